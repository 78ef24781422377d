"""The weight-streaming GEMM (few rows, sizes off the 64-wide grid): its tile
edges (4, 8, 16, 32 rows; 16 to 64 weight rows; 128 K a step, 4 waves), every
weight and activation format, ragged n and k, scale planes at any alignment,
E8M0 byte 255, and uneven MoE groups.  References are float64 products of the
dequantized operands; f32 sums of k terms in another order stay within
sqrt(k) 2^-23 of the products' norm, far below the 1e-5 of rms used here."""
import numpy as np
import pytest

import mxfp4hip as M
import oracle as O
from mlp_data import MlpData

pytestmark = pytest.mark.gpu
E2M1 = np.array([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6])


def mxfp4(rng, n, k):
    q = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    s = rng.integers(118, 136, (n, k // 32), dtype=np.uint8)
    v = E2M1[np.stack([q & 15, q >> 4], -1).reshape(n, k)] * np.repeat(2.0 ** (s.astype(np.float64) - 127), 32, 1)
    return q, s, v


def close(got, ref, tol=1e-5):
    rms = np.sqrt((ref ** 2).mean())
    err = np.abs(got.astype(np.float64) - ref).max() / rms
    assert err <= tol, err


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16, 17, 32, 33, 65])
@pytest.mark.parametrize("n,k", [(64, 128), (1, 32), (130, 1056), (1000, 640), (2048, 96)])
def test_matmul_tile_edges(dev, m, n, k):
    rng = np.random.default_rng(m * 7 + n + k)
    q, s, w = mxfp4(rng, n, k)
    dq, ds = dev.upload(q), dev.upload(s)
    for adt, npdt in ((M.DT_F16, np.float16), (M.DT_F32, np.float32)):
        a = rng.standard_normal((m, k)).astype(npdt)
        da, dc = dev.upload(a), dev.alloc(m * n * 4 + 64)
        dev.upload(np.full(16, 0x7E7E7E7E, np.uint32), M.DevBuf(dev, dc.ptr + m * n * 4, 64))
        dev.mxfp4_matmul(da, adt, dq, dc, M.DT_F32, m, n, k, ds)
        close(dev.download(dc, np.float32, (m, n)), a.astype(np.float64) @ w.T)
        assert (dev.download(dc.offset(m * n * 4), np.uint32, (16,)) == 0x7E7E7E7E).all()  # nothing past the end
        da.free(), dc.free()
    dq.free(), ds.free()


@pytest.mark.parametrize("off", [1, 2, 4, 8])
def test_matmul_scale_plane_alignment(dev, off):
    """The scale copy's 16-byte, 8-byte and byte paths give the same bits."""
    m, n, k = 9, 192, 1024
    rng = np.random.default_rng(off)
    q, s, _ = mxfp4(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float16)
    da, dq, ds, dc = dev.upload(a), dev.upload(q), dev.upload(s), dev.alloc(m * n * 4)
    sh = dev.alloc(s.size + 16)
    dev.upload(s, M.DevBuf(dev, sh.ptr + off, s.size))
    outs = []
    for sc in (ds, M.DevBuf(dev, sh.ptr + off, s.size)):
        dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F32, m, n, k, sc)
        outs.append(dev.download(dc, np.uint32, (m, n)))
    assert np.array_equal(*outs)
    for b in (da, dq, ds, dc, sh):
        b.free()


@pytest.mark.parametrize("adt,npdt", [(M.DT_F16, np.float16), (M.DT_F32, np.float32)])
@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (16, 100, 96), (32, 2000, 1056), (33, 512, 64)])
def test_gemm_f16_weights(dev, adt, npdt, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(npdt)
    b = (rng.standard_normal((n, k)) * 0.05).astype(np.float16)
    da, db, dc = dev.upload(a), dev.upload(b), dev.alloc(m * n * 4)
    dev.gemm_f16(da, adt, db, dc, m, n, k)
    close(dev.download(dc, np.float32, (m, n)), a.astype(np.float64) @ b.astype(np.float64).T)
    for x in (da, db, dc):
        x.free()


@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (8, 192, 256), (9, 4096, 384), (17, 64, 1152), (33, 128, 4096)])
def test_gemm_i8_exact(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    b = rng.integers(-127, 128, (n, k)).astype(np.int8)
    da, db, dc = dev.upload(a), dev.upload(b), dev.alloc(m * n * 4)
    dev.gemm_i8(da, db, dc, m, n, k)
    assert np.array_equal(dev.download(dc, np.int32, (m, n)), a.astype(np.int64) @ b.astype(np.int64).T)
    for x in (da, db, dc):
        x.free()


@pytest.mark.parametrize("wfmt", [M.WFMT_FP8_E4M3, M.WFMT_FP8_E5M2, M.WFMT_INT8, M.WFMT_INT4, M.WFMT_W8A8])
@pytest.mark.parametrize("T,H,I", [(1, 128, 256), (9, 1152, 640), (24, 640, 1152), (40, 256, 4608)])
def test_format_mlp(dev, wfmt, T, H, I):
    d = MlpData(dev, T, H, I, seed=T + H + wfmt, wfmt=wfmt)
    out = dev.alloc(T * H * 2)
    dev.fmt_mlp_forward(wfmt, T, H, I, d.x, d.weights, out)
    x, ((qg, sg), (qu, su), (qd, sd)) = d.host()
    rel, cos = O.mlp_error(dev.download(out, np.float16, (T, H)), O.mlp_format(wfmt, x, qg, sg, qu, su, qd, sd, H, I))
    assert rel <= O.MAX_ABS_REL_TOL and cos >= O.COSINE_TOL, (rel, cos)
    out.free()
    d.free()


@pytest.mark.parametrize("m,k", [(3, 1056), (20, 4096)])
def test_matmul_byte_255(dev, m, k):
    """Byte 255 is +inf: a block of it gives +-inf, or NaN where a code is
    zero or signs meet, and only in its own column."""
    n = 48
    rng = np.random.default_rng(k)
    q, s, w = mxfp4(rng, n, k)
    a = np.abs(rng.standard_normal((m, k)).astype(np.float16)) + np.float16(0.1)
    q[5, 64:80] = 0x22  # column 5, one block of positive codes: +inf
    s[5, 4] = 255
    q[40, -16:] = 0xAA  # column 40, the last block negative: -inf
    s[40, -1] = 255
    s[17, 0] = 255      # column 17, random codes: NaN (zeros or both signs among 32)
    da, dq, ds, dc = dev.upload(a), dev.upload(q), dev.upload(s), dev.alloc(m * n * 4)
    dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F32, m, n, k, ds)
    got = dev.download(dc, np.float32, (m, n))
    assert (got[:, 5] == np.inf).all() and (got[:, 40] == -np.inf).all() and np.isnan(got[:, 17]).all()
    keep = [c for c in range(n) if c not in (5, 17, 40)]
    close(got[:, keep], (a.astype(np.float64) @ w.T)[:, keep])
    for b in (da, dq, ds, dc):
        b.free()


@pytest.mark.parametrize("I", [160, 192, 224])
def test_int4_last_scale_infinite(dev, I):
    """An infinite f16 scale on a row's last block, where K ends within a
    128-K step: +-inf where the block's codes have one sign, nowhere else."""
    T, H = 5, 128
    d = MlpData(dev, T, H, I, seed=I, wfmt=M.WFMT_INT4)
    x, mats = d.host()
    x = np.abs(x) + np.float16(0.1)
    for q, _ in mats[:2]:
        q[I - 32:] = 0x11  # the last 32 mid channels are positive
    qd, sd = mats[2]
    qd[5, -16:], qd[H - 1, -16:] = 0x11, 0xFF
    sd[[5, H - 1], -1] = np.inf
    for host, buf in [(x, d.x)] + [(h, b) for hs, bs in zip(mats, d.mats) for h, b in zip(hs, bs)]:
        dev.upload(host, buf)
    out = dev.alloc(T * H * 2)
    dev.fmt_mlp_forward(M.WFMT_INT4, T, H, I, d.x, d.weights, out)
    got = dev.download(out, np.float16, (T, H))
    assert (got[:, 5] == np.inf).all() and (got[:, H - 1] == -np.inf).all(), got[:, [5, H - 1]]
    keep = np.setdiff1d(np.arange(H), [5, H - 1])
    sd[[5, H - 1], -1] = 1
    ref = O.mlp_format(M.WFMT_INT4, x, *mats[0], *mats[1], *mats[2], H, I)
    rel, cos = O.mlp_error(got[:, keep], ref[:, keep])
    assert rel <= O.MAX_ABS_REL_TOL and cos >= O.COSINE_TOL, (rel, cos)
    out.free()
    d.free()


@pytest.mark.parametrize("counts,H,I", [
    ([25, 0, 3, 17, 1, 8, 9, 33], 512, 384),   # 16-row tiles, all tile bodies, an empty group
    ([90, 1, 40, 33], 256, 1152),              # 32-row tiles
    ([40, 2], 192, 64),                        # sizes the GEMV does not take
])
def test_moe_uneven(dev, counts, H, I):
    E, T = len(counts), sum(counts)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, H)).astype(np.float16)
    mats = []
    for n, k in ((E * I, H), (E * I, H), (E * H, I)):
        q, s = O.mxfp4_quantize(rng.normal(0, 0.05, (n, k)).astype(np.float32))
        mats.append((q, s))
    bufs = [(dev.upload(q), dev.upload(s)) for q, s in mats]
    dx, out = dev.upload(x), dev.alloc(T * H * 2)
    dev.moe_forward(H, I, counts, dx, M.Device.weights(*bufs), out)
    got = dev.download(out, np.float16, (T, H))
    t0 = 0
    for e, c in enumerate(counts):
        if c:
            (qg, sg), (qu, su), (qd, sd) = [(q[e * n:(e + 1) * n], s[e * n:(e + 1) * n])
                                            for (q, s), n in zip(mats, (I, I, H))]
            ref = O.mlp_mxfp4(O.MLP_F16, x[t0:t0 + c], qg, sg, qu, su, qd, sd, H, I)
            rel, cos = O.mlp_error(got[t0:t0 + c], ref)
            assert rel <= O.MAX_ABS_REL_TOL and cos >= O.COSINE_TOL, (e, rel, cos)
        t0 += c
    for b in (dx, out, *[y for z in bufs for y in z]):
        b.free()
