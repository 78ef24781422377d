"""The prefill tile GEMM: edges of its 128-wide tiles (and one whole 256-wide
product), K stages that leave a remainder of its ring, every weight format, E8M0
byte 255; test_gpu_kernels.py has the 256-wide tile's edges and formats.  References are float64 products of the dequantized operands; f32 sums of
k terms in another order stay within sqrt(k) 2^-23 of the products' norm, far
below the 1e-5 of rms used for f32 results; an f16 store is the f32 one rounded."""
import numpy as np
import pytest

import mxfp4hip as M
from mlp_data import MlpData
from test_gpu_stream import E2M1, close, mxfp4

pytestmark = pytest.mark.gpu


# (m, n, k) on the 128-wide tile (4096 x 4096 x 512: the 256-wide one; K = 256: the
# 64-K-stage family): whole, one row or 64 channels past a tile, one row short; then
# K that ends a quarter, half or three quarters into a group of four stages, or in
# the middle of a stage
SHAPES = [(1024, 4096, 256), (1281, 8128, 768), (1000, 4160, 512), (4096, 4096, 512), (4095, 4160, 768), (4097, 2112, 1280),
          (1281, 8128, 320), (4095, 4160, 384), (4095, 4160, 448), (1500, 5013, 288), (4095, 4131, 416), (4097, 2099, 1440)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_matmul_mxfp4(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    q, s, w = mxfp4(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float16)
    da, dq, ds, dc = dev.upload(a), dev.upload(q), dev.upload(s), dev.alloc(m * n * 4 + 64)
    dev.upload(np.full(16, 0x7E7E7E7E, np.uint32), M.DevBuf(dev, dc.ptr + m * n * 4, 64))
    dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F32, m, n, k, ds)
    ref = a.astype(np.float64) @ w.T
    got = dev.download(dc, np.float32, (m, n))
    close(got, ref)
    assert (dev.download(dc.offset(m * n * 4), np.uint32, (16,)) == 0x7E7E7E7E).all()  # nothing past the end
    dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F16, m, n, k, ds)
    assert np.array_equal(dev.download(dc, np.float16, (m, n)), got.astype(np.float16))
    for b in (da, dq, ds, dc):
        b.free()


@pytest.mark.parametrize("k", [512, 800, 1376])
def test_matmul_e8m0_255(dev, k):
    """Byte 255 is +inf: the columns it reaches follow IEEE, the others stand."""
    m, n = 4096, 4160
    rng = np.random.default_rng(5)
    q, s, w = mxfp4(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float16)
    a[7, :] = 0
    a[9, 40] = np.inf
    cols = [0, 255, 300, 4159]
    for c in cols:
        s[c, 3] = 255
    s[300, 3], s[300, -1] = 130, 255  # the row's last block
    w[300] = E2M1[np.stack([q[300] & 15, q[300] >> 4], -1).reshape(k)] * np.repeat(2.0 ** (np.where(s[300] == 255, 127, s[300]).astype(np.float64) - 127), 32)
    q[255, 48:64], w[255, 96:128] = 0x22, 1  # positive codes only: +-inf where the signs of x agree, as in rows 0 to 5
    a[:6] = np.abs(a[:6])
    with np.errstate(invalid="ignore"):
        blk = (w[cols].reshape(len(cols), k // 32, 32) * np.where(s[cols] == 255, np.inf, 1.0)[:, :, None]).reshape(len(cols), k)
        ref = (a[:64].astype(np.float64)[:, None, :] * blk[None]).sum(-1)
    da, dq, ds, dc = dev.upload(a), dev.upload(q), dev.upload(s), dev.alloc(m * n * 4)
    dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F32, m, n, k, ds)
    got = dev.download(dc, np.float32, (m, n))
    assert (ref[:6, 1] == np.inf).all() and np.isnan(ref[7]).all()
    np.testing.assert_array_equal(got[:64, cols].astype(np.float64), ref)  # all NaN or infinite
    keep = np.setdiff1d(np.arange(n), cols)
    rows = np.setdiff1d(np.arange(m), [9])
    close(got[np.ix_(rows, keep)], a[rows].astype(np.float64) @ w[keep].T)
    assert not np.isfinite(got[9, keep]).any()
    for b in (da, dq, ds, dc):
        b.free()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_f16_weights(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float16)
    b = (rng.standard_normal((n, k)) * 0.05).astype(np.float16)
    da, db, dc = dev.upload(a), dev.upload(b), dev.alloc(m * n * 4)
    dev.gemm_f16(da, M.DT_F16, db, dc, m, n, k)
    close(dev.download(dc, np.float32, (m, n)), a.astype(np.float64) @ b.astype(np.float64).T)
    for x in (da, db, dc):
        x.free()


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 256), (4095, 4160, 896), (3841, 4160, 1280)])
def test_gemm_i8_exact(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    b = rng.integers(-127, 128, (n, k)).astype(np.int8)
    da, db, dc = dev.upload(a), dev.upload(b), dev.alloc(m * n * 4)
    dev.gemm_i8(da, db, dc, m, n, k)
    # whole numbers up to k 127^2 < 2^53: exact in float64
    assert np.array_equal(dev.download(dc, np.int32, (m, n)), (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.int64))
    for x in (da, db, dc):
        x.free()


@pytest.mark.parametrize("fmt", [0, -1, M.WFMT_FP8_E4M3, M.WFMT_FP8_E5M2, M.WFMT_INT8, M.WFMT_INT4, M.WFMT_W8A8])
@pytest.mark.parametrize("tokens,h,i", [(1281, 1024, 2816), (4095, 2304, 2304), (2049, 768, 4096), (4095, 1888, 1696)])
def test_mlp_rows(dev, fmt, tokens, h, i):
    """Rows of a large batch against the same rows alone, which other kernels
    run: f32 sums in another order, so f16 mids and results differ by a step
    (2^-10 relative, results up to 6 rms) at most.  -1: REFROW (f32 result)."""
    if fmt == M.WFMT_W8A8 and (h % 128 or i % 128):
        pytest.skip("W8A8 takes multiples of 128")
    d = MlpData(dev, tokens, h, i, seed=tokens + fmt, wfmt=max(fmt, 0))
    out = dev.alloc(tokens * h * 4)
    npdt = np.float32 if fmt < 0 else np.float16

    def run(t, x):
        if fmt > 0:
            dev.fmt_mlp_forward(fmt, t, h, i, x, d.weights, out)
        else:
            dev.mlp_forward(M.MLP_REFROW if fmt else M.MLP_FUSED, t, h, i, x, d.weights, out)
        return dev.download(out, npdt, (t, h))

    got = run(tokens, d.x)
    for lo in (0, tokens // 2, tokens - 24):
        close(got[lo:lo + 24], run(24, M.DevBuf(dev, d.x.ptr + lo * h * 2, 48 * h)).astype(np.float64), 6 * 2 ** -10)
    out.free()
    d.free()
