"""Every GEMM kernel at sizes that the launchers send to it, against the oracle or
a float64 product: the K-step-32 kernel (h), the 64-K-stage family (q) and the
256-wide prefill tile, each in the formats and epilogues it has.  ROUTES lists
(sizes, kernel) of every case; test_routes.py checks it where there is no GPU, so
a rule that moves a case to another kernel shows there.  Tolerances: f32 sums of
k terms in another order stay within sqrt(k) 2^-23 of the products' norm, far
below the 1e-5 of rms used for f32 results (f32 activations as two f16 terms:
2^-22 a value); MLPs are held to the oracle's tolerance."""
import types

import numpy as np
import pytest

import gemm_route as R
import mxfp4hip as M
import oracle as O
from mlp_data import MlpData, sample_rows
from test_gpu_moe import MoeData
from test_gpu_stream import close, mxfp4

pytestmark = pytest.mark.gpu
TOL, COS = O.MAX_ABS_REL_TOL, O.COSINE_TOL
FP8_INT = [M.WFMT_FP8_E4M3, M.WFMT_FP8_E5M2, M.WFMT_INT8, M.WFMT_INT4]

# (activations, weights, m, n, k, kernel): plain products.  h: 64- and 128-row
# tiles, a ragged last row tile, n off 32 and off 64.  tile256: ragged in both
# directions, K in the middle of a stage and of a group of four.
MATMULS = [(a, b, *s) for a in (R.F16, R.F32) for b in (R.MXFP4, R.W_F16)
           for s in ((600, 801, 160, "h"), (1500, 2075, 96, "h"))]
MATMULS += [(R.F32, b, 2048, 2080, 1056, "h") for b in (R.MXFP4, R.W_F16)]
MATMULS += [(R.F16, R.MXFP4, 2049, 7040, 288, "tile256"), (R.F16, R.MXFP4, 1500, 10691, 352, "tile256"),
            (R.F16, R.W_F16, 1500, 10691, 352, "tile256"), (R.F16, R.W_F16, 4096, 4096, 512, "tile256"),
            (R.F16, R.MXFP4, 1024, 4096, 256, "q"), (R.F16, R.W_F16, 1024, 4096, 256, "q")]

# (tokens, hidden, intermediate, gate/up kernel, down kernel), by weight format (0
# FUSED, -1 REFROW)
MLPS = [(f, *s) for f in (0, -1, *FP8_INT) for s in (
    (300, 160, 2080, "h", "stream"), (1500, 2080, 96, "stream", "h"))]
MLPS += [(f, 700, 1088, 1024, "q", "q") for f in (0, -1)]
MLPS += [(f, 260, 2048, 1024, "q", "q") for f in (M.WFMT_FP8_E4M3, M.WFMT_FP8_E5M2, M.WFMT_INT8, M.WFMT_W8A8)]
MLPS += [(M.WFMT_INT4, 900, 2048, 1024, "q", "q")]
MLPS += [(f, 700, 1632, 10880, "tile256", "stream" if f <= 0 else "tile128") for f in (0, -1, *FP8_INT)]
MLPS += [(M.WFMT_W8A8, 1000, 896, 7936, "tile256", "q"), (M.WFMT_W8A8, 4095, 4096, 2048, "tile256", "tile256")]

I8 = [(999, 16320, 1152), (1000, 15872, 896)]                       # tile256
E8M0_255 = [("gate", 700, 1088, 1024), ("down", 700, 1088, 1024)]   # q, q
INT4_SCALES = [(200, 2048, 4096, "q", "stream"), (128, 4096, 14336, "tile128", "q"), (32, 4096, 14336, "stream", "stream")]
MOE_Q = ([700, 0, 650, 17], 7168, 512)


@pytest.mark.parametrize("a,b,m,n,k,kernel", MATMULS)
def test_matmul(dev, a, b, m, n, k, kernel):
    assert R.route(a, b, R.STORE_F32, m, n, k) == kernel
    rng = np.random.default_rng(m + n + k)
    x = rng.standard_normal((m, k)).astype(np.float32 if a == R.F32 else np.float16)
    adt = M.DT_F32 if a == R.F32 else M.DT_F16
    dx, dc = dev.upload(x), dev.alloc(m * n * 4 + 64)
    dev.upload(np.full(16, 0x7E7E7E7E, np.uint32), M.DevBuf(dev, dc.ptr + m * n * 4, 64))
    bufs = [dx, dc]
    if b == R.MXFP4:
        q, s, w = mxfp4(rng, n, k)
        bufs += [dev.upload(q), dev.upload(s)]
        dev.mxfp4_matmul(dx, adt, bufs[2], dc, M.DT_F32, m, n, k, bufs[3])
    else:
        w = (rng.standard_normal((n, k)) * 0.05).astype(np.float16).astype(np.float64)
        bufs.append(dev.upload(w.astype(np.float16)))
        dev.gemm_f16(dx, adt, bufs[2], dc, m, n, k)
    got = dev.download(dc, np.float32, (m, n))
    close(got, x.astype(np.float64) @ w.T)
    assert (dev.download(dc.offset(m * n * 4), np.uint32, (16,)) == 0x7E7E7E7E).all()  # nothing past the end
    if b == R.MXFP4:  # the same sums, rounded
        dev.mxfp4_matmul(dx, adt, bufs[2], dc, M.DT_F16, m, n, k, bufs[3])
        assert np.array_equal(dev.download(dc, np.float16, (m, n)), got.astype(np.float16))
    for buf in bufs:
        buf.free()


def run(dev, d, fmt):
    out = dev.alloc(d.T * d.H * 4)
    if fmt > 0:
        dev.fmt_mlp_forward(fmt, d.T, d.H, d.I, d.x, d.weights, out)
    else:
        dev.mlp_forward(M.MLP_REFROW if fmt else M.MLP_FUSED, d.T, d.H, d.I, d.x, d.weights, out)
    got = dev.download(out, np.float32 if fmt < 0 else np.float16, (d.T, d.H))
    out.free()
    return got


def oracle(d, fmt, rows):
    x, ((qg, sg), (qu, su), (qd, sd)) = d.host()
    if fmt > 0:
        return O.mlp_format(fmt, x, qg, sg, qu, su, qd, sd, d.H, d.I, rows=rows, threads=16)
    return O.mlp_mxfp4(O.MLP_REFROW if fmt else O.MLP_F16, x, qg, sg, qu, su, qd, sd, d.H, d.I, rows=rows, threads=16)


@pytest.mark.parametrize("fmt,t,h,i,up,down", MLPS)
def test_mlp(dev, fmt, t, h, i, up, down):
    assert R.mlp_routes(fmt, t, h, i) == (up, down)
    d = MlpData(dev, t, h, i, seed=t + fmt, wfmt=max(fmt, 0))
    rows = sample_rows(t, 16)
    got = run(dev, d, fmt)
    assert np.isfinite(got).all()
    rel, cos = O.mlp_error(got[rows], oracle(d, fmt, rows))
    print(f"format {fmt} {t} x {h} x {i}: rel={rel:.3e} cos={cos:.7f}", flush=True)
    # the reference row (swiglu_half, f32 stores): as in test_gpu_shapes.py
    assert rel <= (2e-3 if fmt == -1 else TOL) and cos >= COS
    d.free()


@pytest.mark.parametrize("m,n,k", I8)
def test_gemm_i8_exact(dev, m, n, k):
    assert R.route(R.I8, R.W_I8, R.STORE_I32, m, n, k) == "tile256"
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.integers(-128, 128, (r, k)).astype(np.int8) for r in (m, n))
    a[0], b[0], a[-1], b[-1] = -128, -128, 127, -128  # the largest sums
    da, db, dc = dev.upload(a), dev.upload(b), dev.alloc(m * n * 4)
    dev.gemm_i8(da, db, dc, m, n, k)
    # whole numbers up to k 2^14 < 2^53: exact in float64
    assert np.array_equal(dev.download(dc, np.int32, (m, n)), (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.int64))
    for x in (da, db, dc):
        x.free()


def plant_255(dev, d, which, row):
    """E8M0 255 on one block of a weight row and on all of the last row, 0 on another."""
    _, s, n, k = d.mats[{"gate": 0, "up": 1, "down": 2}[which]]
    sc = dev.download(s, np.uint8, (n, k // 32))
    sc[row, 2], sc[n - 1], sc[100, 0] = 255, 255, 0
    dev.upload(sc, s)


def same_nonfinite(got, ref):
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(ref))
    fin = np.isfinite(ref)
    assert not fin.all()
    if fin.any():
        rel, cos = O.mlp_error(got[fin], ref[fin])
        assert rel <= TOL and cos >= COS


@pytest.mark.parametrize("which,t,h,i", E8M0_255)
def test_64_k_stage_e8m0_255(dev, which, t, h, i):
    """Byte 255 (+inf in the reference, MXFP4Kernels.metal:26-29) on the 64-K-stage
    family's f16 x MXFP4 form, in the gate/up and the down GEMM."""
    assert R.mlp_routes(0, t, h, i) == ("q", "q")
    d = MlpData(dev, t, h, i, seed=7)
    plant_255(dev, d, which, 3)
    rows = sample_rows(t, 48)
    same_nonfinite(run(dev, d, 0)[rows].astype(np.float64), oracle(d, 0, rows))
    d.free()


def test_256_tile_e8m0_255(dev):
    """The 256-tile runs a wave's K loop again where byte 255 made its sums NaN:
    the columns follow IEEE, the others stand, K in the middle of a stage."""
    m, n, k = 1500, 10691, 352
    assert R.route(R.F16, R.MXFP4, R.STORE_F32, m, n, k) == "tile256"
    rng = np.random.default_rng(11)
    q, s, w = mxfp4(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    x[:4] = np.abs(x[:4]) + np.float16(0.25)
    x[m - 1] = 0                                     # 0 x inf: NaN
    cols = [0, 255, 256, n - 1]
    for c in cols:
        s[c, 10] = 255                               # the last block, half a stage
        q[c, 160:176] = 0x22                         # codes +1.0
    da, dq, ds, dc = dev.upload(x), dev.upload(q), dev.upload(s), dev.alloc(m * n * 4)
    dev.mxfp4_matmul(da, M.DT_F16, dq, dc, M.DT_F32, m, n, k, ds)
    got = dev.download(dc, np.float32, (m, n))
    assert (got[:4, cols] == np.inf).all() and np.isnan(got[m - 1, cols]).all()
    signs = np.sign(x[:, 320:].astype(np.float32))   # inf of each product's sign: one infinity, or NaN if both (or a 0)
    assert np.array_equal(np.isposinf(got[:, cols[1]]), (signs > 0).all(1)) and not np.isfinite(got[:, cols]).any()
    keep = np.setdiff1d(np.arange(n), cols)
    close(got[:, keep], x.astype(np.float64) @ w[keep].T)
    for b in (da, dq, ds, dc):
        b.free()


@pytest.mark.parametrize("t,h,i,up,down", INT4_SCALES)
def test_int4_scale_planes_4_byte_aligned(dev, t, h, i, up, down):
    """INT4 scale planes at a 4-byte boundary give the bits of aligned ones: the
    deep ring's LDS copy (q, gate/up), the 2-slot and split-K forms that load a
    chunk's scales from memory (q, down), the tile kernel and streaming."""
    assert R.mlp_routes(M.WFMT_INT4, t, h, i) == (up, down)
    d = MlpData(dev, t, h, i, seed=43, wfmt=M.WFMT_INT4)
    ref = run(dev, d, M.WFMT_INT4)
    assert np.isfinite(ref).all()
    moved = []
    for _, s, n, k in d.mats:
        host = dev.download(s, np.uint8, (n * (k // 32) * 2,))
        moved.append(dev.upload(np.concatenate([np.zeros(4, np.uint8), host, np.zeros(12, np.uint8)])))
    d.weights = M.Device.weights(*[(q, types.SimpleNamespace(ptr=b.ptr + 4)) for (q, _, _, _), b in zip(d.mats, moved)])
    assert np.array_equal(run(dev, d, M.WFMT_INT4).view(np.uint16), ref.view(np.uint16))
    for b in moved:
        b.free()
    d.free()


def test_moe_64_k_stage_long_k(dev):
    """Grouped gate/up on the 64-K-stage family at 7168 K: its E8M0 scales (28 KB a
    workgroup) do not fit the LDS copy, so each lane loads a chunk's with one
    8-byte load; planes at a 4-byte boundary take byte loads, and give the same
    bits."""
    counts, h, i = MOE_Q
    assert not R.moe_streams(counts, R.SWIGLU_F16, i, h) and not R.moe_streams(counts, R.STORE_F16, h, i)
    d = MoeData(dev, counts, h, i, seed=95)
    got = d.run()
    rows, t0 = [], 0
    for cnt in counts:
        rows += [t0, t0 + cnt // 2, t0 + cnt - 1] if cnt else []
        t0 += cnt
    rel, cos = O.mlp_error(got[rows], d.oracle(rows=rows)[rows])
    assert np.isfinite(got).all() and rel <= TOL and cos >= COS
    moved = []
    for _, s, n, k in d.mats:
        host = dev.download(s, np.uint8, (n * (k // 32),))
        moved.append(dev.upload(np.concatenate([np.zeros(4, np.uint8), host, np.zeros(12, np.uint8)])))
    d.weights = M.Device.weights(*[(q, types.SimpleNamespace(ptr=b.ptr + 4)) for (q, _, _, _), b in zip(d.mats, moved)])
    assert np.array_equal(d.run().view(np.uint16), got.view(np.uint16))
    for b in moved:
        b.free()
    d.free()
