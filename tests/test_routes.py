"""Which kernel a GEMM runs on (host logic, no GPU): the launchers' rules against
GEMMs where one side was measured at least 1.2 times as fast as the other."""
import pytest

import test_gpu_kernels as G
from gemm_route import (E4M3, F16, F32, I8, INT4, INT8, MXFP4, STORE_F16, STORE_F32, STORE_I32, SWIGLU_F16,
                        SWIGLU_F32, W_F16, W_I8, mlp_routes, moe_streams, route)


# (activations, weights, epilogue, m, n, k, streaming is faster): us streaming / tiled
ON_GRID = [
    (F16, MXFP4, STORE_F16, 1001, 3648, 512, False),    # 24.7 / 9.2
    (F16, MXFP4, SWIGLU_F16, 1856, 1344, 128, False),   # 23.9 / 6.6
    (F16, MXFP4, STORE_F16, 512, 7168, 512, False),     # 23.7 / 9
    (F16, MXFP4, STORE_F16, 1458, 1088, 1216, False),   # 21.6 / 12.7
    (F16, MXFP4, SWIGLU_F16, 34, 12416, 2560, False),   # 26.0 / 14.1
    (F16, E4M3, SWIGLU_F16, 385, 1408, 256, False),     # 15.6 / 4.8
    (F16, E4M3, SWIGLU_F16, 1072, 640, 1408, False),    # 26.9 / 16.3
    (F16, INT8, SWIGLU_F16, 1179, 1920, 256, False),    # 37.7 / 8.6
    (F16, INT4, STORE_F16, 1096, 4032, 256, False),     # 29.5 / 8.9
    (F16, INT4, STORE_F16, 1024, 2944, 2560, False),    # 46.2 / 25.6
    (I8, W_I8, SWIGLU_F32, 1664, 640, 256, False),      # 23.6 / 6.2
    (I8, W_I8, STORE_F16, 440, 2688, 512, False),       # 18.4 / 9.3
    (F16, W_F16, STORE_F32, 820, 960, 512, False),      # 27 / 13 (1014 rows)
    (F32, W_F16, STORE_F16, 2680, 384, 832, False),     # 46.7 / 23.5
    (F16, MXFP4, SWIGLU_F16, 40, 2048, 7168, True),     # 11.9 / 19.9
    (F16, MXFP4, STORE_F16, 40, 7168, 2048, True),
    (F16, MXFP4, SWIGLU_F16, 64, 2048, 7168, True),     # 12.4 / 21.0
    (F16, MXFP4, SWIGLU_F16, 8, 14336, 4096, True),     # 17.7 / 22.0
    (F16, E4M3, STORE_F16, 64, 7168, 2048, True),       # 12.5 / 16.0
    (F16, INT4, SWIGLU_F16, 73, 128, 128, True),        # 2.9 / 4.9
    (I8, W_I8, SWIGLU_F32, 64, 2048, 7168, True),       # 14.3 / 18.6
    (F32, MXFP4, STORE_F16, 64, 4096, 4096, True),      # 15.4 / 24.7
]


@pytest.mark.parametrize("ak,bk,epi,m,n,k,stream", ON_GRID)
def test_streaming_where_it_is_faster(ak, bk, epi, m, n, k, stream):
    assert (route(ak, bk, epi, m, n, k) == "stream") is stream


# us streaming / the K-step-32 kernel
OFF_GRID = [
    (F32, W_F16, STORE_F16, 1536, 864, 128, False),     # 31.7 / 4.8
    (F16, MXFP4, SWIGLU_F16, 2004, 800, 160, False),    # 20.8 / 5.6
    (F16, E4M3, STORE_F16, 1616, 1056, 64, False),      # 15.9 / 4.6
    (F16, INT8, SWIGLU_F16, 1488, 672, 128, False),     # 19.4 / 5.9
    (F16, INT4, STORE_F16, 609, 1632, 192, False),      # 11.8 / 4.7
    (F16, W_F16, STORE_F32, 820, 960, 96, False),       # 9.5 / 3.1
    (F32, W_F16, STORE_F16, 1344, 1152, 3552, False),   # 145 / 75
    (F16, MXFP4, STORE_F16, 257, 2080, 5536, True),     # 23 / 125
    (F16, MXFP4, STORE_F16, 1, 2080, 5536, True),       # 5.9 / 108
    (F16, INT4, STORE_F16, 120, 8736, 1248, True),      # 19.2 / -
]


@pytest.mark.parametrize("ak,bk,epi,m,n,k,stream", OFF_GRID)
def test_streaming_off_the_grid(ak, bk, epi, m, n, k, stream):
    assert (route(ak, bk, epi, m, n, k) == "stream") is stream


@pytest.mark.parametrize("counts,n,k,stream", [
    ([14] * 62 + [5, 5], 320, 448, False),   # 64 experts, 878 tokens, 448 -> 320 -> 448: 31 us a pass streaming, 18 tiled
    ([7] * 64, 448, 128, False),             # 64 experts, 452 tokens, 128 -> 448
    ([4] * 60 + [25, 7, 0, 0], 2048, 7168, True),   # 281 / 712
    ([64] * 8, 2048, 7168, True),            # 130 / 166
    ([128] * 8, 1408, 4096, False),          # 104 / 90
    ([94] * 32, 1024, 2304, False),          # 153 / 101
])
def test_grouped_streaming_where_it_is_faster(counts, n, k, stream):
    assert moe_streams(counts, SWIGLU_F16, n, k) is stream


def test_gpu_cases_reach_their_kernels():
    for a, b, m, n, k, kernel in G.MATMULS:
        assert route(a, b, STORE_F32, m, n, k) == kernel, (a, b, m, n, k)
    for fmt, t, h, i, up, down in G.MLPS:
        assert mlp_routes(fmt, t, h, i) == (up, down), (fmt, t, h, i)
    for m, n, k in G.I8:
        assert route(I8, W_I8, STORE_I32, m, n, k) == "tile256"
    for _, t, h, i in G.E8M0_255:
        assert mlp_routes(0, t, h, i) == ("q", "q")
    for t, h, i, up, down in G.INT4_SCALES:
        assert mlp_routes(G.M.WFMT_INT4, t, h, i) == (up, down)
    counts, h, i = G.MOE_Q
    assert not moe_streams(counts, SWIGLU_F16, i, h) and not moe_streams(counts, STORE_F16, h, i)
