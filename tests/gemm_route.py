"""The kernel that a GEMM runs on (host logic of the library, no GPU), for tests
written for one kernel: they check that their sizes still reach it."""
import ctypes
import struct

import mxfp4hip as M

F16, F32, I8, F8X2 = range(4)                                            # activations
W_F16, MXFP4, E4M3, E5M2, INT8, INT4, W_I8 = range(7)                    # weights
STORE_F32, STORE_F16, SWIGLU_F16, SWIGLU_HALF, SWIGLU_F32, STORE_I32, SWIGLU_F8X2 = range(7)
KERNELS = ("small", "stream", "kq", "tile128", "tile256", "q", "h")


def route(ak, bk, epi, m, n, k):
    """One of KERNELS, for operands at 16-byte boundaries."""
    args = bytearray(160)
    struct.pack_into("3i", args, 64, m, n, k)                            # QGemmArgs: eight pointers, then m, n, k
    f = getattr(M.load(), "_ZN2mx11gemm_kernelEiiiRKNS_9QGemmArgsE")
    return KERNELS[f(ak, bk, epi, (ctypes.c_char * 160).from_buffer(args))]


def mlp_routes(fmt, t, h, i):
    """(gate/up, down) of an MLP.  fmt: 0 FUSED, -1 REFROW, or a weight format."""
    if fmt == M.WFMT_W8A8:
        return route(I8, W_I8, SWIGLU_F32, t, i, h), route(I8, W_I8, STORE_F16, t, h, i)
    bk = {0: MXFP4, -1: MXFP4, M.WFMT_FP8_E4M3: E4M3, M.WFMT_FP8_E5M2: E5M2, M.WFMT_INT8: INT8, M.WFMT_INT4: INT4}[fmt]
    up, down = (SWIGLU_HALF, STORE_F32) if fmt == -1 else (SWIGLU_F16, STORE_F16)
    return route(F16, bk, up, t, i, h), route(F16, bk, down, t, h, i)


def moe_streams(counts, epi, n, k):
    """Whether a grouped GEMM runs on the streaming kernel."""
    table = (ctypes.c_int * 262)()                                       # off[257], then the strides
    for e, c in enumerate(counts):
        table[e + 1] = table[e] + c
    f = getattr(M.load(), "_ZN2mx19stream_wins_groupedEiiiRKNS_10GroupTableEi")
    f.restype = ctypes.c_bool
    return f(epi, n, k, table, len(counts))
