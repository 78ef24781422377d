"""Epilogues that a GEMM launcher does not have are refused before any launch
(CPU: an unrefused call would reach the runtime and report the missing device)."""
import ctypes
import os
import struct

import pytest

import mxfp4hip as M

INVALID = 1  # hipErrorInvalidValue
STORE_F32, STORE_F16, SWIGLU_F16, SWIGLU_HALF, SWIGLU_F32, STORE_I32, SWIGLU_F8X2 = range(7)
pytestmark = pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="a GPU is present: unrefused calls would launch")


@pytest.mark.parametrize("epi", [STORE_F32, SWIGLU_HALF, SWIGLU_F32, STORE_I32, SWIGLU_F8X2])
@pytest.mark.parametrize("rows", [20, 200])
def test_grouped_epilogues(epi, rows):
    """Grouped launches write f16 only: SwiGLU to f16 and the f16 store."""
    args = bytearray(160)
    struct.pack_into("3i", args, 64, rows, 256, 4096)  # QGemmArgs: eight pointers, then m, n, k
    table = bytearray(1048)
    struct.pack_into("3i", table, 0, 0, rows, rows + 1)
    f = getattr(M.load(), "_ZN2mx21launch_gemm_q_groupedEiRKNS_9QGemmArgsERKNS_10GroupTableEiP12ihipStream_t")
    buf = lambda b: (ctypes.c_char * len(b)).from_buffer(b)
    assert f(epi, buf(args), buf(table), 2, None) == INVALID


@pytest.mark.parametrize("epi", [SWIGLU_F32, STORE_I32, SWIGLU_F8X2])
@pytest.mark.parametrize("dtype", [M.DT_F16, M.DT_F32])
def test_off_grid_epilogues(epi, dtype):
    args = bytearray(72)
    struct.pack_into("Pi", args, 0, 0, dtype)          # GemmArgs: a, its dtype, five pointers, m, n, k
    struct.pack_into("3i", args, 56, 4, 96, 160)
    f = getattr(M.load(), "_ZN2mx13launch_gemm_hEiiRKNS_8GemmArgsEP12ihipStream_t")
    assert f(1, epi, (ctypes.c_char * 72).from_buffer(args), None) == INVALID
