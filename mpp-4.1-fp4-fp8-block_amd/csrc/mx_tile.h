// mx_tile.h - launchers of the prefill tile GEMM's instances (mx_gemm_tile.h).
#pragma once

#include <hip/hip_runtime.h>

#include "mx_internal.h"

namespace mx {
namespace tile {

// side: 256 or 128 (tile rows and weight rows)
hipError_t launch_mxfp4(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_int4(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_e4m3(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_e5m2(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_int8(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_f16(int side, int epi, const QGemmArgs& g, hipStream_t st);
hipError_t launch_i8(int epi, const QGemmArgs& g, hipStream_t st);  // W8A8: 256

}  // namespace tile
}  // namespace mx
