// mx_stream.h - launchers of the weight-streaming GEMM (mx_gemm_stream.h),
// shared by its instance files and the choice between them (mx_stream.cpp).
#pragma once

#include "mx_internal.h"

namespace mx {
namespace stream {

constexpr int kScales = 16384;  // LDS for the scale copy (a launch takes fewer groups when K needs more)

struct Args {
  const void* a;
  const float* a_scale;             // AK_I8: per activation row
  const uint8_t *b0, *b1;           // weights (b1: up)
  const uint8_t *s0, *s1;           // scales
  void* c;
  int m, n, k, epi;                 // n: weight rows (SwiGLU: channels); grouped: m of the largest group
  int m_tiles, n_tiles;             // set by the launcher
};

// rows: activation rows of a tile (4, 8, 16 or 32), ng: groups of 16 weight rows of a workgroup (1, 2 or 4)
hipError_t launch_mxfp4(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_f32_mxfp4(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_e4m3(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_e5m2(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_int8(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_i8(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_f16(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_f32_f16(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_int4(const Args& g, int rows, int ng, hipStream_t st);
hipError_t launch_mxfp4_grouped(const Args& g, const GroupTable& gt, int groups, int rows, int ng, hipStream_t st);

}  // namespace stream
}  // namespace mx
