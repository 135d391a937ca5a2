// Shared definitions for the mi_fe HIP library (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cstdarg>

#include "../../include/mife.h"

namespace mife {

// Thread-local last-error text, returned by mife_last_error().
void set_error(const char* fmt, ...);

#define MIFE_CHECK_HIP(expr)                                                  \
  do {                                                                        \
    hipError_t _e = (expr);                                                   \
    if (_e != hipSuccess) {                                                   \
      ::mife::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                        __FILE__, __LINE__);                                  \
      return MIFE_ERR_HIP;                                                    \
    }                                                                         \
  } while (0)

#define MIFE_REQUIRE(cond, code, ...)  \
  do {                                 \
    if (!(cond)) {                     \
      ::mife::set_error(__VA_ARGS__);  \
      return (code);                   \
    }                                  \
  } while (0)

constexpr int kWave = 64;

// Wavefront sum (64 lanes), the result in every lane.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// A double from another lane of the same 16-lane row (DPP control CTRL).
template <int CTRL>
__device__ __forceinline__ double row_lane(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// An eight-byte value of lane `lane`, as a scalar.
template <typename V>
__device__ __forceinline__ V lane_value(V v, int lane) {
  static_assert(sizeof(V) == 8, "eight bytes");
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned int lo = __builtin_amdgcn_readlane((int)(unsigned int)u, lane);
  const unsigned int hi = __builtin_amdgcn_readlane((int)(unsigned int)(u >> 32), lane);
  return __builtin_bit_cast(V, ((unsigned long long)hi << 32) | lo);
}

template <int CTRL>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sums over aligned groups of 8 or 16 lanes, the same bits in every lane of a group.
template <typename T>
__device__ __forceinline__ T sum8(T v) {
  v += row_lane<0xB1>(v);         // quad_perm [1,0,3,2]
  v += row_lane<0x4E>(v);         // quad_perm [2,3,0,1]
  return v + row_lane<0x141>(v);  // row_half_mirror
}
__device__ __forceinline__ double sum16(double v) {
  v = sum8(v);
  return v + row_lane<0x140>(v);  // row_mirror
}

// The FP64 sum (64 active lanes), the same bits in every lane: pairs, quads, eights
// and sixteens by DPP, the four row sums through scalar registers.  A reduction in
// LDS shuffles is a chain of six round trips to the LDS, of which a solver's
// iteration holds several.
__device__ __forceinline__ double wave_sum(double v) {
  v = sum16(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// Block-wide sum; `scratch` must hold blockDim.x/64 values. All threads get the result.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* scratch) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  const int nw = (blockDim.x + kWave - 1) / kWave;
  T s = 0;
  for (int i = 0; i < nw; ++i) s += scratch[i];
  return s;
}

inline int div_up(long long a, long long b) { return (int)((a + b - 1) / b); }

}  // namespace mife
