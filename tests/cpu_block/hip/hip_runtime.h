// Runs device code of this library on the CPU, one block at a time, every thread of
// the block a fiber: enough of the HIP names for kernels without matrix instructions.
// A barrier that some threads of a block never reach (they have returned) is counted,
// and non-temporal loads are counted.  Lanes exchange values when all lanes of their
// wavefront that can run have come to an exchange.
#pragma once
#include <ucontext.h>

#include <algorithm>
#include <bit>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)

using std::max;
using std::min;
struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct int4 {
  int x, y, z, w;
};
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0;
inline const char* hipGetErrorString(hipError_t) { return ""; }

namespace emu {
struct Index {
  int x, y, z;
};
enum Wait { kRun, kWave, kBlock, kDone };
struct Fiber {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack;
  Wait wait;
  uint64_t slot[2];  // exchanged values, by parity of the exchange
  unsigned ops;
};
inline Index thread, block, block_dim, grid_dim;
inline std::vector<Fiber> fibers;
inline ucontext_t home;
inline int current;
inline long partial_barriers, streamed_loads;
inline std::function<void()> body;

inline void yield(Wait w) {
  Fiber& f = fibers[current];
  f.wait = w;
  swapcontext(&f.ctx, &home);
}
inline void entry() {
  body();
  fibers[current].wait = kDone;
  swapcontext(&fibers[current].ctx, &home);
}
// value of lane `from` of this wavefront
inline uint64_t exchange(uint64_t v, int from) {
  Fiber& f = fibers[current];
  const int at = f.ops++ & 1, wave0 = current & ~63;
  f.slot[at] = v;
  yield(kWave);
  return fibers[wave0 + (from & 63)].slot[at];
}
inline void run_block(int threads) {
  fibers = std::vector<Fiber>(threads);
  for (int t = 0; t < threads; ++t) {
    Fiber& f = fibers[t];
    f.stack.reset(new char[1 << 16]);
    f.wait = kRun;
    f.ops = 0;
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.get();
    f.ctx.uc_stack.ss_size = 1 << 16;
    f.ctx.uc_link = &home;
    makecontext(&f.ctx, entry, 0);
  }
  while (true) {
    int at[4] = {0, 0, 0, 0};
    for (int t = 0; t < threads; ++t) {
      if (fibers[t].wait == kRun) {
        current = t;
        thread = {t, 0, 0};
        swapcontext(&home, &fibers[t].ctx);
      }
      ++at[fibers[t].wait];
    }
    if (at[kDone] == threads) return;
    const Wait next = at[kWave] ? kWave : kBlock;
    if (next == kBlock && at[kDone]) ++partial_barriers;
    for (auto& f : fibers)
      if (f.wait == next) f.wait = kRun;
  }
}
template <typename F>
void launch(dim3 grid, int threads, F&& f) {
  body = f;
  block_dim = {threads, 1, 1};
  grid_dim = {(int)grid.x, (int)grid.y, (int)grid.z};
  for (unsigned y = 0; y < grid.y; ++y)
    for (unsigned x = 0; x < grid.x; ++x) {
      block = {(int)x, (int)y, 0};
      run_block(threads);
    }
}
template <typename T>
T load(const T* p) {
  ++streamed_loads;
  return *p;
}
inline int dpp_lane(int ctrl) {
  const int l = current & 63;
  switch (ctrl) {
    case 0xB1: return l ^ 1;
    case 0x4E: return l ^ 2;
    case 0x141: return l ^ 7;
    case 0x140: return l ^ 15;
  }
  std::abort();
}
}  // namespace emu

#define threadIdx emu::thread
#define blockIdx emu::block
#define blockDim emu::block_dim
#define gridDim emu::grid_dim
#define __builtin_nontemporal_load(p) emu::load(p)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, l) ((int)emu::exchange((uint32_t)(v), (l)))
#define __builtin_amdgcn_mov_dpp(v, c, a, b, d) ((int)emu::exchange((uint32_t)(v), emu::dpp_lane(c)))
inline void __syncthreads() { emu::yield(emu::kBlock); }
template <typename T>
T __shfl_xor(T v, int off, int = 64) {
  uint64_t u = 0;
  std::memcpy(&u, &v, sizeof(T));
  u = emu::exchange(u, (emu::current & 63) ^ off);
  std::memcpy(&v, &u, sizeof(T));
  return v;
}
template <typename T>
T atomicAdd(T* p, T v) {
  const T o = *p;
  *p += v;
  return o;
}
inline int __double2loint(double v) { return (int)(uint32_t)std::bit_cast<uint64_t>(v); }
inline int __double2hiint(double v) { return (int)(std::bit_cast<uint64_t>(v) >> 32); }
inline double __hiloint2double(int h, int l) { return std::bit_cast<double>((uint64_t)(uint32_t)h << 32 | (uint32_t)l); }
inline long long __double_as_longlong(double v) { return std::bit_cast<long long>(v); }
inline double __longlong_as_double(long long v) { return std::bit_cast<double>(v); }
inline int __float_as_int(float v) { return std::bit_cast<int>(v); }
inline float __int_as_float(int v) { return std::bit_cast<float>(v); }
