// Grouped (segmented) Jacobi CG: many independent sparse systems -- the
// requests of a serving batch -- iterate together, two launches per iteration for
// the whole group.
//
// Each system ("segment") keeps its matrix in shared pools at its own offsets
// -- CSR, or SELL-64 with int32 or 16-bit slice-relative columns -- and its
// vectors in shared vector pools; column indices are local to the segment.  A
// block table assigns every block of a launch to one segment and a contiguous
// row range (CSR) or slice range (SELL, one slice per wavefront) of it, so each
// block's partial sums belong to exactly one segment.  Every block of the next launch
// reduces its segment's partials itself, in one fixed order (deterministic, and
// independent of which other segments share the launch); the segment's first block
// records its CG scalars in the other of two state slots, and a one-block-per-segment
// finisher ends a run of iterations.  Converged segments stop at once: their blocks
// return on entry.  Nothing here allocates, synchronises or issues memsets, so a
// chunk of iterations can be captured in a HIP graph and replayed.
//
// Precision per segment (mife_segment.prec).  MIFE_F64 segments iterate in
// FP64 throughout.  MIFE_F32 segments iterate in FP32 (FP32 values, vectors
// and products, FP64 scalars) with reliable updates in FP64, as the
// single-solve mife_refine: the FP64 solution x accumulates the FP32
// correction x32, and whenever a segment's FP32 residual has fallen by
// inner_rtol since its last replacement (tested every check_every iterations),
// x += x32 and the FP32 residual is replaced by the true residual b - A64 x
// computed with the FP64 values; p and q = A p are kept and
// beta = (r.z)_replaced / (r.z)_before-the-step.  Such a segment is done when
// its true FP64 residual meets its tolerance (or at its iteration limit); the
// FP32 recurrence never stops it by itself.  Both kinds share every launch: a
// block takes the branch of its segment's precision.
//
// What bounds it: the matrices of the active segments, read once per iteration.  For
// sixteen FP64 requests of 9 to 139 MB (501 MB) served together, of which the large
// elasticity ones run on to the end, a serving took 223.6 ms with finishers after every
// product and update, replacement passes at every check and all matrices read past the
// caches; 190 ms with the two launches, the passes at the end of a run only (no mixed
// request) and 210 MB of the matrices left to the Infinity Cache; 186 ms with the
// wavefronts of a block sharing a SELL3 slice and the sums formed during the product
// (all sixteen active: product 127 -> 107 us; the last 139 MB one alone: 29.5 -> 25.9).
// One wavefront per SELL3 slice with the sums formed during the product: 188.4 ms.
// One 3,600-slice elasticity request alone: sell3_slices.  A stream of 640 requests, 256 at a
// time, is bound by its large elasticity matrices: 78 solves/s FP64 before and after, 40 to 45
// in mixed precision.
#include "mife_common.hpp"
#include "mife_profile.hpp"
#include "mife_sparse.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mife {

namespace grouped {

constexpr int kL = 8;                  // CSR: lanes per row
constexpr int kRowsPerBlock = 256 / kL;
constexpr int kCsrRows = 4 * kRowsPerBlock;
constexpr int kSlicesPerBlock = 4;     // SELL: one slice per wavefront
constexpr int kSell3Waves = 4;         // SELL3: wavefronts that share a slice (or take one each, sell3_slices)
constexpr int kSell3Rows = 3 * kSlice;
constexpr int kUpdateBlocks = 4;       // blocks of one unit (SELL3: a slice) whose rows one block of the update takes

struct SegState {
  double rz, beta, rr, bb, tol2, rr_true;
  double rz_prev;  // r.z before the last step
  double rr_rep;   // mixed precision: FP32 r.r right after the last replacement
  int iters, maxit, done;
  int pause;       // mixed precision: waiting for an FP64 replacement
  int mixed;       // the segment iterates in FP32 with FP64 reliable updates
  int pad;
};

// The vector pools: FP64 segments use the first set, FP32 segments the second
// (both at the segment's row_off).
struct Vecs {
  double *dinv, *r, *z, *p, *q;
  float *dinv32, *r32, *z32, *p32, *q32, *x32;
};

// Partial values per block slot: 0 and 1 the update's r.z and r.r, 2 the product's
// p.q (a product reads the former while it writes the latter); the initial and
// replaced residuals use the slots from 0.
constexpr int kNumParts = 4;
constexpr int kPartPq = 2;
constexpr int kReplaceGrid = 2048;  // grid of the (mostly idle) replacement passes

struct Block {
  int32_t seg;
  int32_t row0;  // first row (CSR) or first slice (SELL), local to the segment
  int32_t rows;  // rows (CSR) or slices (SELL)
  int32_t part;  // index of this block's partial slot
  int32_t p0, p1;  // the segment's partial slots
  int32_t keep;    // SELL: read the matrix with plain loads (the Infinity Cache keeps it)
  int32_t upd;     // blocks whose rows one block of the update takes
};

struct View {
  const mife_segment* segs;
  const Block* blocks;
  const int32_t* rp;
  const int32_t* col;
  const uint16_t* col16;
  const int32_t* cbase;
  const double* val;
  const float* val32;  // FP32 copy of the values (mixed precision), or null
  SegState* st;   // two slots of nst states each; between runs of iterations the first holds
  double* parts;  // kNumParts values per partial slot: parts[v * cap + slot]
  int cap;
  int nst;
};

// y_row = (A x)_row for the rows of this block's segment, 8 lanes per row;
// vpool is the value pool of the precision T.
template <typename T>
__device__ __forceinline__ T row_dot(const View& V, const mife_segment& S, const T* __restrict__ vpool,
                                     const T* __restrict__ x, int row, int sub) {
  const int32_t* rp = V.rp + S.rp_off;
  const int32_t* col = V.col + S.nz_off;
  const T* val = vpool + S.nz_off;
  const T* xs = x + S.row_off;
  const int k0 = rp[row], k1 = rp[row + 1];
  T a = 0;
  for (int k = k0 + sub; k < k1; k += kL) a += val[k] * xs[col[k]];
#pragma unroll
  for (int off = kL / 2; off > 0; off >>= 1) a += __shfl_xor(a, off, kL);
  return a;
}

// SELL: (A x) of lane `lane`'s row of slice s of the segment (complete sum).
template <typename T>
__device__ __forceinline__ T slice_dot(const View& V, const mife_segment& S, bool keep, const T* __restrict__ vpool,
                                       const T* __restrict__ x, int s, int lane) {
  const int32_t* sp = V.rp + S.rp_off;
  const T* val = vpool + S.nz_off;
  const T* xs = x + S.row_off;
  if (S.cb_off >= 0) {
    const uint16_t* c16 = V.col16 + S.nz_off;
    const int32_t* cb = V.cbase + S.cb_off;
    return keep ? sell16_row<T, T, false>(sp, c16, cb, val, xs, s, lane)
                : sell16_row<T, T, true>(sp, c16, cb, val, xs, s, lane);
  }
  const int32_t* c32 = V.col + S.nz_off;
  return keep ? sell_row<T, T, false>(sp, c32, val, xs, s, lane) : sell_row<T, T, true>(sp, c32, val, xs, s, lane);
}

// block_walk of a block whose wavefronts take a SELL3 slice each (Block::upd == 1): the hook
// first, so that no register holds its operands during the product.
template <typename T, typename P, typename F, typename H>
__device__ __forceinline__ void wave_slices_walk(const View& V, const Block& B, const mife_segment& S,
                                                 const T* __restrict__ vpool, const T* __restrict__ x, P&& pre, F&& f,
                                                 H& hook) {
  hook_now(hook);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave >= B.rows) return;
  const int s = B.row0 + wave;
  const int32_t* sp = V.rp + S.rp_off;
  const int base = sp[s], len = (sp[s + 1] - base) / kSlice;
  T ax[3];
  const uint16_t* c16 = V.col16 + S.nz_off + base + lane;
  const T* v = vpool + S.nz_off + (size_t)9 * base + lane;
  const T* xs = x + S.row_off + 3 * (size_t)V.cbase[S.cb_off + s];
  if (B.keep) sell3_sum<T, T, false>(c16, v, xs, len, 0, 1, ax);
  else sell3_sum<T, T, true>(c16, v, xs, len, 0, 1, ax);
  const int row = s * kSell3Rows + 3 * lane;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    if (row + c < S.n) f(row + c, ax[c], pre(row + c));
}

// Calls f(row, (A x)_row, pre(row)) for every row of block B (by one lane per row).
// On the SELL storages pre's loads and the hook's are in flight during the product;
// hook.stage() and hook.finish() run once per block, a barrier apart, before any f.
template <typename T, typename P, typename F, typename H>
__device__ __forceinline__ void block_walk(const View& V, const Block& B, const mife_segment& S,
                                           const T* __restrict__ vpool, const T* __restrict__ x, P&& pre, F&& f,
                                           H& hook) {
  using PV = decltype(pre(0));
  PV pv = {};
  if (B.upd == 1) {
    wave_slices_walk<T>(V, B, S, vpool, x, pre, f, hook);
    return;
  }
  if (S.format == MIFE_FMT_SELL3 && B.rows > 0) {
    // node rows: lane k of the slice gives rows 3 (64 s + k) + c; block columns in
    // the 16-bit column pool at the segment's value offset.  The wavefronts' shares
    // meet in LDS, from where a thread takes the whole row next to its neighbour's.
    __shared__ T share[kSell3Waves][kSell3Rows];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int s = B.row0;
    const int32_t* sp = V.rp + S.rp_off;
    const int base = sp[s], len = (sp[s + 1] - base) / kSlice;
    const int t = threadIdx.x, row = s * kSell3Rows + t;
    const bool own = t < kSell3Rows && row < S.n;
    if (own) pv = pre(row);
    T ax[3];
    const uint16_t* c16 = V.col16 + S.nz_off + base + lane;
    const T* v = vpool + S.nz_off + (size_t)9 * base + lane;
    const T* xs = x + S.row_off + 3 * (size_t)V.cbase[S.cb_off + s];
    if (B.keep) sell3_sum<T, T, false>(c16, v, xs, len, wave, kSell3Waves, ax);
    else sell3_sum<T, T, true>(c16, v, xs, len, wave, kSell3Waves, ax);
#pragma unroll
    for (int c = 0; c < 3; ++c) share[wave][3 * lane + c] = ax[c];
    hook.stage();
    __syncthreads();
    hook.finish();
    if (own) f(row, (share[0][t] + share[1][t]) + (share[2][t] + share[3][t]), pv);
    return;
  }
  if (S.format == MIFE_FMT_SELL) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int s = B.row0 + wave, row = s * kSlice + lane;
    const bool own = wave < B.rows && row < S.n;
    if (own) pv = pre(row);
    T ax = 0;
    if (wave < B.rows) ax = slice_dot<T>(V, S, B.keep != 0, vpool, x, s, lane);
    hook_now(hook);
    if (own) f(row, ax, pv);
    return;
  }
  hook_now(hook);
  if (S.format != MIFE_FMT_CSR) return;  // the block of an empty segment
  const int lr = threadIdx.x / kL, sub = threadIdx.x % kL;
  for (int row = B.row0 + lr; row < B.row0 + B.rows; row += kRowsPerBlock) {
    const T ax = row_dot<T>(V, S, vpool, x, row, sub);
    if (sub == 0) f(row, ax, pre(row));
  }
}

// Calls f(row, (A x)_row) for every row of a block (by one lane per row); for passes that
// read a matrix once between products: nothing of it is kept.
template <typename T, typename F>
__device__ __forceinline__ void block_rows(const View& V, Block B, const mife_segment& S,
                                           const T* __restrict__ vpool, const T* __restrict__ x, F&& f) {
  NoHook none;
  B.keep = 0;
  block_walk<T>(V, B, S, vpool, x, [](int) { return 0; }, [&](int row, T ax, int) { f(row, ax); }, none);
}

// First and last row of block B.
__device__ __forceinline__ void block_row_range(const Block& B, const mife_segment& S, int& r0, int& r1) {
  if (S.format == MIFE_FMT_SELL3) {
    r0 = B.row0 * 3 * kSlice;
    r1 = min(S.n, (B.row0 + B.rows) * 3 * kSlice);
  } else if (S.format == MIFE_FMT_SELL) {
    r0 = B.row0 * kSlice;
    r1 = min(S.n, (B.row0 + B.rows) * kSlice);
  } else {
    r0 = B.row0;
    r1 = B.row0 + B.rows;
  }
}

// Partials of a segment's updates, and the rows of one of them.
__device__ __forceinline__ int update_blocks(const Block& B) {
  return (B.p1 - B.p0 + B.upd - 1) / B.upd;
}
__device__ __forceinline__ void update_row_range(const Block& B, const mife_segment& S, int& r0, int& r1) {
  const bool csr = S.format == MIFE_FMT_CSR;
  const int units = kUpdateBlocks * (csr ? kCsrRows : S.format == MIFE_FMT_SELL3 ? 1 : kSlicesPerBlock);
  Block all = B;
  all.row0 = (B.part - B.p0) * units;
  all.rows = min(units, (csr ? S.n : S.n_slices) - all.row0);
  block_row_range(all, S, r0, r1);
}

template <int NV, int V0 = 0>
__device__ __forceinline__ void store_partials(const View& V, int slot, double (&m)[NV]) {
  __shared__ double red[NV][4];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const double s = wave_sum(m[v]);
    if ((threadIdx.x & 63) == 0) red[v][threadIdx.x >> 6] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int v = 0; v < NV; ++v) V.parts[(size_t)(V0 + v) * V.cap + slot] = red[v][0] + red[v][1] + red[v][2] + red[v][3];
  }
}

}  // namespace grouped

using namespace grouped;

template <typename T>
__device__ __forceinline__ void diag_body(const View& V, const Block& B, const mife_segment& S,
                                          const T* __restrict__ vpool, T* __restrict__ dinv) {
  if (S.format == MIFE_FMT_SELL3) {
    // node row k: its block at node column k (before the padding, whose column
    // is also k), values 0, 4 and 8
    const int32_t* sp = V.rp + S.rp_off;
    const T* val = vpool + S.nz_off;
    for (int t = threadIdx.x; t < B.rows * kSlice; t += blockDim.x) {
      const int s = B.row0 + t / kSlice, lane = t % kSlice;
      const int k = s * kSlice + lane;
      if (3 * k >= S.n) continue;
      const int base = sp[s], len = (sp[s + 1] - base) / kSlice, cb = V.cbase[S.cb_off + s];
      int jd = -1;
      for (int j = 0; j < len; ++j)
        if (cb + (int)V.col16[S.nz_off + base + j * kSlice + lane] == k) {
          jd = j;
          break;
        }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T d = jd >= 0 ? val[(size_t)9 * (base + jd * kSlice) + 4 * c * kSlice + lane] : (T)0;
        dinv[S.row_off + 3 * k + c] = d != (T)0 ? (T)1 / d : (T)1;
      }
    }
    return;
  }
  int r0, r1;
  block_row_range(B, S, r0, r1);
  const int row = r0 + (int)threadIdx.x;
  if (row >= r1) return;
  T d = 0;
  const T* val = vpool + S.nz_off;
  if (S.format == MIFE_FMT_SELL) {
    const int32_t* sp = V.rp + S.rp_off;
    const int s = row / kSlice, lane = row - s * kSlice;
    for (int e = sp[s] + lane; e < sp[s + 1]; e += kSlice) {
      const int c = S.cb_off >= 0 ? V.cbase[S.cb_off + s] + (int)V.col16[S.nz_off + e] : V.col[S.nz_off + e];
      if (c == row && val[e] != (T)0) {
        d = val[e];
        break;
      }
    }
  } else {
    const int32_t* rp = V.rp + S.rp_off;
    const int32_t* col = V.col + S.nz_off;
    for (int k = rp[row]; k < rp[row + 1]; ++k)
      if (col[k] == row) d = val[k];
  }
  dinv[S.row_off + row] = d != (T)0 ? (T)1 / d : (T)1;
}

// Jacobi diagonal D^-1 of the segment's precision
__global__ __launch_bounds__(256) void gcg_diag_kernel(View V, Vecs W) {
  const Block B = V.blocks[blockIdx.x];
  const mife_segment S = V.segs[B.seg];
  if (S.prec == MIFE_F32)
    diag_body<float>(V, B, S, V.val32, W.dinv32);
  else
    diag_body<double>(V, B, S, V.val, W.dinv);
}

// FP64 segment: r = b - A x, z = D^-1 r, p = q = 0.
// FP32 segment: r64 = b - A64 x, r32 = r64, z32 = D^-1 r32, p32 = q32 = x32 = 0.
// Partials r.z, r.r, b.b and (FP32 segments) r64.r64.
__global__ __launch_bounds__(256) void gcg_init_kernel(View V, Vecs W, const double* __restrict__ b,
                                                       const double* __restrict__ x) {
  const Block B = V.blocks[blockIdx.x];
  const mife_segment S = V.segs[B.seg];
  double m[kNumParts] = {0.0, 0.0, 0.0, 0.0};
  if (S.prec == MIFE_F32) {
    block_rows<double>(V, B, S, V.val, x, [&](int row, double ax) {
      const long long g = S.row_off + row;
      const double r64 = b[g] - ax;
      const float ri = (float)r64;
      const float zi = W.dinv32[g] * ri;
      W.r32[g] = ri;
      W.z32[g] = zi;
      W.p32[g] = 0.0f;
      W.q32[g] = 0.0f;
      W.x32[g] = 0.0f;
      m[0] += (double)ri * (double)zi;
      m[1] += (double)ri * (double)ri;
      m[2] += b[g] * b[g];
      m[3] += r64 * r64;
    });
  } else {
    block_rows<double>(V, B, S, V.val, x, [&](int row, double ax) {
      const long long g = S.row_off + row;
      const double ri = b[g] - ax;
      const double zi = W.dinv[g] * ri;
      W.r[g] = ri;
      W.z[g] = zi;
      W.p[g] = 0.0;
      W.q[g] = 0.0;
      m[0] += ri * zi;
      m[1] += ri * ri;
      m[2] += b[g] * b[g];
    });
  }
  store_partials<kNumParts>(V, B.part, m);
}

// Fixed-order sums, in every thread, of values V0 .. V0 + NV - 1 of the partial slots
// [p0, p1) of a segment.
template <int NV, int V0 = 0>
__device__ __forceinline__ void part_sums(const View& V, int p0, int p1, double (&out)[NV]) {
  __shared__ double red[NV][4];
  double a[NV] = {};
  for (int k = p0 + threadIdx.x; k < p1; k += blockDim.x)
#pragma unroll
    for (int v = 0; v < NV; ++v) a[v] += V.parts[(size_t)(V0 + v) * V.cap + k];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const double s = wave_sum(a[v]);
    if ((threadIdx.x & 63) == 0) red[v][threadIdx.x >> 6] = s;
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; ++v) out[v] = red[v][0] + red[v][1] + red[v][2] + red[v][3];
}

// one block per segment: its slots are [seg_parts[k], seg_parts[k+1]) (k = position
// of the segment in the table)
template <int NV>
__device__ __forceinline__ void seg_sums(const View& V, const int32_t* __restrict__ seg_parts, int k,
                                         double (&out)[NV]) {
  part_sums<NV>(V, seg_parts[k], seg_parts[k + 1], out);
}

__global__ __launch_bounds__(256) void gfin_init_kernel(View V, const int32_t* __restrict__ seg_parts,
                                                        const int32_t* __restrict__ seg_ids) {
  const int s = seg_ids[blockIdx.x];
  double out[kNumParts];
  seg_sums<kNumParts>(V, seg_parts, blockIdx.x, out);
  if (threadIdx.x == 0) {
    SegState& g = V.st[s];
    const mife_segment S = V.segs[s];
    const bool mixed = S.prec == MIFE_F32;
    g.rz = out[0];
    g.rr = out[1];
    g.bb = out[2];
    g.beta = 0.0;
    g.rz_prev = 0.0;
    g.rr_rep = out[1];
    g.iters = 0;
    g.maxit = S.maxit;
    g.tol2 = S.rtol * S.rtol;
    g.rr_true = mixed ? out[3] : -1.0;
    g.pause = 0;
    g.mixed = mixed ? 1 : 0;
    g.done = ((mixed ? out[3] : out[1]) <= g.tol2 * out[2] || S.maxit <= 0) ? 1 : 0;
  }
}

__device__ __forceinline__ bool seg_idle(const SegState& g) { return g.done || g.pause; }

// The scalars of a segment after an iteration's update (sums rz, rr).  FP64 segments:
// done when the recurrence residual meets the tolerance or at maxit.  FP32 segments
// pause for a replacement at maxit and, on a CHECK iteration, once r.r has fallen by
// delta2 since the last replacement or below a quarter of the target.
template <bool CHECK>
__device__ __forceinline__ void seg_advance(SegState& g, double rz, double rr, double delta2) {
  g.rz_prev = g.rz;
  g.beta = g.rz != 0.0 ? rz / g.rz : 0.0;
  g.rz = rz;
  g.rr = rr;
  g.iters += 1;
  if (!g.mixed) {
    g.done = (rr <= g.tol2 * g.bb || g.iters >= g.maxit) ? 1 : 0;
  } else if (g.iters >= g.maxit || (CHECK && (rr <= delta2 * g.rr_rep || rr <= 0.25 * g.tol2 * g.bb))) {
    g.pause = 1;
  }
}

// The state of a segment at iteration k for a block of its product: beta and the
// stopping tests from the previous update's partials (pending), left in the other
// state slot by the segment's first block.  A run's finisher sums them the same way, so
// the iterates do not depend on where the runs end.
struct SegHook {
  static constexpr bool kActive = true;
  static constexpr int kHeld = 3;
  const View& V;
  const Block& B;
  const SegState& in;
  SegState* out;  // null: not the first block's first thread
  double* red;
  int count;      // partials of the update
  bool pending, stop;
  double beta, v[kHeld];
  __device__ __forceinline__ SegHook(const View& view, const Block& blk, const SegState& g, SegState* o, bool pend,
                                     double* r)
      : V(view), B(blk), in(g), out(o), red(r), count(update_blocks(blk)), pending(pend), stop(false), beta(0.0) {
    // wavefront w takes half w >> 1 of sum w & 1
#pragma unroll
    for (int u = 0; u < kHeld; ++u) v[u] = pend && first() + 128 * u < count ? part(first() + 128 * u) : 0.0;
  }
  __device__ __forceinline__ int first() const { return 64 * (threadIdx.x >> 7) + (threadIdx.x & 63); }
  __device__ __forceinline__ double part(int i) const {
    return V.parts[(size_t)(threadIdx.x >> 6 & 1) * V.cap + B.p0 + i];
  }
  __device__ __forceinline__ void stage() {
    if (!pending) return;
    double a = (v[0] + v[1]) + v[2];
    for (int i = first() + 128 * kHeld; i < count; i += 128) a += part(i);
    const double s = wave_sum(a);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  }
  __device__ __forceinline__ void finish() {
    if (pending) {
      advance<false>(0.0);
    } else {
      beta = in.beta;
      if (out) *out = in;
    }
  }
  template <bool CHECK>
  __device__ __forceinline__ void advance(double delta2) {
    SegState c = in;
    seg_advance<CHECK>(c, red[0] + red[2], red[1] + red[3], delta2);
    beta = c.beta;
    stop = seg_idle(c);
    if (out) *out = c;
  }
};

template <typename T>
struct RowZpq {
  T z, p, q;
};

template <typename T>
__device__ __forceinline__ void spmv_body(const View& V, const Block& B, const mife_segment& S, SegHook& hook,
                                          const T* __restrict__ vpool, const T* __restrict__ z,
                                          T* __restrict__ p, T* __restrict__ q) {
  double m[1] = {0.0};
  block_walk<T>(
      V, B, S, vpool, z,
      [&](int row) {
        const long long g = S.row_off + row;
        return RowZpq<T>{z[g], p[g], q[g]};
      },
      [&](int row, T az, const RowZpq<T>& o) {
        if (hook.stop) return;
        const long long g = S.row_off + row;
        const T beta = (T)hook.beta;
        const T pi = o.z + beta * o.p;
        const T qi = az + beta * o.q;
        p[g] = pi;
        q[g] = qi;
        m[0] += (double)pi * (double)qi;
      },
      hook);
  if (hook.stop) return;
  store_partials<1, kPartPq>(V, B.part, m);
}

// Iteration k of a run: p = z + beta p ; q = A z + beta q ; partial p.q (in the
// segment's precision).  A run's first iteration takes the state as it is; later ones
// find the previous update's sums while their product's loads are in flight (a segment
// that turns out to have converged drops this one product).
__global__ __launch_bounds__(256) void gcg_spmv_kernel(View V, Vecs W, int k, int pending) {
  __shared__ double red[4];
  const Block B = V.blocks[blockIdx.x];
  const SegState& in = V.st[(k & 1) * V.nst + B.seg];
  SegState* out = threadIdx.x == 0 && B.part == B.p0 ? &V.st[((k + 1) & 1) * V.nst + B.seg] : nullptr;
  if (seg_idle(in)) {
    if (out) *out = in;
    return;
  }
  SegHook hook(V, B, in, out, pending != 0, red);
  const mife_segment S = V.segs[B.seg];
  if (S.prec == MIFE_F32)
    spmv_body<float>(V, B, S, hook, V.val32, W.z32, W.p32, W.q32);
  else
    spmv_body<double>(V, B, S, hook, V.val, W.z, W.p, W.q);
}

template <typename T>
__device__ __forceinline__ void update_body(const View& V, const Block& B, const mife_segment& S, double rz,
                                            T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                            const T* __restrict__ p, const T* __restrict__ q,
                                            const T* __restrict__ dinv) {
  constexpr int D = 4;  // rows per thread in flight: all of a block's (3 x 256 SELL3, 4 x 256 SELL, 2 x 256 CSR)
  int r0, r1;
  update_row_range(B, S, r0, r1);
  T xi[D], ri[D], pi[D], qi[D], di[D];
#pragma unroll
  for (int u = 0; u < D; ++u) {
    const int row = r0 + 256 * u + (int)threadIdx.x;
    const long long g = S.row_off + (row < r1 ? row : r0);
    if (row < r1) xi[u] = x[g], ri[u] = r[g], pi[u] = p[g], qi[u] = q[g], di[u] = dinv[g];
  }
  double pq[1];
  part_sums<1, kPartPq>(V, B.p0, B.p1, pq);
  const T alpha = (T)(pq[0] != 0.0 ? rz / pq[0] : 0.0);
  double m[2] = {0.0, 0.0};
#pragma unroll
  for (int u = 0; u < D; ++u) {
    const int row = r0 + 256 * u + (int)threadIdx.x;
    if (row < r1) {
      const long long g = S.row_off + row;
      x[g] = xi[u] + alpha * pi[u];
      const T rn = ri[u] - alpha * qi[u];
      const T zn = di[u] * rn;
      r[g] = rn;
      z[g] = zn;
      m[0] += (double)rn * (double)zn;
      m[1] += (double)rn * (double)rn;
    }
  }
  store_partials<2>(V, B.part, m);
}

// alpha = r.z / p.q from the product's partials; x += alpha p ; r -= alpha q ;
// z = D^-1 r ; partials r.z, r.r (x: the FP64 solution of FP64 segments; FP32 segments
// update their correction x32).  Block i of a segment takes the rows of blocks
// kUpdateBlocks i onwards; the rest return (the first ones work, not every
// kUpdateBlocks-th, so that all XCDs have work).
__global__ __launch_bounds__(256) void gcg_update_kernel(View V, Vecs W, double* __restrict__ x, int k) {
  const Block B = V.blocks[blockIdx.x];
  if (B.part - B.p0 >= update_blocks(B)) return;
  const SegState& g = V.st[((k + 1) & 1) * V.nst + B.seg];
  if (seg_idle(g)) return;
  const mife_segment S = V.segs[B.seg];
  if (S.prec == MIFE_F32)
    update_body<float>(V, B, S, g.rz, W.x32, W.r32, W.z32, W.p32, W.q32, W.dinv32);
  else
    update_body<double>(V, B, S, g.rz, x, W.r, W.z, W.p, W.q, W.dinv);
}

// End of a run of `count` iterations, one block per segment: the last one's scalars
// (unless the segment already stopped), left in the first state slot.
__global__ __launch_bounds__(256) void gfin_beta_kernel(View V, const int32_t* __restrict__ seg_parts, int count,
                                                        double delta2) {
  __shared__ double red[4];
  const Block B = V.blocks[seg_parts[blockIdx.x]];
  const SegState in = V.st[(count & 1) * V.nst + B.seg];
  SegState* out = threadIdx.x == 0 ? &V.st[B.seg] : nullptr;
  if (seg_idle(in)) {
    if (out) *out = in;
    return;
  }
  SegHook hook(V, B, in, out, true, red);
  hook.stage();
  __syncthreads();
  hook.advance<true>(delta2);
}

// Reliable update, part 1 (paused segments): x += x32, x32 = 0.  Grid-stride
// over the block table.
__global__ __launch_bounds__(256) void gmx_fold_kernel(View V, Vecs W, int n_blocks, double* __restrict__ x) {
  for (int bi = blockIdx.x; bi < n_blocks; bi += gridDim.x) {
    const Block B = V.blocks[bi];
    const SegState& g = V.st[B.seg];
    if (!g.pause || g.done) continue;
    const mife_segment S = V.segs[B.seg];
    int r0, r1;
    block_row_range(B, S, r0, r1);
    for (int row = r0 + threadIdx.x; row < r1; row += 256) {
      const long long i = S.row_off + row;
      x[i] += (double)W.x32[i];
      W.x32[i] = 0.0f;
    }
  }
}

// Reliable update, part 2 (paused segments): r64 = b - A64 x with the FP64
// values, r32 = r64, z32 = D^-1 r32; partials r32.z32, r32.r32, r64.r64.
// Grid-stride over the block table.
__global__ __launch_bounds__(256) void gmx_replace_kernel(View V, Vecs W, int n_blocks, const double* __restrict__ b,
                                                          const double* __restrict__ x) {
  for (int bi = blockIdx.x; bi < n_blocks; bi += gridDim.x) {
    const Block B = V.blocks[bi];
    const SegState& g = V.st[B.seg];
    if (!g.pause || g.done) continue;
    const mife_segment S = V.segs[B.seg];
    double m[3] = {0.0, 0.0, 0.0};
    block_rows<double>(V, B, S, V.val, x, [&](int row, double ax) {
      const long long i = S.row_off + row;
      const double r64 = b[i] - ax;
      const float ri = (float)r64;
      const float zi = W.dinv32[i] * ri;
      W.r32[i] = ri;
      W.z32[i] = zi;
      m[0] += (double)ri * (double)zi;
      m[1] += (double)ri * (double)ri;
      m[2] += r64 * r64;
    });
    store_partials<3>(V, B.part, m);
    __syncthreads();  // the block's LDS partials are reused by its next table entry
  }
}

// Reliable update, part 3 (one block per paused segment): beta from the
// replaced r.z (0 when the replaced r.r exceeds the recurrence's by
// kRestartGrowth), the true residual and the stopping test; resumes the segment.
__global__ __launch_bounds__(256) void gfin_replace_kernel(View V, const int32_t* __restrict__ seg_parts,
                                                           const int32_t* __restrict__ seg_ids) {
  const int s = seg_ids[blockIdx.x];
  if (!V.st[s].pause || V.st[s].done) return;
  double out[3];
  seg_sums<3>(V, seg_parts, blockIdx.x, out);
  if (threadIdx.x == 0) {
    SegState& g = V.st[s];
    g.beta = (g.rz_prev != 0.0 && out[1] <= kRestartGrowth * g.rr) ? out[0] / g.rz_prev : 0.0;
    g.rz = out[0];
    g.rr = out[1];
    g.rr_rep = out[1];
    g.rr_true = out[2];
    g.pause = 0;
    g.done = (out[2] <= g.tol2 * g.bb || g.iters >= g.maxit) ? 1 : 0;
  }
}

// true residual ||b - A x||^2 of the listed segments
__global__ __launch_bounds__(256) void gcg_resid_kernel(View V, const double* __restrict__ b,
                                                        const double* __restrict__ x) {
  const Block B = V.blocks[blockIdx.x];
  const mife_segment S = V.segs[B.seg];
  double m[1] = {0.0};
  block_rows<double>(V, B, S, V.val, x, [&](int row, double ax) {
    const double ri = b[S.row_off + row] - ax;
    m[0] += ri * ri;
  });
  store_partials<1>(V, B.part, m);
}

__global__ __launch_bounds__(256) void gfin_resid_kernel(View V, const int32_t* __restrict__ seg_parts,
                                                         const int32_t* __restrict__ seg_ids) {
  const int s = seg_ids[blockIdx.x];
  double out[1];
  seg_sums<1>(V, seg_parts, blockIdx.x, out);
  if (threadIdx.x == 0) V.st[s].rr_true = out[0];
}

}  // namespace mife

using namespace mife;
using namespace mife::grouped;

namespace {

// Device layout of a table, carved from the caller's work buffer:
//   mife_segment[max_seg] (by slot) | Block[max_blocks] | seg_parts[max_seg+1] |
//   seg_ids[max_seg] | parts[kNumParts * max_blocks]
// The per-slot CG scalars live in a separate state buffer, so tables can be
// rebuilt (segments joining or leaving) while the other segments keep iterating.
struct Layout {
  mife_segment* segs;
  Block* blocks;
  int32_t* seg_parts;
  int32_t* seg_ids;
  double* parts;
};

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

Layout carve(void* work, int max_seg, int max_blocks) {
  char* p = (char*)work;
  Layout L;
  size_t off = 0;
  L.segs = (mife_segment*)(p + off);
  off = align256(off + sizeof(mife_segment) * max_seg);
  L.blocks = (Block*)(p + off);
  off = align256(off + sizeof(Block) * max_blocks);
  L.seg_parts = (int32_t*)(p + off);
  off = align256(off + sizeof(int32_t) * (max_seg + 1));
  L.seg_ids = (int32_t*)(p + off);
  off = align256(off + sizeof(int32_t) * max_seg);
  L.parts = (double*)(p + off);
  return L;
}

}  // namespace

extern "C" {

size_t mife_grouped_state_bytes(int max_segments) { return 2 * sizeof(SegState) * (size_t)max_segments + 256; }

size_t mife_grouped_work_bytes(int max_segments, int max_blocks) {
  size_t b = 0;
  b = align256(b + sizeof(mife_segment) * max_segments);
  b = align256(b + sizeof(Block) * max_blocks);
  b = align256(b + sizeof(int32_t) * (max_segments + 1));
  b = align256(b + sizeof(int32_t) * max_segments);
  b += sizeof(double) * kNumParts * (size_t)max_blocks + 256;
  return b;
}

// Slices that a block of a SELL3 product takes: one, its wavefronts sharing it, or four, one
// each.  Sharing gives a small segment blocks enough for the chip.  A large one has them
// anyway, and then long runs per wavefront, a quarter of the partials and a hook before the
// product cost less.  Shared / one each, ms for one elasticity request to 1e-8, FP64: 810
// slices 49.7 / 55.2, 1,451 86.4 / 88.8, 1,871 133.6 / 127.8, 3,600 305.6 / 289.9 (product 96
// -> 91 us, update 13 -> 10); FP32 with FP64 replacements: 810 slices 88.1 / 88.5, 1,099 123
// / 113, 1,871 219 / 215, 3,600 545 / 446.  By the segment's own size alone, so that its
// sums do not depend on what it shares a launch with.
static int sell3_slices(int n_slices, int prec) { return n_slices < (prec == MIFE_F32 ? 1000 : 1700) ? 1 : 4; }

int mife_grouped_blocks(int n_rows) { return std::max(1, div_up(n_rows, kCsrRows)); }

int mife_grouped_setup(const mife_segment* segs_host, int n_seg, int max_segments, int max_blocks,
                       int* n_blocks_out, void* table_host, void* work, void* stream) {
  MIFE_REQUIRE(segs_host && work && n_blocks_out && table_host, MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  MIFE_REQUIRE(n_seg >= 0 && n_seg <= max_segments, MIFE_ERR_ARG, "too many segments (%d > %d)", n_seg,
               max_segments);
  // host staging buffer (caller-owned pinned or pageable memory of
  // mife_grouped_work_bytes) holding segs | blocks | seg_parts | seg_ids
  Layout D = carve(work, max_segments, max_blocks);
  Layout H = carve(table_host, max_segments, max_blocks);
  int nb = 0;
  double kept = 0.0;  // bytes of the matrices read with plain loads so far (27 entries per row)
  for (int k = 0; k < n_seg; ++k) {
    const mife_segment& S = segs_host[k];
    MIFE_REQUIRE(S.n >= 0, MIFE_ERR_ARG, "segment %d has %d rows", k, S.n);
    MIFE_REQUIRE(S.slot >= 0 && S.slot < max_segments, MIFE_ERR_ARG, "segment slot %d out of range", S.slot);
    MIFE_REQUIRE(S.format == MIFE_FMT_CSR || (S.format == MIFE_FMT_SELL && S.n_slices == div_up(S.n, kSlice)) ||
                     (S.format == MIFE_FMT_SELL3 && S.n % 3 == 0 && S.n_slices == div_up(S.n / 3, kSlice) &&
                      S.cb_off >= 0),
                 MIFE_ERR_ARG, "segment %d: format %d / n_slices %d", k, S.format, S.n_slices);
    MIFE_REQUIRE(S.prec == MIFE_F64 || S.prec == MIFE_F32, MIFE_ERR_ARG, "segment %d: precision %d", k, S.prec);
    H.segs[S.slot] = S;
    H.seg_parts[k] = nb;
    H.seg_ids[k] = S.slot;
    const bool sell = S.format != MIFE_FMT_CSR;
    const int per = S.format == MIFE_FMT_SELL3 ? sell3_slices(S.n_slices, S.prec) : sell ? kSlicesPerBlock : kCsrRows;
    const int units = sell ? S.n_slices : S.n;
    // as many matrices as the Infinity Cache holds stay there between the products.  A
    // product reads a value of the segment's precision and its share of a column per
    // entry; how many entries a row has is not in the table, so trilinear rows are assumed
    // (a wrong guess costs cache hits, nothing else)
    const bool nodes = S.format == MIFE_FMT_SELL3;
    const double value = S.prec == MIFE_F32 ? 4.0 : 8.0;
    const double column = nodes ? 2.0 / 9.0 : S.cb_off >= 0 && S.format == MIFE_FMT_SELL ? 2.0 : 4.0;
    const double bytes = (nodes ? 81.0 : 27.0) * S.n * (value + column);
    const int keep = kept + bytes <= kKeepMost ? 1 : 0;
    if (keep) kept += bytes;
    const int p0 = nb, p1 = nb + std::max(1, div_up(units, per));
    int r0 = 0;
    do {
      MIFE_REQUIRE(nb < max_blocks, MIFE_ERR_ARG, "block table full (%d blocks)", max_blocks);
      H.blocks[nb] = Block{S.slot, r0, std::max(0, std::min(per, units - r0)), nb, p0, p1, keep,
                            S.format == MIFE_FMT_SELL3 ? kUpdateBlocks / per : kUpdateBlocks};
      ++nb;
      r0 += per;
    } while (r0 < units);
  }
  H.seg_parts[n_seg] = nb;
  hipStream_t st = (hipStream_t)stream;
  if (n_seg > 0) {
    MIFE_CHECK_HIP(hipMemcpyAsync(D.segs, H.segs, sizeof(mife_segment) * max_segments, hipMemcpyHostToDevice, st));
    MIFE_CHECK_HIP(hipMemcpyAsync(D.blocks, H.blocks, sizeof(Block) * nb, hipMemcpyHostToDevice, st));
    MIFE_CHECK_HIP(
        hipMemcpyAsync(D.seg_parts, H.seg_parts, sizeof(int32_t) * (n_seg + 1), hipMemcpyHostToDevice, st));
    MIFE_CHECK_HIP(hipMemcpyAsync(D.seg_ids, H.seg_ids, sizeof(int32_t) * n_seg, hipMemcpyHostToDevice, st));
    MIFE_CHECK_HIP(hipStreamSynchronize(st));  // the host staging buffer may be reused at once
  }
  *n_blocks_out = nb;
  return MIFE_OK;
}

static View make_view(const Layout& D, void* state, const mife_pools* P, int cap, int max_seg) {
  return View{D.segs, D.blocks, P->rp,           P->col,  P->col16, P->cbase,
              P->val, P->val32, (SegState*)state, D.parts, cap,      max_seg};
}

static Vecs make_vecs(double* vec5, float* vec6, int64_t rows) {
  return Vecs{vec5, vec5 + rows, vec5 + 2 * rows, vec5 + 3 * rows, vec5 + 4 * rows,
              vec6, vec6 + rows, vec6 + 2 * rows, vec6 + 3 * rows, vec6 + 4 * rows, vec6 + 5 * rows};
}

int mife_grouped_cg_init(int n_seg, int n_blocks, int max_segments, int max_blocks, const mife_pools* pools,
                         const double* b, const double* x, double* vec5, float* vec6, int64_t pool_rows, void* work,
                         void* state, void* stream) {
  MIFE_REQUIRE(pools && pools->rp && pools->val && pools->val32 && b && x && vec5 && vec6 && work && state,
               MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  if (n_seg == 0) return MIFE_OK;
  hipStream_t s = (hipStream_t)stream;
  Layout D = carve(work, max_segments, max_blocks);
  View V = make_view(D, state, pools, max_blocks, max_segments);
  Vecs W = make_vecs(vec5, vec6, pool_rows);
  gcg_diag_kernel<<<n_blocks, 256, 0, s>>>(V, W);
  gcg_init_kernel<<<n_blocks, 256, 0, s>>>(V, W, b, x);
  gfin_init_kernel<<<n_seg, 256, 0, s>>>(V, D.seg_parts, D.seg_ids);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

int mife_grouped_cg_iterate(int n_seg, int n_blocks, int max_segments, int max_blocks, const mife_pools* pools,
                            const double* b, double* x, double* vec5, float* vec6, int64_t pool_rows,
                            int iterations, int check_every, double inner_rtol, void* work, void* state,
                            void* stream) {
  MIFE_REQUIRE(pools && pools->rp && pools->val && pools->val32 && b && x && vec5 && vec6 && work && state,
               MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  MIFE_REQUIRE(check_every >= 1 && inner_rtol > 0.0 && inner_rtol < 1.0, MIFE_ERR_ARG,
               "invalid check_every %d / inner_rtol %g", check_every, inner_rtol);
  if (n_seg == 0) return MIFE_OK;
  hipStream_t s = (hipStream_t)stream;
  Layout D = carve(work, max_segments, max_blocks);
  View V = make_view(D, state, pools, max_blocks, max_segments);
  Vecs W = make_vecs(vec5, vec6, pool_rows);
  const double delta2 = inner_rtol * inner_rtol;
  const int rg = std::min(n_blocks, kReplaceGrid);
  for (int it = 0, k = 0; it < iterations; ++it, ++k) {
    const int tk = prof::begin(s);
    gcg_spmv_kernel<<<n_blocks, 256, 0, s>>>(V, W, k, k > 0 ? 1 : 0);
    prof::end(tk, s, prof::kGroupedSpmv);
    const int tk2 = prof::begin(s);
    gcg_update_kernel<<<n_blocks, 256, 0, s>>>(V, W, x, k);
    prof::end(tk2, s, prof::kGroupedUpdate);
    if ((it + 1) % check_every == 0 || it + 1 == iterations) {
      gfin_beta_kernel<<<n_seg, 256, 0, s>>>(V, D.seg_parts, k + 1, delta2);
      k = -1;  // the next iteration starts a run
      gmx_fold_kernel<<<rg, 256, 0, s>>>(V, W, n_blocks, x);
      const int tk3 = prof::begin(s);
      gmx_replace_kernel<<<rg, 256, 0, s>>>(V, W, n_blocks, b, x);
      prof::end(tk3, s, prof::kGroupedReplace);
      gfin_replace_kernel<<<n_seg, 256, 0, s>>>(V, D.seg_parts, D.seg_ids);
    }
  }
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

int mife_grouped_cg_residual(int n_seg, int n_blocks, int max_segments, int max_blocks, const mife_pools* pools,
                             const double* b, const double* x, void* work, void* state, void* stream) {
  MIFE_REQUIRE(pools && pools->rp && pools->val && b && x && work && state, MIFE_ERR_POINTER_IS_NULL,
               "null pointer argument");
  if (n_seg == 0) return MIFE_OK;
  hipStream_t s = (hipStream_t)stream;
  Layout D = carve(work, max_segments, max_blocks);
  View V = make_view(D, state, pools, max_blocks, max_segments);
  gcg_resid_kernel<<<n_blocks, 256, 0, s>>>(V, b, x);
  gfin_resid_kernel<<<n_seg, 256, 0, s>>>(V, D.seg_parts, D.seg_ids);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

int mife_grouped_cg_status(int max_segments, const void* state, int* iters, int* done, double* relres,
                           void* stream) {
  MIFE_REQUIRE(state && iters && done && relres, MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  hipStream_t s = (hipStream_t)stream;
  std::vector<SegState> h(max_segments);
  MIFE_CHECK_HIP(hipMemcpyAsync(h.data(), state, sizeof(SegState) * max_segments, hipMemcpyDeviceToHost, s));
  MIFE_CHECK_HIP(hipStreamSynchronize(s));
  for (int i = 0; i < max_segments; ++i) {
    iters[i] = h[i].iters;
    done[i] = h[i].done;
    const double rr = h[i].rr_true >= 0.0 ? h[i].rr_true : h[i].rr;
    relres[i] = h[i].bb > 0.0 ? sqrt(rr / h[i].bb) : 0.0;
  }
  return MIFE_OK;
}

}  // extern "C"
