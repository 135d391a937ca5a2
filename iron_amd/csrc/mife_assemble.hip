// Element integration + scatter-add into CSR values.
//
// One 64-lane wavefront integrates one element (trilinear hexahedra: eight, further
// down): lanes gather the element's
// node coordinates into LDS, one lane per Gauss point forms dx/dxi, its
// inverse and |J| (always FP64), then the lanes build the physical gradients
// B[(g,i)][a] and contract K = B^T W B in the value precision T, and finally
// add K into the CSR values through the precomputed position map.  Colours
// are launched one after another, so every CSR entry is updated by at most one
// wavefront per launch and the summation order is fixed (deterministic).
#include "mife_common.hpp"
#include "mife_grid.hpp"
#include "mife_profile.hpp"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace mife {

struct Mat3 {
  double a[3][3];
};

// 2x2 / 3x3 inverse by cofactors (maths.F90 InvertFullDP ordering of terms), every
// multiply-add written out: the bits do not depend on what the compiler fuses around it.
template <int DIM>
__device__ __forceinline__ double invert(const double (&A)[3][3], double (&B)[3][3]) {
#pragma clang fp contract(off)
  // a b - c d
  auto minor = [](double a, double b, double c, double d) {
#pragma clang fp contract(off)
    return fma(a, b, -(c * d));
  };
  if constexpr (DIM == 2) {
    const double det = minor(A[0][0], A[1][1], A[1][0], A[0][1]);
    B[0][0] = A[1][1] / det;
    B[0][1] = -A[0][1] / det;
    B[1][0] = -A[1][0] / det;
    B[1][1] = A[0][0] / det;
    return det;
  } else {
    double det = fma(A[0][0] * A[1][1], A[2][2], (A[0][1] * A[1][2]) * A[2][0]);
    det = fma(A[0][2] * A[1][0], A[2][1], det);
    det = fma(-(A[0][0] * A[2][1]), A[1][2], det);
    det = fma(-(A[1][0] * A[0][1]), A[2][2], det);
    det = fma(-(A[2][0] * A[1][1]), A[0][2], det);
    B[0][0] = minor(A[1][1], A[2][2], A[2][1], A[1][2]) / det;
    B[1][0] = minor(A[1][2], A[2][0], A[2][2], A[1][0]) / det;
    B[2][0] = minor(A[1][0], A[2][1], A[2][0], A[1][1]) / det;
    B[0][1] = minor(A[2][1], A[0][2], A[0][1], A[2][2]) / det;
    B[1][1] = minor(A[2][2], A[0][0], A[0][2], A[2][0]) / det;
    B[2][1] = minor(A[2][0], A[0][1], A[0][0], A[2][1]) / det;
    B[0][2] = minor(A[0][1], A[1][2], A[1][1], A[0][2]) / det;
    B[1][2] = minor(A[0][2], A[1][0], A[1][2], A[0][0]) / det;
    B[2][2] = minor(A[0][0], A[1][1], A[1][0], A[0][1]) / det;
    return det;
  }
}

template <typename T>
__device__ __forceinline__ void add_value(T* p, T v, bool atomic) {
  if (atomic) atomicAdd(p, v);
  else *p += v;
}

// N values into the CSR (no address: none).  They are distinct entries and no other
// element of the launch touches them (atomic: they may), so every old value is loaded
// before the first sum is stored: one round trip instead of N (a 23 x 19 x 21
// triquadratic mesh, eight colour launches: 219 -> 180 us).
template <typename T, int N>
__device__ __forceinline__ void add_values(T* const (&at)[N], const T (&v)[N], bool atomic) {
  if (atomic) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (at[k]) atomicAdd(at[k], v[k]);
    return;
  }
  T old[N];
#pragma unroll
  for (int k = 0; k < N; ++k) old[k] = at[k] ? *at[k] : (T)0;
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (at[k]) *at[k] = old[k] + v[k];
}

// As above for entries p of one CSR (p < 0: none), an index instead of an address each (with
// addresses the triquadratic scatter of 1,000 elements took 113 us instead of 108).
template <typename T, int N>
__device__ __forceinline__ void add_values(T* __restrict__ vals, const int (&p)[N], const T (&v)[N], bool atomic) {
  if (atomic) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (p[k] >= 0) atomicAdd(&vals[p[k]], v[k]);
    return;
  }
  T old[N];
#pragma unroll
  for (int k = 0; k < N; ++k) old[k] = p[k] >= 0 ? vals[p[k]] : (T)0;
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (p[k] >= 0) vals[p[k]] = old[k] + v[k];
}

// Stage layout of a structured (grid) assembly.  With row m = (c, a), column
// n = (c2, b), node a = (ax, ay, az) on the element's NB^3 lattice and element
// e = ex + nx (ey + ny ez), entry (m, n) of element e sits at
//   [ez][ey][c][az][ay][c2][bz][by][ex][ax][bx],
// i.e. stripe U = (ez ny + ey) SU + u(c, az, ay, c2, bz, by), SU = NC^2 NB^4 stripes
// per element row, each stripe nx NB^2 values long.  The entries that one x-line
// of CSR rows needs for one y/z neighbour block are then one contiguous stripe.
// The element kernels write the layout block-wise: each wavefront puts its
// element's entries into LDS as [u][wave][NB^2], and after a block barrier the
// block stores stripe by stripe, so the entries of the block's consecutive
// elements along x go out as one contiguous run per stripe.  Blocks are dealt to
// the eight XCDs in contiguous ranges (block b runs on XCD b % 8), so blocks that
// share a cache line share an L2.
template <int NN, int NC>
struct GridStripe {
  static constexpr int NB = NN == 8 ? 2 : 3, B2 = NB * NB, SU = NC * NC * B2 * B2;
  // LDS slot of entry (m, n) of wavefront w's element
  static __device__ __forceinline__ int slot(int m, int n, int w, int wpb) {
    const int c = m / NN, a = m - c * NN, c2 = n / NN, b = n - c2 * NN;
    const int u = ((((c * NB + a / B2) * NB + (a / NB) % NB) * NC + c2) * NB + b / B2) * NB + (b / NB) % NB;
    return (u * wpb + w) * B2 + (a % NB) * NB + b % NB;
  }
  // stage offset of element e's stripe-0 run
  static __device__ __forceinline__ long long base(long long e, int nx, int ny) {
    const long long ex = e % nx, eyz = e / nx;
    return (eyz * SU * nx + ex) * B2;
  }
  // logical block: contiguous ranges per XCD in a grid stage (gridDim.x a multiple of 8)
  static __device__ __forceinline__ int block(int nx) {
    if (nx <= 0) return blockIdx.x;
    return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  }
  // block-wide store of the LDS slots K of WPB elements (sbase[w] < 0: element slot w
  // is empty)
  template <typename T, int WPB>
  static __device__ __forceinline__ void store(const T* K, const long long* sbase, int nx, T* stage) {
    const long long stride = (long long)nx * B2;
    for (int f = threadIdx.x; f < SU * WPB * B2; f += blockDim.x) {
      const int u = f / (WPB * B2), r = f - u * (WPB * B2), w = r / B2, j = r - w * B2;
      const long long b = sbase[w];
      if (b >= 0) stage[b + u * stride + j] = K[f];
    }
  }
};

// Per-Gauss-point geometry of one element held in LDS by its wavefront.
template <int DIM, int NN, int NG>
struct GeomLDS {
  double x[NN * DIM];
  double ji[NG][DIM][DIM];  // dxi_j/dx_i stored as ji[g][j][i]
  double rwg[NG];           // |J| * w_g
};

template <int DIM, int NN, int NG>
__device__ __forceinline__ void element_geometry(GeomLDS<DIM, NN, NG>& G, const double* __restrict__ coords,
                                                 const int32_t* __restrict__ enodes, long long e,
                                                 const double* __restrict__ dN, const double* __restrict__ w,
                                                 int lane, bool active) {
  if (active && lane < NN) {
    const long long node = enodes[e * NN + lane];
#pragma unroll
    for (int d = 0; d < DIM; ++d) G.x[lane * DIM + d] = coords[node * DIM + d];
  }
  __syncthreads();
  // dx/dxi at Gauss point g = lane % 32: the node sum split between the two
  // half-waves (nodes below and from NN / 2), the halves added across lanes
  // l and l + 32 (NG <= 32), else one lane per Gauss point
  constexpr bool SPLIT = NG <= 32;
  const int g = SPLIT ? (lane & 31) : lane;
  double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  if (active && g < NG) {
    const int a0 = SPLIT && lane >= 32 ? NN / 2 : 0, a1 = SPLIT && lane < 32 ? NN / 2 : NN;
    for (int a = a0; a < a1; ++a) {
#pragma unroll
      for (int j = 0; j < DIM; ++j) {
        const double dn = dN[(g * NN + a) * DIM + j];
#pragma unroll
        for (int d = 0; d < DIM; ++d) J[d][j] += G.x[a * DIM + d] * dn;
      }
    }
  }
  if constexpr (SPLIT) {
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
      for (int j = 0; j < DIM; ++j) J[d][j] += __shfl_xor(J[d][j], 32);
  }
  if (active && lane < NG) {
    double Ji[3][3];
    const double det = invert<DIM>(J, Ji);
#pragma unroll
    for (int j = 0; j < DIM; ++j)
#pragma unroll
      for (int i = 0; i < DIM; ++i) G.ji[g][j][i] = Ji[j][i];
    G.rwg[g] = fabs(det) * w[g];
  }
  __syncthreads();
}

// ------------------------------------------------------------ scalar field
// Inputs of one scalar assembly (one mesh, one set of CSR values).
template <typename T>
struct ScalarJob {
  const double* coords;
  const int32_t* enodes;
  const int32_t* edofs;
  const double* kappa;
  const double* source;
  const int32_t* pos;   // NULL: structured (the element matrices go to the stage at vals)
  T* vals;
  double* svec;
};

// Where a structured assembly's element source vectors go ([e][NN], or NULL), and its
// elements in x and y (GridStripe layout).
struct ScalarStage {
  double* source = nullptr;
  int gnx = 0, gny = 0;
};

// One element per wavefront (element e when `active`); every wavefront of the
// block calls it the same number of times (it holds block barriers).
template <int DIM, int NN, int NG, typename T, int WPB>
__device__ __forceinline__ void scalar_element(const ScalarJob<T>& J, long long e, bool active,
                                               const double* __restrict__ dN, const double* __restrict__ N,
                                               const double* __restrict__ w, bool atomic) {
  constexpr int KD = NG * DIM;
  __shared__ GeomLDS<DIM, NN, NG> geo[WPB];
  __shared__ T sB[WPB][KD * NN];
  __shared__ T sW[WPB][KD];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  GeomLDS<DIM, NN, NG>& G = geo[wv];
  element_geometry<DIM, NN, NG>(G, J.coords, J.enodes, e, dN, w, lane, active);
  const double ke = (active && J.kappa) ? J.kappa[e] : 1.0;
  if (active) {
    for (int t = lane; t < NG * NN; t += 64) {
      const int g = t / NN, a = t - (t / NN) * NN;
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        double b = 0.0;
#pragma unroll
        for (int j = 0; j < DIM; ++j) b += dN[(g * NN + a) * DIM + j] * G.ji[g][j][i];
        sB[wv][(g * DIM + i) * NN + a] = (T)b;
      }
    }
    for (int k = lane; k < KD; k += 64) sW[wv][k] = (T)(G.rwg[k / DIM] * ke);
  }
  __syncthreads();
  if (active) {
    const T* B = sB[wv];
    const T* W = sW[wv];
    for (int t = lane; t < NN * NN; t += 64) {
      const int m = t / NN, n = t - (t / NN) * NN;
      T acc = 0;
#pragma unroll 9
      for (int k = 0; k < KD; ++k) acc += W[k] * B[k * NN + m] * B[k * NN + n];
      add_value(&J.vals[J.pos[e * (NN * NN) + t]], acc, atomic);
    }
    if (J.source && J.svec && lane < NN) {
      // Rounded product and sum, unfused whatever the caller inlines around them
      // (a kernel whose `atomic` is a constant would otherwise fuse them).
#pragma clang fp contract(off)
      double s = 0.0;
      for (int g = 0; g < NG; ++g) s = fma(N[g * NN + lane], G.rwg[g], s);
      s = s * J.source[e];
      add_value(&J.svec[J.edofs[e * NN + lane]], s, atomic);
    }
  }
}

template <int DIM, int NN, int NG, typename T, int WPB>
__global__ __launch_bounds__(64 * WPB) void scalar_assemble_kernel(
    const double* __restrict__ coords, const int32_t* __restrict__ enodes, const int32_t* __restrict__ edofs,
    const double* __restrict__ kappa, const double* __restrict__ source, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ order, int elem_begin, int elem_count, const double* __restrict__ dN,
    const double* __restrict__ N, const double* __restrict__ w, T* __restrict__ vals, double* __restrict__ svec,
    bool atomic) {
  const int idx = (int)blockIdx.x * WPB + (threadIdx.x >> 6);
  const bool active = idx < elem_count;
  long long e = 0;
  if (active) e = order ? order[elem_begin + idx] : (long long)elem_begin + idx;
  scalar_element<DIM, NN, NG, T, WPB>(
      ScalarJob<T>{coords, enodes, edofs, kappa, source, pos, vals, svec}, e, active, dN, N, w, atomic);
}

// ------------------------------------------------ trilinear elements, eight per wavefront
// A wavefront integrates eight elements: lane = (element, Gauss point) forms dx/dxi,
// its inverse and the point's physical gradients in registers, and the eight points'
// contributions to an entry meet by DPP inside the element's eight lanes.  With one
// element per wavefront only 16 of 64 lanes formed geometry, and the sums read 72 LDS
// values per entry.  In launches of few elements G = 8 such groups of lanes share an
// element, a row of its matrix each.  All forms (structured, coloured, batched; whatever
// G) run this code, with every multiply-add written out, so their sums agree bit for bit.
// E elements to a block of 8 E G threads.
template <int E>
struct Q1Tables {
  double dN[8 * 8 * 3];
  double X[E][8][3];
};

// Geometry of lane's (element, Gauss point q): ji[j][i] = dxi_j/dx_i, and |J| w_q.
// Holds two block barriers.
template <int E, int G = 1>
__device__ __forceinline__ double q1_geometry(Q1Tables<E>& S, const double* __restrict__ coords,
                                              const int32_t* __restrict__ enodes, long long e, bool active,
                                              const double* __restrict__ dN, const double* __restrict__ w,
                                              double (&ji)[3][3]) {
  const int el = threadIdx.x / (8 * G), q = threadIdx.x & 7;
  __syncthreads();  // the tables of an earlier pass are done with
  for (int t = threadIdx.x; t < 8 * 8 * 3; t += 8 * E * G) S.dN[t] = dN[t];
  if (active && (threadIdx.x >> 3) % G == 0) {
    const long long node = enodes[e * 8 + q];
#pragma unroll
    for (int d = 0; d < 3; ++d) S.X[el][q][d] = coords[node * 3 + d];
  }
  __syncthreads();
  double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double dn = S.dN[(q * 8 + a) * 3 + j];
#pragma unroll
      for (int d = 0; d < 3; ++d) J[d][j] = fma(S.X[el][a][d], dn, J[d][j]);
    }
  const double det = invert<3>(J, ji);
  return fabs(det) * w[q];
}

// One scalar element per 8 G lanes (e and J are those lanes' own); every thread of the
// block calls it.
template <typename T, bool GRID, int E, int G>
__device__ __forceinline__ void q1_scalar_elements(const ScalarJob<T>& J, const ScalarStage& Q, long long e, bool active,
                                                   const double* __restrict__ dN, const double* __restrict__ N,
                                                   const double* __restrict__ w, bool atomic) {
#pragma clang fp contract(off)
  using GS = GridStripe<8, 1>;
  __shared__ Q1Tables<E> S;
  __shared__ double rw[E][8];
  __shared__ T sK[E * 64];
  __shared__ long long sbase[E];
  const int el = threadIdx.x / (8 * G), q = threadIdx.x & 7, g = (threadIdx.x >> 3) % G;
  double ji[3][3];
  const double rwg = q1_geometry<E, G>(S, J.coords, J.enodes, e, active, dN, w, ji);
  const double ke = (active && J.kappa) ? J.kappa[e] : 1.0;
  const T W = (T)(rwg * ke);
  auto gradient = [&](int a, T (&b)[3]) {
    const double* d = &S.dN[(q * 8 + a) * 3];
#pragma unroll
    for (int i = 0; i < 3; ++i) b[i] = (T)fma(d[0], ji[0][i], fma(d[1], ji[1][i], d[2] * ji[2][i]));
  };
  T B[8][3];
#pragma unroll
  for (int a = 0; a < 8; ++a) gradient(a, B[a]);
  rw[el][q] = rwg;
  auto entry = [&](int m, int n, const T (&bm)[3], bool mine) {  // and its transpose
    const T v = sum8(fma(W * bm[0], B[n][0], fma(W * bm[1], B[n][1], W * bm[2] * B[n][2])));
    if (mine) {
      sK[GRID ? GS::slot(m, n, el, E) : el * 64 + m * 8 + n] = v;
      sK[GRID ? GS::slot(n, m, el, E) : el * 64 + n * 8 + m] = v;
    }
  };
  if constexpr (G == 8) {  // row g of the upper triangle
    T bg[3];
    gradient(g, bg);
#pragma unroll
    for (int n = 0; n < 8; ++n) entry(g, n, bg, n >= g && q == n);
  } else {  // all of it, entry t in lane t % 8
    int t = 0;
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int n = m; n < 8; ++n, ++t) entry(m, n, B[m], q == (t & 7));
  }
  if (GRID && q == 0 && g == 0) sbase[el] = active ? GS::base(e, Q.gnx, Q.gny) : -1;
  __syncthreads();
  if constexpr (GRID) {
    GS::template store<T, E>(sK, sbase, Q.gnx, J.vals);
  } else {
    // the wavefront's elements one by one, a lane per entry: the lanes of a store lie in
    // eight rows (a row per lane instead, in eight elements at once, touched 64 lines:
    // 61 x 47 x 53 elements, atomic, 283 us FP64 and 306 us FP32; 159 and 122 us so)
    constexpr int N = 8 / G;
    const int lane = threadIdx.x & 63, el0 = (threadIdx.x >> 6) * N;
    T* at[N];
    T v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      at[i] = nullptr;
      if (__builtin_amdgcn_readlane((int)active, 8 * i)) {
        at[i] = lane_value(J.vals, 8 * i) + lane_value(J.pos, 8 * i)[lane_value(e, 8 * i) * 64 + lane];
        v[i] = sK[(el0 + i) * 64 + lane];
      }
    }
    add_values(at, v, atomic);
  }
  if (active && g == 0 && J.source && (J.svec || Q.source)) {
    double s = 0.0;
#pragma unroll
    for (int p = 0; p < 8; ++p) s = fma(N[p * 8 + q], rw[el][p], s);
    s = s * J.source[e];
    if (Q.source)
      Q.source[e * 8 + q] = s;
    else
      add_value(&J.svec[J.edofs[e * 8 + q]], s, atomic);
  }
}

// Measured on 61 x 47 x 53 elements with moved nodes, FP64, structured: 187 us with
// one element per wavefront, 55 us now (78 MB of element matrices stored).
template <typename T, bool GRID, int E, int G>
__global__ __launch_bounds__(8 * E * G) void q1_scalar_kernel(ScalarJob<T> J, ScalarStage Q, const int32_t* __restrict__ order,
                                                        int elem_begin, int elem_count,
                                                        const double* __restrict__ dN, const double* __restrict__ N,
                                                        const double* __restrict__ w, bool atomic) {
  const int blk = GRID ? GridStripe<8, 1>::block(Q.gnx) : (int)blockIdx.x;
  const int idx = blk * E + (threadIdx.x / (8 * G));
  const bool active = idx < elem_count;
  long long e = 0;
  if (active) e = order ? order[elem_begin + idx] : (long long)elem_begin + idx;
  q1_scalar_elements<T, GRID, E, G>(J, Q, e, active, dN, N, w, atomic);
}

// ------------------------------------------------ triquadratic, on MFMA
// K = B^T diag(W) B with B[(g,i)][a] = dphi_a/dx_i at Gauss point g (81 x 27,
// padded to 84 x 32) runs as 16x16x4 MFMA tiles: tile (ti, tj) of K takes 21
// steps over the padded (g,i) axis, A operand = B^T rows, B operand = W B.  K is
// symmetric, so tiles (0,0), (0,1), (1,1) are formed and (1,0) is written as
// the transpose of (0,1).  At step t lane l forms the two gradients
// B[4t + l/16][16c + l%16], c = 0, 1, from the reference gradients (LDS) and
// dxi/dx: each is its A-operand entry and, times W, its B-operand entry.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of accumulator register i of lane l (column l % 16)
  static __device__ __forceinline__ int row(int lane, int i) { return 4 * i + (lane >> 4); }
};
template <>
struct Mfma16<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int i) { return 4 * (lane >> 4) + i; }
};

// GRID: the element matrices go to the stage (four wavefronts per SIMD hide the
// operand formation); else they are added into the CSR values, 16 entries per lane at
// once, which takes the registers of two.
constexpr int kQ2Waves = 4;

template <typename T, bool GRID>
__global__ __launch_bounds__(64 * kQ2Waves) __attribute__((amdgpu_waves_per_eu(GRID ? 4 : 2))) void q2_assemble_mfma_kernel(
    const double* __restrict__ coords, const int32_t* __restrict__ enodes, const int32_t* __restrict__ edofs,
    const double* __restrict__ kappa, const double* __restrict__ source, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ order, int elem_begin, int elem_count, const double* __restrict__ dN,
    const double* __restrict__ N, const double* __restrict__ w, T* __restrict__ vals, double* __restrict__ svec,
    bool atomic, double* __restrict__ sstage, int gnx, int gny) {
  constexpr int NN = 27, NG = 27, KD = 81, STEPS = 21, WPB = kQ2Waves;
  using M = Mfma16<T>;
  using GS = GridStripe<NN, 1>;
  // the element matrices of a grid stage reuse the LDS of the reference
  // gradients and geometry once every wavefront is past its products
  struct Tables {
    double dN[NG * NN * 3];
    GeomLDS<3, NN, NG> geo[WPB];
  };
  union Shared {
    Tables t;
    T K[WPB * NN * NN];
  };
  static_assert(sizeof(T) * WPB * NN * NN <= sizeof(Tables), "element matrices exceed the tables' LDS");
  __shared__ Shared sh;
  __shared__ long long sbase[WPB];
  double* sdN = sh.t.dN;
  for (int t = threadIdx.x; t < NG * NN * 3; t += blockDim.x) sdN[t] = dN[t];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int idx = GS::block(gnx) * WPB + wv;
  const bool active = idx < elem_count;
  long long e = 0;
  if (active) e = order ? order[elem_begin + idx] : (long long)elem_begin + idx;
  GeomLDS<3, NN, NG>& G = sh.t.geo[wv];
  element_geometry<3, NN, NG>(G, coords, enodes, e, sdN, w, lane, active);
  if (!GRID && !active) return;  // the scatter holds no further barrier
  const int kq = lane >> 4, col = lane & 15;
  typename M::v4 k00 = {0, 0, 0, 0}, k01 = {0, 0, 0, 0}, k11 = {0, 0, 0, 0};
  double s = 0.0;
  if (active) {
    const double ke = kappa ? kappa[e] : 1.0;
    // lane's two operand positions: a = col and a = 16 + col (the latter is padding for col >= 11)
    auto grad = [&](int k, int a) -> T {
      if (k >= KD || a >= NN) return (T)0;
      const int g = k / 3, i = k - 3 * (k / 3);
      const double* d = &sdN[(g * NN + a) * 3];
      return (T)(d[0] * G.ji[g][0][i] + d[1] * G.ji[g][1][i] + d[2] * G.ji[g][2][i]);
    };
#pragma unroll 3
    for (int t = 0; t < STEPS; ++t) {
      const int k = 4 * t + kq;
      const T wk = k < KD ? (T)(G.rwg[k / 3] * ke) : (T)0;
      const T a0 = grad(k, col), a1 = grad(k, 16 + col);
      k00 = M::mac(a0, a0 * wk, k00);
      k01 = M::mac(a0, a1 * wk, k01);
      k11 = M::mac(a1, a1 * wk, k11);
    }
    if (source && (svec || sstage) && lane < NN) {
      for (int g = 0; g < NG; ++g) s += N[g * NN + lane] * G.rwg[g];
      s *= source[e];
    }
  }
  if constexpr (!GRID) {
    const int32_t* pe = pos + e * (NN * NN);
    const bool second = 16 + col < NN;
    int p[16];
    T v[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = M::row(lane, i);
      // tile (0,0): m = r, n = col; tile (0,1) and its transpose: n = 16 + col;
      // tile (1,1): m = 16 + r, n = 16 + col
      p[4 * i] = pe[r * NN + col];
      p[4 * i + 1] = second ? pe[r * NN + 16 + col] : -1;
      p[4 * i + 2] = second ? pe[(16 + col) * NN + r] : -1;
      p[4 * i + 3] = second && 16 + r < NN ? pe[(16 + r) * NN + 16 + col] : -1;
      v[4 * i] = k00[i];
      v[4 * i + 1] = v[4 * i + 2] = k01[i];
      v[4 * i + 3] = k11[i];
    }
    add_values(vals, p, v, atomic);
    if (source && svec && lane < NN) add_value(&svec[edofs[e * NN + lane]], s, atomic);
    return;
  }
  // grid stage: the element source vector in element order, the matrix in stripes
  if (active && source && sstage && lane < NN) sstage[e * NN + lane] = s;
  __syncthreads();  // every wavefront is done with the tables
  if (active) {
    T* K = sh.K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = M::row(lane, i);
      K[GS::slot(r, col, wv, WPB)] = k00[i];
      if (16 + col < NN) {
        K[GS::slot(r, 16 + col, wv, WPB)] = k01[i];
        K[GS::slot(16 + col, r, wv, WPB)] = k01[i];
      }
      if (16 + r < NN && 16 + col < NN) K[GS::slot(16 + r, 16 + col, wv, WPB)] = k11[i];
    }
  }
  if (lane == 0) sbase[wv] = active ? GS::base(e, gnx, gny) : -1;
  __syncthreads();
  GS::template store<T, WPB>(sh.K, sbase, gnx, vals);
}

// ------------------------------------------------------- linear elasticity
// Trilinear elasticity.  The coefficients are constant over an element, so its 24 x 24
// matrix is a combination of the nine products S_kl[n][m] = sum_g w_g B[g][n][k]
// B[g][m][l]: diagonal block (c,c) is sum_k diagC[c][k] S_kk, and block (i,j) with
// the pair's (Ca, Cb) is Ca S_ij + Cb S_ji for i < j (linear_elasticity_routines.F90:
// 1255-1286; the lower blocks are the transposes).  A wavefront forms the gradients of
// eight elements, lane = (element, Gauss point), and then takes the elements in turn,
// lane = node pair (n, m): nine sums in registers, 72 multiply-adds, from which the
// lane's nine entries follow.  As one GEMM on MFMA with the coefficients inside the
// operands the same matrix took 30 tile steps and as many LDS-formed operands.
template <typename T>
struct ElasticJob {
  const double* coords;
  const int32_t* enodes;
  const double* material;
  const int32_t* pos;
  T* vals;
  int gnx, gny;  // GRID: elements in x and y (GridStripe layout)
};

// Element 4 i + w of a block belongs to wavefront w (lanes 8 i .. 8 i + 7, i < turns, hold its
// number and arrays): in turn i the four wavefronts take consecutive elements, whose
// entries leave through LDS in runs of 16 values.  Half of the gradients are in LDS
// at a time, which keeps two blocks on a CU.
constexpr int kElasticElems = 32;  // at most, in a block of 256 threads (4 per turn)
__device__ __forceinline__ int q1_elastic_slot() { return 4 * ((threadIdx.x & 63) >> 3) + (threadIdx.x >> 6); }

template <typename T, bool GRID>
__device__ __forceinline__ void q1_elastic_elements(const ElasticJob<T>& J, long long e, bool active, int turns,
                                                    const double* __restrict__ dN, const double* __restrict__ w,
                                                    bool atomic) {
#pragma clang fp contract(off)
  using GS = GridStripe<8, 3>;
  constexpr int kWaves = kElasticElems / 8, kHalf = 4, kRun = kWaves * GS::B2;
  __shared__ Q1Tables<kElasticElems> S;
  __shared__ T sB[kWaves][kHalf][8][8][3];
  __shared__ T sW[kWaves][8][8];
  __shared__ T sC[kWaves][8][15];  // diagC[3][3], then (Ca, Cb) of the pairs (0,1), (0,2), (1,2)
  __shared__ T sK[GRID ? 2 : 1][GRID ? GS::SU * kRun : 1];
  __shared__ long long sbase[kWaves][8];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i8 = lane >> 3, q = lane & 7;
  double ji[3][3];
  const double rwg = q1_geometry(S, J.coords, J.enodes, e, active, dN, w, ji);
  T B[8][3];
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const double* d = &S.dN[(q * 8 + a) * 3];
    // dphidx(a,mi) = sum_ni DXI_DX(mi,ni) dphi/dxi_ni   (linear_elasticity_routines.F90:1245-1252)
#pragma unroll
    for (int mi = 0; mi < 3; ++mi) B[a][mi] = (T)fma(ji[mi][0], d[0], fma(ji[mi][1], d[1], ji[mi][2] * d[2]));
  }
  sW[wv][i8][q] = (T)rwg;
  if (q == 0) sbase[wv][i8] = GRID && active ? GS::base(e, J.gnx, J.gny) : -1;
  if (q == 0 && active) {
    const double* mat = J.material + e * 6;
    const double E1 = mat[0], E2 = mat[1], E3 = mat[2], v13 = mat[3], v23 = mat[4], v12 = mat[5];
    const double v31 = v13, v32 = v23, v21 = v12;
    const double gama = 1.0 / (1.0 - v12 * v21 - v23 * v32 - v31 * v13 - 2.0 * v21 * v32 * v13);
    const double C11 = E1 * (1.0 - v23 * v32) * gama, C22 = E2 * (1.0 - v13 * v31) * gama;
    const double C33 = E3 * (1.0 - v12 * v21) * gama;
    const double C12 = E1 * (v21 + v31 * v23) * gama, C13 = E1 * (v31 + v21 * v32) * gama;
    const double C23 = E2 * (v32 + v12 * v31) * gama;
    const double C44 = E2 / (2.0 * (1.0 + v23)), C55 = E1 / (2.0 * (1.0 + v13)), C66 = E3 / (2.0 * (1.0 + v12));
    const double coef[15] = {C11, C66, C44, C66, C22, C55, C44, C55, C33, C12, C66, C13, C44, C23, C55};
#pragma unroll
    for (int k = 0; k < 15; ++k) sC[wv][i8][k] = (T)coef[k];
  }
  const int n = lane >> 3, m = lane & 7;
  const long long stride = (long long)J.gnx * GS::B2;  // GRID
  for (int half = 0; kHalf * half < turns; ++half) {
    __syncthreads();
    if ((i8 >> 2) == half) {
#pragma unroll
      for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int k = 0; k < 3; ++k) sB[wv][i8 & 3][q][a][k] = B[a][k];
    }
    __syncthreads();
    for (int h = 0; h < kHalf && kHalf * half + h < turns; ++h) {
      const int it = kHalf * half + h;
      const bool on = __builtin_amdgcn_readlane((int)active, 8 * it) != 0;
      T P[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const T wg = sW[wv][it][g];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const T bn = wg * sB[wv][h][g][n][k];
#pragma unroll
          for (int l = 0; l < 3; ++l) P[k][l] = fma(bn, sB[wv][h][g][m][l], P[k][l]);
        }
      }
      const T* C = sC[wv][it];
      T K[3][3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        K[c][c] = fma(C[3 * c], P[0][0], fma(C[3 * c + 1], P[1][1], C[3 * c + 2] * P[2][2]));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = i + 1; j < 3; ++j) {
          const T Ca = C[9 + 2 * (i + j - 1)], Cb = C[10 + 2 * (i + j - 1)];
          K[i][j] = fma(Ca, P[i][j], Cb * P[j][i]);
          K[j][i] = fma(Ca, P[j][i], Cb * P[i][j]);
        }
      if constexpr (GRID) {
        T* Ks = sK[it & 1];
        const int at = ((n >> 1) * 12 + (m >> 1)) * kRun + wv * GS::B2 + (n & 1) * 2 + (m & 1);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int c2 = 0; c2 < 3; ++c2) Ks[at + (48 * c + 4 * c2) * kRun] = K[c][c2];
        __syncthreads();  // the other buffer is written next: its stores are done by the barrier after
        const int r = threadIdx.x % kRun, u0 = threadIdx.x / kRun;
        const long long b = sbase[r / GS::B2][it];
        if (b >= 0) {
          T* out = J.vals + b + u0 * stride + r % GS::B2;
#pragma unroll
          for (int k = 0; k < GS::SU * kRun / 256; ++k) out[(256 / kRun) * k * stride] = Ks[threadIdx.x + 256 * k];
        }
      } else if (on) {
        const long long ee = lane_value(e, 8 * it);
        const int32_t* pe = lane_value(J.pos, 8 * it) + ee * 576 + n * 24 + m;
        T* vals = lane_value(J.vals, 8 * it);
        int p[9];
        T v[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          p[k] = pe[(k / 3) * 192 + (k % 3) * 8];
          v[k] = K[k / 3][k % 3];
        }
        add_values(vals, p, v, atomic);
      }
    }
  }
}

// GRID: a structured assembly's stage (elements in order, gnx x gny per z-layer).
// Measured on 63 x 41 x 38 elements with moved nodes, FP64, structured: 337 us as one
// MFMA GEMM per element, 148 us now (452 MB of element matrices stored); 190 us with the
// entries stored straight from registers in runs of four values.
template <typename T, bool GRID>
__global__ __launch_bounds__(256) void q1_elastic_kernel(ElasticJob<T> J, const int32_t* __restrict__ order,
                                                         int elem_begin, int elem_count, int turns,
                                                         const double* __restrict__ dN, const double* __restrict__ w,
                                                         bool atomic) {
  const int blk = GRID ? GridStripe<8, 3>::block(J.gnx) : (int)blockIdx.x;
  const int slot = q1_elastic_slot(), idx = blk * 4 * turns + slot;
  const bool active = slot < 4 * turns && idx < elem_count;
  long long e = 0;
  if (active) e = order ? order[elem_begin + idx] : (long long)elem_begin + idx;
  q1_elastic_elements<T, GRID>(J, e, active, turns, dN, w, atomic);
}

// ------------------------------------------- many meshes in one launch
// A batch assembles the CSR values of many independent trilinear meshes (the
// requests a server admits together): one launch per colour and element kind
// covers every mesh of the batch.  A launch walks a list of segments -- the
// elements of one colour of one mesh -- as one flattened index space; each
// element's lanes find its segment by bisection and run the same element code as
// the one-mesh kernels, so a mesh's values are bit for bit those of its own
// assembly.  Blocks loop over the index space (a resident grid).
struct BatchJob {
  const double* coords;
  const int32_t* enodes;
  const int32_t* edofs;
  const double* coef;
  const double* source;
  const int32_t* pos;
  const int32_t* order;
  void* vals;
  double* svec;
};

struct BatchSeg {
  int32_t job;     // index into the job table
  int32_t begin;   // first position of the colour in the job's element order
  int32_t prefix;  // first flattened index of the segment
  int32_t pad;
};

constexpr int kBatchGrid = 2048;

__device__ __forceinline__ const BatchSeg& batch_seg(const BatchSeg* __restrict__ segs, int nseg, int idx) {
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (segs[mid].prefix <= idx)
      lo = mid;
    else
      hi = mid - 1;
  }
  return segs[lo];
}

template <typename T, int E, int G>
__global__ __launch_bounds__(8 * E * G) void scalar_batch_kernel(const BatchJob* __restrict__ jobs,
                                                           const BatchSeg* __restrict__ segs, int nseg, int total,
                                                           const double* __restrict__ dN,
                                                           const double* __restrict__ N,
                                                           const double* __restrict__ w) {
  for (int base = blockIdx.x * E; base < total; base += gridDim.x * E) {
    const int idx = base + threadIdx.x / (8 * G);
    const bool active = idx < total;
    ScalarJob<T> J{};
    long long e = 0;
    if (active) {
      const BatchSeg sg = batch_seg(segs, nseg, idx);
      const BatchJob B = jobs[sg.job];
      J = ScalarJob<T>{B.coords, B.enodes, B.edofs, B.coef, B.source, B.pos, (T*)B.vals, B.svec};
      e = B.order[sg.begin + idx - sg.prefix];
    }
    q1_scalar_elements<T, false, E, G>(J, ScalarStage{}, e, active, dN, N, w, false);
  }
}

template <typename T, int TURNS>
__global__ __launch_bounds__(256) void elastic_batch_kernel(const BatchJob* __restrict__ jobs,
                                                            const BatchSeg* __restrict__ segs, int nseg, int total,
                                                            const double* __restrict__ dN,
                                                            const double* __restrict__ w) {
  for (int base = blockIdx.x * 4 * TURNS; base < total; base += gridDim.x * 4 * TURNS) {
    const int slot = q1_elastic_slot(), idx = base + slot;
    const bool active = slot < 4 * TURNS && idx < total;
    ElasticJob<T> J{};
    long long e = 0;
    if (active) {
      const BatchSeg sg = batch_seg(segs, nseg, idx);
      const BatchJob B = jobs[sg.job];
      J = ElasticJob<T>{B.coords, B.enodes, B.coef, B.pos, (T*)B.vals, 0, 0};
      e = B.order[sg.begin + idx - sg.prefix];
    }
    q1_elastic_elements<T, false>(J, e, active, TURNS, dN, w, false);
  }
}

// Trilinear scalar elements per block (E) and groups of eight lanes per element (G) from
// the elements of a launch.  Few elements: a wavefront each, its eight groups taking a row
// of the matrix; such launches are as long as one wavefront, and eight launches make a
// coloured assembly (16^3 elements, 512 to a launch: 45 us, 65 with eight elements per
// wavefront, 52 with an element per wavefront and sums in LDS; 24^3, 1,728 to a launch: 60,
// 68, 62; 32^3: 88, 78, 82).  Then eight elements per wavefront, a wavefront per block;
// from 200,000 elements blocks of four (100^3 atomic: 995 us FP64, 773 FP32 one by one,
// 990 and 752 with four; 61 x 47 x 53 structured 74 and 76).
template <typename F>
static void q1_scalar_launch(long long count, F&& f) {
  using std::integral_constant;
  if (count < 2048) f(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  else if (count < 200000) f(integral_constant<int, 8>{}, integral_constant<int, 1>{});
  else f(integral_constant<int, 32>{}, integral_constant<int, 1>{});
}

// Elements that a wavefront of a trilinear elasticity launch takes, one after the other: as
// few as leave the chip full.  FP64, us with 1 / 2 / 4 / 8: staged 8^3 elements 20 / 21 / 23 /
// 28, 16^3 37 / 31 / 31 / 36, 24^3 75 / 58 / 53 / 50; coloured, an eighth of the elements to
// a launch, 16^3 67 / 86 / 123 / 199, 32^3 225 / 201 / 215 / 271, 45^3 630 / 553 / 570 / 545
// (at 8 all its blocks are resident), 61 x 47 x 53 1203 / 1055 / 1030 / 1114.  FP32 holds more
// wavefronts: 45^3 375 / 389 / 353 / 366, 61 x 47 x 53 609 / 600 / 641 / 574.  Atomic adds
// bound the atomic form: 1224 / 1236 / 1215 / 1261 there, FP32 951 / 954 / 957 / 962.
// Batches (many meshes, a colour of all to a launch; the number is a constant of their
// kernels, as a variable it cost 10%): 8 meshes of 8^3, 512 to a launch, 87 / 101 / 133 /
// 200, 16 of 12^3 (3,456) 232 / 188 / 206 / 261, 4 of 24^3 (6,912) 415 / 350 / 324 / 348,
// 2 of 60^3 (54,000) 3378 / 3334 / 3343 / 3352, FP32 2136 / 1905 / 1792 / 1850.
enum class Form { kStage, kColour, kAtomic, kBatch };
template <typename T>
static int elastic_turns(long long count, Form form) {
  if (form == Form::kAtomic) return sizeof(T) == 4 || count < 8192 ? 1 : 4;
  if (form == Form::kBatch)
    return count < 1024 ? 1 : count < 6144 ? 2 : sizeof(T) == 8 || count < 16384 ? 4 : 8;
  if (form == Form::kStage) return count < 1024 ? 1 : count < 4096 ? 2 : count < 8192 ? 4 : 8;
  if (sizeof(T) == 4) return count < 4096 ? 1 : count < 8192 ? 2 : count < 16384 ? 4 : 8;
  return count < 4096 ? 1 : count < 8192 ? 2 : count < 16384 ? 8 : 4;
}

template <int DIM, int NN, int NG, typename T>
static int launch_scalar(const mife_element_desc* d, int n_elem, const double* coords, const int32_t* enodes,
                         const int32_t* edofs, const double* kappa, const double* source, const int32_t* pos,
                         const int32_t* order, const int32_t* cptr, int ncol, T* vals, double* svec,
                         hipStream_t s) {
  constexpr int WPB = (sizeof(T) * NG * DIM * NN > 12000) ? 1 : 4;
  constexpr bool kMfma = DIM == 3 && NN == 27 && NG == 27;
  const int tk = prof::begin(s);
  auto launch = [&](const int32_t* ord, int begin, int count, bool atomic) {
    if constexpr (DIM == 3 && NN == 8 && NG == 8)
      q1_scalar_launch(count, [&](auto per, auto groups) {
        constexpr int E = decltype(per)::value, G = decltype(groups)::value;
        q1_scalar_kernel<T, false, E, G><<<div_up(count, E), 8 * E * G, 0, s>>>(
            ScalarJob<T>{coords, enodes, edofs, kappa, source, pos, vals, svec}, ScalarStage{}, ord, begin, count,
            d->dN, d->N, d->w, atomic);
      });
    else if constexpr (kMfma)
      q2_assemble_mfma_kernel<T, false><<<div_up(count, kQ2Waves), 64 * kQ2Waves, 0, s>>>(
          coords, enodes, edofs, kappa, source, pos, ord, begin, count, d->dN, d->N, d->w, vals, svec, atomic, nullptr,
          0, 0);
    else
      scalar_assemble_kernel<DIM, NN, NG, T, WPB><<<div_up(count, WPB), 64 * WPB, 0, s>>>(
          coords, enodes, edofs, kappa, source, pos, ord, begin, count, d->dN, d->N, d->w, vals, svec, atomic);
  };
  if (!order) {
    launch(nullptr, 0, n_elem, true);
  } else {
    for (int c = 0; c < ncol; ++c) {
      const int cnt = cptr[c + 1] - cptr[c];
      if (cnt > 0) launch(order, cptr[c], cnt, false);
    }
  }
  prof::end(tk, s, sizeof(T) == 8 ? prof::kAssembleScalar : prof::kAssembleScalar32);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

template <typename T>
static int launch_elastic(const mife_element_desc* d, int n_elem, const double* coords, const int32_t* enodes,
                          const double* material, const int32_t* pos, const int32_t* order, const int32_t* cptr,
                          int ncol, T* vals, hipStream_t s) {
  const int tk = prof::begin(s);
  auto launch = [&](const int32_t* ord, int begin, int count, bool atomic) {
    const int turns = elastic_turns<T>(count, atomic ? Form::kAtomic : Form::kColour);
    q1_elastic_kernel<T, false><<<div_up(count, 4 * turns), 256, 0, s>>>(
        ElasticJob<T>{coords, enodes, material, pos, vals, 0, 0}, ord, begin, count, turns, d->dN, d->w, atomic);
  };
  if (!order) {
    launch(nullptr, 0, n_elem, true);
  } else {
    for (int c = 0; c < ncol; ++c) {
      const int cnt = cptr[c + 1] - cptr[c];
      if (cnt > 0) launch(order, cptr[c], cnt, false);
    }
  }
  prof::end(tk, s, sizeof(T) == 8 ? prof::kAssembleElastic : prof::kAssembleElastic32);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

// --------------------------------------------- structured (grid) assembly
// On a generated regular mesh (elements and nodes numbered x fastest, as iron's
// generated mesh numbers them; one or three components in separated DOF order)
// every CSR row is the tensor product of 1-D neighbour ranges, so a row and the
// elements that touch it follow from the node's grid index.  The assembly then
// runs as two passes: the element kernels store every element matrix in the
// GridStripe layout (one launch, no colouring), and this kernel writes each CSR row whole --
// entry by entry the sum of the element entries that meet there, in the order of
// the element colours (parity of the element index per direction), which is the
// order in which the coloured scatter adds them, so the values are bit for bit
// those of the coloured scatter.  No position map is read and no value is read
// back.  The 1-D neighbour arithmetic is in mife_grid.hpp.
//
// One wavefront (one block) per (component c, x-line (iy, iz), run of R
// consecutive nodes ix, R = P (64 / (P^2 + 2P)) so that the run's pairs fit the
// 64 lanes).  Lane l takes one pair (ix, jx): CSR row (c, ix, iy, iz) and its
// x-neighbour offset qx.  The wavefront walks the y/z neighbour blocks
// (c2, qz, qy) of the x-line, which are the same for every lane, so the y/z
// index arithmetic is wave-uniform.  In the GridStripe layout the entries of
// block (c2, qz, qy) for the element slots (sy, sz) are stripe U, nx NB^2
// values, of which lane l reads X = ex NB^2 + ax NB + bx for its element slots
// sx.  Per (c2, qz) the lanes first issue the loads of all qy, then sum each
// entry's (up to eight) element values in colour order -- parity of the element
// index per direction, z slowest, the order of the coloured scatter -- and put
// the sums in LDS, where each row's (c2, qz) piece, cy cx entries, is
// contiguous as in the CSR row; the pieces are then stored row by row.  Units
// are dealt to the eight XCDs in contiguous ranges (block b runs on XCD b % 8),
// so the x-lines that share stripes share an L2.
// stage: element matrices in the GridStripe layout; sstage (NC == 1, may be
// NULL): element source vectors [E][NN].  Every row must hold the full grid
// stencil (the host checks the element DOFs); entries beyond a row's stored
// length are not written.
template <typename T, typename I, int P, int NC>
__global__ __launch_bounds__(64) void grid_gather_kernel(int nx, int ny, int nz, int runs, int n_units,
                                                         const int32_t* __restrict__ row_ptr,
                                                         const T* __restrict__ stage, T* __restrict__ vals,
                                                         const double* __restrict__ sstage,
                                                         double* __restrict__ svec) {
  constexpr int NB = P + 1, NN = NB * NB * NB, PER = P * P + 2 * P, R = P * (64 / PER), Q = 2 * P + 1;
  constexpr int SU = NC * NC * NB * NB * NB * NB;
  __shared__ T piece[Q * 64];
  const int Nx = P * nx + 1, Ny = P * ny + 1, Nz = P * nz + 1;
  const int unit = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (unit >= n_units) return;  // whole block: no barrier is reached
  const int lane = threadIdx.x;
  const int run = unit % runs, line = unit / runs;
  const int iy = line % Ny, iz = (line / Ny) % Nz, c = line / (Ny * Nz);
  const int r0 = run * R, r1 = min(r0 + R, Nx);
  const long long rowline = ((long long)c * Nz + iz) * ((long long)Ny * Nx) + (long long)iy * Nx;
  const int t0 = x_pair_start(r0, P, nx), npairs = x_pair_start(r1, P, nx) - t0;
  // wave-uniform y/z ranges
  int ly, hy, lz, hz;
  elem_range(iy, P, ny, ly, hy);
  elem_range(iz, P, nz, lz, hz);
  const int cy = P * (hy - ly) + P + 1, cz = P * (hz - lz) + P + 1;
  // lane's pair: row ix, neighbour jx, x element slots
  const bool act = lane < npairs;
  int ix = r0, jx = r0;
  if (act) x_pair(t0 + lane, P, ix, jx);
  int lx, hx, ljx, hjx;
  elem_range(ix, P, nx, lx, hx);
  elem_range(jx, P, nx, ljx, hjx);
  const int cx = P * (hx - lx) + P + 1, qx = jx - P * lx;
  const int ax = max(lx, ljx), bx = min(hx, hjx);
  int X[2];
  bool xv[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int ex = elem_of_parity(ax, bx, s);
    xv[s] = act && ex >= 0;
    X[s] = xv[s] ? (ex * NB + (ix - P * ex)) * NB + (jx - P * ex) : 0;
  }
  // LDS place of the lane's entry qy of a piece: rows' pieces back to back
  const int wslot = cy * (x_pair_start(ix, P, nx) - t0) + qx;
  // store plan: LDS slot k = lane + 64 i holds entry k of the pieces, i.e. of
  // row fix = row of pair t0 + k / cy, at (c2 cz + qz) cy cx(fix) + local
  int fpos[Q], fcx[Q], flen[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int k = lane + 64 * i;
    fpos[i] = -1;
    fcx[i] = 0;
    flen[i] = 0;
    if (k < cy * npairs) {
      int fix, fjx;
      x_pair(t0 + k / cy, P, fix, fjx);
      int flx, fhx;
      elem_range(fix, P, nx, flx, fhx);
      const int rp = row_ptr[rowline + fix];
      fpos[i] = rp + (k - cy * (x_pair_start(fix, P, nx) - t0));
      fcx[i] = P * (fhx - flx) + P + 1;
      flen[i] = row_ptr[rowline + fix + 1];
    }
  }
  const I stripe = (I)nx * (NB * NB);
  for (int c2 = 0; c2 < NC; ++c2) {
    for (int qz = 0; qz < cz; ++qz) {
      const int jz = P * lz + qz;
      int ljz, hjz;
      elem_range(jz, P, nz, ljz, hjz);
      const int az = max(lz, ljz), bz = min(hz, hjz);
      int ez[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) ez[s] = elem_of_parity(az, bz, s);
      // loads of every qy first (no use before all are issued)
      T v[Q][2][2][2];
      bool yv[Q][2];
#pragma unroll
      for (int qy = 0; qy < Q; ++qy) {
        const int jy = P * ly + qy;
        int ljy, hjy;
        elem_range(jy, P, ny, ljy, hjy);
        const int ay = max(ly, ljy), by = min(hy, hjy);
#pragma unroll
        for (int sy = 0; sy < 2; ++sy) {
          const int ey = qy < cy ? elem_of_parity(ay, by, sy) : -1;
          yv[qy][sy] = ey >= 0;
#pragma unroll
          for (int sz = 0; sz < 2; ++sz) {
            if (ey < 0 || ez[sz] < 0) continue;
            const I U = ((I)ez[sz] * ny + ey) * SU +
                        (((((c * NB + (iz - P * ez[sz])) * NB + (iy - P * ey)) * NC + c2) * NB + (jz - P * ez[sz])) *
                             NB +
                         (jy - P * ey));
            const T* st = stage + U * stripe;
#pragma unroll
            for (int sx = 0; sx < 2; ++sx)
              if (xv[sx]) v[qy][sz][sy][sx] = st[X[sx]];
          }
        }
      }
#pragma unroll
      for (int qy = 0; qy < Q; ++qy) {
        if (qy >= cy) continue;
        T sum = (T)0;
#pragma unroll
        for (int sz = 0; sz < 2; ++sz) {
          if (ez[sz] < 0) continue;
#pragma unroll
          for (int sy = 0; sy < 2; ++sy) {
            if (!yv[qy][sy]) continue;
#pragma unroll
            for (int sx = 0; sx < 2; ++sx)
              if (xv[sx]) sum += v[qy][sz][sy][sx];
          }
        }
        if (act) piece[wslot + qy * cx] = sum;
      }
      __syncthreads();
      const int blk = (c2 * cz + qz) * cy;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int at = fpos[i] + blk * fcx[i];
        if (fpos[i] >= 0 && at < flen[i]) vals[at] = piece[lane + 64 * i];
      }
      __syncthreads();
    }
  }
  if (NC == 1 && sstage && act && jx == ix) {
    double sv = 0.0;
#pragma unroll
    for (int col = 0; col < 8; ++col) {
      const int ex = elem_of_parity(lx, hx, col & 1), ey = elem_of_parity(ly, hy, (col >> 1) & 1),
                ez = elem_of_parity(lz, hz, col >> 2);
      if (ex < 0 || ey < 0 || ez < 0) continue;
      const long long e = ex + (long long)nx * (ey + (long long)ny * ez);
      const int a = (ix - P * ex) + NB * ((iy - P * ey) + NB * (iz - P * ez));
      sv += sstage[e * NN + a];
    }
    svec[rowline + ix] = sv;
  }
}

template <typename T>
static size_t grid_stage_bytes(long long E, int nn, int nc) {
  const size_t nd = (size_t)nc * nn;
  return ((size_t)E * nd * nd * sizeof(T) + 255) / 256 * 256 + (nc == 1 ? (size_t)E * nn * sizeof(double) : 0);
}

template <typename T, int P, int NC>
static int launch_grid(const mife_element_desc* d, const int* ne, const double* coords, const int32_t* enodes,
                       const double* coef, const double* source, const int32_t* row_ptr, long long n_rows, T* vals,
                       double* svec, void* stage, hipStream_t s) {
  constexpr int NB = P + 1, NN = NB * NB * NB, ND = NC * NN;
  const long long E = (long long)ne[0] * ne[1] * ne[2];
  T* kst = (T*)stage;
  double* sst = (NC == 1 && source && svec)
      ? (double*)((char*)stage + ((size_t)E * ND * ND * sizeof(T) + 255) / 256 * 256)
      : nullptr;
  const int tk = prof::begin(s);
  // multiples of the XCD count
  [[maybe_unused]] const int grid_e = div_up(div_up(E, kQ2Waves), 8) * 8;
  if constexpr (NC == 1) {
    if constexpr (NN == 27) {
      q2_assemble_mfma_kernel<T, true><<<grid_e, 64 * kQ2Waves, 0, s>>>(coords, enodes, nullptr, coef, source, nullptr,
                                                                        nullptr, 0, (int)E, d->dN, d->N, d->w, kst,
                                                                        nullptr, false, sst, ne[0], ne[1]);
    } else {
      q1_scalar_launch(E, [&](auto per, auto groups) {
        constexpr int PE = decltype(per)::value, G = decltype(groups)::value;
        q1_scalar_kernel<T, true, PE, G><<<div_up(div_up(E, PE), 8) * 8, 8 * PE * G, 0, s>>>(
            ScalarJob<T>{coords, enodes, nullptr, coef, source, nullptr, kst, nullptr},
            ScalarStage{sst, ne[0], ne[1]}, nullptr, 0,
            (int)E, d->dN, d->N, d->w, false);
      });
    }
  } else {
    const int turns = elastic_turns<T>(E, Form::kStage);
    q1_elastic_kernel<T, true><<<div_up(div_up(E, 4 * turns), 8) * 8, 256, 0, s>>>(
        ElasticJob<T>{coords, enodes, coef, nullptr, kst, ne[0], ne[1]}, nullptr, 0, (int)E, turns, d->dN, d->w,
        false);
  }
  constexpr int R = P * (64 / (P * P + 2 * P));
  const int runs = div_up(P * ne[0] + 1, R);
  const long long units = (long long)NC * (P * ne[1] + 1) * (P * ne[2] + 1) * runs;
  const int blocks = div_up(units, 8) * 8;  // a multiple of the XCD count
  if ((size_t)E * ND * ND < (size_t(1) << 31))
    grid_gather_kernel<T, int, P, NC><<<blocks, 64, 0, s>>>(ne[0], ne[1], ne[2], runs, (int)units, row_ptr, kst, vals,
                                                           sst, sst ? svec : nullptr);
  else
    grid_gather_kernel<T, long long, P, NC><<<blocks, 64, 0, s>>>(ne[0], ne[1], ne[2], runs, (int)units, row_ptr, kst,
                                                                 vals, sst, sst ? svec : nullptr);
  const int key = NC == 1 ? (sizeof(T) == 8 ? prof::kAssembleScalar : prof::kAssembleScalar32)
                          : (sizeof(T) == 8 ? prof::kAssembleElastic : prof::kAssembleElastic32);
  prof::end(tk, s, key);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}

}  // namespace mife

using namespace mife;

extern "C" size_t mife_assemble_grid_stage_bytes(int n_elem, int n_nodes, int n_comp, int prec) {
  if (n_elem <= 0 || n_nodes <= 0 || (n_comp != 1 && n_comp != 3)) return 0;
  return prec == MIFE_F32 ? grid_stage_bytes<float>(n_elem, n_nodes, n_comp)
                          : grid_stage_bytes<double>(n_elem, n_nodes, n_comp);
}

extern "C" int mife_assemble_grid(const mife_element_desc* d, const int32_t* n_elem, int n_comp,
                                  const double* coords, const int32_t* elem_nodes, const double* coef,
                                  const double* source, const int32_t* row_ptr, int64_t n_rows, int prec, void* vals,
                                  double* src_vec, void* stage, size_t stage_bytes, void* stream) {
  MIFE_REQUIRE(d && n_elem && coords && elem_nodes && row_ptr && vals && stage && d->dN && d->w,
               MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  MIFE_REQUIRE(d->dim == 3, MIFE_ERR_ARG, "the grid assembly is 3-D");
  MIFE_REQUIRE(prec == MIFE_F64 || prec == MIFE_F32, MIFE_ERR_ARG, "invalid precision %d", prec);
  MIFE_REQUIRE(n_comp == 1 || n_comp == 3, MIFE_ERR_ARG, "%d components (1: scalar field, 3: elasticity)", n_comp);
  MIFE_REQUIRE(n_comp == 1 || coef, MIFE_ERR_POINTER_IS_NULL, "elasticity without material");
  MIFE_REQUIRE(n_comp == 1 || !source, MIFE_ERR_ARG, "a source vector is a scalar-field term");
  MIFE_REQUIRE(!source || !src_vec || d->N, MIFE_ERR_POINTER_IS_NULL, "source given without basis values N");
  MIFE_REQUIRE(n_elem[0] > 0 && n_elem[1] > 0 && n_elem[2] > 0, MIFE_ERR_ARG, "empty grid");
  int P = 0;
  if (d->n_nodes == 8 && d->n_gauss == 8) P = 1;
  if (d->n_nodes == 27 && d->n_gauss == 27 && n_comp == 1) P = 2;
  MIFE_REQUIRE(P > 0, MIFE_ERR_ARG, "grid assembly element: %d nodes, %d Gauss points, %d components", d->n_nodes,
               d->n_gauss, n_comp);
  const long long E = (long long)n_elem[0] * n_elem[1] * n_elem[2];
  const long long Nn = (long long)(P * n_elem[0] + 1) * (P * n_elem[1] + 1) * (P * n_elem[2] + 1);
  MIFE_REQUIRE(E < (1LL << 31) && n_rows < (1LL << 31) && n_rows == n_comp * Nn, MIFE_ERR_ARG,
               "%lld rows given, the grid has %lld nodes x %d components", (long long)n_rows, Nn, n_comp);
  const size_t need = prec == MIFE_F32 ? grid_stage_bytes<float>(E, d->n_nodes, n_comp)
                                       : grid_stage_bytes<double>(E, d->n_nodes, n_comp);
  MIFE_REQUIRE(stage_bytes >= need, MIFE_ERR_ARG, "stage of %zu bytes, %zu needed (mife_assemble_grid_stage_bytes)",
               stage_bytes, need);
  hipStream_t s = (hipStream_t)stream;
  const int ne[3] = {n_elem[0], n_elem[1], n_elem[2]};
  if (n_comp == 3) {
    if (prec == MIFE_F64)
      return launch_grid<double, 1, 3>(d, ne, coords, elem_nodes, coef, nullptr, row_ptr, n_rows, (double*)vals,
                                       nullptr, stage, s);
    return launch_grid<float, 1, 3>(d, ne, coords, elem_nodes, coef, nullptr, row_ptr, n_rows, (float*)vals, nullptr,
                                    stage, s);
  }
  if (P == 2) {
    if (prec == MIFE_F64)
      return launch_grid<double, 2, 1>(d, ne, coords, elem_nodes, coef, source, row_ptr, n_rows, (double*)vals,
                                       src_vec, stage, s);
    return launch_grid<float, 2, 1>(d, ne, coords, elem_nodes, coef, source, row_ptr, n_rows, (float*)vals, src_vec,
                                    stage, s);
  }
  if (prec == MIFE_F64)
    return launch_grid<double, 1, 1>(d, ne, coords, elem_nodes, coef, source, row_ptr, n_rows, (double*)vals,
                                     src_vec, stage, s);
  return launch_grid<float, 1, 1>(d, ne, coords, elem_nodes, coef, source, row_ptr, n_rows, (float*)vals, src_vec,
                                  stage, s);
}

extern "C" int mife_assemble_scalar(const mife_element_desc* d, int n_elem, const double* coords,
                                    const int32_t* elem_nodes, const int32_t* elem_dofs, const double* kappa,
                                    const double* source, const int32_t* pos, const int32_t* order,
                                    const int32_t* colour_ptr_host, int n_colours, int prec, void* vals,
                                    double* src_vec, void* stream) {
  MIFE_REQUIRE(d && coords && elem_nodes && elem_dofs && pos && vals && d->dN && d->w, MIFE_ERR_POINTER_IS_NULL,
               "null pointer argument");
  MIFE_REQUIRE(!source || d->N, MIFE_ERR_POINTER_IS_NULL, "source given without basis values N");
  MIFE_REQUIRE(!order || colour_ptr_host, MIFE_ERR_POINTER_IS_NULL, "colour order without colour_ptr");
  MIFE_REQUIRE(prec == MIFE_F64 || prec == MIFE_F32, MIFE_ERR_ARG, "invalid precision %d", prec);
  if (n_elem == 0) return MIFE_OK;
  hipStream_t s = (hipStream_t)stream;
  const int key = d->dim * 10000 + d->n_nodes * 100 + d->n_gauss;
#define SCALAR_CASE(DIM, NN, NG)                                                                            \
  case DIM * 10000 + NN * 100 + NG:                                                                        \
    if (prec == MIFE_F64)                                                                                   \
      return launch_scalar<DIM, NN, NG, double>(d, n_elem, coords, elem_nodes, elem_dofs, kappa, source,   \
                                                pos, order, colour_ptr_host, n_colours, (double*)vals,     \
                                                src_vec, s);                                               \
    return launch_scalar<DIM, NN, NG, float>(d, n_elem, coords, elem_nodes, elem_dofs, kappa, source, pos, \
                                             order, colour_ptr_host, n_colours, (float*)vals, src_vec, s);
  switch (key) {
    SCALAR_CASE(2, 4, 4)
    SCALAR_CASE(2, 9, 9)
    SCALAR_CASE(3, 8, 8)
    SCALAR_CASE(3, 27, 27)
    SCALAR_CASE(3, 8, 27)
    default:
      set_error("unsupported scalar element (dim=%d, nodes=%d, gauss=%d)", d->dim, d->n_nodes, d->n_gauss);
      return MIFE_ERR_ARG;
  }
#undef SCALAR_CASE
}

extern "C" int mife_assemble_elastic(const mife_element_desc* d, int n_elem, const double* coords,
                                     const int32_t* elem_nodes, const int32_t* elem_dofs, const double* material,
                                     const int32_t* pos, const int32_t* order, const int32_t* colour_ptr_host,
                                     int n_colours, int prec, void* vals, void* stream) {
  (void)elem_dofs;
  MIFE_REQUIRE(d && coords && elem_nodes && material && pos && vals && d->dN && d->w, MIFE_ERR_POINTER_IS_NULL,
               "null pointer argument");
  MIFE_REQUIRE(!order || colour_ptr_host, MIFE_ERR_POINTER_IS_NULL, "colour order without colour_ptr");
  MIFE_REQUIRE(d->dim == 3, MIFE_ERR_ARG, "linear elasticity kernel is 3-D only");
  MIFE_REQUIRE(prec == MIFE_F64 || prec == MIFE_F32, MIFE_ERR_ARG, "invalid precision %d", prec);
  if (n_elem == 0) return MIFE_OK;
  hipStream_t s = (hipStream_t)stream;
  if (d->n_nodes == 8 && d->n_gauss == 8) {
    if (prec == MIFE_F64)
      return launch_elastic<double>(d, n_elem, coords, elem_nodes, material, pos, order, colour_ptr_host,
                                          n_colours, (double*)vals, s);
    return launch_elastic<float>(d, n_elem, coords, elem_nodes, material, pos, order, colour_ptr_host,
                                       n_colours, (float*)vals, s);
  }
  set_error("unsupported elastic element (nodes=%d, gauss=%d)", d->n_nodes, d->n_gauss);
  return MIFE_ERR_ARG;
}

namespace {

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

}  // namespace

extern "C" size_t mife_assemble_batch_work_bytes(int n_jobs, int max_colours) {
  const size_t nj = (size_t)std::max(n_jobs, 1);
  return align256(sizeof(BatchJob) * nj) + sizeof(BatchSeg) * nj * (size_t)std::max(max_colours, 1) + 256;
}

extern "C" int mife_assemble_batch(const mife_element_desc* scalar_desc, const mife_element_desc* elastic_desc,
                                   int n_jobs, const mife_assembly_job* jobs, int max_colours, int prec,
                                   void* table_host, void* work, void* stream) {
  MIFE_REQUIRE(n_jobs >= 0 && max_colours >= 0, MIFE_ERR_ARG, "invalid job count %d / colour bound %d", n_jobs,
               max_colours);
  if (n_jobs == 0) return MIFE_OK;
  MIFE_REQUIRE(jobs && table_host && work, MIFE_ERR_POINTER_IS_NULL, "null pointer argument");
  MIFE_REQUIRE(prec == MIFE_F64 || prec == MIFE_F32, MIFE_ERR_ARG, "invalid precision %d", prec);
  bool any_scalar = false, any_elastic = false, any_source = false;
  for (int k = 0; k < n_jobs; ++k) {
    const mife_assembly_job& J = jobs[k];
    MIFE_REQUIRE(J.kind == MIFE_JOB_SCALAR || J.kind == MIFE_JOB_ELASTIC, MIFE_ERR_ARG, "job %d: kind %d", k, J.kind);
    MIFE_REQUIRE(J.n_elem >= 0 && J.n_colours >= 0 && J.n_colours <= max_colours, MIFE_ERR_ARG,
                 "job %d: %d elements in %d colours (bound %d)", k, J.n_elem, J.n_colours, max_colours);
    if (J.n_elem == 0) continue;
    MIFE_REQUIRE(J.coords && J.elem_nodes && J.pos && J.order && J.colour_ptr_host && J.vals,
                 MIFE_ERR_POINTER_IS_NULL, "job %d: null pointer", k);
    MIFE_REQUIRE(J.colour_ptr_host[0] == 0 && J.colour_ptr_host[J.n_colours] == J.n_elem, MIFE_ERR_ARG,
                 "job %d: colour pointers do not cover its %d elements", k, J.n_elem);
    if (J.kind == MIFE_JOB_SCALAR) {
      any_scalar = true;
      if (J.source && J.src_vec) {
        MIFE_REQUIRE(J.elem_dofs, MIFE_ERR_POINTER_IS_NULL, "job %d: source without element DOFs", k);
        any_source = true;
      }
    } else {
      any_elastic = true;
      MIFE_REQUIRE(J.coef, MIFE_ERR_POINTER_IS_NULL, "job %d: elasticity without material", k);
    }
  }
  if (any_scalar) {
    MIFE_REQUIRE(scalar_desc && scalar_desc->dN && scalar_desc->w, MIFE_ERR_POINTER_IS_NULL, "scalar basis missing");
    MIFE_REQUIRE(scalar_desc->dim == 3 && scalar_desc->n_nodes == 8 && scalar_desc->n_gauss == 8, MIFE_ERR_ARG,
                 "batched scalar assembly takes trilinear elements with 2x2x2 Gauss points");
    MIFE_REQUIRE(!any_source || scalar_desc->N, MIFE_ERR_POINTER_IS_NULL, "source given without basis values N");
  }
  if (any_elastic) {
    MIFE_REQUIRE(elastic_desc && elastic_desc->dN && elastic_desc->w, MIFE_ERR_POINTER_IS_NULL,
                 "elastic basis missing");
    MIFE_REQUIRE(elastic_desc->dim == 3 && elastic_desc->n_nodes == 8 && elastic_desc->n_gauss == 8, MIFE_ERR_ARG,
                 "batched elastic assembly takes trilinear elements with 2x2x2 Gauss points");
  }
  // host table: jobs | segments of launch 0 | segments of launch 1 | ...
  char* H = (char*)table_host;
  BatchJob* hj = (BatchJob*)H;
  BatchSeg* hs = (BatchSeg*)(H + align256(sizeof(BatchJob) * n_jobs));
  for (int k = 0; k < n_jobs; ++k) {
    const mife_assembly_job& J = jobs[k];
    hj[k] = BatchJob{J.coords, J.elem_nodes, J.elem_dofs, J.coef, J.source, J.pos, J.order, J.vals, J.src_vec};
  }
  struct Launch {
    int kind, seg0, nseg, total;
  };
  std::vector<Launch> launches;
  int ns = 0;
  for (int c = 0; c < max_colours; ++c) {
    for (int kind : {MIFE_JOB_SCALAR, MIFE_JOB_ELASTIC}) {
      Launch L{kind, ns, 0, 0};
      for (int k = 0; k < n_jobs; ++k) {
        const mife_assembly_job& J = jobs[k];
        if (J.kind != kind || J.n_elem == 0 || c >= J.n_colours) continue;
        const int cnt = J.colour_ptr_host[c + 1] - J.colour_ptr_host[c];
        if (cnt <= 0) continue;
        MIFE_REQUIRE((long long)L.total + cnt < (1LL << 31), MIFE_ERR_ARG, "batch too large");
        hs[ns++] = BatchSeg{k, J.colour_ptr_host[c], L.total, 0};
        ++L.nseg;
        L.total += cnt;
      }
      if (L.nseg > 0) launches.push_back(L);
    }
  }
  hipStream_t s = (hipStream_t)stream;
  const size_t bytes = align256(sizeof(BatchJob) * n_jobs) + sizeof(BatchSeg) * (size_t)std::max(ns, 1);
  MIFE_CHECK_HIP(hipMemcpyAsync(work, table_host, bytes, hipMemcpyHostToDevice, s));
  MIFE_CHECK_HIP(hipStreamSynchronize(s));  // the host table may be reused at once
  const BatchJob* dj = (const BatchJob*)work;
  const BatchSeg* ds = (const BatchSeg*)((char*)work + align256(sizeof(BatchJob) * n_jobs));
  const int tk = prof::begin(s);
  for (const Launch& L : launches) {
    // blocks of `per` elements and `waves` wavefronts, as many as are resident
    auto grid = [&](int per, int waves) {
      return std::max(1, std::min(div_up(L.total, per), kBatchGrid * 4 / waves));
    };
    if (L.kind == MIFE_JOB_SCALAR) {
      q1_scalar_launch(L.total, [&](auto per, auto groups) {
        constexpr int E = decltype(per)::value, G = decltype(groups)::value;
        if (prec == MIFE_F64)
          scalar_batch_kernel<double, E, G><<<grid(E, E * G / 8), 8 * E * G, 0, s>>>(dj, ds + L.seg0, L.nseg, L.total, scalar_desc->dN,
                                                                   scalar_desc->N, scalar_desc->w);
        else
          scalar_batch_kernel<float, E, G><<<grid(E, E * G / 8), 8 * E * G, 0, s>>>(dj, ds + L.seg0, L.nseg, L.total, scalar_desc->dN,
                                                                  scalar_desc->N, scalar_desc->w);
      });
    } else {
      auto elastic = [&](auto zero) {
        using T = decltype(zero);
        auto go = [&](auto turns) {
          constexpr int TURNS = decltype(turns)::value;
          elastic_batch_kernel<T, TURNS><<<grid(4 * TURNS, 4), 256, 0, s>>>(dj, ds + L.seg0, L.nseg, L.total,
                                                                            elastic_desc->dN, elastic_desc->w);
        };
        switch (elastic_turns<T>(L.total, Form::kBatch)) {
          case 1: go(std::integral_constant<int, 1>{}); break;
          case 2: go(std::integral_constant<int, 2>{}); break;
          case 4: go(std::integral_constant<int, 4>{}); break;
          default: go(std::integral_constant<int, 8>{}); break;
        }
      };
      if (prec == MIFE_F64) elastic(0.0);
      else elastic(0.0f);
    }
  }
  prof::end(tk, s, prof::kAssembleBatch);
  MIFE_CHECK_HIP(hipGetLastError());
  return MIFE_OK;
}
