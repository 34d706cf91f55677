// omx_lu.hip -- blocked complex LU for CDNA4.
//
// Right-looking blocked factorisation P A = L U of a column-major Np x Np
// complex matrix (Np a multiple of the block size NB), in complex FP64
// (double2) or complex FP32 (float2).  Two pivot searches:
//   block (default)  diag_lu: partial pivoting among the rows of the panel's
//                  diagonal block, in one workgroup, which also inverts L11
//                  and U11; the solver recovers full accuracy by iterative
//                  refinement and refactors with the tournament if that fails
//   partial        tournament pivoting (TSLU, tslu_panel): register-resident
//                  partial-pivoting LUs of row chunks nominate candidate
//                  rows, a tree of merges picks the NB pivot rows, and its root
//                  writes the gather map, the block's factors and inverses
// Shared by both:
//   panel_mul      the two panel triangular solves as in-place MFMA products
//                  with the inverses: U12 = L11^{-1} A12, L21 = A21 U11^{-1};
//                  block pivoting applies its interchanges here
//   laswp_map      the tournament's row interchanges on the other columns, as
//                  one parallel gather/scatter
//   gemm_tile      A22 -= L21 U12 as complex products on the matrix cores:
//                  v_mfma_f64_16x16x4f64 (FP64) or v_mfma_f32_16x16x4f32
//                  (FP32), four real MFMAs per complex tile product, planar
//                  re/im operands staged through LDS; panels are taken in
//                  pairs so that the bulk update runs with K = 2 NB (groups of
//                  four, K = 4 NB, with gemm_split)
//   gemm_split     the FP32 bulk update (groups of four panels, K = 4 NB) on the
//                  bf16 matrix cores: operands split in three bf16 terms, six
//                  products per real product, FP32 accumulation (FP32-accurate)
//   trsv_kernel    sync-free blocked triangular solves: workgroup k owns
//                  block row k, consumes earlier blocks as they are
//                  published (tagged words) and applies its stored
//                  diagonal-block inverse
// Look-ahead: the pivoting of panel k+1 runs on a second stream while the
// bulk of panel k's trailing update runs on the first.
// This replaces the ScaLAPACK pzgesv path (scalapack/LinearSystemSolver.hpp:84-91)
// and Eigen's ColPivHouseholderQR (PreconditionedMatrixSolver.h:58, 75).
#include <climits>
#include <type_traits>
#include <vector>

#include "omx_kernels.hpp"

namespace omx {

template <typename T> struct CT;
// MFMA 16x16x4: lane l feeds A[l%16][l/16] and B[l/16][l%16]; accumulator
// register v of lane l holds D[row(l, v)][l%16] with
//   FP64 (v_mfma_f64_16x16x4f64): row = 4 v + l/16
//   FP32 (v_mfma_f32_16x16x4f32): row = 4 (l/16) + v
template <> struct CT<double2> {
  using R = double;
  typedef double V4 __attribute__((ext_vector_type(4)));
  static __device__ inline V4 mfma(R a, R b, V4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ inline int row(int lane, int v) { return 4 * v + (lane >> 4); }
};
template <> struct CT<float2> {
  using R = float;
  typedef float V4 __attribute__((ext_vector_type(4)));
  static __device__ inline V4 mfma(R a, R b, V4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ inline int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// Plain complex pair for register-resident arrays (the HIP vector types are
// unions that the compiler keeps in scratch memory when held in arrays).
template <typename R> struct Cx {
  R x, y;
};
template <typename T> using CxOf = Cx<decltype(T{}.x)>;
template <typename R> __device__ inline Cx<R> cx(R a, R b) { return Cx<R>{a, b}; }

template <typename T> __device__ inline T cm(T a, T b) {
  T r;
  r.x = a.x * b.x - a.y * b.y;
  r.y = a.x * b.y + a.y * b.x;
  return r;
}
template <typename T> __device__ inline T csub(T a, T b) {
  T r;
  r.x = a.x - b.x;
  r.y = a.y - b.y;
  return r;
}
template <typename T> __device__ inline double mag2(T a) { return (double)a.x * a.x + (double)a.y * a.y; }
// Whether a pivot counts as one (an FP64 square that underflows does not)
__device__ inline bool nonzero(Cx<double> a) { return mag2(a) > 0.0; }
__device__ inline bool nonzero(Cx<float> a) { return fabsf(a.x) + fabsf(a.y) > 0.0f; }
// Reciprocal: the hardware estimate refined by Newton's iteration
// r <- r + r (1 - d r), which doubles the number of correct bits per step:
// one step after the single-precision estimate (within 1 ulp), two after the
// double-precision one (about 23 correct bits).
__device__ inline float rcp_nr(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(r, __builtin_fmaf(-d, r, 1.0f), r);
}
__device__ inline double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}
__device__ inline float fmx(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fmx(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <typename T> __device__ inline T crecip(T a) {
  // 1 / a by Smith's scaling: with s the smaller and b the larger component
  // in magnitude, q = s / b, 1 / a = (1, -q) / (b + s q) for |re| >= |im| and
  // (q, -1) / (b + s q) otherwise, so no intermediate overflows
  using R = decltype(a.x);
  const bool re = fabs(a.x) >= fabs(a.y);
  const R b = re ? a.x : a.y, sm = re ? a.y : a.x;
  const R q = sm * rcp_nr(b), id = rcp_nr(fmx(sm, q, b));
  T r;
  r.x = re ? id : q * id;
  r.y = re ? -q * id : -id;
  return r;
}
// v - a b with fused multiply-adds
template <typename R> __device__ inline Cx<R> cfms(Cx<R> v, Cx<R> a, Cx<R> b) {
  Cx<R> r;
  r.x = fmx(-a.x, b.x, fmx(a.y, b.y, v.x));
  r.y = fmx(-a.x, b.y, fmx(-a.y, b.x, v.y));
  return r;
}

// Componentwise select (a ternary on the aggregate would go through memory).
template <typename R> __device__ inline Cx<R> csel(bool p, Cx<R> a, Cx<R> b) {
  Cx<R> r;
  r.x = p ? a.x : b.x;
  r.y = p ? a.y : b.y;
  return r;
}

// Value of lane l (wave-uniform) of a complex register pair.
__device__ inline double rdl1(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}
__device__ inline float rdl1(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
template <typename R> __device__ inline Cx<R> rdl(Cx<R> v, int l) { return Cx<R>{rdl1(v.x, l), rdl1(v.y, l)}; }

// Loads and stores with the nontemporal hint, for data a kernel streams once
// (a product's matrix, a bulk update's C tile): they stay out of the caches'
// replacement, which keeps the reused operands there.  In the FP64 product
// this raised 6.0 to 6.8 TB/s (N = 10240) and 5.6 to 6.0 TB/s (64 systems of
// N = 3840).
__device__ inline cplx ld_stream(const cplx *p) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  const d2 v = __builtin_nontemporal_load(reinterpret_cast<const d2 *>(p));
  return cplx{v.x, v.y};
}
__device__ inline float2 ld_stream(const float2 *p) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = __builtin_nontemporal_load(reinterpret_cast<const f2 *>(p));
  float2 r;
  r.x = v.x;
  r.y = v.y;
  return r;
}
// 16 bytes
__device__ inline void ld_stream16(const cplx *p, cplx (&e)[1]) { e[0] = ld_stream(p); }
__device__ inline void ld_stream16(const float2 *p, float2 (&e)[2]) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 v = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(p));
  e[0].x = v.x;
  e[0].y = v.y;
  e[1].x = v.z;
  e[1].y = v.w;
}
__device__ inline void st_stream(float2 *p, float2 c) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = {c.x, c.y};
  __builtin_nontemporal_store(v, reinterpret_cast<f2 *>(p));
}

__global__ void iota_kernel(int *p, int n, int sp) {
  p += (size_t)blockIdx.z * sp;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = i;
}

// ------------------------------------------------------------------ panel
// Maximum of an unsigned key over the 64 lanes of a wave, returned to every
// lane: row shifts build each 16-lane row's maximum in its lane 15, two row
// broadcasts combine the rows into lane 63.
__device__ inline unsigned wave_max_u32(unsigned x) {
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true));  // row_shr:1
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true));  // row_shr:2
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true));  // row_shr:4
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true));  // row_shr:8
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false));  // row_bcast:15
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false));  // row_bcast:31
  return (unsigned)__builtin_amdgcn_readlane((int)x, 63);
}

// Value of lane K of each row of 16 lanes (DPP row_newbcast), to the whole row.
template <int K> __device__ inline float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xF, 0xF, false));
}
template <int K> __device__ inline double row_bcast(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + K, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + K, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
template <int K, typename R> __device__ inline Cx<R> row_bcast(Cx<R> v) {
  return Cx<R>{row_bcast<K>(v.x), row_bcast<K>(v.y)};
}
// f(integral_constant<0>) ... f(integral_constant<N - 1>)
template <int N, int I = 0, typename F> __device__ __forceinline__ void each(F &&f) {
  if constexpr(I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// [L11^{-1} | U11^{-1}] of the factored block F (column-major, 65 apart, rinv the
// reciprocals of its diagonal, 0 for a zero) into dinv, by a workgroup of 8 waves, in place of F: the 16 x 16 diagonal blocks by
// substitution (waves 0-3 those of L11, waves 4-7 of U11; a row of 16 lanes
// holds all rows of 4 columns, so row k reaches them by DPP), then the blocks off
// the diagonal by X21 = -L22^{-1} (L21 L11^{-1}) and X12 = -U11^{-1} (U12
// U22^{-1}) on the matrix cores, 16 and then 32 wide.
//
// Bound: the serial chain.  A substitution over all 64 rows, lane = row, with
// row k broadcast by lane reads, took 64 steps of 16 complex updates: 22 us
// (FP64) of the panel's 65 us; these 15 steps and 4 products take 9 us (FP64; 7 FP32).
template <typename T> __device__ __forceinline__ void invert_block(CxOf<T> *F, const CxOf<T> *rinv, T *dinv) {
  using C = CxOf<T>;
  using R = typename CT<T>::R;
  using V4 = typename CT<T>::V4;
  const int t = threadIdx.x, lane = t & 63, q = __builtin_amdgcn_readfirstlane(t >> 6), li = lane & 15, g = lane >> 4;
  const C zero{}, one{1, 0};
  const bool low = q < 4;  // this wave works on L11, else on U11
  {
    const int o = 16 * (q & 3);
    C x[4], f[16];
#pragma unroll
    for(int k = 0; k < 16; ++k) f[k] = F[(o + k) * 65 + o + li];  // row li of the block
#pragma unroll
    for(int m = 0; m < 4; ++m) x[m] = csel(4 * g + m == li, one, zero);
    if(low) {
      // unit lower: for k: row i -= L[i][k] row k, i > k
      each<15>([&](auto ic) {
        constexpr int k = decltype(ic)::value;
        const C lik = csel(li > k, f[k], zero);
#pragma unroll
        for(int m = 0; m < 4; ++m) x[m] = cfms(x[m], lik, row_bcast<k>(x[m]));
      });
#pragma unroll
      for(int m = 0; m < 4; ++m)
        if(li > 4 * g + m) F[(o + 4 * g + m) * 65 + o + li] = x[m];
    } else {
      // U^{-1} = (D^{-1} U)^{-1} D^{-1} with D = diag(U): a unit-upper sweep
      // (row i -= (U[i][k] / U[i][i]) row k, i < k, k = 15..1), then column j
      // scaled by 1 / U[j][j]
      const C ri = rinv[o + li];
      each<15>([&](auto ic) {
        constexpr int k = 15 - decltype(ic)::value;
        const C uik = csel(li < k, cm(f[k], ri), zero);
#pragma unroll
        for(int m = 0; m < 4; ++m) x[m] = cfms(x[m], uik, row_bcast<k>(x[m]));
      });
#pragma unroll
      for(int m = 0; m < 4; ++m)
        if(li <= 4 * g + m) F[(o + 4 * g + m) * 65 + o + li] = cm(x[m], rinv[o + 4 * g + m]);
    }
  }
  // element (i, k) of the triangular factor's inverse, both within its diagonal block
  auto tri = [&](bool lo, int i, int k) {
    const C v = F[k * 65 + i];
    return lo ? csel(i > k, v, csel(i == k, one, zero)) : csel(i <= k, v, zero);
  };
  // D += S a b over steps k = k0 .. k0 + 3 + 4 (n - 1), a(k) of row li, b(s, k) of column li
  auto mac = [](V4 &dr, V4 &di, C a, C b) {
    dr = CT<T>::mfma(a.x, b.x, dr);
    di = CT<T>::mfma(a.x, b.y, di);
    dr = CT<T>::mfma(-a.y, b.y, dr);
    di = CT<T>::mfma(a.y, b.x, di);
  };
  __syncthreads();
  if(q < 2 || q > 5) {
    // pairs of 16: waves 0, 1 of L11, waves 6, 7 of U11 (each on a SIMD, and so a
    // matrix core, of its own).  The first product's
    // accumulators are the second's right operand as they stand: register v
    // holds row(lane, v), and any order of k will do
    const int p = q & 1, r0 = 32 * p + (low ? 16 : 0), c0 = 32 * p + (low ? 0 : 16);
    V4 tr = {0, 0, 0, 0}, ti = {0, 0, 0, 0}, xr = {0, 0, 0, 0}, xi = {0, 0, 0, 0};
    C l[4], m[4], r[4];
#pragma unroll
    for(int s = 0; s < 4; ++s) {
      m[s] = F[(c0 + 4 * s + g) * 65 + r0 + li];
      r[s] = tri(low, c0 + 4 * s + g, c0 + li);
      l[s] = tri(low, r0 + li, r0 + CT<T>::row(lane, s));
    }
#pragma unroll
    for(int s = 0; s < 4; ++s) mac(tr, ti, m[s], r[s]);
#pragma unroll
    for(int s = 0; s < 4; ++s) mac(xr, xi, C{-l[s].x, -l[s].y}, C{tr[s], ti[s]});
    // the block written here is read by this wave alone
#pragma unroll
    for(int v = 0; v < 4; ++v) F[(c0 + li) * 65 + r0 + CT<T>::row(lane, v)] = C{xr[v], xi[v]};
  }
  __syncthreads();
  {
    // the pair of 32: a wave one 16 x 16 tile (rows 16 a, columns 16 b) of the
    // two products, the first one's result passed on in F; of the triangles'
    // zero blocks one half of the steps is left out
    const int a = q & 1, b = (q >> 1) & 1, r0 = low ? 32 : 0, c0 = low ? 0 : 32;
    V4 tr = {0, 0, 0, 0}, ti = {0, 0, 0, 0}, xr = {0, 0, 0, 0}, xi = {0, 0, 0, 0};
    C m[8], r[8];
#pragma unroll
    for(int s = 0; s < 8; ++s) {
      m[s] = F[(c0 + 4 * s + g) * 65 + r0 + 16 * a + li];
      r[s] = tri(low, c0 + 4 * s + g, c0 + 16 * b + li);
    }
    if(!low || b == 0)
#pragma unroll
      for(int s = 0; s < 4; ++s) mac(tr, ti, m[s], r[s]);
    if(low || b == 1)
#pragma unroll
      for(int s = 4; s < 8; ++s) mac(tr, ti, m[s], r[s]);
    __syncthreads();
#pragma unroll
    for(int v = 0; v < 4; ++v) F[(c0 + 16 * b + li) * 65 + r0 + 16 * a + CT<T>::row(lane, v)] = C{tr[v], ti[v]};
#pragma unroll
    for(int s = 0; s < 8; ++s) m[s] = tri(low, r0 + 16 * a + li, r0 + 4 * s + g);
    __syncthreads();
#pragma unroll
    for(int s = 0; s < 8; ++s) r[s] = F[(c0 + 16 * b + li) * 65 + r0 + 4 * s + g];
    if(low || a == 0)
#pragma unroll
      for(int s = 0; s < 4; ++s) mac(xr, xi, C{-m[s].x, -m[s].y}, r[s]);
    if(!low || a == 1)
#pragma unroll
      for(int s = 4; s < 8; ++s) mac(xr, xi, C{-m[s].x, -m[s].y}, r[s]);
    __syncthreads();
#pragma unroll
    for(int v = 0; v < 4; ++v) F[(c0 + 16 * b + li) * 65 + r0 + 16 * a + CT<T>::row(lane, v)] = C{xr[v], xi[v]};
  }
  __syncthreads();
#pragma unroll
  for(int m = 0; m < 16; ++m) {
    const C v = tri(low, lane, 16 * (q & 3) + m);
    T o;
    o.x = v.x;
    o.y = v.y;
    dinv[(low ? 0 : 4096) + (16 * (q & 3) + m) * 64 + lane] = o;
  }
}

// Tournament pivoting (TSLU, Grigori, Demmel and Xiang 2011): the panel's pivot
// rows are chosen by a tree of local partial-pivoting LUs of up to 64 RPL rows,
// each in one workgroup of 8 waves: the leaves nominate 64 rows of their chunk,
// a merge takes the candidates of RPL sets, and the last one (the root, which
// may be a leaf) also writes the selected rows' factors (wlu, column-major 64 x
// 64), their inverses, the gather map that brings the rows to the top
// (mdst <- msrc, at most 128 entries) and the permutation.
//
// As diag_lu, which stands below: a wave holds 8 columns, here of RPL rows per
// lane; the owner of a column takes the largest |.|^2 of the rows left, in FP64 (the
// upper words are compared first, the lower ones when lanes tie; the first row on
// ties), and the waves of later columns follow by the published steps.  A pivot row sits in one of RPL register slots:
// the step branches on the slot, uniform in the wave.  The multipliers of four
// panels of 8 columns are kept; the owner of a fifth waits until the waves behind
// it have read the first.
//
// Bound: the chain of 64 pivot steps, per level of the tree.  With 128 rows per
// workgroup in 256 threads, three barriers a column and a tree of fan-in two,
// plus the inverses by one thread a column in a kernel of its own, the panels of
// an FP64 system of 1500 took 1.0 ms each and the solve 26.5 ms; with a barrier
// every 8 columns instead of the published steps 96 us a level and 7.3 ms; now 54 us
// and 4.76 ms.
template <typename T, int RPL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(1, 2))) void tslu_panel(
    const T *A, size_t lda, int Np, int j0, int gin, const int *cin, int *cout, T *wlu, T *dinv, int *mdst, int *msrc,
    int *mcnt, int *perm, int *status) {
  using C = CxOf<T>;
  constexpr int ROWS = 64 * RPL, RING = 4, LM = RING * 8 * ROWS, FB = 64 * 65;
  // the multipliers of RING panels of 8 columns ([step][row]), and after the last
  // of them the factored block
  __shared__ C buf[LM > FB ? LM : FB];
  // step c, once published: 1 + its row's place, + 1024 for a zero pivot; the
  // reciprocals (64 more slots in both take the other lanes' stores); the panels
  // that wave q has read; the step of each place
  __shared__ int step[128], seen[8], pos[ROWS];
  __shared__ C rinv[128];
  __shared__ int rid[ROWS], outpos[64], wtop[64];
  const int t = threadIdx.x, lane = t & 63, q = __builtin_amdgcn_readfirstlane(t >> 6), g = blockIdx.x;
  const bool root = gridDim.x == 1;
  const C zero{};
  const int r0 = j0 + g * ROWS;
  const int R = cin ? 64 * min(RPL, gin - RPL * g) : min(ROWS, Np - r0);
  if(t < R) rid[t] = cin ? cin[g * ROWS + t] : r0 + t;
  if(t < 64) step[t] = 0;
  if(t < 8) seen[t] = 0;
  if(t < ROWS) pos[t] = -1;
  __syncthreads();
  C v[RPL][8];
  bool used[RPL];
#pragma unroll
  for(int s = 0; s < RPL; ++s) {
    const int idx = lane + 64 * s;
    used[s] = idx >= R;
    const T *row = A + (size_t)(j0 + 8 * q) * lda + (idx < R ? rid[idx] : j0);
#pragma unroll
    for(int j = 0; j < 8; ++j) {
      const T a = row[(size_t)j * lda];
      v[s][j] = idx < R ? C{a.x, a.y} : zero;
    }
  }
  // columns from .. 7 of the row in slot sl of lane b (both uniform)
  auto pivot_row = [&](int sl, int b, C(&pr)[8], int from) {
#pragma unroll
    for(int s = 0; s < RPL; ++s)
      if(sl == s) {
#pragma unroll
        for(int j = 0; j < 8; ++j)
          if(j >= from) pr[j] = rdl(v[s][j], b);
      }
  };
  // the steps of the earlier owners
#pragma unroll 1
  for(int c = 0; c < 8 * q; ++c) {
    int e;
    do
      e = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&step[c], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    while(e == 0);
    e = (e & 1023) - 1;
    const int sl = e >> 6, b = e & 63;
    const C *lm = buf + (c & (8 * RING - 1)) * ROWS + lane;
    C pr[8], l[RPL];
#pragma unroll
    for(int s = 0; s < RPL; ++s) {
      l[s] = lm[64 * s];
      used[s] = used[s] || (s == sl && lane == b);
    }
    pivot_row(sl, b, pr, 0);
#pragma unroll
    for(int s = 0; s < RPL; ++s)
#pragma unroll
      for(int j = 0; j < 8; ++j) v[s][j] = cfms(v[s][j], l[s], pr[j]);
    if((c & 7) == 7 && lane == 0)
      __hip_atomic_store(&seen[q], c / 8 + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // its own: the ring's slots are free once every later wave has read panel q -
  // RING (they wait for earlier panels only, so this ends)
  if(q >= RING)
    for(int o = q + 1; o < 8; ++o)
      while(__builtin_amdgcn_readfirstlane(
                __hip_atomic_load(&seen[o], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) < q - RING + 1) {
      }
  __builtin_amdgcn_s_setprio(3);
#pragma unroll
  for(int jj = 0; jj < 8; ++jj) {
    const int c = 8 * q + jj;
    // this lane's candidate: its largest row left, the first on ties (NaN counts as
    // large: every step finds a row of its own)
    C best = v[0][jj];
    double kx = -1.0;
    int slot_of = 0;
    bool have = false;
#pragma unroll
    for(int s = 0; s < RPL; ++s) {
      const double m = mag2(v[s][jj]);
      const bool take = !used[s] && !(m <= kx);
      best = csel(take, v[s][jj], best);
      kx = take ? m : kx;
      slot_of = take ? s : slot_of;
      have = have || take;
    }
    // every lane the reciprocal of its own candidate while the maximum is found
    const bool sing = !(kx > 0.0);
    const C ir = csel(sing, zero, crecip(best));
    const unsigned hi = have ? (unsigned)__double2hiint(kx) : 0u;
    const unsigned M = wave_max_u32(hi);
    unsigned long long tied = __ballot(have && hi == M);
    if(tied & (tied - 1)) {  // the lower words among the lanes that tie in the upper one
      const unsigned lo = have && hi == M ? (unsigned)__double2loint(kx) : 0u;
      const unsigned L = wave_max_u32(lo);
      tied = __ballot(have && hi == M && lo == L);
    }
    int sl = 0, b = 0;
#pragma unroll
    for(int s = RPL - 1; s >= 0; --s) {
      const unsigned long long m = tied & __ballot(slot_of == s);
      if(m) {
        sl = s;
        b = __ffsll((long long)m) - 1;
      }
    }
    sl = __builtin_amdgcn_readfirstlane(sl);
    b = __builtin_amdgcn_readfirstlane(b);
    C pr[8];
    pivot_row(sl, b, pr, jj);
    const C ip = rdl(ir, b);
    C *lm = buf + (c & (8 * RING - 1)) * ROWS + lane;
#pragma unroll
    for(int s = 0; s < RPL; ++s) {
      used[s] = used[s] || (s == sl && lane == b);
      const C l = csel(used[s], zero, cm(v[s][jj], ip));
      v[s][jj] = csel(used[s], v[s][jj], l);
      lm[64 * s] = l;
#pragma unroll
      for(int j = jj + 1; j < 8; ++j) v[s][j] = cfms(v[s][j], l, pr[j]);
    }
    // published after the multipliers: a wave's LDS stores are done in order
    const int slot = lane == b ? c : 64 + lane;
    rinv[slot] = ir;
    asm volatile("" ::: "memory");
    __hip_atomic_store(&step[slot], (sing ? 1025 : 1) + 64 * sl + lane, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __builtin_amdgcn_s_setprio(0);
  __syncthreads();  // all steps published and all multipliers read
  const int own = step[lane], mine = (own & 1023) - 1;  // the place of step `lane`
  if(!root) {
    if(q == 0) cout[g * 64 + lane] = rid[mine];
    return;
  }
  if(q == 0) {
    pos[mine] = lane;
    const unsigned long long zm = __ballot(own > 1024);
    if(zm && lane == 0) atomicCAS(&status[0], 0, j0 + __ffsll((long long)zm));
  }
  __syncthreads();
  int mypos[RPL];
#pragma unroll
  for(int s = 0; s < RPL; ++s) mypos[s] = pos[lane + 64 * s];
  // the selected rows' factors in pivoted order
#pragma unroll
  for(int s = 0; s < RPL; ++s)
    if(mypos[s] >= 0) {
#pragma unroll
      for(int j = 0; j < 8; ++j) {
        const int col = 8 * q + j;
        buf[col * 65 + mypos[s]] = v[s][j];
        T o;
        o.x = v[s][j].x;
        o.y = v[s][j].y;
        wlu[col * 64 + mypos[s]] = o;
      }
    }
  if(t < 64) wtop[t] = 0;
  __syncthreads();
  if(q == 0) {
    // winner lane goes to row j0 + lane; the top rows that did not win take the
    // places of the winners from further down, in order
    const int X = rid[mine];
    const bool in_top = X < j0 + 64;
    if(in_top) wtop[X - j0] = 1;
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const unsigned long long om = __ballot(!in_top);
    if(!in_top) outpos[__popcll(om & below)] = X;
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    const bool gone = wtop[lane] == 0;  // row j0 + lane is displaced
    const unsigned long long gm = __ballot(gone), mm = __ballot(X != j0 + lane);
    const int v0 = perm[X], v1 = perm[j0 + lane];
    // every lane's reads have returned before the first write
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int n0 = __popcll(mm);
    if(X != j0 + lane) {
      const int i = __popcll(mm & below);
      mdst[i] = j0 + lane;
      msrc[i] = X;
      perm[j0 + lane] = v0;
    }
    if(gone) {
      const int i = __popcll(gm & below), dst = outpos[i];
      mdst[n0 + i] = dst;
      msrc[n0 + i] = j0 + lane;
      perm[dst] = v1;
    }
    if(lane == 0) *mcnt = n0 + __popcll(gm);
  }
  invert_block<T>(buf, rinv, dinv);
}

// Rows per lane of tslu_panel, and so the tree's fan-in: as many as the
// register file holds (four FP64 rows of 8 columns need three times the
// scratch; FP64 solves with 3 / 2 rows: N = 1500 7.9 / 8.5 ms, N = 4000 28.9 /
// 30.8 ms).
template <typename T> struct TsluCfg {
  static constexpr int RPL = sizeof(T) == 16 ? 3 : 4;
};

// Diagonal-block pivoting: LU with partial pivoting restricted to the 64 x 64
// diagonal block of the panel (rows are chosen among the block's rows; the
// interchanges are applied to whole rows), then the inverses of L11 and U11.
// One workgroup of 8 waves.  Elimination: wave q holds columns 8 q .. 8 q + 7 of
// every row in registers, lane = row; rows are not moved (the pivot order is
// recorded instead).  The waves run without barriers: the owner of a column
// chooses the pivot (DPP maximum of a 32-bit key: max(|re|, |im|) as a float with
// the row in the low bits), leaves the multipliers in LDS and counts the step as
// published; the waves of later columns follow the count, so the next owner has
// applied all but the last steps when its own begin.  Every lane takes the
// reciprocal of its own entry while the maximum is on its way.  Writes the
// factored block into A, the inverses into dinv ([L11^{-1} | U11^{-1}],
// column-major), the block's row map (row j0 + i <- msrc[i]) and the permutation.
//
// Bound: the chain of 64 pivot steps (maximum, multiplier, the next column's
// update) at 2.4 GHz.  With a barrier a panel of 8 columns, the reciprocal after
// the maximum and inverses by substitution: 65 us FP64, 47 us FP32; now 35 and
// 26, of which the elimination takes 21 and 17.
template <typename T>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(1, 2))) void diag_lu(T *A, size_t lda, int j0, T *dinv, int *msrc, int *perm,
                                               int *status, BatchStrides bs) {
  using C = CxOf<T>;
  {
    const int z = blockIdx.z;
    A += z * bs.a;
    dinv += z * bs.inv;
    msrc += (size_t)z * bs.map;
    perm += (size_t)z * bs.perm;
    status += (size_t)z * bs.status;
  }
  // step c, once published: 1 + its row, + 128 for a zero pivot; the pivots'
  // reciprocals (in both, 64 more slots take what the other lanes write: a store
  // without a branch); the step of each row
  __shared__ int step[128], pos[64];
  __shared__ C rinv[128];
  // factored block in pivoted order, column-major [c * 65 + r]; before, the
  // multipliers of step c at [c * 64 + row] (0 on rows already chosen).  One
  // storage: the kernel's LDS stays small enough to start beside the bulk
  // update's workgroups
  __shared__ C F[64 * 65];
  const int t = threadIdx.x, lane = t & 63, q = __builtin_amdgcn_readfirstlane(t >> 6);
  const C zero{};
  C v[8];
#pragma unroll
  for(int j = 0; j < 8; ++j) {
    T a = A[(size_t)(j0 + 8 * q + j) * lda + j0 + lane];
    v[j] = C{a.x, a.y};
  }
  if(t < 64) step[t] = 0;
  __syncthreads();
  // The steps of the earlier owners, each published before it is read; owners
  // wait for earlier ones only, so every wait ends
  bool used = false;
#pragma unroll 1
  for(int c = 0; c < 8 * q; ++c) {
    int e;
    do
      e = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&step[c], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    while(e == 0);
    const int b = (e & 127) - 1;
    const C l = F[c * 64 + lane];
    used = used || lane == b;
#pragma unroll
    for(int j = 0; j < 8; ++j) v[j] = cfms(v[j], l, rdl(v[j], b));
  }
  __builtin_amdgcn_s_setprio(3);
#pragma unroll
  for(int jj = 0; jj < 8; ++jj) {
    const int c = 8 * q + jj;
    const float mx = (float)fmax(fabs((double)v[jj].x), fabs((double)v[jj].y));
    const unsigned key = used ? 0u : ((__float_as_uint(mx) & ~0x7Fu) | (unsigned)(127 - lane));
    const bool sing = !nonzero(v[jj]);
    const C ir = csel(sing, zero, crecip(v[jj]));
    const int e = (sing ? 129 : 1) + lane;
    const int b = 127 - (int)(wave_max_u32(key) & 127);
    used = used || lane == b;
    const C ip = rdl(ir, b);
    const C l = csel(used, zero, cm(v[jj], ip));
    v[jj] = csel(used, v[jj], l);
    F[c * 64 + lane] = l;
#pragma unroll
    for(int j = jj + 1; j < 8; ++j) v[j] = cfms(v[j], l, rdl(v[j], b));
    // published after the multipliers: a wave's LDS stores are done in order
    const int slot = lane == b ? c : 64 + lane;
    rinv[slot] = ir;
    asm volatile("" ::: "memory");
    __hip_atomic_store(&step[slot], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __builtin_amdgcn_s_setprio(0);
  __syncthreads();  // all steps published and all multipliers read
  const int own = step[lane], src = (own & 127) - 1;  // the row of step `lane`
  if(q == 0) pos[src] = lane;
  __syncthreads();
  const int mypos = pos[lane];
#pragma unroll
  for(int j = 0; j < 8; ++j) {
    const int col = 8 * q + j;
    F[col * 65 + mypos] = v[j];
    T o;
    o.x = v[j].x;
    o.y = v[j].y;
    A[(size_t)(j0 + col) * lda + j0 + mypos] = o;
  }
  // the first zero pivot, row map and running permutation (the last wave)
  if(q == 7) {
    const unsigned long long zm = __ballot(own > 128);
    if(zm && lane == 0) atomicCAS(&status[0], 0, j0 + __ffsll((long long)zm));
    const int old = perm[j0 + src];
    msrc[lane] = j0 + src;
    __builtin_amdgcn_wave_barrier();
    perm[j0 + lane] = old;
  }
  __syncthreads();
  invert_block<T>(F, rinv, dinv);
}

// ------------------------------------------------------------------ panel products
// The products with a panel's 64 x 64 inverses, in place, a strip of 16 NT rows or
// columns per workgroup of 4 waves:
//   blockIdx.x < nright   L21 = A21 U11^{-1} on rows first_r ..
//   then                  U12 = L11^{-1} (P A12) on columns first_c .., the block's
//                         interchanges applied as the strip is read (ms, null: none)
// PAIR: the second panel of a pair.  L21 as above; a strip of the columns goes
// through both panels: U12 of p0, block row p1 -= L(p1, p0) U12, U12 of p1.
//
// The strip is staged in LDS; wave w takes 16 of the block's 64 rows (columns),
// its part of the 64 x 64 operands in registers straight from memory, all loads
// of the chain first.  Either product is written so that the accumulators'
// lanes run along the columns of A.
//
// Bound: launch and load latency while the strips are fewer than the chip's
// workgroups, the matrix cores above.  These were 64-wide blocks (few workgroups,
// each 16 us FP64 and 9 us FP32) with the interchanges and the update of block
// row p1 in launches of their own: five launches a pair that are now one.
template <typename T, int NT, bool PAIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void panel_mul(
    T *A, size_t lda, int p0, int p1, int nright, int first_r, int first_c, const T *d0, const T *d1, const int *ms0,
    const int *ms1, BatchStrides bs) {
  using C = CxOf<T>;
  using V4 = typename CT<T>::V4;
  constexpr int W = 16 * NT, LD = 65;
  A += blockIdx.z * bs.a;
  d0 += blockIdx.z * bs.inv;
  if(PAIR) d1 += blockIdx.z * bs.inv;
  __shared__ C S0[W * LD], S1[PAIR ? W * LD : 1];
  const int t = threadIdx.x, lane = t & 63, li = lane & 15, g = lane >> 4;
  // the waves' shares of a triangular product differ: spread them over the SIMDs
  const int tw = __builtin_amdgcn_readfirstlane(t >> 6), w = (tw + blockIdx.x) & 3;
  auto ld = [](const T *p) {
    const T v = *p;
    return C{v.x, v.y};
  };
  auto st = [](T *p, decltype(T{}.x) x, decltype(T{}.x) y) {
    T v;
    v.x = x;
    v.y = y;
    *p = v;
  };
  // x += over k of a(row li, k) b(k, column li), k = 4 s + g in step s
  auto mac = [](V4 &xr, V4 &xi, C a, C b) {
    xr = CT<T>::mfma(a.x, b.x, xr);
    xi = CT<T>::mfma(a.x, b.y, xi);
    xr = CT<T>::mfma(-a.y, b.y, xr);
    xi = CT<T>::mfma(a.y, b.x, xi);
  };
  if((int)blockIdx.x < nright) {
    const int off = first_r + W * blockIdx.x, j0 = PAIR ? p1 : p0;
    const T *M = (PAIR ? d1 : d0) + kNB * kNB;
    C m[16], v[4 * NT];
#pragma unroll
    for(int i = 0; i < 4 * NT; ++i) {
      const int e = t + 256 * i, r = e % W, k = e / W;
      v[i] = ld(A + (size_t)(j0 + k) * lda + off + r);
    }
#pragma unroll
    for(int s = 0; s < 16; ++s) m[s] = ld(M + (16 * w + li) * kNB + 4 * s + g);
#pragma unroll
    for(int i = 0; i < 4 * NT; ++i) {
      const int e = t + 256 * i, r = e % W, k = e / W;
      S0[r * LD + k] = v[i];
    }
    __syncthreads();
    V4 xr[NT], xi[NT];
#pragma unroll
    for(int n = 0; n < NT; ++n) xr[n] = xi[n] = V4{0, 0, 0, 0};
#pragma unroll
    for(int c = 0; c < 4; ++c)
      if(c <= w)  // U11^{-1} is zero below the diagonal
#pragma unroll
        for(int s = 4 * c; s < 4 * c + 4; ++s)
#pragma unroll
          for(int n = 0; n < NT; ++n) mac(xr[n], xi[n], m[s], S0[(16 * n + li) * LD + 4 * s + g]);
#pragma unroll
    for(int n = 0; n < NT; ++n)
#pragma unroll
      for(int v = 0; v < 4; ++v)
        st(A + (size_t)(j0 + 16 * w + CT<T>::row(lane, v)) * lda + off + 16 * n + li, xr[n][v], xi[n][v]);
    return;
  }
  const int off = first_c + W * ((int)blockIdx.x - nright);
  C m0[16], m1[PAIR ? 16 : 1], m2[PAIR ? 16 : 1], v[4 * NT];
  // lane k takes row k of the interchanged block
  const int s0 = ms0 ? ms0[(size_t)blockIdx.z * bs.map + lane] : p0 + lane;
  const int s1 = PAIR ? ms1[(size_t)blockIdx.z * bs.map + lane] - p1 : 0;
#pragma unroll
  for(int s = 0; s < 16; ++s) m0[s] = ld(d0 + (4 * s + g) * kNB + 16 * w + li);
#pragma unroll
  for(int i = 0; i < 4 * NT; ++i) v[i] = ld(A + (size_t)(off + 4 * i + tw) * lda + s0);
  V4 cr[NT], ci[NT];
  if constexpr(PAIR) {
#pragma unroll
    for(int n = 0; n < NT; ++n)
#pragma unroll
      for(int k = 0; k < 4; ++k) {
        const C x = ld(A + (size_t)(off + 16 * n + CT<T>::row(lane, k)) * lda + p1 + 16 * w + li);
        cr[n][k] = x.x;
        ci[n][k] = x.y;
      }
#pragma unroll
    for(int s = 0; s < 16; ++s) {
      const C x = ld(A + (size_t)(p0 + 4 * s + g) * lda + p1 + 16 * w + li);
      m1[s] = C{-x.x, -x.y};
    }
#pragma unroll
    for(int s = 0; s < 16; ++s) m2[s] = ld(d1 + (4 * s + g) * kNB + 16 * w + li);
  }
#pragma unroll
  for(int i = 0; i < 4 * NT; ++i) S0[(4 * i + tw) * LD + lane] = v[i];
  __syncthreads();
  V4 xr[NT], xi[NT];
  auto left = [&](const C *S, const C(&m)[16]) {
#pragma unroll
    for(int n = 0; n < NT; ++n) xr[n] = xi[n] = V4{0, 0, 0, 0};
#pragma unroll
    for(int c = 0; c < 4; ++c)
      if(c <= w)  // L11^{-1} is zero above the diagonal
#pragma unroll
        for(int s = 4 * c; s < 4 * c + 4; ++s)
#pragma unroll
          for(int n = 0; n < NT; ++n) mac(xr[n], xi[n], S[(16 * n + li) * LD + 4 * s + g], m[s]);
  };
  auto store = [&](int j0) {
#pragma unroll
    for(int n = 0; n < NT; ++n)
#pragma unroll
      for(int k = 0; k < 4; ++k)
        st(A + (size_t)(off + 16 * n + CT<T>::row(lane, k)) * lda + j0 + 16 * w + li, xr[n][k], xi[n][k]);
  };
  left(S0, m0);
  store(p0);
  if constexpr(PAIR) {
#pragma unroll
    for(int n = 0; n < NT; ++n)
#pragma unroll
      for(int k = 0; k < 4; ++k) S1[(16 * n + CT<T>::row(lane, k)) * LD + 16 * w + li] = C{xr[n][k], xi[n][k]};
    __syncthreads();
#pragma unroll
    for(int s = 0; s < 16; ++s)
#pragma unroll
      for(int n = 0; n < NT; ++n) mac(cr[n], ci[n], S1[(16 * n + li) * LD + 4 * s + g], m1[s]);
    // S0 was read out before the last barrier
#pragma unroll
    for(int n = 0; n < NT; ++n)
#pragma unroll
      for(int k = 0; k < 4; ++k) S0[(16 * n + CT<T>::row(lane, k)) * LD + 16 * w + li] = C{cr[n][k], ci[n][k]};
    __syncthreads();
    // p1's interchanges on the strip: a wave 4 NT of its columns
    C y[4 * NT];
#pragma unroll
    for(int i = 0; i < 4 * NT; ++i) y[i] = S0[(4 * i + tw) * LD + s1];
    // S1's readers are past the barrier
#pragma unroll
    for(int i = 0; i < 4 * NT; ++i) S1[(4 * i + tw) * LD + lane] = y[i];
    __syncthreads();
    left(S1, m2);
    store(p1);
  }
}
// Strip width: 16 while that fills the chip no more than twice, else 32 (the
// 64 x 64 operands are then read half as often).  The line is not sharp: with 256 /
// 512 / 1024 / 4096 strips FP64 solves of 2208 take 3.67 / 3.68 / 3.66 / 3.67 ms, mixed
// ones of 10240 31.6 / 31.6 / 31.7 / 31.7.
constexpr long kWideStrips = 512;
template <typename T, bool PAIR>
void panel_products(T *A, size_t lda, int p0, int p1, int rows, int first_r, int cols, int first_c, const T *d0,
                    const T *d1, const int *ms0, const int *ms1, hipStream_t st, int nb, BatchStrides bs) {
  if(rows + cols <= 0) return;
  const bool wide = (long)(rows + cols) / 16 * nb > kWideStrips;
  const int w = wide ? 32 : 16;
  const dim3 grid(rows / w + cols / w, 1, nb);
  if(wide)
    hipLaunchKernelGGL((panel_mul<T, 2, PAIR>), grid, dim3(256), 0, st, A, lda, p0, p1, rows / w, first_r, first_c, d0,
                       d1, ms0, ms1, bs);
  else
    hipLaunchKernelGGL((panel_mul<T, 1, PAIR>), grid, dim3(256), 0, st, A, lda, p0, p1, rows / w, first_r, first_c, d0,
                       d1, ms0, ms1, bs);
}

// ------------------------------------------------------------------ swaps
// Tournament pivoting: applies the gather map (rows mdst[i] <- msrc[i], i < *mcnt <=
// 128) to every column: each workgroup handles 8 columns, reads all moved entries
// into registers, then writes them back.  The columns j0 .. j0 + NB - 1 then take
// the factored block from wlu.
template <typename T>
__global__ __launch_bounds__(256) void laswp_map(T *A, size_t lda, int Np, const int *__restrict__ mdst,
                                                 const int *__restrict__ msrc, const int *__restrict__ mcnt,
                                                 const T *__restrict__ wlu, int j0) {
  const int m = *mcnt;
  const int cl = threadIdx.x / 32, li = threadIdx.x % 32, col = blockIdx.x * 8 + cl;
  T v[4];
  int d[4];
  if(col < Np) {
    T *a = A + (size_t)col * lda;
#pragma unroll
    for(int k = 0; k < 4; ++k) {
      int i = li + 32 * k;
      d[k] = i < m ? mdst[i] : -1;
      if(i < m) v[k] = a[msrc[i]];
    }
  }
  __syncthreads();
  if(col < Np) {
    T *a = A + (size_t)col * lda;
#pragma unroll
    for(int k = 0; k < 4; ++k)
      if(d[k] >= 0) a[d[k]] = v[k];
  }
  if(col >= j0 && col < j0 + kNB) {
    // the moves into the block's rows came from this column's 32 lanes, half a
    // wave: in order before these stores
    T *a = A + (size_t)col * lda + j0;
    const T *w = wlu + (col - j0) * kNB;
    __builtin_amdgcn_wave_barrier();
    a[li] = w[li];
    a[li + 32] = w[li + 32];
  }
}

// Deferred interchanges of block pivoting: panel k = blockIdx.y (>= 1)
// applies its map (NB rows at k NB) to the columns left of it.
template <typename T>
__global__ __launch_bounds__(256) void laswp_left(T *A, size_t lda, const int *__restrict__ msrc, BatchStrides bs) {
  A += blockIdx.z * bs.a;
  msrc += (size_t)blockIdx.z * bs.map;
  const int k = blockIdx.y + 1;
  const int cl = threadIdx.x / 32, li = threadIdx.x % 32;
  T *a = A + (size_t)(blockIdx.x * 8 + cl) * lda;
  if(blockIdx.x * 8 >= k * kNB) return;  // whole workgroup past the panel
  T v[2];
#pragma unroll
  for(int q = 0; q < 2; ++q) v[q] = a[msrc[k * kNB + li + 32 * q]];
  __syncthreads();
#pragma unroll
  for(int q = 0; q < 2; ++q) a[k * kNB + li + 32 * q] = v[q];
}

// ------------------------------------------------------------------ gemm
// Trailing update:
// C[row0 + m, col0 + n] -= sum_{k < KD} A[row0 + m, k0 + k] A[k0 + k, col0 + n]
// for m < M, n < N.  A TM x TN tile per workgroup of WGM x WGN waves, each
// wave (TM/WGM) x (TN/WGN) as 16 x 16 MFMA blocks with separate real and
// imaginary accumulators; K is staged through LDS in chunks of BK (planar
// re/im, rows padded to 16 banks) and the next chunk is fetched into
// registers while the current one is multiplied.
template <typename T, int TM, int TN, int KD, int WGM, int WGN, int BK>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_tile(T *A, size_t lda, int row0, int col0, int k0, int M,
                                                           int N, size_t sA) {
  A += blockIdx.z * sA;
  using R = typename CT<T>::R;
  using V4 = typename CT<T>::V4;
  constexpr int NT = 64 * WGM * WGN, PAD = 16;
  constexpr int WM = TM / WGM, WN = TN / WGN, FM = WM / 16, FN = WN / 16;
  constexpr int LA = TM * BK / NT, LB = TN * BK / NT;
  static_assert(LA * NT == TM * BK && LB * NT == TN * BK, "tile not divisible");
  __shared__ R As[2][BK][TM + PAD];
  __shared__ R Bs[2][BK][TN + PAD];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, wm = wv % WGM, wn = wv / WGM;
  const int bm = blockIdx.x * TM, bn = blockIdx.y * TN;
  V4 cr[FM][FN], ci[FM][FN];
#pragma unroll
  for(int a = 0; a < FM; ++a)
#pragma unroll
    for(int b = 0; b < FN; ++b) {
      cr[a][b] = V4{0, 0, 0, 0};
      ci[a][b] = V4{0, 0, 0, 0};
    }
  R ar_[LA], ai_[LA], br_[LB], bi_[LB];
  auto gload = [&](int kc) {
#pragma unroll
    for(int i = 0; i < LA; ++i) {
      const int idx = t + NT * i, r = idx % TM, kk = idx / TM;
      ar_[i] = 0;
      ai_[i] = 0;
      if(bm + r < M) {
        const T v = A[(size_t)(k0 + kc + kk) * lda + row0 + bm + r];
        ar_[i] = v.x;
        ai_[i] = v.y;
      }
    }
#pragma unroll
    for(int i = 0; i < LB; ++i) {
      const int idx = t + NT * i, kb = idx % BK, c = idx / BK;
      br_[i] = 0;
      bi_[i] = 0;
      if(bn + c < N) {
        const T v = A[(size_t)(col0 + bn + c) * lda + k0 + kc + kb];
        br_[i] = v.x;
        bi_[i] = v.y;
      }
    }
  };
  gload(0);
#pragma unroll 1
  for(int kc = 0; kc < KD; kc += BK) {
    __syncthreads();  // the previous chunk has been read out of LDS
#pragma unroll
    for(int i = 0; i < LA; ++i) {
      const int idx = t + NT * i, r = idx % TM, kk = idx / TM;
      As[0][kk][r] = ar_[i];
      As[1][kk][r] = ai_[i];
    }
#pragma unroll
    for(int i = 0; i < LB; ++i) {
      const int idx = t + NT * i, kb = idx % BK, c = idx / BK;
      Bs[0][kb][c] = br_[i];
      Bs[1][kb][c] = bi_[i];
    }
    __syncthreads();
    if(kc + BK < KD) gload(kc + BK);
#pragma unroll
    for(int ks = 0; ks < BK / 4; ++ks) {
      const int kr = ks * 4 + (lane >> 4), li = lane & 15;
      R xr[FM], xi[FM], nxi[FM], yr[FN], yi[FN];
#pragma unroll
      for(int a = 0; a < FM; ++a) {
        xr[a] = As[0][kr][wm * WM + a * 16 + li];
        xi[a] = As[1][kr][wm * WM + a * 16 + li];
        nxi[a] = -xi[a];
      }
#pragma unroll
      for(int b = 0; b < FN; ++b) {
        yr[b] = Bs[0][kr][wn * WN + b * 16 + li];
        yi[b] = Bs[1][kr][wn * WN + b * 16 + li];
      }
#pragma unroll
      for(int a = 0; a < FM; ++a)
#pragma unroll
        for(int b = 0; b < FN; ++b) cr[a][b] = CT<T>::mfma(xr[a], yr[b], cr[a][b]);
#pragma unroll
      for(int a = 0; a < FM; ++a)
#pragma unroll
        for(int b = 0; b < FN; ++b) ci[a][b] = CT<T>::mfma(xr[a], yi[b], ci[a][b]);
#pragma unroll
      for(int a = 0; a < FM; ++a)
#pragma unroll
        for(int b = 0; b < FN; ++b) cr[a][b] = CT<T>::mfma(nxi[a], yi[b], cr[a][b]);
#pragma unroll
      for(int a = 0; a < FM; ++a)
#pragma unroll
        for(int b = 0; b < FN; ++b) ci[a][b] = CT<T>::mfma(xi[a], yr[b], ci[a][b]);
    }
  }
  // C -= the products: the loads of a group of EA block rows are all issued
  // before its first store (M and N are multiples of 16, so each 16 x 16
  // block is wholly in or out of range); FP64 takes one block row at a time
  // to stay within the register budget of four waves per SIMD
  constexpr int EA = sizeof(R) == 8 ? 1 : FM;
#pragma unroll
  for(int a0 = 0; a0 < FM; a0 += EA) {
    R vr[EA][FN][4], vi[EA][FN][4];
#pragma unroll
    for(int a = 0; a < EA; ++a)
#pragma unroll
      for(int b = 0; b < FN; ++b) {
        const int n = bn + wn * WN + b * 16 + (lane & 15), mb = bm + wm * WM + (a0 + a) * 16;
        const T *cp = A + (size_t)(col0 + n) * lda + row0;
#pragma unroll
        for(int v = 0; v < 4; ++v) {
          vr[a][b][v] = 0;
          vi[a][b][v] = 0;
          if(n < N && mb < M) {
            const T c = cp[mb + CT<T>::row(lane, v)];
            vr[a][b][v] = c.x;
            vi[a][b][v] = c.y;
          }
        }
      }
#pragma unroll
    for(int a = 0; a < EA; ++a)
#pragma unroll
      for(int b = 0; b < FN; ++b) {
        const int n = bn + wn * WN + b * 16 + (lane & 15), mb = bm + wm * WM + (a0 + a) * 16;
        if(n >= N || mb >= M) continue;
        T *cp = A + (size_t)(col0 + n) * lda + row0;
#pragma unroll
        for(int v = 0; v < 4; ++v) {
          T c;
          c.x = vr[a][b][v] - cr[a0 + a][b][v];
          c.y = vi[a][b][v] - ci[a0 + a][b][v];
          cp[mb + CT<T>::row(lane, v)] = c;
        }
      }
  }
}

// Tile configuration of the trailing updates (fastest of a sweep at
// M = N = 10112, K = 128: 103 TFLOP/s complex FP32, 55 TFLOP/s complex FP64).
template <typename T> struct UpdTile {
  static constexpr int TM = 128, TN = 64, WGM = 4, WGN = 2, BK = 16;
};

// Tile of the thin updates (K = NB, one of M and N = NB) on the panel
// chain: small tiles for many workgroups (fastest of a sweep at
// 10112 x 64 x 64: 7.9 us FP32, 15.7 us FP64, against 18.2 and 29.5 with
// UpdTile).
struct ThinTile {
  static constexpr int TM = 32, TN = 32, WGM = 2, WGN = 2, BK = 16;
};

// C -= A B over an M x N block (M, N multiples of 64) with K = KD.
template <typename T, int KD, typename U = UpdTile<T>>
void trailing_update(T *A, size_t lda, int row0, int col0, int k0, int M, int N, hipStream_t st, int nb = 1,
                     size_t sA = 0) {
  if(M <= 0 || N <= 0) return;
  hipLaunchKernelGGL((gemm_tile<T, U::TM, U::TN, KD, U::WGM, U::WGN, U::BK>),
                     dim3((M + U::TM - 1) / U::TM, (N + U::TN - 1) / U::TN, nb), dim3(64 * U::WGM * U::WGN), 0, st, A,
                     lda, row0, col0, k0, M, N, sA);
}

// ------------------------------------------------------------------ split-bf16 bulk update
// The complex-FP32 bulk update C -= A B (K = KD) on the bf16 matrix cores:
// every FP32 operand x is split in three bf16 terms x = x1 + x2 + x3 (each
// the round-to-nearest bf16 of what the previous ones leave; x - x1 - x2 - x3
// is below 2^-24 |x|) and the six products x_i y_j with i + j <= 4 (1-based)
// are accumulated in FP32 by v_mfma_f32_32x32x16_bf16: the result has the
// accuracy of an FP32 product (the dropped terms are below 2^-24 |x y|) at
// six bf16 instructions per real product, against the FP32 MFMA's 1/16 of the
// bf16 rate.
//
// The complex product is a real one over k' = 2 k + part:
//   D[n][m] = sum_k' X[n][k'] Y[k'][m],   X[n][2k] = Re B(k,n), X[n][2k+1] = Im B(k,n)
//   Re: Y[2k][m] = Re A(m,k), Y[2k+1][m] = -Im A(m,k)
//   Im: Y[2k][m] = Im A(m,k), Y[2k+1][m] =  Re A(m,k)
// X is B's column in its natural (re, im) storage; both Y are formed from the
// staged A by a sign flip or a swap of the bf16 halves of each 32-bit word.
// D's lanes run along m, so the epilogue reads and writes C's columns in
// 128-byte runs.
//
// LDS holds the three split planes of a K chunk as 16-byte units (4 complex k
// of one row of A or one column of B); the global loads of chunk c + 1 are in
// flight while chunk c is multiplied.  Workgroups are numbered so that each XCD takes a contiguous range of
// tiles, walked in groups of GM tile rows (operands reused from its L2).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x16 mfma_bf16_32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

// f[0..7] -> three words of 8 bf16 each (x1, x2, x3 of every value)
__device__ inline void split_bf16x3(const float *f, u32x4 &h, u32x4 &m, u32x4 &l) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  auto pack = [](float a, float b) {  // one conversion for both
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  };
  auto rest = [](float x, unsigned half) { return x - __uint_as_float(half); };
#pragma unroll
  for(int d = 0; d < 4; ++d) {
    const float x = f[2 * d], y = f[2 * d + 1];
    h[d] = pack(x, y);
    const float x1 = rest(x, h[d] << 16), y1 = rest(y, h[d] & 0xffff0000u);
    m[d] = pack(x1, y1);
    l[d] = pack(rest(x1, m[d] << 16), rest(y1, m[d] & 0xffff0000u));
  }
}

// A wave of the 4 holds 64 x 64 of the tile in 128 accumulator registers, so that
// an operand read from LDS feeds two instructions, and the planes of one chunk
// take 48 KB: two workgroups share a CU, the one's loads, splitting and C tile
// beside the other's products.
//
// Bound: the matrix cores.  Per K = 128 at M = N = 9984 a pass costs 416 us (245
// TFLOP/s complex, six times that in bf16) and 200 us for C and the ends: 165
// TFLOP/s with K = 128, 198 with K = 256.  Eight waves of 32 x 64 in one
// workgroup per CU, double-buffered, C fetched during the last chunk: 154 and
// 185.  The products and their order, and so the bits, are the same.
template <int TM, int TN, int KD, int WGM, int WGN, int BK, int GM>
__global__ __launch_bounds__(64 * WGM * WGN, 2) void gemm_split(float2 *A, size_t lda, int row0, int col0, int k0,
                                                               int M, int N, size_t sA) {
  A += blockIdx.z * sA;
  constexpr int NT = 64 * WGM * WGN;
  constexpr int WM = TM / WGM, WN = TN / WGN, FM = WM / 32, FN = WN / 32;
  constexpr int KG = BK / 4, NC = KD / BK;
  constexpr int UA = TM * KG / NT, UB = TN * KG / NT;
  static_assert(UA * NT == TM * KG && UB * NT == TN * KG, "tile not divisible");
  static_assert(FM >= 1 && FN >= 1 && BK % 8 == 0 && KD % BK == 0, "tile shape");
  __shared__ u32x4 Ys[3][KG][TM];
  __shared__ u32x4 Xs[3][KG][TN];
  const int gx = (M + TM - 1) / TM, gy = (N + TN - 1) / TN, T = gx * gy;
  int L = blockIdx.x;
  const int full = T / 8 * 8;
  if(L < full) L = (L % 8) * (full / 8) + L / 8;
  const int per = GM * gy, g0 = (L / per) * GM, gsz = min(gx - g0, GM), r = L % per;
  const int bm = (g0 + r % gsz) * TM, bn = (r / gsz) * TN;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), wm = wv % WGM, wn = wv / WGM;
  f32x16 accR[FM][FN], accI[FM][FN];
#pragma unroll
  for(int a = 0; a < FM; ++a)
#pragma unroll
    for(int b = 0; b < FN; ++b) {
      accR[a][b] = f32x16{};
      accI[a][b] = f32x16{};
    }
  // rows and columns past the end read the last one: their products are not stored
  const float2 *pa[UA], *pb[UB];
#pragma unroll
  for(int i = 0; i < UA; ++i) {
    const int u = t + NT * i, m = u % TM, kg = u / TM;
    pa[i] = A + (size_t)(k0 + 4 * kg) * lda + row0 + min(bm + m, M - 1);
  }
#pragma unroll
  for(int i = 0; i < UB; ++i) {
    const int u = t + NT * i, kg = u % KG, n = u / KG;
    pb[i] = A + (size_t)(col0 + min(bn + n, N - 1)) * lda + k0 + 4 * kg;
  }
  float ga[UA][8], gb[UB][8];
  auto gload = [&](int kc) {
#pragma unroll
    for(int i = 0; i < UA; ++i)
#pragma unroll
      for(int j = 0; j < 4; ++j) {
        const float2 v = pa[i][(size_t)(kc + j) * lda];
        ga[i][2 * j] = v.x;
        ga[i][2 * j + 1] = v.y;
      }
#pragma unroll
    for(int i = 0; i < UB; ++i) {
      const float4 *p = reinterpret_cast<const float4 *>(pb[i] + kc);
      const float4 p0 = p[0], p1 = p[1];
      gb[i][0] = p0.x;
      gb[i][1] = p0.y;
      gb[i][2] = p0.z;
      gb[i][3] = p0.w;
      gb[i][4] = p1.x;
      gb[i][5] = p1.y;
      gb[i][6] = p1.z;
      gb[i][7] = p1.w;
    }
  };
  gload(0);
#pragma unroll 1
  for(int c = 0; c < NC; ++c) {
    __syncthreads();  // the previous chunk has been read out of LDS
#pragma unroll
    for(int i = 0; i < UA; ++i) {
      const int u = t + NT * i, m = u % TM, kg = u / TM;
      u32x4 h, md, lo;
      split_bf16x3(ga[i], h, md, lo);
      Ys[0][kg][m] = h;
      Ys[1][kg][m] = md;
      Ys[2][kg][m] = lo;
    }
#pragma unroll
    for(int i = 0; i < UB; ++i) {
      const int u = t + NT * i, kg = u % KG, n = u / KG;
      u32x4 h, md, lo;
      split_bf16x3(gb[i], h, md, lo);
      Xs[0][kg][n] = h;
      Xs[1][kg][n] = md;
      Xs[2][kg][n] = lo;
    }
    __syncthreads();
    if(c + 1 < NC) gload((c + 1) * BK);
#pragma unroll
    for(int ks = 0; ks < BK / 8; ++ks) {
      // lane l feeds rows/columns l % 32 at k' = 16 ks + 8 (l / 32) .. + 7
      const int kg = 2 * ks + (lane >> 5), li = lane & 31;
      u32x4 x[3][FN], yr[3][FM], yi[3][FM];
#pragma unroll
      for(int s = 0; s < 3; ++s) {
#pragma unroll
        for(int b = 0; b < FN; ++b) x[s][b] = Xs[s][kg][wn * WN + 32 * b + li];
#pragma unroll
        for(int a = 0; a < FM; ++a) {
          const u32x4 y = Ys[s][kg][wm * WM + 32 * a + li];
#pragma unroll
          for(int d = 0; d < 4; ++d) {
            yr[s][a][d] = y[d] ^ 0x80000000u;
            yi[s][a][d] = (y[d] >> 16) | (y[d] << 16);
          }
        }
      }
      // the small products first
      constexpr int SY[6] = {2, 1, 0, 1, 0, 0}, SX[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
      for(int p = 0; p < 6; ++p)
#pragma unroll
        for(int a = 0; a < FM; ++a)
#pragma unroll
          for(int b = 0; b < FN; ++b) {
            accR[a][b] = mfma_bf16_32(x[SX[p]][b], yr[SY[p]][a], accR[a][b]);
            accI[a][b] = mfma_bf16_32(x[SX[p]][b], yi[SY[p]][a], accI[a][b]);
          }
    }
  }
  // C's tile: lane l, register v of block (a, b) holds D[n][m] with
  // m = 32 a + l % 32, n = 32 b + 8 (v / 4) + 4 (l / 32) + v % 4; M and N are
  // multiples of 32, so each 32 x 32 block is wholly in or out of range.  Read
  // and written with the nontemporal hint (2 % at M = N = 9984)
#pragma unroll
  for(int b = 0; b < FN; ++b)
#pragma unroll
    for(int a = 0; a < FM; ++a) {
      const int mb = bm + wm * WM + 32 * a, nb = bn + wn * WN + 32 * b;
      if(mb >= M || nb >= N) continue;
      float2 *cp = A + (size_t)(col0 + nb + 4 * (lane >> 5)) * lda + row0 + mb + (lane & 31);
      float2 c[16];
#pragma unroll
      for(int v = 0; v < 16; ++v) c[v] = ld_stream(cp + (size_t)(8 * (v / 4) + (v % 4)) * lda);
#pragma unroll
      for(int v = 0; v < 16; ++v) {
        c[v].x -= accR[a][b][v];
        c[v].y -= accI[a][b][v];
        st_stream(cp + (size_t)(8 * (v / 4) + (v % 4)) * lda, c[v]);
      }
    }
}

// Tile of the split-bf16 update (fastest of a sweep at M = N = 9984 and at 16
// systems of 2304; 128 x 64 with 2 or 4 waves, chunks of 8 double-buffered and 8
// waves are within 8 % or slower).
struct SplitTile {
  static constexpr int TM = 128, TN = 128, WGM = 2, WGN = 2, BK = 16, GM = 8;
};

// The bulk update with K = KD (2 NB or 4 NB): split-bf16 for FP32 factors when
// `split`, gemm_tile otherwise.  M and N are multiples of 64.
constexpr int kThinTiles = 512;  // two split tiles for every CU
template <typename T, int KD = 2 * kNB>
void bulk_update(T *A, size_t lda, int row0, int col0, int k0, int M, int N, hipStream_t st, int nb, size_t sA,
                 bool split) {
  if(M <= 0 || N <= 0) return;
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128) * nb;
  if((M <= 2 * kNB || N <= 2 * kNB) && (!split || tiles < kThinTiles)) {
    // the next pair's columns or a second pair's block rows (on the panel chain's
    // critical path): small tiles over many workgroups finish sooner than a few
    // large split tiles (128 rows by 1800 columns: 9 us against 29); a batch's
    // fill the chip with split tiles as well
    trailing_update<T, KD, ThinTile>(A, lda, row0, col0, k0, M, N, st, nb, sA);
    return;
  }
  if constexpr(std::is_same<T, float2>::value) {
    if(split) {
      using U = SplitTile;
      const int tiles = ((M + U::TM - 1) / U::TM) * ((N + U::TN - 1) / U::TN);
      hipLaunchKernelGGL((gemm_split<U::TM, U::TN, KD, U::WGM, U::WGN, U::BK, U::GM>), dim3(tiles, 1, nb),
                         dim3(64 * U::WGM * U::WGN), 0, st, A, lda, row0, col0, k0, M, N, sA);
      return;
    }
  }
  trailing_update<T, KD>(A, lda, row0, col0, k0, M, N, st, nb, sA);
}

// ------------------------------------------------------------------ links
// The triangular solves' links (FP64 factors, variant 1) Linv_k L[k, k-1] (blockIdx.y = 0, k = blockIdx.x +
// 1) and Uinv_k U[k, k+1] (1, k = blockIdx.x), beside the inverses they are formed
// with: 64 x 64, column-major.  Wave w takes 16 rows.
template <typename T>
__global__ __launch_bounds__(256) void link_kernel(const T *A, size_t lda, const T *dinv, T *links, BatchStrides bs) {
  using C = CxOf<T>;
  using V4 = typename CT<T>::V4;
  const bool up = blockIdx.y;
  const int k = blockIdx.x + (up ? 0 : 1), kc = up ? k + 1 : k - 1;
  const size_t at = blockIdx.z * bs.inv + (size_t)k * 2 * kNB * kNB + (up ? kNB * kNB : 0);
  const T *M = dinv + at, *B = A + blockIdx.z * bs.a + (size_t)kc * kNB * lda + (size_t)k * kNB;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, li = lane & 15, g = lane >> 4;
  C m[16];
#pragma unroll
  for(int s = 0; s < 16; ++s) {
    const T v = M[(4 * s + g) * kNB + 16 * w + li];
    m[s] = C{v.x, v.y};
  }
#pragma unroll
  for(int n = 0; n < 4; ++n) {
    V4 xr = {0, 0, 0, 0}, xi = {0, 0, 0, 0};
#pragma unroll
    for(int s = 0; s < 16; ++s) {
      const T v = B[(size_t)(16 * n + li) * lda + 4 * s + g];
      xr = CT<T>::mfma(v.x, m[s].x, xr);
      xi = CT<T>::mfma(v.x, m[s].y, xi);
      xr = CT<T>::mfma(-v.y, m[s].y, xr);
      xi = CT<T>::mfma(v.y, m[s].x, xi);
    }
#pragma unroll
    for(int v = 0; v < 4; ++v) {
      T o;
      o.x = xr[v];
      o.y = xi[v];
      links[at + (16 * n + CT<T>::row(lane, v)) * kNB + 16 * w + li] = o;
    }
  }
}

void lu_links(const double2 *A, int Np, size_t lda, const LuWork &w, hipStream_t st) {
  double2 *dinv = reinterpret_cast<double2 *>(w.dinv);
  if(w.links && Np > kNB)
    hipLaunchKernelGGL((link_kernel<double2>), dim3(Np / kNB - 1, 2, w.nb), dim3(256), 0, st, A, lda, dinv,
                       dinv + links_at(Np), w.bs);
}

// ------------------------------------------------------------------ driver
// Panels of NB columns are taken in pairs (p0 = J, p1 = J + NB), and pairs in
// groups of one or two, so that the bulk of the trailing update runs with K = 2 NB
// or 4 NB.
//
// Block pivoting (interchanges stay inside a panel's 64 rows), two streams:
// sb (panel work) runs group s+1 while st (bulk updates) finishes group s.
//   sb  diag_lu p0; L21(p0) and U12(p0) on p1's columns; p1's columns -=
//       L21(p0) U12(p0); diag_lu p1
//   sb  (groups of two) L21(p1) and U12 of both on the second pair's columns;
//       these columns' update with K = 2 NB; the second pair as the first
//   sb  after st's bulk update of group s-1, on the far columns: U12(p0), block
//       row p1 -= L(p1, p0) U12(p0), U12(p1) (one launch); (groups of two) the
//       second pair's block rows' update with K = 2 NB, then their U12
//   st  A22 -= [L21 ..] [U12; ..]: the next group's columns first, pair by pair
//       (sb starts on them), then the rest
// Interchanges on the columns left of each panel are applied once at the end
// (panels touch disjoint rows, so their order does not matter).
//
// Tournament (partial) pivoting: one stream for the panel sequence, sb for
// the tournaments; every interchange is applied at once to all columns.
// Progress mark of a factorisation (see LuWork::ev_mark).
inline void mark(LuWork &w, hipStream_t st) {
  (void)hipEventRecord(w.ev_mark, st);
  if(w.on_mark) w.on_mark(w.mark_arg);
}

template <typename T>
int lu_factor(T *A, int Np, size_t lda, LuWork &w, hipStream_t st, LuProf *prof) {
  if(Np % kNB) return -1;
  const bool block = w.pivot == kPivotBlock;
  const int nb = w.nb;
  const BatchStrides bs = w.bs;
  if(!block && nb != 1) return -3;  // the tournament factors one system at a time
  hipStream_t sb = w.aux;
  T *wlu = reinterpret_cast<T *>(w.wlu);
  T *dinv = reinterpret_cast<T *>(w.dinv);
  auto dk = [&](int j0) { return dinv + (size_t)(j0 / kNB) * 2 * kNB * kNB; };
  hipLaunchKernelGGL(iota_kernel, dim3((Np + 255) / 256, 1, nb), dim3(256), 0, st, w.perm, Np, bs.perm);
  if(prof) {
    prof->used = 0;
    prof->gemm_flop = 0.0;
    prof->gemm_launches = 0;
  }
  auto links = [&] {
    if constexpr(std::is_same<T, double2>::value) lu_links(A, Np, lda, w, st);
  };
  if(block) {
    // G panels a group: quads (two pairs), whose bulk update has K = 4 NB, where
    // that update is the split-bf16 one, which C's traffic holds back at K = 2 NB;
    // pairs where gemm_tile does it, which the matrix cores bound at either K and
    // whose quads only lengthen the panel chain.  Mixed solves with quads / pairs:
    // N = 2720 4.63 / 4.70 ms, 10240 42.9 / 44.9 ms, 16 wavelengths of 2560 226 / 233
    // ms; FP64, N = 2208 4.48 / 4.10 ms
    constexpr bool f32 = std::is_same<T, float2>::value;
    const int G = f32 && w.split ? 4 : 2;
    // a pair's panels (the second if two); its columns are up to date
    auto pair = [&](int p0, bool two) {
      const int p1 = p0 + kNB;
      hipLaunchKernelGGL((diag_lu<T>), dim3(1, 1, nb), dim3(512), 0, sb, A, lda, p0, dk(p0), w.msrc + p0, w.perm,
                         w.status, bs);
      if(!two) return;
      panel_products<T, false>(A, lda, p0, p1, Np - p1, p1, kNB, p1, dk(p0), nullptr, w.msrc + p0, nullptr, sb, nb, bs);
      trailing_update<T, kNB, ThinTile>(A, lda, p1, p1, p0, Np - p1, kNB, sb, nb, bs.a);
      hipLaunchKernelGGL((diag_lu<T>), dim3(1, 1, nb), dim3(512), 0, sb, A, lda, p1, dk(p1), w.msrc + p1, w.perm,
                         w.status, bs);
    };
    // L21 of a pair's second panel on rows >= p0 + 2 NB (when l21); U12 of both on
    // cols columns from c0
    auto through = [&](int p0, bool l21, int cols, int c0) {
      const int p1 = p0 + kNB, below = p1 + kNB;
      panel_products<T, true>(A, lda, p0, p1, l21 ? Np - below : 0, below, cols, c0, dk(p0), dk(p1), w.msrc + p0,
                              w.msrc + p1, sb, nb, bs);
    };
    // ev_next, ev_piv: the next group's first and second pair are up to date
    (void)hipEventRecord(w.ev_next, st);
    (void)hipEventRecord(w.ev_piv, st);
    (void)hipEventRecord(w.ev_bulk, st);
    for(int J = 0, pi = 0; J < Np; J += G * kNB, ++pi) {
      const int np = std::min(G, (Np - J) / kNB);  // panels of this group
      const int q = J + 2 * kNB, far = J + np * kNB, restf = Np - far;
      const bool rec = prof && pi < prof->cap;
      hipEvent_t *pe = rec ? prof->ev + 4 * pi : nullptr;
      (void)hipStreamWaitEvent(sb, w.ev_next, 0);
      if(rec) (void)hipEventRecord(pe[0], sb);
      pair(J, np > 1);
      if(np > 2) {
        // the second pair's columns: through the first, then its update
        (void)hipStreamWaitEvent(sb, w.ev_piv, 0);
        through(J, true, (np - 2) * kNB, q);
        bulk_update<T>(A, lda, q, q, J, Np - q, (np - 2) * kNB, sb, nb, bs.a, w.split);
        pair(q, np > 3);
      }
      const int last = far - 2 * kNB;  // the group's last pair
      if(rec) (void)hipEventRecord(pe[1], sb);
      if(restf > 0) {
        (void)hipStreamWaitEvent(sb, w.ev_bulk, 0);
        if(G == 4) {
          through(J, false, restf, far);
          bulk_update<T>(A, lda, q, far, J, 2 * kNB, restf, sb, nb, bs.a, w.split);
        }
        through(last, true, restf, far);  // and L21 of the last panel
      }
      (void)hipEventRecord(w.ev_pan, sb);
      (void)hipStreamWaitEvent(st, w.ev_pan, 0);
      if(rec) (void)hipEventRecord(pe[2], st);
      if(restf > 0) {
        auto bulk = [&](int c0, int n) {
          if constexpr(f32)
            if(G == 4) return bulk_update<T, 4 * kNB>(A, lda, far, c0, J, restf, n, st, nb, bs.a, w.split);
          bulk_update<T>(A, lda, far, c0, J, restf, n, st, nb, bs.a, w.split);
        };
        // the next group's first pair, its second, and the rest
        int c0 = far;
        const int n1 = std::min(2 * kNB, Np - c0);
        bulk(c0, n1);
        (void)hipEventRecord(w.ev_next, st);
        c0 += n1;
        if(G == 4) {
          const int n2 = std::min(2 * kNB, Np - c0);
          bulk(c0, n2);
          (void)hipEventRecord(w.ev_piv, st);
          c0 += n2;
        }
        bulk(c0, Np - c0);
        (void)hipEventRecord(w.ev_bulk, st);
        if(rec) {
          prof->gemm_flop += 8.0 * (double)restf * restf * (G * kNB) * nb;
          prof->gemm_launches += (restf > n1 ? 2 : 1) + (G == 4 && Np - far > 4 * kNB ? 1 : 0);
        }
      }
      if(rec) {
        (void)hipEventRecord(pe[3], st);
        prof->used = pi + 1;
      }
      if(w.ev_mark && far >= w.mark_col && J < w.mark_col) mark(w, st);
    }
    if(w.ev_mark && Np < w.mark_col) mark(w, st);
    if(Np > kNB)
      hipLaunchKernelGGL((laswp_left<T>), dim3((Np - kNB) / 8, Np / kNB - 1, nb), dim3(256), 0, st, A, lda,
                         w.msrc, bs);
    links();
    return 0;
  }

  // ---- tournament pivoting
  auto pivoting = [&](int j0) {
    (void)hipEventRecord(w.ev_next, st);
    (void)hipStreamWaitEvent(sb, w.ev_next, 0);
    constexpr int RPL = TsluCfg<T>::RPL;
    static_assert(64 * RPL >= kPanelRows, "the candidate lists are sized for workgroups of kPanelRows rows");
    int gin = 0, buf = 0;
    for(int g = (Np - j0 + 64 * RPL - 1) / (64 * RPL);; g = (g + RPL - 1) / RPL) {
      hipLaunchKernelGGL((tslu_panel<T, RPL>), dim3(g), dim3(512), 0, sb, A, lda, Np, j0, gin,
                         gin ? w.cand[buf] : nullptr, w.cand[buf ^ 1], wlu, dk(j0), w.mdst, w.msrc, w.mcnt, w.perm,
                         w.status);
      if(g == 1) break;
      gin = g;
      buf ^= 1;
    }
    (void)hipEventRecord(w.ev_piv, sb);
  };
  // interchanges on every column, and the factored block
  auto swaps = [&](int j0) {
    (void)hipStreamWaitEvent(st, w.ev_piv, 0);
    hipLaunchKernelGGL((laswp_map<T>), dim3(Np / 8), dim3(256), 0, st, A, lda, Np, w.mdst, w.msrc, w.mcnt, wlu, j0);
  };
  // L21 and U12 of panel j0
  auto solves = [&](int j0) {
    const int rest = Np - j0 - kNB;
    panel_products<T, false>(A, lda, j0, 0, rest, j0 + kNB, rest, j0 + kNB, dk(j0), nullptr, nullptr, nullptr, st, 1, bs);
  };
  if((Np + kPanelRows - 1) / kPanelRows > w.gmax) return -2;
  pivoting(0);
  for(int J = 0, pi = 0; J < Np; J += 2 * kNB, ++pi) {
    const int p0 = J, p1 = J + kNB;
    const bool rec = prof && pi < prof->cap;
    hipEvent_t *pe = rec ? prof->ev + 4 * pi : nullptr;
    if(rec) (void)hipEventRecord(pe[0], st);
    swaps(p0);
    solves(p0);
    const int rest1 = Np - p1 - kNB;
    if(p1 < Np) {
      trailing_update<T, kNB, ThinTile>(A, lda, p1, p1, p0, Np - p1, kNB, st);
      pivoting(p1);
      // rows from below (not yet updated with p0 beyond p1) may move into
      // block row p1: interchange first, then update the block row
      swaps(p1);
      trailing_update<T, kNB, ThinTile>(A, lda, p1, p1 + kNB, p0, kNB, rest1, st);
      solves(p1);
    }
    if(rec) {
      (void)hipEventRecord(pe[1], st);
      (void)hipEventRecord(pe[2], st);
    }
    if(p1 < Np && rest1 > 0) {
      const int Jn = p1 + kNB;
      bulk_update<T>(A, lda, Jn, Jn, p0, rest1, kNB, st, 1, 0, w.split);
      pivoting(Jn);
      bulk_update<T>(A, lda, Jn, Jn + kNB, p0, rest1, rest1 - kNB, st, 1, 0, w.split);
      if(rec) {
        prof->gemm_flop += 8.0 * (double)rest1 * rest1 * (2 * kNB);
        prof->gemm_launches += rest1 > kNB ? 2 : 1;
      }
    }
    if(rec) {
      (void)hipEventRecord(pe[3], st);
      prof->used = pi + 1;
    }
    if(w.ev_mark && p1 + kNB >= w.mark_col && p0 < w.mark_col) mark(w, st);
  }
  if(w.ev_mark && Np < w.mark_col) mark(w, st);
  links();
  return 0;
}

// ------------------------------------------------------------------ solves
// Publication tags of the triangular solves: the low 4 bits of both 64-bit
// words of a published x entry hold 1 (the lower solve) or 2 (the upper
// solve), which changes the value by at most 2^-48 of itself.  The tags are
// fixed, so results do not depend on the history of launches.
constexpr unsigned long long kTagMask = 0xFull;
__device__ inline double with_tag(double v, unsigned tg) {
  return __longlong_as_double((long long)(((unsigned long long)__double_as_longlong(v) & ~kTagMask) | tg));
}
// The permuted right-hand side, with the tag bits cleared: a word the
// triangular solves have not yet published can never carry their tag.
__global__ void gather_kernel(const cplx *b, const int *perm, cplx *y, int Np, BatchStrides bs, const int *live) {
  const size_t z = blockIdx.z;
  if(live && !live[z * KF_COUNT]) return;
  b += z * bs.vec;
  y += z * bs.vec;
  perm += z * bs.perm;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < Np) {
    const cplx v = b[perm[i]];
    y[i] = mk(with_tag(v.x, 0u), with_tag(v.y, 0u));
  }
}

// Sync-free blocked triangular solve.  Workgroup K owns SB consecutive
// 64-row blocks (a super-block).  Far phase: it consumes the blocks x_b of
// earlier super-blocks as they are published and accumulates
// L[super-block rows, b] x_b, with the next 64 x 16 tile slice of each thread
// prefetched into registers while the current one is multiplied.  Near phase: the
// super-block's own blocks are solved in sequence inside the workgroup -- the
// contributions of the blocks just solved, then the stored inverse of the
// diagonal block -- so only every SB-th link of the chain crosses
// workgroups.  SB = 1 with links: the neighbour's contribution comes last, by one
// product with the stored Dinv_k L[k, k-1]: what waits on the chain's last link
// is that product alone, the rest and the inverse having been applied before (a
// solve of N = 2208: 95 -> 70 us; forming the links takes 12 us).  FP64 factors
// only: a product of FP32 factors would have to be rounded to 32 bits between the
// FP64 sums of the two products it replaces (and gave 71 -> 62 us at N = 2176).
// With PRE the near phase's tiles (diagonal-block inverses and
// the intra-super-block L tiles) are loaded into registers at kernel start
// (PRE = 1) or after the far phase (PRE = 2).  Thread t handles row
// r = t % 64 and columns 16 (t / 64) .. 16 (t / 64) + 15 of every tile.
//
// Publication: a solved block is written with device-coherent (agent-scope)
// 64-bit stores whose low bits carry the solve's tag, and nothing else: a
// consumer polls the block's words themselves with device-coherent loads
// until every word carries the tag, so it needs no flag, no ordering between
// stores, and no second read.  Each 64-bit word is single-copy atomic, and
// the words it replaces carry another tag (0 in the right-hand side the
// gather wrote, 1 from the lower solve before the upper one), so a tagged
// word is always the new value.  Neither side writes back or invalidates the L2.
template <typename T, bool LOWER, int SB, int PRE>
__global__ __launch_bounds__(256) void trsv_kernel(const T *__restrict__ A, size_t lda, int Np,
                                                   const T *__restrict__ dinv, cplx *x,
                                                   int *status, BatchStrides bs, const int *live,
                                                   const T *__restrict__ links) {
  constexpr int NB = kNB;
  constexpr int NI = SB * (SB - 1) / 2;
  const size_t zs = blockIdx.z;
  if(live && !live[zs * KF_COUNT]) return;  // the whole system: no workgroup waits for it
  A += zs * bs.a;
  dinv += zs * bs.inv;
  x += zs * bs.vec;
  constexpr unsigned tg = LOWER ? 1u : 2u;
  const int nblk = Np / NB, nsb = (nblk + SB - 1) / SB;
  const int K = LOWER ? blockIdx.x : nsb - 1 - blockIdx.x;
  const int kb0 = K * SB, nb = min(SB, nblk - kb0);
  const int t = threadIdx.x, r = t & 63;
  const int cq = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform
  constexpr int CH = 8;  // far blocks taken per round
  __shared__ cplx xs[CH * NB];
  __shared__ cplx part[4][NB];
  __shared__ cplx part2[SB][4][NB];
  __shared__ int nready_s;
  __shared__ cplx rhs[SB][NB];
  __shared__ cplx xsb[SB][NB];
  // right-hand sides of the super-block (only this workgroup writes them)
  cplx b0[SB];
#pragma unroll
  for(int s = 0; s < SB; ++s) b0[s] = (t < NB && s < nb) ? x[(size_t)(kb0 + s) * NB + t] : mk(0.0);
  // the thread's 16 entries of a 64 x 64 tile at base (column-major, leading
  // dimension ld): a wave-uniform column address plus the lane's row offset
  auto tile = [&](const T *base, size_t ld, T (&dst)[16]) {
    const T *col = base + (size_t)(cq * 16) * ld;
#pragma unroll
    for(int cc = 0; cc < 16; ++cc) dst[cc] = col[(size_t)cc * ld + (unsigned)r];
  };
  // diagonal-block inverse of block k, and the tile L[k, kc] (column-major in A)
  auto inv_base = [&](int k) { return dinv + (size_t)k * 2 * NB * NB + (LOWER ? 0 : NB * NB); };
  auto a_base = [&](int k, int kc) { return A + (size_t)kc * NB * lda + (size_t)k * NB; };
  // near-phase tiles: mv[s] = inverse of block kb0+s; lv[idx(s, s')] = L[kb0+s, kb0+s']
  T mv[PRE ? SB : 1][16], lv[PRE ? (NI > 0 ? NI : 1) : 1][16];
  auto preload = [&]() {
#pragma unroll
    for(int s = 0; s < SB; ++s)
      if(s < nb) tile(inv_base(kb0 + s), NB, mv[PRE ? s : 0]);
    int q = 0;
#pragma unroll
    for(int s = 0; s < SB; ++s)
#pragma unroll
      for(int s2 = 0; s2 < SB; ++s2) {
        if(LOWER ? (s2 < s) : (s2 > s)) {
          if(s < nb && s2 < nb) tile(a_base(kb0 + s, kb0 + s2), lda, lv[PRE ? q : 0]);
          ++q;
        }
      }
  };
  if(PRE == 1) preload();
  const int nfar_all = LOWER ? kb0 : nblk - (kb0 + nb);
  const bool lk = SB == 1 && links != nullptr && nfar_all > 0;
  const int nfar = nfar_all - (lk ? 1 : 0);
  T wl[SB == 1 ? 16 : 1];
  if constexpr(SB == 1)
    if(lk) tile(links + zs * bs.inv + (size_t)kb0 * 2 * NB * NB + (LOWER ? 0 : NB * NB), NB, wl);
  auto fblk = [&](int j) { return LOWER ? j : nblk - 1 - j; };  // j-th far block in order of publication
  // wave 0, one entry per lane: the far blocks from j0 on, as far as they are
  // published (at least one, at most CH, none past end), into xs: each poll reads
  // a whole block and keeps it when every word carries the tag; the blocks after
  // a published one are tried at once
  auto poll = [&](int j0, int end) {
    unsigned spins = 0;
    int nr = 0;
    bool drain = false;
    while(nr < CH && j0 + nr < end) {
      const unsigned long long *src =
          reinterpret_cast<const unsigned long long *>(x + (size_t)fblk(j0 + nr) * NB + t);
      const unsigned long long re = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned long long im = __hip_atomic_load(src + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool ok = (re & kTagMask) == tg && (im & kTagMask) == tg;
      if(__ballot(ok) == ~0ull) {
        xs[nr * NB + t] = mk(__longlong_as_double((long long)re), __longlong_as_double((long long)im));
        ++nr;
        continue;
      }
      if(nr > 0) break;
      if(__builtin_amdgcn_readfirstlane(
             __hip_atomic_load(&status[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) {
        drain = true;
        break;
      }
      if(++spins > (1u << 24)) {
        if(t == 0) __hip_atomic_store(&status[1], 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        drain = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if(drain) {  // a timed-out wait: finish with zeros (the host reports the error)
      nr = min(CH, end - j0);
      for(int c = 0; c < nr; ++c) xs[c * NB + t] = mk(0.0);
    }
    if(t == 0) nready_s = nr;
  };
  // ---- far phase
  cplx acc[SB];
#pragma unroll
  for(int s = 0; s < SB; ++s) acc[s] = mk(0.0);
  T cur[16], nxt[16];
  if(nfar > 0) tile(a_base(kb0, fblk(0)), lda, cur);
  for(int j0 = 0; j0 < nfar;) {
    if(t < 64) poll(j0, nfar);
    __syncthreads();
    const int nr = nready_s;
    for(int c = 0; c < nr; ++c) {
      const int j = j0 + c, b = fblk(j);
#pragma unroll
      for(int s = 0; s < SB; ++s) {
        if(s < nb) {
          // prefetch the next slice: (s + 1, b) or (0, next far block)
          const bool inner = s + 1 < nb;
          if(inner || j + 1 < nfar) tile(inner ? a_base(kb0 + s + 1, b) : a_base(kb0, fblk(j + 1)), lda, nxt);
#pragma unroll
          for(int cc = 0; cc < 16; ++cc) {
            const T v = cur[cc];
            const cplx xv = xs[c * NB + cq * 16 + cc];
            acc[s].x += (double)v.x * xv.x - (double)v.y * xv.y;
            acc[s].y += (double)v.x * xv.y + (double)v.y * xv.x;
          }
#pragma unroll
          for(int cc = 0; cc < 16; ++cc) cur[cc] = nxt[cc];
        }
      }
    }
    __syncthreads();
    j0 += nr;
  }
  if(PRE == 2) preload();
  // right-hand sides of the super-block's blocks minus the far contributions
#pragma unroll
  for(int s = 0; s < SB; ++s) part2[s][cq][r] = acc[s];
  __syncthreads();
  if(t < NB) {
#pragma unroll
    for(int s = 0; s < SB; ++s)
      if(s < nb) rhs[s][t] = b0[s] - (part2[s][0][t] + part2[s][1][t] + part2[s][2][t] + part2[s][3][t]);
  }
  __syncthreads();
  // ---- near phase: the super-block's blocks in order
#pragma unroll
  for(int i = 0; i < SB; ++i) {
    const int s = LOWER ? i : SB - 1 - i;  // compile-time index; blocks past nb are skipped
    if(s < nb) {
      const int k = kb0 + s;
      // contributions of the blocks of this super-block solved before
      cplx a = mk(0.0);
      int q = 0;
      bool any = false;
#pragma unroll
      for(int ss = 0; ss < SB; ++ss)
#pragma unroll
        for(int s2 = 0; s2 < SB; ++s2) {
          if(LOWER ? (s2 < ss) : (s2 > ss)) {
            if(ss == s && s2 < nb) {
              any = true;
              T lt[16];
              if(PRE) {
#pragma unroll
                for(int cc = 0; cc < 16; ++cc) lt[cc] = lv[PRE ? q : 0][cc];
              } else {
                tile(a_base(k, kb0 + s2), lda, lt);
              }
#pragma unroll
              for(int cc = 0; cc < 16; ++cc) {
                const cplx xv = xsb[s2][cq * 16 + cc];
                a.x += (double)lt[cc].x * xv.x - (double)lt[cc].y * xv.y;
                a.y += (double)lt[cc].x * xv.y + (double)lt[cc].y * xv.x;
              }
            }
            ++q;
          }
        }
      if(any) {
        part[cq][r] = a;
        __syncthreads();
        if(t < NB) xs[t] = rhs[s][t] - (part[0][t] + part[1][t] + part[2][t] + part[3][t]);
      } else {
        if(t < NB) xs[t] = rhs[s][t];
      }
      __syncthreads();
      // x_k = (diagonal block)^{-1} r
      T m[16];
      if(PRE) {
#pragma unroll
        for(int cc = 0; cc < 16; ++cc) m[cc] = mv[PRE ? s : 0][cc];
      } else {
        tile(inv_base(k), NB, m);
      }
      cplx y = mk(0.0);
#pragma unroll
      for(int cc = 0; cc < 16; ++cc) {
        const cplx sv = xs[cq * 16 + cc];
        y.x += (double)m[cc].x * sv.x - (double)m[cc].y * sv.y;
        y.y += (double)m[cc].x * sv.y + (double)m[cc].y * sv.x;
      }
      part[cq][r] = y;
      __syncthreads();
      cplx sum = mk(0.0);
      if(t < NB) sum = part[0][t] + part[1][t] + part[2][t] + part[3][t];
      if constexpr(SB == 1)
        if(lk) {
          if(t < 64) poll(nfar, nfar_all);
          __syncthreads();
          cplx l = mk(0.0);
#pragma unroll
          for(int cc = 0; cc < 16; ++cc) {
            const cplx xv = xs[cq * 16 + cc];
            l.x += (double)wl[cc].x * xv.x - (double)wl[cc].y * xv.y;
            l.y += (double)wl[cc].x * xv.y + (double)wl[cc].y * xv.x;
          }
          part[cq][r] = l;
          __syncthreads();
          if(t < NB) sum = sum - (part[0][t] + part[1][t] + part[2][t] + part[3][t]);
        }
      if(t < NB) {
        const cplx xk = mk(with_tag(sum.x, tg), with_tag(sum.y, tg));
        xsb[s][t] = xk;
        unsigned long long *dst = reinterpret_cast<unsigned long long *>(x + (size_t)k * NB + t);
        __hip_atomic_store(dst, (unsigned long long)__double_as_longlong(xk.x), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + 1, (unsigned long long)__double_as_longlong(xk.y), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();  // part and xs are rewritten by the next block
    }
  }
}

// Super-block size and near-phase prefetch of the triangular solves (the
// complex-FP64 tiles of a prefetch would not fit in the register file):
// variant 0 is the default, 1 one block per workgroup (every link crosses
// workgroups, least work per link), 2 four blocks per workgroup with the
// near-phase tiles loaded as used (fewer cross-workgroup links).
template <typename T> struct TrsvCfg;
template <> struct TrsvCfg<float2> {
  static constexpr int SB[kTrsvVariants] = {2, 1, 4};
  static constexpr int PRE[kTrsvVariants] = {1, 1, 0};
};
template <> struct TrsvCfg<double2> {
  static constexpr int SB[kTrsvVariants] = {2, 1, 4};
  static constexpr int PRE[kTrsvVariants] = {2, 2, 0};
};

template <typename T, int V>
static void trsv_pair(const T *A, int Np, size_t lda, LuWork &w, cplx *x, int nz, hipStream_t st) {
  constexpr int SB = TrsvCfg<T>::SB[V];
  constexpr int PRE = TrsvCfg<T>::PRE[V];
  const T *dinv = reinterpret_cast<const T *>(w.dinv), *links = nullptr;
  if(std::is_same<T, double2>::value && w.links) links = dinv + links_at(Np);
  const int nblk = Np / kNB, nsb = (nblk + SB - 1) / SB;
  hipLaunchKernelGGL((trsv_kernel<T, true, SB, PRE>), dim3(nsb, 1, nz), dim3(256), 0, st, A, lda, Np, dinv, x,
                     w.status, w.bs, w.live, links);
  hipLaunchKernelGGL((trsv_kernel<T, false, SB, PRE>), dim3(nsb, 1, nz), dim3(256), 0, st, A, lda, Np, dinv, x,
                     w.status, w.bs, w.live, links);
}

template <typename T>
void lu_solve(const T *A, int Np, size_t lda, LuWork &w, const cplx *b, cplx *x, hipStream_t st) {
  const int nz = w.nb;
  hipLaunchKernelGGL(gather_kernel, dim3((Np + 255) / 256, 1, nz), dim3(256), 0, st, b, w.perm, x, Np, w.bs, w.live);
  switch(w.trsv) {
  case 1: trsv_pair<T, 1>(A, Np, lda, w, x, nz, st); break;
  case 2: trsv_pair<T, 2>(A, Np, lda, w, x, nz, st); break;
  default: trsv_pair<T, 0>(A, Np, lda, w, x, nz, st); break;
  }
}

void bulk_update_probe(float2 *A, int Np, size_t lda, int nb, size_t sA, bool split, hipStream_t st) {
  const int m = Np - 4 * kNB;
  if(m <= 0) return;
  if(split) {
    bulk_update<float2, 4 * kNB>(A, lda, 4 * kNB, 4 * kNB, 0, m, m, st, nb, sA, true);
    return;
  }
  for(int k0 : {0, 2 * kNB}) bulk_update<float2>(A, lda, 4 * kNB, 4 * kNB, k0, m, m, st, nb, sA, false);
}

template int lu_factor<double2>(double2 *, int, size_t, LuWork &, hipStream_t, LuProf *);
template int lu_factor<float2>(float2 *, int, size_t, LuWork &, hipStream_t, LuProf *);
template void lu_solve<double2>(const double2 *, int, size_t, LuWork &, const cplx *, cplx *, hipStream_t);
template void lu_solve<float2>(const float2 *, int, size_t, LuWork &, const cplx *, cplx *, hipStream_t);

// ------------------------------------------------------------------ gemv
// y = A x for the FP64 matrix (residuals and GMRES) or its complex-FP32 copy
// (entries widened to FP64, FP64 vectors and sums), two-stage column split: 256
// rows by a run of columns per workgroup, 16 bytes of a column per thread and
// load (two FP32 rows, one FP64).
//
// Bound: HBM, once enough loads are in flight.  FP32, N = 49152: 3171 us with one
// row per thread and 32 parts (6.1 TB/s), 2772 with two and 16 (6.97); N = 10240:
// 191 and 128 us (6.5 TB/s).
template <typename T>
__global__ __launch_bounds__(sizeof(T) == 8 ? 128 : 256) void gemv_part_kernel(const T *__restrict__ A, size_t lda,
                                                                              int N, const cplx *__restrict__ x,
                                                                              cplx *part, int chunk, size_t sA,
                                                                              size_t sv, const int *flag) {
  constexpr int RPT = 16 / sizeof(T), TPB = 256 / RPT;
  const size_t zs = blockIdx.z;
  if(flag && !flag[zs * KF_COUNT]) return;
  A += zs * sA;
  x += zs * sv;
  part += (size_t)blockIdx.z * gridDim.y * N;
  __shared__ cplx xs[512];
  const int r = blockIdx.x * 256 + threadIdx.x * RPT;
  const int c0 = blockIdx.y * chunk, c1 = min(N, c0 + chunk);
  cplx acc[RPT];
#pragma unroll
  for(int i = 0; i < RPT; ++i) acc[i] = mk(0.0);
  for(int cb = c0; cb < c1; cb += 512) {
    int ce = min(c1, cb + 512);
    __syncthreads();
    for(int i = threadIdx.x; i < ce - cb; i += TPB) xs[i] = x[cb + i];
    __syncthreads();
    if(r < N) {
      const T *a = A + (size_t)cb * lda + r;
      int n = ce - cb;
#pragma unroll 8
      for(int c = 0; c < n; ++c) {
        T e[RPT];
        ld_stream16(a + (size_t)c * lda, e);
#pragma unroll
        for(int i = 0; i < RPT; ++i) {
          const double vx = e[i].x, vy = e[i].y;
          acc[i].x += vx * xs[c].x - vy * xs[c].y;
          acc[i].y += vx * xs[c].y + vy * xs[c].x;
        }
      }
    }
  }
  if(r < N)
#pragma unroll
    for(int i = 0; i < RPT; ++i) part[(size_t)blockIdx.y * N + r + i] = acc[i];
}
// Column parts of a product: the fewest (the longest runs of columns, the fewest
// partial vectors) that still give `want` workgroups.  FP64: 1280, about five per
// CU.  Measured on 3840 x 3840 systems: 6.75 TB/s with 8 parts for 64 systems
// against 5.94 with 32, 6.20 with 24 parts for 4 systems; one system with 32 / 64 /
// 96 parts: N = 2176 32.4 / 21.5 / 16.8 us, 2752 44 / 28 / 22, 5120 100 / 62 / 65,
// 10240 254 / 296 / 264.  FP32: 2560 of half the threads.  Few rows (N < 1280)
// keep 32 parts: the product is 4 us with either, and the next kernel adds them up.
inline int gemv_parts(int N, int nz, int most, int want) {
  const long rb = (N + 255) / 256;
  if(nz <= 1 && rb <= 5) return kGemvSplit;
  for(int s : {8, 12, 16, 24, 32, 48, 64, 96})
    if(s >= most || rb * nz * s >= want) return std::min(s, most);
  return most;
}
int gemv_partial(const cplx *A, size_t lda, int N, const cplx *x, cplx *part, hipStream_t st, int nb, size_t sA,
                 size_t sv, const int *flag, int live) {
  const int ns = gemv_parts(N, live, nb == 1 ? kGemvSplitMax : kGemvSplit, 1280), chunk = (N + ns - 1) / ns;
  hipLaunchKernelGGL(gemv_part_kernel<cplx>, dim3((N + 255) / 256, ns, nb), dim3(256), 0, st, A, lda, N, x, part,
                     chunk, sA, sv, flag);
  return ns;
}
int gemv_partial(const float2 *A, size_t lda, int N, const cplx *x, cplx *part, hipStream_t st, const int *flag) {
  // N even, A's columns on 16 bytes: the padded order is a multiple of 64
  const int ns = gemv_parts(N, 1, kGemvSplitMax, 2560), chunk = (N + ns - 1) / ns;
  hipLaunchKernelGGL(gemv_part_kernel<float2>, dim3((N + 255) / 256, ns, 1), dim3(128), 0, st, A, lda, N, x, part,
                     chunk, (size_t)0, (size_t)0, flag);
  return ns;
}

// ------------------------------------------------------------------ products of half the blocks
// Objects j of a workgroup (their sum over j leaves it once): as many as leave 1536
// workgroups, at most 8 and an eighth of the objects.  Not a number of chunks that 8
// divides: workgroups go to the 8 XCDs in turn, and a chunk's work grows with its
// index.  Times in us with 1, 2, 4, 8 objects: FP64, 66 objects of n = 126 (n = 2 nmax
// (nmax + 2)) 120, 110, 136, 206; 171 of 48 123, 112, 105, 111; 513 of 96 3220, 3160,
// 3137, 3135; 251 of 96 770, 767, 763, 999 (32 chunks of 8).
inline int sym_chunk(int P, int nb) {
  int ch = (int)std::max(1L, std::min({8L, (long)P / 8, (long)nb * P * P / 3072}));
  while(ch > 1 && (P + ch - 1) / ch % 8 == 0) ++ch;
  return ch;
}
size_t sym_scratch(int P, int nmax, int nb) {
  const size_t n = 2 * (size_t)nmax * (nmax + 2), ch = sym_chunk(P, nb), nc = (P + ch - 1) / ch;
  return nb * (nc * P + (size_t)P * (P - 1) / 2) * n;
}
// Small blocks leave a thread few columns between the barriers of its objects.
// Whole / half products, us: FP64 n = 6, N = 8202 167 / 628; n = 16, N = 8208 161 / 149,
// 24016 1377 / 1130; n = 30, N = 8220 164 / 140.  FP32 n = 16, N = 24016 709 / 849; n =
// 30, N = 8220 89 / 105, 24030 694 / 745; n = 48, N = 8208 89 / 78; n = 70 (rows of 560
// bytes), N = 8260 93 / 96, 24010 725 / 677, 49210 3006 / 2558; n = 96, N = 8256 86 / 66.
bool sym_pays(int nmax, bool f32) { return nmax >= (f32 ? 4 : 2); }
__device__ inline cplx sym_T(const SymArgs &a, const cplx *ov, int j, int pol, int n) {
  return ov[(((size_t)a.tkind * a.P + j) * 2 + pol) * (a.nmax + 1) + n];
}
// Row p's degree and polarisation, and its parity factor: (-1)^n, times -1 for TM.
__device__ inline double sym_sign(int p, int nf, int &n, int &pol) {
  int m;
  pol = p >= nf;
  unflat(p % nf, n, m);
  return ((n & 1) != 0) != (pol != 0) ? -1.0 : 1.0;
}
// The size by which a row's factors are compared: |T| falls like x^(2n+1) of the
// size parameter x, and its square underflows from degree 8 on at x = 2e-10
__device__ inline double sym_mag(cplx v) { return fmax(fabs(v.x), fabs(v.y)); }
__device__ inline cplx sym_widen(cplx v) { return v; }
__device__ inline cplx sym_widen(float2 v) { return cplx{(double)v.x, (double)v.y}; }

// Block (chunk c of objects j, object i < j): thread t is row p = t % n, the
// columns u, u + G, .. of u = t / n.  The sums over j of y_i go to part[c][i], each
// y_j's to z[pair].
//
// Bound: HBM, at half the bytes of the plain product, and the barriers between
// objects.  N = 49152 (n = 96): FP32 2.78 -> 1.86 ms, 5.2 TB/s of the half, FP64 5.50 ->
// 3.38, 5.7 TB/s; N = 10240 (n = 160), FP64: 249 -> 171 us, 4.9 TB/s; N = 2142: 20 -> 28,
// so single systems take it from kSymN on, where sym_pays.
template <typename T>
__global__ __launch_bounds__(512) void sym_pairs(SymArgs a, const T *__restrict__ A, const cplx *__restrict__ x, int CH,
                                                int G) {
  const int c = blockIdx.x, i = blockIdx.y, zs = blockIdx.z, P = a.P, nf = a.nmax * (a.nmax + 2), n = 2 * nf;
  if(a.flag && !a.flag[(size_t)zs * KF_COUNT]) return;
  const int j1 = min(P, (c + 1) * CH);
  if(j1 <= i + 1) return;  // no object of the chunk past i
  A += zs * a.sA;
  x += zs * a.sv;
  const cplx *ov = a.ov + zs * a.zov;
  const int nc = (P + CH - 1) / CH;
  cplx *part = a.scratch + zs * (((size_t)nc * P + (size_t)P * (P - 1) / 2) * n), *z = part + (size_t)nc * P * n;
  extern __shared__ cplx sh[];
  // the objects' vectors, with and without the signs; the column groups' sums
  cplx *xi = sh, *si = sh + n, *xj = sh + 2 * n, *sj = sh + 3 * n, *red = sh + 4 * n;
  const int t = threadIdx.x, u = t / n, p = t % n;
  const bool in = u < G;
  auto load = [&](int o, cplx *v, cplx *sv) {
    for(int q = t; q < n; q += blockDim.x) {
      int d, pl;
      const cplx e = x[(size_t)o * n + q];
      v[q] = e;
      sv[q] = sym_sign(q, nf, d, pl) * e;
    }
  };
  load(i, xi, si);
  int deg, pol;
  const double sp = sym_sign(p, nf, deg, pol);
  const cplx Ti = sym_T(a, ov, i, pol, deg);
  cplx acc = mk(0.0);
  // Columns by E, the next E (of the next object after the last) on their way while
  // these are summed: the barriers between objects then wait for no load.  E: four
  // waves a SIMD in either type (by 8 objects, FP64 with 4 / 6 / 8: N = 49152 3.67 /
  // 3.69 / 4.03 ms, 10240 176 / 205 / 193 us; FP32: 2.31 / 2.20 / 2.26 ms)
  constexpr int E = sizeof(T) == 8 ? 6 : 4;
  const int j0 = max(i + 1, c * CH), cnt = n / G, steps = (cnt + E - 1) / E;
  cplx Tn = sym_T(a, ov, j0, pol, deg);
  T cur[E], nxt[E];
  // the block whose row is the larger: S_ij times x_j, and with the signs x_i for
  // y_j; or S_ji times x_i, and with the signs x_j for y_i
  auto base = [&](int j, bool own) {
    return A + (size_t)((own ? j : i) * n + u) * a.lda + (size_t)(own ? i : j) * n + p;
  };
  auto fetch = [&](const T *e, int b, T(&d)[E]) {
#pragma unroll
    for(int k = 0; k < E; ++k) d[k] = ld_stream(e + (size_t)(G * min(E * b + k, cnt - 1)) * a.lda);
  };
  bool own = sym_mag(Ti) >= sym_mag(Tn);
  const T *e = base(j0, own);
  if(in) fetch(e, 0, cur);
  for(int j = j0; j < j1; ++j) {
    const cplx Tj = Tn;
    if(j + 1 < j1) Tn = sym_T(a, ov, j + 1, pol, deg);
    __syncthreads();
    load(j, xj, sj);
    __syncthreads();
    cplx f = mk(0.0), h = mk(0.0);
    const bool ownj = own;
    if(in) {
      const cplx *v = ownj ? xj : xi, *w = ownj ? si : sj;
      for(int b = 0; b < steps; ++b) {
        if(b + 1 < steps) {
          fetch(e, b + 1, nxt);
        } else if(j + 1 < j1) {
          own = sym_mag(Ti) >= sym_mag(Tn);
          e = base(j + 1, own);
          fetch(e, 0, nxt);
        }
#pragma unroll
        for(int k = 0; k < E; ++k) {
          const int q = u + G * (E * b + k);
          if(E * b + k < cnt) {
            const cplx m = sym_widen(cur[k]);
            f = f + m * v[q];
            h = h + m * w[q];
          }
        }
#pragma unroll
        for(int k = 0; k < E; ++k) cur[k] = nxt[k];
      }
      const cplx big = ownj ? Ti : Tj, small = ownj ? Tj : Ti;
      h = sp * ((sym_mag(big) > 0.0 ? small / big : mk(0.0)) * h);
    }
    const cplx yi = ownj ? f : h;
    cplx yj = ownj ? h : f;
    acc = acc + yi;
    if(G > 1) {
      if(in && u > 0) red[(u - 1) * n + p] = yj;
      __syncthreads();
      if(u == 0)
        for(int g = 1; g < G; ++g) yj = yj + red[(g - 1) * n + p];
    }
    if(u == 0) z[((size_t)j * (j - 1) / 2 + i) * n + p] = yj;
  }
  if(G > 1) {
    __syncthreads();
    if(in && u > 0) red[(u - 1) * n + p] = acc;
    __syncthreads();
    if(u == 0)
      for(int g = 1; g < G; ++g) acc = acc + red[(g - 1) * n + p];
  }
  if(u == 0) part[((size_t)c * P + i) * n + p] = acc;
}
// y of object i: x (the unit blocks), the parts of its row and the pairs (k, i), k < i.
__global__ __launch_bounds__(256) void sym_sum(SymArgs a, const cplx *__restrict__ x, cplx *y, int CH) {
  const int r = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6, zs = blockIdx.z, P = a.P;
  if(a.flag && !a.flag[(size_t)zs * KF_COUNT]) return;
  const int n = 2 * a.nmax * (a.nmax + 2), nc = (P + CH - 1) / CH;
  const cplx *part = a.scratch + zs * (((size_t)nc * P + (size_t)P * (P - 1) / 2) * n), *z = part + (size_t)nc * P * n;
  __shared__ cplx red[3][64];
  cplx s = mk(0.0);
  if(r < P * n) {  // the waves share the terms
    const int i = r / n, p = r % n, c0 = (i + 1) / CH;
    if(i + 1 < P)
#pragma unroll 4
      for(int c = c0 + w; c < nc; c += 4) s = s + part[((size_t)c * P + i) * n + p];
#pragma unroll 4
    for(int k = w; k < i; k += 4) s = s + z[((size_t)i * (i - 1) / 2 + k) * n + p];
  }
  if(w > 0) red[w - 1][threadIdx.x & 63] = s;
  __syncthreads();
  if(w > 0 || r >= a.Np) return;
  const int l = threadIdx.x & 63;
  y[zs * a.sv + r] = x[zs * a.sv + r] + ((s + red[0][l]) + (red[1][l] + red[2][l]));
}
template <typename T> void sym_run(const SymArgs &a, const T *A, const cplx *x, cplx *y, hipStream_t st) {
  const int n = 2 * a.nmax * (a.nmax + 2), CH = sym_chunk(a.P, a.nb), nc = (a.P + CH - 1) / CH;
  // column groups (of one size) that fill the waves best, 512 threads at most
  int G = 1;
  auto fill = [&](int g) { return (double)(n * g) / ((n * g + 63) / 64 * 64); };
  for(int g = 2; n * g <= 512; ++g)
    if(n % g == 0 && fill(g) > fill(G) + 0.03) G = g;
  hipLaunchKernelGGL((sym_pairs<T>), dim3(nc, a.P - 1, a.nb), dim3((n * G + 63) / 64 * 64),
                     sizeof(cplx) * (4 + G - 1) * n, st, a, A, x, CH, G);
  hipLaunchKernelGGL(sym_sum, dim3((a.Np + 63) / 64, 1, a.nb), dim3(256), 0, st, a, x, y, CH);
}
void sym_product(const SymArgs &a, const cplx *A, const cplx *x, cplx *y, hipStream_t st) { sym_run(a, A, x, y, st); }
void sym_product(const SymArgs &a, const float2 *A, const cplx *x, cplx *y, hipStream_t st) { sym_run(a, A, x, y, st); }

}  // namespace omx
