// omx_krylov.hip -- restarted flexible GMRES with its small algebra on the
// device, for nb systems in lockstep (system = blockIdx.y).
//
// One Arnoldi step after the product's partial sums is four launches:
//   kry_dots    w = the product; partial sums of V^H w
//   kry_orth    h = the sums; w -= V h; partial sums of the second pass
//   kry_orth2   the second pass; partial sums of |w|^2
//   kry_next    v_{j+1} = w / |w|; the system's first block rotates its
//               Hessenberg column (Gmres_Zcomp, PreconditionedMatrix.cpp:
//               892-985) and decides whether the system has converged
// Each block adds up the partial sums it needs by itself (they fit the L2), so
// no launch does nothing but reduce.  A cycle ends with kry_solve_y (the
// triangular system), kry_update (x += Z y) and kry_tiny; it begins with
// kry_resid (b - A x) and kry_begin (the decisions of the restart).
//
// Flags in device memory gate every kernel, the products and the
// preconditioner's solves, so the host may enqueue the next step before it
// knows whether this one converged: a step after the last does nothing.
//
// Bound: launch latency at small orders, the matrix product at large ones.  An
// Arnoldi step used to be eleven launches, three copies and a wait for the
// host's rotations: 70 us beside a product of 250 us at N = 10240, now 30 us.
// The refinement of 3 spheres of nmax 6 (N = 288) went from 650 to 340 us, an
// ordinary group of 16 clusters from 13.9 to 12.1 ms.
#include <algorithm>

#include "omx_kernels.hpp"

namespace omx {

namespace {

constexpr int kRows = 256;  // rows of a block, one per thread

__device__ inline cplx wave_red(cplx v) {
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_xor(v.x, o, 64);
    v.y += __shfl_xor(v.y, o, 64);
  }
  return v;
}
__device__ inline double wave_red(double v) {
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// Sum of one double per thread of a 256-thread block, to every thread.
__device__ inline double block_red(double v, double *lds) {
  v = wave_red(v);
  __syncthreads();
  if((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  return (lds[0] + lds[1]) + (lds[2] + lds[3]);
}

struct Sys {  // system z's part of the state
  cplx *H, *g, *cs, *sn, *y, *h;
  double *sc;
  int *fl;
  __device__ Sys(const KryState &s, int z) {
    const size_t m = s.m;
    cplx *c = s.c + (size_t)z * kry_cplx(s.m);
    H = c;
    g = H + m * (m + 1);
    cs = g + m + 1;
    sn = cs + m;
    y = sn + m;
    h = y + m;
    sc = s.sc + (size_t)z * KS_COUNT;
    fl = s.fl + (size_t)z * KF_COUNT;
  }
};

// part[blk][k] of system z: partial sums of block blk
__device__ inline cplx *part_of(const KryState &s, int pass, int z) {
  return s.part + ((size_t)pass * gridDim.y + z) * gridDim.x * (s.m + 2);
}
__device__ inline double *nrm_of(const KryState &s, int which, int z) {
  return s.pnrm + ((size_t)which * gridDim.y + z) * gridDim.x;
}

// hs[k] = sum over the blocks of part[blk][k], k < nv, by the whole block.
__device__ inline void sum_parts(const cplx *part, int ld, int nblk, int nv, cplx *hs, cplx *tmp) {
  const int t = threadIdx.x;
  for(int k0 = 0; k0 < nv; k0 += kRows) {
    const int nk = min(kRows, nv - k0), G = kRows / nk, k = t % nk, g = t / nk;
    cplx s = mk(0.0);
    if(g < G)
      for(int b = g; b < nblk; b += G) s = s + part[(size_t)b * ld + k0 + k];
    __syncthreads();
    tmp[t] = s;
    __syncthreads();
    if(t < nk) {
      for(int q = 1; q < G; ++q) s = s + tmp[q * nk + t];
      hs[k0 + t] = s;
    }
  }
  __syncthreads();
}
__device__ inline cplx shfl_xor(cplx v, int o) { return cplx{__shfl_xor(v.x, o, 64), __shfl_xor(v.y, o, 64)}; }
// (sum of a) + (sum of b) + ((sum of c) + (sum of d)) over the wave, each sum by
// halves (lanes 32 apart, 16 apart, ..), to every lane: the first two halvings
// take two and four of the sums at once, in the lanes the others leave.
__device__ inline cplx wave_red4(cplx a, cplx b, cplx c, cplx d) {
  const bool hi = threadIdx.x & 32, hj = threadIdx.x & 16;
  auto pick = [](bool p, cplx x, cplx y) { return cplx{p ? x.x : y.x, p ? x.y : y.y}; };
  const cplx u = pick(hi, b, a) + shfl_xor(pick(hi, a, b), 32);
  const cplx v = pick(hi, d, c) + shfl_xor(pick(hi, c, d), 32);
  cplx s = pick(hj, v, u) + shfl_xor(pick(hj, u, v), 16);
#pragma unroll
  for(int o = 8; o > 0; o >>= 1) s = s + shfl_xor(s, o);
  s = s + shfl_xor(s, 32);
  return s + shfl_xor(s, 16);
}

// Partial sums of V_k^H w over the block's rows, k < nv, into out[k]: a wave takes
// every fourth k over all 256 rows, one reduction each (with 64 rows a wave, and
// so four reductions for every k, the step's two passes took 28 us instead of 16
// at N = 2720, j = 35; the same sums).
__device__ inline void dots(const cplx *V, size_t ldk, int nv, cplx w, int n, cplx *out, cplx (&ws)[kRows]) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, r0 = blockIdx.x * kRows + lane;
  __syncthreads();
  ws[t] = w;
  __syncthreads();
  cplx x[4];
#pragma unroll
  for(int i = 0; i < 4; ++i) x[i] = ws[lane + 64 * i];
#pragma unroll 2
  for(int k = wv; k < nv; k += 4) {
    const cplx *v = V + (size_t)k * ldk + r0;
    cplx e[4];
#pragma unroll
    for(int i = 0; i < 4; ++i) {
      e[i] = mk(0.0);
      if(r0 + 64 * i < n) e[i] = conj(v[64 * i]) * x[i];
    }
    const cplx s = wave_red4(e[0], e[1], e[2], e[3]);
    if(lane == 0) out[k] = s;
  }
}

__global__ __launch_bounds__(kRows) void kry_dots(KryState s, const cplx *gpart, int ns, size_t sg) {
  const int z = blockIdx.y, j = s.j, r = blockIdx.x * kRows + threadIdx.x;
  const Sys q(s, z);
  if(!q.fl[KF_LIVE]) return;
  __shared__ cplx ws[kRows];
  cplx w = mk(0.0);
  cplx *W = s.w + z * s.sv;
  if(r < s.n) {
    if(ns > 0) {
      const cplx *g = gpart + z * sg + r;
#pragma unroll 8
      for(int k = 0; k < ns; ++k) w = w + g[(size_t)k * s.n];
      W[r] = w;
    } else {
      w = W[r];
    }
  }
  dots(s.V + z * s.sz, s.ldk, j + 1, w, s.n, part_of(s, 0, z) + (size_t)blockIdx.x * (s.m + 2), ws);
}

__global__ __launch_bounds__(kRows) void kry_orth(KryState s) {
  const int z = blockIdx.y, j = s.j, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  if(!q.fl[KF_LIVE]) return;
  __shared__ cplx ws[kRows], hs[260];
  sum_parts(part_of(s, 0, z), s.m + 2, gridDim.x, j + 1, hs, ws);
  if(blockIdx.x == 0)
    for(int k = t; k <= j; k += kRows) q.h[k] = hs[k];
  const cplx *V = s.V + z * s.sz;
  cplx w = mk(0.0);
  if(r < s.n) {
    w = s.w[z * s.sv + r];
#pragma unroll 8
    for(int k = 0; k <= j; ++k) w = w - V[(size_t)k * s.ldk + r] * hs[k];
    s.w[z * s.sv + r] = w;
  }
  dots(V, s.ldk, j + 1, w, s.n, part_of(s, 1, z) + (size_t)blockIdx.x * (s.m + 2), ws);
}

__global__ __launch_bounds__(kRows) void kry_orth2(KryState s) {
  const int z = blockIdx.y, j = s.j, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  if(!q.fl[KF_LIVE]) return;
  __shared__ cplx tmp[kRows], hs[260];
  __shared__ double lds[4];
  sum_parts(part_of(s, 1, z), s.m + 2, gridDim.x, j + 1, hs, tmp);
  if(blockIdx.x == 0)
    for(int k = t; k <= j; k += kRows) q.h[k] = q.h[k] + hs[k];
  const cplx *V = s.V + z * s.sz;
  double e = 0.0;
  if(r < s.n) {
    cplx w = s.w[z * s.sv + r];
#pragma unroll 8
    for(int k = 0; k <= j; ++k) w = w - V[(size_t)k * s.ldk + r] * hs[k];
    s.w[z * s.sv + r] = w;
    e = norm2(w);
  }
  e = block_red(e, lds);
  if(t == 0) nrm_of(s, 0, z)[blockIdx.x] = e;
}

__device__ inline double sum_norms(const double *p, int nblk, double *lds) {
  double e = 0.0;
  for(int b = threadIdx.x; b < nblk; b += kRows) e += p[b];
  return block_red(e, lds);
}

__global__ __launch_bounds__(kRows) void kry_next(KryState s, int *host) {
  const int z = blockIdx.y, j = s.j, m = s.m, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  if(!q.fl[KF_LIVE]) {
    if(blockIdx.x == 0 && t == 0) host[2 * z] = 0;
    return;
  }
  __shared__ double lds[4];
  __shared__ cplx hc[260], cs[260], sn[260];
  const double hn = sqrt(sum_norms(nrm_of(s, 0, z), gridDim.x, lds));
  if(r < s.n && hn > 0.0) s.V[z * s.sz + (size_t)(j + 1) * s.ldk + r] = (1.0 / hn) * s.w[z * s.sv + r];
  if(blockIdx.x) return;
  for(int k = t; k <= j; k += kRows) hc[k] = q.h[k];
  for(int k = t; k < j; k += kRows) {
    cs[k] = q.cs[k];
    sn[k] = q.sn[k];
  }
  __syncthreads();
  if(t == 0) {
    cplx a = hc[0];
    for(int i = 0; i < j; ++i) {  // the rotations so far
      const cplx b = hc[i + 1];
      hc[i] = cs[i].x * a + sn[i] * b;
      a = -(conj(sn[i]) * a) + cs[i].x * b;
    }
    // the new one, of (a, hn)
    const double aa = cabs(a), den = hypot(aa, hn);
    double c = 1.0;
    cplx n = mk(0.0);
    if(den > 0.0) {
      c = aa / den;
      n = (aa > 0.0 ? a / aa : mk(1.0)) * (hn / den);
    }
    hc[j] = c * a + hn * n;
    q.cs[j] = mk(c);
    q.sn[j] = n;
    const cplx gj = q.g[j], gn = -(conj(n) * gj);
    q.g[j] = c * gj;
    q.g[j + 1] = gn;
    const int its = ++q.fl[KF_ITS];
    q.fl[KF_J] = j + 1;
    const double goal = 0.5 * s.tol * q.sc[KS_BN], left = cabs(gn);
    const bool go = !(left <= goal) && left == left && hn > 0.0 && its < s.maxit;
    q.fl[KF_LIVE] = go ? 1 : 0;
    // 0: done; otherwise alive, with the binary digits to the goal
    host[2 * z] = go ? 1 : 0;
    host[2 * z + 1] = go && goal > 0.0 ? max(0, ilogb(left / goal)) : 0;
    __threadfence_system();
  }
  __syncthreads();
  for(int k = t; k <= j; k += kRows) q.H[(size_t)j * (m + 1) + k] = hc[k];
}

// y of the system's triangular system H y = g (jz x jz), by columns.
__global__ __launch_bounds__(kRows) void kry_solve_y(KryState s) {
  const int z = blockIdx.x, m = s.m, t = threadIdx.x;
  const Sys q(s, z);
  if(!q.fl[KF_ACTIVE]) return;
  __shared__ cplx a[260], yi;
  const int jj = q.fl[KF_J];
  for(int i = t; i < jj; i += kRows) a[i] = q.g[i];
  __syncthreads();
  for(int i = jj - 1; i >= 0; --i) {
    const cplx *Hc = q.H + (size_t)i * (m + 1);
    if(t == 0) yi = a[i] / Hc[i];
    __syncthreads();
    const cplx y = yi;
    for(int k = t; k < i; k += kRows) a[k] = a[k] - Hc[k] * y;
    if(t == 0) q.y[i] = y;
    __syncthreads();
  }
}

// x += Z y, and the partial norms of the correction and of x.
__global__ __launch_bounds__(kRows) void kry_update(KryState s, cplx *x) {
  const int z = blockIdx.y, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  if(!q.fl[KF_ACTIVE]) return;
  __shared__ cplx ys[260];
  __shared__ double lds[4];
  const int jj = q.fl[KF_J];
  for(int i = t; i < jj; i += kRows) ys[i] = q.y[i];
  __syncthreads();
  double e = 0.0, f = 0.0;
  if(r < s.n) {
    const cplx *Z = s.Z + z * s.sz + r;
    cplx d = mk(0.0);
#pragma unroll 4
    for(int k = 0; k < jj; ++k) d = d + Z[(size_t)k * s.ldk] * ys[k];
    cplx *xr = x + z * s.sv + r;
    const cplx v = *xr + d;
    *xr = v;
    e = norm2(d);
    f = norm2(v);
  }
  e = block_red(e, lds);
  f = block_red(f, lds);
  if(t == 0) {
    nrm_of(s, 0, z)[blockIdx.x] = e;
    nrm_of(s, 1, z)[blockIdx.x] = f;
  }
}

// A correction below the FP64 resolution of x ends the refinement: a batch's
// system at once (its cycle may have ended with steps to go: neither flag stays),
// a single one after its residual has been formed.
__global__ __launch_bounds__(kRows) void kry_tiny(KryState s, int nblk, int nb, int at_once) {
  const int z = blockIdx.x;
  const Sys q(s, z);
  if(!q.fl[KF_ACTIVE]) return;
  __shared__ double lds[4];
  const double d = sqrt(sum_norms(s.pnrm + (size_t)z * nblk, nblk, lds));
  const double x = sqrt(sum_norms(s.pnrm + ((size_t)nb + z) * nblk, nblk, lds));
  if(threadIdx.x == 0 && d <= 1e-16 * x) {
    q.fl[KF_TINY] = 1;
    if(at_once) q.fl[KF_ACTIVE] = q.fl[KF_LIVE] = 0;
  }
}

// r = b - A x (b alone without a product), and the partial norms of r and b.
__global__ __launch_bounds__(kRows) void kry_resid(KryState s, const cplx *b, const cplx *gpart, int ns, size_t sg,
                                                   int first) {
  const int z = blockIdx.y, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  if(!first && !q.fl[KF_ACTIVE]) return;
  __shared__ double lds[4];
  double e = 0.0, f = 0.0;
  if(r < s.n) {
    const cplx bv = b[z * s.sv + r];
    cplx v = bv;
    if(ns > 0) {
      const cplx *g = gpart + z * sg + r;
      cplx a = mk(0.0);
#pragma unroll 8
      for(int k = 0; k < ns; ++k) a = a + g[(size_t)k * s.n];
      v = bv - a;
    } else if(ns < 0) {  // the product is in w
      v = bv - s.w[z * s.sv + r];
    }
    s.r[z * s.sv + r] = v;
    e = norm2(v);
    f = norm2(bv);
  }
  e = block_red(e, lds);
  f = block_red(f, lds);
  if(t == 0) {
    nrm_of(s, 0, z)[blockIdx.x] = e;
    if(first) nrm_of(s, 1, z)[blockIdx.x] = f;
  }
}

// The restart's decisions, and v_0 = r / |r|.  Stops at the tolerance, at maxit
// steps, after a tiny correction, and at the FP64 floor: a cycle that did not
// halve the residual once it is within the acceptance band (<= 1e3 tol), or two
// of them (for a single system only below 1e-10: further up a slow phase of the
// restarted iteration is waited out).
__global__ __launch_bounds__(kRows) void kry_begin(KryState s, cplx *x, int first, int batch, int *host) {
  const int z = blockIdx.y, t = threadIdx.x, r = blockIdx.x * kRows + t;
  const Sys q(s, z);
  const bool lead = blockIdx.x == 0 && t == 0;
  __shared__ double lds[4];
  if(!first && !q.fl[KF_ACTIVE]) {
    if(lead) host[2 * z] = 0;
    return;
  }
  const double beta = sqrt(sum_norms(nrm_of(s, 0, z), gridDim.x, lds));
  const double bn = first ? sqrt(sum_norms(nrm_of(s, 1, z), gridDim.x, lds)) : q.sc[KS_BN];
  if(first && bn == 0.0) {  // zero right-hand side: zero solution
    if(r < s.n) x[z * s.sv + r] = mk(0.0);
  } else if(r < s.n && beta > 0.0) {
    s.V[z * s.sz + r] = (1.0 / beta) * s.r[z * s.sv + r];
  }
  if(!lead) return;
  // (a single system's NaN right-hand side: a NaN residual, which no caller accepts;
  // a batch's is left as it is)
  const double prev = first ? 0.0 : q.sc[KS_PREV], res = bn == 0.0 || (batch && !(bn > 0.0)) ? 0.0 : beta / bn;
  int stall = first ? 0 : q.fl[KF_STALL];
  const int its = first ? 0 : q.fl[KF_ITS];
  bool go = !(first && bn == 0.0) && !(res <= s.tol) && its < s.maxit && res == res;
  if(!first && q.fl[KF_TINY]) go = false;
  if(go) {
    if(prev > 0.0 && beta > 0.5 * prev && (batch || res < 1e-10)) {
      if(++stall >= 2 || res <= 1e3 * s.tol) go = false;
    } else {
      stall = 0;
    }
  }
  q.sc[KS_BN] = bn;
  q.sc[KS_PREV] = beta;
  q.sc[KS_RES] = res;
  q.g[0] = mk(beta);
  q.fl[KF_LIVE] = q.fl[KF_ACTIVE] = go ? 1 : 0;
  q.fl[KF_J] = 0;
  q.fl[KF_ITS] = its;
  q.fl[KF_STALL] = stall;
  q.fl[KF_TINY] = 0;
  host[2 * z] = go ? 1 : 0;
  host[2 * z + 1] = go && s.tol > 0.0 ? max(0, ilogb(res / (0.5 * s.tol))) : 0;
  __threadfence_system();
}

dim3 grid(const KryState &s) { return dim3((s.n + kRows - 1) / kRows, s.nb); }

}  // namespace

int kry_blocks(int n) { return (n + kRows - 1) / kRows; }

void kry_step(const KryState &s, const cplx *gpart, int ns, size_t sg, int *host, hipStream_t st) {
  hipLaunchKernelGGL(kry_dots, grid(s), dim3(kRows), 0, st, s, gpart, ns, sg);
  hipLaunchKernelGGL(kry_orth, grid(s), dim3(kRows), 0, st, s);
  hipLaunchKernelGGL(kry_orth2, grid(s), dim3(kRows), 0, st, s);
  hipLaunchKernelGGL(kry_next, grid(s), dim3(kRows), 0, st, s, host);
}
void kry_end_cycle(const KryState &s, cplx *x, bool tiny, bool batch, hipStream_t st) {
  hipLaunchKernelGGL(kry_solve_y, dim3(s.nb), dim3(kRows), 0, st, s);
  hipLaunchKernelGGL(kry_update, grid(s), dim3(kRows), 0, st, s, x);
  if(tiny) hipLaunchKernelGGL(kry_tiny, dim3(s.nb), dim3(kRows), 0, st, s, kry_blocks(s.n), s.nb, batch ? 1 : 0);
}
void kry_restart(const KryState &s, const cplx *b, cplx *x, const cplx *gpart, int ns, size_t sg, bool first,
                 bool batch, int *host, hipStream_t st) {
  hipLaunchKernelGGL(kry_resid, grid(s), dim3(kRows), 0, st, s, b, gpart, ns, sg, first ? 1 : 0);
  hipLaunchKernelGGL(kry_begin, grid(s), dim3(kRows), 0, st, s, x, first ? 1 : 0, batch ? 1 : 0, host);
}

}  // namespace omx
