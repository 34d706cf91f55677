// omx_aca.hip -- adaptive cross approximation of the coupling blocks and the
// compressed matrix-vector product.
//
//   aca_kernel       ACA_compression (PreconditionedMatrix.cpp:763-862) with
//                    getMaxInd (:864-889): one workgroup per admissible block
//   aca_pack_kernel  the factors of each block, U (n x r) then V (r x n),
//                    copied from the n x n staging slots into a packed pool
//   aca_vt_kernel    t_b = V_b x_j for every compressed block b = (i, j)
//   aca_rows_kernel  partial y_i over a group of block row i's blocks:
//                    dense S_ij x_j or U_b t_b (matvec, :1058-1085)
//   aca_sum_kernel   y = x + sum of the partials (the identity diagonal blocks)
#include "omx_kernels.hpp"

namespace omx {

namespace {

__device__ inline double wave_sum(double v) {
  for(int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Largest value, first index on ties (getMaxInd keeps the first strict maximum).
__device__ inline void wave_argmax(double &v, int &i) {
  for(int o = 32; o > 0; o >>= 1) {
    double ov = __shfl_xor(v, o);
    int oi = __shfl_xor(i, o);
    if(ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
}

}  // namespace

// One wave per block; lane l owns rows / columns l + 64 g, g < R (n <= 64 R <=
// 256).  Step k: the residual row I_k against the k terms so far, its
// largest unused entry J_k, v_k = row / pivot, the residual column J_k -> u_k,
// the reference's norm estimate (the cross terms over p <= k-2 and the first
// k entries, unconjugated, :826-843) and its stopping test for k >= 1, then
// I_{k+1} = largest unused entry of u_k.  A residual row or column with no
// non-zero candidate ends the iteration with the terms so far (they reproduce
// the block exactly).
//
// Bound: the latency of a step's dependent reads, so by the blocks in flight.
// With 256 threads a block, most of them idle at n = 70, and eight barriers a
// step: 7.9 ms for the 90 000 blocks of 300 spheres; now 4.4 ms.
template <int R> __global__ __launch_bounds__(64, R < 3 ? 4 : 2) void aca_kernel(AcaArgs a) {
  const int b = blockIdx.x, lane = threadIdx.x, n = a.n;
  const cplx *A = a.A + (size_t)b * n * n;
  cplx *U = a.U + (size_t)b * n * n, *V = a.V + (size_t)b * n * n;
  __shared__ cplx coef[64 * R], uk[64 * R], vk[64 * R];
  bool usedR[R], usedC[R];
#pragma unroll
  for(int g = 0; g < R; ++g) usedR[g] = usedC[g] = lane + 64 * g >= n;
  // index of the largest |x| not used (the first on ties), -1 when all are zero
  auto argmax = [&](const cplx(&x)[R], const bool(&used)[R]) {
    double v = -1.0;
    int i = lane;
#pragma unroll
    for(int g = 0; g < R; ++g) {
      const double m = used[g] ? -1.0 : cabs(x[g]);
      if(m > v) {
        v = m;
        i = lane + 64 * g;
      }
    }
    wave_argmax(v, i);
    return v > 0.0 ? i : -1;
  };
  double norma = 0.0;
  int ik = 0, r = 0;
  for(int k = 0; k < n; ++k) {
#pragma unroll
    for(int g = 0; g < R; ++g) usedR[g] = usedR[g] || lane + 64 * g == ik;
    for(int p = lane; p < k; p += 64) coef[p] = U[(size_t)p * n + ik];  // U(I_k, p)
    __syncthreads();
    cplx rv[R], u[R];
#pragma unroll
    for(int g = 0; g < R; ++g) {
      const int t = lane + 64 * g;
      rv[g] = mk(0.0);
      if(t < n) {
        const cplx e = A[(size_t)t * n + ik];
        cplx s = mk(0.0);
#pragma unroll 4
        for(int p = 0; p < k; ++p) s = s + coef[p] * V[(size_t)p * n + t];
        rv[g] = e - s;
      }
    }
    const int jk = argmax(rv, usedC);
    if(jk < 0) break;
    cplx piv = mk(0.0);
#pragma unroll
    for(int g = 0; g < R; ++g) {
      if(jk >> 6 == g) piv = cplx{__shfl(rv[g].x, jk & 63, 64), __shfl(rv[g].y, jk & 63, 64)};
      usedC[g] = usedC[g] || lane + 64 * g == jk;
    }
    double sv[R], su[R];
    __syncthreads();
#pragma unroll
    for(int g = 0; g < R; ++g) {
      const int t = lane + 64 * g;
      cplx v = mk(0.0);
      if(t < n) {
        v = rv[g] / piv;
        V[(size_t)k * n + t] = v;
        vk[t] = v;
      }
      sv[g] = norm2(v);
    }
    for(int p = lane; p < k; p += 64) coef[p] = V[(size_t)p * n + jk];  // V(p, J_k)
    __syncthreads();
#pragma unroll
    for(int g = 0; g < R; ++g) {
      const int t = lane + 64 * g;
      u[g] = mk(0.0);
      if(t < n) {
        const cplx e = A[(size_t)jk * n + t];
        cplx s = mk(0.0);
#pragma unroll 4
        for(int p = 0; p < k; ++p) s = s + coef[p] * U[(size_t)p * n + t];
        u[g] = e - s;
        U[(size_t)k * n + t] = u[g];
        uk[t] = u[g];
      }
      su[g] = norm2(u[g]);
    }
    __syncthreads();
    double SU = 0.0, SV = 0.0, CR = 0.0;
#pragma unroll
    for(int g = 0; g < R; ++g) {
      const int t = lane + 64 * g;
      double cross = 0.0;
      if(t < k - 1) {  // p = t
        cplx p1 = mk(0.0), p2 = mk(0.0);
#pragma unroll 4
        for(int q = 0; q < k; ++q) {
          p1 = p1 + U[(size_t)t * n + q] * uk[q];
          p2 = p2 + V[(size_t)t * n + q] * vk[q];
        }
        cross = cabs(p1) * cabs(p2);
      }
      SU += wave_sum(su[g]);
      SV += wave_sum(sv[g]);
      if(64 * g < k - 1) CR += wave_sum(cross);
    }
    const double cn = sqrt(SU), rn = sqrt(SV);
    bool stop = false;
    if(k == 0) {
      norma = cn * cn * (rn * rn);
    } else {
      norma = norma + cn * cn * (rn * rn) + 2.0 * CR;
      stop = a.eps * sqrt(norma) >= cn * rn;
    }
    r = k + 1;
    if(stop) break;
    const int in = argmax(u, usedR);
    if(in < 0) break;
    ik = in;
    __syncthreads();
  }
  if(lane == 0) a.rank[b] = r;
}

__global__ void aca_pack_kernel(const cplx *U, const cplx *V, int n, const int *rank, cplx *pool, const size_t *off) {
  const int b = blockIdx.x;
  const size_t m = (size_t)n * rank[b];
  const cplx *u = U + (size_t)b * n * n, *v = V + (size_t)b * n * n;
  cplx *d = pool + off[b];
  for(size_t e = threadIdx.x; e < m; e += blockDim.x) {
    d[e] = u[e];
    d[m + e] = v[e];
  }
}

// A wave per compressed block: four rows of V at a time, 16 lanes each, x_j in NI
// registers a lane (n <= 16 NI).  With a row per wave and all 64 lanes on it (n =
// 70: a second pass of 6) the reductions bound it: 282 us a product for the 0.92
// GB of V of 300 spheres, now 178 us (5.2 TB/s; a loop over blocks in six
// workgroups a CU, each with the next descriptor on its way: 201).
template <int NI> __global__ __launch_bounds__(256) void aca_vt_kernel(AcaOp op, const cplx *x) {
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if(e >= op.naca) return;
  const AcaDesc d = op.desc[op.acalist[e]];
  const int n = op.n, r = d.rank, lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
  cplx xs[NI];
#pragma unroll
  for(int i = 0; i < NI; ++i) {
    xs[i] = mk(0.0);
    if(li + 16 * i < n) xs[i] = x[(size_t)d.j * n + li + 16 * i];
  }
  const cplx *Vb = d.M + (size_t)n * r;
  // H fours of rows at once, their loads first
  constexpr int H = NI < 10 ? 2 : 1;
  for(int p0 = 0; p0 < r; p0 += 4 * H) {
    cplx v[H][NI];
#pragma unroll
    for(int h = 0; h < H; ++h)
#pragma unroll
      for(int i = 0; i < NI; ++i) {
        const int p = p0 + 4 * h + g;
        v[h][i] = mk(0.0);
        if(p < r && li + 16 * i < n) v[h][i] = Vb[(size_t)p * n + li + 16 * i];
      }
#pragma unroll
    for(int h = 0; h < H; ++h) {
      const int p = p0 + 4 * h + g;
      cplx s = mk(0.0);
#pragma unroll
      for(int i = 0; i < NI; ++i) s = s + v[h][i] * xs[i];
#pragma unroll
      for(int o = 8; o > 0; o >>= 1) {
        s.x += __shfl_xor(s.x, o, 64);
        s.y += __shfl_xor(s.y, o, 64);
      }
      if(p < r && li == 0) op.t[d.toff + p] = s;
    }
  }
}

// The group's blocks of a block row, dealt to the four waves: four columns at a
// time, 16 lanes each, the rows' sums in NI registers a lane throughout; the
// column groups' and the waves' sums meet at the end.  With a thread a row (n =
// 70: a second wave of 6) and the right operand staged between barriers for every
// block: 184 us a product, now 177 us (5.3 TB/s).
template <int NI> __global__ __launch_bounds__(256) void aca_rows_kernel(AcaOp op, const cplx *x) {
  const int gr = blockIdx.x, i0 = blockIdx.y, n = op.n, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, li = lane & 15;
  __shared__ cplx sum[3][16 * NI];
  cplx acc[NI];
#pragma unroll
  for(int i = 0; i < NI; ++i) acc[i] = mk(0.0);
  const int end = op.rowptr[i0 + 1], step = op.G * 4;
  int e = op.rowptr[i0] + gr + op.G * w;
  AcaDesc nx{};
  if(e < end) nx = op.desc[e];
  for(; e < end; e += step) {
    const AcaDesc d = nx;
    if(e + step < end) nx = op.desc[e + step];
    const int m = d.rank < 0 ? n : d.rank;
    const cplx *src = d.rank < 0 ? x + (size_t)d.j * n : op.t + d.toff;
    constexpr int H = NI < 10 ? 2 : 1;
    for(int c0 = 0; c0 < m; c0 += 4 * H) {
      cplx v[H][NI], b[H];
#pragma unroll
      for(int h = 0; h < H; ++h) {
        const int c = c0 + 4 * h + g;
        b[h] = mk(0.0);
        if(c < m) b[h] = src[c];
#pragma unroll
        for(int i = 0; i < NI; ++i) {
          v[h][i] = mk(0.0);
          if(c < m && li + 16 * i < n) v[h][i] = d.M[(size_t)c * n + li + 16 * i];
        }
      }
#pragma unroll
      for(int h = 0; h < H; ++h)
#pragma unroll
        for(int i = 0; i < NI; ++i) acc[i] = acc[i] + v[h][i] * b[h];
    }
  }
#pragma unroll
  for(int i = 0; i < NI; ++i) {
#pragma unroll
    for(int o = 32; o >= 16; o >>= 1) {
      acc[i].x += __shfl_xor(acc[i].x, o, 64);
      acc[i].y += __shfl_xor(acc[i].y, o, 64);
    }
    if(w > 0 && g == 0) sum[w - 1][li + 16 * i] = acc[i];
  }
  __syncthreads();
  if(w == 0 && g == 0)
#pragma unroll
    for(int i = 0; i < NI; ++i)
      if(li + 16 * i < n) {
        const int q = li + 16 * i;
        op.part[((size_t)gr * op.P + i0) * n + q] = ((acc[i] + sum[0][q]) + sum[1][q]) + sum[2][q];
      }
}

__global__ void aca_sum_kernel(AcaOp op, const cplx *x, cplx *y) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(e >= (size_t)op.Np) return;
  cplx s = x[e];
  if(e < (size_t)op.N) {
    const size_t i = e / op.n, q = e % op.n;
    for(int g = 0; g < op.G; ++g) s = s + op.part[((size_t)g * op.P + i) * op.n + q];
  }
  y[e] = s;
}

void run_aca(const AcaArgs &a, hipStream_t st) {
  switch((a.n + 63) / 64) {
  case 1: hipLaunchKernelGGL(aca_kernel<1>, dim3(a.nblk), dim3(64), 0, st, a); break;
  case 2: hipLaunchKernelGGL(aca_kernel<2>, dim3(a.nblk), dim3(64), 0, st, a); break;
  case 3: hipLaunchKernelGGL(aca_kernel<3>, dim3(a.nblk), dim3(64), 0, st, a); break;
  default: hipLaunchKernelGGL(aca_kernel<4>, dim3(a.nblk), dim3(64), 0, st, a); break;
  }
}

void run_aca_pack(const cplx *U, const cplx *V, int n, int nblk, const int *rank, cplx *pool, const size_t *off,
                  hipStream_t st) {
  hipLaunchKernelGGL(aca_pack_kernel, dim3(nblk), dim3(256), 0, st, U, V, n, rank, pool, off);
}

// The kernels of the smallest NI with n <= 16 NI, of the register counts that
// n = 2 nmax (nmax + 2) = 6 16 30 48 70 96 126 160 198 240 come to.
template <int NI> void run_products(const AcaOp &op, const cplx *x, hipStream_t st) {
  constexpr int next = NI < 3 ? NI + 1 : NI == 3 ? 5 : NI == 5 ? 6 : NI < 10 ? NI + 2 : NI == 10 ? 13 : 16;
  if constexpr(NI < 16)
    if(op.n > 16 * NI) return run_products<next>(op, x, st);
  if(op.naca > 0) hipLaunchKernelGGL(aca_vt_kernel<NI>, dim3((op.naca + 3) / 4), dim3(256), 0, st, op, x);
  if(op.G > 0) hipLaunchKernelGGL(aca_rows_kernel<NI>, dim3(op.G, op.P), dim3(256), 0, st, op, x);
}

void aca_matvec(const AcaOp &op, const cplx *x, cplx *y, hipStream_t st) {
  run_products<1>(op, x, st);
  hipLaunchKernelGGL(aca_sum_kernel, dim3((op.Np + 255) / 256), dim3(256), 0, st, op, x, y);
}

}  // namespace omx
