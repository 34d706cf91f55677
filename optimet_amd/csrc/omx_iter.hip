// omx_iter.hip -- level-1 kernels: conversions, padding, norms and the
// element-wise unpreconditioning steps (Solver.cpp:57-116).
#include <type_traits>

#include "omx_kernels.hpp"

namespace omx {

// y[i] = x[i] * ov[kind][obj][pol][deg(i)] - sub[i], over the N = 2 nf P unknowns
// of system blockIdx.z
__global__ void vmul_ov_k(cplx *y, const cplx *x, const cplx *ov, int kind, int P, int nmax, const cplx *sub,
                          int n, size_t zvec, size_t zov) {
  y += blockIdx.z * zvec;
  x += blockIdx.z * zvec;
  ov += blockIdx.z * zov;
  if(sub) sub += blockIdx.z * zvec;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  const int nf = nmax * (nmax + 2);
  int obj = i / (2 * nf), r = i % (2 * nf);
  int pol = r >= nf, q = r % nf, deg, m;
  unflat(q, deg, m);
  cplx v = x[i] * ov[(((size_t)kind * P + obj) * 2 + pol) * (nmax + 1) + deg];
  if(sub) v = v - sub[i];
  y[i] = v;
}

constexpr int kRedBlocks = 128;
__global__ __launch_bounds__(256) void nrm2_k(const cplx *x, int n, double *part) {
  __shared__ double red[256];
  double s = 0.0;
  for(int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) s += norm2(x[i]);
  red[threadIdx.x] = s;
  __syncthreads();
  for(int st = 128; st > 0; st >>= 1) {
    if(threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if(threadIdx.x == 0) part[blockIdx.x] = red[0];
}
__global__ void nrm2_reduce_k(const double *part, int nb, double *out) {
  __shared__ double red[128];
  double s = 0.0;
  for(int b = threadIdx.x; b < nb; b += 128) s += part[b];
  red[threadIdx.x] = s;
  __syncthreads();
  for(int st = 64; st > 0; st >>= 1) {
    if(threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if(threadIdx.x == 0) *out = red[0];
}

static inline dim3 g1(int n) { return dim3((n + 255) / 256); }

// y = (complex float) x over n elements (grid-stride: n may exceed 2^31)
__global__ void demote_k(float2 *y, const cplx *x, size_t n) {
  for(size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    y[i] = make_float2((float)x[i].x, (float)x[i].y);
}
void demote(float2 *y, const cplx *x, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(demote_k, dim3(4096), dim3(256), 0, st, y, x, n);
}
__global__ void zero_ints_k(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = 0;
}
void zero_ints(int *p, int n, hipStream_t st) { hipLaunchKernelGGL(zero_ints_k, g1(n), dim3(256), 0, st, p, n); }

// dst (Nd x Nd, column-major) = src (Ns x Ns, leading dimension Ns) bordered
// by the identity (grid-stride: Nd^2 may exceed 2^31)
template <typename D>
__global__ void pad_matrix_k(D *dst, int Nd, const cplx *src, int Ns) {
  const size_t n = (size_t)Nd * Nd;
  for(size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const int j = (int)(e / Nd), i = (int)(e % Nd);
    const cplx v = (i < Ns && j < Ns) ? src[(size_t)j * Ns + i] : mk(i == j ? 1.0 : 0.0);
    if constexpr(std::is_same<D, cplx>::value)
      dst[e] = v;
    else
      dst[e] = make_float2((float)v.x, (float)v.y);
  }
}
void pad_matrix64(cplx *dst, int Nd, const cplx *src, int Ns, hipStream_t st) {
  hipLaunchKernelGGL(pad_matrix_k<cplx>, dim3(4096), dim3(256), 0, st, dst, Nd, src, Ns);
}
void pad_matrix32(float2 *dst, int Nd, const cplx *src, int Ns, hipStream_t st) {
  hipLaunchKernelGGL(pad_matrix_k<float2>, dim3(4096), dim3(256), 0, st, dst, Nd, src, Ns);
}
// dst[0, Nd) = src[0, Ns) followed by zeros
__global__ void pad_vector_k(cplx *dst, int Nd, const cplx *src, int Ns) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < Nd) dst[i] = i < Ns ? src[i] : mk(0.0);
}
void pad_vector(cplx *dst, int Nd, const cplx *src, int Ns, hipStream_t st) {
  hipLaunchKernelGGL(pad_vector_k, g1(Nd), dim3(256), 0, st, dst, Nd, src, Ns);
}
void vmul_ov(cplx *y, const cplx *x, const cplx *ov, int kind, int P, int nmax, const cplx *sub, int n,
             hipStream_t st, int nb, size_t zvec, size_t zov) {
  hipLaunchKernelGGL(vmul_ov_k, dim3((n + 255) / 256, 1, nb), dim3(256), 0, st, y, x, ov, kind, P, nmax, sub, n, zvec,
                     zov);
}
void nrm2sq(const cplx *x, int n, double *part, double *out, hipStream_t st) {
  int nb = std::min(kRedBlocks, (n + 255) / 256);
  hipLaunchKernelGGL(nrm2_k, dim3(nb), dim3(256), 0, st, x, n, part);
  hipLaunchKernelGGL(nrm2_reduce_k, dim3(1), dim3(128), 0, st, part, nb, out);
}

}  // namespace omx
