// omx_fields.hip -- field maps: E and H at omega and 2 omega at given points
// (Result::getEHFields, Result.cpp:74-301, with Result::setFields, :797-933).
//
//   fields_owner    the first sphere that holds each point (Geometry::checkInner,
//                   Geometry.cpp:147-163), or P outside all of them
//   fields_outside  partial sums of the scattered and incident waves at the
//                   outside points: one wave per (64 points, objects)
//   fields_sum      the partial sums added in a fixed order, with their factors
//   fields_inside   one workgroup per inside point: internal waves and the SH
//                   bulk term (Geometry::COEFFpartSH, symbol::CXm1 / CXp1)
//
// The vector spherical waves are those of AuxCoefficients
// (AuxCoefficients.cpp:30-343): Wigner functions W, dW by the reference's
// recurrence, its 1e-6 shift of the polar angle on the z axis included.
// Negative orders come from the positive ones, W_n^{-m} = (-1)^m W_n^m and
// likewise dW; on the axis the reference shifts pi - theta for m < 0 the same
// way, across the pole, which turns the sign of dW_n^{-m} around.
//
// Bound: FP64 VALU.  A point and object pair costs about 25 FP64 operations per
// harmonic and frequency; 24 objects at nmax 6 and 6561 points are 0.4 G of
// them, about 10 us at the FP64 rate.  A lane is a point and a wave walks the
// objects, so every lane works, the expansion coefficients are wave-uniform
// (scalar loads) and the sum over objects stays in registers; objects are
// also split over workgroups where the points alone do not fill the device.
// Measured at that size (nmax 6, 81 x 81 points, second harmonic): 0.19 ms for
// the four kernels, against 9.6 ms for one workgroup per point with a thread
// per object (25 of 256 threads at work, radial and Wigner tables in scratch).
#include <algorithm>

#include "omx_kernels.hpp"

namespace omx {

namespace {

__device__ inline void to_cart(double st, double ct, double sp, double cp, const cplx v[3], cplx out[3]) {
  // Tools::toProjection
  out[0] = st * cp * v[0] + ct * cp * v[1] - sp * v[2];
  out[1] = st * sp * v[0] + ct * sp * v[1] + cp * v[2];
  out[2] = ct * v[0] - st * v[1];
}
__device__ inline void to_sph(double x, double y, double z, double &r, double &t, double &p) {
  // Tools::toSpherical
  r = sqrt(x * x + y * y + z * z);
  t = r > 0.0 ? acos(z / r) : 0.0;
  p = r > 0.0 ? atan2(y, x) : 0.0;
}
__device__ inline bool on_axis(double the) { return (fabs(the) < 1e-10) || (fabs(the) - kPi + 1e-10 > 0.0); }

// Constants of the Wigner recurrence, in LDS: rt = sqrt(n^2 - m^2), ri its
// reciprocal, i2 = 1 / (2n + 1), dn the harmonics' normalisation, sq =
// sqrt((2n - 1) / 2n) (the step of W_n^n).
template <int NMAX> struct FieldTab {
  static constexpr int S = NMAX + 1;
  double rt[(NMAX + 2) * S], ri[(NMAX + 2) * S], i2[NMAX + 2], dn[NMAX + 2], sq[NMAX + 2];
  __device__ void fill() {
    for(int e = threadIdx.x; e < (NMAX + 2) * S; e += blockDim.x) {
      const int n = e / S, m = e % S;
      const double v = n > m ? sqrt((double)(n * n - m * m)) : 0.0;
      rt[e] = v;
      ri[e] = n > m ? 1.0 / v : 0.0;
    }
    for(int n = threadIdx.x; n < NMAX + 2; n += blockDim.x) {
      i2[n] = 1.0 / (2 * n + 1);
      dn[n] = n ? sqrt((2.0 * n + 1.0) / (4.0 * kPi * (n * (n + 1)))) : 0.0;
      sq[n] = n ? sqrt((2.0 * n - 1.0) / (2.0 * n)) : 1.0;
    }
  }
};

// Radial functions of one expansion, taken at n = 1, 2, ..: z_n and z_n'.  One
// type for both kinds, so that the harmonic sums exist once in the kernel.
struct Radial {
  cplx iz, f, g;  // 1 / z; h_n^(1), h_{n+1}^(1), upward
  const cplx *v;  // regular (non-null): j_0 .. j_{nmax+1} in memory
  __device__ Radial(cplx z, const cplx *vals) : v(vals) {
    iz = mk(1.0) / z;
    f = g = mk(0.0);
    if(v || hypot(z.x, z.y) <= kErrEps) return;
    const cplx eiz = cexp_(mk(-z.y, z.x));
    const cplx f0 = mk(0.0, -1.0) * eiz * iz;
    f = -(eiz * (z + mk(0.0, 1.0))) * (iz * iz);
    g = (3.0 * f) * iz - f0;
  }
  __device__ void at(int n, cplx &z, cplx &d) {
    if(v) {
      f = v[n];
      g = v[n + 1];
    }
    z = f;
    d = ((double)n * f) * iz - g;
    const cplx h = ((2.0 * n + 3.0) * g) * iz - f;
    f = g;
    g = h;
  }
};

// Sums over the harmonics of one expansion about a centre at this lane's point
// (Rr, Rt, Rp) relative to it: sE = sum M_p a_p + N_p b_p, sH = sum N_p a_p +
// M_p b_p, Cartesian; a and b wave-uniform.  Degree by degree: the angular
// sums over m in registers (one pair +-m at a time), then the radial factors.
template <int NMAX>
__device__ __forceinline__ void expansion(const FieldTab<NMAX> &tb, double Rt, double Rp, cplx Kr, Radial rad,
                                          const cplx *__restrict__ a, const cplx *__restrict__ b, cplx sE[3],
                                          cplx sH[3]) {
  constexpr int S = NMAX + 1;
  const bool axis = on_axis(Rt);
  const double vig = axis ? Rt + 1e-6 : Rt;
  const double x = cos(vig), isv = 1.0 / sin(vig), s1 = sqrt((1.0 - x) * (1.0 + x));
  double st, ct, sp, cp;
  sincos(Rt, &st, &ct);
  sincos(Rp, &sp, &cp);
  const double ia = axis ? 1.0 / ct : 1.0 / st;  // A = m dW / cos on the axis, m W / sin off it
  const double sg = axis ? -1.0 : 1.0;
  cplx e[S];  // exp(i m phi)
  e[0] = mk(1.0);
#pragma unroll
  for(int m = 1; m <= NMAX; ++m) e[m] = e[m - 1] * mk(cp, sp);
  double Wp[S], W[S], Wn[S];  // degrees n - 1, n, n + 1
#pragma unroll
  for(int m = 0; m <= NMAX; ++m) Wp[m] = W[m] = Wn[m] = 0.0;
  double wmm = s1 * tb.sq[1];
  Wp[0] = 1.0;
  W[0] = x;
  if(NMAX >= 1) W[1] = wmm;
  const cplx iKr = mk(1.0) / Kr;
  cplx e3[3] = {mk(0.0), mk(0.0), mk(0.0)}, h3[3] = {mk(0.0), mk(0.0), mk(0.0)};
#pragma unroll 1
  for(int n = 1; n <= NMAX; ++n) {
    const double *r0 = tb.rt + n * S, *r1 = r0 + S, *q1 = tb.ri + (n + 1) * S;
    const double tn = (2.0 * n + 1.0) * x, fn = n * tb.i2[n] * isv, gn = (n + 1) * tb.i2[n] * isv;
    wmm = wmm * s1 * tb.sq[n + 1];
    cplx wa = mk(0.0), wb = mk(0.0), da = mk(0.0), db = mk(0.0), aa = mk(0.0), ab = mk(0.0);
    const int p0 = n * (n + 1) - 1;
#pragma unroll
    for(int m = 0; m <= NMAX; ++m) {
      if(m > n) continue;
      Wn[m] = (tn * W[m] - r0[m] * Wp[m]) * q1[m];
      const double dW = r1[m] * Wn[m] * fn - r0[m] * Wp[m] * gn;
      if(m == 0) {
        const cplx ua = a[p0], ub = b[p0];
        wa = wa + W[0] * ua;
        wb = wb + W[0] * ub;
        da = da + dW * ua;
        db = db + dW * ub;
        continue;
      }
      const double A = m * ia * (axis ? dW : W[m]);
      // (-1)^m exp(i m phi) {a, b}_m and exp(-i m phi) {a, b}_{-m}
      const cplx ep = (m & 1) ? -e[m] : e[m], em = conj(e[m]);
      const cplx pa = ep * a[p0 - m], pb = ep * b[p0 - m], ma = em * a[p0 + m], mb = em * b[p0 + m];
      wa = wa + W[m] * (pa + ma);
      wb = wb + W[m] * (pb + mb);
      da = da + dW * (pa + sg * ma);
      db = db + dW * (pb + sg * mb);
      aa = aa + A * (pa - sg * ma);
      ab = ab + A * (pb - sg * mb);
    }
    cplx z, d;
    rad.at(n, z, d);
    const double dn = tb.dn[n];
    const cplx zt = dn * z, izt = mk(-zt.y, zt.x);
    const cplx zz = (iKr * dn) * (Kr * d + z), izz = mk(-zz.y, zz.x);
    const cplx zr = (iKr * (dn * (n * (n + 1)))) * z;
    e3[0] = e3[0] + zr * wb;
    e3[1] = e3[1] + izt * aa + zz * db;
    e3[2] = e3[2] + izz * ab - zt * da;
    h3[0] = h3[0] + zr * wa;
    h3[1] = h3[1] + zz * da + izt * ab;
    h3[2] = h3[2] + izz * aa - zt * db;
#pragma unroll
    for(int m = 0; m <= NMAX; ++m) {
      Wp[m] = W[m];
      W[m] = m == n + 1 ? wmm : Wn[m];
    }
  }
  to_cart(st, ct, sp, cp, e3, sE);
  to_cart(st, ct, sp, cp, h3, sH);
}

__global__ __launch_bounds__(256) void fields_owner(FieldArgs a) {
#pragma clang fp contract(off)
  const int ip = blockIdx.x * blockDim.x + threadIdx.x;
  if(ip >= a.npts) return;
  const double px = a.pts[3 * ip], py = a.pts[3 * ip + 1], pz = a.pts[3 * ip + 2];
  int in = a.P;
  for(int j = 0; j < a.P; ++j) {
    const double dx = px - a.xyz[3 * j], dy = py - a.xyz[3 * j + 1], dz = pz - a.xyz[3 * j + 2];
    if(sqrt(dx * dx + dy * dy + dz * dz) <= a.radius[j]) {
      in = j;
      break;
    }
  }
  a.owner[ip] = in;
}

// Grid (tiles of 64 points, slices, frequencies); wave w of slice s takes the
// tasks 4 s + w, 4 s + w + 4 slices, ..: objects 0 .. P-1 and, at omega, the
// incident wave as task P.  part[z][slice][6][npts].
template <int NMAX>
__global__ __launch_bounds__(256, 2) void fields_outside(FieldArgs a) {
  __shared__ FieldTab<NMAX> tb;
  __shared__ cplx jv[64 * (NMAX + 2)];  // j_n of the one wave that takes the incident task
  __shared__ cplx red[3][6][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ns = gridDim.y, sl = blockIdx.y, fz = blockIdx.z, nf = NMAX * (NMAX + 2);
  tb.fill();
  __syncthreads();
  const int ip = blockIdx.x * 64 + lane;
  const bool out = ip < a.npts && a.owner[ip] == a.P;
  const cplx k = fz ? 2.0 * a.waveK : a.waveK;
  const cplx *x = fz ? a.xsh : a.x;
  const int ntask = a.P + (fz ? 0 : 1);
  cplx acc[6];
#pragma unroll
  for(int c = 0; c < 6; ++c) acc[c] = mk(0.0);
  if(out) {
    const double px = a.pts[3 * ip], py = a.pts[3 * ip + 1], pz = a.pts[3 * ip + 2];
#pragma unroll 1
    for(int task = 4 * sl + w; task < ntask; task += 4 * ns) {
      double Rr, Rt, Rp;
      cplx sE[3], sH[3];
      const bool inc = task == a.P;  // the incident wave about the origin
      double cx = 0.0, cy = 0.0, cz = 0.0;
      const cplx *co = a.inc;
      if(!inc) {
        cx = a.xyz[3 * task];
        cy = a.xyz[3 * task + 1];
        cz = a.xyz[3 * task + 2];
        co = x + (size_t)task * 2 * nf;
      }
      to_sph(px - cx, py - cy, pz - cz, Rr, Rt, Rp);
      cplx *jl = jv + lane * (NMAX + 2);
      if(inc) sph_values_to(0, Rr * k, NMAX + 2, jl);
      expansion<NMAX>(tb, Rt, Rp, Rr * k, Radial(Rr * k, inc ? jl : nullptr), co, co + nf, sE, sH);
#pragma unroll
      for(int c = 0; c < 3; ++c) {
        acc[c] = acc[c] + sE[c];
        acc[3 + c] = acc[3 + c] + sH[c];
      }
    }
  }
  if(w > 0) {
#pragma unroll
    for(int c = 0; c < 6; ++c) red[w - 1][c][lane] = acc[c];
  }
  __syncthreads();
  if(w == 0 && out) {
#pragma unroll
    for(int c = 0; c < 6; ++c)
      a.part[(((size_t)fz * ns + sl) * 6 + c) * a.npts + ip] =
          acc[c] + red[0][c][lane] + red[1][c][lane] + red[2][c][lane];
  }
}

__global__ __launch_bounds__(256) void fields_sum(FieldArgs a, int ns) {
  const int ip = blockIdx.x * blockDim.x + threadIdx.x, fz = blockIdx.y;
  if(ip >= a.npts || a.owner[ip] != a.P) return;
  const cplx k0 = mk(a.omega * sqrt(kEps0 * kMu0)), iZ = mk(0.0, -1.0) / csqrt_(a.bg_mu / a.bg_eps);
  for(int c = 0; c < 6; ++c) {
    cplx s = mk(0.0);
    for(int q = 0; q < ns; ++q) s = s + a.part[(((size_t)fz * ns + q) * 6 + c) * a.npts + ip];
    const int o = 3 * ip + c % 3;
    if(fz == 0) {
      if(c < 3) a.E[o] = s; else a.H[o] = s * iZ;
    } else {
      if(c < 3) a.Esh[o] = s * k0; else a.Hsh[o] = s * (iZ * k0);
    }
  }
}

__device__ inline cplx wave_total(cplx v) {
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_xor(v.x, o, 64);
    v.y += __shfl_xor(v.y, o, 64);
  }
  return v;
}

// One workgroup per point inside a sphere.  Waves 0-1 take the harmonics of
// the internal wave at omega, waves 2-3 those at 2 omega; then all threads
// share the bilinear sums of the bulk term, output harmonic kk = t % nf, over
// the (n1, n2) factors of the radius tabulated once in LDS (the products of
// radial functions of symbol::CXm1 / CXp1, Symbol.cpp:474-655); only the table
// entries with M1 + M2 = M are visited (all others vanish).
template <int NMAX>
__global__ __launch_bounds__(256) void fields_inside(FieldArgs a) {
  constexpr int S = NMAX + 1, NF = NMAX * (NMAX + 2);
  const int ip = blockIdx.x, j = a.owner[ip];
  if(j == a.P) return;
  __shared__ cplx jw[NMAX + 2], js[NMAX + 2], f[NMAX + 2], d[NMAX + 2], d2[NMAX + 2], em[S];
  __shared__ double Wt[S * S], dWt[S * S], At[S * S];
  __shared__ cplx cs[NF], ds[NF];
  __shared__ cplx tab[6][NMAX * NMAX];
  __shared__ cplx red[2][256];
  __shared__ cplx wsum[4][6];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  double Rr, Rt, Rp;
  to_sph(a.pts[3 * ip] - a.xyz[3 * j], a.pts[3 * ip + 1] - a.xyz[3 * j + 1], a.pts[3 * ip + 2] - a.xyz[3 * j + 2], Rr,
         Rt, Rp);
  const bool axis = on_axis(Rt);
  const cplx k0 = mk(a.omega * sqrt(kEps0 * kMu0));
  const cplx ki = k0 * csqrt_((a.eps[j] / mk(kEps0)) * (a.mu[j] / mk(kMu0)));
  const cplx ksh = (2.0 * k0) * csqrt_((a.eps_sh[j] / mk(kEps0)) * (a.mu[j] / mk(kMu0)));
  const cplx kj = a.omega * csqrt_(a.eps[j] * a.mu[j]);
  if(t == 0) sph_values_to(0, Rr * ki, NMAX + 2, jw);
  if(t == 64 && a.sh) sph_values_to(0, Rr * ksh, NMAX + 2, js);
  if(t == 128 && a.sh) sph_values_to(0, Rr * kj, NMAX + 2, f);
  if(t >= 192 && t < 192 + S) {  // Wigner functions of order m at every degree
    const int m = t - 192;
    const double vig = axis ? Rt + 1e-6 : Rt, x = cos(vig), sv = sin(vig);
    const double ia = axis ? 1.0 / cos(Rt) : 1.0 / sin(Rt);
    const double s1 = sqrt((1.0 - x) * (1.0 + x));
    double W = 1.0, Wp = 0.0;
    for(int i = 1; i <= m; ++i) W = W * s1 * sqrt((2.0 * i - 1.0) / (2.0 * i));
    for(int n = m; n <= NMAX; ++n) {
      const double r0 = sqrt((double)(n * n - m * m)), r1 = sqrt((double)((n + 1) * (n + 1) - m * m));
      const double Wn = ((2.0 * n + 1.0) * x * W - r0 * Wp) / r1;
      const double dW = (n * r1 * Wn - (n + 1) * r0 * Wp) / ((2.0 * n + 1.0) * sv);
      Wt[n * S + m] = W;
      dWt[n * S + m] = dW;
      At[n * S + m] = m == 0 ? 0.0 : m * ia * (axis ? dW : W);
      Wp = W;
      W = Wn;
    }
    em[m] = mk(cos(m * Rp), sin(m * Rp));
  }
  if(a.sh)
    for(int p = t; p < NF; p += 256) {
      cs[p] = a.xint[(size_t)j * 2 * NF + p];
      ds[p] = a.xint[(size_t)j * 2 * NF + NF + p];
    }
  __syncthreads();
  // the angular functions of harmonic (n, m), any sign of m, with the factor
  // (-1)^m exp(i m phi)
  auto angular = [&](int n, int m, double &W, double &dW, double &A, cplx &e) {
    const int am = abs(m), i = n * S + am;
    const double o = (am & 1) ? -1.0 : 1.0, sg = axis ? -1.0 : 1.0;
    W = Wt[i];
    dW = dWt[i];
    A = At[i];
    if(m < 0) {
      dW = sg * dW;
      A = -sg * A;
      e = conj(em[am]);
    } else {
      e = o * em[am];
    }
  };
  cplx v[6];
#pragma unroll
  for(int c = 0; c < 6; ++c) v[c] = mk(0.0);
  {
    const int fz = t >> 7, p = t & 127;
    if(p < NF && (fz == 0 || a.sh)) {
      const cplx *co = (fz ? a.xintsh : a.xint) + (size_t)j * 2 * NF, *jn = fz ? js : jw;
      const cplx Kr = Rr * (fz ? ksh : ki), iKr = mk(1.0) / Kr;
      int n, m;
      unflat(p, n, m);
      double W, dW, A;
      cplx e;
      angular(n, m, W, dW, A, e);
      const double dn = sqrt((2.0 * n + 1.0) / (4.0 * kPi * (n * (n + 1))));
      const cplx z = jn[n], zd = ((double)n * z) / Kr - jn[n + 1], g = dn * e;
      const cplx zz = iKr * (Kr * zd + z), zr = iKr * (((double)(n * (n + 1))) * z);
      const cplx ap = g * co[p], bp = g * co[NF + p];
      const cplx Mt = z * mk(0.0, A), Mp = z * mk(-dW), Nr = zr * W, Nt = zz * dW, Np = zz * mk(0.0, A);
      v[0] = Nr * bp;
      v[1] = Mt * ap + Nt * bp;
      v[2] = Mp * ap + Np * bp;
      v[3] = Nr * ap;
      v[4] = Nt * ap + Mt * bp;
      v[5] = Np * ap + Mp * bp;
    }
  }
#pragma unroll
  for(int c = 0; c < 6; ++c) {
    const cplx s = wave_total(v[c]);
    if(lane == 0) wsum[w][c] = s;
  }
  const double st = sin(Rt), ct = cos(Rt), sp = sin(Rp), cp = cos(Rp);
  const cplx mi = mk(0.0, -1.0);
  __syncthreads();
  cplx oE[3], oH[3];
  if(t == 0 || (t == 128 && a.sh)) {
    cplx e3[3], h3[3];
    for(int c = 0; c < 3; ++c) {
      e3[c] = wsum[w][c] + wsum[w + 1][c];
      h3[c] = wsum[w][3 + c] + wsum[w + 1][3 + c];
    }
    to_cart(st, ct, sp, cp, e3, oE);
    to_cart(st, ct, sp, cp, h3, oH);
    const cplx iZ = mi / csqrt_(a.mu[j] / (t ? a.eps_sh[j] : a.eps[j]));
    for(int c = 0; c < 3; ++c) {
      if(t == 0) {
        a.E[3 * ip + c] = oE[c];
        a.H[3 * ip + c] = oH[c] * iZ;
      } else {
        oE[c] = oE[c] * k0;  // the bulk term is added below
        a.Hsh[3 * ip + c] = oH[c] * (iZ * k0);
      }
    }
  }
  if(!a.sh) return;
  // E_gamma: the bulk (gamma) source of the fundamental internal field
  const cplx zz = Rr * kj;
  const double ir = 1.0 / Rr;
  if(t <= NMAX) {
    cplx dv = mk(0.0);
    if(hypot(zz.x, zz.y) > kErrEps) dv = -f[t + 1] + (((double)t) * f[t]) / zz;
    if(zz.y == 0.0) dv.y = 0.0;
    d[t] = dv;
  }
  __syncthreads();
  if(t <= NMAX) {
    cplx dv = mk(0.0);
    if(t >= 1 && hypot(zz.x, zz.y) > kErrEps) {  // bessel3der (Bessel.h:230-231)
      dv = -(mk((double)t) / zz) * d[t] + (mk((double)t) / (zz * zz)) * f[t] + d[t - 1];
      if(zz.y == 0.0) dv.y = 0.0;
    }
    d2[t] = dv;
  }
  __syncthreads();
  const cplx ik2 = mk(1.0) / (kj * kj);
  for(int e = t; e < NMAX * NMAX; e += 256) {
    const int n1 = e / NMAX + 1, n2 = e % NMAX + 1;
    const double s4 = sqrt((double)n1 * n2 * (n1 + 1) * (n2 + 1));
    const cplx j1 = f[n1], j2 = f[n2], dj1 = d[n1], dj2 = d[n2];
    const cplx b1 = kj * dj1 + j1 * ir, b2 = kj * dj2 + j2 * ir;
    const cplx a1 = kj * kj * d2[n1] - (ir * ir) * j1 + ir * kj * dj1;
    const cplx a2 = kj * kj * d2[n2] - (ir * ir) * j2 + ir * kj * dj2;
    tab[0][e] = j1 * dj2 * kj + kj * dj1 * j2;
    tab[1][e] = ik2 * (a1 * b2 + a2 * b1);
    tab[2][e] = ik2 * (s4 * ((ir * ir) * (kj * dj1 * j2 + j1 * kj * dj2) - (2.0 * ir * ir * ir) * (j1 * j2)));
    tab[3][e] = j1 * dj2;
    tab[4][e] = ik2 * (b2 * b1);
    tab[5][e] = ik2 * (s4 * ((ir * ir) * (j1 * j2)));
  }
  __syncthreads();
  {
    constexpr int parts = 256 / NF;
    const int kk = t % NF, part = t / NF;
    cplx xm = mk(0.0), xp = mk(0.0);
    if(part < parts) {
      const size_t sz = (size_t)NF * NF * NF, base = (size_t)kk * NF * NF;
      const double *W00 = a.tab + 6 * sz + base, *W11 = a.tab + 5 * sz + base, *Wm = a.tab + 4 * sz + base;
      int n, m;
      unflat(kk, n, m);
      for(int p = part; p < NF; p += parts) {
        int n1, m1;
        unflat(p, n1, m1);
        const int m2 = m - m1;
        const cplx cp_ = cs[p], dp = ds[p];
        for(int n2 = max(1, abs(m2)); n2 <= NMAX; ++n2) {
          const int q = flat(n2, m2), e = (n1 - 1) * NMAX + n2 - 1;
          const double w00 = W00[p * NF + q], w11 = W11[p * NF + q], wm = Wm[p * NF + q];
          const cplx cc = cp_ * cs[q], dq = dp * ds[q];
          xm = xm + (w00 * cc) * tab[0][e] + dq * (w11 * tab[1][e] + wm * tab[2][e]);
          xp = xp + (w00 * cc) * tab[3][e] + dq * (w11 * tab[4][e] + wm * tab[5][e]);
        }
      }
    }
    red[0][t] = xm;
    red[1][t] = xp;
  }
  __syncthreads();
  cplx g3[3] = {mk(0.0), mk(0.0), mk(0.0)};
  if(t < NF) {
    constexpr int parts = 256 / NF;
    cplx xm = mk(0.0), xp = mk(0.0);
    for(int q = 0; q < parts; ++q) {
      xm = xm + red[0][q * NF + t];
      xp = xp + red[1][q * NF + t];
    }
    int n, m;
    unflat(t, n, m);
    const double snn = sqrt((double)n * (n + 1)), dn = sqrt((2.0 * n + 1.0) / (4.0 * kPi * (n * (n + 1))));
    const cplx pre = (-mk(kEps0) / a.eps_sh[j]) * a.gamma[j];
    double W, dW, A;
    cplx e;
    angular(n, m, W, dW, A, e);
    // X(-1) = dm dn sqrt(n(n+1)) e (W, 0, 0); X(+1) = dm dn e (0, dW, iA)
    const cplx g = dn * e, gm = g * (pre * xm), gp = g * (pre * ((snn * ir) * xp));
    g3[0] = (snn * W) * gm;
    g3[1] = dW * gp;
    g3[2] = mk(0.0, A) * gp;
  }
#pragma unroll
  for(int c = 0; c < 3; ++c) {
    const cplx s = wave_total(g3[c]);
    if(lane == 0) wsum[w][c] = s;
  }
  __syncthreads();
  if(t == 128) {
    cplx e3[3], g[3];
    for(int c = 0; c < 3; ++c) e3[c] = wsum[0][c] + wsum[1][c];
    to_cart(st, ct, sp, cp, e3, g);
    for(int c = 0; c < 3; ++c) a.Esh[3 * ip + c] = oE[c] + g[c];
  }
}

template <int NMAX> void launch_fields(const FieldArgs &a, int ns, hipStream_t st) {
  const int tiles = (a.npts + 63) / 64, nfq = a.sh ? 2 : 1;
  hipLaunchKernelGGL(fields_owner, dim3((a.npts + 255) / 256), dim3(256), 0, st, a);
  hipLaunchKernelGGL(fields_outside<NMAX>, dim3(tiles, ns, nfq), dim3(256), 0, st, a);
  hipLaunchKernelGGL(fields_sum, dim3((a.npts + 255) / 256, nfq), dim3(256), 0, st, a, ns);
  hipLaunchKernelGGL(fields_inside<NMAX>, dim3(a.npts), dim3(256), 0, st, a);
}

}  // namespace

// Slices of the objects: as many as give 2048 workgroups (two of four waves
// per SIMD pair and CU, what the registers allow), at most one task a wave.
int fields_slices(int P, int npts, int sh) {
  const int tiles = (npts + 63) / 64, nfq = sh ? 2 : 1;
  return std::max(1, std::min((P + 1 + 3) / 4, 2048 / (tiles * nfq)));
}

void run_fields(const FieldArgs &a, hipStream_t st) {
  const int ns = fields_slices(a.P, a.npts, a.sh);
  switch(a.nmax) {
  case 1: launch_fields<1>(a, ns, st); break;
  case 2: launch_fields<2>(a, ns, st); break;
  case 3: launch_fields<3>(a, ns, st); break;
  case 4: launch_fields<4>(a, ns, st); break;
  case 5: launch_fields<5>(a, ns, st); break;
  case 6: launch_fields<6>(a, ns, st); break;
  case 7: launch_fields<7>(a, ns, st); break;
  case 8: launch_fields<8>(a, ns, st); break;
  case 9: launch_fields<9>(a, ns, st); break;
  case 10: launch_fields<10>(a, ns, st); break;
  default: break;
  }
}

}  // namespace omx
