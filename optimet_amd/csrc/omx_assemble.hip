// omx_assemble.hip -- coefficient generation and matrix assembly on CDNA4.
//
// Kernels:
//   objects_kernel     Mie T-matrices and auxiliary per-object vectors
//                      (Scatterer.cpp:39-412, Geometry.cpp:86-145)
//   pair_kernel        Stout translation coefficients of one sphere pair
//                      (TranslationAdditionCoefficients.cpp:71-135,
//                      Coupling.cpp:30-87) fused with the block write
//                      S_ij = -T_i [[A^T,B^T],[B^T,A^T]] (PreconditionedMatrix.cpp:350-400)
//   origin_kernel      regular coupling from the origin per object: local
//                      incident field, Q_i = T_i inc_i (PreconditionedMatrix.cpp:1327-1345,
//                      Excitation.cpp:79-129) and the column weights of the
//                      scattering cross section (Result.cpp:579-647)
//   cross_kernel       per-object cross-section partial sums (Result.cpp:557-761)
//   pad_kernel         identity padding of the matrix up to the LU block size
//
// The Stout recurrence decouples into independent "rows": for a fixed
// instance (k or its negative-m twin), fixed m and fixed k = m + kappa, the
// diagonal recurrence (n = m) followed by the off-diagonal recurrence in n
// needs only the neighbours l-1, l+1 of the previous step.  Each row is
// mapped to 2*nmax+1 consecutive lanes of a wave (lane = l); neighbours come
// from cross-lane shuffles, and the rows stay in registers from one degree to
// the next, so every degree costs one step per row.
#include <utility>

#include "omx_kernels.hpp"

namespace omx {

// ------------------------------------------------------------------ objects
// One workgroup of two waves per object.  Output ov[kind][obj][2][nmax+1] (TE
// at [0], TM at [1]).  Bound: the latency of a Miller recurrence (about 60
// complex divisions in a row); the seven Bessel sets of an object run side by
// side in lanes of the two waves (five j_n, two h_n), then every (frequency,
// degree) has a lane of its own.  One thread per object, with the sets one
// after another and its arrays in scratch, took 151 us for 3 objects at nmax
// 6, which every solve waits for; this takes 23.
__global__ __launch_bounds__(128) void objects_kernel(ObjArgs a) {
  const int i = blockIdx.x, t = threadIdx.x;
  if(a.omz) {  // system blockIdx.z of a batch
    const int z = blockIdx.z;
    a.omega = a.omz[z];
    a.eps += (size_t)z * a.P;
    a.eps_sh += (size_t)z * a.P;
    a.ov += z * a.zov;
    if(z > 0) a.sph = nullptr;  // the geometry is common: system 0 writes it
  }
  const int nmax = a.nmax, S = nmax + 1;
  auto OV = [&](int kind, int pol, int n) -> cplx & {
    return a.ov[(((size_t)kind * a.P + i) * 2 + pol) * S + n];
  };
  if(t == 127 && a.sph) {
    // spherical coordinates of the centre (Tools.cpp:250-258)
    double x = a.xyz[3 * i], y = a.xyz[3 * i + 1], z = a.xyz[3 * i + 2];
    double r = sqrt(x * x + y * y + z * z);
    const double th = r > 0.0 ? acos(z / r) : 0.0, ph = r > 0.0 ? atan2(y, x) : 0.0;
    double *o = a.sph + kSphDoubles * i;
    o[0] = r > 0.0 ? r : 0.0;
    o[1] = sin(th);
    o[2] = cos(th);
    o[3] = sin(ph);
    o[4] = cos(ph);
  }
  const double R = a.radius[i];
  const cplx eps = a.eps[i], mu = a.mu[i], eps_sh = a.eps_sh[i], mu_sh = mu;
  const cplx bge = a.bg_eps, bgm = a.bg_mu;
  // Bessel sets: 0, 1: j_n at r0 and rho r0 (omega); 2, 3: the same at
  // 2 omega; 4: j_n at k_j R (SH source); 5, 6: h_n at r0 (omega, 2 omega)
  __shared__ cplx bf[7][kMaxNmax + 2], bd[7][kMaxNmax + 2];
  const int set = t < 5 ? t : (t == 64 || t == 65) ? t - 59 : -1;
  if(set >= 0) {
    const int f = set < 4 ? set >> 1 : set - 5;  // 0: omega, 1: 2 omega
    double om = (f == 1 ? 2.0 : 1.0) * a.omega;
    cplx ks = om * csqrt_((f == 1 ? eps_sh : eps) * (f == 1 ? mu_sh : mu));
    cplx kb = om * csqrt_(bge * bgm);
    cplx rho = ks / kb, r0 = kb * R;
    cplx z = (set < 4 && (set & 1)) ? rho * r0 : r0;
    if(set == 4) {
      cplx kj = a.omega * csqrt_(eps * mu);
      z = R * kj;
    }
    sph_bessel(set >= 5, z, nmax, bf[set], bd[set]);
  }
  __syncthreads();
  if(t < 2 * nmax) {
    const int f = t / nmax, n = t % nmax + 1;  // f = 0: omega, f = 1: 2 omega
    const cplx zeta_b2 = csqrt_(bgm / bge);
    double om = (f == 0 ? 1.0 : 2.0) * a.omega;
    cplx ks = om * csqrt_((f ? eps_sh : eps) * (f ? mu_sh : mu));
    cplx kb = om * csqrt_(bge * bgm);
    cplx rho = ks / kb, r0 = kb * R;
    cplx mu_s = f ? mu_sh : mu;
    cplx mu_sob = mu_s / bgm;
    // Riccati functions of degree n
    const cplx jf = bf[2 * f][n], jd = bd[2 * f][n], rf = bf[2 * f + 1][n], rd = bd[2 * f + 1][n];
    const cplx hf = bf[5 + f][n], hd = bd[5 + f][n];
    const cplx psi = r0 * jf, dpsi = r0 * jd + jf, ksi = r0 * hf, dksi = r0 * hd + hf;
    const cplx psr = (r0 * rho) * rf, dpsr = (r0 * rho) * rd + rf;
    cplx zeta_j2 = f ? csqrt_(mu_sh / eps_sh) : csqrt_(mu / eps);
    cplx zb = zeta_b2 / zeta_j2;
    cplx xb = kb * R, xi2 = ks * R;
    // T (Scatterer.cpp:70-84) / T_SH (:131-145)
    cplx te = (psi / ksi) * (mu_sob * dpsi / psi - rho * dpsr / psr) / (rho * dpsr / psr - mu_sob * dksi / ksi);
    cplx tm = (psi / ksi) * (mu_sob * dpsr / psr - rho * dpsi / psi) / (rho * dksi / ksi - mu_sob * dpsr / psr);
    OV(f ? OV_TSH : OV_T, 0, n) = te;
    OV(f ? OV_TSH : OV_T, 1, n) = tm;
    if(f == 0) {
      // Iaux (Scatterer.cpp:297-312)
      cplx mu_j = mu, mu_0 = bgm, I = mk(0.0, 1.0);
      OV(OV_IAUX, 0, n) = (mu_j * rho) / (mu_0 * rho * dpsr * psi - mu_j * psr * dpsi) * I;
      OV(OV_IAUX, 1, n) = (mu_j * rho) / (mu_j * psi * dpsr - mu_0 * rho * psr * dpsi) * I;
      // absorption weights (Geometry.cpp:126-140), real part kept in .x
      cplx t1 = I * rho * mu_0 * conj(mu_j) * conj(psr) * dpsr;
      double t2 = cabs(mu_j * psr * dpsi - mu_0 * rho * dpsr * psi);
      OV(OV_CABS, 0, n) = mk(t1.x / (t2 * t2));
      t1 = I * conj(rho) * mu_0 * mu_j * conj(psr) * dpsr;
      t2 = cabs(mu_0 * rho * psr * dpsi - mu_j * dpsr * psi);
      OV(OV_CABS, 1, n) = mk(t1.x / (t2 * t2));
    } else {
      // IauxSH1 (Scatterer.cpp:343-357), IauxSH2 (:390-404)
      OV(OV_IAUXSH1, 0, n) = (-xi2 * ksi) / (xb * psr);
      OV(OV_IAUXSH1, 1, n) = (-xi2 * dksi) / (xb * dpsr);
      cplx bnpp = (zb * xb * dpsr) / (zb * ksi * dpsr - psr * dksi);
      cplx anpp = (zb * xb * psr) / (zb * psr * dksi - ksi * dpsr);
      OV(OV_IAUXSH2, 0, n) = bnpp * ((-xi2 * ksi) / (xb * psr) + (xi2 * dksi) / (zb * xb * dpsr));
      OV(OV_IAUXSH2, 1, n) = anpp * ((-xi2 * dksi) / (xb * dpsr) + (xi2 * ksi) / (zb * xb * psr));
      // TSH1_outer (Scatterer.cpp:200-208), TSH2_outer (:250-260)
      OV(OV_TSH1O, 0, n) = -xb * psr / (zb * ksi * dpsr - psr * dksi);
      OV(OV_TSH1O, 1, n) = -xb * dpsr / (zb * psr * dksi - ksi * dpsr);
      OV(OV_TSH2O, 0, n) = zb * xb * dpsr / (zb * ksi * dpsr - psr * dksi);
      OV(OV_TSH2O, 1, n) = zb * xb * psr / (zb * psr * dksi - ksi * dpsr);
    }
  }
  // radial data of the SH source (Symbol.cpp:52-78): j_n(k_j R) and k_j j_n' + j_n / R
  if(t >= 64 && t <= 64 + nmax) {
    const int n = t - 64;
    cplx kj = a.omega * csqrt_(eps * mu);
    OV(OV_SHRAD, 0, n) = bf[4][n];
    OV(OV_SHRAD, 1, n) = kj * bd[4][n] + bf[4][n] / R;
  }
}

// ------------------------------------------------------------------ tables
// Shape of a workgroup of the pair and origin kernels.  A recurrence row (inst,
// m, k) takes L lanes of a wave (lane = l); a wave holds G rows of consecutive k
// and S waves all of them, for the orders (inst, m) dealt to it: MS sets of S
// waves share the 2 nmax + 1 orders, GR for each.  Two sets where the state of
// all orders would not fit beside the rest of a kernel's registers without
// losing a workgroup per CU, one set where it does (nmax 6) or where two would
// leave a lane 128 registers (nmax 9, 10).  S, us, with one / two sets: nmax 5,
// 150 spheres 913 / 917; nmax 6, 128 spheres 707 / 808; nmax 7, 100 spheres 1163
// / 1170; nmax 8, 64 spheres with V 1425 / 1420; nmax 10, 60 spheres 1456 / 2396.
template <int NMAX> struct PairCfg {
  static constexpr int L = 2 * NMAX + 1, G = 64 / L, S = (L + G - 1) / G;
  static constexpr int MS = NMAX <= 3 ? 4 : NMAX == 6 || NMAX >= 9 ? 1 : 2;
  static constexpr int NW = S * MS, NT = 64 * NW, GR = (L + MS - 1) / MS;
};

// LDS workspace of one pair (or one object-origin coupling).
template <int NMAX>
struct PairLDS {
  static constexpr int L = 2 * NMAX + 1;           // lanes per recurrence row
  static constexpr int NL = (NMAX + 1) * (NMAX + 1); // (l, K) entries per (n, M), l <= NMAX
  static constexpr int NF = NMAX * (NMAX + 2);
  static constexpr int KD = 3 * NMAX + 1;          // diagonal rows: k = -2 nmax .. nmax
  cplx h[2][L + 1];          // z_l(k R) for the +m and -m instances
  union {
    cplx Y[L * L];           // Y_l^k, index l*l + l + k (read before T is first written)
    cplx T[(2 * NMAX + 1) * NL]; // C(n, M, l, K) of the current n, index (M+n)*NL + l*l+l+K
  };
  cplx D[2 * KD * L];        // C(n, n, l, k) of the current n, [inst][k + 2 nmax][l]
  cplx Ti[2 * NF];           // row scale -T_i (assembly) or incident vector (origin)
  double w[NF];              // column weights (origin kernel)
  __device__ PairLDS() {}
};

// Division by a fixed complex z (Smith's scaling, as cplx's operator/) whose
// two real divisions by the common d use its reciprocal: with rd the rounded
// 1 / d, q = x rd and q + (x - q d) rd by fused multiply-adds is the rounded
// x / d (Markstein 1990), in three instructions instead of about thirty.
struct DivBy {
  double r, d, rd;
  bool re;
  __device__ DivBy(cplx z) {
    re = fabs(z.x) >= fabs(z.y);
    r = re ? z.y / z.x : z.x / z.y;
    d = re ? z.x + z.y * r : z.x * r + z.y;
    rd = 1.0 / d;
  }
  __device__ double real(double x) const {
    const double q = x * rd;
    return fma(fma(-q, d, x), rd, q);
  }
  __device__ cplx operator()(cplx a) const {
    return re ? mk(real(a.x + a.y * r), real(a.y - a.x * r)) : mk(real(a.x * r + a.y), real(a.y * r - a.x));
  }
};

// Computes z_l and Y_l^k for pair vector R (r, theta, phi) and wavenumber k.
template <int NMAX>
__device__ void pair_setup(PairLDS<NMAX> &s, double Rr, double Rt, double Rp, cplx k, bool hankel,
                           const double *__restrict__ coef) {
  constexpr int L = PairLDS<NMAX>::L;
  int t = threadIdx.x;
  if(t < 2) {
    // +m instance: k; -m instance: conj(k) (regular) or -conj(k) (irregular)
    // (TranslationAdditionCoefficients.h:72-74)
    cplx kk = (t == 0) ? k : (hankel ? -conj(k) : conj(k));
    sph_values_to<DivBy>(hankel ? 1 : 0, Rr * kk, L + 1, s.h[t]);
  } else if(t >= 64 && t < 64 + L) {
    // normalised associated Legendre, column |k| = am, rows l = am .. L-1; all
    // coefficients are loaded before the recurrence starts
    const int am = t - 64;
    const double *LP = coef + CF_DEG * kCoefStride + CF_LEGP, *LA = coef + CF_LEGA * kCoefStride + am,
                 *LB = coef + CF_LEGB * kCoefStride + am;
    double la[L], lb[L];
    la[0] = lb[0] = 0.0;
#pragma unroll
    for(int l = 1; l < L; ++l) {
      la[l] = LA[l * l + l];
      lb[l] = LB[l * l + l];
    }
    double x = cos(Rt), sx = sin(Rt);
    double p = 1.0 / sqrt(4.0 * kPi);
#pragma unroll
    for(int i = 1; i < L; ++i) {
      const double v = p * (LP[i] * sx);
      p = i <= am ? v : p;
    }
    double pm2 = 0.0, pm1 = 0.0;
    cplx e = mk(cos(am * Rp), sin(am * Rp));
    double sg = (am % 2) ? -1.0 : 1.0;
#pragma unroll
    for(int l = 0; l < L; ++l) {
      double pl = la[l] * (x * pm1 - lb[l] * pm2);
      if(l == am + 1) pl = la[l] * x * p;
      if(l == am) pl = p;
      if(l >= am) {
        pm2 = pm1;
        pm1 = pl;
        cplx y = pl * e;
        s.Y[l * l + l + am] = y;
        if(am > 0) s.Y[l * l + l - am] = sg * conj(y);
      }
    }
  }
}

// f(0), f(1), .. f(N - 1) with the index a compile-time constant from the
// start, so that arrays indexed by it stay in registers.
template <int N, class F> __device__ __forceinline__ void static_for(F &&f) {
  [&]<int... I>(std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
  }(std::make_integer_sequence<int, N>{});
}

// Value of the next / previous lane (wave_shl / wave_shr by one).
template <int CTRL> __device__ inline double dpp_d(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
constexpr int kFromNext = 0x130, kFromPrev = 0x138;

// The recurrence of every row, one harmonic degree a step, with the rows' state
// in registers: C(n, m, l, k) of this and the previous degree.
//
// Off-diagonal rows (m < n): the two coefficients of a step depend on (l, k)
// alone, so a lane loads them once for every order and degree; what depends on
// (n, m) is wave-uniform.  A row-step is about 30 instructions.
// Diagonal values C(n, n, l, k) depend on the previous degree's at k - 1, that
// is on k - n alone: one chain for every k - n, held in LDS and advanced by all
// threads, starts every row.
//
// Measured (one workgroup, clocks per degree at nmax 6): 2000 against 10000 with
// rows dealt to lanes regardless of m, each forming its indices and loading four
// coefficients a step, and the diagonal steps repeated by every row.
template <int NMAX> struct Recurrence {
  using Cfg = PairCfg<NMAX>;
  static constexpr int L = Cfg::L, NL = PairLDS<NMAX>::NL, KD = PairLDS<NMAX>::KD;
  static constexpr int NT = Cfg::NT, GR = Cfg::GR, ITEMS = 2 * KD * L, IT = (ITEMS + NT - 1) / NT;
  cplx cur[GR], prev[GR];
  double ca, cb;         // a lane's coefficients of an off-diagonal step: of l - 1 and l + 1
  int l, k, ms;          // lane's degree and order; its wave's set of orders
  bool rowok, tabok;     // the lane holds a row entry; one that goes into the table
  double da[IT], db[IT]; // an item's coefficients of a diagonal step: of l + 1 and l - 1
  cplx dv[IT];           // its value
  static __device__ int ci(int nn, int mm) { return nn * nn + nn + mm; }
  // item of the diagonal chains: instance, k and l
  static __device__ __forceinline__ bool item(int i, int &inst, int &kk, int &ll) {
    const int e = threadIdx.x + i * NT;
    inst = e / (KD * L);
    kk = (e / L) % KD - 2 * NMAX;
    ll = e % L;
    return e < ITEMS;
  }
  __device__ __forceinline__ void store_diag(PairLDS<NMAX> &s) const {
    static_for<IT>([&](auto c) {
      constexpr int i = c;
      if((int)threadIdx.x + i * NT < ITEMS) s.D[threadIdx.x + i * NT] = dv[i];
    });
  }
  // A lane's places and coefficients (before the pair's setup, which hides the
  // latency of the loads).
  __device__ __forceinline__ void init(const double *__restrict__ coef) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = lane / L, kr = (wave % Cfg::S) * Cfg::G + rg;
    l = lane % L;
    k = kr - NMAX;
    ms = wave / Cfg::S;
    rowok = rg < Cfg::G && kr < L;
    tabok = rowok && l <= NMAX && abs(k) <= l;
    const double *CAP = coef + CF_AP * kCoefStride, *CAM = coef + CF_AM * kCoefStride;
    const double *CBP = coef + CF_BP * kCoefStride, *CBM = coef + CF_BM * kCoefStride;
    ca = (rowok && l >= 1 && abs(k) <= l - 1) ? CAP[ci(l - 1, k)] : 0.0;
    cb = (rowok && l < L - 1 && abs(k) <= l + 1) ? CAM[ci(l + 1, k)] : 0.0;
    static_for<IT>([&](auto c) {
      constexpr int i = c;
      int inst, kk, ll;
      const bool ok = item(i, inst, kk, ll);
      const int kd = kk - 1;
      da[i] = (ok && ll < L - 1 && abs(kd) <= ll + 1) ? CBM[ci(ll + 1, kd)] : 0.0;
      db[i] = (ok && ll >= 1 && abs(kd) <= ll - 1) ? CBP[ci(ll - 1, kd)] : 0.0;
    });
  }
  // D_0(l) = C(0, 0, l, kappa) (TranslationAdditionCoefficients.cpp:102-111)
  // into s.D; the caller synchronises before the first step.
  __device__ __forceinline__ void start(PairLDS<NMAX> &s) {
    const double s4pi = sqrt(4.0 * kPi);
    static_for<IT>([&](auto c) {
      constexpr int i = c;
      int inst, kk, ll;
      const bool ok = item(i, inst, kk, ll);
      dv[i] = mk(0.0);
      if(ok && abs(kk) <= ll) {
        cplx hb = s.h[inst][ll];
        if(ll == 0 && kk == 0)
          dv[i] = hb;
        else {
          double fac = s4pi * (((ll + kk) % 2 == 0) ? 1.0 : -1.0);
          dv[i] = fac * (s.Y[ll * ll + ll - kk] * hb);
        }
      }
    });
    store_diag(s);
    static_for<GR>([&](auto c) { cur[c] = prev[c] = mk(0.0); });
  }
  // Degree t (called for t = 1, 2, ..) from s.D of degree t - 1: the table
  // C(t, M, l, K), |M| <= t, l <= NMAX, |K| <= l, into s.T.  The caller
  // synchronises, then store_diag's degree t into s.D, then synchronises again
  // before the next step.
  __device__ __forceinline__ void step(PairLDS<NMAX> &s, int t, bool hankel, const double *__restrict__ coef) {
    const double *CAM = coef + CF_AM * kCoefStride, *CIA = coef + CF_IAP * kCoefStride,
                 *CIB = coef + CF_IBP * kCoefStride;
    // off-diagonal steps to (t, m, l, k) (:119-124) of the rows with m < t
    static_for<GR>([&](auto ic) {
      constexpr int i = ic;
      const int e = ms + i * Cfg::MS;
      const int inst = e <= NMAX ? 0 : 1, m = inst ? e - NMAX : e;
      if(e >= L || m >= t) return;
      const double c0 = CAM[ci(t - 1, m)], c3 = CIA[ci(t - 1, m)];
      cplx c = cur[i];
      if(m == t - 1) {  // the row starts from its diagonal value
        cplx d = mk(0.0);
        if(rowok) d = s.D[(inst * KD + k + 2 * NMAX) * L + l];
        // a value of its own: a choice between the two places to load from
        // would keep the whole state in memory
        asm volatile("" : "+v"(d.x), "+v"(d.y));
        c = d;
      }
      const double lx = dpp_d<kFromPrev>(c.x), ly = dpp_d<kFromPrev>(c.y);
      const double hx = dpp_d<kFromNext>(c.x), hy = dpp_d<kFromNext>(c.y);
      cplx nw;
      nw.x = fma(hx, cb, fma(lx, ca, -(prev[i].x * c0))) * c3;
      nw.y = fma(hy, cb, fma(ly, ca, -(prev[i].y * c0))) * c3;
      prev[i] = c;
      cur[i] = nw;
      if(tabok) put(s, t, inst, m, k, l, hankel, nw);
    });
    // diagonal steps to (t, t, l, k) (:113-117)
    const double c3 = CIB[ci(t - 1, t - 1)];
    static_for<IT>([&](auto ic) {
      constexpr int i = ic;
      int inst, kk, ll;
      const bool ok = item(i, inst, kk, ll);
      cplx lo = mk(0.0), hi = mk(0.0);
      if(ok && kk > -2 * NMAX) {
        const cplx *d = s.D + (inst * KD + kk - 1 + 2 * NMAX) * L + ll;
        if(ll > 0) lo = d[-1];
        if(ll < L - 1) hi = d[1];
      }
      dv[i].x = fma(lo.x, db[i], hi.x * da[i]) * c3;
      dv[i].y = fma(lo.y, db[i], hi.y * da[i]) * c3;
      if(ok && ll <= NMAX && abs(kk) <= ll) put(s, t, inst, t, kk, ll, hankel, dv[i]);
    });
  }
  // C(t, m, l, k) of instance 0, or C(t, -m, l, -k) from instance 1, into the table
  static __device__ __forceinline__ void put(PairLDS<NMAX> &s, int t, int inst, int m, int k, int l, bool hankel, cplx v) {
    if(inst == 0) {
      s.T[(m + t) * NL + l * l + l + k] = v;
    } else {
      const int M = -m, K = -k;
      const int e = hankel ? (t + M + l + K) : (K + M);
      v = conj(v);
      if(e % 2) v = -v;
      s.T[(M + t) * NL + l * l + l + K] = v;
    }
  }
};

template <int NMAX>
__device__ inline cplx tget(const PairLDS<NMAX> &s, int n, int M, int l, int K) {
  constexpr int NL = PairLDS<NMAX>::NL;
  if(abs(M) > n || l < 0 || abs(K) > l) return mk(0.0);
  return s.T[(M + n) * NL + l * l + l + K];
}

// Per-row (q = (l, K)) factors of the A / B formulas (Coupling.cpp:30-51).
struct QFac {
  int l, K;
  double lam, mu, b1, b2, g0, g1, g2;
};
__device__ inline QFac qfac(int q, const double *__restrict__ coef) {
  QFac f;
  unflat(q, f.l, f.K);
  const int i = f.l * f.l + f.l + f.K;
  f.lam = coef[CF_DEG * kCoefStride + CF_NU + f.l];
  f.mu = coef[CF_DEG * kCoefStride + CF_MU + f.l];
  f.b1 = coef[CF_A1 * kCoefStride + i];
  f.b2 = coef[CF_A2 * kCoefStride + i];
  f.g0 = coef[CF_G0 * kCoefStride + i];
  f.g1 = coef[CF_G1 * kCoefStride + i];
  f.g2 = coef[CF_G2 * kCoefStride + i];
  return f;
}

// A(p, q) and B(p, q) for p = (n, M) (object j harmonic) and row q.
template <int NMAX>
__device__ inline void coeff_AB(const PairLDS<NMAX> &s, int n, int M, const QFac &f, const double *__restrict__ coef,
                                cplx &A, cplx &B) {
  const double nu = coef[CF_DEG * kCoefStride + CF_NU + n];
  const double a1 = coef[CF_A1 * kCoefStride + n * n + n + M], a2 = coef[CF_A2 * kCoefStride + n * n + n + M];
  int l = f.l, K = f.K;
  cplx t0 = tget(s, n, M, l, K), tp = tget(s, n, M + 1, l, K + 1), tm = tget(s, n, M - 1, l, K - 1);
  A = (0.5 * f.lam * nu) * ((double)(2 * K * M) * t0 + (a1 * f.b1) * tp + (a2 * f.b2) * tm);
  cplx u0 = tget(s, n, M, l - 1, K), up = tget(s, n, M + 1, l - 1, K + 1), um = tget(s, n, M - 1, l - 1, K - 1);
  cplx v = ((double)(2 * M) * f.g0) * u0 + (a1 * f.g1) * up - (a2 * f.g2) * um;
  double fb = -0.5 * f.mu * nu;
  B = mk(-fb * v.y, fb * v.x);  // (0, fb) * v
}

// Pair vector r_i - r_j through Cartesian coordinates (Spherical.h:129-131);
// the angles' sines and cosines come from objects_kernel.
__device__ inline void pair_vector(const double *sph, int i, int j, double &r, double &t, double &p) {
  const double *a = sph + kSphDoubles * i, *b = sph + kSphDoubles * j;
  double xi = a[0] * a[1] * a[4], yi = a[0] * a[1] * a[3], zi = a[0] * a[2];
  double xj = b[0] * b[1] * b[4], yj = b[0] * b[1] * b[3], zj = b[0] * b[2];
  double dx = xi - xj, dy = yi - yj, dz = zi - zj;
  r = sqrt(dx * dx + dy * dy + dz * dz);
  if(r > 0.0) {
    t = acos(dz / r);
    p = atan2(dy, dx);
  } else {
    t = p = 0.0;
  }
}

// ------------------------------------------------------------------ assembly
// One block per unordered pair i <= j (block rows i and j, triangular index
// blockIdx.x), or per listed pair i < j (pair-list mode: S_ij and S_ji in two
// consecutive slots); blockIdx.y = 1 takes the launch's second matrix (V
// beside S).  S_ji comes from them by the parity of the translation: A_pq(-R) = (-1)^(n+l) A_pq(R), B_pq(-R) = -(-1)^(n+l) B_pq(R)
// for p of degree n and q of degree l, scaled by -T_j.
// Bound: the blocks' stores, 24 bytes an entry with the FP32 copy, as far as the
// serial setup of a pair (radial functions, Legendre functions: about 5 us) is
// hidden by the CU's other workgroups.  S alone, P = 512, nmax 6: 11.8 ms, 4.9
// TB/s (21.6 before the recurrences kept their state); S and V, P = 64, nmax 8:
// 1.40 ms, 3.6 TB/s (2.52); one pair alone, nmax 6: 30 us (90).  (The reference computes
// the ordered pair j, i through its own pair vector, equal to rounding).
template <int NMAX>
__global__ __launch_bounds__(PairCfg<NMAX>::NT) void pair_kernel(PairArgs a) {
  constexpr int NF = PairLDS<NMAX>::NF;
  __shared__ PairLDS<NMAX> s;
  const int P = a.P;
  if(blockIdx.y) {  // the second matrix of the launch
    a.tkind = a.tkind2;
    a.k = a.k2;
    a.kz = a.kz2;
    a.S64 = a.V64;
    a.S32 = a.V32;
  }
  if(a.kz) {  // system blockIdx.z of a batch
    const int z = blockIdx.z;
    a.k = a.kz[z];
    a.ov += z * a.zov;
    if(a.S64) a.S64 += z * a.zS;
    if(a.S32) a.S32 += z * a.zS;
  }
  int i, j;
  size_t x0, y0;
  if(a.plist) {  // unordered pair blockIdx.x of a list, its two blocks in slots of their own
    const int pid = a.plist[blockIdx.x];
    i = pid / P;
    j = pid % P;
    if(a.S64) a.S64 += 2 * blockIdx.x * a.zblk;
    if(a.S32) a.S32 += 2 * blockIdx.x * a.zblk;
  } else {  // triangular index k = j (j + 1) / 2 + i, i <= j
    const int k = blockIdx.x;
    int jj = (int)((sqrt(8.0 * k + 1.0) - 1.0) * 0.5);
    while((jj + 1) * (jj + 2) / 2 <= k) ++jj;
    while(jj * (jj + 1) / 2 > k) --jj;
    j = jj;
    i = k - jj * (jj + 1) / 2;
  }
  const int ci = i, cj = j;  // i <= j
  size_t x1, y1;             // the mirrored block S_{cj ci}
  size_t mo = 0;             // and its offset (a list's second slot)
  if(a.plist) {
    x0 = y0 = x1 = y1 = 0;
    mo = a.zblk;
  } else {
    x0 = (size_t)ci * 2 * NF;
    y0 = (size_t)cj * 2 * NF;
    x1 = y0;
    y1 = x0;
  }
  const int t = threadIdx.x;
  const int cg = blockDim.x / NF;  // column groups
  const int q = t % NF, grp = t / NF;
  const bool qact = grp < cg;
  if(i == j) {  // identity diagonal block
    for(int c = grp; c < 2 * NF && qact; c += cg) {
      for(int h = 0; h < 2; ++h) {
        int r = q + h * NF;
        double v = (r == c) ? 1.0 : 0.0;
        size_t idx = (y0 + c) * a.lda + x0 + r;
        if(a.S64) a.S64[idx] = mk(v);
        if(a.S32) a.S32[idx] = make_float2((float)v, 0.0f);
      }
    }
    return;
  }
  // row scale -T_ci
  for(int r = t; r < 2 * NF; r += blockDim.x) {
    int nn, mm;
    unflat(r % NF, nn, mm);
    s.Ti[r] = -a.ov[(((size_t)a.tkind * P + ci) * 2 + (r >= NF)) * (NMAX + 1) + nn];
  }
  double Rr, Rt, Rp;
  pair_vector(a.sph, ci, cj, Rr, Rt, Rp);
  const bool ident = fabs(Rr) < kErrEps;  // Coupling.cpp:82-84
  Recurrence<NMAX> rec;
  rec.init(a.coef);
  const QFac f = qfac(q, a.coef);
  if(!ident) pair_setup<NMAX>(s, Rr, Rt, Rp, a.k, true, a.coef);
  __syncthreads();
  const cplx Tq = s.Ti[q], Tq2 = s.Ti[q + NF];
  // row scale -T_cj of the mirrored block, and this row's parity (-1)^l
  cplx Uq = mk(0.0), Uq2 = mk(0.0);
  if(qact) {
    Uq = -a.ov[(((size_t)a.tkind * P + cj) * 2 + 0) * (NMAX + 1) + f.l];
    Uq2 = -a.ov[(((size_t)a.tkind * P + cj) * 2 + 1) * (NMAX + 1) + f.l];
  }
  const double sq = (f.l & 1) ? -1.0 : 1.0;
  if(!ident) rec.start(s);
  __syncthreads();
#pragma unroll 1
  for(int n = 1; n <= NMAX; ++n) {
    if(!ident) rec.step(s, n, true, a.coef);
    __syncthreads();
    if(!ident) rec.store_diag(s);
    if(qact) {
      for(int M = n - grp; M >= -n; M -= cg) {
        int p = flat(n, M);
        cplx A, B;
        if(ident) {
          A = mk(p == q ? 1.0 : 0.0);
          B = mk(0.0);
        } else {
          coeff_AB<NMAX>(s, n, M, f, a.coef, A, B);
        }
        cplx v00 = Tq * A, v10 = Tq2 * B, v01 = Tq * B, v11 = Tq2 * A;
        size_t c0 = (y0 + p) * a.lda + x0, c1 = (y0 + NF + p) * a.lda + x0;
        if(a.S64) {
          a.S64[c0 + q] = v00;
          a.S64[c0 + NF + q] = v10;
          a.S64[c1 + q] = v01;
          a.S64[c1 + NF + q] = v11;
        }
        if(a.S32) {
          a.S32[c0 + q] = make_float2((float)v00.x, (float)v00.y);
          a.S32[c0 + NF + q] = make_float2((float)v10.x, (float)v10.y);
          a.S32[c1 + q] = make_float2((float)v01.x, (float)v01.y);
          a.S32[c1 + NF + q] = make_float2((float)v11.x, (float)v11.y);
        }
        {
          const double sa = (n & 1) ? -sq : sq;
          const cplx Am = sa * A, Bm = (-sa) * B;
          const cplx w00 = Uq * Am, w10 = Uq2 * Bm, w01 = Uq * Bm, w11 = Uq2 * Am;
          const size_t d0 = mo + (y1 + p) * a.lda + x1, d1 = mo + (y1 + NF + p) * a.lda + x1;
          if(a.S64) {
            a.S64[d0 + q] = w00;
            a.S64[d0 + NF + q] = w10;
            a.S64[d1 + q] = w01;
            a.S64[d1 + NF + q] = w11;
          }
          if(a.S32) {
            a.S32[d0 + q] = make_float2((float)w00.x, (float)w00.y);
            a.S32[d0 + NF + q] = make_float2((float)w10.x, (float)w10.y);
            a.S32[d1 + q] = make_float2((float)w01.x, (float)w01.y);
            a.S32[d1 + NF + q] = make_float2((float)w11.x, (float)w11.y);
          }
        }
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ origin
// Block (j, f): object j, f = 0 at k (local incident field, Q, weights),
// f = 1 at 2k (weights for the second-harmonic scattering cross section; only
// launched with the second harmonic).  Bound: latency, one workgroup per
// object beside the whole assembly.  All threads take the coefficients of a
// degree into LDS, then threads 0 .. nf-1 add them up row by row (in the order
// of p) while the later waves add up the column weights.  With a row's thread
// computing its coefficients one after another and the weights by LDS atomics
// this took 185 us at nmax 6 (3 objects) and 479 at nmax 8 (64), in front of the
// pairs; now 37, and 167 beside the pairs.
template <int NMAX>
__global__ __launch_bounds__(PairCfg<NMAX>::NT) void origin_kernel(OriginArgs a) {
  constexpr int NF = PairLDS<NMAX>::NF, NT = PairCfg<NMAX>::NT;
  __shared__ PairLDS<NMAX> s;
  __shared__ cplx sA[(2 * NMAX + 1) * NF], sB[(2 * NMAX + 1) * NF];
  const int j = blockIdx.x, fq = blockIdx.y;
  const int t = threadIdx.x;
  const int P = a.P;
  if(a.kz) {  // system blockIdx.z of a batch
    const int z = blockIdx.z;
    a.k = a.kz[z];
    a.ov += z * a.zov;
    a.incloc += z * a.zvec;
    a.Q += z * a.zvec;
    a.w += z * a.zw;
  }
  // incident vector [a_inc; b_inc] in s.Ti
  for(int r = t; r < 2 * NF; r += NT) s.Ti[r] = a.inc[r];
  // Rrel = toSpherical(toCartesian(vR_j) - 0) (Excitation.cpp:81)
  double Rr, Rt, Rp;
  {
    const double *o = a.sph + kSphDoubles * j;
    double x = o[0] * o[1] * o[4], y = o[0] * o[1] * o[3], z = o[0] * o[2];
    Rr = sqrt(x * x + y * y + z * z);
    Rt = Rr > 0.0 ? acos(z / Rr) : 0.0;
    Rp = Rr > 0.0 ? atan2(y, x) : 0.0;
  }
  const bool ident = fabs(Rr) < kErrEps;
  cplx k = fq == 0 ? a.k : 2.0 * a.k;
  const int cg = NT / NF, q = t % NF, grp = t / NF;
  Recurrence<NMAX> rec;
  rec.init(a.coef);
  const QFac f = qfac(q, a.coef);
  if(!ident) pair_setup<NMAX>(s, Rr, Rt, Rp, k, false, a.coef);
  __syncthreads();
  cplx acc0 = mk(0.0), acc1 = mk(0.0);
  if(!ident) rec.start(s);
  __syncthreads();
  constexpr int W0 = (NF + 63) / 64;  // the first wave that holds no row
  const int lane = t & 63, wave = t >> 6;
#pragma unroll 1
  for(int n = 1; n <= NMAX; ++n) {
    if(!ident) rec.step(s, n, false, a.coef);
    __syncthreads();
    if(!ident) rec.store_diag(s);
    if(grp < cg)
      for(int e = grp; e <= 2 * n; e += cg) {  // M = n - e
        cplx A, B;
        if(ident) {
          A = mk(flat(n, n - e) == q ? 1.0 : 0.0);
          B = mk(0.0);
        } else {
          coeff_AB<NMAX>(s, n, n - e, f, a.coef, A, B);
        }
        sA[e * NF + q] = A;
        sB[e * NF + q] = B;
      }
    __syncthreads();
    if(t < NF) {
      for(int e = 0; e <= 2 * n; ++e) {
        const int p = flat(n, n - e);
        const cplx A = sA[e * NF + t], B = sB[e * NF + t];
        // inc_local[q] = sum_p A(p,q) a_p + B(p,q) b_p ; [nf+q]: B a + A b
        acc0 = acc0 + A * s.Ti[p] + B * s.Ti[NF + p];
        acc1 = acc1 + B * s.Ti[p] + A * s.Ti[NF + p];
      }
    } else if(wave >= W0) {
      for(int e = wave - W0; e <= 2 * n; e += NT / 64 - W0) {
        double w = 0.0;
        for(int r = lane; r < NF; r += 64) w += norm2(sA[e * NF + r]) + norm2(sB[e * NF + r]);
#pragma unroll
        for(int o = 32; o > 0; o >>= 1) w += __shfl_xor(w, o, 64);
        if(lane == 0) s.w[flat(n, n - e)] = w;
      }
    }
  }
  __syncthreads();
  if(t < NF) {
    if(fq == 0) {
      int nn, mm;
      unflat(t, nn, mm);
      const cplx te = a.ov[(((size_t)OV_T * P + j) * 2 + 0) * (NMAX + 1) + nn];
      const cplx tm = a.ov[(((size_t)OV_T * P + j) * 2 + 1) * (NMAX + 1) + nn];
      a.incloc[(size_t)j * 2 * NF + t] = acc0;
      a.incloc[(size_t)j * 2 * NF + NF + t] = acc1;
      a.Q[(size_t)j * 2 * NF + t] = te * acc0;
      a.Q[(size_t)j * 2 * NF + NF + t] = tm * acc1;
    }
    a.w[((size_t)fq * P + j) * NF + t] = s.w[t];
  }
}

// ------------------------------------------------------------------ cross sections
// Block (j, z): partial sums [Cext, Csca, Cabs, Csca_SH] of object j, system z.
__global__ void cross_kernel(CrossArgs a) {
  const int j = blockIdx.x, z = blockIdx.z, t = threadIdx.x;
  a.x += z * a.zvec;
  if(a.xsh) a.xsh += z * a.zvec;
  a.incloc += z * a.zvec;
  a.w += z * a.zw;
  a.ov += z * a.zov;
  a.out += (size_t)z * 4 * a.P;
  const int nf = a.nmax * (a.nmax + 2), S = a.nmax + 1;
  __shared__ double red[4][256];
  double c[4] = {0, 0, 0, 0};
  for(int q = t; q < nf; q += blockDim.x) {
    int n, m;
    unflat(q, n, m);
    size_t b = (size_t)j * 2 * nf;
    cplx x0 = a.x[b + q], x1 = a.x[b + nf + q];
    cplx i0 = a.incloc[b + q], i1 = a.incloc[b + nf + q];
    c[0] += (conj(i0) * x0 + conj(i1) * x1).x;
    double w = a.w[(size_t)j * nf + q];
    c[1] += w * (norm2(x0) + norm2(x1));
    double ca0 = a.ov[(((size_t)OV_CABS * a.P + j) * 2 + 0) * S + n].x;
    double ca1 = a.ov[(((size_t)OV_CABS * a.P + j) * 2 + 1) * S + n].x;
    double m0 = cabs(x0), m1 = cabs(x1);
    c[2] += m0 * m0 * ca0 + m1 * m1 * ca1;
    if(a.xsh) {
      cplx y0 = a.xsh[b + q], y1 = a.xsh[b + nf + q];
      double w2 = a.w[((size_t)a.P + j) * nf + q];
      c[3] += w2 * (norm2(y0) + norm2(y1));
    }
  }
  for(int e = 0; e < 4; ++e) red[e][t] = c[e];
  __syncthreads();
  for(int st = blockDim.x / 2; st > 0; st >>= 1) {
    if(t < st)
      for(int e = 0; e < 4; ++e) red[e][t] += red[e][t + st];
    __syncthreads();
  }
  if(t < 4) a.out[(size_t)j * 4 + t] = red[t][0];
}

// ------------------------------------------------------------------ padding
// Rows/columns N..Np-1 of an Np x Np matrix: identity on the diagonal, zero
// elsewhere, so the padded system has the same solution in its first N rows.
// The border's entries only: the d rows below each column c < N, then the d
// columns behind, d = Np - N.
template <typename T>
__global__ void pad_kernel(T *A, int N, int Np, size_t lda, size_t zs) {
  A += blockIdx.z * zs;
  const int d = Np - N;
  const size_t below = (size_t)d * N, e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(e >= below + (size_t)d * Np) return;
  const size_t c = e < below ? e / d : N + (e - below) / Np;
  const size_t r = e < below ? N + e % d : (e - below) % Np;
  T v{};
  if(r == c) v.x = 1;
  A[c * lda + r] = v;
}

// ------------------------------------------------------------------ launchers
template <int NMAX>
static void launch_pair(const PairArgs &a, hipStream_t st, int nb) {
  hipLaunchKernelGGL(pair_kernel<NMAX>, dim3(a.plist ? a.nlist : a.P * (a.P + 1) / 2, a.V64 || a.V32 ? 2 : 1, nb),
                     dim3(PairCfg<NMAX>::NT), 0, st, a);
}
template <int NMAX>
static void launch_origin(const OriginArgs &a, hipStream_t st, int nb) {
  hipLaunchKernelGGL(origin_kernel<NMAX>, dim3(a.P, a.sh ? 2 : 1, nb), dim3(PairCfg<NMAX>::NT), 0, st, a);
}

#define OMX_NMAX_SWITCH(nmax, F, ...) \
  switch(nmax) {                      \
  case 1: F<1>(__VA_ARGS__); break;   \
  case 2: F<2>(__VA_ARGS__); break;   \
  case 3: F<3>(__VA_ARGS__); break;   \
  case 4: F<4>(__VA_ARGS__); break;   \
  case 5: F<5>(__VA_ARGS__); break;   \
  case 6: F<6>(__VA_ARGS__); break;   \
  case 7: F<7>(__VA_ARGS__); break;   \
  case 8: F<8>(__VA_ARGS__); break;   \
  case 9: F<9>(__VA_ARGS__); break;   \
  case 10: F<10>(__VA_ARGS__); break; \
  default: break;                     \
  }

void run_objects(const ObjArgs &a, hipStream_t st, int nb) {
  hipLaunchKernelGGL(objects_kernel, dim3(a.P, 1, nb), dim3(128), 0, st, a);
}
void run_pairs(const PairArgs &a, hipStream_t st, int nb) { OMX_NMAX_SWITCH(a.nmax, launch_pair, a, st, nb); }
void run_origin(const OriginArgs &a, hipStream_t st, int nb) { OMX_NMAX_SWITCH(a.nmax, launch_origin, a, st, nb); }
void run_cross(const CrossArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(cross_kernel, dim3(a.P, 1, a.nb), dim3(256), 0, st, a);
}
void run_pad64(cplx *A, int N, int Np, size_t lda, hipStream_t st, int nb, size_t zs) {
  if(Np == N) return;
  const size_t n = (size_t)(Np - N) * (N + Np);
  hipLaunchKernelGGL(pad_kernel<double2>, dim3((unsigned)((n + 255) / 256), 1, nb), dim3(256), 0, st, reinterpret_cast<double2 *>(A), N, Np, lda, zs);
}
void run_pad32(float2 *A, int N, int Np, size_t lda, hipStream_t st, int nb, size_t zs) {
  if(Np == N) return;
  const size_t n = (size_t)(Np - N) * (N + Np);
  hipLaunchKernelGGL(pad_kernel<float2>, dim3((unsigned)((n + 255) / 256), 1, nb), dim3(256), 0, st, A, N, Np, lda, zs);
}

// Coefficient tables (CF_*), at index n*n + n + m of each for n <= kCoefN: one
// thread per entry.
__global__ void fill_coef_kernel(double *h) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= kCoefStride) return;
  auto at = [&](int kind) -> double & { return h[kind * kCoefStride + i]; };
  int n = (int)sqrt((double)i);
  const int m = i - n * n - n;
  const double ap = a_plus(n, m), bp = b_plus(n, m);
  at(CF_AP) = ap;
  at(CF_AM) = a_minus(n, m);
  at(CF_BP) = bp;
  at(CF_BM) = b_minus(n, m);
  at(CF_IAP) = ap != 0.0 ? 1.0 / ap : 0.0;
  at(CF_IBP) = bp != 0.0 ? 1.0 / bp : 0.0;
  at(CF_A1) = sqrt((double)((n - m) * (n + m + 1)));
  at(CF_A2) = sqrt((double)((n + m) * (n - m + 1)));
  at(CF_G0) = sqrt((double)((n - m) * (n + m)));
  at(CF_G1) = n > m ? sqrt((double)((n - m) * (n - m - 1))) : 0.0;
  at(CF_G2) = n > -m ? sqrt((double)((n + m) * (n + m - 1))) : 0.0;
  double la = 0.0, lb = 0.0;
  const int l = n, am = m;
  if(am >= 0 && l == am + 1) la = sqrt(2.0 * am + 3.0);
  if(am >= 0 && l >= am + 2) {
    la = sqrt((4.0 * l * l - 1.0) / ((double)l * l - (double)am * am));
    lb = sqrt(((l - 1.0) * (l - 1.0) - (double)am * am) / (4.0 * (l - 1.0) * (l - 1.0) - 1.0));
  }
  at(CF_LEGA) = la;
  at(CF_LEGB) = lb;
  // by degree: entry i of the table is CF_NU, CF_MU or CF_LEGP + d
  const int d = i < CF_MU ? i - CF_NU : i < CF_LEGP ? i - CF_MU : i - CF_LEGP;
  double v = 0.0;
  if(d >= 1 && d <= kCoefN) {
    if(i < CF_MU)
      v = 1.0 / sqrt((double)(d * (d + 1)));
    else if(i < CF_LEGP)
      v = sqrt((double)(2 * d + 1) / (double)((2 * d - 1) * d * (d + 1)));
    else
      v = -sqrt((2.0 * d + 1.0) / (2.0 * d));
  }
  at(CF_DEG) = v;
}
void fill_coef(double *d, hipStream_t st) {
  hipLaunchKernelGGL(fill_coef_kernel, dim3((kCoefStride + 255) / 256), dim3(256), 0, st, d);
}

}  // namespace omx
