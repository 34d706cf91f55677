// omx_capi.hip -- the C ABI (include/optimet_mi355x.h): context, device
// buffers, the update()/solve() sequence of solver::PreconditionedMatrix
// (PreconditionedMatrixSolver.h:45-100) and the iterative solvers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <complex>
#include <functional>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <map>
#include <mutex>
#include <thread>
#include <tuple>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/optimet_mi355x.h"
#include "omx_kernels.hpp"
#include "omx_sh.hpp"

using omx::cplx;

namespace {

thread_local std::string g_err;

struct OmxError : std::runtime_error {
  int code;
  OmxError(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define HIPCHK(x)                                                                                   \
  do {                                                                                              \
    hipError_t e_ = (x);                                                                            \
    if(e_ != hipSuccess)                                                                            \
      throw OmxError(e_ == hipErrorOutOfMemory ? OMX_ERR_MEMORY : OMX_ERR_DEVICE,                   \
                     std::string(#x) + ": " + hipGetErrorString(e_));                               \
  } while(0)

// Device buffer owned by the context.
struct DBuf {
  void *p = nullptr;
  size_t bytes = 0;
  void ensure(size_t b, size_t *total) {
    if(b <= bytes && p) return;
    release(total);
    if(b == 0) return;
    HIPCHK(hipMalloc(&p, b));
    bytes = b;
    *total += b;
  }
  void release(size_t *total) {
    if(p) {
      (void)hipFree(p);
      *total -= bytes;
    }
    p = nullptr;
    bytes = 0;
  }
  template <typename T> T *as() const { return static_cast<T *>(p); }
};

// A part of a DBuf.
struct DView {
  void *p = nullptr;
  template <typename T> T *as() const { return static_cast<T *>(p); }
};

// Device state of the iterations of nb systems (omx_krylov.hip), the pinned words
// that tell the host how each step ended (a ring of kTicks), and their events.
struct KryWs {
  static constexpr int kTicks = 4;
  DBuf c, sc, fl, part, pnrm;
  int *pin = nullptr;    // [kTicks][nb][2], then the final scalars, flags and two status words
  size_t pin_bytes = 0;
  hipEvent_t ev[kTicks] = {};
  static size_t tick_ints(int nb) { return 2 * (size_t)nb; }
  void ensure(int n, int m, int nb, size_t *T) {
    const size_t blk = omx::kry_blocks(n);
    c.ensure(sizeof(cplx) * omx::kry_cplx(m) * nb, T);
    sc.ensure(sizeof(double) * omx::KS_COUNT * nb, T);
    fl.ensure(sizeof(int) * omx::KF_COUNT * nb, T);
    part.ensure(sizeof(cplx) * 2 * nb * blk * (m + 2), T);
    pnrm.ensure(sizeof(double) * 2 * nb * blk, T);
    const size_t b =
        sizeof(double) * omx::KS_COUNT * nb + sizeof(int) * (omx::KF_COUNT * nb + kTicks * tick_ints(nb) + 2);
    if(pin_bytes < b) {
      if(pin) (void)hipHostFree(pin);
      pin = nullptr;
      pin_bytes = 0;
      HIPCHK(hipHostMalloc(reinterpret_cast<void **>(&pin), b));
      pin_bytes = b;
    }
    for(hipEvent_t &e : ev)
      if(!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  void release(size_t *T) {
    DBuf *b[] = {&c, &sc, &fl, &part, &pnrm};
    for(DBuf *x : b) x->release(T);
    if(pin) (void)hipHostFree(pin);
    pin = nullptr;
    pin_bytes = 0;
    for(hipEvent_t &e : ev) {
      if(e) (void)hipEventDestroy(e);
      e = nullptr;
    }
  }
};

// Normwise backward error accepted from a refinement that stopped above its
// residual band: 1000 units of FP64 roundoff.
const double kBackwardErrorBound = 1e3 * 1.1e-16;

// The inner solve of OMX_SOLVER_GMRES32_IR: one GMRES cycle of at most
// kInnerSteps steps on the complex-FP32 copy, stopped at kInnerTol relative
// residual (the FP32 matrix holds S to about 6e-8, so the inner solve can
// gain about six digits per outer step).
constexpr int kInnerSteps = 30;
constexpr double kInnerTol = 1e-6;

constexpr int kMarkN = 9216;  // see omx_solve
constexpr int kSymN = 8192;   // see sym_args
// OMX_SOLVER_AUTO: systems of order N >= kAutoKrylovN start with the mixed
// Krylov, within a budget of outer steps whose matvecs cost what the mixed LU
// would (8/3 N^3 flop at about 140 TFLOP/s against an 8 N^2-byte product at
// about 6 TB/s: 0.0143 N products, kInnerSteps + 1 of them per outer step),
// and fall back to the mixed LU + refinement on the same matrices when it
// does not converge; smaller systems go to the LU directly.
constexpr int kAutoKrylovN = 16384;
inline int auto_krylov_steps(int N) { return std::max(4, (int)(0.0143 * N / (kInnerSteps + 1))); }
// Below kAutoKrylovN, with the second harmonic: V's mixed LU starts at once on
// the second stream pair (V does not depend on the fundamental solution), and
// S is first tried with FP64 GMRES beside it, so that S's solve is hidden
// while it takes less than V's factorisation.  Its budget is the products
// that cost what an LU would (8/3 N^3 flop at about 125 TFLOP/s against a
// 16 N^2-byte FP64 product at about 6 TB/s: N / 125); S falls back to its own
// mixed LU when GMRES has not converged by then.
inline int auto_gmres64_steps(int N) { return std::max(20, N / 125); }
// Batched sweeps take the same rule (S by lockstep FP64 GMRES beside V's
// batched factorisation, within twice that budget) from this order on; below
// it the budget (2 N / 125 < 33 products) is under what such systems need.
constexpr int kSweepKrylovN = 2048;

const double kMu0 = 4.0 * omx::kPi * 1e-7;
const double kEps0 = 1.0 / (kMu0 * omx::kC0 * omx::kC0);

}  // namespace

struct omx_context {
  int device = 0;
  hipStream_t st = nullptr;
  hipEvent_t ev[8];
  size_t total = 0;
  // geometry
  int P = 0, nmax = 0, nf = 0, N = 0, Np = 0;
  std::vector<double> xyz, radius;
  std::vector<cplx> eps, mu, eps_sh, ksippp, ksiparppar, gamma;  // absolute eps, mu; relative ones kept below
  cplx bg_eps_r = omx::mk(1.0), bg_mu_r = omx::mk(1.0);
  bool have_geom = false, have_exc = false;
  // excitation
  double lambda = 0, theta = 0, phi = 0;
  cplx eth = omx::mk(1.0), eph = omx::mk(0.0);
  int sh = 0;
  // solver
  int kind = OMX_SOLVER_LU64;
  int kind_req = OMX_SOLVER_LU64;  // as set; OMX_SOLVER_AUTO resolves into kind at each update
  int auto_budget = 0;             // outer Krylov steps of OMX_SOLVER_AUTO (0: the cost model)
  bool krylov_s = false;           // OMX_SOLVER_AUTO: S tried with FP64 GMRES beside V's factorisation
  bool autotune = true;            // sweeps and solves pick their bulk product and triangular solves by timing
  bool tuned = false, tuned_split = true;  // the single-system choice of the last update
  int pivot = OMX_PIVOT_BLOCK;
  // fraction of S's columns factored before V's factorisation starts
  // (OMX_SH_OVERLAP overrides; 0 starts both together)
  double sh_overlap = 0.5;
  // OMX_SOLVER_AUTO with S by GMRES: fraction of V's columns factored before
  // S's GMRES starts (OMX_KRYLOV_MARK overrides; 0 starts both together), from
  // N = kMarkN on by default
  double krylov_mark = -1.0;
  int lu32_gemm = OMX_GEMM_BF16X3;
  int fallbacks = 0;
  double tol = 1e-16;
  int maxit = 300, restart = 40;
  // state
  bool updated = false, solved = false;
  bool factored = false, factored_sh = false;
  bool dirty32 = false, dirty32_sh = false;  // the FP32 matrix holds factors, not S (V)
  int cg_nmax = 0;
  // device buffers
  DBuf d_geo;  // the geometry's arrays, one after another (upload_geometry)
  DView d_xyz, d_radius, d_eps, d_mu, d_eps_sh, d_kppp, d_kpar, d_gam;
  DBuf d_sph, d_ov, d_inc, d_incloc, d_Q, d_w,
      d_coef, d_S64, d_S32, d_V64, d_V32, d_x, d_xsh, d_xint, d_xintsh, d_K, d_K1, d_cross, d_cg, d_abscoef, d_abssh,
      d_absbes,
      d_fpts, d_fout, d_fown, d_fpart;
  DBuf d_perm, d_cand, d_map, d_status, d_wlu;
  hipStream_t aux = nullptr;
  hipEvent_t lu_ev[4] = {nullptr, nullptr, nullptr, nullptr};
  // the second-harmonic system's own streams, events, status and maps, so
  // its factorisation can run beside the fundamental solve
  hipStream_t st2 = nullptr, aux2 = nullptr;
  hipEvent_t lu_ev2[4] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t xev[4] = {nullptr, nullptr, nullptr, nullptr};
  DBuf d_status2, d_map2;
  std::vector<hipEvent_t> pev2;
  omx::LuProf prof2{};
  DBuf d_basis, d_basisZ, d_w1, d_w2, d_r, d_nrm, d_gpart, d_sym;
  KryWs kry;
  // pinned host staging of the geometry, and the event after its last copy
  double *geo_pin = nullptr;
  int geo_pin_n = 0;
  // pinned staging of the solution vectors
  char *out_pin = nullptr;
  size_t out_pin_bytes = 0;
  hipEvent_t geo_ev = nullptr;
  hipEvent_t mv_ev[2] = {nullptr, nullptr};  // around a product, with profiling on
  // omx_update's times (start, objects done, assembly done) and its joins
  bool upd_timed = false;
  hipEvent_t uev[3] = {nullptr, nullptr, nullptr}, ujoin[2] = {nullptr, nullptr};
  omx::LuWork lu{}, lu_sh{};
  bool links_room = false;  // alloc_lu leaves room for links
  bool profile = false;
  std::vector<hipEvent_t> pev;
  omx::LuProf prof{};
  double prof_gemm_ms = 0, prof_panel_ms = 0, prof_flop = 0, prof_total_ms = 0;
  int prof_launches = 0;
  DBuf d_perm2;
  DBuf d_dinv, d_dinv2, d_F64, d_F64sh;  // diagonal-block inverses; FP64 factors (the FP64 matrices stay intact)
  // wavelength sweeps: per-system buffers of one batch ([system][...])
  struct Sweep {
    DBuf S64, S32, V64, V32, F64, F64sh, eps, eps_sh, ov, incloc, Q, w, x, xint, xsh, xintsh, K, K1, cross, abscoef,
        abssh, absbes;
    DBuf perm, perm2, dinv, dinv2, map, status, basis, basisZ, r, w1, w2, gpart, kz, omz, map2, status2;
    KryWs kry;
    void release(size_t *T) {
      DBuf *b[] = {&S64, &S32, &V64, &V32, &F64, &F64sh, &eps, &eps_sh, &ov, &incloc, &Q, &w, &x, &xint, &xsh, &xintsh,
                   &K, &K1, &cross, &abscoef, &abssh, &absbes, &perm, &perm2, &dinv, &dinv2, &map, &status, &basis,
                   &basisZ, &r, &w1, &w2, &gpart, &kz, &omz, &map2, &status2};
      for(DBuf *p : b) p->release(T);
      kry.release(T);
    }
  } sw;
  // ACA-compressed operators S (0) and V (1) of OMX_SOLVER_ACA_GMRES
  struct AcaMat {
    int n = 0, P = 0, G = 0, naca = 0, ndense = 0, rmax = 0;
    double rsum = 0, bytes = 0, ref_mb = 0;
    std::vector<int> rank;           // [i P + j]: r, -1 dense, 0 diagonal
    std::vector<const cplx *> where;  // [i P + j]: U (compressed) or the block (dense)
    std::vector<DBuf> pools;          // factor pools, one per compression chunk (kept for the next build)
    DBuf dense, desc, rowptr, acalist, t, part;
    bool built = false;
    // forgets the operator; its device buffers stay for the next one of its shape (a
    // scan rebuilds it at every wavelength; freeing and mapping gigabytes again took
    // 6 of 28 ms per solve of 300 spheres at nmax 5, and 140 of 173 ms in a
    // process that had solved larger systems before)
    void reset() {
      rank.clear();
      where.clear();
      built = false;
      bytes = ref_mb = rsum = 0;
      naca = ndense = rmax = 0;
    }
    void release(size_t *T) {
      for(auto &p : pools) p.release(T);
      pools.clear();
      DBuf *b[] = {&dense, &desc, &rowptr, &acalist, &t, &part};
      for(DBuf *x : b) x->release(T);
      reset();
    }
  } aca[2];
  DBuf d_acaA, d_acaU, d_acaV, d_acaR, d_acaOff, d_plist;
  // the inner GMRES of OMX_SOLVER_GMRES32_IR: its own basis and vectors
  struct GmresWs {
    DBuf basis, r, w1, gpart;
    KryWs kry;
    void release(size_t *T) {
      DBuf *b[] = {&basis, &r, &w1, &gpart};
      for(DBuf *x : b) x->release(T);
      kry.release(T);
    }
  } ws_in;
  // Captured factorisations (omx_set_graphs): executable graphs of S's
  // factorisation (s1, then s2 after V's start mark) and V's, and the state
  // they were captured for; one set for single solves, one for sweep chunks
  struct FactorGraphs {
    hipGraphExec_t s1 = nullptr, s2 = nullptr, v = nullptr;
    std::vector<uintptr_t> key;
    void reset() {
      hipGraphExec_t *g[] = {&s1, &s2, &v};
      for(hipGraphExec_t *x : g) {
        if(*x) (void)hipGraphExecDestroy(*x);
        *x = nullptr;
      }
      key.clear();
    }
  } fg, fg_sweep;
  bool graphs = false;
  int graph_captures = 0, graph_launches = 0;
  omx_stats stats{};
  void *scratch = nullptr;  // this device's address of the no-allocation solve's scratch array
  long long mv_calls = 0;  // FP64 matrix-vector products since the last omx_set_profile
  double mv_ms = 0, mv_bytes = 0;
  double omega() const { return omx::kC0 * (2.0 * omx::kPi / lambda); }
  cplx waveK() const {
    std::complex<double> b = std::sqrt(std::complex<double>(bg_eps_r.x, bg_eps_r.y) *
                                       std::complex<double>(bg_mu_r.x, bg_mu_r.y));
    double k0 = 2.0 * omx::kPi / lambda;
    return omx::mk(k0 * b.real(), k0 * b.imag());
  }
};

namespace {

template <typename F> int guard(F &&f) {
  try {
    f();
    return OMX_OK;
  } catch(OmxError &e) {
    g_err = e.what();
    return e.code;
  } catch(std::exception &e) {
    g_err = e.what();
    return OMX_ERR_ARG;
  }
}

// A call that fails leaves none of its work in flight.  The status words of a
// factorisation are looked at with the first steps of its refinement enqueued, and V's
// factorisation runs on the second stream while S's solve may fail; the next call
// starts on the first stream, in the same workspaces.
struct DrainOnError {
  omx_context *c;
  int before = std::uncaught_exceptions();
  ~DrainOnError() {
    if(std::uncaught_exceptions() <= before) return;
    for(hipStream_t s : {c->st, c->aux, c->st2, c->aux2}) (void)hipStreamSynchronize(s);
  }
};

cplx C(const double *p, int i) { return omx::mk(p[2 * i], p[2 * i + 1]); }

bool use32(int kind) { return kind == OMX_SOLVER_LU32_IR || kind == OMX_SOLVER_GMRES32_IR; }
bool is_lu(int kind) { return kind == OMX_SOLVER_LU64 || kind == OMX_SOLVER_LU32_IR; }

void alloc_lu(omx_context *c, omx::LuWork &w, DBuf &perm, DBuf &dinv, bool second) {
  const int Np = c->Np;
  const int gmax = (Np + omx::kPanelRows - 1) / omx::kPanelRows + 1;
  dinv.ensure(sizeof(cplx) * omx::dinv_elems(Np, c->links_room), &c->total);
  perm.ensure(sizeof(int) * Np, &c->total);
  // tournament scratch: one half per system, as S and V may be factored
  // at the same time
  c->d_cand.ensure(sizeof(int) * 4 * gmax * omx::kNB, &c->total);
  c->d_wlu.ensure(sizeof(cplx) * 2 * omx::kNB * omx::kNB, &c->total);
  if(!second) {
    c->d_map.ensure(sizeof(int) * (3 * ((size_t)Np + 2 * omx::kNB)), &c->total);
    c->d_status.ensure(64, &c->total);
  } else {
    c->d_map2.ensure(sizeof(int) * (3 * ((size_t)Np + 2 * omx::kNB)), &c->total);
    c->d_status2.ensure(64, &c->total);
  }
  DBuf &map = second ? c->d_map2 : c->d_map;
  DBuf &status = second ? c->d_status2 : c->d_status;
  HIPCHK(hipMemsetAsync(status.p, 0, 64, c->st));
  w = omx::LuWork{};
  w.perm = perm.as<int>();
  const int half = second ? 1 : 0;
  w.cand[0] = c->d_cand.as<int>() + (2 * half) * gmax * omx::kNB;
  w.cand[1] = c->d_cand.as<int>() + (2 * half + 1) * gmax * omx::kNB;
  w.mdst = map.as<int>();
  w.msrc = map.as<int>() + (Np + 2 * omx::kNB);
  w.mcnt = map.as<int>() + 2 * (Np + 2 * omx::kNB);
  w.status = status.as<int>();
  w.wlu = c->d_wlu.as<cplx>() + (size_t)half * omx::kNB * omx::kNB;
  w.dinv = dinv.p;
  w.pivot = c->pivot;
  hipEvent_t *ev = second ? c->lu_ev2 : c->lu_ev;
  w.aux = second ? c->aux2 : c->aux;
  w.ev_next = ev[0];
  w.ev_piv = ev[1];
  w.ev_bulk = ev[2];
  w.ev_pan = ev[3];
  w.gmax = gmax;
}

// The triangular-solve variant of a system's factors; FP64 ones solved by variant 1
// take links.
void set_trsv(omx_context *c, omx::LuWork &w, DBuf &dinv, int trsv) {
  w.trsv = trsv;
  w.links = c->kind == OMX_SOLVER_LU64 && trsv == 1;
  dinv.ensure(sizeof(cplx) * omx::dinv_elems(c->Np, w.links), &c->total);
  w.dinv = dinv.p;
}

// The geometry's arrays on the device in one copy: mu, eps, eps_sh and the
// susceptibilities (complex, P each), then the centres and radii.  The staging
// is pinned, and rewritten only once the copy before has left it.
constexpr int kGeoDoubles = 6 * 2 + 3 + 1;
void upload_geometry(omx_context *c) {
  if(!c->d_coef.p) {  // the assembly's coefficient tables, once per context
    c->d_coef.ensure(sizeof(double) * omx::CF_COUNT * omx::kCoefStride, &c->total);
    omx::fill_coef(c->d_coef.as<double>(), c->st);
  }
  const size_t P = c->P;
  const int n = kGeoDoubles * c->P;
  if(c->geo_pin_n < n) {
    HIPCHK(hipEventSynchronize(c->geo_ev));
    if(c->geo_pin) (void)hipHostFree(c->geo_pin);
    c->geo_pin = nullptr;
    c->geo_pin_n = 0;
    HIPCHK(hipHostMalloc(reinterpret_cast<void **>(&c->geo_pin), sizeof(double) * n));
    c->geo_pin_n = n;
  }
  HIPCHK(hipEventSynchronize(c->geo_ev));
  DView *cv[] = {&c->d_mu, &c->d_eps, &c->d_eps_sh, &c->d_kppp, &c->d_kpar, &c->d_gam};
  const std::vector<cplx> *src[] = {&c->mu, &c->eps, &c->eps_sh, &c->ksippp, &c->ksiparppar, &c->gamma};
  double *h = c->geo_pin, *d = c->d_geo.as<double>();
  for(int e = 0; e < 6; ++e) {
    std::memcpy(h + 2 * P * e, src[e]->data(), sizeof(cplx) * P);
    cv[e]->p = d + 2 * P * e;
  }
  std::memcpy(h + 12 * P, c->xyz.data(), sizeof(double) * 3 * P);
  std::memcpy(h + 15 * P, c->radius.data(), sizeof(double) * P);
  c->d_xyz.p = d + 12 * P;
  c->d_radius.p = d + 15 * P;
  HIPCHK(hipMemcpyAsync(d, h, sizeof(double) * n, hipMemcpyHostToDevice, c->st));
  HIPCHK(hipEventRecord(c->geo_ev, c->st));
}

// (Re)allocates every size-dependent buffer.
void alloc_all(omx_context *c) {
  const int P = c->P, nf = c->nf, N = c->N, Np = c->Np, S = c->nmax + 1;
  size_t *T = &c->total;
  c->d_geo.ensure(sizeof(double) * kGeoDoubles * P, T);
  c->d_sph.ensure(sizeof(double) * omx::kSphDoubles * P, T);
  c->d_ov.ensure(sizeof(cplx) * omx::OV_COUNT * P * 2 * S, T);
  c->d_inc.ensure(sizeof(cplx) * 2 * nf, T);
  c->d_incloc.ensure(sizeof(cplx) * N, T);
  c->d_Q.ensure(sizeof(cplx) * Np, T);
  c->d_w.ensure(sizeof(double) * 2 * P * nf, T);
  c->d_x.ensure(sizeof(cplx) * Np, T);
  c->d_xsh.ensure(sizeof(cplx) * Np, T);
  c->d_xint.ensure(sizeof(cplx) * Np, T);
  c->d_xintsh.ensure(sizeof(cplx) * Np, T);
  c->d_K.ensure(sizeof(cplx) * Np, T);
  c->d_K1.ensure(sizeof(cplx) * Np, T);
  c->d_cross.ensure(sizeof(double) * 4 * P, T);
  c->d_abscoef.ensure(sizeof(cplx) * P * nf, T);
  c->d_abssh.ensure(sizeof(double) * P, T);
  c->d_absbes.ensure(sizeof(cplx) * P * omx::kAbsBes, T);
  c->d_r.ensure(sizeof(cplx) * Np, T);
  c->d_w1.ensure(sizeof(cplx) * Np, T);
  c->d_w2.ensure(sizeof(cplx) * Np, T);
  c->d_gpart.ensure(sizeof(cplx) * Np * omx::gemv_part_rows(1), T);
  c->d_nrm.ensure(sizeof(double) * 256, T);
}

// Gives back the compression's staging (not needed by the operators).
void aca_release_staging(omx_context *c) {
  for(DBuf *x : {&c->d_acaA, &c->d_acaU, &c->d_acaV}) x->release(&c->total);
}

void alloc_matrices(omx_context *c) {
  const size_t n2 = (size_t)c->Np * c->Np;
  size_t *T = &c->total;
  if(c->kind != OMX_SOLVER_ACA_GMRES) aca_release_staging(c);
  // FP64 matrix: factorised (LU64), streamed (GMRES) or the residual operator
  // (IR); the compressed operators of ACA replace it
  bool need64 = c->kind != OMX_SOLVER_ACA_GMRES;
  bool need32 = use32(c->kind);
  if(need64) c->d_S64.ensure(sizeof(cplx) * n2, T); else c->d_S64.release(T);
  if(need32) c->d_S32.ensure(sizeof(float2) * n2, T); else c->d_S32.release(T);
  if(c->sh) {
    if(need64) c->d_V64.ensure(sizeof(cplx) * n2, T); else c->d_V64.release(T);
    if(need32) c->d_V32.ensure(sizeof(float2) * n2, T); else c->d_V32.release(T);
  } else {
    c->d_V64.release(T);
    c->d_V32.release(T);
  }
  const bool f64 = c->kind == OMX_SOLVER_LU64;
  if(f64) c->d_F64.ensure(sizeof(cplx) * n2, T); else c->d_F64.release(T);
  if(f64 && c->sh) c->d_F64sh.ensure(sizeof(cplx) * n2, T); else c->d_F64sh.release(T);
  c->d_basis.ensure(sizeof(cplx) * (size_t)c->Np * (c->restart + 1), T);
  // preconditioned (flexible) GMRES keeps M^{-1} v_j: the LU kinds and the mixed Krylov
  const bool flex = is_lu(c->kind) || c->kind == OMX_SOLVER_GMRES32_IR;
  if(flex) c->d_basisZ.ensure(sizeof(cplx) * (size_t)c->Np * (c->restart + 1), T);
  else c->d_basisZ.release(T);
  if(c->kind == OMX_SOLVER_GMRES32_IR) {
    auto &w = c->ws_in;
    const size_t Np = (size_t)c->Np;
    w.basis.ensure(sizeof(cplx) * Np * (kInnerSteps + 1), T);
    w.r.ensure(sizeof(cplx) * Np, T);
    w.w1.ensure(sizeof(cplx) * Np, T);
    w.gpart.ensure(sizeof(cplx) * Np * omx::gemv_part_rows(1), T);
  } else {
    c->ws_in.release(T);
  }
  alloc_lu(c, c->lu, c->d_perm, c->d_dinv, false);
  if(c->sh) alloc_lu(c, c->lu_sh, c->d_perm2, c->d_dinv2, true);
}

float elapsed(omx_context *c, int a, int b) {
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev[a], c->ev[b]);
  return ms;
}

// ------------------------------------------------------------------ ACA
// Scattering_matrix_ACA_FF / _SH (PreconditionedMatrix.cpp:489-551,
// 696-759) on the device: block (i, j != i) is compressed when
// |c_i - c_j| >= 2 (r_i + r_j) (:526; the distance of Tools::findDistance on
// the reader's spherical coordinates, Tools.cpp:30-44) and kept dense
// otherwise.  Dense blocks are assembled by the pair kernel straight into
// their pool; compressed blocks are assembled chunk by chunk into n x n
// staging slots, compressed there (aca_kernel, at most n terms each) and
// their factors packed into a pool of exactly sum 2 n r entries per chunk,
// so the full matrix never exists on the device.
constexpr double kAcaEps = 1e-3;            // PreconditionedMatrix.cpp:774
constexpr double kAcaStagingBytes = 1.5e9;  // assembly + factor staging of one chunk

// Gives back the compressed operators and their staging (another solver kind,
// or omx_trim).
void aca_release(omx_context *c) {
  c->aca[0].release(&c->total);
  c->aca[1].release(&c->total);
  aca_release_staging(c);
}

// A buffer kept from the operator before: allocated again when it is too small or
// more than twice what is wanted, with spare (want) where memory allows.
void fit(DBuf &b, size_t need, size_t want, size_t *T) {
  if(b.p && b.bytes >= need && b.bytes <= 2 * want) return;
  b.release(T);
  try {
    b.ensure(want, T);
  } catch(OmxError &e) {
    if(e.code != OMX_ERR_MEMORY || want == need) throw;
    (void)hipGetLastError();
    b.ensure(need, T);
  }
}

void aca_build(omx_context *c, bool shf) {
  omx_context::AcaMat &m = c->aca[shf ? 1 : 0];
  size_t *T = &c->total;
  const int P = c->P, nmax = c->nmax, n = 2 * c->nf;
  // kept between updates of one cluster's shape (a scan, an optimiser's loop) only
  if(m.P && (m.P != P || m.n != n)) {
    m.release(T);
    aca_release_staging(c);
  }
  m.reset();
  const size_t n2 = (size_t)n * n;
  hipStream_t st = c->st;
  m.n = n;
  m.P = P;
  m.rank.assign((size_t)P * P, 0);
  m.where.assign((size_t)P * P, nullptr);
  // centres through the reader's Cartesian -> spherical -> Cartesian round trip
  std::vector<double> ctr(3 * (size_t)P);
  for(int i = 0; i < P; ++i) {
    const double x = c->xyz[3 * i], y = c->xyz[3 * i + 1], z = c->xyz[3 * i + 2];
    const double r = std::sqrt(x * x + y * y + z * z);
    const double th = r > 0.0 ? std::acos(z / r) : 0.0, ph = r > 0.0 ? std::atan2(y, x) : 0.0;
    ctr[3 * i] = r * std::sin(th) * std::cos(ph);
    ctr[3 * i + 1] = r * std::sin(th) * std::sin(ph);
    ctr[3 * i + 2] = r * std::cos(th);
  }
  // unordered pairs i < j; blocks 2 b (i, j) and 2 b + 1 (j, i) of pair b
  std::vector<int> dl, al;
  for(int i = 0; i < P; ++i)
    for(int j = i + 1; j < P; ++j) {
      const double d = std::sqrt(std::pow(ctr[3 * j] - ctr[3 * i], 2.0) + std::pow(ctr[3 * j + 1] - ctr[3 * i + 1], 2.0) +
                                 std::pow(ctr[3 * j + 2] - ctr[3 * i + 2], 2.0));
      if(d >= 2.0 * (c->radius[i] + c->radius[j])) {
        al.push_back(i * P + j);
      } else {
        dl.push_back(i * P + j);
        m.rank[(size_t)i * P + j] = m.rank[(size_t)j * P + i] = -1;
      }
    }
  m.ndense = 2 * (int)dl.size();
  m.naca = 2 * (int)al.size();
  // block 2 b + h of a pair list as i P + j
  auto block = [P](const std::vector<int> &l, size_t b) {
    const int pid = l[b / 2];
    return b & 1 ? (size_t)(pid % P) * P + pid / P : (size_t)pid;
  };
  cplx k = c->waveK();
  if(shf) k = omx::mk(2.0 * k.x, 2.0 * k.y);  // PreconditionedMatrix.cpp:725
  omx::PairArgs base{P, nmax, shf ? omx::OV_TSH : omx::OV_T, k, c->d_sph.as<double>(), c->d_ov.as<cplx>(),
                     c->d_coef.as<double>(), (size_t)n, nullptr, nullptr};
  base.zblk = n2;  // S_ij of pair b at 2 b n2, S_ji behind it
  const size_t listn = std::max(dl.size(), (size_t)1);
  size_t used = 0;  // pools
  if(!m.ndense) m.dense.release(T);
  if(m.ndense) {
    fit(m.dense, sizeof(cplx) * n2 * m.ndense, sizeof(cplx) * n2 * m.ndense, T);
    c->d_plist.ensure(sizeof(int) * listn, T);
    HIPCHK(hipMemcpyAsync(c->d_plist.p, dl.data(), sizeof(int) * dl.size(), hipMemcpyHostToDevice, st));
    omx::PairArgs pa = base;
    pa.S64 = m.dense.as<cplx>();
    pa.plist = c->d_plist.as<int>();
    pa.nlist = (int)dl.size();
    omx::run_pairs(pa, st);
    for(int b = 0; b < m.ndense; ++b) m.where[block(dl, b)] = m.dense.as<cplx>() + b * n2;
    HIPCHK(hipStreamSynchronize(st));  // dl and the list buffer are reused below
  }
  if(m.naca) {
    // blocks of a chunk: whole pairs
    const int C = 2 * (int)std::max<double>(1.0, std::min<double>(m.naca / 2, kAcaStagingBytes / (96.0 * n2)));
    for(DBuf *b : {&c->d_acaA, &c->d_acaU, &c->d_acaV}) fit(*b, sizeof(cplx) * n2 * C, sizeof(cplx) * n2 * C, T);
    c->d_acaR.ensure(sizeof(int) * C, T);
    c->d_acaOff.ensure(sizeof(size_t) * C, T);
    c->d_plist.ensure(sizeof(int) * std::max((size_t)C, listn), T);
    std::vector<int> rk(C);
    std::vector<size_t> off(C);
    size_t chunk = 0;
    for(int b0 = 0; b0 < m.naca; b0 += C, ++chunk) {
      const int nb = std::min(C, m.naca - b0);
      HIPCHK(hipMemcpyAsync(c->d_plist.p, al.data() + b0 / 2, sizeof(int) * (nb / 2), hipMemcpyHostToDevice, st));
      omx::PairArgs pa = base;
      pa.S64 = c->d_acaA.as<cplx>();
      pa.plist = c->d_plist.as<int>();
      pa.nlist = nb / 2;
      omx::run_pairs(pa, st);
      omx::AcaArgs aa{n, nb, kAcaEps, c->d_acaA.as<cplx>(), c->d_acaU.as<cplx>(), c->d_acaV.as<cplx>(),
                      c->d_acaR.as<int>()};
      omx::run_aca(aa, st);
      HIPCHK(hipMemcpyAsync(rk.data(), c->d_acaR.p, sizeof(int) * nb, hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      size_t tot = 0;
      for(int b = 0; b < nb; ++b) {
        if(rk[b] < 1 || rk[b] > n) throw OmxError(OMX_ERR_DEVICE, "ACA returned rank " + std::to_string(rk[b]));
        off[b] = tot;
        tot += 2 * (size_t)n * rk[b];
      }
      if(m.pools.size() <= chunk) m.pools.emplace_back();
      DBuf &pool = m.pools[chunk];
      // an eighth to spare when it has to grow: ranks vary a little from one
      // wavelength to the next
      fit(pool, sizeof(cplx) * tot, sizeof(cplx) * (tot + tot / 8), T);
      HIPCHK(hipMemcpyAsync(c->d_acaOff.p, off.data(), sizeof(size_t) * nb, hipMemcpyHostToDevice, st));
      omx::run_aca_pack(c->d_acaU.as<cplx>(), c->d_acaV.as<cplx>(), n, nb, c->d_acaR.as<int>(), pool.as<cplx>(),
                        c->d_acaOff.as<size_t>(), st);
      for(int b = 0; b < nb; ++b) {
        m.rank[block(al, b0 + b)] = rk[b];
        m.where[block(al, b0 + b)] = pool.as<cplx>() + off[b];
      }
      HIPCHK(hipStreamSynchronize(st));  // off, rk and the list buffer are reused
    }
    used = chunk;
  }
  for(; m.pools.size() > used; m.pools.pop_back()) m.pools.back().release(T);
  // descriptors, block row by block row
  std::vector<omx::AcaDesc> desc;
  std::vector<int> rowptr(P + 1, 0), acalist;
  int toff = 0;
  m.bytes = 0;
  m.ref_mb = (double)P * n2 * 16.0 / 1e6;  // identity blocks
  for(int i = 0; i < P; ++i) {
    rowptr[i] = (int)desc.size();
    for(int j = 0; j < P; ++j) {
      const int r = m.rank[(size_t)i * P + j];
      if(i == j) continue;
      omx::AcaDesc d{m.where[(size_t)i * P + j], j, r, 0};
      if(r > 0) {
        d.toff = toff;
        toff += r;
        acalist.push_back((int)desc.size());
        m.bytes += 32.0 * n * r;
        m.ref_mb += 2.0 * n * r * 16.0 / 1e6;
        m.rmax = std::max(m.rmax, r);
        m.rsum += r;
      } else {
        m.bytes += 16.0 * n2;
        m.ref_mb += n2 * 16.0 / 1e6;
      }
      desc.push_back(d);
    }
  }
  rowptr[P] = (int)desc.size();
  // one round of the chip, six workgroups a CU
  m.G = P > 1 ? std::max(1, std::min((P + 2) / 4, 1536 / P)) : 0;
  m.desc.ensure(sizeof(omx::AcaDesc) * std::max<size_t>(desc.size(), 1), T);
  m.rowptr.ensure(sizeof(int) * (P + 1), T);
  m.acalist.ensure(sizeof(int) * std::max<size_t>(acalist.size(), 1), T);
  m.t.ensure(sizeof(cplx) * std::max(toff, 1), T);
  m.part.ensure(sizeof(cplx) * (size_t)std::max(m.G, 1) * P * n, T);
  if(!desc.empty())
    HIPCHK(hipMemcpyAsync(m.desc.p, desc.data(), sizeof(omx::AcaDesc) * desc.size(), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(m.rowptr.p, rowptr.data(), sizeof(int) * (P + 1), hipMemcpyHostToDevice, st));
  if(!acalist.empty())
    HIPCHK(hipMemcpyAsync(m.acalist.p, acalist.data(), sizeof(int) * acalist.size(), hipMemcpyHostToDevice, st));
  HIPCHK(hipStreamSynchronize(st));  // the host vectors end here
  m.built = true;
}

// y = S x (V x) with the compressed operator, on stream st.
void aca_apply(omx_context *c, bool shf, const cplx *x, cplx *y, hipStream_t st) {
  omx_context::AcaMat &m = c->aca[shf ? 1 : 0];
  if(!m.built) throw OmxError(OMX_ERR_STATE, "no compressed operator");
  omx::AcaOp op{c->P, m.n, c->N, c->Np, m.G, m.desc.as<omx::AcaDesc>(), m.rowptr.as<int>(), m.acalist.as<int>(),
                m.naca, m.t.as<cplx>(), m.part.as<cplx>()};
  omx::aca_matvec(op, x, y, st);
}

// The error that a factorisation's status words tell of, if any.
void throw_status(const int *s) {
  if(s[1]) throw OmxError(OMX_ERR_DEVICE, "device wait timed out (code " + std::to_string(s[1]) + ")");
  if(s[0]) throw OmxError(OMX_ERR_SINGULAR, "zero pivot at column " + std::to_string(s[0] - 1));
}

// ------------------------------------------------------------------ GMRES
// Right-preconditioned restarted GMRES in FP64 with classical Gram-Schmidt (two
// passes), in flexible form: the preconditioned vectors M^{-1} v_j are kept, so
// the end of a cycle needs no further preconditioner application.  nb systems
// run in lockstep, each with its own Hessenberg matrix and stopping state; one
// that has converged drops out of the products and solves.  The algebra runs on
// the device (omx_krylov.hip); the host only learns, a step later, which systems
// go on.
struct Krylov {
  omx_context *c;
  int n, nb;
  hipStream_t s;
  KryWs &ws;
  cplx *V, *Z;            // bases; Z of the preconditioned vectors (V itself without one)
  cplx *r, *w, *gpart;
  // the operator: FP64 matrices A (sA apart), or their complex-FP32 copy, or a
  // product given as a function
  const cplx *A = nullptr;
  size_t sA = 0;
  const float2 *A32 = nullptr;
  std::function<void(const cplx *, cplx *)> op = nullptr;
  double op_bytes = 0.0;
  // with scratch: the Arnoldi steps' products from half the blocks (the residuals
  // come from the whole matrix)
  omx::SymArgs sym{};
  // out = M^{-1} in for the systems whose flag is set (identity when null)
  std::function<void(const cplx *in, cplx *out, const int *live)> prec = nullptr;
  bool x_zero = false;     // x starts at 0: no product before the first cycle
  bool one_cycle = false;  // and no residual after it (a fixed-cost preconditioner)
  bool batch = false;      // the batched sweeps' stopping rules
  bool lazy = false;       // never enqueue a step that may turn out not to be needed
  const int *status = nullptr;  // the factorisation's status words, looked at once the first step is known
  std::vector<double> res;
  std::vector<int> its;
  int bits = 0;            // binary digits between the residual and its goal, as last known

  // Enqueues A x into gpart (returns the column parts) or w (returns 0).
  int product(const cplx *x, const int *flag, int live, bool step) {
    const bool prof = c->profile;
    if(prof) HIPCHK(hipEventRecord(c->mv_ev[0], s));
    int ns = 0;
    if(op)
      op(x, w);
    else if(step && sym.scratch) {
      omx::SymArgs a = sym;
      a.flag = flag;
      if(A32)
        omx::sym_product(a, A32, x, w, s);
      else
        omx::sym_product(a, A, x, w, s);
    }
    else if(A32)
      ns = omx::gemv_partial(A32, (size_t)c->Np, n, x, gpart, s, flag);
    else
      ns = omx::gemv_partial(A, (size_t)c->Np, n, x, gpart, s, nb, sA, (size_t)n, flag, std::max(1, live));
    if(prof) {
      HIPCHK(hipEventRecord(c->mv_ev[1], s));
      HIPCHK(hipEventSynchronize(c->mv_ev[1]));
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, c->mv_ev[0], c->mv_ev[1]));
      c->mv_ms += ms;
    }
    return ns;
  }
  void count(int live, bool step) {
    if(live < 1) return;
    ++c->mv_calls;
    const double half = step && sym.scratch ? 0.5 : 1.0;
    c->mv_bytes += (op ? op_bytes : half * (A32 ? 8.0 : 16.0) * n * (double)n) * live;
  }
  // Solves A x = b; x holds the initial guesses.  res: the final relative
  // residuals, its: the iterations.  (A one-cycle solve leaves both unread.)
  void solve(const cplx *b, cplx *x, double tol, int maxit, int m) {
    ws.ensure(n, m, nb, &c->total);
    const bool never = lazy || c->profile || op != nullptr;
    omx::KryState st{n,
                     m,
                     nb,
                     0,
                     tol,
                     maxit,
                     ws.c.as<cplx>(),
                     ws.sc.as<double>(),
                     ws.fl.as<int>(),
                     ws.part.as<cplx>(),
                     ws.pnrm.as<double>(),
                     V,
                     prec ? Z : V,
                     (size_t)n * nb,
                     (size_t)n,
                     r,
                     w,
                     (size_t)n};
    const int *live = st.fl + omx::KF_LIVE, *active = st.fl + omx::KF_ACTIVE;
    int tick = -1, known = -1;  // the last event recorded, and the last one waited for
    auto slot = [&](int t) { return ws.pin + (size_t)(t % KryWs::kTicks) * KryWs::tick_ints(nb); };
    auto mark = [&] {
      ++tick;
      HIPCHK(hipEventRecord(ws.ev[tick % KryWs::kTicks], s));
    };
    // waits for the next event: the systems that go on, and the digits left
    int nlive = nb, last_bits = 0, restart = 0;
    double left = 0.0;  // steps to the goal after the last known one, by its gain
    double *hs = reinterpret_cast<double *>(ws.pin + KryWs::kTicks * KryWs::tick_ints(nb));
    int *hf = reinterpret_cast<int *>(hs + omx::KS_COUNT * nb), *hst = hf + omx::KF_COUNT * nb;
    if(status) HIPCHK(hipMemcpyAsync(hst, status, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
    auto wait = [&] {
      const int before = nlive;
      ++known;
      HIPCHK(hipEventSynchronize(ws.ev[known % KryWs::kTicks]));
      if(status && known == 0) throw_status(hst);
      const int *h = slot(known);
      nlive = bits = 0;
      for(int z = 0; z < nb; ++z)
        if(h[2 * z]) {
          ++nlive;
          bits = std::max(bits, h[2 * z + 1]);
        }
      const int gain = last_bits - bits;
      left = known != restart && gain > 0 ? (double)bits / gain : 0.0;
      last_bits = bits;
      if(known != restart) count(before, true);
    };
    int ns = 0;
    if(!x_zero && !one_cycle) {
      ns = product(x, nullptr, nb, false);
      if(op) ns = -1;
      count(nb, false);
    }
    omx::kry_restart(st, b, x, gpart, ns, (size_t)std::max(0, ns) * n, true, batch, slot(tick + 1), s);
    mark();
    if(never) wait();
    while(known < tick || nlive > 0) {
      bool over = false;
      for(int j = 0; j < m && !over; ++j) {
        st.j = j;
        const cplx *vj = V + (size_t)j * st.ldk, *pj = vj;
        if(prec) {
          cplx *zj = Z + (size_t)j * st.ldk;
          prec(vj, zj, live);
          pj = zj;
        }
        ns = product(pj, live, nlive, true);
        omx::kry_step(st, gpart, ns, (size_t)ns * n, slot(tick + 1), s);
        mark();
        // Go on at once when the steps enqueued since the last known one are
        // surely not enough (its gain repeated, and one to spare); otherwise
        // wait for the outcomes, oldest first
        while(known < tick && !over) {
          const int open = tick - known;
          if(!never && j + 1 < m && left > open + 0.5 && open < KryWs::kTicks - 1) break;
          wait();
          over = nlive == 0;
        }
      }
      while(known < tick) wait();
      omx::kry_end_cycle(st, x, !one_cycle, batch, s);
      if(one_cycle) return;
      ns = product(x, active, nb, false);
      if(op) ns = -1;
      count(nb, false);
      omx::kry_restart(st, b, x, gpart, ns, (size_t)std::max(0, ns) * n, false, batch, slot(tick + 1), s);
      mark();
      restart = tick;
      wait();
    }
    HIPCHK(hipMemcpyAsync(hs, st.sc, sizeof(double) * omx::KS_COUNT * nb, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(hf, st.fl, sizeof(int) * omx::KF_COUNT * nb, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    res.resize(nb);
    its.resize(nb);
    for(int z = 0; z < nb; ++z) {
      res[z] = hs[omx::KS_COUNT * z + omx::KS_RES];
      its[z] = hf[omx::KF_COUNT * z + omx::KF_ITS];
    }
  }
};

hipStream_t sys_stream(const omx_context *c, bool shf) { return shf ? c->st2 : c->st; }

void check_status(omx_context *c, bool shf = false) {
  int s[2] = {0, 0};
  hipStream_t st = sys_stream(c, shf);
  HIPCHK(hipMemcpyAsync(s, (shf ? c->d_status2 : c->d_status).p, sizeof(s), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  throw_status(s);
}

omx::LuProf *prof_begin(omx_context *c, bool shf) {
  if(!c->profile) return nullptr;
  std::vector<hipEvent_t> &pev = shf ? c->pev2 : c->pev;
  omx::LuProf &prof = shf ? c->prof2 : c->prof;
  int cap = c->Np / omx::kNB + 1;
  if((int)pev.size() < 4 * cap + 2) {
    for(auto e : pev) (void)hipEventDestroy(e);
    pev.assign(4 * cap + 2, nullptr);
    for(auto &e : pev) HIPCHK(hipEventCreate(&e));
  }
  prof.ev = pev.data() + 2;
  prof.cap = cap;
  HIPCHK(hipEventRecord(pev[0], sys_stream(c, shf)));
  return &prof;
}
void prof_end(omx_context *c, bool shf) {
  if(!c->profile) return;
  std::vector<hipEvent_t> &pev = shf ? c->pev2 : c->pev;
  omx::LuProf &prof = shf ? c->prof2 : c->prof;
  HIPCHK(hipEventRecord(pev[1], sys_stream(c, shf)));
  HIPCHK(hipEventSynchronize(pev[1]));
  float ms = 0;
  for(int i = 0; i < prof.used; ++i) {
    hipEvent_t *e = prof.ev + 4 * i;
    HIPCHK(hipEventElapsedTime(&ms, e[0], e[1]));
    c->prof_panel_ms += ms;
    HIPCHK(hipEventElapsedTime(&ms, e[2], e[3]));
    c->prof_gemm_ms += ms;
  }
  HIPCHK(hipEventElapsedTime(&ms, pev[0], pev[1]));
  c->prof_total_ms += ms;
  c->prof_flop += prof.gemm_flop;
  c->prof_launches += prof.gemm_launches;
}

// Enqueues the factorisation of S (V) with pivot mode pv on the system's
// stream; the status is checked by the caller.
void factor_enqueue(omx_context *c, bool shf, int pv) {
  omx::LuWork &lu = shf ? c->lu_sh : c->lu;
  cplx *A64 = (shf ? c->d_V64 : c->d_S64).as<cplx>();
  const int Np = c->Np;
  const size_t lda = (size_t)Np, n2 = lda * Np;
  hipStream_t st = sys_stream(c, shf);
  omx::zero_ints((shf ? c->d_status2 : c->d_status).as<int>(), 4, st);  // a kernel: this may be captured
  lu.pivot = pv;
  lu.split = c->tuned ? c->tuned_split : c->lu32_gemm == OMX_GEMM_BF16X3;
  omx::LuProf *prof = prof_begin(c, shf);
  int rc;
  if(c->kind == OMX_SOLVER_LU64) {
    cplx *F64 = (shf ? c->d_F64sh : c->d_F64).as<cplx>();
    HIPCHK(hipMemcpyAsync(F64, A64, sizeof(cplx) * n2, hipMemcpyDeviceToDevice, st));
    rc = omx::lu_factor<double2>(reinterpret_cast<double2 *>(F64), Np, lda, lu, st, prof);
  } else {
    float2 *A32 = (shf ? c->d_V32 : c->d_S32).as<float2>();
    bool &dirty = shf ? c->dirty32_sh : c->dirty32;
    if(dirty) omx::demote(A32, A64, n2, st);  // an earlier factorisation overwrote it
    dirty = true;
    rc = omx::lu_factor<float2>(A32, Np, lda, lu, st, prof);
  }
  if(rc) throw OmxError(OMX_ERR_DEVICE, "lu_factor launch failed (" + std::to_string(rc) + ")");
  prof_end(c, shf);
  (shf ? c->factored_sh : c->factored) = true;
}

// ------------------------------------------------------------------ graphs
// With omx_set_graphs on, the block-pivoting factorisations are captured once
// per state (the key: order, kind, pivoting, product, whether the FP32 copy
// must be refreshed first, and every buffer address the kernels take) and
// replayed afterwards.  S's capture is cut at V's start mark into two graphs
// and V's factorisation is captured on its own stream pair, so a replay keeps
// the eager overlap: S's first part, then V on the second stream after it
// beside S's rest.  Inside the captures every clear is a kernel.

void end_capture_quietly(hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if(hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(st, &g);
    if(g) (void)hipGraphDestroy(g);
  }
  (void)hipGetLastError();
}

hipGraphExec_t instantiate(hipGraph_t g) {
  if(!g) return nullptr;
  size_t n = 0;
  HIPCHK(hipGraphGetNodes(g, nullptr, &n));
  hipGraphExec_t e = nullptr;
  if(n) HIPCHK(hipGraphInstantiate(&e, g, nullptr, nullptr, 0));
  return e;
}

std::vector<uintptr_t> single_key(omx_context *c, bool with_v, int mark) {
  const bool split = c->tuned ? c->tuned_split : c->lu32_gemm == OMX_GEMM_BF16X3;
  std::vector<uintptr_t> k{1,
                           (uintptr_t)with_v,
                           (uintptr_t)c->Np,
                           (uintptr_t)c->kind,
                           (uintptr_t)c->pivot,
                           (uintptr_t)split,
                           (uintptr_t)mark,
                           (uintptr_t)c->dirty32,
                           (uintptr_t)(with_v && c->dirty32_sh)};
  const omx::LuWork *lw[] = {&c->lu, &c->lu_sh};
  for(const omx::LuWork *w : lw) {
    const void *p[] = {w->perm, w->mdst, w->msrc, w->mcnt, w->status, w->dinv, w->aux};
    for(const void *x : p) k.push_back((uintptr_t)x);
    k.push_back((uintptr_t)w->links);
  }
  const void *b[] = {c->d_S64.p, c->d_S32.p, c->d_V64.p, c->d_V32.p, c->d_F64.p, c->d_F64sh.p, c->d_status.p,
                     c->d_status2.p};
  for(const void *x : b) k.push_back((uintptr_t)x);
  return k;
}

struct CaptureMark {
  omx_context *c;
  hipGraph_t g1 = nullptr, gv = nullptr;
};

// At V's start mark inside S's capture: close S's first graph, capture V's
// factorisation on the second stream pair, and reopen S's capture (the
// look-ahead's next waits are on events recorded in the new capture).
void capture_at_mark(void *arg) {
  auto *cm = static_cast<CaptureMark *>(arg);
  omx_context *c = cm->c;
  HIPCHK(hipStreamEndCapture(c->st, &cm->g1));
  HIPCHK(hipStreamBeginCapture(c->st2, hipStreamCaptureModeThreadLocal));
  factor_enqueue(c, true, c->pivot);
  HIPCHK(hipStreamEndCapture(c->st2, &cm->gv));
  HIPCHK(hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
  HIPCHK(hipEventRecord(c->lu.ev_next, c->st));
  HIPCHK(hipEventRecord(c->lu.ev_piv, c->st));
  HIPCHK(hipEventRecord(c->lu.ev_bulk, c->st));
}

// Enqueues S's factorisation (and V's from S's mark column on, with_v) as
// graph launches, capturing them first when the state has changed.
void factor_graphed(omx_context *c, bool with_v, int mark) {
  auto &g = c->fg;
  std::vector<uintptr_t> key = single_key(c, with_v, mark);
  if(g.key != key) {
    g.reset();
    CaptureMark cm{c};
    hipGraph_t g2 = nullptr;
    omx::LuWork &lu = c->lu;
    auto unmark = [&] {
      lu.ev_mark = nullptr;
      lu.on_mark = nullptr;
      lu.mark_arg = nullptr;
    };
    const bool d32 = c->dirty32, d32sh = c->dirty32_sh;
    try {
      HIPCHK(hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
      if(with_v) {
        lu.ev_mark = c->xev[0];
        lu.mark_col = mark;
        lu.on_mark = capture_at_mark;
        lu.mark_arg = &cm;
      }
      factor_enqueue(c, false, c->pivot);
      unmark();
      HIPCHK(hipStreamEndCapture(c->st, with_v ? &g2 : &cm.g1));
      if(with_v && !cm.gv) throw OmxError(OMX_ERR_DEVICE, "factorisation capture: V's start mark was not reached");
      g.s1 = instantiate(cm.g1);
      g.s2 = instantiate(g2);
      g.v = instantiate(cm.gv);
    } catch(...) {
      unmark();
      end_capture_quietly(c->st);
      end_capture_quietly(c->st2);
      hipGraph_t gs[] = {cm.g1, cm.gv, g2};
      for(hipGraph_t x : gs)
        if(x) (void)hipGraphDestroy(x);
      g.reset();
      c->dirty32 = d32;
      c->dirty32_sh = d32sh;
      c->factored = c->factored_sh = false;
      throw;
    }
    hipGraph_t gs[] = {cm.g1, cm.gv, g2};
    for(hipGraph_t x : gs)
      if(x) (void)hipGraphDestroy(x);
    g.key = key;
    ++c->graph_captures;
  }
  // what factor_enqueue leaves behind
  const bool split = c->tuned ? c->tuned_split : c->lu32_gemm == OMX_GEMM_BF16X3;
  c->lu.pivot = c->pivot;
  c->lu.split = split;
  if(c->kind != OMX_SOLVER_LU64) c->dirty32 = true;
  c->factored = true;
  if(g.s1) HIPCHK(hipGraphLaunch(g.s1, c->st));
  if(with_v) {
    c->lu_sh.pivot = c->pivot;
    c->lu_sh.split = split;
    if(c->kind != OMX_SOLVER_LU64) c->dirty32_sh = true;
    c->factored_sh = true;
    HIPCHK(hipEventRecord(c->xev[0], c->st));
    HIPCHK(hipStreamWaitEvent(c->st2, c->xev[0], 0));
    if(g.v) HIPCHK(hipGraphLaunch(g.v, c->st2));
  }
  if(g.s2) HIPCHK(hipGraphLaunch(g.s2, c->st));
  ++c->graph_launches;
}

// The target may sit below the FP64 residual floor of an ill-conditioned
// system: a solution whose normwise backward error ||b - A x|| / (||A||_F ||x||
// + ||b||) is within 1000 units of FP64 roundoff is accepted (the relative
// residual's floor is u ||A|| ||x|| / ||b||, far above u when x is large).  The
// bound is a constant: it does not grow with tol, so a caller's loose tol
// never lets an FP32-quality answer through.
bool backward_stable(omx_context *c, const cplx *A64, const cplx *rhs, const cplx *x, double res, hipStream_t st) {
  const size_t Np = (size_t)c->Np;
  auto nrm = [&](const cplx *v) {
    omx::nrm2sq(v, c->Np, c->d_nrm.as<double>() + 1, c->d_nrm.as<double>(), st);
    double e = 0.0;
    HIPCHK(hipMemcpyAsync(&e, c->d_nrm.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return std::sqrt(e);
  };
  const double bn = nrm(rhs), xn = nrm(x);
  double a2 = 0.0;
  const size_t n2 = Np * Np, chunk = (size_t)1 << 28;
  for(size_t off = 0; off < n2; off += chunk) {
    omx::nrm2sq(A64 + off, (int)std::min(chunk, n2 - off), c->d_nrm.as<double>() + 1, c->d_nrm.as<double>(), st);
    double v = 0.0;
    HIPCHK(hipMemcpyAsync(&v, c->d_nrm.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    a2 += v;
  }
  const double eta = (res * bn) / (std::sqrt(a2) * xn + bn);
  return eta <= kBackwardErrorBound;
}

// The scratch of such products, or none when memory is short (the products then read
// the whole matrix).
cplx *sym_ensure(omx_context *c, size_t elems) {
  try {
    c->d_sym.ensure(sizeof(cplx) * elems, &c->total);
  } catch(OmxError &e) {
    if(e.code != OMX_ERR_MEMORY) throw;
    (void)hipGetLastError();
    return nullptr;
  }
  return c->d_sym.as<cplx>();
}

// Products of the assembled S (V) from half its blocks, from N = kSymN on (below,
// the caches hold much of the matrix: N = 2142 20 us whole, 28 from its half; 10240
// 249 and 171) and for the block orders that gain by it; without scratch otherwise.
omx::SymArgs sym_args(omx_context *c, bool shf, bool f32) {
  omx::SymArgs a{c->P, c->nmax, c->Np, (size_t)c->Np, c->d_ov.as<cplx>(), shf ? omx::OV_TSH : omx::OV_T, nullptr};
  if(c->kind == OMX_SOLVER_ACA_GMRES || !c->updated || c->P < 2 || c->N < kSymN || !omx::sym_pays(c->nmax, f32))
    return a;
  a.scratch = sym_ensure(c, omx::sym_scratch(c->P, c->nmax, 1));
  return a;
}

// Solves (S or V) x = rhs with the context's solver kind, on the system's
// stream (a factorisation already enqueued by factor_enqueue is used).
void solve_system(omx_context *c, bool shf, const cplx *rhs, cplx *x, int *iters, double *res) {
  omx::LuWork &lu = shf ? c->lu_sh : c->lu;
  cplx *A64 = (shf ? c->d_V64 : c->d_S64).as<cplx>();
  bool &fact = shf ? c->factored_sh : c->factored;
  const int Np = c->Np;
  const size_t lda = (size_t)Np;
  hipStream_t st = sys_stream(c, shf);
  DBuf &status = shf ? c->d_status2 : c->d_status;
  Krylov gm{c,          Np,
            1,          st,
            c->kry,     c->d_basis.as<cplx>(),
            c->d_basisZ.as<cplx>(), c->d_r.as<cplx>(),
            c->d_w1.as<cplx>(),     c->d_gpart.as<cplx>()};
  gm.A = A64;
  auto run = [&](cplx *xx, int maxit) {
    gm.solve(rhs, xx, c->tol, maxit, c->restart);
    *iters = gm.its[0];
    *res = gm.res[0];
  };
  // (V's FP64 products read the whole matrix: those of S were measured, and of the
  // choices that a size makes only the mixed Krylov has any of V's, about five a solve)
  if(!is_lu(c->kind) && !shf) gm.sym = sym_args(c, shf, false);
  if(c->kind == OMX_SOLVER_ACA_GMRES) {  // Gmres_Zcomp on the compressed operator
    gm.op = [c, shf, st](const cplx *in, cplx *out) { aca_apply(c, shf, in, out, st); };
    gm.op_bytes = c->aca[shf ? 1 : 0].bytes;
  }
  // mixed Krylov: the preconditioner is one GMRES cycle on the FP32 copy
  auto &wi = c->ws_in;
  Krylov inner{c,      Np,
               1,      st,
               wi.kry, wi.basis.as<cplx>(),
               nullptr, wi.r.as<cplx>(),
               wi.w1.as<cplx>(), wi.gpart.as<cplx>()};
  if(c->kind == OMX_SOLVER_GMRES32_IR) {
    float2 *A32w = (shf ? c->d_V32 : c->d_S32).as<float2>();
    bool &dirty = shf ? c->dirty32_sh : c->dirty32;
    if(dirty) omx::demote(A32w, A64, (size_t)Np * lda, st);  // an earlier factorisation overwrote it
    dirty = false;
    inner.A32 = A32w;
    inner.sym = sym_args(c, shf, true);
    inner.one_cycle = true;
    gm.lazy = true;  // its preconditioner is a solve of its own
    gm.prec = [&inner, &gm, Np, st](const cplx *in, cplx *out, const int *) {
      HIPCHK(hipMemsetAsync(out, 0, sizeof(cplx) * Np, st));
      // no further than the outer residual has to go (its last known distance to
      // the goal, a factor of four to spare): the last step of a cycle and the
      // ones that follow a restart need a digit or two, not six.  N = 49152: 59 ->
      // 40 inner products
      inner.solve(in, out, std::max(kInnerTol, std::ldexp(1.0, -(gm.bits + 3))), kInnerSteps, kInnerSteps);
    };
  }
  if(!is_lu(c->kind)) {
    const bool try_first = c->kind_req == OMX_SOLVER_AUTO;
    try {
      HIPCHK(hipMemsetAsync(status.p, 0, 16, st));
      HIPCHK(hipMemsetAsync(x, 0, sizeof(cplx) * Np, st));
      const int maxit =
          try_first ? std::min(c->maxit, c->auto_budget > 0 ? c->auto_budget : auto_krylov_steps(c->N)) : c->maxit;
      gm.x_zero = true;
      run(x, maxit);
      gm.x_zero = false;
      check_status(c, shf);
      if(!(*res <= 1e3 * c->tol) && (c->kind == OMX_SOLVER_ACA_GMRES || !backward_stable(c, A64, rhs, x, *res, st)))
        throw OmxError(OMX_ERR_NOCONV, "GMRES stopped at relative residual " + std::to_string(*res));
      return;
    } catch(OmxError &e) {
      if(!(try_first && e.code == OMX_ERR_NOCONV)) throw;
      c->kind = OMX_SOLVER_LU32_IR;  // the same S and S32: on to the mixed LU
      ++c->fallbacks;
    }
  }
  if(!shf && c->krylov_s && !fact) {
    // FP64 GMRES on S while V factorises; S's own mixed LU if it falls short
    omx::zero_ints(status.as<int>(), 4, st);
    HIPCHK(hipMemsetAsync(x, 0, sizeof(cplx) * Np, st));
    const int maxit = std::min(c->maxit, c->auto_budget > 0 ? c->auto_budget : auto_gmres64_steps(c->N));
    gm.sym = sym_args(c, shf, false);
    gm.x_zero = true;
    run(x, maxit);
    gm.x_zero = false;
    gm.sym = omx::SymArgs{};
    if(*res <= 1e3 * c->tol || backward_stable(c, A64, rhs, x, *res, st)) return;
    ++c->fallbacks;
  }
  const bool f64 = c->kind == OMX_SOLVER_LU64;
  cplx *F64 = (shf ? c->d_F64sh : c->d_F64).as<cplx>();
  float2 *A32 = (shf ? c->d_V32 : c->d_S32).as<float2>();
  // Block pivoting first (when selected); a zero pivot or a refinement that
  // does not converge falls back to tournament (partial) pivoting.
  const int first = fact ? lu.pivot : c->pivot;
  for(int pv = first; pv <= OMX_PIVOT_PARTIAL; ++pv) {
    const bool last = pv == OMX_PIVOT_PARTIAL;
    try {
      if(!fact || lu.pivot != pv) factor_enqueue(c, shf, pv);
      gm.status = status.as<int>();  // zero pivots of this factorisation
      if(f64) {
        gm.prec = [F64, &lu, Np, lda, st](const cplx *in, cplx *out, const int *live) {
          lu.live = live;
          omx::lu_solve<double2>(reinterpret_cast<const double2 *>(F64), Np, lda, lu, in, out, st);
          lu.live = nullptr;
        };
        omx::lu_solve<double2>(reinterpret_cast<const double2 *>(F64), Np, lda, lu, rhs, x, st);
        if(pv == OMX_PIVOT_PARTIAL) {  // plain FP64 LU with partial pivoting
          gm.status = nullptr;
          check_status(c, shf);
          *iters = 0;
          *res = -1.0;
          return;
        }
      } else {
        gm.prec = [A32, &lu, Np, lda, st](const cplx *in, cplx *out, const int *live) {
          lu.live = live;
          omx::lu_solve<float2>(A32, Np, lda, lu, in, out, st);
          lu.live = nullptr;
        };
        omx::lu_solve<float2>(A32, Np, lda, lu, rhs, x, st);  // x0 = M^{-1} b
      }
      run(x, c->maxit);
      check_status(c, shf);
      // the target may sit below the FP64 residual floor of an ill-conditioned
      // system; a stagnated refinement within 1000x of it is accepted, and so
      // is one whose normwise backward error ||b - A x|| / (||A||_F ||x|| + ||b||)
      // is within 1000x of the FP64 unit roundoff (the relative residual's
      // floor is u ||A|| ||x|| / ||b||, far above u when x is large).  That
      // bound is a constant: it does not grow with tol, so a caller's loose
      // tol never lets an FP32-quality answer through.
      if(!(*res <= 1e3 * c->tol) && !backward_stable(c, A64, rhs, x, *res, st))
        throw OmxError(OMX_ERR_NOCONV, "refinement stopped at relative residual " + std::to_string(*res) +
                                           ", backward error above " + std::to_string(kBackwardErrorBound));
      return;
    } catch(OmxError &e) {
      if(last || (e.code != OMX_ERR_SINGULAR && e.code != OMX_ERR_NOCONV)) throw;
      ++c->fallbacks;
      fact = false;
    }
  }
}

// Buffers of a batch of nb systems of order Np (mixed: FP32 copies too).
// Enqueues V's factorisation from a host thread of its own: the enqueueing
// of a factorisation proceeds at the device's pace, so enqueued from the
// calling thread it would hold back S's iterative solve (which needs the host
// between its products) until V's factorisation had run.  join() rethrows an
// error of the thread; the destructor joins without rethrowing.
struct SideEnqueue {
  std::thread t;
  std::exception_ptr err;
  void start(omx_context *c, void (*f)(void *)) {
    run(c->device, [c, f] { f(c); });
  }
  void run(int device, std::function<void()> job) {
    t = std::thread([this, device, job] {
      try {
        HIPCHK(hipSetDevice(device));
        job();
      } catch(...) {
        err = std::current_exception();
      }
    });
  }
  void join() {
    if(t.joinable()) t.join();
    if(err) {
      std::exception_ptr e = err;
      err = nullptr;
      std::rethrow_exception(e);
    }
  }
  ~SideEnqueue() {
    if(t.joinable()) t.join();
  }
};

void sweep_alloc(omx_context *c, int nb, bool f64, bool sh) {
  auto &w = c->sw;
  size_t *T = &c->total;
  const size_t Np = c->Np, n2 = Np * Np, P = c->P, S = c->nmax + 1;
  const int m = c->restart;
  aca_release_staging(c);
  w.S64.ensure(sizeof(cplx) * n2 * nb, T);
  if(f64) {
    w.F64.ensure(sizeof(cplx) * n2 * nb, T);
    w.S32.release(T);
  } else {
    w.S32.ensure(sizeof(float2) * n2 * nb, T);
    w.F64.release(T);
  }
  if(sh) {
    w.V64.ensure(sizeof(cplx) * n2 * nb, T);
    if(f64) w.F64sh.ensure(sizeof(cplx) * n2 * nb, T); else w.V32.ensure(sizeof(float2) * n2 * nb, T);
  }
  w.eps.ensure(sizeof(cplx) * P * nb, T);
  w.eps_sh.ensure(sizeof(cplx) * P * nb, T);
  w.ov.ensure(sizeof(cplx) * omx::OV_COUNT * P * 2 * S * nb, T);
  for(DBuf *b : {&w.incloc, &w.Q, &w.x, &w.xint, &w.xsh, &w.xintsh, &w.K, &w.K1, &w.r, &w.w1, &w.w2})
    b->ensure(sizeof(cplx) * Np * nb, T);
  w.w.ensure(sizeof(double) * 2 * P * c->nf * nb, T);
  w.cross.ensure(sizeof(double) * 4 * P * nb, T);
  w.abscoef.ensure(sizeof(cplx) * P * c->nf * nb, T);
  w.abssh.ensure(sizeof(double) * P * nb, T);
  w.absbes.ensure(sizeof(cplx) * P * omx::kAbsBes * nb, T);
  for(DBuf *b : {&w.perm, &w.perm2}) b->ensure(sizeof(int) * Np * nb, T);
  w.map.ensure(sizeof(int) * Np * nb, T);
  w.status.ensure(sizeof(int) * 4 * nb, T);
  if(sh) {  // V's factorisation runs beside S's: maps and status words of its own
    w.map2.ensure(sizeof(int) * Np * nb, T);
    w.status2.ensure(sizeof(int) * 4 * nb, T);
  }
  w.basis.ensure(sizeof(cplx) * Np * (m + 1) * nb, T);
  w.basisZ.ensure(sizeof(cplx) * Np * (m + 1) * nb, T);
  w.gpart.ensure(sizeof(cplx) * Np * omx::gemv_part_rows(nb), T);
  w.kz.ensure(sizeof(cplx) * 2 * nb, T);
  w.omz.ensure(sizeof(double) * nb, T);
}

// Bytes of one system of a large batch (sweep_alloc, and the scratch of the half
// products with S by GMRES).
double sweep_bytes(const omx_context *c, bool krylov_s) {
  const bool f64 = c->kind == OMX_SOLVER_LU64;
  const double Np = c->Np, nm = c->sh ? 2.0 : 1.0;
  const double vectors = 12.0 + 2.0 * (c->restart + 1) + omx::kGemvSplit;
  return nm * Np * Np * (f64 ? 32.0 : 24.0) + 16.0 * Np * vectors + 32.0 * omx::dinv_elems(c->Np, f64) +
         (krylov_s ? 16.0 * omx::sym_scratch(c->P, c->nmax, 1) : 0.0);
}

// One system's or a batch's triangular-solve variant: see set_trsv.
omx::LuWork sweep_lu(omx_context *c, int nb, bool second, int trsv) {
  auto &w = c->sw;
  const int Np = c->Np;
  omx::LuWork lw{};
  lw.perm = (second ? w.perm2 : w.perm).as<int>();
  lw.links = c->kind == OMX_SOLVER_LU64 && trsv == 1;
  lw.trsv = trsv;
  lw.msrc = (second ? w.map2 : w.map).as<int>();
  lw.status = (second ? w.status2 : w.status).as<int>();
  // V's factorisation runs on the second stream pair, beside S's work
  lw.aux = second ? c->aux2 : c->aux;
  const hipEvent_t *ev = second ? c->lu_ev2 : c->lu_ev;
  lw.ev_next = ev[0];
  lw.ev_piv = ev[1];
  lw.ev_bulk = ev[2];
  lw.ev_pan = ev[3];
  lw.gmax = 0;
  lw.pivot = omx::kPivotBlock;
  lw.split = c->lu32_gemm == OMX_GEMM_BF16X3;
  lw.nb = nb;
  lw.bs.a = (size_t)Np * Np;
  lw.bs.inv = omx::dinv_elems(Np, lw.links);
  DBuf &dinv = second ? w.dinv2 : w.dinv;
  dinv.ensure(sizeof(cplx) * lw.bs.inv * nb, &c->total);
  lw.dinv = dinv.p;
  lw.bs.vec = (size_t)Np;
  lw.bs.perm = Np;
  lw.bs.map = Np;
  lw.bs.status = 4;
  return lw;
}

// The lockstep iteration of a batch on the FP64 matrices A (Np^2 apart), in the
// sweep's buffers: basis vector k of system z at V + (k nb + z) Np.
Krylov sweep_krylov(omx_context *c, int nb, const cplx *A) {
  auto &w = c->sw;
  Krylov gm{c,     c->Np,
            nb,    c->st,
            w.kry, w.basis.as<cplx>(),
            w.basisZ.as<cplx>(), w.r.as<cplx>(),
            w.w1.as<cplx>(),     w.gpart.as<cplx>()};
  gm.A = A;
  gm.sA = (size_t)c->Np * c->Np;
  gm.batch = true;
  return gm;
}

// ------------------------------------------------------------------ autotuner
// Per shape (device, padded order, batch, factor type) the batched sweeps
// pick the bulk-update product of FP32 factors (split-bf16 with K = 256 or FP32
// MFMA with K = 128, timed on the same 256 columns' worth of update) and
// the triangular-solve variant by timing every candidate on the batch's own
// buffers before its first chunk (zeroed matrices, identity permutations:
// the kernels have no value-dependent branches, so the times are those of the
// real work), once per process.  A candidate replaces the default only when
// it is at least 5% faster, so tuning again returns the same choice unless
// two candidates sit at that margin.  The choices are kept per process and
// can be read back (omx_tune_query).
struct TuneChoice {
  bool split = true;
  int trsv = 0;
  double t_prod[2] = {0, 0};                   // ms: split-bf16, FP32 MFMA (FP32 factors only)
  double t_trsv[omx::kTrsvVariants] = {0, 0, 0};  // ms per batched LU solve
};
std::mutex g_tune_mu;
std::map<std::tuple<int, int, int, int>, TuneChoice> g_tune;  // (device, Np, nb, fp64)
constexpr double kTuneMargin = 0.95;

bool tune_lookup(const omx_context *c, int nb, bool f64, TuneChoice *out) {
  std::lock_guard<std::mutex> g(g_tune_mu);
  auto it = g_tune.find(std::make_tuple(c->device, c->Np, nb, f64 ? 1 : 0));
  if(it != g_tune.end()) *out = it->second;
  return it != g_tune.end();
}

double time_median(hipStream_t st, const std::function<void()> &f, int reps = 5) {
  hipEvent_t a, b;
  HIPCHK(hipEventCreate(&a));
  HIPCHK(hipEventCreate(&b));
  std::vector<float> ts;
  try {
    f();  // warm-up
    for(int r = 0; r < reps; ++r) {
      HIPCHK(hipEventRecord(a, st));
      f();
      HIPCHK(hipEventRecord(b, st));
      HIPCHK(hipEventSynchronize(b));
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, a, b));
      ts.push_back(ms);
    }
  } catch(...) {
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    throw;
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  std::sort(ts.begin(), ts.end());
  return ts[ts.size() / 2];
}

// A solve's share of forming the links: a factorisation is applied about three times,
// to the right-hand side and in two refinement steps.
double links_share(const double2 *F, int Np, const omx::LuWork &lw, hipStream_t st) {
  return time_median(st, [&] { omx::lu_links(F, Np, (size_t)Np, lw, st); }) / 3.0;
}

// The tuned choice for this batch (tuning it first if needed); runs on the
// chunk's buffers before the chunk fills them.
TuneChoice sweep_tune(omx_context *c, int nb, bool f64) {
  TuneChoice ch;
  if(tune_lookup(c, nb, f64, &ch)) return ch;
  auto &w = c->sw;
  const int Np = c->Np;
  const size_t n2 = (size_t)Np * Np, lda = (size_t)Np;
  hipStream_t st = c->st;
  ch.split = c->lu32_gemm == OMX_GEMM_BF16X3;
  void *F = f64 ? w.F64.p : w.S32.p;
  const size_t fbytes = (f64 ? sizeof(double2) : sizeof(float2)) * n2 * nb;
  HIPCHK(hipMemsetAsync(F, 0, fbytes, st));
  if(!f64 && Np > 4 * omx::kNB) {  // a smaller factorisation has no bulk update
    float2 *A = static_cast<float2 *>(F);
    ch.t_prod[0] = time_median(st, [&] { omx::bulk_update_probe(A, Np, lda, nb, n2, true, st); });
    ch.t_prod[1] = time_median(st, [&] { omx::bulk_update_probe(A, Np, lda, nb, n2, false, st); });
    const int dflt = ch.split ? 0 : 1, other = 1 - dflt;
    if(ch.t_prod[other] < kTuneMargin * ch.t_prod[dflt]) ch.split = other == 0;
    HIPCHK(hipMemsetAsync(F, 0, fbytes, st));
  }
  // triangular solves on zeroed factors and inverses, identity permutations
  std::vector<int> ident((size_t)Np * nb);
  for(int z = 0; z < nb; ++z)
    for(int i = 0; i < Np; ++i) ident[(size_t)z * Np + i] = i;
  HIPCHK(hipMemcpyAsync(w.perm.p, ident.data(), sizeof(int) * ident.size(), hipMemcpyHostToDevice, st));
  const size_t before = w.dinv.bytes;
  (void)sweep_lu(c, nb, false, 1);  // room for the links
  HIPCHK(hipMemsetAsync(w.dinv.p, 0, w.dinv.bytes, st));
  HIPCHK(hipMemsetAsync(w.r.p, 0, w.r.bytes, st));
  for(int v = 0; v < omx::kTrsvVariants; ++v) {
    omx::LuWork lw = sweep_lu(c, nb, false, v);
    ch.t_trsv[v] = time_median(st, [&] {
      if(f64)
        omx::lu_solve<double2>(static_cast<const double2 *>(F), Np, lda, lw, w.r.as<cplx>(), w.w2.as<cplx>(), st);
      else
        omx::lu_solve<float2>(static_cast<const float2 *>(F), Np, lda, lw, w.r.as<cplx>(), w.w2.as<cplx>(), st);
    });
    if(lw.links) ch.t_trsv[v] += links_share(static_cast<const double2 *>(F), Np, lw, st);
  }
  int best = 0;
  for(int v = 1; v < omx::kTrsvVariants; ++v)
    if(ch.t_trsv[v] < ch.t_trsv[best]) best = v;
  ch.trsv = ch.t_trsv[best] < kTuneMargin * ch.t_trsv[0] ? best : 0;
  if(ch.trsv != 1 && w.dinv.bytes > before) w.dinv.release(&c->total);
  HIPCHK(hipStreamSynchronize(st));  // ident ends here
  std::lock_guard<std::mutex> g(g_tune_mu);
  g_tune[std::make_tuple(c->device, Np, nb, f64 ? 1 : 0)] = ch;
  return ch;
}

// The single-system LU solves (omx_update / omx_solve) tune the same way,
// with batch 1 and the context's own buffers (before the assembly fills
// them).
TuneChoice single_tune(omx_context *c, bool f64) {
  TuneChoice ch;
  const int Np = c->Np;
  const size_t n2 = (size_t)Np * Np, lda = (size_t)Np;
  hipStream_t st = c->st;
  ch.split = c->lu32_gemm == OMX_GEMM_BF16X3;
  void *F = f64 ? c->d_F64.p : c->d_S32.p;
  const size_t fbytes = (f64 ? sizeof(double2) : sizeof(float2)) * n2;
  HIPCHK(hipMemsetAsync(F, 0, fbytes, st));
  if(!f64 && Np > 4 * omx::kNB) {  // a smaller factorisation has no bulk update
    float2 *A = static_cast<float2 *>(F);
    ch.t_prod[0] = time_median(st, [&] { omx::bulk_update_probe(A, Np, lda, 1, 0, true, st); });
    ch.t_prod[1] = time_median(st, [&] { omx::bulk_update_probe(A, Np, lda, 1, 0, false, st); });
    const int dflt = ch.split ? 0 : 1, other = 1 - dflt;
    if(ch.t_prod[other] < kTuneMargin * ch.t_prod[dflt]) ch.split = other == 0;
    HIPCHK(hipMemsetAsync(F, 0, fbytes, st));
  }
  std::vector<int> ident(Np);
  for(int i = 0; i < Np; ++i) ident[i] = i;
  HIPCHK(hipMemcpyAsync(c->d_perm.p, ident.data(), sizeof(int) * Np, hipMemcpyHostToDevice, st));
  omx::LuWork &lw = c->lu;
  set_trsv(c, lw, c->d_dinv, 1);  // room for the links
  HIPCHK(hipMemsetAsync(c->d_dinv.p, 0, c->d_dinv.bytes, st));
  HIPCHK(hipMemsetAsync(c->d_r.p, 0, c->d_r.bytes, st));
  for(int v = 0; v < omx::kTrsvVariants; ++v) {
    lw.trsv = v;
    lw.links = f64 && v == 1;
    ch.t_trsv[v] = time_median(st, [&] {
      if(f64)
        omx::lu_solve<double2>(static_cast<const double2 *>(F), Np, lda, lw, c->d_r.as<cplx>(), c->d_w2.as<cplx>(),
                               st);
      else
        omx::lu_solve<float2>(static_cast<const float2 *>(F), Np, lda, lw, c->d_r.as<cplx>(), c->d_w2.as<cplx>(), st);
    });
    if(lw.links) ch.t_trsv[v] += links_share(static_cast<const double2 *>(F), Np, lw, st);
  }
  int best = 0;
  for(int v = 1; v < omx::kTrsvVariants; ++v)
    if(ch.t_trsv[v] < ch.t_trsv[best]) best = v;
  ch.trsv = ch.t_trsv[best] < kTuneMargin * ch.t_trsv[0] ? best : 0;
  HIPCHK(hipStreamSynchronize(st));  // ident ends here
  std::lock_guard<std::mutex> g(g_tune_mu);
  g_tune[std::make_tuple(c->device, Np, 1, f64 ? 1 : 0)] = ch;
  return ch;
}

// One batch of a wavelength sweep: nb systems (wavelengths lam[z], absolute
// permittivities eps[z * P + i], eps_sh[z * P + i]) assembled, factorised and
// refined side by side.  Systems whose factorisation hit a zero pivot or whose
// refinement did not converge are flagged in bad[z] for the caller to redo
// one at a time with partial pivoting.
void sweep_chunk(omx_context *c, int nb, const double *lam, const cplx *eps, const cplx *eps_sh, double *x_sca,
                 double *x_int, double *x_sca_sh, double *x_int_sh, double *xs, std::vector<int> &bad,
                 std::vector<int> &iters, std::vector<double> &resid, bool krylov_s) {
  const bool f64 = c->kind == OMX_SOLVER_LU64, sh = c->sh;
  sweep_alloc(c, nb, f64, sh);
  const TuneChoice tune = c->autotune ? sweep_tune(c, nb, f64) : TuneChoice{c->lu32_gemm == OMX_GEMM_BF16X3, 0};
  auto &w = c->sw;
  const int P = c->P, nmax = c->nmax, N = c->N, Np = c->Np;
  const size_t n2 = (size_t)Np * Np, lda = (size_t)Np;
  const size_t ovs = (size_t)omx::OV_COUNT * P * 2 * (nmax + 1), ws = (size_t)2 * P * c->nf;
  hipStream_t st = c->st;
  HIPCHK(hipMemcpyAsync(w.eps.p, eps, sizeof(cplx) * P * nb, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(w.eps_sh.p, eps_sh, sizeof(cplx) * P * nb, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemsetAsync(w.status.p, 0, w.status.bytes, st));
  if(sh) HIPCHK(hipMemsetAsync(w.status2.p, 0, w.status2.bytes, st));
  HIPCHK(hipMemsetAsync(w.Q.p, 0, w.Q.bytes, st));
  HIPCHK(hipMemsetAsync(c->d_status.p, 0, 16, st));
  const cplx bge = kEps0 * c->bg_eps_r, bgm = kMu0 * c->bg_mu_r;
  std::complex<double> bgn = std::sqrt(std::complex<double>(c->bg_eps_r.x, c->bg_eps_r.y) *
                                       std::complex<double>(c->bg_mu_r.x, c->bg_mu_r.y));
  // plane-wave coefficients do not depend on the wavelength (Excitation.cpp:48-75)
  omx::IncArgs ia{nmax, c->theta, c->phi, c->eth, c->eph, c->d_inc.as<cplx>()};
  omx::run_incident(ia, st);
  cplx *cS64 = w.S64.as<cplx>(), *cV64 = w.V64.as<cplx>();
  float2 *cS32 = w.S32.as<float2>(), *cV32 = w.V32.as<float2>();
  // per-system wavenumbers (k at omega, 2k at 2 omega) and angular frequencies;
  // every assembly kernel then covers the whole batch in one launch (system in blockIdx.z)
  std::vector<cplx> hk(2 * nb);
  std::vector<double> hom(nb);
  for(int z = 0; z < nb; ++z) {
    const double k0 = 2.0 * omx::kPi / lam[z];
    hom[z] = omx::kC0 * k0;
    hk[z] = omx::mk(k0 * bgn.real(), k0 * bgn.imag());
    hk[nb + z] = omx::mk(2.0 * hk[z].x, 2.0 * hk[z].y);  // PreconditionedMatrix.cpp:592
  }
  HIPCHK(hipMemcpyAsync(w.kz.p, hk.data(), sizeof(cplx) * 2 * nb, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(w.omz.p, hom.data(), sizeof(double) * nb, hipMemcpyHostToDevice, st));
  const cplx *kz = w.kz.as<cplx>();
  omx::ObjArgs oa{P, nmax, hom[0], bge, bgm, c->d_xyz.as<double>(), c->d_radius.as<double>(), w.eps.as<cplx>(),
                  c->d_mu.as<cplx>(), w.eps_sh.as<cplx>(), c->d_sph.as<double>(), w.ov.as<cplx>()};
  oa.omz = w.omz.as<double>();
  oa.zov = ovs;
  omx::run_objects(oa, st, nb);
  omx::OriginArgs og{P, nmax, hk[0], c->d_sph.as<double>(), w.ov.as<cplx>(), c->d_coef.as<double>(),
                     c->d_inc.as<cplx>(), w.incloc.as<cplx>(), w.Q.as<cplx>(), w.w.as<double>(), sh};
  og.kz = kz;
  og.zov = ovs;
  og.zvec = lda;
  og.zw = ws;
  // beside the pairs, as in omx_update
  HIPCHK(hipEventRecord(c->ujoin[0], st));
  HIPCHK(hipStreamWaitEvent(c->st2, c->ujoin[0], 0));
  omx::run_origin(og, c->st2, nb);
  HIPCHK(hipEventRecord(c->ujoin[1], c->st2));
  omx::PairArgs pa{P, nmax, omx::OV_T, hk[0], c->d_sph.as<double>(), w.ov.as<cplx>(), c->d_coef.as<double>(), lda,
                   cS64, f64 ? nullptr : cS32};
  pa.kz = kz;
  pa.zov = ovs;
  pa.zS = n2;
  if(sh) {  // V in the same launch
    pa.tkind2 = omx::OV_TSH;
    pa.kz2 = kz + nb;
    pa.V64 = cV64;
    pa.V32 = f64 ? nullptr : cV32;
  }
  omx::run_pairs(pa, st, nb);
  omx::run_pad64(cS64, N, Np, lda, st, nb, n2);
  if(!f64) omx::run_pad32(cS32, N, Np, lda, st, nb, n2);
  if(sh) {
    omx::run_pad64(cV64, N, Np, lda, st, nb, n2);
    if(!f64) omx::run_pad32(cV32, N, Np, lda, st, nb, n2);
  }
  HIPCHK(hipStreamWaitEvent(st, c->ujoin[1], 0));
  HIPCHK(hipGetLastError());
  auto status_scan = [&](std::vector<int> &flag, bool second) {
    std::vector<int> h(4 * nb);
    HIPCHK(hipMemcpyAsync(h.data(), (second ? w.status2 : w.status).p, sizeof(int) * 4 * nb, hipMemcpyDeviceToHost,
                          st));
    int g[2];
    HIPCHK(hipMemcpyAsync(g, c->d_status.p, sizeof(g), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if(h[1] || g[1]) throw OmxError(OMX_ERR_DEVICE, "device wait timed out in a batched solve");
    for(int z = 0; z < nb; ++z)
      if(h[4 * z]) flag[z] = 1;
  };
  // factorisation of S (V) for every system, enqueued on stream fst
  auto factor = [&](bool second, omx::LuWork &lw, hipStream_t fst) -> void * {
    cplx *A64 = second ? cV64 : cS64;
    void *F;
    int rc;
    if(f64) {
      F = (second ? w.F64sh : w.F64).p;
      HIPCHK(hipMemcpyAsync(F, A64, sizeof(cplx) * n2 * nb, hipMemcpyDeviceToDevice, fst));
      rc = omx::lu_factor<double2>(static_cast<double2 *>(F), Np, lda, lw, fst, nullptr);
    } else {
      F = (second ? w.V32 : w.S32).p;
      rc = omx::lu_factor<float2>(static_cast<float2 *>(F), Np, lda, lw, fst, nullptr);
    }
    if(rc) throw OmxError(OMX_ERR_DEVICE, "batched lu_factor launch failed (" + std::to_string(rc) + ")");
    return F;
  };
  // V does not depend on the fundamental solution: its factorisation starts
  // on the second stream pair right after the assembly and runs beside S's
  // factorisation and refinement; V's refinement waits for it
  omx::LuWork lwS = sweep_lu(c, nb, false, tune.trsv), lwV{};
  lwS.split = tune.split;
  if(sh) {
    lwV = sweep_lu(c, nb, true, tune.trsv);
    lwV.split = tune.split;
  }
  void *FS = f64 ? w.F64.p : w.S32.p, *FV = sh ? (f64 ? w.F64sh.p : w.V32.p) : nullptr;
  SideEnqueue vq;
  if(krylov_s) {
    // S is solved by GMRES (no factorisation); V's factorisation is enqueued
    // from a host thread of its own so that S's iterations start at once
    HIPCHK(hipEventRecord(c->xev[0], st));
    vq.run(c->device, [&] {
      HIPCHK(hipStreamWaitEvent(c->st2, c->xev[0], 0));
      factor(true, lwV, c->st2);
      HIPCHK(hipEventRecord(c->xev[1], c->st2));
    });
  } else if(c->graphs) {
    // captured once per batch shape and buffers, then replayed chunk after chunk
    auto &g = c->fg_sweep;
    std::vector<uintptr_t> key{2, (uintptr_t)nb, (uintptr_t)Np, (uintptr_t)f64, (uintptr_t)sh, (uintptr_t)tune.split,
                               (uintptr_t)lwS.links};
    const void *p[] = {w.S64.p, w.S32.p, w.V64.p, w.V32.p, w.F64.p, w.F64sh.p, w.perm.p, w.perm2.p, w.map.p,
                       w.map2.p, w.status.p, w.status2.p, w.dinv.p, w.dinv2.p};
    for(const void *x : p) key.push_back((uintptr_t)x);
    if(g.key != key) {
      g.reset();
      hipGraph_t gs = nullptr, gv = nullptr;
      try {
        if(sh) {
          HIPCHK(hipStreamBeginCapture(c->st2, hipStreamCaptureModeThreadLocal));
          factor(true, lwV, c->st2);
          HIPCHK(hipStreamEndCapture(c->st2, &gv));
        }
        HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        factor(false, lwS, st);
        HIPCHK(hipStreamEndCapture(st, &gs));
        g.s1 = instantiate(gs);
        g.v = instantiate(gv);
      } catch(...) {
        end_capture_quietly(c->st2);
        end_capture_quietly(st);
        if(gs) (void)hipGraphDestroy(gs);
        if(gv) (void)hipGraphDestroy(gv);
        g.reset();
        throw;
      }
      if(gs) (void)hipGraphDestroy(gs);
      if(gv) (void)hipGraphDestroy(gv);
      g.key = key;
      ++c->graph_captures;
    }
    if(sh) {
      HIPCHK(hipEventRecord(c->xev[0], st));
      HIPCHK(hipStreamWaitEvent(c->st2, c->xev[0], 0));
      if(g.v) HIPCHK(hipGraphLaunch(g.v, c->st2));
      HIPCHK(hipEventRecord(c->xev[1], c->st2));
    }
    if(g.s1) HIPCHK(hipGraphLaunch(g.s1, st));
    ++c->graph_launches;
  } else {
    if(sh) {
      HIPCHK(hipEventRecord(c->xev[0], st));
      HIPCHK(hipStreamWaitEvent(c->st2, c->xev[0], 0));
      factor(true, lwV, c->st2);
      HIPCHK(hipEventRecord(c->xev[1], c->st2));
    }
    factor(false, lwS, st);
  }
  // refinement of every system of S (V); per-system convergence flags
  auto refine = [&](bool second, omx::LuWork &lw, void *F, const cplx *rhs, cplx *x, bool from_x = false) {
    status_scan(bad, second);
    cplx *A64 = second ? cV64 : cS64;
    Krylov gm = sweep_krylov(c, nb, A64);
    gm.prec = [c, F, &lw, Np, lda, f64](const cplx *in, cplx *out, const int *live) {
      lw.live = live;
      if(f64)
        omx::lu_solve<double2>(static_cast<const double2 *>(F), Np, lda, lw, in, out, c->st);
      else
        omx::lu_solve<float2>(static_cast<const float2 *>(F), Np, lda, lw, in, out, c->st);
      lw.live = nullptr;
    };
    if(!from_x) gm.prec(rhs, x, nullptr);  // else: start from the iterate x holds
    // the batch runs in lockstep until its slowest system stops: a system
    // still short of the target after four restart cycles is left to the
    // one-at-a-time path (partial pivoting) instead of holding the batch
    const int bmax = nb > 1 ? std::min(c->maxit, 4 * c->restart) : c->maxit;
    gm.solve(rhs, x, c->tol, bmax, c->restart);
    status_scan(bad, second);
    for(int z = 0; z < nb; ++z) {
      if(!(gm.res[z] <= 1e3 * c->tol)) bad[z] = 1;
      iters[2 * z + (second ? 1 : 0)] = gm.its[z];
      resid[2 * z + (second ? 1 : 0)] = gm.res[z];
    }
  };
  if(krylov_s) {
    // lockstep FP64 GMRES on every system of S, from zero, within twice the
    // single-system budget (S's solve runs beside V's factorisation); a
    // system short of the target is left to the one-at-a-time path
    status_scan(bad, false);
    Krylov gm = sweep_krylov(c, nb, cS64);
    if((double)N * N * nb >= (double)kSymN * kSymN && omx::sym_pays(nmax, false)) {  // as sym_args
      gm.sym = omx::SymArgs{P,  nmax, (int)Np, lda, w.ov.as<cplx>(), omx::OV_T, sym_ensure(c, omx::sym_scratch(P, nmax, nb)),
                            nb, (size_t)Np * Np, lda, ovs};
    }
    cplx *Sx = w.x.as<cplx>();
    gm.x_zero = true;
    HIPCHK(hipMemsetAsync(Sx, 0, sizeof(cplx) * lda * nb, st));
    const int budget = std::min(c->maxit, c->auto_budget > 0 ? c->auto_budget : 2 * auto_gmres64_steps(c->N));
    gm.solve(w.Q.as<cplx>(), Sx, c->tol, budget, c->restart);
    bool short_any = false;
    for(int z = 0; z < nb; ++z) {
      short_any |= !(gm.res[z] <= 1e3 * c->tol);
      iters[2 * z] = gm.its[z];
      resid[2 * z] = gm.res[z];
    }
    if(short_any) {
      // S factored for the batch after all; every system refined from its
      // GMRES iterate (those already at the target stop at once)
      factor(false, lwS, st);
      refine(false, lwS, FS, w.Q.as<cplx>(), Sx, true);
      ++c->fallbacks;
    }
  } else {
    refine(false, lwS, FS, w.Q.as<cplx>(), w.x.as<cplx>());
  }
  omx::vmul_ov(w.xint.as<cplx>(), w.x.as<cplx>(), w.ov.as<cplx>(), omx::OV_IAUX, P, nmax, nullptr, N, st, nb, lda, ovs);
  if(sh) {
    if(c->cg_nmax != nmax) {
      size_t nf = (size_t)c->nf, sz = nf * nf * nf;
      c->d_cg.ensure(sizeof(double) * 9 * sz, &c->total);
      omx::run_cg(nmax, c->d_cg.as<double>(), st);
      c->cg_nmax = nmax;
    }
    HIPCHK(hipMemsetAsync(w.K.p, 0, w.K.bytes, st));
    omx::ShArgs sa{P, nmax, hom[0], bge, bgm, c->d_radius.as<double>(), w.eps.as<cplx>(), c->d_mu.as<cplx>(),
                   w.eps_sh.as<cplx>(), c->d_kppp.as<cplx>(), c->d_kpar.as<cplx>(), c->d_gam.as<cplx>(),
                   w.ov.as<cplx>(), c->d_cg.as<double>(), w.xint.as<cplx>(), w.K.as<cplx>(), w.K1.as<cplx>()};
    sa.nb = nb;
    sa.omz = w.omz.as<double>();
    sa.zvec = lda;
    sa.zov = ovs;
    omx::run_shsrc(sa, st);
    vq.join();  // V's factorisation enqueued (and its event recorded) before the wait below
    HIPCHK(hipStreamWaitEvent(st, c->xev[1], 0));  // V's factorisation
    refine(true, lwV, FV, w.K.as<cplx>(), w.xsh.as<cplx>());
    omx::vmul_ov(w.xintsh.as<cplx>(), w.xsh.as<cplx>(), w.ov.as<cplx>(), omx::OV_IAUXSH1, P, nmax, w.K1.as<cplx>(), N,
                 st, nb, lda, ovs);
  }
  // cross sections (Result.cpp:557-761)
  omx::CrossArgs ca{P, nmax, w.x.as<cplx>(), sh ? w.xsh.as<cplx>() : nullptr, w.incloc.as<cplx>(), w.w.as<double>(),
                    w.ov.as<cplx>(), w.cross.as<double>()};
  ca.nb = nb;
  ca.zvec = lda;
  ca.zw = ws;
  ca.zov = ovs;
  omx::run_cross(ca, st);
  // SH absorption (Result.cpp:763-794), every system in one batch
  if(sh) {
    omx::AbsShArgs aa{P, nmax, hom[0], bge, bgm, c->d_radius.as<double>(), w.eps.as<cplx>(), c->d_mu.as<cplx>(),
                      w.eps_sh.as<cplx>(), c->d_gam.as<cplx>(), c->d_cg.as<double>(), w.xint.as<cplx>(),
                      w.xintsh.as<cplx>(), w.abscoef.as<cplx>(), w.abssh.as<double>()};
    aa.bes = w.absbes.as<cplx>();
    aa.omz = w.omz.as<double>();
    aa.nb = nb;
    aa.zvec = lda;
    omx::run_abssh(aa, st);
  }
  std::vector<double> part((size_t)4 * P * nb), pabs((size_t)P * nb, 0.0);
  HIPCHK(hipMemcpyAsync(part.data(), w.cross.p, sizeof(double) * part.size(), hipMemcpyDeviceToHost, st));
  if(sh) HIPCHK(hipMemcpyAsync(pabs.data(), w.abssh.p, sizeof(double) * pabs.size(), hipMemcpyDeviceToHost, st));
  auto cp = [&](double *dst, const DBuf &b) {
    if(dst)
      HIPCHK(hipMemcpy2DAsync(dst, sizeof(cplx) * N, b.p, sizeof(cplx) * Np, sizeof(cplx) * N, nb,
                              hipMemcpyDeviceToHost, st));
  };
  cp(x_sca, w.x);
  cp(x_int, w.xint);
  if(sh) {
    cp(x_sca_sh, w.xsh);
    cp(x_int_sh, w.xintsh);
  }
  HIPCHK(hipStreamSynchronize(st));
  if(xs)
    for(int z = 0; z < nb; ++z) {
      double sm[4] = {0, 0, 0, 0};
      for(int j = 0; j < P; ++j)
        for(int e = 0; e < 4; ++e) sm[e] += part[(size_t)z * 4 * P + 4 * j + e];
      const double rk = 2.0 * omx::kPi / lam[z] * bgn.real();
      double sa = 0.0;
      for(int j = 0; j < P; ++j) sa += pabs[(size_t)z * P + j];
      xs[5 * z + 0] = (-1. / (rk * rk)) * sm[0];  // Result.cpp:576
      xs[5 * z + 1] = (1. / (rk * rk)) * sm[1];   // Result.cpp:646
      xs[5 * z + 2] = (1. / (rk * rk)) * sm[2];   // Result.cpp:675
      xs[5 * z + 3] = sh ? (1.0 / (4.0 * c->bg_eps_r.x * c->bg_mu_r.x)) * sm[3] : 0.0;  // Result.cpp:760
      xs[5 * z + 4] = sa;                                                               // Result.cpp:763-794
    }
}

// ------------------------------------------------------------------ no-allocation solve
// omx_dense_solve_noalloc keeps every work array of its factorisation and
// triangular solves in one file-scope device array, so a call allocates
// nothing.  Each device holds its own copy for the life of the process; the
// host learns that copy's address once per device (hipGetSymbolAddress in
// omx_create, with the device current) and passes that address to kernels:
// the array's name in host code is not a device address.
constexpr int kNoAllocMaxN = 4096;  // largest order (and padded order) served
constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }
struct NoAllocLayout {
  static constexpr int Np = kNoAllocMaxN;
  static constexpr int gmax = Np / omx::kPanelRows + 1;
  static constexpr size_t status = 0;  // 16 ints
  static constexpr size_t perm = status + align256(16 * sizeof(int));  // Np ints
  static constexpr size_t cand = perm + align256(Np * sizeof(int));  // 2 x gmax x 64 ints
  static constexpr size_t map = cand + align256(2 * gmax * omx::kNB * sizeof(int));  // 3 x (Np + 128) ints
  static constexpr size_t wlu = map + align256(3 * (Np + 2 * omx::kNB) * sizeof(int));  // 64 x 64 complex
  static constexpr size_t dinv = wlu + align256(omx::kNB * omx::kNB * sizeof(cplx));  // 2 x 64 x Np complex
  static constexpr size_t rhs = dinv + align256(2 * omx::kNB * (size_t)Np * sizeof(cplx));  // Np complex
  static constexpr size_t x = rhs + align256(Np * sizeof(cplx));  // Np complex
  static constexpr size_t bytes = x + align256(Np * sizeof(cplx));
};
static_assert(NoAllocLayout::bytes < (9u << 20), "no-allocation scratch stays under 9 MiB");

static __device__ __align__(256) unsigned char scratch[NoAllocLayout::bytes];

std::mutex g_scratch_mu;
std::vector<void *> g_scratch_addr;  // per device, filled once

// Device address of this device's scratch array (the device must be current).
void *scratch_address(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if((int)g_scratch_addr.size() <= device) g_scratch_addr.resize(device + 1, nullptr);
  if(!g_scratch_addr[device]) {
    void *p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if(!p) throw OmxError(OMX_ERR_DEVICE, "hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_addr[device] = p;
  }
  return g_scratch_addr[device];
}

// Clears n ints (a kernel rather than a memset, so the call also suits code
// that records it into a graph).
__global__ void zero_ints_kernel(int *p, int n) {
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}
// rb[0, N) = b, rb[N, Np) = 0: the right-hand side of the padded system.
__global__ void stage_rhs_kernel(const cplx *b, cplx *rb, int N, int Np) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < Np) rb[i] = i < N ? b[i] : omx::mk(0.0);
}

}  // namespace

extern "C" {

const char *omx_last_error(void) { return g_err.c_str(); }

int omx_create(omx_context **out, int device) {
  return guard([&] {
    if(!out) throw OmxError(OMX_ERR_ARG, "null context pointer");
    int n = 0;
    HIPCHK(hipGetDeviceCount(&n));
    if(device < 0 || device >= n) throw OmxError(OMX_ERR_DEVICE, "no HIP device " + std::to_string(device));
    auto *c = new omx_context();
    if(const char *e = std::getenv("OMX_SH_OVERLAP")) c->sh_overlap = std::atof(e);
    if(const char *e = std::getenv("OMX_KRYLOV_MARK")) c->krylov_mark = std::atof(e);
    c->device = device;
    try {
      HIPCHK(hipSetDevice(device));
      HIPCHK(hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking));
      HIPCHK(hipStreamCreateWithFlags(&c->aux, hipStreamNonBlocking));
      HIPCHK(hipStreamCreateWithFlags(&c->st2, hipStreamNonBlocking));
      HIPCHK(hipStreamCreateWithFlags(&c->aux2, hipStreamNonBlocking));
      for(auto &e : c->lu_ev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      for(auto &e : c->lu_ev2) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      for(auto &e : c->xev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      for(auto &e : c->ev) HIPCHK(hipEventCreate(&e));
      for(auto &e : c->uev) HIPCHK(hipEventCreate(&e));
      for(hipEvent_t *e : {&c->geo_ev, &c->ujoin[0], &c->ujoin[1]})
        HIPCHK(hipEventCreateWithFlags(e, hipEventDisableTiming));
      omx::upload_factorials();
      c->scratch = scratch_address(device);
    } catch(...) {
      omx_destroy(c);
      throw;
    }
    *out = c;
  });
}

void omx_destroy(omx_context *c) {
  if(!c) return;
  (void)hipSetDevice(c->device);
  if(c->st) (void)hipStreamSynchronize(c->st);
  if(c->st2) (void)hipStreamSynchronize(c->st2);
  c->fg.reset();
  c->fg_sweep.reset();
  c->d_status2.release(&c->total);
  c->d_map2.release(&c->total);
  DBuf *bufs[] = {&c->d_geo, &c->d_sph, &c->d_ov, &c->d_inc, &c->d_incloc, &c->d_Q, &c->d_w, &c->d_coef, &c->d_S64,
                  &c->d_S32, &c->d_V64, &c->d_V32, &c->d_x, &c->d_xsh, &c->d_xint, &c->d_xintsh, &c->d_K,
                  &c->d_K1, &c->d_cross, &c->d_cg, &c->d_perm, &c->d_cand, &c->d_map,
                  &c->d_wlu, &c->d_status, &c->d_basis, &c->d_basisZ, &c->d_w1, &c->d_w2, &c->d_r,
                  &c->d_nrm, &c->d_gpart, &c->d_sym, &c->d_perm2,
                  &c->d_dinv, &c->d_dinv2, &c->d_F64, &c->d_F64sh, &c->d_abscoef, &c->d_abssh, &c->d_absbes,
                  &c->d_fpts, &c->d_fout, &c->d_fown, &c->d_fpart};
  for(DBuf *b : bufs) b->release(&c->total);
  c->sw.release(&c->total);
  c->aca[0].release(&c->total);
  c->aca[1].release(&c->total);
  c->ws_in.release(&c->total);
  c->kry.release(&c->total);
  DBuf *abufs[] = {&c->d_acaA, &c->d_acaU, &c->d_acaV, &c->d_acaR, &c->d_acaOff, &c->d_plist};
  for(DBuf *b : abufs) b->release(&c->total);
  for(auto &e : c->ev)
    if(e) (void)hipEventDestroy(e);
  for(auto e : c->pev)
    if(e) (void)hipEventDestroy(e);
  for(auto e : c->lu_ev)
    if(e) (void)hipEventDestroy(e);
  for(auto e : c->lu_ev2)
    if(e) (void)hipEventDestroy(e);
  for(auto e : c->xev)
    if(e) (void)hipEventDestroy(e);
  for(hipEvent_t e : {c->mv_ev[0], c->mv_ev[1], c->geo_ev, c->uev[0], c->uev[1], c->uev[2], c->ujoin[0], c->ujoin[1]})
    if(e) (void)hipEventDestroy(e);
  for(auto e : c->pev2)
    if(e) (void)hipEventDestroy(e);
  if(c->aux2) (void)hipStreamDestroy(c->aux2);
  if(c->st2) (void)hipStreamDestroy(c->st2);
  if(c->aux) (void)hipStreamDestroy(c->aux);
  if(c->st) (void)hipStreamDestroy(c->st);
  if(c->geo_pin) (void)hipHostFree(c->geo_pin);
  if(c->out_pin) (void)hipHostFree(c->out_pin);
  delete c;
}

int omx_set_geometry(omx_context *c, int nobj, int nmax, const double *xyz, const double *radius,
                     const double *eps_r, const double *mu_r, const double *eps_r_sh, const double *ksippp,
                     const double *ksiparppar, const double *gamma, const double *bg_eps_r,
                     const double *bg_mu_r) {
  return guard([&] {
    if(!c || nobj < 1 || nmax < 1 || nmax > omx::kMaxNmax || !xyz || !radius || !eps_r || !mu_r)
      throw OmxError(OMX_ERR_ARG, "invalid geometry (1 <= nmax <= 10, nobj >= 1, arrays non-null)");
    HIPCHK(hipSetDevice(c->device));
    // Geometry::pushObject rejects overlapping spheres (Geometry.cpp:39-51)
    for(int i = 0; i < nobj; ++i)
      for(int j = 0; j < i; ++j) {
        double dx = xyz[3 * i] - xyz[3 * j], dy = xyz[3 * i + 1] - xyz[3 * j + 1], dz = xyz[3 * i + 2] - xyz[3 * j + 2];
        if(std::sqrt(dx * dx + dy * dy + dz * dz) <= radius[i] + radius[j])
          throw OmxError(OMX_ERR_OVERLAP, "spheres " + std::to_string(j) + " and " + std::to_string(i) + " overlap");
      }
    for(int i = 0; i < nobj; ++i)
      if(!(radius[i] > 0.0) || !std::isfinite(eps_r[2 * i]) || !std::isfinite(eps_r[2 * i + 1]))
        throw OmxError(OMX_ERR_ARG, "non-positive radius or non-finite permittivity at sphere " + std::to_string(i));
    c->P = nobj;
    c->nmax = nmax;
    c->nf = nmax * (nmax + 2);
    c->N = 2 * c->nf * nobj;
    c->Np = (c->N + omx::kNB - 1) / omx::kNB * omx::kNB;
    c->xyz.assign(xyz, xyz + 3 * nobj);
    c->radius.assign(radius, radius + nobj);
    c->eps.resize(nobj);
    c->mu.resize(nobj);
    c->eps_sh.resize(nobj);
    c->ksippp.resize(nobj);
    c->ksiparppar.resize(nobj);
    c->gamma.resize(nobj);
    for(int i = 0; i < nobj; ++i) {
      c->eps[i] = kEps0 * C(eps_r, i);
      c->mu[i] = kMu0 * C(mu_r, i);
      c->eps_sh[i] = eps_r_sh ? kEps0 * C(eps_r_sh, i) : omx::mk(kEps0);
      c->ksippp[i] = ksippp ? C(ksippp, i) : omx::mk(0.0);
      c->ksiparppar[i] = ksiparppar ? C(ksiparppar, i) : omx::mk(0.0);
      c->gamma[i] = gamma ? C(gamma, i) : omx::mk(0.0);
    }
    c->bg_eps_r = bg_eps_r ? C(bg_eps_r, 0) : omx::mk(1.0);
    c->bg_mu_r = bg_mu_r ? C(bg_mu_r, 0) : omx::mk(1.0);
    c->have_geom = true;
    c->updated = c->solved = false;
  });
}

int omx_set_excitation(omx_context *c, double wavelength, double theta, double phi, const double *etheta,
                       const double *ephi, int sh) {
  return guard([&] {
    if(!c || !(wavelength > 0.0)) throw OmxError(OMX_ERR_ARG, "invalid excitation");
    c->lambda = wavelength;
    c->theta = theta;
    c->phi = phi;
    c->eth = etheta ? C(etheta, 0) : omx::mk(1.0);
    c->eph = ephi ? C(ephi, 0) : omx::mk(0.0);
    c->sh = sh ? 1 : 0;
    c->have_exc = true;
    c->updated = c->solved = false;
  });
}

int omx_set_solver(omx_context *c, int kind, double tol, int maxit, int restart) {
  return guard([&] {
    if(!c || kind < 0 || kind > 5 || !(tol > 0.0) || maxit < 1 || restart < 1 || restart > 256)
      throw OmxError(OMX_ERR_ARG, "invalid solver settings");
    c->kind = c->kind_req = kind;
    c->tol = tol;
    c->maxit = maxit;
    c->restart = restart;
    c->updated = c->solved = false;
  });
}

int omx_set_auto_budget(omx_context *c, int steps) {
  return guard([&] {
    if(!c || steps < 0) throw OmxError(OMX_ERR_ARG, "invalid budget");
    c->auto_budget = steps;
  });
}

int omx_set_graphs(omx_context *c, int on) {
  return guard([&] {
    if(!c) throw OmxError(OMX_ERR_ARG, "null context");
    HIPCHK(hipSetDevice(c->device));
    c->graphs = on != 0;
    if(!c->graphs) {
      HIPCHK(hipStreamSynchronize(c->st));
      HIPCHK(hipStreamSynchronize(c->st2));
      c->fg.reset();
      c->fg_sweep.reset();
    }
  });
}

int omx_set_autotune(omx_context *c, int on) {
  return guard([&] {
    if(!c) throw OmxError(OMX_ERR_ARG, "null context");
    c->autotune = on != 0;
  });
}

int omx_tune_query(int device, int Np, int nb, int fp64, int *split, int *trsv, double *times) {
  return guard([&] {
    std::lock_guard<std::mutex> g(g_tune_mu);
    auto it = g_tune.find(std::make_tuple(device, Np, nb, fp64 ? 1 : 0));
    if(it == g_tune.end()) throw OmxError(OMX_ERR_STATE, "shape not tuned");
    const TuneChoice &ch = it->second;
    if(split) *split = ch.split ? 1 : 0;
    if(trsv) *trsv = ch.trsv;
    if(times) {
      times[0] = ch.t_prod[0];
      times[1] = ch.t_prod[1];
      for(int v = 0; v < omx::kTrsvVariants; ++v) times[2 + v] = ch.t_trsv[v];
    }
  });
}

int omx_tune_reset(void) {
  std::lock_guard<std::mutex> g(g_tune_mu);
  g_tune.clear();
  return OMX_OK;
}

int omx_set_pivoting(omx_context *c, int mode) {
  return guard([&] {
    if(!c || (mode != OMX_PIVOT_BLOCK && mode != OMX_PIVOT_PARTIAL)) throw OmxError(OMX_ERR_ARG, "invalid pivoting");
    c->pivot = mode;
    c->factored = c->factored_sh = false;
    c->solved = false;
  });
}

int omx_set_lu32_gemm(omx_context *c, int mode) {
  return guard([&] {
    if(!c || (mode != OMX_GEMM_BF16X3 && mode != OMX_GEMM_FP32)) throw OmxError(OMX_ERR_ARG, "invalid gemm mode");
    c->lu32_gemm = mode;
    c->factored = c->factored_sh = false;
    c->solved = false;
  });
}

int omx_set_cg_tables(omx_context *c, int nmax, const double *const *tables) {
  return guard([&] {
    if(!c || nmax < 1 || nmax > omx::kMaxNmax || !tables) throw OmxError(OMX_ERR_ARG, "invalid tables");
    HIPCHK(hipSetDevice(c->device));
    size_t nf = (size_t)nmax * (nmax + 2), sz = nf * nf * nf;
    c->d_cg.ensure(sizeof(double) * 9 * sz, &c->total);
    for(int t = 0; t < 9; ++t) {
      if(!tables[t]) throw OmxError(OMX_ERR_ARG, "null table");
      HIPCHK(hipMemcpyAsync(c->d_cg.as<double>() + t * sz, tables[t], sizeof(double) * sz, hipMemcpyHostToDevice,
                            c->st));
    }
    HIPCHK(hipStreamSynchronize(c->st));
    c->cg_nmax = nmax;
  });
}

int omx_build_cg_tables(omx_context *c, int nmax) {
  return guard([&] {
    if(!c || nmax < 1 || nmax > omx::kMaxNmax) throw OmxError(OMX_ERR_ARG, "invalid nmax");
    HIPCHK(hipSetDevice(c->device));
    size_t nf = (size_t)nmax * (nmax + 2), sz = nf * nf * nf;
    c->d_cg.ensure(sizeof(double) * 9 * sz, &c->total);
    omx::run_cg(nmax, c->d_cg.as<double>(), c->st);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->st));
    c->cg_nmax = nmax;
  });
}

int omx_update(omx_context *c) {
  return guard([&] {
    if(!c || !c->have_geom || !c->have_exc) throw OmxError(OMX_ERR_STATE, "geometry and excitation must be set");
    HIPCHK(hipSetDevice(c->device));
    if(c->kind_req == OMX_SOLVER_AUTO)
      c->kind = c->N >= kAutoKrylovN ? OMX_SOLVER_GMRES32_IR : OMX_SOLVER_LU32_IR;
    c->krylov_s = c->kind_req == OMX_SOLVER_AUTO && c->kind == OMX_SOLVER_LU32_IR && c->sh;
    if(c->kind != OMX_SOLVER_ACA_GMRES) aca_release(c);
    alloc_all(c);
    const bool tune = c->autotune && is_lu(c->kind), f64 = c->kind == OMX_SOLVER_LU64;
    TuneChoice t;
    const bool known = tune && tune_lookup(c, 1, f64, &t);
    c->links_room = tune && f64 && (!known || t.trsv == 1);
    alloc_matrices(c);
    c->tuned = false;
    if(tune && !known) {
      t = single_tune(c, f64);
      if(c->links_room && t.trsv != 1) {  // no links after all
        c->d_dinv.release(&c->total);
        c->d_dinv2.release(&c->total);
      }
    }
    c->tuned = tune;
    if(tune) {
      set_trsv(c, c->lu, c->d_dinv, t.trsv);
      if(c->sh) set_trsv(c, c->lu_sh, c->d_dinv2, t.trsv);
      c->tuned_split = t.split;
    }
    const int P = c->P, nmax = c->nmax;
    // The plane wave and the objects' origin couplings run on the second
    // stream beside the pairs: they need the objects only, and one workgroup
    // per object leaves the device to the pairs.  The call returns once all is
    // enqueued; whatever reads its results follows on the context's stream.
    hipStream_t st = c->st, st2 = c->st2;
    HIPCHK(hipEventRecord(c->uev[0], st));
    upload_geometry(c);
    const double omega = c->omega();
    const cplx bge = kEps0 * c->bg_eps_r, bgm = kMu0 * c->bg_mu_r;
    omx::ObjArgs oa{P, nmax, omega, bge, bgm, c->d_xyz.as<double>(), c->d_radius.as<double>(),
                    c->d_eps.as<cplx>(), c->d_mu.as<cplx>(), c->d_eps_sh.as<cplx>(), c->d_sph.as<double>(),
                    c->d_ov.as<cplx>()};
    omx::run_objects(oa, st);
    HIPCHK(hipEventRecord(c->uev[1], st));
    HIPCHK(hipEventRecord(c->ujoin[0], st));
    HIPCHK(hipStreamWaitEvent(st2, c->ujoin[0], 0));
    omx::IncArgs ia{nmax, c->theta, c->phi, c->eth, c->eph, c->d_inc.as<cplx>()};
    omx::run_incident(ia, st2);
    HIPCHK(hipMemsetAsync(c->d_Q.p, 0, sizeof(cplx) * c->Np, st2));
    omx::OriginArgs og{P, nmax, c->waveK(), c->d_sph.as<double>(), c->d_ov.as<cplx>(), c->d_coef.as<double>(),
                       c->d_inc.as<cplx>(), c->d_incloc.as<cplx>(), c->d_Q.as<cplx>(), c->d_w.as<double>(), c->sh};
    omx::run_origin(og, st2);
    HIPCHK(hipEventRecord(c->ujoin[1], st2));
    const size_t lda = (size_t)c->Np;
    if(c->kind == OMX_SOLVER_ACA_GMRES) {
      if(!c->sh) c->aca[1].release(&c->total);
      auto build = [&] {
        aca_build(c, false);
        if(c->sh) aca_build(c, true);
      };
      try {
        build();
      } catch(OmxError &e) {  // without what is kept from the operators before
        if(e.code != OMX_ERR_MEMORY) throw;
        (void)hipGetLastError();
        aca_release(c);
        build();
      }
    } else {
      omx::PairArgs pa{P, nmax, omx::OV_T, c->waveK(), c->d_sph.as<double>(), c->d_ov.as<cplx>(),
                       c->d_coef.as<double>(), lda, c->d_S64.as<cplx>(), c->d_S32.as<float2>()};
      if(c->sh) {  // V in the same launch
        pa.tkind2 = omx::OV_TSH;
        pa.k2 = omx::mk(2.0 * pa.k.x, 2.0 * pa.k.y);  // PreconditionedMatrix.cpp:592
        pa.V64 = c->d_V64.as<cplx>();
        pa.V32 = c->d_V32.as<float2>();
      }
      omx::run_pairs(pa, st);
      if(c->d_S64.p) omx::run_pad64(c->d_S64.as<cplx>(), c->N, c->Np, lda, st);
      if(c->d_S32.p) omx::run_pad32(c->d_S32.as<float2>(), c->N, c->Np, lda, st);
      if(c->sh) {
        if(c->d_V64.p) omx::run_pad64(c->d_V64.as<cplx>(), c->N, c->Np, lda, st);
        if(c->d_V32.p) omx::run_pad32(c->d_V32.as<float2>(), c->N, c->Np, lda, st);
      }
    }
    HIPCHK(hipStreamWaitEvent(st, c->ujoin[1], 0));
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->uev[2], st));
    c->upd_timed = true;
    c->stats.N = c->N;
    c->stats.Np = c->Np;
    c->stats.device_bytes = c->total;
    c->updated = true;
    c->solved = false;
    c->factored = c->factored_sh = false;
    c->dirty32 = c->dirty32_sh = false;
  });
}

// The nine Clebsch-Gordan-type tables of the SH source for the context's
// nmax (Symbol.cpp:1036-1451), built once per nmax.
void ensure_cg(omx_context *c, hipStream_t st) {
  if(c->cg_nmax == c->nmax) return;
  size_t nf = (size_t)c->nf, sz = nf * nf * nf;
  c->d_cg.ensure(sizeof(double) * 9 * sz, &c->total);
  omx::run_cg(c->nmax, c->d_cg.as<double>(), st);
  c->cg_nmax = c->nmax;
}

// The second-harmonic source K and K1 of the context's x_int
// (PreconditionedMatrix.cpp:1347-1436, Geometry.cpp:250-310), on stream st.
void sh_source(omx_context *c, hipStream_t st) {
  HIPCHK(hipMemsetAsync(c->d_K.p, 0, sizeof(cplx) * c->Np, st));
  omx::ShArgs sa{c->P, c->nmax, c->omega(), kEps0 * c->bg_eps_r, kMu0 * c->bg_mu_r, c->d_radius.as<double>(),
                 c->d_eps.as<cplx>(), c->d_mu.as<cplx>(), c->d_eps_sh.as<cplx>(), c->d_kppp.as<cplx>(),
                 c->d_kpar.as<cplx>(), c->d_gam.as<cplx>(), c->d_ov.as<cplx>(), c->d_cg.as<double>(),
                 c->d_xint.as<cplx>(), c->d_K.as<cplx>(), c->d_K1.as<cplx>()};
  omx::run_shsrc(sa, st);
}

// The solution vectors to the caller's arrays (null: left out), after all of the
// context's work on its first stream: through pinned staging, so that the
// copies take one wait between them.
void read_vectors(omx_context *c, double *x_sca, double *x_int, double *x_sca_sh, double *x_int_sh) {
  double *dst[] = {x_sca, x_int, c->sh ? x_sca_sh : nullptr, c->sh ? x_int_sh : nullptr};
  const DBuf *src[] = {&c->d_x, &c->d_xint, &c->d_xsh, &c->d_xintsh};
  const size_t b = sizeof(cplx) * c->N;
  if(c->out_pin_bytes < 4 * b) {
    if(c->out_pin) (void)hipHostFree(c->out_pin);
    c->out_pin = nullptr;
    c->out_pin_bytes = 0;
    HIPCHK(hipHostMalloc(reinterpret_cast<void **>(&c->out_pin), 4 * b));
    c->out_pin_bytes = 4 * b;
  }
  for(int e = 0; e < 4; ++e)
    if(dst[e]) HIPCHK(hipMemcpyAsync(c->out_pin + e * b, src[e]->p, b, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  for(int e = 0; e < 4; ++e)
    if(dst[e]) std::memcpy(dst[e], c->out_pin + e * b, b);
}

int omx_solve(omx_context *c, double *x_sca, double *x_int, double *x_sca_sh, double *x_int_sh) {
  return guard([&] {
    if(!c || !c->updated) throw OmxError(OMX_ERR_STATE, "omx_update must precede omx_solve");
    HIPCHK(hipSetDevice(c->device));
    DrainOnError drain{c};
    const int N = c->N, P = c->P, nmax = c->nmax;
    double tf = 0, ts = 0, tsh = 0;
    HIPCHK(hipEventRecord(c->ev[0], c->st));
    // V does not depend on the fundamental solution, only its right-hand
    // side does: its factorisation runs on the second stream pair beside the
    // fundamental solve (not while profiling, which times each factorisation
    // alone)
    const bool lu_kind = is_lu(c->kind);
    const bool graphed =
        c->graphs && lu_kind && !c->profile && c->pivot == OMX_PIVOT_BLOCK && !c->factored && !c->krylov_s;
    SideEnqueue vq;
    if(c->sh && lu_kind && !c->factored_sh && !c->profile) {
      // V's factorisation starts once S's has passed a fraction of its
      // columns (by then S's trailing updates no longer fill the device),
      // and overlaps the rest of it and the fundamental refinement
      // (V's work is enqueued right at the mark, in the middle of S's
      // enqueueing: a wait on the mark event enqueued only after all of S's
      // work was seen to hold V back until S's end)
      const int mark = c->krylov_s ? 0 : (int)(c->sh_overlap * c->Np);
      auto start_v = [](void *arg) {
        omx_context *cc = static_cast<omx_context *>(arg);
        HIPCHK(hipStreamWaitEvent(cc->st2, cc->xev[0], 0));
        factor_enqueue(cc, true, cc->pivot);
      };
      if(mark > 0 && graphed) {
        factor_graphed(c, true, mark);
      } else if(mark > 0 && !c->factored) {
        c->lu.ev_mark = c->xev[0];
        c->lu.mark_col = mark;
        c->lu.on_mark = start_v;
        c->lu.mark_arg = c;
        try {
          factor_enqueue(c, false, c->pivot);
        } catch(...) {
          c->lu.ev_mark = nullptr;
          c->lu.on_mark = nullptr;
          throw;
        }
        c->lu.ev_mark = nullptr;
        c->lu.on_mark = nullptr;
      } else if(c->krylov_s && !c->factored) {
        // From kMarkN on, S's GMRES starts once V's factorisation has passed
        // krylov_mark of its columns: the first columns carry most of the
        // bulk-update work, which the GMRES products would only slow down, and
        // the panel-bound rest leaves the device room for them.  Below, the whole
        // factorisation is panel-bound and both start together.  Solves with 0 /
        // 0.25 / 0.5: N = 1280 2.89 / 3.29 / 3.57 ms, 2720 5.05 / 5.71 / 6.08, 5120
        // 11.4 / 11.7 / 12.6, 7200 21.0 / 22.6 / 24.0, 10240 42.1 / 41.6 / 43.0
        HIPCHK(hipEventRecord(c->xev[0], c->st));
        const double frac = c->krylov_mark >= 0.0 ? c->krylov_mark : c->N >= kMarkN ? 0.25 : 0.0;
        const int kmark = (int)(frac * c->Np);
        if(kmark > 0) {
          c->lu_sh.ev_mark = c->xev[3];
          c->lu_sh.mark_col = kmark;
          c->lu_sh.on_mark = nullptr;
        }
        vq.start(c, start_v);
        if(kmark > 0) {
          try {
            vq.join();  // V's factorisation enqueued, with its mark recorded
          } catch(...) {
            c->lu_sh.ev_mark = nullptr;
            throw;
          }
          c->lu_sh.ev_mark = nullptr;
          HIPCHK(hipStreamWaitEvent(c->st, c->xev[3], 0));
        }
      } else {
        HIPCHK(hipEventRecord(c->xev[0], c->st));
        start_v(c);
      }
    }
    if(graphed && !c->factored) factor_graphed(c, false, 0);
    // X_sca = S^{-1} Q (PreconditionedMatrixSolver.h:58)
    solve_system(c, false, c->d_Q.as<cplx>(), c->d_x.as<cplx>(), &c->stats.iterations, &c->stats.residual);
    HIPCHK(hipEventRecord(c->ev[1], c->st));
    // X_int = X_sca (.) Iaux (Solver.cpp:57-77)
    omx::vmul_ov(c->d_xint.as<cplx>(), c->d_x.as<cplx>(), c->d_ov.as<cplx>(), omx::OV_IAUX, P, nmax, nullptr, N, c->st);
    HIPCHK(hipEventRecord(c->ev[2], c->st));
    if(c->sh) {
      ensure_cg(c, c->st);
      HIPCHK(hipEventRecord(c->ev[3], c->st));
      sh_source(c, c->st);
      HIPCHK(hipEventRecord(c->ev[4], c->st));
      // the second-harmonic solve runs on the second stream, after the source
      // (and after V's factorisation has been enqueued there)
      HIPCHK(hipEventRecord(c->xev[1], c->st));
      vq.join();
      HIPCHK(hipStreamWaitEvent(c->st2, c->xev[1], 0));
      solve_system(c, true, c->d_K.as<cplx>(), c->d_xsh.as<cplx>(), &c->stats.iterations_sh, &c->stats.residual_sh);
      // X_int_SH = X_sca_SH (.) IauxSH1 - K1ana (Solver.cpp:95-116)
      omx::vmul_ov(c->d_xintsh.as<cplx>(), c->d_xsh.as<cplx>(), c->d_ov.as<cplx>(), omx::OV_IAUXSH1, P, nmax,
                   c->d_K1.as<cplx>(), N, c->st2);
      HIPCHK(hipEventRecord(c->xev[2], c->st2));
      HIPCHK(hipStreamWaitEvent(c->st, c->xev[2], 0));
      HIPCHK(hipEventRecord(c->ev[5], c->st));
    }
    HIPCHK(hipGetLastError());
    read_vectors(c, x_sca, x_int, x_sca_sh, x_int_sh);
    ts += elapsed(c, 0, 2);
    if(c->sh) {
      tsh = elapsed(c, 3, 4);
      ts += elapsed(c, 4, 5);
    }
    c->stats.t_factor_ms = tf;
    c->stats.t_solve_ms = ts;
    c->stats.t_sh_source_ms = tsh;
    c->solved = true;
  });
}

// ------------------------------------------------------------------ groups
// Batch buffers of a group solve in the leader context: the sweep's buffers
// that the batched factorisation, triangular solves and lockstep refinement
// use, at the group's padded order L->Np.
void group_alloc(omx_context *L, int nb, bool f64, bool sh) {
  auto &w = L->sw;
  size_t *T = &L->total;
  const size_t Np = L->Np, n2 = Np * Np;
  const int m = L->restart;
  aca_release_staging(L);
  w.S64.ensure(sizeof(cplx) * n2 * nb, T);
  if(f64) w.F64.ensure(sizeof(cplx) * n2 * nb, T); else w.S32.ensure(sizeof(float2) * n2 * nb, T);
  if(sh) {
    w.V64.ensure(sizeof(cplx) * n2 * nb, T);
    if(f64) w.F64sh.ensure(sizeof(cplx) * n2 * nb, T); else w.V32.ensure(sizeof(float2) * n2 * nb, T);
  }
  for(DBuf *b : {&w.Q, &w.x, &w.xsh, &w.K, &w.r, &w.w1, &w.w2}) b->ensure(sizeof(cplx) * Np * nb, T);
  for(DBuf *b : {&w.perm, &w.perm2}) b->ensure(sizeof(int) * Np * nb, T);
  for(DBuf *b : {&w.map, &w.map2}) b->ensure(sizeof(int) * Np * nb, T);
  for(DBuf *b : {&w.status, &w.status2}) b->ensure(sizeof(int) * 4 * nb, T);
  w.basis.ensure(sizeof(cplx) * Np * (m + 1) * nb, T);
  w.basisZ.ensure(sizeof(cplx) * Np * (m + 1) * nb, T);
  w.gpart.ensure(sizeof(cplx) * Np * omx::gemv_part_rows(nb), T);
  L->d_status.ensure(64, T);
}

int omx_solve_group(omx_context *L, int n, omx_context *const *mem) {
  return guard([&] {
    if(!L || n < 1 || !mem) throw OmxError(OMX_ERR_ARG, "omx_solve_group: leader, count and members required");
    for(int i = 0; i < n; ++i) {
      omx_context *m = mem[i];
      if(!m || m == L) throw OmxError(OMX_ERR_ARG, "omx_solve_group: member " + std::to_string(i) + " invalid");
      if(!m->updated) throw OmxError(OMX_ERR_STATE, "omx_solve_group: member " + std::to_string(i) + " not updated");
      if(m->device != L->device) throw OmxError(OMX_ERR_ARG, "omx_solve_group: members must share the leader's device");
      if(m->kind != mem[0]->kind || (m->kind != OMX_SOLVER_LU64 && m->kind != OMX_SOLVER_LU32_IR))
        throw OmxError(OMX_ERR_ARG, "omx_solve_group: members need one LU kind (lu64 or lu32ir)");
      if((m->sh != 0) != (mem[0]->sh != 0)) throw OmxError(OMX_ERR_ARG, "omx_solve_group: mixed SH flags");
      for(int j = 0; j < i; ++j)
        if(mem[j] == m) throw OmxError(OMX_ERR_ARG, "omx_solve_group: a member appears twice");
    }
    HIPCHK(hipSetDevice(L->device));
    DrainOnError drain{L};
    const bool f64 = mem[0]->kind == OMX_SOLVER_LU64, sh = mem[0]->sh != 0;
    int Np = 0;
    for(int i = 0; i < n; ++i) Np = std::max(Np, mem[i]->Np);
    // the leader runs the batch at the largest padded order with the first
    // member's refinement settings, in its sweep buffers only; its own
    // sizes and settings come back on every exit
    struct Restore {
      omx_context &c;
      int N, Np, kind, sh, maxit, restart, gemm;
      double tol;
      ~Restore() {
        c.N = N;
        c.Np = Np;
        c.kind = kind;
        c.sh = sh;
        c.maxit = maxit;
        c.restart = restart;
        c.lu32_gemm = gemm;
        c.tol = tol;
      }
    } restore{*L, L->N, L->Np, L->kind, L->sh, L->maxit, L->restart, L->lu32_gemm, L->tol};
    L->Np = Np;
    L->N = Np;
    L->kind = mem[0]->kind;
    L->sh = sh;
    L->tol = mem[0]->tol;
    L->maxit = mem[0]->maxit;
    L->restart = mem[0]->restart;
    L->lu32_gemm = mem[0]->lu32_gemm;
    const int nb = n;
    const size_t n2 = (size_t)Np * Np, lda = (size_t)Np;
    group_alloc(L, nb, f64, sh);
    const TuneChoice tune = L->autotune ? sweep_tune(L, nb, f64) : TuneChoice{L->lu32_gemm == OMX_GEMM_BF16X3, 0};
    auto &w = L->sw;
    hipStream_t st = L->st;
    for(DBuf *b : {&w.status, &w.status2}) HIPCHK(hipMemsetAsync(b->p, 0, b->bytes, st));
    HIPCHK(hipMemsetAsync(L->d_status.p, 0, 16, st));
    // the members' matrices and right-hand sides, bordered by the identity
    cplx *S64 = w.S64.as<cplx>(), *V64 = sh ? w.V64.as<cplx>() : nullptr;
    for(int z = 0; z < nb; ++z) HIPCHK(hipStreamWaitEvent(st, mem[z]->uev[2], 0));
    for(int z = 0; z < nb; ++z) {
      omx_context *m = mem[z];
      omx::pad_matrix64(S64 + z * n2, Np, m->d_S64.as<cplx>(), m->Np, st);
      if(f64) omx::pad_matrix64(w.F64.as<cplx>() + z * n2, Np, m->d_S64.as<cplx>(), m->Np, st);
      else omx::pad_matrix32(w.S32.as<float2>() + z * n2, Np, m->d_S64.as<cplx>(), m->Np, st);
      if(sh) {
        omx::pad_matrix64(V64 + z * n2, Np, m->d_V64.as<cplx>(), m->Np, st);
        if(f64) omx::pad_matrix64(w.F64sh.as<cplx>() + z * n2, Np, m->d_V64.as<cplx>(), m->Np, st);
        else omx::pad_matrix32(w.V32.as<float2>() + z * n2, Np, m->d_V64.as<cplx>(), m->Np, st);
      }
      omx::pad_vector(w.Q.as<cplx>() + z * lda, Np, m->d_Q.as<cplx>(), m->N, st);
    }
    HIPCHK(hipGetLastError());
    void *FS = f64 ? w.F64.p : w.S32.p, *FV = sh ? (f64 ? w.F64sh.p : w.V32.p) : nullptr;
    auto factor = [&](void *F, omx::LuWork &lw, hipStream_t fst) {
      const int rc = f64 ? omx::lu_factor<double2>(static_cast<double2 *>(F), Np, lda, lw, fst, nullptr)
                         : omx::lu_factor<float2>(static_cast<float2 *>(F), Np, lda, lw, fst, nullptr);
      if(rc) throw OmxError(OMX_ERR_DEVICE, "batched lu_factor launch failed (" + std::to_string(rc) + ")");
    };
    omx::LuWork lwS = sweep_lu(L, nb, false, tune.trsv), lwV{};
    lwS.split = tune.split;
    if(sh) {
      lwV = sweep_lu(L, nb, true, tune.trsv);
      lwV.split = tune.split;
      HIPCHK(hipEventRecord(L->xev[0], st));
      HIPCHK(hipStreamWaitEvent(L->st2, L->xev[0], 0));
      factor(FV, lwV, L->st2);
      HIPCHK(hipEventRecord(L->xev[1], L->st2));
    }
    factor(FS, lwS, st);
    std::vector<int> bad(nb, 0), iters(2 * nb, 0);
    std::vector<double> resid(2 * nb, 0.0);
    auto status_scan = [&](bool second) {
      std::vector<int> h(4 * nb);
      HIPCHK(hipMemcpyAsync(h.data(), (second ? w.status2 : w.status).p, sizeof(int) * 4 * nb,
                            hipMemcpyDeviceToHost, st));
      int g[2];
      HIPCHK(hipMemcpyAsync(g, L->d_status.p, sizeof(g), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      if(h[1] || g[1]) throw OmxError(OMX_ERR_DEVICE, "device wait timed out in a group solve");
      for(int z = 0; z < nb; ++z)
        if(h[4 * z]) bad[z] = 1;
    };
    auto refine = [&](bool second, omx::LuWork &lw, void *F, const cplx *A64, const cplx *rhs, cplx *x) {
      status_scan(second);
      Krylov gm = sweep_krylov(L, nb, A64);
      gm.prec = [L, F, &lw, Np, lda, f64](const cplx *in, cplx *out, const int *live) {
        lw.live = live;
        if(f64)
          omx::lu_solve<double2>(static_cast<const double2 *>(F), Np, lda, lw, in, out, L->st);
        else
          omx::lu_solve<float2>(static_cast<const float2 *>(F), Np, lda, lw, in, out, L->st);
        lw.live = nullptr;
      };
      gm.prec(rhs, x, nullptr);
      const int bmax = nb > 1 ? std::min(L->maxit, 4 * L->restart) : L->maxit;
      gm.solve(rhs, x, L->tol, bmax, L->restart);
      status_scan(second);
      for(int z = 0; z < nb; ++z) {
        if(!(gm.res[z] <= 1e3 * L->tol)) bad[z] = 1;
        iters[2 * z + (second ? 1 : 0)] = gm.its[z];
        resid[2 * z + (second ? 1 : 0)] = gm.res[z];
      }
    };
    // fundamental: S x = Q for every member, then each member's x and x_int
    refine(false, lwS, FS, S64, w.Q.as<cplx>(), w.x.as<cplx>());
    for(int z = 0; z < nb; ++z) {
      omx_context *m = mem[z];
      HIPCHK(hipMemcpyAsync(m->d_x.p, w.x.as<cplx>() + z * lda, sizeof(cplx) * m->Np, hipMemcpyDeviceToDevice, st));
      omx::vmul_ov(m->d_xint.as<cplx>(), m->d_x.as<cplx>(), m->d_ov.as<cplx>(), omx::OV_IAUX, m->P, m->nmax, nullptr,
                   m->N, st);
    }
    if(sh) {
      // each member's SH source from its own x_int, then V x = K in one batch
      for(int z = 0; z < nb; ++z) {
        omx_context *m = mem[z];
        ensure_cg(m, st);
        sh_source(m, st);
        omx::pad_vector(w.K.as<cplx>() + z * lda, Np, m->d_K.as<cplx>(), m->N, st);
      }
      HIPCHK(hipStreamWaitEvent(st, L->xev[1], 0));  // V's factorisation
      refine(true, lwV, FV, V64, w.K.as<cplx>(), w.xsh.as<cplx>());
      for(int z = 0; z < nb; ++z) {
        omx_context *m = mem[z];
        HIPCHK(hipMemcpyAsync(m->d_xsh.p, w.xsh.as<cplx>() + z * lda, sizeof(cplx) * m->Np, hipMemcpyDeviceToDevice,
                              st));
        omx::vmul_ov(m->d_xintsh.as<cplx>(), m->d_xsh.as<cplx>(), m->d_ov.as<cplx>(), omx::OV_IAUXSH1, m->P, m->nmax,
                     m->d_K1.as<cplx>(), m->N, st);
      }
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    HIPCHK(hipStreamSynchronize(L->st2));
    for(int z = 0; z < nb; ++z) {
      omx_context *m = mem[z];
      if(bad[z]) {
        // zero pivot in the block or a refinement short of the target: this
        // member alone, with the single-system path and its fallbacks
        if(omx_solve(m, nullptr, nullptr, nullptr, nullptr) != OMX_OK)
          throw OmxError(OMX_ERR_NOCONV, "omx_solve_group: member " + std::to_string(z) + ": " + omx_last_error());
        ++L->fallbacks;
        continue;
      }
      m->stats.iterations = iters[2 * z];
      m->stats.iterations_sh = iters[2 * z + 1];
      m->stats.residual = resid[2 * z];
      m->stats.residual_sh = resid[2 * z + 1];
      m->solved = true;
    }
    L->stats.sweep_batch = nb;
  });
}

int omx_read_solution(omx_context *c, double *x_sca, double *x_int, double *x_sca_sh, double *x_int_sh) {
  return guard([&] {
    if(!c || !c->solved) throw OmxError(OMX_ERR_STATE, "no solution: omx_solve or omx_solve_group first");
    HIPCHK(hipSetDevice(c->device));
    read_vectors(c, x_sca, x_int, x_sca_sh, x_int_sh);
  });
}

int omx_cross_sections(omx_context *c, double *out4) {
  return guard([&] {
    if(!c || !c->solved || !out4) throw OmxError(OMX_ERR_STATE, "omx_solve must precede omx_cross_sections");
    HIPCHK(hipSetDevice(c->device));
    omx::CrossArgs ca{c->P, c->nmax, c->d_x.as<cplx>(), c->sh ? c->d_xsh.as<cplx>() : nullptr,
                      c->d_incloc.as<cplx>(), c->d_w.as<double>(), c->d_ov.as<cplx>(), c->d_cross.as<double>()};
    omx::run_cross(ca, c->st);
    std::vector<double> part(4 * c->P);
    HIPCHK(hipMemcpyAsync(part.data(), c->d_cross.p, sizeof(double) * part.size(), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    double s[4] = {0, 0, 0, 0};
    for(int j = 0; j < c->P; ++j)
      for(int e = 0; e < 4; ++e) s[e] += part[4 * j + e];
    double rk = c->waveK().x;
    out4[0] = (-1. / (rk * rk)) * s[0];  // Result.cpp:576
    out4[1] = (1. / (rk * rk)) * s[1];   // Result.cpp:646
    out4[2] = (1. / (rk * rk)) * s[2];   // Result.cpp:675
    out4[3] = c->sh ? (1.0 / (4.0 * c->bg_eps_r.x * c->bg_mu_r.x)) * s[3] : 0.0;  // Result.cpp:760
  });
}

int omx_absorption_cross_section_sh(omx_context *c, double *out) {
  return guard([&] {
    if(!c || !c->solved || !out) throw OmxError(OMX_ERR_STATE, "omx_solve must precede omx_absorption_cross_section_sh");
    if(!c->sh || c->cg_nmax != c->nmax) throw OmxError(OMX_ERR_STATE, "no second-harmonic solution");
    HIPCHK(hipSetDevice(c->device));
    omx::AbsShArgs aa{c->P, c->nmax, c->omega(), kEps0 * c->bg_eps_r, kMu0 * c->bg_mu_r, c->d_radius.as<double>(),
                      c->d_eps.as<cplx>(), c->d_mu.as<cplx>(), c->d_eps_sh.as<cplx>(), c->d_gam.as<cplx>(),
                      c->d_cg.as<double>(), c->d_xint.as<cplx>(), c->d_xintsh.as<cplx>(), c->d_abscoef.as<cplx>(),
                      c->d_abssh.as<double>()};
    aa.bes = c->d_absbes.as<cplx>();
    omx::run_abssh(aa, c->st);
    HIPCHK(hipGetLastError());
    std::vector<double> part(c->P);
    HIPCHK(hipMemcpyAsync(part.data(), c->d_abssh.p, sizeof(double) * c->P, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    double s = 0.0;
    for(double v : part) s += v;
    *out = s;
  });
}

int omx_fields(omx_context *c, int npts, const double *xyz, double *E, double *H, double *E_sh, double *H_sh) {
  return guard([&] {
    if(!c || !c->solved) throw OmxError(OMX_ERR_STATE, "omx_solve must precede omx_fields");
    if(npts < 1 || !xyz || !E || !H) throw OmxError(OMX_ERR_ARG, "omx_fields: points and E, H outputs required");
    const bool sh = E_sh || H_sh;
    if(sh && (!E_sh || !H_sh)) throw OmxError(OMX_ERR_ARG, "omx_fields: E_sh and H_sh go together");
    if(sh && (!c->sh || c->cg_nmax != c->nmax)) throw OmxError(OMX_ERR_STATE, "no second-harmonic solution");
    HIPCHK(hipSetDevice(c->device));
    const int chunk = 1 << 16;
    const int cap = std::min(npts, chunk);
    c->d_fpts.ensure(sizeof(double) * 3 * cap, &c->total);
    c->d_fout.ensure(sizeof(cplx) * 12 * cap, &c->total);
    c->d_fown.ensure(sizeof(int) * cap, &c->total);
    // the last chunk is smaller than the others and may take more slices
    const int tail = npts % chunk ? npts % chunk : cap;
    const size_t pe = std::max((size_t)omx::fields_slices(c->P, cap, sh) * cap,
                               (size_t)omx::fields_slices(c->P, tail, sh) * tail);
    c->d_fpart.ensure(sizeof(cplx) * (sh ? 12 : 6) * pe, &c->total);
    for(int i0 = 0; i0 < npts; i0 += chunk) {
      const int n = std::min(chunk, npts - i0);
      cplx *o = c->d_fout.as<cplx>();
      HIPCHK(hipMemcpyAsync(c->d_fpts.p, xyz + 3 * (size_t)i0, sizeof(double) * 3 * n, hipMemcpyHostToDevice, c->st));
      omx::FieldArgs fa{c->P, c->nmax, sh ? 1 : 0, n, c->omega(), c->waveK(), kEps0 * c->bg_eps_r, kMu0 * c->bg_mu_r,
                        c->d_xyz.as<double>(), c->d_radius.as<double>(), c->d_eps.as<cplx>(), c->d_mu.as<cplx>(),
                        c->d_eps_sh.as<cplx>(), c->d_gam.as<cplx>(), sh ? c->d_cg.as<double>() : nullptr,
                        c->d_inc.as<cplx>(), c->d_x.as<cplx>(), c->d_xint.as<cplx>(), c->d_xsh.as<cplx>(),
                        c->d_xintsh.as<cplx>(), c->d_fpts.as<double>(), o, o + 3 * (size_t)cap, o + 6 * (size_t)cap,
                        o + 9 * (size_t)cap, c->d_fown.as<int>(), c->d_fpart.as<cplx>()};
      omx::run_fields(fa, c->st);
      HIPCHK(hipGetLastError());
      const size_t b = sizeof(cplx) * 3 * n, off = 6 * (size_t)i0;
      HIPCHK(hipMemcpyAsync(E + off, o, b, hipMemcpyDeviceToHost, c->st));
      HIPCHK(hipMemcpyAsync(H + off, o + 3 * (size_t)cap, b, hipMemcpyDeviceToHost, c->st));
      if(sh) {
        HIPCHK(hipMemcpyAsync(E_sh + off, o + 6 * (size_t)cap, b, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipMemcpyAsync(H_sh + off, o + 9 * (size_t)cap, b, hipMemcpyDeviceToHost, c->st));
      }
      HIPCHK(hipStreamSynchronize(c->st));
    }
  });
}

int omx_scattering_size(const omx_context *c) { return c ? c->N : 0; }

int omx_get_stats(const omx_context *c, omx_stats *out) {
  if(!c || !out) return OMX_ERR_ARG;
  *out = c->stats;
  if(c->upd_timed && hipEventSynchronize(c->uev[2]) == hipSuccess) {
    float ms = 0;
    if(hipEventElapsedTime(&ms, c->uev[0], c->uev[2]) == hipSuccess) out->t_update_ms = ms;
    if(hipEventElapsedTime(&ms, c->uev[1], c->uev[2]) == hipSuccess) out->t_assemble_ms = ms;
  }
  out->device_bytes = c->total;
  out->t_lu_gemm_ms = c->prof_gemm_ms;
  out->lu_gemm_flop = c->prof_flop;
  out->lu_gemm_launches = c->prof_launches;
  out->t_lu_panel_ms = c->prof_panel_ms;
  out->t_factor_total_ms = c->prof_total_ms;
  out->pivot_fallbacks = c->fallbacks;
  out->matvec_calls = (int)c->mv_calls;
  out->t_matvec_ms = c->mv_ms;
  out->matvec_bytes = c->mv_bytes;
  out->graph_captures = c->graph_captures;
  out->graph_launches = c->graph_launches;
  return OMX_OK;
}

int omx_set_profile(omx_context *c, int on) {
  return guard([&] {
    if(!c) throw OmxError(OMX_ERR_ARG, "null context");
    HIPCHK(hipSetDevice(c->device));
    for(auto &e : c->mv_ev)
      if(on && !e) HIPCHK(hipEventCreate(&e));
    c->profile = on != 0;
    c->prof_gemm_ms = c->prof_panel_ms = c->prof_flop = c->prof_total_ms = 0;
    c->prof_launches = 0;
    c->mv_calls = 0;
    c->mv_ms = 0;
    c->mv_bytes = 0;
  });
}

int omx_read_matrix(omx_context *c, int which, double *out) {
  return guard([&] {
    if(!c || !c->updated || !out) throw OmxError(OMX_ERR_STATE, "no assembled matrix");
    const DBuf &b = which == 0 ? c->d_S64 : c->d_V64;
    if(!b.p) throw OmxError(OMX_ERR_STATE, "matrix not held in FP64");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemcpy2DAsync(out, sizeof(cplx) * c->N, b.p, sizeof(cplx) * c->Np, sizeof(cplx) * c->N, c->N,
                            hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
  });
}

int omx_read_matrix_block(omx_context *c, int which, int row0, int col0, int nrows, int ncols, double *out) {
  return guard([&] {
    if(!c || !c->updated || !out) throw OmxError(OMX_ERR_STATE, "no assembled matrix");
    if(row0 < 0 || col0 < 0 || nrows < 1 || ncols < 1 || row0 + nrows > c->N || col0 + ncols > c->N)
      throw OmxError(OMX_ERR_ARG, "block outside the N x N matrix");
    const DBuf &b = which == 0 ? c->d_S64 : c->d_V64;
    if(!b.p) throw OmxError(OMX_ERR_STATE, "matrix not held in FP64");
    HIPCHK(hipSetDevice(c->device));
    const cplx *src = b.as<cplx>() + (size_t)col0 * c->Np + row0;
    HIPCHK(hipMemcpy2DAsync(out, sizeof(cplx) * nrows, src, sizeof(cplx) * c->Np, sizeof(cplx) * nrows, ncols,
                            hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
  });
}

int omx_aca_info(omx_context *c, int which, int *ranks, double *info) {
  return guard([&] {
    if(!c || which < 0 || which > 1) throw OmxError(OMX_ERR_ARG, "invalid arguments");
    const omx_context::AcaMat &m = c->aca[which];
    if(!m.built) throw OmxError(OMX_ERR_STATE, "no compressed operator (OMX_SOLVER_ACA_GMRES and omx_update first)");
    if(ranks) std::copy(m.rank.begin(), m.rank.end(), ranks);
    if(info) {
      info[0] = m.bytes;
      info[1] = 16.0 * (double)c->N * c->N;
      info[2] = m.ref_mb;
      info[3] = m.naca;
      info[4] = m.ndense;
      info[5] = m.rmax;
      info[6] = m.naca ? m.rsum / m.naca : 0.0;
    }
  });
}

int omx_aca_block(omx_context *c, int which, int i, int j, int *rank, double *U, double *V) {
  return guard([&] {
    if(!c || which < 0 || which > 1 || !rank || !U || !V) throw OmxError(OMX_ERR_ARG, "invalid arguments");
    const omx_context::AcaMat &m = c->aca[which];
    if(!m.built) throw OmxError(OMX_ERR_STATE, "no compressed operator (OMX_SOLVER_ACA_GMRES and omx_update first)");
    if(i < 0 || j < 0 || i >= m.P || j >= m.P) throw OmxError(OMX_ERR_ARG, "block outside the cluster");
    HIPCHK(hipSetDevice(c->device));
    const size_t b = (size_t)i * m.P + j, n = m.n;
    const int r = m.rank[b];
    *rank = r;
    if(r < 0) {
      HIPCHK(hipMemcpyAsync(U, m.where[b], sizeof(cplx) * n * n, hipMemcpyDeviceToHost, c->st));
    } else if(r > 0) {
      HIPCHK(hipMemcpyAsync(U, m.where[b], sizeof(cplx) * n * r, hipMemcpyDeviceToHost, c->st));
      HIPCHK(hipMemcpyAsync(V, m.where[b] + n * r, sizeof(cplx) * n * r, hipMemcpyDeviceToHost, c->st));
    }
    HIPCHK(hipStreamSynchronize(c->st));
  });
}

int omx_read_vector(omx_context *c, int which, double *out) {
  return guard([&] {
    if(!c || !c->updated || !out) throw OmxError(OMX_ERR_STATE, "nothing assembled");
    const DBuf *b = which == 0 ? &c->d_Q : which == 1 ? &c->d_K : which == 2 ? &c->d_K1 : &c->d_incloc;
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemcpyAsync(out, b->p, sizeof(cplx) * c->N, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
  });
}

int omx_dense_solve(omx_context *c, int N, const double *A, const double *b, double *x, int kind) {
  return guard([&] {
    if(!c || N < 1 || !A || !b || !x || (kind != OMX_SOLVER_LU64 && kind != OMX_SOLVER_LU32_IR))
      throw OmxError(OMX_ERR_ARG, "invalid dense solve");
    HIPCHK(hipSetDevice(c->device));
    DrainOnError drain{c};
    // reuse the context machinery with a synthetic "geometry" of the right
    // size; the geometry's sizes, solver kind and SH flag come back on every
    // exit (a failed solve must not leave the dense sizes behind: the next
    // omx_update would size its buffers from them)
    omx_context &ctx = *c;
    struct Restore {
      omx_context &c;
      int N, Np, kind, sh;
      ~Restore() {
        c.N = N;
        c.Np = Np;
        c.kind = kind;
        c.sh = sh;
        c.updated = false;
        c.solved = false;
        c.factored = c.factored_sh = false;
      }
    } restore{ctx, ctx.N, ctx.Np, ctx.kind, ctx.sh};
    ctx.N = N;
    ctx.Np = (N + omx::kNB - 1) / omx::kNB * omx::kNB;
    ctx.kind = kind;
    ctx.sh = 0;
    ctx.updated = false;
    ctx.links_room = false;
    const size_t Np = ctx.Np;
    ctx.d_x.ensure(sizeof(cplx) * Np, &ctx.total);
    ctx.d_Q.ensure(sizeof(cplx) * Np, &ctx.total);
    ctx.d_r.ensure(sizeof(cplx) * Np, &ctx.total);
    ctx.d_w1.ensure(sizeof(cplx) * Np, &ctx.total);
    ctx.d_w2.ensure(sizeof(cplx) * Np, &ctx.total);
    ctx.d_gpart.ensure(sizeof(cplx) * Np * omx::gemv_part_rows(1), &ctx.total);
    ctx.d_nrm.ensure(sizeof(double) * 256, &ctx.total);
    alloc_matrices(&ctx);
    HIPCHK(hipMemsetAsync(ctx.d_Q.p, 0, sizeof(cplx) * Np, ctx.st));
    HIPCHK(hipMemcpyAsync(ctx.d_Q.p, b, sizeof(cplx) * N, hipMemcpyHostToDevice, ctx.st));
    HIPCHK(hipMemcpy2DAsync(ctx.d_S64.p, sizeof(cplx) * Np, A, sizeof(cplx) * N, sizeof(cplx) * N, N,
                            hipMemcpyHostToDevice, ctx.st));
    omx::run_pad64(ctx.d_S64.as<cplx>(), N, (int)Np, Np, ctx.st);
    if(kind == OMX_SOLVER_LU32_IR) {
      std::vector<float2> a32((size_t)N * N);
      for(size_t i = 0; i < a32.size(); ++i) a32[i] = make_float2((float)A[2 * i], (float)A[2 * i + 1]);
      HIPCHK(hipMemcpy2DAsync(ctx.d_S32.p, sizeof(float2) * Np, a32.data(), sizeof(float2) * N, sizeof(float2) * N, N,
                              hipMemcpyHostToDevice, ctx.st));
      omx::run_pad32(ctx.d_S32.as<float2>(), N, (int)Np, Np, ctx.st);
      HIPCHK(hipStreamSynchronize(ctx.st));
    }
    ctx.factored = false;
    ctx.dirty32 = false;
    int it = 0;
    double res = 0;
    solve_system(&ctx, false, ctx.d_Q.as<cplx>(), ctx.d_x.as<cplx>(), &it, &res);
    HIPCHK(hipMemcpyAsync(x, ctx.d_x.p, sizeof(cplx) * N, hipMemcpyDeviceToHost, ctx.st));
    HIPCHK(hipStreamSynchronize(ctx.st));
    ctx.stats.iterations = it;
    ctx.stats.residual = res;
  });
}

int omx_solve_sweep(omx_context *c, int nl, const double *lambdas, const double *eps_r, const double *eps_r_sh,
                    int batch, double *x_sca, double *x_int, double *x_sca_sh, double *x_int_sh, double *xs,
                    int *iterations) {
  return guard([&] {
    if(!c || !c->have_geom || !c->have_exc || nl < 1 || !lambdas || batch < 0)
      throw OmxError(OMX_ERR_ARG, "invalid sweep (geometry, excitation and wavelengths required)");
    // the automatic choice in a batched sweep: V's mixed LU, and with the
    // second harmonic S by lockstep FP64 GMRES beside V's factorisation
    if(c->kind_req == OMX_SOLVER_AUTO) c->kind = OMX_SOLVER_LU32_IR;
    const bool krylov_s = c->kind_req == OMX_SOLVER_AUTO && c->sh && c->N >= kSweepKrylovN;
    if(!is_lu(c->kind)) throw OmxError(OMX_ERR_ARG, "sweeps need an LU solver kind");
    for(int l = 0; l < nl; ++l)
      if(!(lambdas[l] > 0.0)) throw OmxError(OMX_ERR_ARG, "non-positive wavelength");
    HIPCHK(hipSetDevice(c->device));
    DrainOnError drain{c};
    alloc_all(c);
    c->d_status.ensure(64, &c->total);
    const int P = c->P, N = c->N;
    // geometry and material constants on the device (as omx_update)
    upload_geometry(c);
    // batch size: at most 64 systems and half of the free device memory
    const double per = sweep_bytes(c, krylov_s);
    size_t fr = 0, tot = 0;
    HIPCHK(hipMemGetInfo(&fr, &tot));
    int nb = batch > 0 ? batch : 64;
    nb = std::max(1, std::min({nb, nl, (int)std::max(1.0, 0.5 * (double)(fr + c->sw.S64.bytes) / per)}));
    std::vector<cplx> eps((size_t)nl * P), eps_sh((size_t)nl * P);
    for(int l = 0; l < nl; ++l)
      for(int i = 0; i < P; ++i) {
        eps[(size_t)l * P + i] = eps_r ? kEps0 * C(eps_r, l * P + i) : c->eps[i];
        eps_sh[(size_t)l * P + i] = eps_r_sh ? kEps0 * C(eps_r_sh, l * P + i) : c->eps_sh[i];
      }
    auto off = [&](double *p, int l, size_t n) { return p ? p + 2 * n * l : nullptr; };
    std::vector<int> redo;
    int itmax[2] = {0, 0};
    double resmax[2] = {0, 0};
    HIPCHK(hipEventRecord(c->ev[6], c->st));
    for(int l0 = 0; l0 < nl; l0 += nb) {
      const int n = std::min(nb, nl - l0);
      std::vector<int> bad(n, 0), its(2 * n, 0);
      std::vector<double> res(2 * n, 0.0);
      sweep_chunk(c, n, lambdas + l0, eps.data() + (size_t)l0 * P, eps_sh.data() + (size_t)l0 * P,
                  off(x_sca, l0, N), off(x_int, l0, N), off(x_sca_sh, l0, N), off(x_int_sh, l0, N),
                  xs ? xs + 5 * l0 : nullptr, bad, its, res, krylov_s);
      for(int z = 0; z < n; ++z) {
        if(bad[z]) redo.push_back(l0 + z);
        if(iterations) {
          iterations[2 * (l0 + z)] = its[2 * z];
          iterations[2 * (l0 + z) + 1] = its[2 * z + 1];
        }
        for(int e = 0; e < 2; ++e) {
          itmax[e] = std::max(itmax[e], its[2 * z + e]);
          if(!bad[z]) resmax[e] = std::max(resmax[e], res[2 * z + e]);
        }
      }
    }
    HIPCHK(hipEventRecord(c->ev[7], c->st));
    HIPCHK(hipEventSynchronize(c->ev[7]));
    const float t_batch = elapsed(c, 6, 7);
    // systems the batch could not solve: one at a time with partial pivoting
    if(!redo.empty()) {
      // the batch's buffers are released first (its results are on the host), so
      // the one-at-a-time solves (which allocate a single system's matrices,
      // copies and bases) never hold memory beside a whole batch: the
      // context's peak stays the batch footprint a scheduler admitted
      c->sw.release(&c->total);
      c->d_sym.release(&c->total);
      const double lam0 = c->lambda;
      const std::vector<cplx> e0 = c->eps, es0 = c->eps_sh;
      const int piv0 = c->pivot;
      c->pivot = OMX_PIVOT_PARTIAL;
      try {
        for(int l : redo) {
          c->lambda = lambdas[l];
          for(int i = 0; i < P; ++i) {
            c->eps[i] = eps[(size_t)l * P + i];
            c->eps_sh[i] = eps_sh[(size_t)l * P + i];
          }
          int rc = omx_update(c);
          if(rc) throw OmxError(rc, omx_last_error());
          rc = omx_solve(c, off(x_sca, l, N), off(x_int, l, N), off(x_sca_sh, l, N), off(x_int_sh, l, N));
          if(rc) throw OmxError(rc, omx_last_error());
          if(xs) {
            rc = omx_cross_sections(c, xs + 5 * l);
            if(rc) throw OmxError(rc, omx_last_error());
            xs[5 * l + 4] = 0.0;
            if(c->sh) {
              rc = omx_absorption_cross_section_sh(c, xs + 5 * l + 4);
              if(rc) throw OmxError(rc, omx_last_error());
            }
          }
          if(iterations) {
            iterations[2 * l] = c->stats.iterations;
            iterations[2 * l + 1] = c->stats.iterations_sh;
          }
          ++c->fallbacks;
        }
      } catch(...) {
        c->lambda = lam0;
        c->eps = e0;
        c->eps_sh = es0;
        c->pivot = piv0;
        throw;
      }
      c->lambda = lam0;
      c->eps = e0;
      c->eps_sh = es0;
      c->pivot = piv0;
      c->updated = c->solved = false;
    }
    c->stats.N = c->N;
    c->stats.Np = c->Np;
    c->stats.iterations = itmax[0];
    c->stats.iterations_sh = itmax[1];
    c->stats.residual = resmax[0];
    c->stats.residual_sh = resmax[1];
    c->stats.t_solve_ms = t_batch;
    c->stats.sweep_batch = nb;
    c->stats.device_bytes = c->total;
  });
}

int omx_mem_info(omx_context *c, size_t *free_bytes, size_t *total_bytes, size_t *held_bytes) {
  return guard([&] {
    if(!c) throw OmxError(OMX_ERR_ARG, "null context");
    HIPCHK(hipSetDevice(c->device));
    size_t fr = 0, tot = 0;
    HIPCHK(hipMemGetInfo(&fr, &tot));
    if(free_bytes) *free_bytes = fr;
    if(total_bytes) *total_bytes = tot;
    if(held_bytes) *held_bytes = c->total;
  });
}

int omx_trim(omx_context *c) {
  return guard([&] {
    if(!c) throw OmxError(OMX_ERR_ARG, "null context");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->st));
    HIPCHK(hipStreamSynchronize(c->st2));
    c->fg.reset();
    c->fg_sweep.reset();
    auto &w = c->sw;
    DBuf *big[] = {&c->d_S64, &c->d_S32, &c->d_V64, &c->d_V32, &c->d_F64, &c->d_F64sh, &w.S64, &w.S32, &w.V64,
                   &w.V32, &w.F64, &w.F64sh, &w.basis, &w.basisZ, &w.gpart, &c->d_basis, &c->d_basisZ,
                   &c->d_gpart,  &c->d_sym};
    for(DBuf *b : big) b->release(&c->total);
    aca_release(c);
    c->ws_in.release(&c->total);
    c->updated = c->solved = false;
    c->factored = c->factored_sh = false;
  });
}

int omx_dense_solve_noalloc(omx_context *c, int N, double *A, size_t lda, const double *b, double *x) {
  return guard([&] {
    if(!c || !A || !b || !x) throw OmxError(OMX_ERR_ARG, "omx_dense_solve_noalloc: null argument");
    if(N < 1 || N > kNoAllocMaxN)
      throw OmxError(OMX_ERR_ARG, "omx_dense_solve_noalloc: N = " + std::to_string(N) + " is outside [1, " +
                                      std::to_string(kNoAllocMaxN) + "], the limit of its scratch array");
    const int Np = (N + omx::kNB - 1) / omx::kNB * omx::kNB;
    if(lda < (size_t)Np)
      throw OmxError(OMX_ERR_ARG, "omx_dense_solve_noalloc: lda = " + std::to_string(lda) +
                                      " is below N rounded up to 64 (" + std::to_string(Np) + ")");
    if(!c->scratch) throw OmxError(OMX_ERR_STATE, "omx_dense_solve_noalloc: context has no scratch address");
    HIPCHK(hipSetDevice(c->device));
    hipStream_t st = c->st;
    using L = NoAllocLayout;
    unsigned char *base = static_cast<unsigned char *>(c->scratch);
    auto ip = [&](size_t off) { return reinterpret_cast<int *>(base + off); };
    omx::LuWork w{};
    w.status = ip(L::status);
    w.perm = ip(L::perm);
    w.cand[0] = ip(L::cand);
    w.cand[1] = ip(L::cand) + L::gmax * omx::kNB;
    w.mdst = ip(L::map);
    w.msrc = ip(L::map) + (L::Np + 2 * omx::kNB);
    w.mcnt = ip(L::map) + 2 * (L::Np + 2 * omx::kNB);
    w.wlu = base + L::wlu;
    w.dinv = base + L::dinv;
    w.aux = c->aux;
    w.ev_next = c->lu_ev[0];
    w.ev_piv = c->lu_ev[1];
    w.ev_bulk = c->lu_ev[2];
    w.ev_pan = c->lu_ev[3];
    w.gmax = L::gmax;
    w.pivot = omx::kPivotPartial;
    w.nb = 1;
    cplx *rb = reinterpret_cast<cplx *>(base + L::rhs), *xs = reinterpret_cast<cplx *>(base + L::x);
    // the array keeps the last call's contents: the status words start at zero
    const int nz = (int)((L::perm - L::status) / sizeof(int));
    hipLaunchKernelGGL(zero_ints_kernel, dim3((nz + 255) / 256), dim3(256), 0, st, ip(L::status), nz);
    hipLaunchKernelGGL(stage_rhs_kernel, dim3((Np + 255) / 256), dim3(256), 0, st, reinterpret_cast<const cplx *>(b),
                       rb, N, Np);
    omx::run_pad64(reinterpret_cast<cplx *>(A), N, Np, lda, st);
    HIPCHK(hipGetLastError());
    const int rc = omx::lu_factor<double2>(reinterpret_cast<double2 *>(A), Np, lda, w, st, nullptr);
    if(rc) throw OmxError(OMX_ERR_DEVICE, "lu_factor launch failed (" + std::to_string(rc) + ")");
    auto status = [&]() {
      int s[2] = {0, 0};
      HIPCHK(hipMemcpyAsync(s, w.status, sizeof(s), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      if(s[1]) throw OmxError(OMX_ERR_DEVICE, "device wait timed out (code " + std::to_string(s[1]) + ")");
      if(s[0]) throw OmxError(OMX_ERR_SINGULAR, "zero pivot at column " + std::to_string(s[0] - 1));
    };
    status();
    omx::lu_solve<double2>(reinterpret_cast<const double2 *>(A), Np, lda, w, rb, xs, st);
    HIPCHK(hipMemcpyAsync(x, xs, sizeof(cplx) * N, hipMemcpyDeviceToDevice, st));
    HIPCHK(hipGetLastError());
    status();
  });
}

}  // extern "C"
