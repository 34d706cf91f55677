// omx_kernels.hpp -- launch interfaces shared by the HIP translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>


#include "omx_math.hpp"

namespace omx {

// per-object vector kinds, layout ov[kind][obj][pol][n], pol 0 = TE, 1 = TM
enum {
  OV_T = 0,      // getTLocal
  OV_TSH,        // getTLocalSH
  OV_IAUX,       // getIaux
  OV_IAUXSH1,    // getIauxSH1
  OV_IAUXSH2,    // getIauxSH2
  OV_TSH1O,      // getTLocalSH1_outer
  OV_TSH2O,      // getTLocalSH2_outer
  OV_CABS,       // getCabsAux (real, in .x)
  OV_SHRAD,      // [0][n] = j_n(k_j R), [1][n] = k_j j_n'(k_j R) + j_n / R
  OV_COUNT
};

constexpr int kCoefN = 2 * kMaxNmax + 2;
constexpr int kCoefStride = (kCoefN + 1) * (kCoefN + 1);
// Tables of square roots that do not depend on the pair, kCoefStride doubles
// each (fill_coef): formed in the kernels they were half of the arithmetic of
// an A / B coefficient and most of a workgroup's setup.
enum {
  CF_AP = 0, CF_AM, CF_BP, CF_BM,  // the recurrence's a+, a-, b+, b- (n, m)
  CF_IAP, CF_IBP,                  // 1 / a+, 1 / b+
  CF_A1, CF_A2,                    // sqrt((n-m)(n+m+1)), sqrt((n+m)(n-m+1))
  CF_G0, CF_G1, CF_G2,             // sqrt((n-m)(n+m)), sqrt((n-m)(n-m-1)), sqrt((n+m)(n+m-1))
  CF_LEGA, CF_LEGB,                // the Legendre recurrence of degree n, order m
  CF_DEG,                          // by degree, at CF_NU, CF_MU, CF_LEGP + n
  CF_COUNT
};
constexpr int CF_NU = 0, CF_MU = 64, CF_LEGP = 128;
// Spherical coordinates of a centre as the assembly keeps them: r, sin and cos
// of the polar angle, sin and cos of the azimuth.
constexpr int kSphDoubles = 5;

struct ObjArgs {
  int P, nmax;
  double omega;
  cplx bg_eps, bg_mu;                // absolute
  const double *xyz, *radius;
  const cplx *eps, *mu, *eps_sh;     // absolute
  double *sph;                       // out: kSphDoubles per centre
  cplx *ov;                          // out: per-object vectors
  // batches (blockIdx.z = system z): omega, eps, eps_sh and ov of system z at
  // omz[z], eps + z P, eps_sh + z P, ov + z zov (omz null: one system)
  const double *omz = nullptr;
  size_t zov = 0;
};

struct IncArgs {
  int nmax;
  double theta, phi;
  cplx etheta, ephi;
  cplx *inc;                         // out: [a_inc (nf); b_inc (nf)]
};

struct PairArgs {
  int P, nmax, tkind;                // tkind: OV_T for S, OV_TSH for V
  cplx k;                            // background wavenumber (k or 2k)
  const double *sph;
  const cplx *ov;
  const double *coef;
  size_t lda;
  cplx *S64;                         // optional FP64 output
  float2 *S32;                       // optional complex-FP32 output
  // batches (blockIdx.z = system z): wavenumber kz[z], ov + z zov, matrices + z zS
  const cplx *kz = nullptr;
  size_t zov = 0, zS = 0;
  // pair list (plist non-null): nlist unordered pairs, pair b = plist[b]
  // (i P + j, i < j): S_ij written to S64 / S32 + 2 b zblk and S_ji to
  // + (2 b + 1) zblk, with leading dimension lda
  const int *plist = nullptr;
  int nlist = 0;
  size_t zblk = 0;
  // a second matrix in the same launch (either pointer non-null): V beside S
  int tkind2 = 0;
  cplx k2 = {0.0, 0.0};
  const cplx *kz2 = nullptr;
  cplx *V64 = nullptr;
  float2 *V32 = nullptr;
};

struct OriginArgs {
  int P, nmax;
  cplx k;
  const double *sph;
  const cplx *ov;
  const double *coef;
  const cplx *inc;
  cplx *incloc;                      // out: N
  cplx *Q;                           // out: N
  double *w;                         // out: [2][P][nf]; the second half (at 2k) with sh only
  int sh;
  // batches (blockIdx.z = system z): wavenumber kz[z], ov + z zov,
  // incloc/Q + z zvec, w + z zw
  const cplx *kz = nullptr;
  size_t zov = 0, zvec = 0, zw = 0;
};

struct CrossArgs {
  int P, nmax;
  const cplx *x, *xsh, *incloc;
  const double *w;
  const cplx *ov;
  double *out;                       // [nb][P][4]
  // nb systems: the vectors zvec, w zw and ov zov apart
  int nb = 1;
  size_t zvec = 0, zw = 0, zov = 0;
};

// Result::getEHFields / setFields (Result.cpp:74-301, 797-933): E and H at
// omega and 2 omega at npts Cartesian points, Cartesian components.
struct FieldArgs {
  int P, nmax, sh, npts;
  double omega;
  cplx waveK, bg_eps, bg_mu;               // background wavenumber; absolute eps, mu
  const double *xyz, *radius;              // object centres (Cartesian) and radii
  const cplx *eps, *mu, *eps_sh, *gamma;   // absolute
  const double *tab;                       // nine tables (SH bulk term inside spheres)
  const cplx *inc;                         // [a_inc; b_inc]
  const cplx *x, *xint, *xsh, *xintsh;     // solution vectors (N each)
  const double *pts;                       // 3 npts
  cplx *E, *H, *Esh, *Hsh;                 // 3 npts each; Esh, Hsh unused without sh
  int *owner;                              // workspace: npts
  cplx *part;                              // workspace: fields_slices() x (sh ? 12 : 6) x npts
};
int fields_slices(int P, int npts, int sh);
void run_fields(const FieldArgs &a, hipStream_t st);

// nb > 1: a batch of nb systems in one launch (the batch fields of the args)
void run_objects(const ObjArgs &a, hipStream_t st, int nb = 1);
void run_incident(const IncArgs &a, hipStream_t st);
void run_pairs(const PairArgs &a, hipStream_t st, int nb = 1);
void run_origin(const OriginArgs &a, hipStream_t st, int nb = 1);
void run_cross(const CrossArgs &a, hipStream_t st);
// identity padding of nb matrices zs elements apart
void run_pad64(cplx *A, int N, int Np, size_t lda, hipStream_t st, int nb = 1, size_t zs = 0);
void run_pad32(float2 *A, int N, int Np, size_t lda, hipStream_t st, int nb = 1, size_t zs = 0);
void fill_coef(double *dev, hipStream_t st);  // CF_COUNT x kCoefStride

// ---------------------------------------------------------------- ACA
struct AcaArgs {
  int n, nblk;       // block order (<= 256) and blocks in the launch
  double eps;        // compression tolerance
  const cplx *A;     // nblk blocks, n x n column-major, n^2 apart
  cplx *U, *V;       // nblk slots of n^2: U column p at U + p n, V row p at V + p n
  int *rank;         // out: nblk
};
void run_aca(const AcaArgs &a, hipStream_t st);
// block b's factors, U (n x r) then V (r x n), copied to pool + off[b]
void run_aca_pack(const cplx *U, const cplx *V, int n, int nblk, const int *rank, cplx *pool, const size_t *off,
                  hipStream_t st);

// One off-diagonal block of a compressed operator: rank -1 dense (n x n
// column-major at M), r > 0 compressed (U n x r at M, V r x n at M + n r,
// V x_j kept at t + toff).
struct AcaDesc {
  const cplx *M;
  int j, rank, toff;
};
struct AcaOp {
  int P, n, N, Np, G;          // G groups of a block row's blocks (0 when P = 1)
  const AcaDesc *desc;         // sorted by block row, rows at rowptr[i] .. rowptr[i+1]
  const int *rowptr, *acalist; // acalist: desc indices of the naca compressed blocks
  int naca;
  cplx *t, *part;              // V x products; partial rows [G][P][n]
};
// y = S x for the compressed operator S (identity diagonal blocks, identity
// on the padding rows N .. Np-1)
void aca_matvec(const AcaOp &op, const cplx *x, cplx *y, hipStream_t st);

// ---------------------------------------------------------------- LU
constexpr int kNB = 64;        // LU block size (panel width, padding granule)
constexpr int kPanelRows = 192; // fewest rows of the panel held by one workgroup (tournament)

// Distances between the systems of a batch (element counts of each buffer);
// all zero for a single system.  A batch runs with blockIdx.z = system.
struct BatchStrides {
  size_t a = 0;    // matrices (elements of T)
  size_t inv = 0;  // per-panel inverse sets (elements of T)
  size_t vec = 0;  // right-hand sides and solutions (complex FP64 elements)
  int perm = 0;    // permutations
  int map = 0;     // row maps (msrc)
  int status = 0;  // status words
};

struct LuWork {
  // device scratch of one factorization
  int *perm;            // Np: final row permutation (row i of P A is row perm[i] of A)
  int *cand[2];         // tournament candidates, ping-pong, [Gmax][NB]
  int *mdst, *msrc;     // gather maps: tournament rows mdst <- msrc, mcnt of 2 NB entries at
  int *mcnt;            // the start; block pivoting row i <- msrc[i]
  int *status;          // [0]: singular pivot column+1, [1]: wait timeout
  void *wlu;            // NB x NB complex: the tournament's selected-block factors
  void *dinv;           // per panel [L11^{-1} | U11^{-1}], 2 NB^2 elements of T, column-major
  bool links = false;   // FP64 factors solved by variant 1: the triangular solves' links follow in dinv
  hipStream_t aux;      // look-ahead stream of the panel pivoting
  hipEvent_t ev_next, ev_piv, ev_bulk, ev_pan;
  int gmax;
  int pivot;            // kPivotBlock or kPivotPartial
  int nb = 1;           // systems in the batch (block pivoting only when > 1)
  BatchStrides bs;      // their strides; the pointers above are system 0's
  const int *live = nullptr;  // lu_solve: systems whose flag (KF_COUNT ints apart) is 0 are left out (null: none)
  int trsv = 0;              // triangular-solve variant (kTrsvVariants; 0: the default)
  bool split = true;             // FP32 factors: bulk updates on the split-bf16 MFMA
  hipEvent_t ev_mark = nullptr;  // when set: recorded on the bulk stream once the
  int mark_col = 0;              // factorisation has passed column mark_col, and
  void (*on_mark)(void *) = nullptr;  // then on_mark(mark_arg) is called (on the host,
  void *mark_arg = nullptr;           // in the middle of the enqueueing)
};
// Elements of T in a factorisation's dinv: 2 NB^2 per panel, and with links as many
// of them, from links_at on.
inline size_t links_at(int Np) { return 2 * (size_t)64 * Np; }
inline size_t dinv_elems(int Np, bool links) { return (links ? 2 : 1) * links_at(Np); }

// Pivot search of a panel: among the rows of its diagonal block only
// (followed by iterative refinement), or over the whole column (tournament).
constexpr int kPivotBlock = 0;
constexpr int kPivotPartial = 1;

// Optional per-launch timing of the factorisation (events on the same stream).
struct LuProf {
  hipEvent_t *ev = nullptr;  // 4 events per panel pair: panel work start/end (look-ahead
                             // stream), bulk update start/end (main stream)
  int cap = 0;               // pairs the pool covers
  int used = 0;              // pairs recorded by the last factorisation
  double gemm_flop = 0.0;    // algorithmic flop of the recorded bulk updates (8 m n k each)
  int gemm_launches = 0;     // their kernel launches
};

// Factor the Np x Np complex matrix in place (P A = L U); T = double2 or float2.
template <typename T>
int lu_factor(T *A, int Np, size_t lda, LuWork &w, hipStream_t st, LuProf *prof = nullptr);
// Triangular-solve variants: super-block size (64-row blocks per workgroup)
// and when the near-phase tiles are loaded (0: as used, 1: at kernel start,
// 2: after the far phase).  Variant 0 is the default of each type.
constexpr int kTrsvVariants = 3;
// The bulk updates of an FP32 factorisation's first four panels on the columns
// behind them (M = N = Np - 256) as it runs them with either product: one with K =
// 256 (split) or two with K = 128, on nb matrices sA apart.  A timing probe for the
// autotuner; nothing to do up to Np = 256.  (A's contents are overwritten.)
void bulk_update_probe(float2 *A, int Np, size_t lda, int nb, size_t sA, bool split, hipStream_t st);
// The triangular solves' links of factored FP64 matrices (with w.links; lu_factor ends
// with them).
void lu_links(const double2 *A, int Np, size_t lda, const LuWork &w, hipStream_t st);
// Solve with the factors: x = A^{-1} b, vectors always complex FP64.
template <typename T>
void lu_solve(const T *A, int Np, size_t lda, LuWork &w, const cplx *b, cplx *x, hipStream_t st);

// ---------------------------------------------------------------- iterative
// Partial sums of y = A x for nb systems (matrices sA, vectors sv apart), or of
// its complex-FP32 copy (FP64 vectors and sums): part[z][k][N], k < the returned
// number of column parts (<= kGemvSplitMax), chosen for `live` working systems.
// Systems whose flag (KF_COUNT ints apart; null: all) is 0 are left out.
int gemv_partial(const cplx *A, size_t lda, int N, const cplx *x, cplx *part, hipStream_t st, int nb = 1,
                 size_t sA = 0, size_t sv = 0, const int *flag = nullptr, int live = 1);
int gemv_partial(const float2 *A, size_t lda, int N, const cplx *x, cplx *part, hipStream_t st,
                 const int *flag = nullptr);
constexpr int kGemvSplit = 32, kGemvSplitMax = 96;  // column parts: most of a batch's product, of a single one's
inline size_t gemv_part_rows(int nb) { return std::max(kGemvSplitMax, kGemvSplit * nb); }  // vectors of partial sums

// y = S x for nb assembled scattering matrices from half their blocks: S_ji[p][q]
// is S_ij[p][q] times (T_j / T_i)[p] and the parity sign of (p, q), so a pair's two
// products read one block, for each row p the one of the larger |T[p]|.
// Scratch: sym_scratch(P, nmax, nb) complex values for nb systems.
struct SymArgs {
  int P, nmax, Np;
  size_t lda;
  const cplx *ov;  // the rows' factors T, of kind tkind (OV_T: S, OV_TSH: V)
  int tkind;
  cplx *scratch;
  int nb = 1;
  size_t sA = 0, sv = 0, zov = 0;  // matrices, vectors and ov of the systems apart
  const int *flag = nullptr;       // systems whose flag (KF_COUNT ints apart) is 0 are left out
};
size_t sym_scratch(int P, int nmax, int nb);
bool sym_pays(int nmax, bool f32);  // whether such a product is the faster one at this block order
void sym_product(const SymArgs &a, const cplx *A, const cplx *x, cplx *y, hipStream_t st);
void sym_product(const SymArgs &a, const float2 *A, const cplx *x, cplx *y, hipStream_t st);

// GMRES with its small algebra on the device (omx_krylov.hip), nb systems in
// lockstep: the state of each, and the vectors they share.
enum { KF_LIVE = 0, KF_ACTIVE, KF_J, KF_ITS, KF_STALL, KF_TINY, KF_COUNT = 8 };  // flags, ints
enum { KS_BN = 0, KS_PREV, KS_RES, KS_COUNT = 4 };                              // scalars, doubles
struct KryState {
  int n, m, nb, j;     // order, restart length (<= 256), systems, step of the cycle
  double tol;
  int maxit;
  cplx *c;             // [nb][kry_cplx(m)]: Hessenberg columns, g, rotations, y, h
  double *sc;          // [nb][KS_COUNT]
  int *fl;             // [nb][KF_COUNT]
  cplx *part;          // [2][nb][kry_blocks(n)][m + 2]
  double *pnrm;        // [2][nb][kry_blocks(n)]
  cplx *V;             // basis: vector k of system z at V + k ldk + z sz
  const cplx *Z;       // preconditioned basis, laid out alike (V itself without one)
  size_t ldk, sz;
  cplx *r, *w;         // residual and work vector, system z at + z sv (as b and x)
  size_t sv;
};
__host__ __device__ inline size_t kry_cplx(int m) {
  return (size_t)m * (m + 1) + (m + 1) + 3 * (size_t)m + (m + 2);
}
int kry_blocks(int n);
// Arnoldi step s.j after its product: partial sums gpart + z sg + k n, k < ns, or
// the product itself in s.w (ns 0).  host (pinned, [nb][2]): the system goes on,
// and the binary digits that its residual has to fall to the goal.
void kry_step(const KryState &s, const cplx *gpart, int ns, size_t sg, int *host, hipStream_t st);
void kry_end_cycle(const KryState &s, cplx *x, bool tiny, bool batch, hipStream_t st);
// b - A x and the restart's decisions; ns as above, 0: no product (x = 0), -1:
// the product is in s.w
void kry_restart(const KryState &s, const cplx *b, cplx *x, const cplx *gpart, int ns, size_t sg, bool first,
                 bool batch, int *host, hipStream_t st);

// level-1 helpers (omx_iter.hip)
void demote(float2 *y, const cplx *x, size_t n, hipStream_t st);                 // y = (c64) x
// p[0..n) = 0 by a kernel (a memset node must not go into a captured graph)
void zero_ints(int *p, int n, hipStream_t st);
// dst (Nd x Nd) = src (Ns x Ns, Ns <= Nd) bordered by the identity, in FP64 or
// rounded to complex FP32; dst[0, Nd) = src[0, Ns) followed by zeros
void pad_matrix64(cplx *dst, int Nd, const cplx *src, int Ns, hipStream_t st);
void pad_matrix32(float2 *dst, int Nd, const cplx *src, int Ns, hipStream_t st);
void pad_vector(cplx *dst, int Nd, const cplx *src, int Ns, hipStream_t st);
void vmul_ov(cplx *y, const cplx *x, const cplx *ov, int kind, int P, int nmax, const cplx *sub, int n,
             hipStream_t st, int nb = 1, size_t zvec = 0, size_t zov = 0);     // y = x (.) ov[kind] - sub
void nrm2sq(const cplx *x, int n, double *part, double *out, hipStream_t st);

}  // namespace omx
