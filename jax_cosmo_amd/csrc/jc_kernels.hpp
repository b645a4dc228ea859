// Kernel argument blocks and host-side launchers shared by the translation
// units of libjc_limber.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace jc {

// Fixed table sizes of the reference discretisation.
constexpr int NCHI = 256;     // chi table nodes, background.py:199 (steps=256)
constexpr int NGROW = 128;    // growth table nodes, background.py:443 (steps=128)
constexpr int NHF_K = 257;    // halofit ln k Simpson nodes, power.py:111 (N=256)
constexpr int NHF_R = 256;    // halofit ln R grid, power.py:92
constexpr int NROMB = 129;    // sigma_8 Romberg samples, power.py:76 (divmax=7)
constexpr int NWL_J = 257;    // per-z weak-lensing Simpson nodes, probes.py:51
constexpr int MAXT = 10;      // tracers per request handled by the Limber kernel
constexpr int NWL_MAX = 10;   // weak-lensing bins per kernel launch

// constants.py:23-27: intrinsic-alignment normalisation C_1 and the critical
// density [h^2 M_sun Mpc^-3]
constexpr double C1_IA = 5.0e-14;
constexpr double RHOCRIT = 2.7750e11;

// Per (cosmology, a-node) record consumed by the Limber kernel, in floats
// (each slot holds 1 + ND floats for the derivative kernels).
enum CoefSlot {
  CF_INV_CHI = 0,  // 1 / max(chi, 1)     (k = (ell + 1/2) / max(chi, 1))
  CF_CHI1,         // max(chi, 1)         (1/k)
  CF_LNINVCHI,     // -ln max(chi, 1)     (ln k)
  CF_WGT,          // Simpson weight * dchi/da / max(chi^2, 1) / c^2
  CF_G2P,          // D(a)^2 * pknorm
  CF_LGRNL,        // log2 R_nl = -log2 k_nl
  CF_RNL,          // R_nl
  CF_KNL,          // k_nl
  CF_AN, CF_BN, CF_LGCF3, CF_GAM3, CF_ALPHA, CF_BETA, CF_NU, CF_F1X3, CF_F2,
  CF_CHI,          // chi(a)
  CF_GROWTH,       // D(a)
  CF_MU,           // halofit mu_n (0 for takahashi2012)
  NCOEF
};
// The record of forward calls in transfer-table mode (same size).  The
// reference's per-point products of an a-node factor and a multipole factor
// are split so that each slot holds everything that depends on a alone: with
// l = ell + 1/2, k = l / max(chi, 1) and y = k R_nl,
//   table position      u = ln(l) invh + FT_Q + FT_T
//   Delta_L^2         d2l = T^2 k^n_s l^3 FT_G3
//   y                     = l FT_YC,  log2 y = log2 l + FT_LA
//   1 + mu/y + nu/y^2     = 1 + (FT_MU + FT_NU / l) / l
//   (c f3 y)^(3-gamma)    = 2^(FT_GAM log2 y + FT_GC)
// and M(a, ell) = l^-3 FT_AW [bracket], whose l^-3 leaves the sum over a.
// Slots 0-15 are read as four float4.
enum FwdSlot {
  FT_Q = 0,  // int32 bits: floor of (-ln max(chi, 1) - lo) invh, and its
  FT_T,      // fraction (lo, invh: the transfer table's grid)
  FT_G3,     // D^2 pknorm / (2 pi^2 max(chi, 1)^3)
  FT_LA,     // log2(R_nl / max(chi, 1))
  FT_YC,     // R_nl / max(chi, 1)
  FT_MU,     // mu_n max(chi, 1) / R_nl
  FT_NU,     // nu_n (max(chi, 1) / R_nl)^2
  FT_BETA,
  FT_F1X3,
  FT_F2,
  FT_GAM,    // 3 - gamma_n
  FT_GC,     // (3 - gamma_n) log2(c_n f3)
  FT_ALPHA,
  FT_BN,
  FT_AN,
  FT_AW,     // 2 pi^2 max(chi, 1)^3 x Simpson weight x dchi/da / max(chi^2, 1) / c^2
  FT_CHI = CF_CHI,
};
static_assert(NCOEF == 20, "FwdSlot shares the record of CoefSlot");
// Per-cosmology record (EH98 constants and the lensing prefactor).
enum CrecSlot {
  CR_FB = 0, CR_FC, CR_INV13KEQ, CR_BETAC18, CR_C14A, CR_SHD, CR_ALPHAB, CR_BETAB,
  CR_BETANODE, CR_LNKSILK, CR_NS, CR_WLCONST, CR_PKNORM, CR_LNINV13, CR_BNODE_SHD, CR_BB_SHD,
  CR_EHLO,    // ln k at the first node of the transfer table
  CR_EHINVH,  // 1 / (its ln k spacing)
  CR_ALPHAG, CR_TQ, CR_NW,  // the no-wiggle transfer form
  NCREC_USED
};
constexpr int NCREC = 21;
// Intervals of the per-cosmology transfer table: cubic Hermite pieces of
// T(k) k^(n_s/2) uniform in ln k over the k range of one forward call (16 KB
// per cosmology; interpolation error below 1e-6 of T).
constexpr int NEHQ = 1023;
// The adjoint's table of theta derivatives has a row of 8 floats (7
// derivatives, one pad) at each of the NEHQ + 1 nodes of the same grid (32 KB
// per cosmology, read through the L2); 4-point Lagrange interpolation.
constexpr int NEHD_ROW = 8;

struct RJob;
struct RCol;

// Segments of the chi and growth tables at a node of the a-grid
// (interpolate.py:12-37): table nodes i, j and the fraction t of
// f[i] + (f[j] - f[i]) t.
struct ASeg {
  double tc, tg;
  int16_t ci, cj, gi, gj;
};

struct TablesArgs {
  const double* params;   // [B][8] Cosmology(...) parameters
  const double* seeds;    // [B][8] d param / d direction (ND = 1; the 7 directions of ND = 7 are the parameters)
  int B, Na;
  const double* a_list;   // [Na] scale factors
  const double* a_wgt;    // [Na] quadrature weight of each node (0 = evaluation only)
  const double* atab_chi; // [256]
  const double* atab_g;   // [128]
  const double* hf_lnk;   // [257]
  const float* hf_k32;    // [257] exp(hf_lnk) as float
  const double* hf_kp;    // [257][4] k^2, k^4, k^6, 0 at k = exp(hf_lnk)
  const double* hf_E;     // [257][256] exp(-(k_i R_j)^2)
  const double* logr;     // [256]
  // cosmology-independent node quantities (host-computed once per context)
  const double* chi_nodes;  // [256][8]: a_i, ln a_i, 1/a_i, a_mid, ln a_mid, 1/a_mid, h_i (chi RK4 in ln a)
  const double* g_nodes;    // [128][8]: x_i, ln x_i, 1/x_i, x_mid, ln x_mid, 1/x_mid (growth RK4 in a)
  const double* gg_nodes;   // [128][8]: as chi_nodes on the growth grid (gamma growth RK4 in ln a)
  const double* romb;       // [129][4]: k, 1/k, ln k, Romberg weight x k (k W(8k))^2/(2 pi^2) at the sigma_8 nodes
  const double* hf_nodes;   // [257][4]: k, 1/k, ln k, Simpson weight x k^3/(2 pi^2) at k = exp(hf_lnk)
  const double* hf_R2;      // [256] R^2 at R = exp(logr)
  const double* a_ln;       // [Na] ln a of the a-grid, or null (computed in the kernel)
  const ASeg* a_seg;        // [Na] table segments of the a-grid, or null
  // kernels local in z: number counts n b H (probes.py:77-99) and the NLA
  // intrinsic-alignment terms of weak-lensing bins (probes.py:102-129)
  int nLoc;
  const double* loc_nb;   // [nLoc][Na] cosmology-independent factor at each node
  const int* loc_col;     // [nLoc] tracer column
  const int* loc_mode;    // [nLoc] LOC_* flags
  int Tpad;
  float* chitab;          // [B][256][2][W] (chi, slope of segment i)
  float* coef;            // [B][Na][NCOEF][W]
  float* crec;            // [B][NCREC][W]
  float* R;               // [B][Na][Tpad][W]
  double* dbg;            // optional [B][DBG_STRIDE] FP64 intermediates
  int dbg_stride;
  const int* dB;          // optional device count: blocks >= *dB exit (grid sized for B)
  int transfer_model;     // 0: eisenhu_osc, 1: eisenhu (no wiggles)
  int halofit_model;      // 0: takahashi2012, 1: smith2003
  int growth_model;       // 0: growth ODE (background.py:443-487), 1: f = Omega_m(a)^gamma (background.py:515-582)
  double gamma;           // growth index of model 1
  // calls in table mode (forward, adjoint): build the transfer table at the end of the
  // table kernel over the ln k range of these multipoles
  float4* ehtab;          // [B][NEHQ] or null
  float* ehtab7;          // adjoint calls: [B][NEHQ + 1][8] theta derivatives at the table's nodes, or null
  const double* ell;      // [n_ell]
  int n_ell;
  // served batches: cosmology c's multipoles are instead the ell of columns
  // rjobs[c].col0 .. rjobs[c].col0 + rjobs[c].n_ell - 1 of rcols, and row
  // c of R holds request c's tracers in its own order (column i = pool
  // tracer rjobs[c].sel[i]; pool tracers it does not select are not written)
  const RJob* rjobs;
  const RCol* rcols;
};


// flags of a z-local kernel: times H(a) always; LOC_INVD: / D(a)
// (inverse_growth_linear_bias); LOC_IA: * Omega_m / D(a) (NLA normalisation)
enum LocMode { LOC_INVD = 1, LOC_IA = 2 };

// a single source plane (delta_nz, probes.py:53-64): chi-table segment and
// offset of its scale factor, and (1 + m)
struct WLSource {
  int32_t on;
  int32_t L;
  float off;
  float fac;
};

struct WLArgs {
  int B, Na, nw;
  int ia;                 // add to the z-local (intrinsic-alignment) values already in R
  const WLSource* src;    // [nw]
  const uint8_t* Lidx;    // [257][Na] chi-table segment of z'_{m,j}
  const float* delta;     // [257][Na] a'_{m,j} - atab[L]
  const float* Nw;        // [5 or NWL_MAX][257][Na] (dx_m/3) w_j n_i(z'_{m,j}) (1 + m_i), zero rows past nw
  const float* zp1;       // [Na] 1 + z_m
  const int* col;         // [nw] tracer column
  const float* chitab;
  const float* coef;
  const float* crec;
  float* R;
  int Tpad;
  const int* dB;          // optional device count of cosmologies (grid sized for B)
  // optional (served batches): row c of R in request c's tracer order, as
  // TablesArgs::rjobs
  const RJob* rjobs;
};

struct LimberArgs {
  int B, Na, n_ell, ncols;  // ncols = B * n_ell
  const double* ell;        // [n_ell]
  const float* coef;
  const float* crec;
  const float* R;
  int Tpad;
  uint32_t wl_mask;         // bit i set: tracer i is weak lensing (ell factor)
  float* out;               // [B][P][n_ell]
  float* out_t;             // [B][P][n_ell] tangent (JVP)
  const float* cbar;        // [B][P][n_ell] cotangent (VJP)
  float* theta_col;         // VJP partials: [ncols][7] per column; launch_adjoint: [B][adj_groups(Na)][slices][7]
  int waves;                // waves per block splitting the a range
  const float4* ehtab;      // [B][NEHQ] transfer table, or null: evaluate EH98 per point
  const float* ehtab7;      // adjoint: [B][NEHQ + 1][8] d/dtheta of the table's function at its nodes
  int mx;                   // forward, n_ell >= 32: contract the pairs on the matrix cores
  // small batches: the a range is also split over `slices` blocks per column
  // group (grid y); each writes its partial outputs, already scaled, to
  // part[slice][...] in the layout of out (then out_t) or theta_col, and
  // launch_slice_sum adds the slices in order
  int slices;               // 1 = no split
  float* part;
};

// waves per block of the forward kernel in table mode (it ignores
// LimberArgs::waves, the tile of the other Limber kernels)
constexpr int FWD_WAVES = 4;

struct PkArgs {            // P(k, a) evaluation at (k_i, a_i) pairs
  int n;                   // points for one cosmology
  const double* k;         // [n]
  const float* coef;       // [Na == n][NCOEF] for that cosmology
  const float* crec;       // [NCREC]
  double* plin;            // [n]
  double* pnl;             // [n]
};

// ---------------------------------------------------------------- ragged batches
// One request of a served batch (all requests of a launch share n_z).
struct RJob {
  int32_t c;          // cosmology row in the launch's tables
  int32_t T;          // tracers of the request (1..10)
  int32_t n_ell;
  uint32_t wl_mask;   // bit i: tracer i of the request is weak lensing
  int64_t out_off;    // float offset of the request's [P][n_ell] output block
  int64_t cbar_off;   // float offset of its cotangent block (adjoint)
  int32_t col0;       // first column of the request in the column list
  int32_t sel[MAXT];  // pool tracer column of each of its tracers
  int32_t pad;
};
// One (request, ell) column; job < 0 pads a column tile.
struct RCol {
  int32_t job;
  int32_t l;
  double ell;
};

struct RaggedArgs {
  const int* ncols;      // device: number of columns (a multiple of 64)
  const RCol* cols;
  const RJob* jobs;
  int Na;
  const float* coef;
  const float* crec;
  const float* R;        // row c: request c's tracers in its own order
  int Tpad;
  float* out;
  const float* cbar;
  const int* njobs;      // adjoint: device count of requests
  float* theta_part;     // adjoint: per block partials, adj_ragged_blocks() rows of 7
  int min_slices;        // adjoint: adj_min_slices of the longest request there can be
  int waves;
  // per-cosmology transfer tables (row c of the launch's tables) and, for
  // the adjoint, their theta derivatives
  const float4* ehtab;   // [rows][NEHQ]
  const float* ehtab7;   // [rows][NEHQ + 1][NEHD_ROW]
  // forward: the a range of each 64-column tile is split over
  // ragged_slices(live tiles) blocks (at most max_slices); partials of
  // slice s go to part + s * part_stride in the layout of out when there is
  // more than one
  int max_slices;
  float* part;
  int64_t part_stride;
};

// The dispatcher deals blocks to the 8 XCDs in turn (block b to XCD b % 8), and each
// XCD has its own L2.  Neighbouring units of work read the same records, so units are
// renumbered to give each XCD one contiguous range of them: a record is then fetched
// into one L2 instead of two or three.  xcd_share: the range of block b's XCD;
// xcd_order: the unit of block b of n (a bijection of [0, n) for any n).
struct XcdShare {
  int first, count;
};
__device__ inline XcdShare xcd_share(int b, int n) {
  const int q = n >> 3, r = n & 7, x = b & 7;
  return {x * q + (x < r ? x : r), q + (x < r ? 1 : 0)};
}
__device__ inline int xcd_order(int b, int n) { return xcd_share(b, n).first + (b >> 3); }

// The adjoint's blocks (jc_adjoint.hip): a cosmology's a-nodes in groups of up
// to 64 (lanes), its multipoles dealt to ADJ_WAVES waves and, where that leaves
// the chip idle, to several blocks.
constexpr int ADJ_WAVES = 4;
// Multipoles whose sums a block takes in FP32 (128 a wave) before they go on in FP64.
// theta-bar's error against sums over 100 at a time stays below 1e-7 of the terms'
// magnitudes (in one go 1.1e-6 at 5000 multipoles, 7e-6 at 20000). 256: the same error,
// 347 us against 320 for 256 cosmologies of 300.
constexpr int ADJ_TERMS = 512;
__host__ __device__ inline int adj_groups(int Na) { return (Na + 63) / 64; }
// Served batches: enough slices of the multipoles for ADJ_FILL blocks (the
// device chooses by its live requests), and at least min_slices, which keep
// the longest request within ADJ_TERMS; a grid of adj_ragged_blocks.
constexpr int ADJ_FILL = 768;
__host__ __device__ inline int adj_min_slices(int n_ell) { return (n_ell + ADJ_TERMS - 1) / ADJ_TERMS; }
__host__ __device__ inline int adj_ragged_slices(int units, int min_slices) {
  int s = units < 1 ? 1 : ADJ_FILL / units;
  s = s < 1 ? 1 : (s > 16 ? 16 : s);
  return s > min_slices ? s : min_slices;
}
inline int adj_ragged_blocks(int max_jobs, int Na, int min_slices) {
  const int u = max_jobs * adj_groups(Na) * min_slices;
  return u > ADJ_FILL ? u : ADJ_FILL;
}

// Slices of a ragged launch with `tiles` live 64-column tiles: enough for
// about 2048 waves, each wave keeping at least 8 a-nodes.
__host__ __device__ inline int ragged_slices(int tiles, int waves, int Na, int max_slices) {
  if (tiles < 1) return 1;
  int s = (2048 + tiles * waves - 1) / (tiles * waves);
  const int smax = Na / (8 * waves);
  s = s < smax ? s : smax;
  s = s < max_slices ? s : max_slices;
  return s < 1 ? 1 : s;
}

// Blocks that hold every unit of `tiles` live tiles or fewer.  An XCD has at most
// t / 8 + 1 of t tiles and ragged_slices gives each at most 2048 / (t waves) + 1
// slices and at most max_slices, so its units are at most 256 / waves + t / 8 +
// max_slices + 1.
inline int ragged_fwd_blocks(int tiles, int waves, int max_slices) {
  return 8 * ((256 + waves - 1) / waves + (tiles + 7) / 8 + max_slices + 1);
}

// launchers (defined next to their kernels)
hipError_t launch_tables(int nd, const TablesArgs& a, hipStream_t s, int num_cu, int variant = 0);
// ctile: cosmologies per block of the forward kernel (1, 2, 4, 8, 16; 0 = by rule)
hipError_t launch_wl(int nd, int ctile, const WLArgs& a, int num_cu, hipStream_t s);
// Gaussian likelihood on block-diagonal covariances (jc_likelihood.hip)
// (strides of element (p, q, l) of a precision array: (p P + q) pair + l ell)
struct PrecLayout {
  int64_t pair, ell;
};
// the reference's sparse format [P][P][n_ell], and one block after the other
inline PrecLayout prec_sparse(int64_t n_ell) { return {n_ell, 1}; }
inline PrecLayout prec_blocks(int64_t P) { return {1, P * P}; }
// ld[n_ell][2]: |det| of block l = ld[l][0] 2^ld[l][1]
hipError_t launch_block_inv(const double* cov, int P, int n_ell, double* inv, PrecLayout lay, double* ld,
                            hipStream_t s);
hipError_t launch_loglike(const float* mu, int B, int P, int n_ell, const double* data, const double* prec,
                          PrecLayout lay, double c0, float* s_out, double* part, double* loglike, hipStream_t s);
// Gaussian KDE n(z) (redshift.py:126-156) at n points from a catalog sorted
// by redshift: out[p] = sum_k w_k N(z_p - z_k; bw) / sum_k w_k
// growth rate and transverse distance of a background call (FP64 slots 6, 7)
hipError_t launch_background_ex(const double* params, const double* a, int n, const double* atab_g,
                                int growth_model, double gamma, double* dbg, hipStream_t s);
// out[o] = sum over s of part[s * n + o], s = 0..slices-1 in order
hipError_t launch_slice_sum(const float* part, int slices, int64_t n, float* out, hipStream_t s);
// dst = src, whole 8-byte words (src may be pinned host memory)
hipError_t launch_stage(const void* src, void* dst, size_t bytes, hipStream_t s);
// jac[b][o][d] = sum over s of part[s][b * 7 + d][o], for B cosmologies and n outputs
hipError_t launch_jac_sum(const float* part, int slices, int64_t B, int64_t n, float* jac, hipStream_t s);
hipError_t launch_kde(const double* z, int64_t n, const double* cz, const double* cw, int64_t ncat, double bw,
                      double wsum, double* out, hipStream_t s);
hipError_t launch_limber(int nd, int T, const LimberArgs& a, hipStream_t s);
// the adjoint in transfer-table mode; its partials theta_col are then summed by
// launch_theta_reduce(theta_col, 1, B, adj_groups(Na) * slices, ...)
hipError_t launch_adjoint(int T, const LimberArgs& a, hipStream_t s);
// theta[B][7] = sum over slices and ell of the per-column partials
// [nsl][B][n_ell][7] (nsl = 1: the partials of an unsliced launch)
hipError_t launch_theta_reduce(const float* theta_col, int nsl, int B, int n_ell, double* theta, hipStream_t s);
hipError_t launch_pk_eval(const PkArgs& a, hipStream_t s);
// for up to max_cols columns
hipError_t launch_limber_ragged(int max_cols, const RaggedArgs& a, hipStream_t s);
hipError_t launch_ragged_adjoint(int max_jobs, const RaggedArgs& a, hipStream_t s);
hipError_t launch_ragged_reduce(int max_jobs, const RaggedArgs& a, double* theta, hipStream_t s);
// dense covariances (jc_dense.hip): in-place lower Cholesky factor of the
// row-major N x N matrix A (log L_ii into dlog[N], *bad set on a
// non-positive pivot; the strict upper triangle is zeroed; inv: DENSE_PANEL^2
// doubles of workspace); the inverses of L's DENSE_SOLVE_BLOCK-row diagonal
// blocks, tri_inverse_size(N) doubles, which the solves take; X = L^-1 R
// (transpose 0) or L^-T R (transpose 1) for B right-hand sides as rows of R,
// which is overwritten; the log-likelihood -1/2 |L^-1 (data - mu_b)|^2 + c0 of
// B means, with Z and X as [B][N] workspaces and dmu (may be null) =
// C^-1 (data - mu_b) as float
constexpr int DENSE_PANEL = 64;
constexpr int DENSE_SOLVE_BLOCK = 512;
inline size_t tri_inverse_size(int64_t N) {
  return (size_t)((N + DENSE_SOLVE_BLOCK - 1) / DENSE_SOLVE_BLOCK) * DENSE_SOLVE_BLOCK * DENSE_SOLVE_BLOCK;
}
// packed lower triangle: row r starts at tri_row(r) doubles and is padded to whole
// 64-byte lines; rows [r0, r1) at src (pinned host memory) into the rows of A
__host__ __device__ inline int64_t tri_row(int64_t r) {
  const int64_t g = r >> 3;
  return 32 * g * (g + 1) + (r & 7) * 8 * (g + 1);
}
hipError_t launch_unpack_lower(const double* src, double* A, int64_t N, int64_t r0, int64_t r1, hipStream_t s);
hipError_t launch_dense_cholesky(double* A, int64_t N, double* inv, double* dlog, int* bad, hipStream_t s);
hipError_t launch_tri_inverse(const double* L, int64_t N, double* inv, hipStream_t s);
hipError_t launch_dense_solve(const double* L, int64_t N, const double* inv, double* R, double* X, int64_t B,
                              int transpose, hipStream_t s);
// N <= DENSE_PANEL: X = L^-1 R (mode 0), L^-T R (1) or L^-T L^-1 R (2)
hipError_t launch_small_solve(const double* L, int N, const double* R, double* X, int64_t B, int mode, hipStream_t s);
// the same for any N, in X and without a workspace, by 64-row blocks of two launches
// each (N = 5500, 256 right-hand sides: 1880 us against 410 with the inverses)
hipError_t launch_dense_solve_in_place(const double* L, int64_t N, double* X, int64_t B, int mode, hipStream_t s);
hipError_t launch_dense_loglike(const float* mu, int64_t B, int64_t N, const double* data, const double* L, double c0,
                                const double* inv, double* Z, double* X, double* loglike, float* dmu, hipStream_t s);
// out[o] = sum of the forward partials of the launch's live slices, for o in
// [range[0], range[1]) (device values), grid sized for max_out floats
hipError_t launch_ragged_slice_sum(const int* ncols, int waves, int Na, int max_slices, const float* part,
                                   int64_t part_stride, const int* range, int64_t max_out, float* out,
                                   hipStream_t s);

}  // namespace jc
