// Per-cosmology tables (FP64), and the KDE n(z).
//
// k_tables: one workgroup per cosmology builds, in FP64,
//   * the chi(a) table: RK4 in ln a of a y-independent right-hand side, i.e.
//     a cumulative Simpson with midpoint nodes (background.py:223-233,
//     scipy/ode.py:6-22), as a parallel prefix sum;
//   * the growth table: RK4 over a of [D, dD/da] (background.py:443-487),
//     the ODE is linear, so each RK4 step is a 2x2 propagator built in
//     parallel and the 127 steps are composed by a parallel prefix product;
//     or, for a Cosmology with gamma, RK4 in ln a of the y-independent
//     dlnD/dlna = Omega_m(a)^gamma (background.py:515-549) as a prefix sum;
//   * sigma_8 normalisation by the 129-sample Romberg table over ln k in
//     [-4, 3] (power.py:56-78, integrate.py:67-159), as the weighted sum of
//     the samples that its extrapolation amounts to;
//   * the halofit sigma^2(R) table on 256 R nodes from a 257-node ln k Simpson
//     (power.py:96-111).  sigma^2(R, a) = D(a)^2 sigma^2(R, 1) exactly, so one
//     table per cosmology replaces the reference's [Na, 257, 256] tensor, and
//     the exp(-(k R)^2) factors are a cosmology-independent resident table;
//   * per a-node: chi, D, the nonlinear scale by the reference's
//     nearest-node interpolation of the decreasing sigma^2 table
//     (power.py:112-115), n_eff and C (power.py:118-139), the Takahashi
//     coefficients (power.py:199-238), the Simpson weight of the Limber
//     integral (angular_cl.py:91-96) and the number-count kernels
//     (probes.py:77-99);
//   * for calls in table mode, beside the a-nodes, the cosmology's transfer
//     table T(k) k^(n_s/2) over the call's ln k range.
// Measured (n_z 512, 100 ell): 1 cosmology 50 -> 31 us, 1024 112 -> 92 us, the
// 7-direction dual form for 256 cosmologies 195 -> 119 us.
#include <type_traits>

#include "jc_records.hpp"

namespace jc {

template <int ND>
struct Seed {
  static JC_D typename Types<ND>::D load(const double* params, const double* seeds, int c, int i) {
    typename Types<ND>::D r;
    r.v = params[c * 8 + i];
#pragma unroll
    for (int d = 0; d < ND; ++d) r.d[d] = seeds[(c * 8 + i) * ND + d];
    return r;
  }
};
// The adjoint's seven directions are the seven parameters themselves (Omega_k,
// parameter 5, has none): constants, which fold into the first operations.
JC_D int param_dir(int i) { return i < 5 ? i : (i == 5 ? -1 : i - 1); }
template <>
struct Seed<7> {
  static JC_D Types<7>::D load(const double* params, const double*, int c, int i) {
    Types<7>::D r;
    r.v = params[c * 8 + i];
#pragma unroll
    for (int d = 0; d < 7; ++d) r.d[d] = d == param_dir(i) ? 1.0 : 0.0;
    return r;
  }
};
template <>
struct Seed<0> {
  static JC_D double load(const double* params, const double*, int c, int i) { return params[c * 8 + i]; }
};

template <class S>
JC_D S zero() { return Make<S>::c(0.0); }

// FP64 (possibly dual) scalar in memory: component i at p[i]
template <class S>
struct DMem {
  static JC_D S ld(const double* p) { return p[0]; }
  static JC_D void st(double* p, const S& x) { p[0] = x; }
};
template <int N>
struct DMem<Dual<double, N>> {
  static JC_D Dual<double, N> ld(const double* p) {
    Dual<double, N> r;
    r.v = p[0];
#pragma unroll
    for (int i = 0; i < N; ++i) r.d[i] = p[1 + i];
    return r;
  }
  static JC_D void st(double* p, const Dual<double, N>& x) {
    p[0] = x.v;
#pragma unroll
    for (int i = 0; i < N; ++i) p[1 + i] = x.d[i];
  }
};

// Table segment of interpolate.py:12-37 on nodes xp[0..n-1] (log-uniform,
// logspace(-3, 0, n)): nearest node (first on ties) clipped to [1, n-2], side
// from clip(x, xp[1], xp[n-2]); the line through both nodes at x is
// f[i] + (f[j] - f[i]) t.
JC_D void logtab_segment(double x, double log10x, const double* xp, int n, int& i, int& j, double& t) {
  double u = (log10x + 3.0) * (double)(n - 1) / 3.0;
  int i0 = (int)::floor(u);
  i0 = i0 < 0 ? 0 : (i0 > n - 1 ? n - 1 : i0);
  int ind = i0;
  // neighbours (covers any rounding in the log index); scan upward so the
  // first index wins ties
  // (clamped candidates repeat an end node, which never wins over its first
  // occurrence; the four reads are independent)
  double best = 1e300;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int q = i0 - 1 + k;
    q = q < 0 ? 0 : (q > n - 1 ? n - 1 : q);
    const double dd = (x - xp[q]) * (x - xp[q]);
    if (dd < best) { best = dd; ind = q; }
  }
  ind = ind < 1 ? 1 : (ind > n - 2 ? n - 2 : ind);
  double xc = x > xp[1] ? x : xp[1];
  xc = xc < xp[n - 2] ? xc : xp[n - 2];
  i = ind;
  j = (xc - xp[ind] < 0.0) ? ind - 1 : ind + 1;
  t = (x - xp[i]) / (xp[j] - xp[i]);
}
template <class S>
JC_D S interp_logtab(double x, double log10x, const double* xp, const S* fp, int n) {
  int i, j;
  double t;
  logtab_segment(x, log10x, xp, n, i, j, t);
  return fp[i] + (fp[j] - fp[i]) * t;
}

// Growth ODE right-hand side coefficients at x (background.py:465-475):
// y' = [[0, 1], [r, -q]] y, given ln x and 1/x.
template <class Sd>
JC_D void growth_qr(const CosmoP<Sd>& cp, double x, double lnx, double ix, Sd& q, Sd& r) {
  const Sd efde = jm::exp(f_de_ln(cp, x, lnx));
  const Sd E2 = Esqr_parts(cp, ix, efde);
  const Sd iE2 = 1.0 / E2;
  Sd omm = cp.Omega_m * (ix * ix * ix) * iE2;
  Sd omde = cp.Omega_de * efde * iE2;
  q = (2.0 - 0.5 * (omm + (1.0 + 3.0 * w_de(cp, x)) * omde)) * ix;
  r = 1.5 * omm * ix * ix;
}

// 2x2 matrix helpers for the growth propagators (row-major m[0..3])
template <class Sd>
JC_D void mat_mul(const Sd* a, const Sd* b, Sd* c) {  // c = a b
  c[0] = a[0] * b[0] + a[1] * b[2];
  c[1] = a[0] * b[1] + a[1] * b[3];
  c[2] = a[2] * b[0] + a[3] * b[2];
  c[3] = a[2] * b[1] + a[3] * b[3];
}

// Read-only data seen through the constant address space: wave-uniform loads
// from it become scalar loads whatever the kernel stores elsewhere (a global
// store of the same type would otherwise stop the compiler from proving the
// data unchanged, and uniform reads would go through the vector memory path).
typedef const __attribute__((address_space(4))) double ConstD;

// Cubic Hermite interpolant on [x_q, x_q + h] at fraction t, from the end
// values f0, f1 and the end derivatives d0, d1 (per unit x).
template <class Sd, class Tt>
JC_D Sd hermite(const Tt& t, double h, const Sd& f0, const Sd& f1, const Sd& d0, const Sd& d1) {
  const Sd e0 = h * d0, e1 = h * d1;
  const Sd c2 = 3.0 * (f1 - f0) - 2.0 * e0 - e1;
  const Sd c3 = 2.0 * (f0 - f1) + e0 + e1;
  return ((c3 * t + c2) * t + e0) * t + f0;
}

template <int W>
JC_D void eh_dtab_node(int c, int q, double lo, double h, const float* crec, float* ehtab7);

// Values of a lane of the wave for scans (plain or dual).
JC_D double shfl_up_s(double x, int d) { return __shfl_up(x, d, 64); }
template <typename T, int N>
JC_D Dual<T, N> shfl_up_s(const Dual<T, N>& x, int d) {
  Dual<T, N> r;
  r.v = __shfl_up(x.v, d, 64);
#pragma unroll
  for (int k = 0; k < N; ++k) r.d[k] = __shfl_up(x.d[k], d, 64);
  return r;
}

JC_D double shfl_xor_s(double x, int m) { return __shfl_xor(x, m, 64); }
template <typename T, int N>
JC_D Dual<T, N> shfl_xor_s(const Dual<T, N>& x, int m) {
  Dual<T, N> r;
  r.v = __shfl_xor(x.v, m, 64);
#pragma unroll
  for (int k = 0; k < N; ++k) r.d[k] = __shfl_xor(x.d[k], m, 64);
  return r;
}
template <class S>
JC_D S wave_sum(S v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = v + shfl_xor_s(v, m);
  return v;
}

// The EH98 constants of the 15 LDS slots, converted by f.
template <class S, class F>
JC_D EHc<S> eh_from(const F& f, int nw) {
  EHc<S> e;
  e.fb = f(0);
  e.fc = f(1);
  e.inv13keq = f(2);
  e.ln_inv13keq = f(3);
  e.beta_c18 = f(4);
  e.c14a = f(5);
  e.sh_d = f(6);
  e.alpha_b = f(7);
  e.beta_b = f(8);
  e.beta_node = f(9);
  e.ln_ksilk = f(10);
  e.bnode_shd = f(11);
  e.bb_shd = f(12);
  e.alpha_g = f(13);
  e.tq = f(14);
  e.nw = nw;
  return e;
}

// First halofit k node past y = k R = 7.75 for the R nodes from 64 r on.
constexpr int HF_ROWS[4] = {NHF_K, 245, 205, 164};

typedef double f64x4 __attribute__((ext_vector_type(4)));

// LDS of the table kernel, in scalars Sd unless said otherwise.  X holds the
// integrands of the background tables first; forward tables use it again for
// the moment products and the transfer table's nodes, the dual kernels keep
// those (X is then the moment tables' space, the nodes the samples').
template <int ND>
struct TabLds {
  static constexpr int CHI = 0;
  static constexpr int G = CHI + NCHI;
  static constexpr int SIG = G + NGROW;              // sigma^2, S_1, S_2, S_3: [4][256]
  static constexpr int SMP = SIG + 4 * NHF_R;        // samples: sigma_8, then halofit
  static constexpr int EH = SMP + NROMB + NHF_K;     // EH98 constants
  static constexpr int TOT = EH + 16;                // scan totals of the waves
  static constexpr int X = ND == 0 ? (TOT + 32 + 3) / 4 * 4 : SIG;  // 32-byte aligned
  static constexpr int KP = ND == 0 ? 0 : (TOT + 32) * (ND + 1);  // dual kernels: k^0 .. k^6 rows, in doubles
  static constexpr int END = ND == 0 ? X + 2048 : TOT + 32 + (4 * NHF_K + ND) / (ND + 1);
  static constexpr size_t bytes() {
    // then floats: halofit P_1 (Sf) and its k, and the task counter
    return sizeof(double) * (ND + 1) * END + sizeof(float) * ((ND + 1) * NHF_K + NHF_K + 3) + 32;
  }
};

// One workgroup per cosmology.  The phases are bound by the issue and latency
// of FP64 chains, so they are few (a barrier each), every thread has work in
// each, and what depends on the a-grid alone (segments and fractions of the
// table interpolations, Romberg weights, powers of k and R) comes from resident
// tables.  The per-a nodes and the nodes of the transfer table are one list of
// 64-node tasks that the waves draw from, so the a-grid's odd node (n_z + 1)
// costs one wave a pass, not all of them.
// WO: floats of a stored scalar.  With ND = 1 and WO = 8 the seven directions
// of a cosmology are seven workgroups, which write one derivative each into the
// records of the adjoint (direction 0 the values too): a few cosmologies leave
// the chip idle, and a workgroup of one direction takes half the time of one of
// seven.
template <int ND, int NT, int MINW, int WO = ND + 1>
__global__ __launch_bounds__(NT, MINW) void k_tables(TablesArgs A) {
  using Sd = typename Types<ND>::D;
  using Sf = typename Types<ND>::F;
  using L = TabLds<ND>;
  constexpr int W = ND + 1, NW = NT / 64;
  constexpr bool SPLIT = WO != W;
  extern __shared__ __align__(16) unsigned char smem[];
  Sd* const lds = reinterpret_cast<Sd*>(smem);
  Sd* const s_chi = lds + L::CHI;
  Sd* const s_g = lds + L::G;
  Sd* const s_sig = lds + L::SIG;
  Sd* const s_S = s_sig + NHF_R;
  Sd* const s_smp = lds + L::SMP;
  Sd* const s_eh = lds + L::EH;
  Sd* const s_tot = lds + L::TOT;
  Sd* const s_x = lds + L::X;
  Sf* const s_p1f = reinterpret_cast<Sf*>(lds + L::END);
  float* const s_k32 = reinterpret_cast<float*>(s_p1f + NHF_K);
  int* const s_next = reinterpret_cast<int*>(s_k32 + NHF_K);

  const int dir = SPLIT ? blockIdx.x % (WO - 1) : 0;
  const int c = SPLIT ? blockIdx.x / (WO - 1) : blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a scalar of the records: its value, and the derivatives
  auto put = [&](float* o, const Sd& v) {
    if constexpr (SPLIT) {
      if (dir == 0) o[0] = (float)v.v;
      o[1 + dir] = (float)v.d[0];
    } else {
      Mem<Sf>::st(o, conv<Sf>(v));
    }
  };
  if (c >= A.B) return;
  if (A.dB && c >= *A.dB) return;  // served batches: grid sized for capacity

  Sd p[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (SPLIT) {
      p[i].v = A.params[c * 8 + i];
      p[i].d[0] = dir == param_dir(i) ? 1.0 : 0.0;
    } else {
      p[i] = Seed<ND>::load(A.params, A.seeds, c, i);
    }
  }
  const CosmoP<Sd> cp = make_cosmo(p);
  for (int i = tid; i < NHF_K; i += NT) s_k32[i] = A.hf_k32[i];
  if (tid == 0) *s_next = 0;
  if constexpr (ND > 0) {
    double* kp = reinterpret_cast<double*>(smem) + L::KP;
    for (int e = tid; e < 4 * NHF_K; e += NT) kp[e] = (e & 3) ? A.hf_kp[e - 1] : 1.0;
  }

  // ------------------------------------------- EH98 constants, background integrands
  // The k-independent EH98 quantities (transfer.py:47-85, 88-97, 109-117,
  // 134-142) once per cosmology, in FP64, by wave 0 beside the other waves'
  // background integrands; the samples read them from LDS and the Limber
  // kernels from the cosmology record.  Forward tables: the independent powers
  // and logarithms on separate lanes (eh_setup_wave).  Dual tables: direction d
  // on lane d, as a chain of one-direction duals.
  if (wave == 0) {
    if constexpr (ND == 0) {
      const EHc<double> eh = eh_setup_wave(cp, lane);
      if (lane == 0) {
        const double vals[15] = {eh.fb, eh.fc, eh.inv13keq, eh.ln_inv13keq, eh.beta_c18, eh.c14a, eh.sh_d,
                                 eh.alpha_b, eh.beta_b, eh.beta_node, eh.ln_ksilk, eh.bnode_shd, eh.bb_shd,
                                 eh.alpha_g, eh.tq};
#pragma unroll
        for (int i = 0; i < 15; ++i) s_eh[i] = vals[i];
      }
    } else if (lane < ND) {
      using D1 = Dual<double, 1>;
      D1 q[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        q[i].v = p[i].v;
        q[i].d[0] = ND == 7 ? (lane == param_dir(i) ? 1.0 : 0.0) : p[i].d[0];
      }
      const EHc<D1> eh = eh_setup(make_cosmo(q));
      const D1 vals[15] = {eh.fb, eh.fc, eh.inv13keq, eh.ln_inv13keq, eh.beta_c18, eh.c14a, eh.sh_d,
                           eh.alpha_b, eh.beta_b, eh.beta_node, eh.ln_ksilk, eh.bnode_shd, eh.bb_shd,
                           eh.alpha_g, eh.tq};
      double* o = reinterpret_cast<double*>(s_eh);
#pragma unroll
      for (int i = 0; i < 15; ++i) {
        if (lane == 0) o[i * W] = vals[i].v;
        o[i * W + 1 + lane] = vals[i].d[0];
      }
    }
  }
  // dchi/dln a at the 256 nodes and RK4 midpoints of the chi table, and the
  // growth ODE's coefficients (or dlnD/dlna of the gamma growth) at the 128
  // nodes and midpoints of the growth table, by the waves past the first
  Sd* const x_chi = s_x;             // [2][256]
  Sd* const x_g = s_x + 2 * NCHI;    // [2][128][2]
  if (wave > 0) {
    for (int t = tid - 64; t < 2 * NCHI + 2 * NGROW; t += NT - 64) {
      if (t < 2 * NCHI) {
        const int i = t & (NCHI - 1), mid = t / NCHI;
        if (mid && i == 0) continue;
        const double* nd = A.chi_nodes + (size_t)i * 8 + 3 * mid;  // a, ln a, 1/a
        const Sd E2 = Esqr_parts(cp, nd[2], jm::exp(f_de_ln(cp, nd[0], nd[1])));
        x_chi[t] = RH * nd[2] / jm::sqrt(E2);  // dchioverda(e^t) e^t
      } else {
        const int u = t - 2 * NCHI, i = u & (NGROW - 1), mid = u / NGROW;
        if (mid && i == 0) continue;
        const double* nd = (A.growth_model == 0 ? A.g_nodes : A.gg_nodes) + (size_t)i * 8 + 3 * mid;
        if (A.growth_model == 0) {
          growth_qr(cp, nd[0], nd[1], nd[2], x_g[2 * u], x_g[2 * u + 1]);
        } else {
          const Sd efde = jm::exp(f_de_ln(cp, nd[0], nd[1]));
          const Sd omm = cp.Omega_m * (nd[2] * nd[2] * nd[2]) / Esqr_parts(cp, nd[2], efde);
          x_g[2 * u] = jm::exp(A.gamma * jm::log(omm));
        }
      }
    }
  }
  __syncthreads();

  // ------------------------------------------- chi and growth tables
  // chi: RK4 in ln a of a y-independent right-hand side, a cumulative Simpson
  // with midpoints; growth ODE: RK4 over a of the linear y' = A(a) y
  // (background.py:443-487).  Each step is y_i = G_i y_{i-1} with G_i = I +
  // h/6 (K1 + 2 K2 + 2 K3 + K4), K1 = A(a_{i-1}), K2 = A(mid)(I + h/2 K1),
  // K3 = A(mid)(I + h/2 K2), K4 = A(a_i)(I + h K3): the same products the
  // reference's RK4 forms, regrouped.  Gamma growth (background.py:515-549):
  // RK4 in t = ln a of the y-independent f(t) from y_0 = ln a_0 with a first
  // step of h = 0.  Prefix sums and products within the waves, then across.
  Sd dchi = zero<Sd>();
  if (tid < NCHI) {
    if (tid > 0)
      dchi = (1.0 / 6.0) * A.chi_nodes[(size_t)tid * 8 + 6] * (x_chi[tid - 1] + 4.0 * x_chi[NCHI + tid] + x_chi[tid]);
    for (int o = 1; o < 64; o <<= 1) {
      const Sd v = shfl_up_s(dchi, o);
      if (lane >= o) dchi = dchi + v;
    }
    if (lane == 63) s_tot[wave] = dchi;
  }
  Sd G[4];
  if (tid < NGROW) {
    const int i = tid;
    if (A.growth_model == 0) {
      if (i == 0) {  // ode.py:6-22: the first step has h = 0
        G[0] = Make<Sd>::c(1.0); G[1] = zero<Sd>(); G[2] = zero<Sd>(); G[3] = Make<Sd>::c(1.0);
      } else {
        const double h = A.atab_g[i] - A.atab_g[i - 1];
        const Sd q0 = x_g[2 * (i - 1)], r0 = x_g[2 * (i - 1) + 1];
        const Sd qm = x_g[2 * (NGROW + i)], rm = x_g[2 * (NGROW + i) + 1];
        const Sd q1 = x_g[2 * i], r1 = x_g[2 * i + 1];
        // the second row of A M for M = I + s K: (r M0 - q M2, r M1 - q M3);
        // its first row is M's second
        const Sd K1[4] = {zero<Sd>(), Make<Sd>::c(1.0), r0, -q0};
        Sd K2[4], K3[4], K4[4];
        auto step = [&](const Sd& r, const Sd& q, const Sd* K, double s, Sd* out) {
          const Sd m2 = s * K[2], m3 = 1.0 + s * K[3];
          out[0] = m2;
          out[1] = m3;
          out[2] = r * (1.0 + s * K[0]) - q * m2;
          out[3] = r * (s * K[1]) - q * m3;
        };
        step(rm, qm, K1, 0.5 * h, K2);
        step(rm, qm, K2, 0.5 * h, K3);
        step(r1, q1, K3, h, K4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          G[e] = ((e == 0 || e == 3) ? 1.0 : 0.0) + 1.0 / 6.0 * h * (K1[e] + 2.0 * K2[e] + 2.0 * K3[e] + K4[e]);
      }
      for (int o = 1; o < 64; o <<= 1) {  // prefix products, later x earlier
        Sd V[4], P[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) V[e] = shfl_up_s(G[e], o);
        mat_mul(G, V, P);
        if (lane >= o) {
#pragma unroll
          for (int e = 0; e < 4; ++e) G[e] = P[e];
        }
      }
    } else {
      G[0] = i == 0 ? Make<Sd>::c(A.gg_nodes[1])
                    : (1.0 / 6.0) * A.gg_nodes[(size_t)i * 8 + 6] *
                          (x_g[2 * (i - 1)] + 4.0 * x_g[2 * (NGROW + i)] + x_g[2 * i]);
      for (int o = 1; o < 64; o <<= 1) {
        const Sd v = shfl_up_s(G[0], o);
        if (lane >= o) G[0] = G[0] + v;
      }
      G[1] = G[2] = G[3] = zero<Sd>();
    }
    if (tid == 63) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s_tot[16 + e] = G[e];
    }
  }
  __syncthreads();
  if (tid < NCHI) {
    Sd before = zero<Sd>(), all = zero<Sd>();
#pragma unroll
    for (int w = 0; w < NCHI / 64; ++w) {
      if (w < wave) before = before + s_tot[w];
      all = all + s_tot[w];
    }
    s_chi[tid] = all - (before + dchi);
  }
  if (tid < NGROW) {
    if (wave == 1) {
      Sd V[4], P[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) V[e] = s_tot[16 + e];
      if (A.growth_model == 0) {
        mat_mul(G, V, P);
#pragma unroll
        for (int e = 0; e < 4; ++e) G[e] = P[e];
      } else {
        G[0] = G[0] + V[0];
      }
    }
    // raw D = (P_i y_0)[0], y_0 = [a_0, 1]; normalised below by the last node's
    const Sd y = A.growth_model == 0 ? G[0] * A.atab_g[0] + G[1] : jm::exp(G[0]);
    s_g[tid] = y;
    if (A.dbg && A.growth_model == 0) G[0] = G[2] * A.atab_g[0] + G[3];  // dD/da
  }

  // ------------------------------------------- EH98 samples
  {
  const EHc<Sd> eh = eh_from<Sd>([&](int i) { return s_eh[i]; }, A.transfer_model);
  if (tid == 0) {
    const Sd vals[18] = {eh.fb, eh.fc, eh.inv13keq, eh.beta_c18, eh.c14a, eh.sh_d, eh.alpha_b, eh.beta_b,
                         eh.beta_node, eh.ln_ksilk, cp.n_s,
                         3.0 * H0 * H0 * cp.Omega_m / 2.0 / C_KMS,  // probes.py:71
                         eh.ln_inv13keq, eh.bnode_shd, eh.bb_shd, eh.alpha_g, eh.tq,
                         Make<Sd>::c(A.transfer_model ? 1.0 : 0.0)};
    constexpr int slot[18] = {CR_FB, CR_FC, CR_INV13KEQ, CR_BETAC18, CR_C14A, CR_SHD, CR_ALPHAB, CR_BETAB,
                              CR_BETANODE, CR_LNKSILK, CR_NS, CR_WLCONST, CR_LNINV13, CR_BNODE_SHD, CR_BB_SHD,
                              CR_ALPHAG, CR_TQ, CR_NW};
    float* cr = A.crec + (size_t)c * NCREC * WO;
#pragma unroll
    for (int i = 0; i < 18; ++i) put(cr + slot[i] * WO, vals[i]);
  }
  // T^2 k^n_s times the resident weights: of the sigma_8 Romberg table
  // (power.py:56-78, integrate.py:67-159: its extrapolation is a fixed linear
  // combination of the samples) and of the halofit ln k Simpson rule with
  // k^3/(2 pi^2) (power.py:96-111), both without the normalisation
  for (int t = tid; t < NROMB + NHF_K; t += NT) {
    const bool rb = t < NROMB;
    const double* nd = rb ? A.romb + 4 * t : A.hf_nodes + 4 * (t - NROMB);  // k, 1/k, ln k, weight
    const Sd T = eh_transfer(eh, nd[0], nd[1], nd[2]);
    const Sd v = nd[3] * (T * T * jm::exp(cp.n_s * nd[2]));
    s_smp[t] = v;
    if (!rb) s_p1f[t - NROMB] = conv<Sf>(v);
  }
  }
  __syncthreads();
  // sigma8^2 / sigma^2(R = 8) (power.py:37-41), by every wave; the growth
  // factor at a = 1 in power.py:48 is the table's last node over itself, 1
  Sd pknorm;
  {
    Sd v = s_smp[lane] + s_smp[64 + lane];
    if (lane == 0) v = v + s_smp[128];
    pknorm = cp.sigma8 * cp.sigma8 / wave_sum(v);
  }
  // growth table, background.py:482
  if (tid < NGROW) {
    const Sd y = s_g[tid], last = s_g[NGROW - 1];
    const Sd g = y / last;
    // background calls: the growth-rate table (background.py:483-484)
    if (A.dbg && A.growth_model == 0) A.dbg[(size_t)c * A.dbg_stride + 768 + tid] = val(G[0] / last * A.atab_g[tid] / g);
    G[0] = g;
  }
  // chi table for the weak-lensing kernel
  if (tid < NCHI) {
    const Sd chi_i = s_chi[tid];
    Sd slope = zero<Sd>();
    if (tid < NCHI - 1) slope = (s_chi[tid + 1] - chi_i) / (A.atab_chi[tid + 1] - A.atab_chi[tid]);
    float* ct = A.chitab + ((size_t)c * NCHI + tid) * 2 * WO;
    put(ct, chi_i);
    put(ct + WO, slope);
  }
  if (tid == 0) put(A.crec + ((size_t)c * NCREC + CR_PKNORM) * WO, pknorm);

  // ------------------------------------------- Gaussian moments
  // of the a = 1 power (without D^2) on the 256 R nodes:
  //   S_p(R_j) = sum_i w_i P1_i y^{2p} exp(-y^2),  y = k_i R_j,  p = 0..3,
  // summed as R_j^{2p} sum_i (w_i P1_i k_i^{2p}) E_ij.
  // S_0 is the halofit sigma^2(R) table (power.py:96-111); S_1 and S_2 are
  // the n_eff and C sums of power.py:118-139 and, with dS_p/dln R =
  // 2p S_p - 2 S_{p+1}, give a cubic Hermite interpolant in ln R that is
  // evaluated at each a-node's R_nl (absolute error ~1e-8 in n_eff and C).
  // Rows past y = 7.75 for every R of a group add nothing in FP64 (e^-60).
  const Sd* raw = s_smp + NROMB;
  if constexpr (ND == 0) {
    // V_ip = w_i P1_i k_i^{2p} in LDS; wave w takes the k nodes w, w + NW, ...,
    // lane l the four R nodes l, l + 64, l + 128, l + 192, so each broadcast
    // read of a V row feeds 16 FMAs and each E row is read once, coalesced (the
    // L1's rate on E's 526 KB is what bounds it); the waves' partial sums are
    // added in a fixed order through LDS.
    ConstD* kp = (ConstD*)A.hf_kp;
    double4* V4 = reinterpret_cast<double4*>(s_x);  // [257] and a zero row; then the partial sums
    if (tid == 0) V4[NHF_K] = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int i = tid; i < NHF_K; i += NT) {
      const double v = raw[i];
      V4[i] = make_double4(v, v * kp[4 * i], v * kp[4 * i + 1], v * kp[4 * i + 2]);
    }
    __syncthreads();
    if (tid < NGROW) s_g[tid] = G[0];  // every thread has read the raw table
    double acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[r][q] = 0.0;
    const double* E = A.hf_E + lane;
    auto rows = [&](int i0, int i1, auto nr) {  // k nodes i0, i0 + NW, ... < i1 for the first nr groups of R
      constexpr int NR = decltype(nr)::value;
      auto term = [&](const double4& v, const double* e) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          acc[r][0] = fma(v.x, e[r], acc[r][0]);
          acc[r][1] = fma(v.y, e[r], acc[r][1]);
          acc[r][2] = fma(v.z, e[r], acc[r][2]);
          acc[r][3] = fma(v.w, e[r], acc[r][3]);
        }
      };
      constexpr int U = 4;  // rows in flight: the loop waits on the L2 otherwise
      int i = i0;
      for (; i + (U - 1) * NW < i1; i += U * NW) {
        double e[U][NR];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int r = 0; r < NR; ++r) e[u][r] = E[(size_t)(i + u * NW) * NHF_R + 64 * r];
#pragma unroll
        for (int u = 0; u < U; ++u) term(V4[i + u * NW], e[u]);
      }
      if (i < i1) {  // the rest, past i1 the last row again against V's zero row
        double e[U - 1][NR];
        const int last = i + (i1 - 1 - i) / NW * NW;
#pragma unroll
        for (int u = 0; u < U - 1; ++u)
#pragma unroll
          for (int r = 0; r < NR; ++r) e[u][r] = E[(size_t)min(i + u * NW, last) * NHF_R + 64 * r];
#pragma unroll
        for (int u = 0; u < U - 1; ++u) term(V4[i + u * NW <= last ? i + u * NW : NHF_K], e[u]);
        i = last + NW;
      }
      return i;
    };
    int i = rows(wave, HF_ROWS[3], std::integral_constant<int, 4>());
    i = rows(i, HF_ROWS[2], std::integral_constant<int, 3>());
    i = rows(i, HF_ROWS[1], std::integral_constant<int, 2>());
    rows(i, NHF_K, std::integral_constant<int, 1>());
    double* red = s_x;  // [2][16][64] per pair of waves
    for (int hw = NW / 2; hw >= 1; hw >>= 1) {
      __syncthreads();  // V, or the previous round's sums, have been read
#pragma unroll
      for (int half = 0; half < (NW > 4 ? 2 : 1); ++half) {
        // (with 8 waves the first round goes in two halves: the space is 2 waves')
        const int w0 = hw > 2 ? 2 * half : 0;
        const int n = hw > 2 ? 2 : hw;
        if (half && hw <= 2) break;
        if (half) __syncthreads();
        if (wave >= hw + w0 && wave < hw + w0 + n) {
#pragma unroll
          for (int q = 0; q < 16; ++q) red[((wave - hw - w0) * 16 + q) * 64 + lane] = acc[q >> 2][q & 3];
        }
        __syncthreads();
        if (wave >= w0 && wave < w0 + n) {
#pragma unroll
          for (int q = 0; q < 16; ++q) acc[q >> 2][q & 3] += red[((wave - w0) * 16 + q) * 64 + lane];
        }
      }
    }
    if (wave == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = lane + 64 * r;
        const double R2 = A.hf_R2[j], f = pknorm * R2;
        s_sig[j] = acc[r][0] * pknorm;
        s_S[j] = acc[r][1] * f;
        s_S[NHF_R + j] = acc[r][2] * (f * R2);
        s_S[2 * NHF_R + j] = acc[r][3] * (f * R2 * R2);
      }
    }
  } else {
    // The dual sums are one product S[j][col] = sum_i E_ij V_i,col with a
    // column per (component, p): 8 (ND = 1) or 32 (ND = 7), on the FP64 matrix
    // cores, 16 x 16 x 4 at a time.  Lane l of an operand holds k node l / 16 of
    // the step; wave w takes the 16-node R tiles w, w + NW, ...
    constexpr int NC = (4 * W + 15) / 16, NTL = 16 / NW;
    const double* rawd = reinterpret_cast<const double*>(raw);
    const int li = lane & 15, lg = lane >> 4;
    __syncthreads();
    if (tid < NGROW) s_g[tid] = G[0];  // every thread has read the raw table
    f64x4 acc[NTL][NC];
#pragma unroll
    for (int t = 0; t < NTL; ++t)
#pragma unroll
      for (int n = 0; n < NC; ++n) acc[t][n] = f64x4{0.0, 0.0, 0.0, 0.0};
    // steps of 4 k nodes, the E rows of U steps in flight; the 257th node last
    auto load = [&](int k, double* e) {
#pragma unroll
      for (int t = 0; t < NTL; ++t) e[t] = A.hf_E[(size_t)k * NHF_R + 16 * (wave + NW * t) + li];
    };
    const double* kp = reinterpret_cast<const double*>(smem) + L::KP;
    auto product = [&](int k, const double* e, bool on) {  // off: the lane's k node counts for nothing
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int col = 16 * n + li, pp = min(col / W, 3), comp = col % W;
        double v = rawd[k * W + comp] * kp[4 * k + pp];
        v = on ? v : 0.0;
#pragma unroll
        for (int t = 0; t < NTL; ++t) acc[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(e[t], v, acc[t][n], 0, 0, 0);
      }
    };
    constexpr int U = 8;
    static_assert((NHF_K - 1) % (4 * U) == 0, "whole steps and one node");
    for (int i = 0; i + 1 < NHF_K; i += 4 * U) {
      double e[U][NTL];
#pragma unroll
      for (int u = 0; u < U; ++u) load(i + 4 * u + lg, e[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) product(i + 4 * u + lg, e[u], true);
    }
    {
      double e[NTL];
      load(NHF_K - 1, e);
      product(NHF_K - 1, e, lg == 0);
    }
    double* out = reinterpret_cast<double*>(s_sig);
#pragma unroll
    for (int t = 0; t < NTL; ++t)
#pragma unroll
      for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * (wave + NW * t) + lg + 4 * r, col = 16 * n + li, pp = col / W, comp = col - pp * W;
          const double R2 = A.hf_R2[j];
          const double f = pp == 0 ? 1.0 : (pp == 1 ? R2 : (pp == 2 ? R2 * R2 : R2 * R2 * R2));
          if (pp < 4) out[(size_t)(pp * NHF_R + j) * W + comp] = acc[t][n][r] * f;
        }
    __syncthreads();
    for (int j = tid; j < 4 * NHF_R; j += NT) s_sig[j] = s_sig[j] * pknorm;
  }
  __syncthreads();

  // ------------------------------------------- per a-node, transfer table
  // The transfer table's range: ln k = ln(ell + 1/2) - ln max(chi, 1) over the
  // call's multipoles and a-nodes; chi falls with a, so its ends are at the
  // first and last node.
  auto segments = [&](int m, Sd& chi, Sd& g) {
    ASeg sg;
    if (A.a_seg) {
      sg = A.a_seg[m];
    } else {
      const double a = A.a_list[m], l10a = ::log10(a);
      int i, j;
      logtab_segment(a, l10a, A.atab_chi, NCHI, i, j, sg.tc);
      sg.ci = (int16_t)i;
      sg.cj = (int16_t)j;
      logtab_segment(a, l10a, A.atab_g, NGROW, i, j, sg.tg);
      sg.gi = (int16_t)i;
      sg.gj = (int16_t)j;
    }
    chi = maxc(s_chi[sg.ci] + (s_chi[sg.cj] - s_chi[sg.ci]) * sg.tc, 0.0);  // background.py:242
    g = s_g[sg.gi] + (s_g[sg.gj] - s_g[sg.gi]) * sg.tg;
    g = minc(maxc(g, 0.0), 1.0);                                            // background.py:488
  };
  const bool tab = (ND == 0 || WO == 8) && A.ehtab;
  float lo = 0.0f, invh = 0.0f;
  double h = 0.0;
  if (tab) {
    // served batches: each cosmology's own multipoles (its request's columns)
    const double* ell = A.ell;
    int n_ell = A.n_ell, stride = 1;
    if (A.rjobs) {
      const RJob& jb = A.rjobs[c];
      ell = &A.rcols[jb.col0].ell;
      n_ell = jb.n_ell;
      stride = (int)(sizeof(RCol) / sizeof(double));
    }
    double l0 = 1e300, l1 = -1e300;
    for (int l = lane; l < n_ell; l += 64) {
      const double v = ell[(size_t)l * stride];
      l0 = fmin(l0, v);
      l1 = fmax(l1, v);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      l0 = fmin(l0, __shfl_xor(l0, o, 64));
      l1 = fmax(l1, __shfl_xor(l1, o, 64));
    }
    Sd ca, cb, g;
    segments(0, ca, g);
    segments(A.Na - 1, cb, g);
    // a margin of a few float ulps of ln k on both sides: every point's
    // position lies inside the table whichever way it is rounded
    constexpr double MARGIN = 2e-5;
    lo = (float)(::log((l0 + 0.5) / fmax(val(ca), 1.0)) - MARGIN);
    const double span = fmax(::log((l1 + 0.5) / fmax(val(cb), 1.0)) + MARGIN - (double)lo, 1e-3);
    // the nodes are x_q = lo + q / invh with invh a float rounded down, so
    // NEHQ intervals cover the range and positions are exact
    invh = (float)(NEHQ / span);
    if ((double)invh * span > (double)NEHQ) invh = nextafterf(invh, 0.0f);
    h = 1.0 / (double)invh;
    if (tid == 0 && dir == 0) {
      A.crec[((size_t)c * NCREC + CR_EHLO) * WO] = lo;
      A.crec[((size_t)c * NCREC + CR_EHINVH) * WO] = invh;
    }
  }
  // T(k) k^(n_s/2) (transfer.py:119-149, power.py:14-18) and its ln k
  // derivative at the table's nodes, in float with forward-mode duals; each
  // value is moved from the float-rounded node to the exact one with its
  // derivative
  // (one direction a workgroup: the samples are too few, the moments' k rows are free)
  float2* s_nd = SPLIT ? reinterpret_cast<float2*>(reinterpret_cast<double*>(smem) + L::KP)
                       : reinterpret_cast<float2*>(ND == 0 ? s_x : s_smp);  // [NEHQ + 1]
  static_assert(!SPLIT || 4 * NHF_K >= NEHQ + 1, "the nodes fit the k rows");
  const float hns = 0.5f * (float)val(cp.n_s);
  auto table_node = [&](int q) {
    using D1 = Dual<float, 1>;
    const EHc<D1> e1 = eh_from<D1>([&](int i) { return Make<D1>::c(val(s_eh[i])); }, A.transfer_model);
    const double xn = (double)lo + (double)q * h;
    D1 x, k, ik;
    x.v = (float)xn;
    x.d[0] = 1.0f;
    k.v = jm::exp(x.v);
    k.d[0] = k.v;
    ik.v = jm::exp(-x.v);
    ik.d[0] = -ik.v;
    const D1 tn = eh_transfer(e1, k, ik, x) * jm::exp(hns * x);
    s_nd[q] = make_float2(tn.v + tn.d[0] * (float)(xn - (double)x.v), tn.d[0]);
  };
  const double c2 = C_KMS * C_KMS;
  const float dlnk = (float)(A.hf_lnk[1] - A.hf_lnk[0]);
  const float lnk0 = (float)A.hf_lnk[0];
  const double lr0 = A.logr[0], hR = A.logr[1] - A.logr[0];
  auto a_node = [&](int m) {
    const double a = A.a_list[m];
    const double lna = A.a_ln ? A.a_ln[m] : ::log(a);
    const double ia = 1.0 / a;
    Sd chi, g;
    segments(m, chi, g);
    const Sd efde = jm::exp(f_de_ln(cp, a, lna));
    const Sd E2 = Esqr_parts(cp, ia, efde);
    const Sd iE2 = 1.0 / E2;
    const Sd sqE = jm::sqrt(E2);
    const Sd dchida = RH * (ia * ia) * (sqE * iE2);                        // background.py:294
    const Sd g2 = g * g;
    // nonlinear scale: interp(1.0, sigma^2(R, a), ln R) with sigma^2 decreasing
    const double g2v = val(g2);
    int lo_j = 0, hi_j = NHF_R;  // first j with g2 * sig_j < 1
    while (lo_j < hi_j) {
      const int mid = (lo_j + hi_j) >> 1;
      if (g2v * val(s_sig[mid]) < 1.0) hi_j = mid; else lo_j = mid + 1;
    }
    int ind;
    if (lo_j == 0) ind = 0;
    else if (lo_j == NHF_R) ind = NHF_R - 1;
    else {
      const double d0 = (1.0 - g2v * val(s_sig[lo_j - 1])) * (1.0 - g2v * val(s_sig[lo_j - 1]));
      const double d1 = (1.0 - g2v * val(s_sig[lo_j])) * (1.0 - g2v * val(s_sig[lo_j]));
      ind = (d1 < d0) ? lo_j : lo_j - 1;
    }
    ind = ind < 1 ? 1 : (ind > NHF_R - 2 ? NHF_R - 2 : ind);
    // clip(1, xp[1], xp[-2]) returns xp[-2] for a decreasing table, so the
    // side is sign(xp[254] - xp[ind]): left segment unless ind == 254
    const double xcl = g2v * val(s_sig[NHF_R - 2]);
    const int nb = (xcl - g2v * val(s_sig[ind]) < 0.0) ? ind - 1 : ind + 1;
    const Sd Sind = g2 * s_sig[ind];
    const Sd Snb = g2 * s_sig[nb];
    const Sd root = A.logr[ind] + (A.logr[nb] - A.logr[ind]) / (Snb - Sind) * (1.0 - Sind);
    constexpr double LN_RMIN = -13.815510557964274;  // ln 1e-6
    const Sd Rnl = maxc(jm::exp(root), 1e-6);                             // power.py:113-115
    // n_eff and C (power.py:118-139): n_eff + 3 = 2 g^2 S1(R_nl),
    // C = (n_eff+3)^2 + 4 g^2 (S1 - S2), S1/S2 by the Hermite interpolant of
    // the moment tables.  Outside the R grid (R_nl < 1e-4 or > 10, only for
    // scale factors well before a = 1/11) the sums are taken directly: float
    // terms, float partial sums of 16 terms, double totals, skipping y < 1e-3
    // (relative size < 1e-12) and y^2 > 40.
    Sd S1, S2;
    const Sd uR = (root - lr0) * (1.0 / hR);
    const int qR = (int)::floor(val(uR));
    if (qR >= 0 && qR <= NHF_R - 2) {
      const Sd tR = uR - (double)qR;
      const Sd* S1t = s_S;
      const Sd* S2t = s_S + NHF_R;
      const Sd* S3t = s_S + 2 * NHF_R;
      S1 = hermite(tR, hR, S1t[qR], S1t[qR + 1], 2.0 * (S1t[qR] - S2t[qR]), 2.0 * (S1t[qR + 1] - S2t[qR + 1]));
      S2 = hermite(tR, hR, S2t[qR], S2t[qR + 1], 4.0 * S2t[qR] - 2.0 * S3t[qR],
                   4.0 * S2t[qR + 1] - 2.0 * S3t[qR + 1]);
    } else {
      Sf Rf = conv<Sf>(Rnl);
      int ibeg = (int)((logf(1e-3f / val(Rf)) - lnk0) / dlnk);
      ibeg = ibeg < 0 ? 0 : (ibeg > NHF_K ? NHF_K : ibeg);
      S1 = zero<Sd>();
      S2 = zero<Sd>();
      for (int i0 = ibeg; i0 < NHF_K; i0 += 16) {
        Sf p1 = Make<Sf>::c(0.0), p2 = Make<Sf>::c(0.0);
        const int iend = i0 + 16 < NHF_K ? i0 + 16 : NHF_K;
        bool stop = false;
        for (int i = i0; i < iend; ++i) {
          Sf y = s_k32[i] * Rf;
          Sf y2 = y * y;
          if (val(y2) > 40.0f) { stop = true; break; }
          Sf ty2 = s_p1f[i] * jm::exp(-y2) * y2;
          p1 += ty2;
          p2 += ty2 * y2;
        }
        S1 = S1 + conv<Sd>(p1);
        S2 = S2 + conv<Sd>(p2);
        if (stop) break;
      }
      S1 = S1 * pknorm;
      S2 = S2 * pknorm;
    }
    const Sd n3 = 2.0 * g2 * S1;
    const Sd n_eff = n3 - 3.0;
    const Sd Cc = n3 * n3 + 4.0 * g2 * (S1 - S2);
    const Sd omm = cp.Omega_m * (ia * ia * ia) * iE2;
    const Sd omde = cp.Omega_de * efde * iE2;
    const HFa<Sd> hf = halofit_coefs(n_eff, Cc, omm, omde, w_de(cp, a), A.halofit_model);
    const Sd chi1 = maxc(chi, 1.0);                                        // angular_cl.py:73
    const Sd invchi = 1.0 / chi1;
    // max(chi^2, 1) = max(chi, 1)^2 (angular_cl.py:91,96)
    const Sd wgt = (A.a_wgt[m] / c2) * dchida * (invchi * invchi);

    float* cf = A.coef + ((size_t)c * A.Na + m) * NCOEF * WO;
    if (ND == 0 && A.ehtab) {  // forward record (FwdSlot)
      if constexpr (ND == 0) {
        const double iRnl = 1.0 / Rnl, yc = Rnl * invchi, iyc = chi1 * iRnl, c3 = chi1 * chi1 * chi1;
        const double lnchi = jm::logf_acc(chi1);
        const double u = (-lnchi - (double)lo) * (double)invh, uf = ::floor(u);
        float4* o = reinterpret_cast<float4*>(cf);
        o[0] = make_float4(__builtin_bit_cast(float, (int)uf), (float)(u - uf),
                           (float)(g2 * pknorm * (invchi * invchi * invchi) * (1.0 / (2.0 * PI * PI))),
                           (float)((fmax(root, LN_RMIN) - lnchi) * 1.4426950408889634));
        o[1] = make_float4((float)yc, (float)(hf.mu_n * iyc), (float)(hf.nu_n * (iyc * iyc)), (float)hf.beta_n);
        o[2] = make_float4((float)hf.f1x3, (float)hf.f2, (float)hf.gam3, (float)(hf.gam3 * hf.lg_cf3));
        o[3] = make_float4((float)hf.alpha_n, (float)hf.b_n, (float)hf.a_n, (float)(2.0 * PI * PI * c3 * wgt));
        cf[FT_CHI] = (float)chi;
      }
    } else {
      put(cf + CF_INV_CHI * WO, invchi);
      put(cf + CF_CHI1 * WO, chi1);
      // the logarithms stored as floats are taken to float accuracy
      put(cf + CF_LNINVCHI * WO, -jm::logf_acc(chi1));
      put(cf + CF_KNL * WO, 1.0 / Rnl);
      put(cf + CF_MU * WO, hf.mu_n);
      put(cf + CF_WGT * WO, wgt);
      put(cf + CF_G2P * WO, g2 * pknorm);
      put(cf + CF_LGRNL * WO, maxc(root, LN_RMIN) * 1.4426950408889634);
      put(cf + CF_RNL * WO, Rnl);
      put(cf + CF_AN * WO, hf.a_n);
      put(cf + CF_BN * WO, hf.b_n);
      put(cf + CF_LGCF3 * WO, hf.lg_cf3);
      put(cf + CF_GAM3 * WO, hf.gam3);
      put(cf + CF_ALPHA * WO, hf.alpha_n);
      put(cf + CF_BETA * WO, hf.beta_n);
      put(cf + CF_NU * WO, hf.nu_n);
      put(cf + CF_F1X3 * WO, hf.f1x3);
      put(cf + CF_F2 * WO, hf.f2);
      put(cf + CF_CHI * WO, chi);
      put(cf + CF_GROWTH * WO, g);
    }

    // z-local kernels, H = H0 sqrt(E^2) (background.py:129-148): number
    // counts n(z) b H (probes.py:87-99) and the NLA terms (probes.py:114-124)
    for (int t = 0; t < A.nLoc; ++t) {
      Sd r = A.loc_nb[(size_t)t * A.Na + m] * (H0 * sqE);
      const int mode = A.loc_mode[t];
      if (mode & LOC_INVD) r = r / g;             // bias.py:38-40: b / D(a)
      if (mode & LOC_IA) r = r * cp.Omega_m / g;  // probes.py:120-122
      // R columns: the pool column, or (served batches) each position of
      // the request that selects the tracer
      const int lc = A.loc_col[t];
      uint32_t cmask = 1u << lc;
      if (A.rjobs) {
        const RJob& jb = A.rjobs[c];
        const int T = jb.T;
        cmask = 0;
#pragma unroll
        for (int i = 0; i < MAXT; ++i) cmask |= (i < T && jb.sel[i] == lc ? 1u : 0u) << i;
      }
      const size_t rb = ((size_t)c * A.Na + m) * A.Tpad;
      for (uint32_t mk = cmask; mk; mk &= mk - 1) put(A.R + (rb + __builtin_ctz(mk)) * WO, r);
    }
    if (A.dbg) {
      double* d = A.dbg + (size_t)c * A.dbg_stride + 1024 + (size_t)m * 8;
      d[0] = val(chi); d[1] = val(g); d[2] = 1.0 / val(Rnl); d[3] = val(n_eff); d[4] = val(Cc);
      d[5] = val(dchida);
    }
  };
  const int na_tasks = (A.Na + 63) / 64, nt_tasks = tab ? (NEHQ + 64) / 64 : 0;
  for (;;) {
    int t = 0;
    if (lane == 0) t = atomicAdd(s_next, 1);
    t = __builtin_amdgcn_readfirstlane(t);
    if (t >= na_tasks + nt_tasks) break;
    if (t < na_tasks) {
      if (64 * t + lane < A.Na) a_node(64 * t + lane);
    } else {
      const int q = 64 * (t - na_tasks) + lane;
      if (q <= NEHQ) {
        if (dir == 0) table_node(q);
        if constexpr (ND == 7) eh_dtab_node<W>(c, q, (double)lo, h, A.crec, A.ehtab7);
        if constexpr (SPLIT) {
          const EHc<Sf> e1 = eh_from<Sf>([&](int i) { return conv<Sf>(s_eh[i]); }, A.transfer_model);
          const float x = (float)((double)lo + (double)q * h), k = jm::exp(x), ik = jm::exp(-x);
          const Sf tn = eh_transfer(e1, k, ik, x) * jm::exp(conv<Sf>(cp.n_s) * (0.5f * x));
          float* o = A.ehtab7 + ((size_t)c * (NEHQ + 1) + q) * NEHD_ROW;
          o[dir] = tn.d[0];
          if (dir == 0) o[7] = 0.0f;
        }
      }
    }
  }
  if (A.dbg && tid < NCHI) {
    double* d = A.dbg + (size_t)c * A.dbg_stride;
    d[tid] = val(s_chi[tid]);
    if (tid < NGROW) d[256 + tid] = val(s_g[tid]);
    d[384 + tid] = val(s_sig[tid]);
    if (tid == 0) d[640] = val(pknorm);
  }
  if (!tab || dir != 0) return;  // uniform over the workgroup
  __syncthreads();
  // cubic Hermite pieces of T(k) k^(n_s/2) between the nodes
  const float hf = (float)h;
  float4* dst = A.ehtab + (size_t)c * NEHQ;
  for (int q = tid; q < NEHQ; q += NT) {
    const float2 n0 = s_nd[q], n1 = s_nd[q + 1];
    const float e0 = hf * n0.y, e1d = hf * n1.y;
    dst[q] = make_float4(n0.x, e0, 3.0f * (n1.x - n0.x) - 2.0f * e0 - e1d, 2.0f * (n0.x - n1.x) + e0 + e1d);
  }
}

// Growth rate and transverse comoving distance at the n scale factors of a
// background call (slots 6 and 7 of each per-a block of dbg), from the table
// kernel's FP64 output for the same call: chi in slot 0 and, for the ODE
// model, the growth-rate table in slots 768..895 of the table block.
__global__ __launch_bounds__(256) void k_background_ex(const double* params, const double* a, int n,
                                                       const double* atab_g, int growth_model, double gamma,
                                                       double* dbg) {
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m >= n) return;
  double p[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = params[i];
  const CosmoP<double> cp = make_cosmo(p);
  double* d = dbg + 1024 + (size_t)m * 8;
  const double x = a[m];
  if (growth_model == 0) {
    d[6] = interp_logtab(x, ::log10(x), atab_g, dbg + 768, NGROW);  // background.py:490-512
  } else {  // background.py:551-582: Omega_m(a)^gamma at a
    const double ix = 1.0 / x;
    const double omm = cp.Omega_m * (ix * ix * ix) / Esqr_parts(cp, ix, ::exp(f_de_ln(cp, x, ::log(x))));
    d[6] = ::exp(gamma * ::log(omm));
  }
  // background.py:297-344: the branch of k = -sign(Omega_k)
  const double ok = cp.Omega_k, sk = ::sqrt(::fabs(ok)), chi = d[0];
  d[7] = ok > 0.0 ? RH / sk * ::sinh(sk * chi / RH) : (ok < 0.0 ? RH / sk * ::sin(sk * chi / RH) : chi);
}

hipError_t launch_background_ex(const double* params, const double* a, int n, const double* atab_g,
                                int growth_model, double gamma, double* dbg, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_background_ex, dim3((n + 255) / 256), dim3(256), 0, s, params, a, n, atab_g, growth_model,
                     gamma, dbg);
  return hipGetLastError();
}

// Forward tables: 1 = 256 threads at 4 waves/SIMD (some register spills), 2 =
// 256 threads at 2 waves/SIMD, 3 = 512 threads at 2 waves/SIMD, 0 = by the
// number of cosmologies: one workgroup per CU takes all of its registers (3)
// while there is at most one for each, two share it (2) up to two each, and
// four (1) beyond.  Measured on 256 CUs, n_z 512, for 3 / 2 / 1 in us: 31 / 36 / 40
// at 1 cosmology, 45 / 52 / 54 at 256, 79 / 58 / 63 at 512, 136 / 105 / 92 at 1024.
// Dual tables: while there is at most one workgroup per CU, one of 512 threads
// per cosmology and direction (the adjoint's seven directions apart); beyond, 256
// threads, and the adjoint's directions together.  Measured, n_z 512: directions
// apart 85 -> 49 us at 1 cosmology, 106 -> 82 at 36, but 105 -> 119 at 73; 512
// threads against 256 for one direction 43 / 51 us at 7 rows, 54 / 64 at 210, 96 / 78
// at 420.
hipError_t launch_tables(int nd, const TablesArgs& a, hipStream_t s, int num_cu, int variant) {
  const size_t sm = nd == 0 ? TabLds<0>::bytes() : (nd == 1 ? TabLds<1>::bytes() : TabLds<7>::bytes());
  if (nd == 0) {
    if (variant == 0) variant = a.B <= num_cu ? 3 : (a.B <= 2 * num_cu ? 2 : 1);
    switch (variant) {
      case 1: hipLaunchKernelGGL((k_tables<0, 256, 4>), dim3(a.B), dim3(256), sm, s, a); break;
      case 3: hipLaunchKernelGGL((k_tables<0, 512, 2>), dim3(a.B), dim3(512), sm, s, a); break;
      default: hipLaunchKernelGGL((k_tables<0, 256, 2>), dim3(a.B), dim3(256), sm, s, a); break;
    }
  } else if (nd == 1) {
    if (a.B <= num_cu) hipLaunchKernelGGL((k_tables<1, 512, 2>), dim3(a.B), dim3(512), sm, s, a);
    else hipLaunchKernelGGL((k_tables<1, 256, 2>), dim3(a.B), dim3(256), sm, s, a);
  } else if (nd == 7 && 7 * (int64_t)a.B <= num_cu && !a.dB) {  // (a.dB: the live count is on the device)
    hipLaunchKernelGGL((k_tables<1, 512, 2, 8>), dim3(7 * a.B), dim3(512), TabLds<1>::bytes(), s, a);
  } else if (nd == 7) {
    hipLaunchKernelGGL((k_tables<7, 256, 1>), dim3(a.B), dim3(256), sm, s, a);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The theta derivatives of the transfer table's function at node q (float duals
// at fixed k), for 4-point Lagrange interpolation in the adjoint kernel.  W = 8
// is the record width: 7 derivatives after each value.
template <int W>
JC_D void eh_dtab_node(int c, int q, double lo, double h, const float* crec, float* ehtab7) {
  using D7 = Dual<float, 7>;
  D7 ns;
  const EHc<D7> e = load_eh<D7, W>(crec + (size_t)c * NCREC * W, ns);
  const float x = (float)(lo + (double)q * h);
  const float k = jm::exp(x), ik = jm::exp(-x);
  const D7 tn = eh_transfer(e, k, ik, x) * jm::exp(ns * (0.5f * x));
  float4* o = reinterpret_cast<float4*>(ehtab7 + ((size_t)c * (NEHQ + 1) + q) * NEHD_ROW);
  o[0] = make_float4(tn.d[0], tn.d[1], tn.d[2], tn.d[3]);
  o[1] = make_float4(tn.d[4], tn.d[5], tn.d[6], 0.0f);
}

// ------------------------------------------------------------------ KDE n(z)
// One thread per evaluation point.  The catalog is sorted by redshift, so a
// point only visits galaxies within 8.5 bandwidths (the rest weigh below
// exp(-36) ~ 2e-16 of the nearest ones); exponentials in float, sums in double.
__global__ void k_kde(const double* __restrict__ z, int64_t n, const double* __restrict__ cz,
                      const double* __restrict__ cw, int64_t ncat, double bw, double scale,
                      double* __restrict__ out) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double zp = z[p];
  const double lo = zp - 8.5 * bw;
  int64_t a = 0, b = ncat;  // first galaxy with cz >= lo
  while (a < b) {
    const int64_t mid = (a + b) >> 1;
    if (cz[mid] < lo) a = mid + 1; else b = mid;
  }
  const double hi = zp + 8.5 * bw;
  const float c2 = (float)(-0.5 / (bw * bw));
  double s = 0.0;
  for (int64_t k = a; k < ncat && cz[k] <= hi; ++k) {
    const float d = (float)(zp - cz[k]);
    s += cw[k] * (double)jm::exp(c2 * d * d);
  }
  out[p] = s * scale;
}

hipError_t launch_kde(const double* z, int64_t n, const double* cz, const double* cw, int64_t ncat, double bw,
                      double wsum, double* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const double scale = 1.0 / (sqrt(2.0 * PI) * bw) / wsum;
  hipLaunchKernelGGL(k_kde, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, z, n, cz, cw, ncat, bw, scale, out);
  return hipGetLastError();
}

}  // namespace jc
