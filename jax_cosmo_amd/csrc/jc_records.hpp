// Device-side readers of the per-cosmology (crec) and per-(cosmology, a)
// (coef) records that the table kernel writes and the Limber and transfer
// table kernels consume.
#pragma once
#include "jc_kernels.hpp"
#include "jc_physics.hpp"

namespace jc {

template <class Sf, int W>
struct PointCoefs {
  Sf invchi, chi1, lninvchi, wgt, g2p, lgRnl, Rnl, knl;
  HFa<Sf> hf;
};

template <class Sf, int W>
JC_D PointCoefs<Sf, W> load_coefs(const float* cf) {
  PointCoefs<Sf, W> r;
  r.invchi = Mem<Sf>::ld(cf + CF_INV_CHI * W);
  r.chi1 = Mem<Sf>::ld(cf + CF_CHI1 * W);
  r.lninvchi = Mem<Sf>::ld(cf + CF_LNINVCHI * W);
  r.wgt = Mem<Sf>::ld(cf + CF_WGT * W);
  r.g2p = Mem<Sf>::ld(cf + CF_G2P * W);
  r.lgRnl = Mem<Sf>::ld(cf + CF_LGRNL * W);
  r.Rnl = Mem<Sf>::ld(cf + CF_RNL * W);
  r.knl = Mem<Sf>::ld(cf + CF_KNL * W);
  r.hf.a_n = Mem<Sf>::ld(cf + CF_AN * W);
  r.hf.b_n = Mem<Sf>::ld(cf + CF_BN * W);
  r.hf.lg_cf3 = Mem<Sf>::ld(cf + CF_LGCF3 * W);
  r.hf.gam3 = Mem<Sf>::ld(cf + CF_GAM3 * W);
  r.hf.alpha_n = Mem<Sf>::ld(cf + CF_ALPHA * W);
  r.hf.beta_n = Mem<Sf>::ld(cf + CF_BETA * W);
  r.hf.nu_n = Mem<Sf>::ld(cf + CF_NU * W);
  r.hf.f1x3 = Mem<Sf>::ld(cf + CF_F1X3 * W);
  r.hf.f2 = Mem<Sf>::ld(cf + CF_F2 * W);
  r.hf.mu_n = Mem<Sf>::ld(cf + CF_MU * W);
  return r;
}

template <class Sf, int W>
JC_D EHc<Sf> load_eh(const float* cr, Sf& ns) {
  EHc<Sf> e;
  e.fb = Mem<Sf>::ld(cr + CR_FB * W);
  e.fc = Mem<Sf>::ld(cr + CR_FC * W);
  e.inv13keq = Mem<Sf>::ld(cr + CR_INV13KEQ * W);
  e.ln_inv13keq = Mem<Sf>::ld(cr + CR_LNINV13 * W);
  e.beta_c18 = Mem<Sf>::ld(cr + CR_BETAC18 * W);
  e.c14a = Mem<Sf>::ld(cr + CR_C14A * W);
  e.sh_d = Mem<Sf>::ld(cr + CR_SHD * W);
  e.alpha_b = Mem<Sf>::ld(cr + CR_ALPHAB * W);
  e.beta_b = Mem<Sf>::ld(cr + CR_BETAB * W);
  e.beta_node = Mem<Sf>::ld(cr + CR_BETANODE * W);
  e.ln_ksilk = Mem<Sf>::ld(cr + CR_LNKSILK * W);
  e.bnode_shd = Mem<Sf>::ld(cr + CR_BNODE_SHD * W);
  e.bb_shd = Mem<Sf>::ld(cr + CR_BB_SHD * W);
  e.alpha_g = Mem<Sf>::ld(cr + CR_ALPHAG * W);
  e.tq = Mem<Sf>::ld(cr + CR_TQ * W);
  e.nw = cr[CR_NW * W] != 0.0f;
  ns = Mem<Sf>::ld(cr + CR_NS * W);
  return e;
}

// The forward record (FwdSlot) of one a-node: four float4.
struct FwdRec {
  float4 a, b, c, d;
};
JC_D FwdRec load_fwd(const float* cf) {
  const float4* p = reinterpret_cast<const float4*>(cf);
  return FwdRec{p[0], p[1], p[2], p[3]};
}

// Per-lane constants of a column in transfer-table mode: l = ell + 1/2, its
// powers and logarithm, and ln(l) in units of the table's spacing, split into
// an integer and a fraction (so that the position within a piece keeps the
// float's whole precision).
struct EllT {
  float l, il, l3, lg;
  int q;
  float t;
};
JC_D EllT ell_tab(double ell, double invh) {
  EllT e;
  const double l = ell + 0.5, ln = ::log(l);
  e.l = (float)l;
  e.il = (float)(1.0 / l);
  e.l3 = (float)(l * l * l);
  e.lg = (float)(ln * 1.4426950408889634);
  const double u = ln * invh, f = ::floor(u);
  e.q = (int)f;
  e.t = (float)(u - f);
  return e;
}
// the l^-3 that the sum over a leaves out
JC_D float ell_m3(double ell) {
  const double l = ell + 0.5;
  return (float)(1.0 / (l * l * l));
}

// Table piece of a point: its index, and its fraction in t.  The table is
// built a margin wider than the call's points, so the clamp acts on
// non-finite cosmologies only.
JC_D int tab_piece(const FwdRec& r, const EllT& e, float& t) {
  const float s = e.t + r.a.y;
  int q = e.q + __builtin_bit_cast(int, r.a.x) + (s >= 1.0f ? 1 : 0);
  t = __builtin_amdgcn_fractf(s);
  return min(max(q, 0), NEHQ - 1);
}

// l^3 M(a, ell) at the table piece cc, fraction t (FwdSlot): P_nl of
// power.py:244-262 with its three quotients over one reciprocal; 34 simple and
// 6 transcendental instructions with tab_piece.
JC_D float fwd_point(const float4& cc, float t, const FwdRec& r, const EllT& e) {
  constexpr float A1 = (float)(0.25 * 1.4426950408889634), A2 = (float)(0.125 * 1.4426950408889634);
  const float tn = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(cc.w, t, cc.z), t, cc.y), t, cc.x);
  const float d2l = ((tn * tn) * e.l3) * r.a.z;
  const float L1 = jm::log2(1.0f + d2l);
  const float y = e.l * r.b.x;
  const float fy2 = y * __builtin_fmaf(y, A2, A1);  // f(y) = y/4 + y^2/8, base 2
  const float eq = jm::exp2(__builtin_fmaf(r.b.w, L1, -fy2));
  const float lgy = e.lg + r.a.w;
  const float yf1 = jm::exp2(r.c.x * lgy);
  const float yf2 = jm::exp2(r.c.y * lgy);
  const float ycg = jm::exp2(__builtin_fmaf(r.c.z, lgy, r.c.w));
  const float d0 = __builtin_fmaf(r.d.x, d2l, 1.0f);
  const float d12 =
      __builtin_fmaf(r.d.y, yf2, 1.0f + ycg) * __builtin_fmaf(e.il, __builtin_fmaf(e.il, r.b.z, r.b.y), 1.0f);
  const float num = __builtin_fmaf(d2l * eq, d12, (r.d.z * yf1) * d0);
  return (r.d.w * num) * __builtin_amdgcn_rcpf(d0 * d12);
}

}  // namespace jc
