// Adjoint of the Limber sum in transfer-table mode: theta-bar = sum over
// (ell, pairs) of Cbar_ij dC_ij/dtheta for theta = (Omega_c, Omega_b, h, n_s,
// sigma8, w0, wa), with C_ij(ell) = F_i F_j sum_a R_i R_j M(a, ell) as in the
// forward kernel.
//
// Everything but T(k) depends on theta through quantities of one a-node: the
// 14 record fields that M is made of and the tracer kernels R_i, whose theta
// derivatives the table and lensing kernels stored.  So the sum over ell is
// taken first, and the derivatives are contracted once per node instead of
// once per point: lane = a-node, loop over ell,
//   V_i = 1/2 sum_j ct_ij R_j (ct symmetric, diagonal doubled),  G = sum_i R_i V_i,
//   Rbar_i += 2 M V_i,   xbar += G dM/dx for each record field x,
// then theta-bar = sum_nodes (sum_x xbar dx/dtheta + sum_i Rbar_i dR_i/dtheta)
// plus T(k)'s own derivative at fixed k, read from the table of theta
// derivatives at every point (4-point Lagrange).  The lanes' 31 sums and the
// node's record stay in registers; the cotangents and the multipole's
// constants are the same for all lanes and come from LDS as broadcasts.
// With lane = (cosmology, ell) instead, every point reads the node's 224 dual
// floats and spends 7 FMAs on each.  Measured, 256 cosmologies x 100 ell x n_z
// 512: 10 tracers 610 -> 160 us; bound by VALU issue (300 instructions a point,
// 120 of them the cotangents' share, which takes 35 of the 160 us) with the LDS
// reads of a point beside it (25 float4, 9 of them gathers: 9 us).  Staging the
// tables costs 5-8 us and the contraction with the derivatives, 58 KB a block,
// 9-13 us.
#include "jc_records.hpp"

namespace jc {

namespace {

// multipoles staged per turn: two per wave, so that with the tables three
// blocks fit a CU's LDS (two points unrolled: no gain)
constexpr int ADJ_EC = 8;
constexpr int ADJ_HDR = 64;  // multipole constants computed per turn

// record fields with a theta derivative, in the order of the node sums: slots
// 2..5 (ln 1/chi, weight, D^2 pknorm, log2 R_nl), 8..16 (a_n .. f2), 19 (mu_n)
constexpr int ADJ_NX = 14;
JC_D int adj_slot(int j) { return j < 4 ? j + CF_LNINVCHI : (j < 13 ? j - 4 + CF_AN : CF_MU); }
static_assert(CF_LNINVCHI == 2 && CF_LGRNL == 5 && CF_AN == 8 && CF_F2 == 16, "adj_slot's ranges");

template <int T>
struct AdjShape {
  static constexpr int P = T * (T + 1) / 2;
  static constexpr int ROW = (P + 3) / 4 * 4 + 4;  // staged cotangents of a multipole; + 4 spreads the banks
  static constexpr int NQ = ADJ_NX + T;            // node sums
  static constexpr int LDS = 4 * NEHQ + 8 * (NEHQ + 1) + ADJ_EC * ROW + 8 * ADJ_HDR;  // floats
  static_assert(ADJ_WAVES * NQ * 64 + 2 * 64 * NQ + 64 <= LDS, "the reduction reuses the tables' space");
};

// What one block reads: `n1 - n0` <= 64 nodes of one cosmology, multipoles
// [l0, l1) of its cotangent block.
struct AdjIn {
  const float* coef;   // [Na][NCOEF][8]
  const float* R;      // [Na][Tpad][8]
  int Tpad;
  const float4* tab;   // [NEHQ]
  const float4* dtab;  // [NEHQ + 1][2]
  float lo, invh;
  const double* ell;   // multipole l at ell[l * estride]
  int estride;
  const float* cbar;   // [P][n_ell]
  int n_ell;
  uint32_t wl_mask;
  int l0, l1, n0, n1;
  float* out;          // [7]
};

template <int T>
JC_D void adjoint_block(const AdjIn& A, float4* lds4) {
  using S = AdjShape<T>;
  constexpr int P = S::P, ROW = S::ROW, NQ = S::NQ;
  constexpr float LN2 = 0.69314718055994531f, LOG2E = 1.4426950408889634f;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nn = A.n1 - A.n0;
  if (A.l0 >= A.l1) {  // no multipoles in this slice
    if (t < 7) A.out[t] = 0.0f;
    return;
  }
  float4* tab = lds4;
  float4* dA = tab + NEHQ;      // derivatives 0..3 at the table's nodes
  float4* dB = dA + NEHQ + 1;   // 4..6: apart, so that neighbouring nodes fill the banks
  float* rows = reinterpret_cast<float*>(dB + NEHQ + 1);
  float* hdr = rows + ADJ_EC * ROW;
  for (int e = t; e < NEHQ; e += 64 * ADJ_WAVES) tab[e] = A.tab[e];
  for (int e = t; e < 2 * (NEHQ + 1); e += 64 * ADJ_WAVES) (e & 1 ? dB : dA)[e >> 1] = A.dtab[e];

  // the node's record in the forward kernel's form (FwdSlot)
  const float* cf = A.coef + (size_t)(A.n0 + min(lane, nn - 1)) * NCOEF * 8;
  const float chi1 = cf[CF_CHI1 * 8], iyc = chi1 * cf[CF_KNL * 8];
  FwdRec r;
  {
    const float ic = cf[CF_INV_CHI * 8], lnic = cf[CF_LNINVCHI * 8];
    const double u = ((double)lnic - (double)A.lo) * (double)A.invh, uf = ::floor(u);
    r.a = make_float4(__builtin_bit_cast(float, (int)uf), (float)(u - uf),
                      cf[CF_G2P * 8] * (ic * ic * ic) * (float)(1.0 / (2.0 * PI * PI)),
                      __builtin_fmaf(lnic, LOG2E, cf[CF_LGRNL * 8]));
    r.b = make_float4(cf[CF_RNL * 8] * ic, cf[CF_MU * 8] * iyc, cf[CF_NU * 8] * (iyc * iyc), cf[CF_BETA * 8]);
    r.c = make_float4(cf[CF_F1X3 * 8], cf[CF_F2 * 8], cf[CF_GAM3 * 8], cf[CF_GAM3 * 8] * cf[CF_LGCF3 * 8]);
    r.d = make_float4(cf[CF_ALPHA * 8], cf[CF_BN * 8], cf[CF_AN * 8],
                      (float)(2.0 * PI * PI) * (chi1 * chi1 * chi1) * cf[CF_WGT * 8]);
  }
  float Rv[T];
#pragma unroll
  for (int i = 0; i < T; ++i) Rv[i] = A.R[((size_t)(A.n0 + min(lane, nn - 1)) * A.Tpad + i) * 8];

  // staging of the cotangents: thread -> multipole t % EC, pairs t / EC + k NP;
  // each pair's power of the lensing factor and its share of V (1/2, diagonal 1)
  constexpr int NP = 64 * ADJ_WAVES / ADJ_EC, KP = (P + NP - 1) / NP;
  const int sl = t % ADJ_EC;
  int wlp[KP];
  float dia[KP];
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    int q = t / ADJ_EC + k * NP, i = 0;
    while (i < T && q >= T - i) q -= T - i++;
    wlp[k] = (int)((A.wl_mask >> i) & 1u) + (int)((A.wl_mask >> min(i + q, 31)) & 1u);
    dia[k] = q == 0 ? 1.0f : 0.5f;
  }
  auto fetch = [&](int l, float* v) {
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const int p = t / ADJ_EC + k * NP;
      v[k] = p < P && l < A.l1 ? A.cbar[(size_t)p * A.n_ell + l] : 0.0f;
    }
  };

  // node sums, all without the node's factor AW
  float aS = 0, aG3 = 0, aY = 0, aAL = 0, aB = 0, aAN = 0, aF1 = 0, aBN = 0, aF2 = 0, aC = 0, aGAM = 0, aMU = 0,
        aNU = 0, aSL = 0;
  float Rb[T], th[7];
#pragma unroll
  for (int i = 0; i < T; ++i) Rb[i] = 0.0f;
#pragma unroll
  for (int d = 0; d < 7; ++d) th[d] = 0.0f;

  auto point = [&](const float* h, const float* row) {
    const float4 h0 = *reinterpret_cast<const float4*>(h), h1 = *reinterpret_cast<const float4*>(h + 4);
    const float hq = h1.x;  // (a scalar: see EllT::q)
    const EllT e{h0.x, h0.y, h0.z, h0.w, __builtin_bit_cast(int, hq), h1.y};
    // the cotangents' share of this node
    float V[T];
#pragma unroll
    for (int i = 0; i < T; ++i) V[i] = 0.0f;
    {
      float cb[P];
#pragma unroll
      for (int p = 0; p < P; ++p) cb[p] = row[p];
      int p = 0;
#pragma unroll
      for (int i = 0; i < T; ++i) {
#pragma unroll
        for (int j = i; j < T; ++j) {
          V[i] = __builtin_fmaf(cb[p], Rv[j], V[i]);
          if (j > i) V[j] = __builtin_fmaf(cb[p], Rv[i], V[j]);
          ++p;
        }
      }
    }
    float G = 0.0f;
#pragma unroll
    for (int i = 0; i < T; ++i) G = __builtin_fmaf(Rv[i], V[i], G);
    G *= h1.z;  // here, not in the cotangents: l^-3 would take 40 bits of their range
    // the bracket S = q1 + q2 of fwd_point, q1 = d2l eq / d0, q2 = a_n yf1 / (A B)
    float ft;
    const int q = tab_piece(r, e, ft);
    const float4 cc = tab[q];
    constexpr float A1 = 0.25f * LOG2E, A2 = 0.125f * LOG2E;
    const float tn = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(cc.w, ft, cc.z), ft, cc.y), ft, cc.x);
    const float w = (tn * tn) * e.l3;
    const float d2l = w * r.a.z;
    const float L1 = jm::log2(1.0f + d2l);
    const float y = e.l * r.b.x;
    const float eq = jm::exp2(__builtin_fmaf(r.b.w, L1, -(y * __builtin_fmaf(y, A2, A1))));
    const float lgy = e.lg + r.a.w;
    const float yf1 = jm::exp2(r.c.x * lgy);
    const float yf2 = jm::exp2(r.c.y * lgy);
    const float ycg = jm::exp2(__builtin_fmaf(r.c.z, lgy, r.c.w));
    const float d0 = __builtin_fmaf(r.d.x, d2l, 1.0f);
    const float Aq = __builtin_fmaf(r.d.y, yf2, 1.0f + ycg);
    const float Bq = __builtin_fmaf(e.il, __builtin_fmaf(e.il, r.b.z, r.b.y), 1.0f);
    const float AB = Aq * Bq;
    const float rden = __builtin_amdgcn_rcpf(d0 * AB);
    const float r0 = rden * AB, r12 = rden * d0;
    const float ge = G * (eq * r0);   // G q1 / d2l
    const float p1 = ge * d2l;        // G q1
    const float gy = G * (yf1 * r12); // G q2 / a_n
    const float p2 = r.d.z * gy;      // G q2
    aS += p1 + p2;
    const float M = (r.d.w * h1.z) * __builtin_fmaf(d2l, eq * r0, r.d.z * (yf1 * r12));
#pragma unroll
    for (int i = 0; i < T; ++i) Rb[i] = __builtin_fmaf(M, V[i], Rb[i]);
    // q1: d ln q1 = (1 - alpha d2l / d0 + beta d2l / (1 + d2l)) d ln d2l
    //               - d2l / d0 dalpha + ln(1 + d2l) dbeta - (y + y^2) / 4 d ln y
    const float dr = d2l * r0;
    const float bd = (r.b.w * d2l) * __builtin_amdgcn_rcpf(1.0f + d2l);
    const float e1 = ge * (__builtin_fmaf(-r.d.x, dr, 1.0f) + bd);
    aG3 = __builtin_fmaf(e1, w, aG3);
    aAL = __builtin_fmaf(-p1, dr, aAL);
    aB = __builtin_fmaf(p1, L1, aB);
    aY = __builtin_fmaf(-p1, __builtin_fmaf(y, y, y), aY);
    // q2 = a_n y^f1 / ((1 + b y^f2 + (c f3 y)^(3 - gamma)) (1 + mu / y + nu / y^2))
    aAN += gy;
    aF1 = __builtin_fmaf(p2, lgy, aF1);
    const float pr = p2 * r12;
    const float pA = -pr * Bq, pB = -(pr * Aq) * e.il;
    const float pb = pA * yf2, pc = pA * ycg;
    aBN += pb;
    aF2 = __builtin_fmaf(pb, lgy, aF2);
    aC += pc;
    aGAM = __builtin_fmaf(pc, lgy, aGAM);
    aMU += pB;
    aNU = __builtin_fmaf(pB, e.il, aNU);
    // T(k): its slope in ln k reaches theta through chi, its derivative at
    // fixed k by 4-point Lagrange interpolation of the nodes' values
    const float Tb = e1 * (2.0f * tn * e.l3 * r.a.z);
    aSL = __builtin_fmaf(Tb, __builtin_fmaf(__builtin_fmaf(3.0f * cc.w, ft, 2.0f * cc.z), ft, cc.y), aSL);
    const int j0 = min(max(q - 1, 0), NEHQ - 3);
    const float s = ft + (float)(q - j0);
    const float s1 = s - 1.0f, s2 = s - 2.0f, s3 = s - 3.0f;
    const float s01 = s * s1, s23 = (s2 * s3) * Tb;
    const float w0 = -(1.0f / 6.0f) * s1 * s23, w1 = 0.5f * s * s23;
    const float w2 = -0.5f * (s01 * s3) * Tb, w3 = (1.0f / 6.0f) * (s01 * s2) * Tb;
    const float wj[4] = {w0, w1, w2, w3};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 a = dA[j0 + j], b = dB[j0 + j];
      th[0] = __builtin_fmaf(wj[j], a.x, th[0]);
      th[1] = __builtin_fmaf(wj[j], a.y, th[1]);
      th[2] = __builtin_fmaf(wj[j], a.z, th[2]);
      th[3] = __builtin_fmaf(wj[j], a.w, th[3]);
      th[4] = __builtin_fmaf(wj[j], b.x, th[4]);
      th[5] = __builtin_fmaf(wj[j], b.y, th[5]);
      th[6] = __builtin_fmaf(wj[j], b.z, th[6]);
    }
  };

  float nv[KP];
  fetch(A.l0 + sl, nv);
  for (int lc = A.l0; lc < A.l1; lc += ADJ_EC) {
    const int hl = (lc - A.l0) % ADJ_HDR;
    __syncthreads();  // the rows (and constants) before these have been read
    if (hl == 0) {
      if (wave == 0) {
        const double ell = A.ell[(size_t)min(lc + lane, A.l1 - 1) * A.estride];
        const EllT e = ell_tab(ell, (double)A.invh);
        const float lf =
            (float)(::sqrt((ell - 1.0) * ell * (ell + 1.0) * (ell + 2.0)) / ((ell + 0.5) * (ell + 0.5)));
        float4* o = reinterpret_cast<float4*>(hdr + lane * 8);
        o[0] = make_float4(e.l, e.il, e.l3, e.lg);
        o[1] = make_float4(__builtin_bit_cast(float, e.q), e.t, ell_m3(ell), lf);
      }
      __syncthreads();
    }
    {
      const float lf = hdr[(hl + sl) * 8 + 7];
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        const float F = wlp[k] == 0 ? 1.0f : (wlp[k] == 1 ? lf : lf * lf);
        const int p = t / ADJ_EC + k * NP;
        if (p < P) rows[sl * ROW + p] = nv[k] * (F * dia[k]);
      }
    }
    __syncthreads();
    if (lc + ADJ_EC < A.l1) fetch(lc + ADJ_EC + sl, nv);
    const int ne = min(ADJ_EC, A.l1 - lc);
#pragma unroll 1
    for (int e = wave; e < ne; e += ADJ_WAVES) point(hdr + (hl + e) * 8, rows + e * ROW);
  }

  // the waves' sums of each node, in order; then wave 0's lanes turn them into
  // cotangents of the record fields
  float* red = reinterpret_cast<float*>(lds4);
  double* xs = reinterpret_cast<double*>(red + ADJ_WAVES * NQ * 64);  // (the weight's cotangent needs the range)
  double* wsum = xs + 64 * NQ;  // [ADJ_WAVES][8]
  const float sums[ADJ_NX] = {aS, aG3, aY, aAL, aB, aAN, aF1, aBN, aF2, aC, aGAM, aMU, aNU, aSL};
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ADJ_NX; ++k) red[(wave * NQ + k) * 64 + lane] = sums[k];
#pragma unroll
  for (int i = 0; i < T; ++i) red[(wave * NQ + ADJ_NX + i) * 64 + lane] = Rb[i];
  __syncthreads();
  auto node_sum = [&](int k) {
    float v = red[k * 64 + lane];
#pragma unroll
    for (int w = 1; w < ADJ_WAVES; ++w) v += red[(w * NQ + k) * 64 + lane];
    return v;
  };
  if (wave == 0) {
    float v[ADJ_NX];
#pragma unroll
    for (int k = 0; k < ADJ_NX; ++k) v[k] = node_sum(k);
    const double AW = r.d.w;
    const double cA = (2.0 * PI * PI) * ((double)chi1 * chi1 * chi1);
    const float yy = 0.25f * v[2];                                   // d / d ln y
    const float la = r.c.x * (r.d.z * v[5]) + r.c.y * (r.d.y * v[7]) + r.c.z * v[9];  // d / d ln y of the powers
    const float mn = r.b.y * v[11] + 2.0f * r.b.z * v[12];
    double* x = xs + lane * NQ;
    // G3, AW, y and the position of the table all carry chi; y and mu / y carry R_nl
    x[0] = AW * (3.0f * (r.a.z * v[1] - v[0]) + (yy + la - mn) + A.invh * v[13]);
    x[1] = cA * v[0];
    x[2] = AW * v[1] / cA;
    x[3] = AW * LN2 * (yy + la - mn);
    x[4] = AW * v[5];
    x[5] = AW * v[7];
    x[6] = AW * LN2 * r.c.z * v[9];
    x[7] = AW * LN2 * (v[10] + cf[CF_LGCF3 * 8] * v[9]);
    x[8] = AW * v[3];
    x[9] = AW * LN2 * v[4];
    x[10] = AW * (iyc * iyc) * v[12];
    x[11] = AW * LN2 * v[6];
    x[12] = AW * LN2 * r.d.y * v[8];
    x[13] = AW * iyc * v[11];
  } else {
#pragma unroll
    for (int i = 0; i < T; ++i)
      if (i % (ADJ_WAVES - 1) == wave - 1) xs[lane * NQ + ADJ_NX + i] = 2.0 * (double)node_sum(ADJ_NX + i);
  }
  __syncthreads();
  // contraction with the stored derivatives in FP64: even threads read
  // (value, d0, d1, d2) of a field, odd threads (d3 .. d6); coalesced
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  auto add = [&](double x, const float* p) {
    const float4 d = *reinterpret_cast<const float4*>(p + (t & 1) * 4);
    s0 += x * (double)(t & 1 ? d.x : d.y);
    s1 += x * (double)(t & 1 ? d.y : d.z);
    s2 += x * (double)(t & 1 ? d.z : d.w);
    if (t & 1) s3 += x * (double)d.w;
  };
  for (int e = t >> 1; e < nn * ADJ_NX; e += 32 * ADJ_WAVES) {
    const int n = e / ADJ_NX, j = e - n * ADJ_NX;
    add(xs[n * NQ + j], A.coef + ((size_t)(A.n0 + n) * NCOEF + adj_slot(j)) * 8);
  }
  for (int e = t >> 1; e < nn * T; e += 32 * ADJ_WAVES) {
    const int n = e / T, i = e - n * T;
    add(xs[n * NQ + ADJ_NX + i], A.R + ((size_t)(A.n0 + n) * A.Tpad + i) * 8);
  }
  // T(k)'s share: the lanes' sums times their node's factor (lanes past the
  // last node repeat it)
  const double aw = lane < nn ? (double)r.d.w : 0.0;
  double o[7];
#pragma unroll
  for (int d = 0; d < 7; ++d) {
    double v = lane < nn ? aw * (double)th[d] : 0.0;
    v += d < 3 ? (t & 1 ? 0.0 : (d == 0 ? s0 : (d == 1 ? s1 : s2)))
               : (t & 1 ? (d == 3 ? s0 : (d == 4 ? s1 : (d == 5 ? s2 : s3))) : 0.0);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    o[d] = v;
  }
  if (lane == 0) {
#pragma unroll
    for (int d = 0; d < 7; ++d) wsum[wave * 8 + d] = o[d];
  }
  __syncthreads();
  if (t < 7) {
    double v = wsum[t];
#pragma unroll
    for (int w = 1; w < ADJ_WAVES; ++w) v += wsum[w * 8 + t];
    A.out[t] = (float)v;
  }
}

}  // namespace

template <int T>
__global__ __launch_bounds__(64 * ADJ_WAVES, 3) void k_adjoint(LimberArgs A) {
  extern __shared__ float4 lds4[];
  const int ngrp = adj_groups(A.Na), per = (A.Na + ngrp - 1) / ngrp;
  const int b = xcd_order(blockIdx.x, gridDim.x);
  const int c = b / ngrp, grp = b - c * ngrp;
  const int chunk = (A.n_ell + A.slices - 1) / A.slices;
  const float* cr = A.crec + (size_t)c * NCREC * 8;
  AdjIn in;
  in.coef = A.coef + (size_t)c * A.Na * NCOEF * 8;
  in.R = A.R + (size_t)c * A.Na * A.Tpad * 8;
  in.Tpad = A.Tpad;
  in.tab = A.ehtab + (size_t)c * NEHQ;
  in.dtab = reinterpret_cast<const float4*>(A.ehtab7 + (size_t)c * (NEHQ + 1) * NEHD_ROW);
  in.lo = cr[CR_EHLO * 8];
  in.invh = cr[CR_EHINVH * 8];
  in.ell = A.ell;
  in.estride = 1;
  in.cbar = A.cbar + (size_t)c * AdjShape<T>::P * A.n_ell;
  in.n_ell = A.n_ell;
  in.wl_mask = A.wl_mask;
  in.l0 = min(A.n_ell, (int)blockIdx.y * chunk);
  in.l1 = min(A.n_ell, in.l0 + chunk);
  in.n0 = grp * per;
  in.n1 = min(A.Na, in.n0 + per);
  in.out = A.theta_col + ((size_t)b * A.slices + blockIdx.y) * 7;
  adjoint_block<T>(in, lds4);
}

template <int T>
static hipError_t launch_adj_T(const LimberArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((k_adjoint<T>), dim3(a.B * adj_groups(a.Na), a.slices), dim3(64 * ADJ_WAVES),
                     AdjShape<T>::LDS * sizeof(float), s, a);
  return hipGetLastError();
}

hipError_t launch_adjoint(int T, const LimberArgs& a, hipStream_t s) {
  if (!a.ehtab || !a.ehtab7 || a.slices < 1 || a.slices > 65535 || a.B < 1 || a.Na < 1) return hipErrorInvalidValue;
  switch (T) {
    case 1: return launch_adj_T<1>(a, s);
    case 2: return launch_adj_T<2>(a, s);
    case 3: return launch_adj_T<3>(a, s);
    case 4: return launch_adj_T<4>(a, s);
    case 5: return launch_adj_T<5>(a, s);
    case 6: return launch_adj_T<6>(a, s);
    case 7: return launch_adj_T<7>(a, s);
    case 8: return launch_adj_T<8>(a, s);
    case 9: return launch_adj_T<9>(a, s);
    case 10: return launch_adj_T<10>(a, s);
    default: return hipErrorInvalidValue;
  }
}

// Served batches: one block per (request, node group, slice of its
// multipoles), the tracer count a constant of the body (a block-uniform
// switch).  The grid is sized for the capacity; blocks past the live ones exit.
__global__ __launch_bounds__(64 * ADJ_WAVES, 3) void k_ragged_adjoint(RaggedArgs A) {
  extern __shared__ float4 lds4[];
  const int ngrp = adj_groups(A.Na), per = (A.Na + ngrp - 1) / ngrp;
  const int units = *A.njobs * ngrp;
  const int nsl = adj_ragged_slices(units, A.min_slices);
  const int live = units * nsl;
  const XcdShare xs = xcd_share(blockIdx.x, live);
  const int xi = blockIdx.x >> 3;
  if (xi >= xs.count) return;
  const int b = xs.first + xi;
  const int y = b % nsl, u = b / nsl, grp = u % ngrp;
  const RJob& jb = A.jobs[u / ngrp];
  const int c = jb.c;
  // (a request takes the slices that itself asks for; its other blocks are empty)
  const int own = adj_ragged_slices(units, adj_min_slices(jb.n_ell));
  const int chunk = (jb.n_ell + own - 1) / own;
  const float* cr = A.crec + (size_t)c * NCREC * 8;
  AdjIn in;
  in.coef = A.coef + (size_t)c * A.Na * NCOEF * 8;
  in.R = A.R + (size_t)c * A.Na * A.Tpad * 8;
  in.Tpad = A.Tpad;
  in.tab = A.ehtab + (size_t)c * NEHQ;
  in.dtab = reinterpret_cast<const float4*>(A.ehtab7 + (size_t)c * (NEHQ + 1) * NEHD_ROW);
  in.lo = cr[CR_EHLO * 8];
  in.invh = cr[CR_EHINVH * 8];
  in.ell = &A.cols[jb.col0].ell;
  in.estride = sizeof(RCol) / sizeof(double);
  in.cbar = A.cbar + jb.cbar_off;
  in.n_ell = jb.n_ell;
  in.wl_mask = jb.wl_mask;
  in.l0 = min(jb.n_ell, y * chunk);
  in.l1 = min(jb.n_ell, in.l0 + chunk);
  in.n0 = grp * per;
  in.n1 = min(A.Na, in.n0 + per);
  in.out = A.theta_part + (size_t)b * 7;
  switch (__builtin_amdgcn_readfirstlane(jb.T)) {
    case 1: adjoint_block<1>(in, lds4); break;
    case 2: adjoint_block<2>(in, lds4); break;
    case 3: adjoint_block<3>(in, lds4); break;
    case 4: adjoint_block<4>(in, lds4); break;
    case 5: adjoint_block<5>(in, lds4); break;
    case 6: adjoint_block<6>(in, lds4); break;
    case 7: adjoint_block<7>(in, lds4); break;
    case 8: adjoint_block<8>(in, lds4); break;
    case 9: adjoint_block<9>(in, lds4); break;
    default: adjoint_block<10>(in, lds4); break;
  }
}

hipError_t launch_ragged_adjoint(int max_jobs, const RaggedArgs& a, hipStream_t s) {
  if (max_jobs < 1 || a.min_slices < 1 || !a.njobs || !a.ehtab || !a.ehtab7 || !a.theta_part) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_ragged_adjoint, dim3(adj_ragged_blocks(max_jobs, a.Na, a.min_slices)), dim3(64 * ADJ_WAVES),
                     AdjShape<MAXT>::LDS * sizeof(float), s, a);
  return hipGetLastError();
}

// theta[row(j)][d] = sum of request j's block partials (FP64, in order): one
// 64-thread block per request, the grid sized for the capacity; lane l adds
// the partials l / 7, l / 7 + 9, ... of parameter l % 7.
__global__ __launch_bounds__(64) void k_ragged_reduce(RaggedArgs A, double* __restrict__ theta) {
  __shared__ double part[63];
  const int j = blockIdx.x;
  if (j >= *A.njobs) return;  // uniform across the block
  const int ngrp = adj_groups(A.Na);
  const int n = ngrp * adj_ragged_slices(*A.njobs * ngrp, A.min_slices);
  const float* p = A.theta_part + (size_t)j * n * 7;
  const int t = threadIdx.x;
  if (t < 63) {
    double v = 0.0;
    for (int e = t; e < n * 7; e += 63) v += (double)p[e];
    part[t] = v;
  }
  __syncthreads();
  if (t < 7) {
    double v = part[t];
    for (int k = 1; k < 9; ++k) v += part[t + 7 * k];
    theta[A.jobs[j].out_off * 7 + t] = v;  // out_off: the request's row in the batch
  }
}

hipError_t launch_ragged_reduce(int max_jobs, const RaggedArgs& a, double* theta, hipStream_t s) {
  if (max_jobs <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ragged_reduce, dim3(max_jobs), dim3(64), 0, s, a, theta);
  return hipGetLastError();
}

}  // namespace jc
