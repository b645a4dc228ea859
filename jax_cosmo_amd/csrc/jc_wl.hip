// Weak-lensing kernels (probes.py:26-84): for each outer node m of the a-grid,
//   q_i(m) = sum_j Nw_i(m, j) clip(chi' - chi_m, 0) / clip(chi', 1),
// the per-z Simpson sum over z'_{m,j}, whose segments, offsets and weighted
// number densities are resident tables; chi' is interpolated in the
// cosmology's chi table.
//
// A block covers 64 consecutive outer nodes m (one per lane) for CT
// cosmologies; its SL waves split the 256 inner nodes j and their partial sums
// are added in LDS in a fixed order (deterministic), each wave adding its
// share of the bins.  Every resident-table element loaded for (m, j) serves CT
// cosmologies; NW = weak-lensing bins held in registers (>= the set's count).
// The last node (a = 1, z = 0) has chi = 0 and so a zero kernel; the lane of the
// node before it writes that zero.
//
// Nodes with chi_m >= 1 (all but the last ones of a fine grid; wave-uniform)
// have chi' >= chi_m >= 1 (the resident tables put no inner node nearer than its
// outer one: past the probe's zmax all of them are the outer node, with zero
// weights), so neither clip acts: f = (chi' - chi_m) / chi', and
// its derivatives are ((chi_m / chi') dchi' - dchi_m) / chi', two FMAs a
// direction, with the 1 / chi' moved to the weights.  ND = 0: 8 instructions and
// a reciprocal a point with 5 bins; bound by the resident tables' path through
// the L2 where few cosmologies share them, by VALU issue beyond (with every
// table read an L1 hit, 49 of 59 us at 1024 cosmologies).  ND = 7: 66
// instructions, bound by VALU issue.  Measured at n_z 512, 5 bins, before and
// after: 10 -> 8 us at 1 cosmology, 74 -> 59 at 1024, 235 -> 179 at 2048 with n_z
// 1024; with 7 directions 36 -> 14 us at 1 and 124 -> 75 at 256.
#include <algorithm>

#include "jc_math.hpp"
#include "jc_kernels.hpp"

namespace jc {

namespace {

// raw buffer loads: the table bases and the bin row offsets stay in SGPRs, so
// one 32-bit byte offset per lane serves all of a node's loads (no 64-bit
// address arithmetic in the loop); loads past a table's end read zero
JC_D __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
JC_D float buf_f32(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

constexpr int WL_M = 64;  // outer nodes per block

// A cosmology's chi table in LDS, [2][W] floats a segment (chi and slope, each
// a value and its derivatives): float2 or float4 rows, and with 7 directions
// four planes of float4, so that the neighbouring segments that the lanes read
// lie next to each other (64-byte rows took four times the LDS cycles).
template <int ND>
JC_D void load_seg(const float* tab, int L, float* chi, float* sl) {
  if constexpr (ND == 0) {
    const float2 v = reinterpret_cast<const float2*>(tab)[L];
    chi[0] = v.x;
    sl[0] = v.y;
  } else if constexpr (ND == 1) {
    const float4 v = reinterpret_cast<const float4*>(tab)[L];
    chi[0] = v.x;
    chi[1] = v.y;
    sl[0] = v.z;
    sl[1] = v.w;
  } else {
    static_assert(ND == 7, "");
    const float4* t = reinterpret_cast<const float4*>(tab) + L;
    const float4 a = t[0], b = t[NCHI], c = t[2 * NCHI], d = t[3 * NCHI];
    chi[0] = a.x; chi[1] = a.y; chi[2] = a.z; chi[3] = a.w;
    chi[4] = b.x; chi[5] = b.y; chi[6] = b.z; chi[7] = b.w;
    sl[0] = c.x; sl[1] = c.y; sl[2] = c.z; sl[3] = c.w;
    sl[4] = d.x; sl[5] = d.y; sl[6] = d.z; sl[7] = d.w;
  }
}

}  // namespace

template <int ND, int CT, int NW, int SL>
__device__ __forceinline__ void wl_block(const WLArgs& A) {
  using Sf = typename Types<ND>::F;
  constexpr int W = ND + 1;
  constexpr int TS = NCHI * 2 * W;                  // floats of a cosmology's table
  extern __shared__ __align__(16) float wl_smem[];  // [CT] tables, then [SL][NW][W][64] partial sums
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = blockIdx.x * WL_M + lane;
  const int c0 = blockIdx.y * CT;
  const int B = A.dB ? min(*A.dB, A.B) : A.B;
  if (c0 >= B) return;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int c = c0 + ct < B ? c0 + ct : B - 1;
    const float4* src = reinterpret_cast<const float4*>(A.chitab + (size_t)c * TS);
    float4* dst = reinterpret_cast<float4*>(wl_smem + ct * TS);
    for (int e = tid; e < TS / 4; e += WL_M * SL) dst[ND == 7 ? (e & 3) * NCHI + (e >> 2) : e] = src[e];
  }
  __syncthreads();
  const int N = A.Na - 1;  // nodes with a nonzero kernel
  const bool active = m < N;
  const int mm = active ? m : N - 1;
  Sf chim[CT];
  float acc[CT][NW][W];
  bool far = true;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int c = c0 + ct < B ? c0 + ct : B - 1;
    chim[ct] = Mem<Sf>::ld(A.coef + (((size_t)c * A.Na + mm) * NCOEF + CF_CHI) * W);
    far = far && val(chim[ct]) >= 1.0f;
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int d = 0; d < W; ++d) acc[ct][i][d] = 0.0f;
  }
  // j = 0 is z' = z, where chi' == chi and the integrand is exactly zero
  constexpr int JS = (NWL_J - 1) / SL;
  const int j0 = 1 + wave * JS;
  const int rs = NWL_J * A.Na;  // elements per table row block (and per bin of the weights)
  const __amdgpu_buffer_rsrc_t rL = buf_rsrc(A.Lidx, rs);
  const __amdgpu_buffer_rsrc_t rD = buf_rsrc(A.delta, rs * 4);
  const __amdgpu_buffer_rsrc_t rN = buf_rsrc(A.Nw, rs * 4 * NW);
  int oL = j0 * A.Na + mm;
  // clip(chi' - chi, 0) / clip(chi', 1) with both clips (probes.py:51); that of
  // chi' itself (background.py:242) cannot change it, since chi >= 0
  auto clipped = [&](int ct, int L, float dl) {
    float x[W], s[W];
    load_seg<ND>(wl_smem + ct * TS, L, x, s);
    Sf chip = Mem<Sf>::ld(x) + Mem<Sf>::ld(s) * dl;
    return maxc(chip - chim[ct], 0.0f) * jm::rcp(maxc(chip, 1.0f));
  };
  if (__all(far)) {
    // the next node's table elements are in flight while this one's are used
    // (deeper prefetches were slower)
    int L, Ln;
    float dl, dln, nw[NW], nwn[NW];
    auto fetch = [&](int& l, float& d, float* n) {
      l = __builtin_amdgcn_raw_buffer_load_b8(rL, oL, 0, 0);
      d = buf_f32(rD, 4 * oL, 0);
#pragma unroll
      for (int i = 0; i < NW; ++i) n[i] = buf_f32(rN, 4 * oL, 4 * i * rs);  // zero rows past nw
      oL += A.Na;
    };
    fetch(Ln, dln, nwn);
#pragma unroll 1
    for (int j = 0; j < JS; ++j) {
      L = Ln;
      dl = dln;
#pragma unroll
      for (int i = 0; i < NW; ++i) nw[i] = nwn[i];
      if (j + 1 < JS) fetch(Ln, dln, nwn);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float x[W], s[W];
        load_seg<ND>(wl_smem + ct * TS, L, x, s);
        const float chip = __builtin_fmaf(s[0], dl, x[0]);
        const float r = __builtin_amdgcn_rcpf(chip);
        const float f = (chip - val(chim[ct])) * r;
        // bins past the set's count carry nw = 0 and f is finite: no guard
#pragma unroll
        for (int i = 0; i < NW; ++i) acc[ct][i][0] = __builtin_fmaf(nw[i], f, acc[ct][i][0]);
        if constexpr (ND > 0) {
          const float q = val(chim[ct]) * r;
          float df[ND];
#pragma unroll
          for (int d = 0; d < ND; ++d)
            df[d] = __builtin_fmaf(__builtin_fmaf(s[1 + d], dl, x[1 + d]), q, -chim[ct].d[d]);
#pragma unroll
          for (int i = 0; i < NW; ++i) {
            const float w = nw[i] * r;
#pragma unroll
            for (int d = 0; d < ND; ++d) acc[ct][i][1 + d] = __builtin_fmaf(w, df[d], acc[ct][i][1 + d]);
          }
        }
      }
    }
  } else {
    for (int j = 0; j < JS; ++j, oL += A.Na) {
      const int L = __builtin_amdgcn_raw_buffer_load_b8(rL, oL, 0, 0);
      const float dl = buf_f32(rD, 4 * oL, 0);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const Sf f = clipped(ct, L, dl);
#pragma unroll
        for (int i = 0; i < NW; ++i)
          Mem<Sf>::st(acc[ct][i], Mem<Sf>::ld(acc[ct][i]) + buf_f32(rN, 4 * oL, 4 * i * rs) * f);
      }
    }
  }
  // single source planes (probes.py:53-64): clip(chi_s - chi, 0) / clip(chi_s, 1)
  if (wave == 0) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (i < A.nw) {
        const WLSource sp = A.src[i];
        if (sp.on) {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            Mem<Sf>::st(acc[ct][i], Mem<Sf>::ld(acc[ct][i]) + sp.fac * clipped(ct, sp.L, sp.off));
        }
      }
    }
  }
  // the waves' sums, one cosmology after the other (the tables' space is
  // reused): wave w adds bins w, w + SL, ... in wave order and stores them
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int d = 0; d < W; ++d) wl_smem[((wave * NW + i) * W + d) * 64 + lane] = acc[ct][i][d];
    __syncthreads();
    const int c = c0 + ct;
    if (c >= B) return;
    const Sf pref = (A.zp1[mm] * chim[ct]) * Mem<Sf>::ld(A.crec + ((size_t)c * NCREC + CR_WLCONST) * W);
    for (int i = wave; i < A.nw; i += SL) {
      Sf r = Mem<Sf>::ld(&wl_smem[(i * W) * 64 + lane], 64);
#pragma unroll
      for (int w = 1; w < SL; ++w) r = r + Mem<Sf>::ld(&wl_smem[((w * NW + i) * W) * 64 + lane], 64);
      r = r * pref;
      // R columns of the bin: the pool column, or (served batches) every
      // position of the request that selects the bin; all MAXT positions are
      // tested so that the loads issue together
      const int cl = A.col[i];
      uint32_t mk = 0;
      if (A.rjobs) {
        const RJob& jb = A.rjobs[c];
#pragma unroll
        for (int p = 0; p < MAXT; ++p) mk |= (p < jb.T && jb.sel[p] == cl ? 1u : 0u) << p;
      } else {
        mk = 1u << cl;
      }
      if (!active) continue;
      for (; mk; mk &= mk - 1) {
        float* dst = A.R + (((size_t)c * A.Na + m) * A.Tpad + __builtin_ctz(mk)) * W;
        Sf v = r;
        if (A.ia) v = v + Mem<Sf>::ld(dst);  // the NLA term written by the table kernel
        Mem<Sf>::st(dst, v);
        // the a = 1 node: zero lensing kernel (chi = 0), the NLA term stays
        if (m == N - 1 && !A.ia) Mem<Sf>::st(dst + (size_t)A.Tpad * W, Make<Sf>::c(0.0));
      }
    }
  }
}

template <int ND, int CT, int NW, int SL>
__global__ __launch_bounds__(WL_M * SL) void k_wl(WLArgs A) {
  wl_block<ND, CT, NW, SL>(A);
}

// Served batches: the grid is made for a full batch, the number of cosmologies
// is on the device.  CT of them share a block in a full batch; below `few` of
// them, which would leave most of the chip idle, two do, and 8 waves
// split the inner nodes (three branches of 50 cosmologies side by side: 40 -> 21 us
// each).
template <int CT, int NW, int SL>
__global__ __launch_bounds__(WL_M * SL) void k_wl_live(WLArgs A, int few) {
  if (*A.dB <= few) wl_block<0, 2, NW, SL>(A);
  else wl_block<0, CT, NW, SL>(A);
}

template <int ND, int CT, int NW, int SL>
static hipError_t wl_launch(const WLArgs& a, int num_cu, hipStream_t s) {
  constexpr int W = ND + 1;
  constexpr size_t sm = std::max((size_t)CT * NCHI * 2 * W, (size_t)SL * NW * W * 64) * sizeof(float);
  static_assert(sm <= 160 * 1024, "LDS of a block");
  const int nb = (a.Na - 1 + WL_M - 1) / WL_M;
  if constexpr (ND == 0 && CT > 2) {
    if (a.dB) {
      // two a block up to 4 blocks of one cosmology per CU (the rule below)
      const int few = std::min(4 * num_cu / nb, a.B);
      const dim3 grid(nb, std::max((few + 1) / 2, (a.B + CT - 1) / CT));
      hipLaunchKernelGGL((k_wl_live<CT, NW, SL>), grid, dim3(WL_M * SL), sm, s, a, few);
      return hipGetLastError();
    }
  }
  const dim3 grid(nb, (a.B + CT - 1) / CT);
  hipLaunchKernelGGL((k_wl<ND, CT, NW, SL>), grid, dim3(WL_M * SL), sm, s, a);
  return hipGetLastError();
}

// Launch shape.  What a wave reads of the resident tables (25 bytes a point)
// comes through the L2 at about 14 TB/s, so the more cosmologies share it the
// better, as long as the blocks still fill the chip; with few blocks 8 waves
// split the inner nodes.  Measured on 256 CUs, n_z 512 (8 node blocks), 5 bins,
// us for 1 / 2 / 4 / 8 cosmologies a block: 8.3 / 8.8 / 10.5 / 17 at 1
// cosmology, 17 / 11.3 / 13.5 / 22 at 64, 50 / 31 / 22 / 26 at 256, 93 / 55 / 37 /
// 38 at 512, 177 / 100 / 66 / 59 at 1024.  A batch of 520 takes 204 us
// with 4 and 208 with 8, one of 700 235 and 232.  Seven directions, (1, 8 waves) / (1, 4)
// / (2, 4): 14 / 23 / 30 at 1, 26 / 31 / 35 at 64, 44 / 44 / 45 at 128, 80 / 78 / 75
// at 256, 312 / 289 / 258 at 1024.  ctile (ND = 0): 0 = by this rule.
template <int NW>
static hipError_t wl_launch_nw(int nd, int ctile, const WLArgs& a, int num_cu, hipStream_t s) {
  const int64_t blocks = (int64_t)((a.Na - 1 + WL_M - 1) / WL_M) * a.B;  // at one cosmology each
  if (nd == 0) {
    if (ctile == 0) ctile = blocks <= num_cu ? 1 : (blocks <= 2 * num_cu ? 2 : (blocks <= 20 * num_cu ? 4 : 8));
    switch (ctile) {
      case 1: return wl_launch<0, 1, NW, 8>(a, num_cu, s);
      case 2: return wl_launch<0, 2, NW, 8>(a, num_cu, s);
      case 4: return wl_launch<0, 4, NW, 8>(a, num_cu, s);
      case 8: return a.dB ? wl_launch<0, 8, NW, 8>(a, num_cu, s) : wl_launch<0, 8, NW, 4>(a, num_cu, s);
      case 16: return wl_launch<0, 16, NW, 4>(a, num_cu, s);
      default: return hipErrorInvalidValue;
    }
  }
  if (nd == 1) return blocks <= num_cu ? wl_launch<1, 1, NW, 8>(a, num_cu, s) : wl_launch<1, 1, NW, 4>(a, num_cu, s);
  if (nd != 7) return hipErrorInvalidValue;
  if constexpr (NW <= 5) {  // (with 10 bins the partial sums of 8 waves would not fit the LDS)
    if (blocks <= 2 * num_cu) return wl_launch<7, 1, NW, 8>(a, num_cu, s);
  }
  return blocks <= 4 * num_cu ? wl_launch<7, 1, NW, 4>(a, num_cu, s) : wl_launch<7, 2, NW, 4>(a, num_cu, s);
}

hipError_t launch_wl(int nd, int ctile, const WLArgs& a, int num_cu, hipStream_t s) {
  if (a.nw < 1 || a.nw > NWL_MAX || a.Na < 2) return hipErrorInvalidValue;
  return a.nw <= 5 ? wl_launch_nw<5>(nd, ctile, a, num_cu, s) : wl_launch_nw<NWL_MAX>(nd, ctile, a, num_cu, s);
}

}  // namespace jc
