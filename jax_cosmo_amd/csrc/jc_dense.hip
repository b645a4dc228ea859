// Dense Gaussian likelihood algebra on the device (likelihood.py:43-61, the
// covariance as one N x N matrix, N = pairs x ell: 5500 for 10 tracers and
// 100 ell).  FP64 throughout, row-major N x N (numpy's layout; the matrix is
// symmetric, so rows and columns are interchangeable on input).  All products
// run on the FP64 matrix cores (v_mfma_f64_16x16x4): a lane holds 4 consecutive
// k of one row, so operands whose k is contiguous in memory come straight from
// global memory as whole 128-byte segments, without LDS.
//
// Cholesky C = L L^T, right-looking in 64-column panels, two launches a panel:
//   k_chol_panel  the panel below its 64 x 64 diagonal block, L21 = A21 L11^-T,
//                 as a product with the block's inverse and one correction;
//   k_chol_syrk   the trailing lower triangle, A22 -= L21 L21^T, 64 x 64 tiles;
//                 its first block then factors and inverts the next panel's
//                 diagonal block (chol64) beside the other tiles.
// Triangular solves for B right-hand sides stored as rows ([B][N]), in
// 512-row blocks whose triangles are inverted first, all at once
// (k_tri_inv64, k_tri_merge): per block one product with its inverse
// (k_solve_diag) and one that removes it from the remaining rows
// (k_solve_update).
// The likelihood of a batch of means: r = data - mu, z = L^-1 r,
// -1/2 |z|^2 + c0 per mean (fixed-order sums), and its derivative with
// respect to the mean, C^-1 r = L^-T z, the adjoint's cotangent.
#include <algorithm>

#include "jc_kernels.hpp"
#include "jc_mma64.hpp"

namespace jc {

constexpr int DB = 64;              // panel width and tile size
constexpr int SB = DENSE_SOLVE_BLOCK;  // rows a solve step takes

typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// (Kernels here ask for 2 waves per SIMD: with a budget above 256 registers the
// compiler keeps accumulators in the accumulation file and copies them in and
// out of every product's loop.)
// Operands of 16 k: lane l takes k = 4 (l / 16) .. + 3 of row l % 16 (element q
// of both operands in one instruction, so any assignment of k to lanes serves).
// row: p[0 .. n) along k, n valid elements from the lane's first (n >= 4: all).
__device__ __forceinline__ d4 frag_row(const double* p, int n) {
  d4 v = {0.0, 0.0, 0.0, 0.0};
  if (n >= 4) {
    const d2u a = *reinterpret_cast<const d2u*>(p), b = *reinterpret_cast<const d2u*>(p + 2);
    v[0] = a[0];
    v[1] = a[1];
    v[2] = b[0];
    v[3] = b[1];
  } else {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q < n) v[q] = p[q];
  }
  return v;
}
// column: the elements are ld apart
__device__ __forceinline__ d4 frag_col(const double* p, size_t ld, int n) {
  d4 v = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (q < n) v[q] = p[q * ld];
  return v;
}
// n steps of 16 k with the operands of the next D in flight (a load from L
// outside the L2 takes longer than a step's products): load(s, q) fills slot q
// with step s, use(q) consumes it.  n is uniform over the wave.
template <int D, class Load, class Use>
__device__ __forceinline__ void pipelined(int n, Load&& load, Use&& use) {
#pragma unroll
  for (int q = 0; q < D; ++q)
    if (q < n) load(q, q);
  for (int s = 0; s < n; s += D) {
#pragma unroll
    for (int q = 0; q < D; ++q) {
      if (s + q < n) {
        use(q);
        if (s + q + D < n) load(s + q + D, q);
      }
    }
  }
}

// ------------------------------------------------------------------ Cholesky
constexpr int LS = DB + 2;  // LDS row stride of a 64 x 64 block

__device__ __forceinline__ double lane_d(double x, int src) {  // src uniform
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, src);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), src);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// 16 x 16 block product from LDS: acc += A B^T (NT: rows of B) or A B
template <bool NT>
__device__ __forceinline__ void lds_mma(const double* A, const double* B, int lane, d4& acc) {
  const int i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = 4 * q + g;
    acc = mfma64(A[i * LS + k], NT ? B[i * LS + k] : B[k * LS + i], acc);
  }
}
__device__ __forceinline__ void lds_put(double* D, int lane, const d4& v) {
#pragma unroll
  for (int r = 0; r < 4; ++r) D[((lane >> 4) + 4 * r) * LS + (lane & 15)] = v[r];
}

// sqrt(d) and its reciprocal for normal d > 0, by Newton from v_rsq_f64
__device__ __forceinline__ double sqrt_rsqrt(double d, double& r) {
  double y = __builtin_amdgcn_rsq(d);
  y = __builtin_fma(0.5 * y, __builtin_fma(-d * y, y, 1.0), y);
  y = __builtin_fma(0.5 * y, __builtin_fma(-d * y, y, 1.0), y);
  r = y;
  const double s = d * y;
  return __builtin_fma(0.5 * y, __builtin_fma(-s, s, d), s);
}

// V (lower triangle by 16 x 16 blocks) = the inverse of the lower triangular
// 64 x 64 block in S, by the 256 threads of a block, from the inverses of its
// 16 x 16 diagonal blocks, which the caller has put into V:
// V21 = -V22 (S21 V11), 16 and 32 wide.
__device__ void tri64_merge(const double* S, double* V) {
  double* Tm = V + 32;  // rows 0-31, columns 32-63: above the inverse's diagonal, not part of it
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  const d4 zero = {0.0, 0.0, 0.0, 0.0};
  if (wave < 2) {
    const int o = 32 * wave;
    d4 v = zero;
    lds_mma<false>(S + (o + 16) * LS + o, V + o * LS + o, lane, v);
    lds_put(Tm + 16 * wave * LS, lane, v);
  }
  __syncthreads();
  if (wave < 2) {
    const int o = 32 * wave;
    d4 v = zero;
    lds_mma<false>(V + (o + 16) * LS + o + 16, Tm + 16 * wave * LS, lane, v);
    lds_put(V + (o + 16) * LS + o, lane, -v);
  }
  __syncthreads();
  // 32 wide: the blocks above V's diagonal inside its halves are not stored
  const int ra = 16 * (wave >> 1), cb = 16 * (wave & 1);
  d4 t = zero;
  for (int c = cb; c < 32; c += 16) lds_mma<false>(S + (32 + ra) * LS + c, V + c * LS + cb, lane, t);
  __syncthreads();  // the 16-wide Tm has been read
  lds_put(Tm + ra * LS + cb, lane, t);
  __syncthreads();
  t = zero;
  for (int c = 0; c <= ra; c += 16) lds_mma<false>(V + (32 + ra) * LS + 32 + c, Tm + c * LS + cb, lane, t);
  lds_put(V + (32 + ra) * LS + cb, lane, -t);
  __syncthreads();
}

// The inverse of the lower triangular 16 x 16 block L by one wave: lane i solves
// x L^T = e_i by columns: a step chains a product and an FMA (by rows it was a dot
// product, 2.9 us a block).
__device__ __forceinline__ void tri16_inverse(const double* L, double* V) {
  const int lane = threadIdx.x & 63, i = lane & 15;
  const double rd = 1.0 / L[i * LS + i];
  double a[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) a[c] = i == c ? 1.0 : 0.0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    a[j] *= lane_d(rd, j);
#pragma unroll
    for (int c = j + 1; c < 16; ++c) a[c] -= a[j] * L[c * LS + j];
  }
  if (lane < 16) {
#pragma unroll
    for (int j = 0; j < 16; ++j) V[j * LS + i] = a[j];
  }
}

// The same as tri64_merge with nothing in V: wave w inverts its 16 x 16 diagonal
// block first.
__device__ void tri64_inverse(const double* S, double* V) {
  const int o = 16 * (threadIdx.x >> 6);
  tri16_inverse(S + o * LS + o, V + o * LS + o);
  tri64_merge(S, V);
}

// chol64's step of 16 columns down `rows` rows of D for any pivots, by one wave in
// LDS: zero, negative and undefined ones (reported), those next to the ends of the
// range, and infinity (a datum of infinite variance: its column of the factor is zero
// but for the diagonal).
__device__ void chol16_any(double* D, int rows, double* V, int* bad) {
  const int lane = threadIdx.x & 63;
  double* r = D + min(lane, rows - 1) * LS;
  auto fence = [] {  // (the wave's LDS operations complete in order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  for (int j = 0; j < 16; ++j) {
    double d = D[j * LS + j];
    if (!(d > 0.0)) {
      d = 1.0;
      if (lane == 0) *bad = 1;
    }
    d = ::sqrt(d);
    const double id = 1.0 / d;
    fence();
    if (lane < rows) r[j] = lane < j ? 0.0 : (lane == j ? d : r[j] * id);
    fence();
    for (int c = j + 1; c < 16; ++c)
      if (lane >= c && lane < rows) r[c] -= r[j] * D[c * LS + j];
    fence();
  }
  tri16_inverse(D, V);
}

// Factors the 64 x 64 block in S (lower triangle; identity past nb) in place
// and leaves the inverse of its factor in the lower triangle (by 16 x 16
// blocks) of V, by the 256 threads of a block.  16 columns at a time: wave 0
// factors them down all rows of the block (row o + i in lane i, so the rows
// below the diagonal come with it; pivots and multipliers by readlane, no
// barrier), then all waves update the rest as 16 x 16 products.  Beside it wave 1
// does the same with 16 rows of the identity below the diagonal block, which
// become its inverse (by substitution afterwards: 3 us more).  One block in LDS 16
// us, 2.4 of them a panel (2.7 as L D L^T with the square roots at the end); with
// barriers between 64 pivots 97 us.
__device__ void chol64(double* S, double* V, int nb, double* dlog, int* bad) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();  // the caller has written S
  auto update = [&](int jb) {  // the rows and columns past block column jb
    const int o = 16 * jb;
    int t = 0;
    for (int ib = jb + 1; ib < 4; ++ib)
      for (int kb = jb + 1; kb <= ib; ++kb, ++t) {
        if ((t & 3) != wave) continue;
        d4 v = {0.0, 0.0, 0.0, 0.0};
        lds_mma<true>(S + 16 * ib * LS + o, S + 16 * kb * LS + o, lane, v);
        double* D = S + 16 * ib * LS + 16 * kb;
#pragma unroll
        for (int r = 0; r < 4; ++r) D[((lane >> 4) + 4 * r) * LS + (lane & 15)] -= v[r];
      }
  };
  // A pivot is a difference of its diagonal element and squares: with the elements
  // in this range it is normal and finite, or not positive.  (Uniform over the block.)
  const double dd = S[lane * (LS + 1)];
  if (!__all(dd >= 0x1p-900 && dd <= 0x1p1020)) {
    for (int jb = 0; jb < 4; ++jb) {
      const int o = 16 * jb;
      __syncthreads();  // every wave has read dd, or updated
      if (wave == 0) chol16_any(S + o * (LS + 1), DB - o, V + o * (LS + 1), bad);
      __syncthreads();
      update(jb);
    }
    __syncthreads();
  } else {
    for (int jb = 0; jb < 4; ++jb) {
      const int o = 16 * jb;
      const int r0 = wave == 0 ? min(o + lane, DB - 1) : o + (lane & 15);
      double* row = S + r0 * LS + o;
      double a[16];
      if (wave < 2) {
#pragma unroll
        for (int c = 0; c < 16; ++c) a[c] = wave == 1 && lane >= 16 ? (lane - 16 == c ? 1.0 : 0.0) : row[c];
      }
      __syncthreads();  // wave 1 has read the block that wave 0 will overwrite
      if (wave < 2) {
        bool ok = true;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const double p = lane_d(a[j], j);
          ok = ok && p > 0.0;
          const double d = p > 0.0 ? p : 1.0;  // keeps the rest finite; the caller reports the failure
          double r;
          const double q = sqrt_rsqrt(d, r);
          a[j] = lane == j ? q : a[j] * r;
#pragma unroll
          for (int c = j + 1; c < 16; ++c) a[c] -= a[j] * lane_d(a[j], c);
        }
        if (wave == 0) {
          if (o + lane < DB) {
#pragma unroll
            for (int c = 0; c < 16; ++c) row[c] = lane >= c ? a[c] : 0.0;
          }
          if (!ok && lane == 0) *bad = 1;
        } else if (lane >= 16 && lane < 32) {
#pragma unroll
          for (int j = 0; j < 16; ++j) V[(o + j) * LS + o + lane - 16] = a[j];
        }
      }
      __syncthreads();
      update(jb);
      __syncthreads();
    }
  }
  if (wave == 3 && lane < nb) dlog[lane] = ::log(S[lane * LS + lane]);
  tri64_merge(S, V);
}

// the diagonal block in S (written by the caller) -> factor in A, inverse in inv
__device__ __forceinline__ void chol64_store(double* A, int64_t N, int64_t k0, double* S, double* V, double* inv,
                                             double* dlog, int* bad) {
  const int nb = (int)min((int64_t)DB, N - k0);
  chol64(S, V, nb, dlog + k0, bad);
  for (int e = threadIdx.x; e < DB * DB; e += 256) {
    const int i = e / DB, j = e - i * DB;
    if (j <= i && i < nb) A[(size_t)(k0 + i) * N + k0 + j] = S[i * LS + j];
    inv[e] = V[i * LS + j];
  }
}

__global__ __launch_bounds__(256, 2) void k_chol_first(double* __restrict__ A, int64_t N, double* __restrict__ inv,
                                                     double* __restrict__ dlog, int* __restrict__ bad) {
  __shared__ double S[DB * LS], V[DB * LS];
  const int nb = (int)min((int64_t)DB, N);
  if (threadIdx.x == 0) *bad = 0;  // (the thread that sets it)
  for (int e = threadIdx.x; e < DB * DB; e += 256) {
    const int i = e / DB, j = e - i * DB;
    S[i * LS + j] = i < nb && j <= i ? A[(size_t)i * N + j] : (i == j ? 1.0 : 0.0);
  }
  chol64_store(A, N, 0, S, V, inv, dlog, bad);
}

// rows i >= k0 + 64: x = a L11^-T, 16 rows a wave (which reads its rows' 64
// columns before it writes them).  The product with the block's inverse alone has a
// residual that grows with the block's condition number and goes into every
// later panel (covariances of condition 1e12 met non-positive pivots); one
// correction, x += (a - x L11^T) L11^-T, brings it back to that of a substitution.
// Products are taken transposed, with the rows of L11 dealt to the operand's lanes
// so that a result comes back as the 4 consecutive columns per lane in which it is
// used and stored.  Average over the panels of N = 2750: 7.3 us without the
// correction, 8.3 with it.
__global__ __launch_bounds__(256, 2) void k_chol_panel(double* __restrict__ A, int64_t N, int64_t k0,
                                                     const double* __restrict__ inv) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int64_t r0 = k0 + DB + ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  if (r0 >= N) return;
  const int p = 4 * (i & 3) + (i >> 2);  // result (g, r) is then row 4 g + r of a 16 x 16 block
  double* const row = A + (size_t)min(r0 + i, N - 1) * N + k0 + 4 * g;
  // everything is in flight at once: blocks (c, s), s <= c, of the inverse and of L11
  d4 a[4], x[4], v[10], l[10];
#pragma unroll
  for (int s = 0; s < 4; ++s) a[s] = frag_row(row + 16 * s, 4);
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int s = 0; s <= c; ++s) {
      v[c * (c + 1) / 2 + s] = frag_row(inv + (16 * c + p) * DB + 16 * s + 4 * g, 4);
      l[c * (c + 1) / 2 + s] = frag_row(A + (size_t)(k0 + 16 * c + p) * N + k0 + 16 * s + 4 * g, 4);
    }
  auto lower = [&](const d4* m, const d4* b, int c) {
    d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s <= c; ++s) mma16(m[c * (c + 1) / 2 + s], b[s], acc);
    return acc;
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) x[c] = lower(v, a, c);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // above L11's diagonal lies whatever the caller had
      const double e = l[c * (c + 3) / 2][q];
      l[c * (c + 3) / 2][q] = 4 * g + q > p ? 0.0 : fmin(e, 0x1p1023);  // (an infinite L_jj has x_j = 0)
    }
    a[c] -= lower(l, x, c);  // the residual
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) x[c] += lower(v, a, c);
  if (r0 + i >= N) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    *reinterpret_cast<d2u*>(row + 16 * c) = d2u{x[c][0], x[c][1]};
    *reinterpret_cast<d2u*>(row + 16 * c + 2) = d2u{x[c][2], x[c][3]};
  }
}

// trailing update of the lower triangle from row/column r0 = k0 + 64: tile
// (ti, tj), tj <= ti, of 64 x 64, 32 x 32 a wave; block 0 (the next panel's
// diagonal block) goes on to factor it
__global__ __launch_bounds__(256, 2) void k_chol_syrk(double* __restrict__ A, int64_t N, int64_t k0,
                                                    double* __restrict__ inv, double* __restrict__ dlog,
                                                    int* __restrict__ bad) {
  __shared__ double S[DB * LS], V[DB * LS];
  const int64_t r0 = k0 + DB;
  const int64_t idx = blockIdx.x;
  int64_t ti = (int64_t)((sqrt(8.0 * (double)idx + 1.0) - 1.0) * 0.5);
  while (ti * (ti + 1) / 2 > idx) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= idx) ++ti;
  const int64_t tj = idx - ti * (ti + 1) / 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  const int64_t ri = r0 + ti * DB + 32 * (wave >> 1), rj = r0 + tj * DB + 32 * (wave & 1);
  d4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  const double* pa[2];
  const double* pb[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    pa[a] = A + (size_t)min(ri + 16 * a + i, N - 1) * N + k0 + 4 * g;
    pb[a] = A + (size_t)min(rj + 16 * a + i, N - 1) * N + k0 + 4 * g;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const d4 a0 = frag_row(pa[0] + 16 * s, 4), a1 = frag_row(pa[1] + 16 * s, 4);
    const d4 b0 = frag_row(pb[0] + 16 * s, 4), b1 = frag_row(pb[1] + 16 * s, 4);
    mma16(a0, b0, acc[0][0]);
    mma16(a0, b1, acc[0][1]);
    mma16(a1, b0, acc[1][0]);
    mma16(a1, b1, acc[1][1]);
  }
  const int nb = (int)min((int64_t)DB, N - r0);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = ri + 16 * a + g + 4 * r, col = rj + 16 * b + i;
        if (idx == 0) {
          const int x = (int)(row - r0), y = (int)(col - r0);
          S[x * LS + y] = x < nb && y <= x ? A[(size_t)row * N + col] - acc[a][b][r] : (x == y ? 1.0 : 0.0);
        } else if (col <= row && row < N) {
          A[(size_t)row * N + col] -= acc[a][b][r];
        }
      }
  if (idx != 0) return;  // uniform over the block
  chol64_store(A, N, r0, S, V, inv, dlog, bad);
}

// the strict upper triangle of the factor is zeroed at the end
__global__ void k_zero_upper(double* __restrict__ A, int64_t N) {
  const int64_t row = blockIdx.y;
  for (int64_t c = row + 1 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < N; c += (int64_t)gridDim.x * blockDim.x)
    A[(size_t)row * N + c] = 0.0;
}

// ------------------------------------------------------------------ triangular solves
// Inverses of the SB x SB diagonal blocks of L, one block after another in
// inv ([ceil(N / SB)][SB][SB], row-major; rows past N count as identity; the
// 64 x 64 sub-blocks above the diagonal are not written).  The forward error
// of a solve by products with the triangles' inverses has the bound of
// substitution, |L^-1| |L| |x| (its residual has not: a factorisation corrects for
// that, k_chol_panel), and the 64 divisions and broadcasts a substitution chains
// per block are gone.
// k_tri_inv64: the 64 x 64 diagonal blocks.
__global__ __launch_bounds__(256, 2) void k_tri_inv64(const double* __restrict__ L, int64_t N, double* __restrict__ inv) {
  __shared__ double S[DB * LS], V[DB * LS];
  const int64_t k0 = (int64_t)blockIdx.x * DB;
  for (int e = threadIdx.x; e < DB * DB; e += 256) {
    const int r = e / DB, c = e - r * DB;
    S[r * LS + c] = k0 + r < N && c <= r ? L[(size_t)(k0 + r) * N + k0 + c] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  tri64_inverse(S, V);
  double* o = inv + (size_t)(blockIdx.x / (SB / DB)) * SB * SB + (size_t)(blockIdx.x % (SB / DB)) * DB * (SB + 1);
  for (int e = threadIdx.x; e < DB * DB; e += 256) {
    const int r = e / DB, c = e - r * DB;
    o[(size_t)r * SB + c] = c / 16 <= r / 16 ? V[r * LS + c] : 0.0;
  }
}

// k_tri_merge: two inverted neighbours of H rows to one of 2 H:
// inv21 = -inv22 (L21 inv11), 16 NC columns per block (grid y), 16 rows a wave.
template <int H, int NC>
__global__ __launch_bounds__(4 * H, H < 256 ? 2 : 4) void k_tri_merge(const double* __restrict__ L, int64_t N,
                                                                      double* __restrict__ inv) {
  constexpr int MS = 16 * NC + 2;  // LDS row stride of the product
  __shared__ double tm[H * MS];
  constexpr int per = SB / (2 * H);
  const int64_t k0 = (int64_t)blockIdx.x * 2 * H;
  double* V = inv + (size_t)(blockIdx.x / per) * SB * SB + (size_t)(blockIdx.x % per) * 2 * H * (SB + 1);
  const int j0 = blockIdx.y * 16 * NC;
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int w0 = 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t lrow = k0 + H + w0 + i;  // rows past N: zero (their columns lie below N)
  d4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = d4{0.0, 0.0, 0.0, 0.0};
  constexpr int D = 4;
  d4 x[D], v[D][NC];
  pipelined<D>((H - j0) / 16, [&](int s, int q) {  // inv11 has no rows above its column
    const int k = j0 + 16 * s + 4 * g;
    x[q] = lrow < N ? frag_row(L + (size_t)lrow * N + k0 + k, 4) : d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < NC; ++c) v[q][c] = frag_col(V + (size_t)k * SB + j0 + 16 * c + i, SB, 4);
  }, [&](int q) {
#pragma unroll
    for (int c = 0; c < NC; ++c) mma16(x[q], v[q][c], acc[c]);
  });
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) tm[(w0 + g + 4 * r) * MS + 16 * c + i] = acc[c][r];
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = d4{0.0, 0.0, 0.0, 0.0};
  pipelined<D>(w0 / 16 + 1, [&](int s, int q) {
    x[q] = frag_row(V + (size_t)(H + w0 + i) * SB + H + 16 * s + 4 * g, 4);
#pragma unroll
    for (int c = 0; c < NC; ++c) v[q][c] = frag_col(tm + (16 * s + 4 * g) * MS + 16 * c + i, MS, 4);
  }, [&](int q) {
#pragma unroll
    for (int c = 0; c < NC; ++c) mma16(x[q], v[q][c], acc[c]);
  });
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) V[(size_t)(H + w0 + g + 4 * r) * SB + j0 + 16 * c + i] = -acc[c][r];
}

// The solves' steps are a chain, so each has to be short: a workgroup takes a
// small tile of the result, its 4 waves every 4th step of 16 k of the same tile,
// and their sums are added through LDS in order.  (A v_mfma_f64_16x16x4 holds its
// SIMD for 75 cycles: one wave per tile chained 32 steps of 300 cycles and more, and
// tiles large enough for that left many SIMDs with none.)  N = 5500, inverses
// included: 256 right-hand sides 657 -> 400 us, one 289 -> 178; 512-row blocks
// against 256 save 90 of that.  256 right-hand sides cost the matrix cores 115 us.

// k_solve_diag: x_k = inv_k r_k (TR: with inv_k's transpose) for the block's
// rows, 16 rows (grid y) of 16 right-hand sides per workgroup; R [B][N] what is
// left of the right-hand sides, X [B][N] the solution.
template <bool TR>
__global__ __launch_bounds__(256, 2) void k_solve_diag(const double* __restrict__ inv, int64_t N, int64_t k0, int64_t B,
                                                     const double* __restrict__ R, double* __restrict__ X) {
  __shared__ double red[4][4][64];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w0 = 16 * blockIdx.y, nb = (int)min((int64_t)SB, N - k0);
  const int64_t b0 = (int64_t)blockIdx.x * 16;
  const double* V = inv + (size_t)(k0 / SB) * SB * SB;
  const double* r = R + (size_t)min(b0 + i, B - 1) * N + k0 + 4 * g;
  const int row = w0 + i;
  const int kb = (TR ? w0 : 0) + 16 * wave;
  const int ke = min((nb + 15) & ~15, TR ? SB : w0 + 16);
  constexpr int D = 8;  // a wave's steps, all in flight
  d4 acc = {0.0, 0.0, 0.0, 0.0}, x[D], v[D];
  pipelined<D>((ke - kb + 63) / 64, [&](int s, int q) {
    const int k = kb + 64 * s;
    x[q] = frag_row(r + k, nb - k - 4 * g);  // (what is left of the block from the lane's first column on)
    v[q] = TR ? frag_col(V + (size_t)(k + 4 * g) * SB + row, SB, 4) : frag_row(V + (size_t)row * SB + k + 4 * g, 4);
  }, [&](int q) { mma16(x[q], v[q], acc); });
#pragma unroll
  for (int q = 0; q < 4; ++q) red[wave][q][lane] = acc[q];
  __syncthreads();
  const int64_t b = b0 + g + 4 * wave;  // wave w adds and writes register w
  if (row >= nb || b >= B) return;
  double s = ((red[0][wave][lane] + red[1][wave][lane]) + red[2][wave][lane]) + red[3][wave][lane];
  if (s != s) {  // something not finite, perhaps only against a zero on the triangle's other side
    const double* rb = R + (size_t)b * N + k0;
    s = 0.0;
    for (int k = TR ? row : 0; k < (TR ? nb : row + 1); ++k) s += rb[k] * V[TR ? (size_t)k * SB + row : (size_t)row * SB + k];
  }
  X[(size_t)b * N + k0 + row] = s;
}

// k_solve_update: removes the solved block of BS rows from the rows still to come
// (forward: after it, r_i -= sum_t L[i][k0+t] x_{k0+t}; TR: before it,
// r_i -= sum_t L[k0+t][i] x_{k0+t}), 32 rows x 16 WB right-hand sides a
// workgroup.  Workgroups are numbered so that one XCD's L2 holds the same rows of
// L for all right-hand sides.  X may be R (the rows read and written are others).
template <bool TR, int WB, int BS>
__global__ __launch_bounds__(256, 2) void k_solve_update(const double* __restrict__ L, int64_t N, int64_t k0, int64_t B,
                                                      int gy, const double* __restrict__ X, double* __restrict__ R) {
  __shared__ double red[4][2 * WB][4][64];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = (int)min((int64_t)BS, N - k0);
  const int id = xcd_order(blockIdx.x, gridDim.x);
  const int64_t row0 = (TR ? 0 : k0 + BS) + (int64_t)(id / gy) * 32, row_end = TR ? k0 : N;
  const int64_t b0 = (int64_t)(id % gy) * (16 * WB);
  const double* x[WB];
  int64_t rw[2];
#pragma unroll
  for (int a = 0; a < WB; ++a) x[a] = X + (size_t)min(b0 + 16 * a + i, B - 1) * N + k0;
#pragma unroll
  for (int c = 0; c < 2; ++c) rw[c] = min(row0 + 16 * c + i, row_end - 1);
  d4 acc[WB][2];
#pragma unroll
  for (int a = 0; a < WB; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[a][c] = d4{0.0, 0.0, 0.0, 0.0};
  constexpr int D = 4;
  d4 xv[D][WB], lv[D][2];
  auto load = [&](int s, int q, int left) {  // left: columns from the lane's first on (4: all)
    const int kk = 64 * s + 16 * wave + 4 * g;
#pragma unroll
    for (int a = 0; a < WB; ++a) xv[q][a] = frag_row(x[a] + kk, left);
#pragma unroll
    for (int c = 0; c < 2; ++c)
      lv[q][c] = TR ? frag_col(L + (size_t)(k0 + kk) * N + rw[c], N, left)
                    : frag_row(L + (size_t)rw[c] * N + k0 + kk, left);
  };
  auto use = [&](int q) {
#pragma unroll
    for (int a = 0; a < WB; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c) mma16(xv[q][a], lv[q][c], acc[a][c]);
  };
  if (nb == BS)
    pipelined<D>(BS / 64, [&](int s, int q) { load(s, q, 4); }, use);
  else
    pipelined<D>((nb - 16 * wave + 63) / 64,
                 [&](int s, int q) { load(s, q, nb - (64 * s + 16 * wave) - 4 * g); }, use);
#pragma unroll
  for (int a = 0; a < WB; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) red[wave][2 * a + c][q][lane] = acc[a][c][q];
  __syncthreads();
  // the 2 WB tiles of 4 registers, in turn to the waves
  for (int e = wave; e < 8 * WB; e += 4) {
    const int t = e >> 2, q = e & 3;
    const int64_t b = b0 + 16 * (t >> 1) + g + 4 * q, row = row0 + 16 * (t & 1) + i;
    if (b < B && row < row_end)
      R[(size_t)b * N + row] -= ((red[0][t][q][lane] + red[1][t][q][lane]) + red[2][t][q][lane]) + red[3][t][q][lane];
  }
}

// Solves with at most 64 rows, all modes in one launch: a wave takes a
// right-hand side, lane i row i, by substitution (10 rows, L^-T L^-1: 64 us a call with
// three launches, 56 with one).  ld: row stride of all three.  X may be R.
__global__ __launch_bounds__(256) void k_solve_small(const double* __restrict__ L, int N, int64_t ld, const double* R,
                                                     double* X, int64_t B, int mode) {
  __shared__ double S[DB * LS];
  const int lane = threadIdx.x & 63;
  for (int e = threadIdx.x; e < DB * DB; e += 256) {
    const int r = e / DB, c = e - r * DB;
    if (r < N && c <= r) S[r * LS + c] = L[(size_t)r * ld + c];
  }
  __syncthreads();
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= B) return;
  const double rd = lane < N ? 1.0 / S[lane * LS + lane] : 0.0;
  double r = lane < N ? R[(size_t)b * ld + lane] : 0.0;
  if (mode != 1) {
    for (int k = 0; k < N; ++k) {
      const double x = lane_d(r, k) * lane_d(rd, k);
      if (lane > k && lane < N) r -= S[lane * LS + k] * x;
      else if (lane == k) r = x;
    }
  }
  if (mode != 0) {
    for (int k = N - 1; k >= 0; --k) {
      const double x = lane_d(r, k) * lane_d(rd, k);
      if (lane < k) r -= S[k * LS + lane] * x;
      else if (lane == k) r = x;
    }
  }
  if (lane < N) X[(size_t)b * ld + lane] = r;
}

// r = data - mu (FP64), [B][N]
__global__ void k_resid(const float* __restrict__ mu, const double* __restrict__ data, int64_t N, int64_t B,
                        double* __restrict__ r) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= N * B) return;
  r[e] = data[e % N] - (double)mu[e];
}

// out[b] = -1/2 sum_i z[b][i]^2 + c0: 256 threads per right-hand side, fixed order
__global__ __launch_bounds__(256) void k_sq_sum(const double* __restrict__ Z, int64_t N, double c0,
                                                double* __restrict__ out) {
  __shared__ double ws[4];
  const int64_t b = blockIdx.x;
  const double* z = Z + (size_t)b * N;
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < N; i += 256) s += z[i] * z[i];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[b] = -0.5 * (((ws[0] + ws[1]) + ws[2]) + ws[3]) + c0;
}

__global__ void k_to_float(const double* __restrict__ x, int64_t n, float* __restrict__ y) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) y[e] = (float)x[e];
}

// one row a block
__global__ __launch_bounds__(256) void k_unpack_lower(const double* __restrict__ src, double* __restrict__ A, int64_t N,
                                                      int64_t r0) {
  const int64_t r = r0 + blockIdx.x;
  const double* in = src + (tri_row(r) - tri_row(r0));
  double* out = A + (size_t)r * N;
#pragma unroll 4
  for (int64_t c = threadIdx.x; c <= r; c += 256) out[c] = in[c];
}

hipError_t launch_unpack_lower(const double* src, double* A, int64_t N, int64_t r0, int64_t r1, hipStream_t s) {
  if (r1 <= r0) return hipSuccess;
  hipLaunchKernelGGL(k_unpack_lower, dim3((unsigned)(r1 - r0)), dim3(256), 0, s, src, A, N, r0);
  return hipGetLastError();
}

hipError_t launch_dense_cholesky(double* A, int64_t N, double* inv, double* dlog, int* bad, hipStream_t s) {
  if (N < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_chol_first, dim3(1), dim3(256), 0, s, A, N, inv, dlog, bad);
  for (int64_t k0 = 0; N - k0 > DB; k0 += DB) {
    const int64_t rest = N - k0 - DB, T = (rest + DB - 1) / DB;
    hipLaunchKernelGGL(k_chol_panel, dim3((unsigned)T), dim3(256), 0, s, A, N, k0, inv);
    hipLaunchKernelGGL(k_chol_syrk, dim3((unsigned)(T * (T + 1) / 2)), dim3(256), 0, s, A, N, k0, inv, dlog, bad);
  }
  hipLaunchKernelGGL(k_zero_upper, dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>((N + 255) / 256, 64)),
                                         (unsigned)N),
                     dim3(256), 0, s, A, N);
  return hipGetLastError();
}

hipError_t launch_tri_inverse(const double* L, int64_t N, double* inv, hipStream_t s) {
  if (N < 1) return hipErrorInvalidValue;
  // whole SB blocks: the merges of a partial last block read identity rows
  const int64_t ns = (N + SB - 1) / SB;
  hipLaunchKernelGGL(k_tri_inv64, dim3((unsigned)(N <= DB ? 1 : ns * (SB / DB))), dim3(256), 0, s, L, N, inv);
  static_assert(SB == 512, "the merges go 64 -> 128 -> 256 -> 512");
  if (N > 64) hipLaunchKernelGGL((k_tri_merge<64, 2>), dim3((unsigned)(ns * 4), 2), dim3(256), 0, s, L, N, inv);
  if (N > 128) hipLaunchKernelGGL((k_tri_merge<128, 2>), dim3((unsigned)(ns * 2), 4), dim3(512), 0, s, L, N, inv);
  if (N > 256) hipLaunchKernelGGL((k_tri_merge<256, 1>), dim3((unsigned)ns, 16), dim3(1024), 0, s, L, N, inv);
  return hipGetLastError();
}

// (16 right-hand sides at most: half the products)
template <bool TR, int BS>
static void solve_update(const double* L, int64_t N, int64_t k0, int64_t B, const double* X, double* R, hipStream_t s) {
  const int64_t rows = TR ? k0 : N - k0 - BS;
  if (rows <= 0) return;
  const int gy = (int)(B <= 16 ? 1 : (B + 31) / 32);
  const dim3 gu((unsigned)((rows + 31) / 32 * gy));
  if (B <= 16) hipLaunchKernelGGL((k_solve_update<TR, 1, BS>), gu, dim3(256), 0, s, L, N, k0, B, gy, X, R);
  else hipLaunchKernelGGL((k_solve_update<TR, 2, BS>), gu, dim3(256), 0, s, L, N, k0, B, gy, X, R);
}

template <bool TR>
static void solve_pass(const double* L, int64_t N, const double* inv, double* R, double* X, int64_t B, hipStream_t s) {
  const int64_t last = (N - 1) / SB * SB;
  for (int64_t step = 0; step <= last; step += SB) {
    const int64_t k0 = TR ? last - step : step, nb = std::min<int64_t>(SB, N - k0);
    const dim3 gd((unsigned)((B + 15) / 16), (unsigned)((nb + 15) / 16));
    hipLaunchKernelGGL((k_solve_diag<TR>), gd, dim3(256), 0, s, inv, N, k0, B, R, X);
    solve_update<TR, SB>(L, N, k0, B, X, R, s);
  }
}

template <bool TR>
static void solve_pass_in_place(const double* L, int64_t N, double* X, int64_t B, hipStream_t s) {
  const int64_t last = (N - 1) / DB * DB;
  for (int64_t step = 0; step <= last; step += DB) {
    const int64_t k0 = TR ? last - step : step;
    hipLaunchKernelGGL(k_solve_small, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, s, L + (size_t)k0 * N + k0,
                       (int)std::min<int64_t>(DB, N - k0), N, X + k0, X + k0, B, TR ? 1 : 0);
    solve_update<TR, DB>(L, N, k0, B, X, X, s);
  }
}

hipError_t launch_dense_solve(const double* L, int64_t N, const double* inv, double* R, double* X, int64_t B,
                              int transpose, hipStream_t s) {
  if (N < 1 || B < 1 || R == X) return hipErrorInvalidValue;
  if (transpose) solve_pass<true>(L, N, inv, R, X, B, s);
  else solve_pass<false>(L, N, inv, R, X, B, s);
  return hipGetLastError();
}

hipError_t launch_small_solve(const double* L, int N, const double* R, double* X, int64_t B, int mode, hipStream_t s) {
  if (N < 1 || N > DB || B < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_solve_small, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, s, L, N, (int64_t)N, R, X, B, mode);
  return hipGetLastError();
}

hipError_t launch_dense_solve_in_place(const double* L, int64_t N, double* X, int64_t B, int mode, hipStream_t s) {
  if (N < 1 || B < 1) return hipErrorInvalidValue;
  if (mode != 1) solve_pass_in_place<false>(L, N, X, B, s);
  if (mode != 0) solve_pass_in_place<true>(L, N, X, B, s);
  return hipGetLastError();
}

hipError_t launch_dense_loglike(const float* mu, int64_t B, int64_t N, const double* data, const double* L, double c0,
                                const double* inv, double* Z, double* X, double* loglike, float* dmu, hipStream_t s) {
  const int64_t n = B * N;
  hipError_t e;
  hipLaunchKernelGGL(k_resid, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, mu, data, N, B, Z);
  if ((e = launch_dense_solve(L, N, inv, Z, X, B, 0, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_sq_sum, dim3((unsigned)B), dim3(256), 0, s, X, N, c0, loglike);
  if (dmu) {
    if ((e = launch_dense_solve(L, N, inv, X, Z, B, 1, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_to_float, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Z, n, dmu);
  }
  return hipGetLastError();
}

}  // namespace jc
