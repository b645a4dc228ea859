// Gaussian likelihood algebra on the device (likelihood.py:9-61,
// sparse.py:295-389), for the block-diagonal covariances the path produces:
// the reference's sparse format [P][P][n_ell] holds, for each ell, a P x P
// block (entry (p, q, l) couples C_p(ell_l) and C_q(ell_l)).
//
// k_block_inv:  per ell, the inverse of the P x P block by Gauss-Jordan
//               elimination (FP64; any invertible block, as sparse.py:295-315
//               inverts) and the product of its pivots, whose magnitude is
//               |det| (sparse.py:322-366).
// k_chi2:       per (ell, group of 32 cosmologies), r = data - mu and
//               s = C_l^-1 r on the FP64 matrix cores; writes s (the
//               derivative of the log-likelihood with respect to mu, the
//               adjoint's cotangent) and r^T s per (cosmology, ell).
// k_chi2_sum:   per cosmology, -1/2 sum_l r^T s in a fixed order plus a
//               constant (deterministic).
//
// Blocks are dealt to the XCDs so that each takes a contiguous range of ell: the
// arrays' innermost index is ell, and neighbours share cache lines.
#include "jc_kernels.hpp"
#include "jc_mma64.hpp"

namespace jc {

constexpr int LK_MAXP = 64;  // pairs per block (10 tracers give 55)

// element (p, q) of block l of a precision array
__device__ __forceinline__ size_t prec_at(const PrecLayout& a, int P, int p, int q, int l) {
  return ((size_t)p * P + q) * a.pair + (size_t)l * a.ell;
}

// Gauss-Jordan with partial pivoting of the P x 2P array A in LDS (the block
// beside the identity, loaded here); pivots to piv.
__device__ void gauss_jordan_pivoting(const double* __restrict__ cov, int P, int n_ell, int l, double* A, double* piv) {
  __shared__ int s_row;
  const int W2 = 2 * P;
  for (int e = threadIdx.x; e < P * W2; e += blockDim.x) {
    const int p = e / W2, q = e - p * W2;
    A[e] = q < P ? cov[((size_t)p * P + q) * n_ell + l] : (q - P == p ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int k = 0; k < P; ++k) {
    // the row at or below k with the largest |A[i][k]|
    if (threadIdx.x == 0) {
      int r = k;
      double best = fabs(A[k * W2 + k]);
      for (int i = k + 1; i < P; ++i) {
        const double v = fabs(A[i * W2 + k]);
        if (v > best) {
          best = v;
          r = i;
        }
      }
      s_row = r;
    }
    __syncthreads();
    const int r = s_row;
    if (r != k) {
      for (int q = threadIdx.x; q < W2; q += blockDim.x) {
        const double t = A[k * W2 + q];
        A[k * W2 + q] = A[r * W2 + q];
        A[r * W2 + q] = t;
      }
      __syncthreads();
    }
    const double pk = A[k * W2 + k];
    if (threadIdx.x == 0) piv[k] = pk;
    const double ip = 1.0 / pk;
    __syncthreads();
    // row k scaled, then every other row i -= A[i][k] * row k
    for (int q = threadIdx.x; q < W2; q += blockDim.x) A[k * W2 + q] *= ip;
    __syncthreads();
    for (int e = threadIdx.x; e < P * W2; e += blockDim.x) {
      const int i = e / W2, q = e - i * W2;
      if (i != k && q != k) A[e] -= A[i * W2 + k] * A[k * W2 + q];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < P; i += blockDim.x)
      if (i != k) A[i * W2 + k] = 0.0;
    __syncthreads();
  }
}

// One workgroup inverts one block, in place and in registers: thread (ti, tj)
// holds the elements (ti + 16 r, tj + 16 c).  A step shares its pivot row and
// column through LDS (two buffers, so one barrier a step) and costs a division
// and 16 FMAs a thread; with the array in LDS, beside the identity, it was four
// barriers and eight times the LDS traffic.  Bound by the chain of P steps.  55 x 55
// blocks, 100 ell: 246 -> 32 us.
// Eliminates on the diagonal (the order that suits the symmetric positive
// definite covariances, whose badly scaled rows row exchanges would mix); a block
// with a non-positive pivot there is started again with partial pivoting, which
// inverts any invertible block.
// ld[l] = the product of the pivots' mantissas and the sum of their exponents
// (|det| = ld[l][0] 2^ld[l][1]; zero or not finite for a singular block).
__global__ __launch_bounds__(256) void k_block_inv(const double* __restrict__ cov, int P, int n_ell,
                                                    double* __restrict__ inv, PrecLayout lay,
                                                    double* __restrict__ ld) {
  extern __shared__ double A[];  // [P][2P], for the pivoting pass
  __shared__ double s_r[2][LK_MAXP], s_c[2][LK_MAXP], s_piv[LK_MAXP];
  const int l = xcd_order(blockIdx.x, n_ell);
  const int ti = threadIdx.x >> 4, tj = threadIdx.x & 15;
  double a[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int p = ti + 16 * r, q = tj + 16 * c;
      a[r][c] = p < P && q < P ? cov[((size_t)p * P + q) * n_ell + l] : 0.0;
    }
  bool bad = false;  // uniform: every thread sees every pivot
#pragma unroll
  for (int kr = 0; kr < 4; ++kr) {
    for (int kk = 0; kk < 16; ++kk) {
      const int k = 16 * kr + kk, u = k & 1;
      if (k >= P || bad) break;
      if (ti == kk)
#pragma unroll
        for (int c = 0; c < 4; ++c) s_r[u][tj + 16 * c] = a[kr][c];
      if (tj == kk)
#pragma unroll
        for (int r = 0; r < 4; ++r) s_c[u][ti + 16 * r] = a[r][kr];
      __syncthreads();
      const double pk = s_r[u][k], ip = 1.0 / pk;
      if (threadIdx.x == 0) s_piv[k] = pk;
      bad = !(pk > 0.0);
      double row[4], col[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) row[c] = s_r[u][tj + 16 * c] * ip;
#pragma unroll
      for (int r = 0; r < 4; ++r) col[r] = s_c[u][ti + 16 * r];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          double v = a[r][c] - col[r] * row[c];
          if (r == kr && ti == kk) v = row[c];
          if (c == kr && tj == kk) v = r == kr && ti == kk ? ip : -(col[r] * ip);
          a[r][c] = v;
        }
    }
  }
  __syncthreads();
  if (bad) gauss_jordan_pivoting(cov, P, n_ell, l, A, s_piv);
  if (threadIdx.x < 64) {
    int e = 0;
    double m = (int)threadIdx.x < P ? frexp(fabs(s_piv[threadIdx.x]), &e) : 1.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      m *= __shfl_xor(m, o);
      e += __shfl_xor(e, o);
    }
    if (threadIdx.x == 0) {
      ld[2 * l] = m;
      ld[2 * l + 1] = (double)e;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int p = ti + 16 * r, q = tj + 16 * c;
      if (p < P && q < P) inv[prec_at(lay, P, p, q, l)] = bad ? A[p * 2 * P + P + q] : a[r][c];
    }
}

// A workgroup per (ell, 32 cosmologies): the precision block and the residuals
// are staged once, all loads in flight together, and S = C_l^-1 R is one product
// of 16 x 16 tiles; wave w takes the cosmologies 16 (w % 2) .. + 15 and the pairs
// 32 (w / 2) .. + 31.  Rows are padded by two doubles (16 rows at a time fall on
// different LDS banks).  One cosmology a wave at a time, with the product on the
// VALU from LDS, waited for its residuals' loads on every turn.  256 means, 55
// pairs, 100 ell: 41 -> 23 us.
constexpr int LK_CB = 32, LK_LS = LK_MAXP + 2;

__global__ __launch_bounds__(256) void k_chi2(const float* __restrict__ mu, int B, int P, int n_ell,
                                               const double* __restrict__ data, const double* __restrict__ prec,
                                               PrecLayout lay, float* __restrict__ s_out, double* __restrict__ part) {
  __shared__ __align__(16) double Pl[LK_MAXP * LK_LS];  // [pair][pair]
  __shared__ __align__(16) double Rl[LK_CB * LK_LS];    // [cosmology][pair]
  __shared__ double sv[2][LK_CB];
  const int l = xcd_order(blockIdx.x, n_ell);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  const int64_t b0 = (int64_t)blockIdx.y * LK_CB;
  const int pad = (P + 15) & ~15;
  // lane p takes pair p of every 4th row; all loads before the first use
  const bool in = lane < P;
  const double dl = in ? data[(size_t)lane * n_ell + l] : 0.0;
  float m[LK_CB / 4];
  double pr[LK_MAXP / 4];
#pragma unroll
  for (int j = 0; j < LK_CB / 4; ++j) {
    const int64_t b = b0 + wave + 4 * j;
    m[j] = in && b < B ? mu[((size_t)b * P + lane) * n_ell + l] : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < LK_MAXP / 4; ++j) {
    const int p = wave + 4 * j;
    pr[j] = in && p < P ? prec[prec_at(lay, P, p, lane, l)] : 0.0;
  }
#pragma unroll
  for (int j = 0; j < LK_CB / 4; ++j)
    Rl[(wave + 4 * j) * LK_LS + lane] = b0 + wave + 4 * j < B ? dl - (double)m[j] : 0.0;
#pragma unroll
  for (int j = 0; j < LK_MAXP / 4; ++j) Pl[(wave + 4 * j) * LK_LS + lane] = pr[j];
  __syncthreads();
  const int bl = 16 * (wave & 1) + i, t0 = 2 * (wave >> 1);
  const double* rb = Rl + bl * LK_LS;
  auto frag = [&](const double* p) { return d4{p[0], p[1], p[2], p[3]}; };
  double v = 0.0;
#pragma unroll
  for (int t = t0; t < t0 + 2; ++t) {
    if (16 * t >= P) break;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k = 4 * g; k < pad; k += 16) mma16(frag(Pl + (16 * t + i) * LK_LS + k), frag(rb + k), acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p = 16 * t + g + 4 * r;  // a padded pair's 0 x inf stays out
      if (p < P) {
        v += rb[p] * acc[r];
        if (s_out && b0 + bl < B) s_out[((size_t)(b0 + bl) * P + p) * n_ell + l] = (float)acc[r];
      }
    }
  }
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  if (g == 0) sv[wave >> 1][bl] = v;
  __syncthreads();
  if (threadIdx.x < LK_CB && b0 + threadIdx.x < B)
    part[(size_t)(b0 + threadIdx.x) * n_ell + l] = sv[0][threadIdx.x] + sv[1][threadIdx.x];
}

// one wave per cosmology: lane j adds ell j, j + 64, ..., then a butterfly
// over the wave (a fixed order)
__global__ __launch_bounds__(64) void k_chi2_sum(const double* __restrict__ part, int n_ell, double c0,
                                                  double* __restrict__ out) {
  const int b = blockIdx.x;
  const int lane = threadIdx.x;
  double s = 0.0;
  for (int l = lane; l < n_ell; l += 64) s += part[(size_t)b * n_ell + l];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  if (lane == 0) out[b] = -0.5 * s + c0;
}

hipError_t launch_block_inv(const double* cov, int P, int n_ell, double* inv, PrecLayout lay, double* ld,
                            hipStream_t s) {
  if (P < 1 || P > LK_MAXP) return hipErrorInvalidValue;
  const size_t sm = (size_t)P * 2 * P * sizeof(double);
  hipLaunchKernelGGL(k_block_inv, dim3(n_ell), dim3(256), sm, s, cov, P, n_ell, inv, lay, ld);
  return hipGetLastError();
}

hipError_t launch_loglike(const float* mu, int B, int P, int n_ell, const double* data, const double* prec,
                          PrecLayout lay, double c0, float* s_out, double* part, double* loglike, hipStream_t s) {
  if (P < 1 || P > LK_MAXP) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_chi2, dim3(n_ell, (B + LK_CB - 1) / LK_CB), dim3(256), 0, s, mu, B, P, n_ell, data, prec, lay,
                     s_out, part);
  hipLaunchKernelGGL(k_chi2_sum, dim3(B), dim3(64), 0, s, part, n_ell, c0, loglike);
  return hipGetLastError();
}

}  // namespace jc
