// Numeric set-up of the multigrid levels (smoothed aggregation, rebuilt at every Newton iteration).
//
// Between its sparse products a set-up needs, per level, the inverse diagonal, the largest
// eigenvalue of D^-1 A (12 Lanczos steps, one matrix product each), the smoother's weights and the
// transfers of the cycle, and at the end the dense inverse of the coarsest operator.  All of it is
// short vectors and small matrices, so launches, not bytes, are what it costs: about a thousand of
// them per set-up and three host reads when written as vector operations.  Here a Lanczos step is
// two launches (the scalars stay on the device as per-block partial sums that the next launch adds up
// itself), a level's copies and permutations are one each, and the dense inverse is one launch per 32
// columns and one more.  Everything is deterministic: sums are taken in a fixed order.
// Assembly, set-up and solve of the 383x383 p-Laplace system (three levels above 286 unknowns, 10 CG
// iterations), pass after pass: 6.48 -> 3.12 ms by this file, 2.20 with the cycle's passes of fne_amg.hip.
// The set-up alone, waited for: 383x383 p-Laplace 4.53 -> 0.89 ms, 320x16x16 beam with six rigid-body
// modes 16.1 -> 8.6, P4 slope by p-multigrid (128,080 unknowns) 6.28 -> 1.32.
#include "fne_common.h"

#include <algorithm>

namespace {

constexpr int kLanThreads = 256;
constexpr int kLanBlocks = 512;   // blocks of the vector kernels = partial sums of |w|^2
constexpr int kLanParts = 1024;   // partial sums of w.v that every block adds up itself; above, one block first
constexpr int kLanSteps = 64;

// sum over the workgroup, the same on every thread (fixed order)
__device__ __forceinline__ double block_sum_all(double v) {
  __shared__ double s_part[kLanThreads / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();  // the last sum's readers are done
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < kLanThreads / 64; ++i) t += s_part[i];
  return t;
}

__device__ __forceinline__ double sum_parts(const double* __restrict__ part, int n) {
  double t = 0.0;
  for (int i = threadIdx.x; i < n; i += kLanThreads) t += part[i];
  return block_sum_all(t);
}

// dinv = 1 / diagonal (1 where that is zero), s = |dinv|^1/2 (finite where an indefinite Hessian has a
// negative diagonal), u = s v0 and partial sums of |v0|^2; w = v0 is read in place
template <typename VT>
__global__ __launch_bounds__(kLanThreads) void lanczos_start_kernel(int n, const VT* __restrict__ vals,
                                                                    const int64_t* __restrict__ diag,
                                                                    const double* __restrict__ v0,
                                                                    double* __restrict__ dinv,
                                                                    double* __restrict__ s, double* __restrict__ u,
                                                                    double* __restrict__ part) {
  double t = 0.0;
  for (int i = blockIdx.x * kLanThreads + threadIdx.x; i < n; i += gridDim.x * kLanThreads) {
    const double a = double(vals[diag[i]]);
    const double di = 1.0 / (a == 0.0 ? 1.0 : a);
    const double si = sqrt(fabs(di)), w = v0[i];
    dinv[i] = di;
    s[i] = si;
    u[i] = si * w;
    t += w * w;
  }
  t = block_sum_all(t);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// v = w / beta; y = S v - beta v_prev with S = D^-1/2 A D^-1/2 (u = D^-1/2 w); partial sums of y.v.
// beta = |w|; the first step has none before it
template <typename VT, int LPR, int FORM>
__global__ __launch_bounds__(kLanThreads) void lanczos_mult_kernel(
    int n, const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, const VT* __restrict__ vals,
    const double* __restrict__ s, const double* __restrict__ u, const double* __restrict__ w,
    const double* __restrict__ v_prev, double* __restrict__ v, double* __restrict__ y,
    const double* __restrict__ norm_part, int n_norm, double* __restrict__ part, double* __restrict__ beta_out) {
  __shared__ double prod[FORM == 2 ? kStreamCap : 1];
  const double nrm = sqrt(sum_parts(norm_part, n_norm));
  if (beta_out && blockIdx.x == 0 && threadIdx.x == 0) *beta_out = nrm;
  const double div = fmax(nrm, 1e-300);
  int row;
  bool leader;
  const double acc =
      csr_form_dot<VT, LPR, FORM>(n, indptr, indices, vals, [&](int c) { return u[c]; }, prod, row, leader);
  double t = 0.0;
  if (leader) {
    const double vi = w[row] / div;
    double yi = s[row] * (acc / div);
    if (v_prev) yi -= nrm * v_prev[row];
    v[row] = vi;
    y[row] = yi;
    t = yi * vi;
  }
  t = block_sum_all(t);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ __launch_bounds__(kLanThreads) void lanczos_join_kernel(const double* __restrict__ part, int n,
                                                                   double* __restrict__ out) {
  const double t = sum_parts(part, n);
  if (threadIdx.x == 0) out[0] = t;
}

// alpha = y.v; w = y - alpha v, u = D^-1/2 w and partial sums of |w|^2
__global__ __launch_bounds__(kLanThreads) void lanczos_update_kernel(int n, const double* __restrict__ y,
                                                                     const double* __restrict__ v,
                                                                     const double* __restrict__ s,
                                                                     double* __restrict__ w, double* __restrict__ u,
                                                                     const double* __restrict__ dot_part, int n_dot,
                                                                     double* __restrict__ part,
                                                                     double* __restrict__ alpha_out) {
  const double alpha = sum_parts(dot_part, n_dot);
  if (blockIdx.x == 0 && threadIdx.x == 0) *alpha_out = alpha;
  double t = 0.0;
  for (int i = blockIdx.x * kLanThreads + threadIdx.x; i < n; i += gridDim.x * kLanThreads) {
    const double wi = y[i] - alpha * v[i];
    w[i] = wi;
    u[i] = s[i] * wi;
    t += wi * wi;
  }
  t = block_sum_all(t);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// Largest eigenvalue of the symmetric tridiagonal (alpha, beta) by multisection: the leading minors of
// x - T are all positive exactly where x is above every eigenvalue (T scaled to its bound, so that
// the minors stay in range; products instead of the pivots' quotients, 17 -> 10 us in a kernel trace).  64 points per
// round, so 6 bits each; 11 rounds.  out = {max(lambda, 1e-300), 1 if every coefficient is finite else 0}.
__global__ __launch_bounds__(kLanThreads) void lanczos_eig_kernel(int k, const double* __restrict__ alpha,
                                                                  const double* __restrict__ beta,
                                                                  const double* __restrict__ norm_part, int n_norm,
                                                                  double* __restrict__ out) {
  const double last = sqrt(sum_parts(norm_part, n_norm));  // checked like the others, not used
  __shared__ double s_a[kLanSteps], s_b[kLanSteps];  // diagonal, and off-diagonal before it
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  if (lane < k) {
    s_a[lane] = alpha[lane];
    s_b[lane] = lane > 0 ? beta[lane - 1] : 0.0;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  double lo = -INFINITY, hi = -INFINITY;
  bool ok = isfinite(last);
  for (int i = 0; i < k; ++i) {
    const double a = s_a[i], bl = fabs(s_b[i]), br = i + 1 < k ? fabs(s_b[i + 1]) : 0.0;
    ok = ok && isfinite(a) && isfinite(bl) && isfinite(br);
    lo = fmax(lo, a);
    hi = fmax(hi, a + bl + br);
  }
  const double bound = fmax(fabs(lo), fabs(hi));
  if (ok && bound > 0.0) {
    const double inv = 1.0 / bound;
    if (lane < k) {
      s_a[lane] *= inv;
      s_b[lane] *= inv;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    lo *= inv;
    hi *= inv;
    for (int round = 0; round < 11; ++round) {
      const double x = lo + (hi - lo) * ((lane + 1) / 65.0);
      bool above = true;
      double p1 = 1.0, p2 = 0.0;
      for (int i = 0; i < k; ++i) {
        const double p = (x - s_a[i]) * p1 - s_b[i] * s_b[i] * p2;
        above = above && p > 0.0;
        p2 = p1;
        p1 = p;
      }
      const unsigned long long m = __ballot(above);
      const int f = m ? __ffsll((long long)m) - 1 : 64;  // first point above the spectrum
      const double xf = __shfl(x, min(f, 63), 64), xp = __shfl(x, max(f - 1, 0), 64);
      if (f > 0) lo = xp;
      if (f < 64) hi = xf;
    }
    lo *= bound;
    hi *= bound;
  }
  if (lane == 0) {
    out[0] = ok ? fmax(0.5 * (lo + hi), 1e-300) : NAN;
    out[1] = ok ? 1.0 : 0.0;
  }
}

// wd = f_wd / lambda dinv; wcheb[k] = f_k / lambda dinv
struct SmootherFactors {
  double wd, cheb[8];
  int n;
};
__global__ __launch_bounds__(kLanThreads) void smoother_weights_kernel(int n, const double* __restrict__ dinv,
                                                                       const double* __restrict__ lam,
                                                                       SmootherFactors f, double* __restrict__ wd,
                                                                       double* __restrict__ wcheb) {
  const double l = lam[0];
  for (int i = blockIdx.x * kLanThreads + threadIdx.x; i < n; i += gridDim.x * kLanThreads) {
    const double di = dinv[i];
    wd[i] = f.wd / l * di;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k < f.n) wcheb[int64_t(k) * n + i] = f.cheb[k] / l * di;
  }
}

// R = P^T by its permutation, and both transfers in the cycle's precision
template <typename VT>
__global__ __launch_bounds__(256) void transfers_kernel(int nnz, const double* __restrict__ p,
                                                        const int64_t* __restrict__ perm, double* __restrict__ r,
                                                        VT* __restrict__ p_cycle, VT* __restrict__ r_cycle) {
  for (int k = blockIdx.x * 256 + threadIdx.x; k < nnz; k += gridDim.x * 256) {
    const double a = p[perm[k]];
    r[k] = a;
    r_cycle[k] = VT(a);
    p_cycle[k] = VT(p[k]);
  }
}

// A = (C + C^T) / 2 by the transpose's permutation, and the cycle's copy
template <typename VT>
__global__ __launch_bounds__(256) void symmetrise_kernel(int nnz, const double* __restrict__ c,
                                                         const int64_t* __restrict__ perm, double* __restrict__ a,
                                                         VT* __restrict__ a_cycle) {
  for (int k = blockIdx.x * 256 + threadIdx.x; k < nnz; k += gridDim.x * 256) {
    const double v = 0.5 * (c[k] + c[perm[k]]);
    a[k] = v;
    if (a_cycle) a_cycle[k] = VT(v);
  }
}

// ---------------------------------------------------------------------------------------------
// Dense inverse of a symmetric positive definite matrix by its Cholesky factor: A = L L^T,
// F = L^-1, A^-1 = F^T F, in 32x32 tiles.  One launch per block column K, a workgroup per tile of the
// lower triangle from row K down.  Each factors A_KK for itself in LDS (32 pivots, one after the other,
// which is cheaper than a launch of its own) and keeps T = L_KK^-1; then, with L_IK = A_IK T^T,
//   row K:     F_KJ = T M_KJ (J < K), F_KK = T
//   rows I>K:  M_IJ -= L_IK (T M_KJ) (J < K), M_IK = -L_IK T, A_IJ -= L_IK L_JK^T (J > K)
// where M is the part of L^-1 that is still being eliminated.  A_IJ lies in the lower tiles and M_IJ in
// the tiles above the diagonal, so nothing that a workgroup reads is written in the same launch.
// Only L_KK is inverted explicitly, whose condition is the square root of A_KK's: the inverse is as
// accurate as LAPACK's potrf and potri (block Gauss-Jordan with explicit inverses of the A_KK themselves
// loses 1e5 of that at condition 1e8 and 33 unknowns).  The pivots are those of an LDL^T factorisation,
// all positive exactly when the matrix is positive definite.  Products by v_mfma 16x16x4 in FP64, a
// quadrant per wavefront.  Bound by the 32 pivots of each launch, one after the other.  Call after call,
// 286 unknowns 152 us, 1,200 unknowns 853 (Gauss-Jordan on the whole square 146 and 1,417, the library's
// factorisation and inverse 993 and 4,230).
// ---------------------------------------------------------------------------------------------
constexpr int kTile = 32, kTs = kTile + 1;  // LDS row stride
typedef double d4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void spd_rows_kernel(int n, int npad, const int32_t* __restrict__ indptr,
                                                       const int32_t* __restrict__ indices,
                                                       const double* __restrict__ vals, double* __restrict__ a,
                                                       double* __restrict__ status) {
  const int row = blockIdx.x;
  double* r = a + size_t(row) * npad;
  for (int j = threadIdx.x; j < npad; j += 256) r[j] = row >= n && j == row ? 1.0 : 0.0;  // identity padding
  __syncthreads();
  if (row < n)
    for (int k = indptr[row] + int(threadIdx.x); k < indptr[row + 1]; k += 256) r[indices[k]] = vals[k];
  if (row == 0 && threadIdx.x == 0) status[0] = 0.0;
}

// out = (a + a^T) / 2
__global__ __launch_bounds__(256) void spd_symmetrise_kernel(int npad, const double* __restrict__ a,
                                                             double* __restrict__ out) {
  __shared__ double t[kTile][kTs];
  const int bi = blockIdx.y * kTile, bj = blockIdx.x * kTile, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int i = ty; i < kTile; i += 8) t[i][tx] = a[size_t(bj + i) * npad + bi + tx];
  __syncthreads();
  for (int i = ty; i < kTile; i += 8)
    out[size_t(bi + i) * npad + bj + tx] = 0.5 * (a[size_t(bi + i) * npad + bj + tx] + t[tx][i]);
}

// the wavefront's 16x16 quadrant of c + X Y (32x32 in LDS, row stride kTs), TX, TY: with X^T, Y^T
template <bool TX, bool TY>
__device__ __forceinline__ d4 tile_product(const double* X, const double* Y, int qi, int qj, int lane, d4 c) {
  const int r = lane & 15, k = lane >> 4;
#pragma unroll
  for (int s = 0; s < kTile / 4; ++s) {
    const int m = 4 * s + k;
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(TX ? X[m * kTs + qi + r] : X[(qi + r) * kTs + m],
                                             TY ? Y[(qj + r) * kTs + m] : Y[m * kTs + qj + r], c, 0, 0, 0);
  }
  return c;
}

__global__ __launch_bounds__(256) void spd_step_kernel(int npad, int K, double* __restrict__ a,
                                                       double* __restrict__ f, double* __restrict__ status) {
  __shared__ double sT[kTile * kTs], sL[kTile * kTs], sR[kTile * kTs];
  __shared__ double s_col[2][kTile], s_row[2][kTile];
  const int tid = threadIdx.x, tx = tid & 31, ty = tid >> 5;
  const int I = K + blockIdx.y, J = blockIdx.x;
  if (J > I) return;  // the whole workgroup
  auto tile = [&](double* m, int i, int j) { return m + (size_t(i) * npad + j) * kTile; };
  const double* akk = tile(a, K, K);
  const double* left = tile(a, I, K);
  const double* right = tile(a, J, K);  // M_KJ above the diagonal, A_JK below
  double* out = I == K ? tile(f, K, J) : (J > K ? tile(a, I, J) : tile(a, J, I));  // F_KJ, A_IJ, M_IJ
  // A_KK in registers, four rows per thread: rows ty + 8 i, column tx
  double m[4], d[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const size_t at = size_t(ty + 8 * i) * npad + tx;
    m[i] = akk[at];
    d[i] = 1.0;
    if (I != K) sL[(ty + 8 * i) * kTs + tx] = left[at];
    if (J != K) sR[(ty + 8 * i) * kTs + tx] = right[at];
  }
  const int lane = tid & 63, wave = tid >> 6, qi = (wave >> 1) * 16, qj = (wave & 1) * 16;
  d4 c = {0, 0, 0, 0};
  if (I != K && J != K) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c[r] = out[size_t(qi + (lane >> 4) + 4 * r) * npad + qj + (lane & 15)];
  }
  bool bad = false;
  // elimination of the rows below each pivot; the columns behind it take up the inverse of the unit
  // lower factor
#pragma unroll
  for (int p = 0; p < kTile; ++p) {
    const int buf = p & 1;
    if (tx == p) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s_col[buf][ty + 8 * i] = m[i];
    }
    if (ty == (p & 7)) s_row[buf][tx] = m[p >> 3];
    __syncthreads();
    const double piv = s_row[buf][p];
    if (!(piv > 0.0) || !isfinite(piv)) bad = true;
    double ip = __builtin_amdgcn_rcp(piv);  // two Newton steps: within an ulp, a third of a division's chain
    ip = fma(ip, fma(-piv, ip, 1.0), ip);
    ip = fma(ip, fma(-piv, ip, 1.0), ip);
    const double rj = tx == p ? ip : s_row[buf][tx] * ip;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = ty + 8 * i;
      if (row > p) m[i] = (tx == p ? 0.0 : m[i]) - s_col[buf][row] * rj;
      if (row == p) d[i] = piv;
    }
  }
  // T = D^-1/2 times the inverse of the unit factor
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = ty + 8 * i;
    m[i] = (tx < row ? m[i] : (tx == row ? 1.0 : 0.0)) / sqrt(d[i]);
  }
  if (I == K && J == K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) out[size_t(ty + 8 * i) * npad + tx] = m[i];
    if (bad && tid == 0) status[0] = 1.0;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) sT[(ty + 8 * i) * kTs + tx] = m[i];
  __syncthreads();
  if (I == K) {
    c = tile_product<false, false>(sT, sR, qi, qj, lane, c);
  } else {
    const d4 z = {0, 0, 0, 0};
    const d4 l = tile_product<false, true>(sL, sT, qi, qj, lane, z);  // L_IK
    d4 g = z;                                                         // T M_KJ, or L_JK
    if (J < K) g = tile_product<false, false>(sT, sR, qi, qj, lane, z);
    if (J > K) g = tile_product<false, true>(sR, sT, qi, qj, lane, z);
    __syncthreads();  // sL and sR are read
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int at = (qi + (lane >> 4) + 4 * r) * kTs + qj + (lane & 15);
      sL[at] = -l[r];
      sR[at] = g[r];
    }
    __syncthreads();
    if (J == K)
      c = tile_product<false, false>(sL, sT, qi, qj, lane, c);
    else if (J < K)
      c = tile_product<false, false>(sL, sR, qi, qj, lane, c);
    else
      c = tile_product<false, true>(sL, sR, qi, qj, lane, c);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) out[size_t(qi + (lane >> 4) + 4 * r) * npad + qj + (lane & 15)] = c[r];
}

// inv = F^T F, tile (I, J) of the lower triangle and its transpose; the next tiles of F are loaded under
// the products
__global__ __launch_bounds__(256) void spd_product_kernel(int n, int npad, const double* __restrict__ f,
                                                          double* __restrict__ inv) {
  __shared__ double sX[kTile * kTs], sY[kTile * kTs];
  const int I = blockIdx.y, J = blockIdx.x, nt = npad / kTile;
  if (J > I) return;
  const int tid = threadIdx.x, tx = tid & 31, ty = tid >> 5;
  const int lane = tid & 63, wave = tid >> 6, qi = (wave >> 1) * 16, qj = (wave & 1) * 16;
  double x[4], y[4];
  auto load = [&](int K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t row = size_t(K * kTile + ty + 8 * i) * npad + tx;
      x[i] = f[row + I * kTile];
      y[i] = f[row + J * kTile];
    }
  };
  d4 c = {0, 0, 0, 0};
  load(I);
  for (int K = I; K < nt; ++K) {
    __syncthreads();  // the last tiles are read
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sX[(ty + 8 * i) * kTs + tx] = x[i];
      sY[(ty + 8 * i) * kTs + tx] = y[i];
    }
    if (K + 1 < nt) load(K + 1);
    __syncthreads();
    c = tile_product<true, false>(sX, sY, qi, qj, lane, c);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = I * kTile + qi + (lane >> 4) + 4 * r, j = J * kTile + qj + (lane & 15);
    if (i < n && j <= i) {
      inv[size_t(i) * n + j] = c[r];
      inv[size_t(j) * n + i] = c[r];
    }
  }
}

// lanes per row and form of the precision argument, as in fne_spmv; false: not valid
bool csr_code(int32_t precision, const void* indices, const void* vals, int& lpr, int& form) {
  lpr = (precision >> 8) & 0xff;
  if (lpr == 0) lpr = 8;
  if (lpr > 64 || (lpr & (lpr - 1))) return false;
  form = csr_form_of(precision) == kCsrFormStream && csr_stream_ok(indices, vals)
             ? 2
             : (csr_use_vec(indices, vals, lpr) ? 1 : 0);
  return true;
}

int64_t lanczos_parts(int32_t n, int lpr) { return (int64_t(n) * lpr + kLanThreads - 1) / kLanThreads; }

template <typename VT>
int lanczos_run(int n, const int32_t* indptr, const int32_t* indices, const VT* vals, int lpr, int form,
                const int64_t* diag, const double* v0, int steps, double* dinv, double* work, double* out,
                hipStream_t st) {
  const int parts = int(lanczos_parts(n, lpr));
  const int nb = std::min(kLanBlocks, (n + kLanThreads - 1) / kLanThreads);
  double* s = work;
  double* u = s + n;
  double* w = u + n;
  double* y = w + n;
  double* va = y + n;
  double* vb = va + n;
  double* norm_part = vb + n;               // [kLanBlocks]
  double* alpha = norm_part + kLanBlocks;   // [kLanSteps]
  double* beta = alpha + kLanSteps;         // [kLanSteps]
  double* joined = beta + kLanSteps;        // [8]
  double* dot_part = joined + 8;            // [parts]
  hipLaunchKernelGGL(lanczos_start_kernel<VT>, dim3(nb), dim3(kLanThreads), 0, st, n, vals, diag, v0, dinv, s, u,
                     norm_part);
  for (int k = 0; k < steps; ++k) {
    double* v = k & 1 ? vb : va;
    const double* v_prev = k == 0 ? nullptr : (k & 1 ? va : vb);
    const double* wk = k == 0 ? v0 : w;
    double* beta_out = k == 0 ? nullptr : beta + k - 1;
#define LAN(L, F)                                                                                               \
  hipLaunchKernelGGL((lanczos_mult_kernel<VT, L, F>), dim3(parts), dim3(kLanThreads), 0, st, n, indptr, indices, \
                     vals, s, u, wk, v_prev, v, y, norm_part, nb, dot_part, beta_out)
#define LAN_L(L)                \
  case L:                       \
    if (form == 2) LAN(L, 2);   \
    else if (form == 1) LAN(L, 1); \
    else LAN(L, 0);             \
    break;
    switch (lpr) {
      LAN_L(1)
      LAN_L(2)
      LAN_L(4)
      LAN_L(8)
      LAN_L(16)
      LAN_L(32)
      LAN_L(64)
    }
#undef LAN_L
#undef LAN
    const double* dots = dot_part;
    int n_dot = parts;
    if (parts > kLanParts) {
      hipLaunchKernelGGL(lanczos_join_kernel, dim3(1), dim3(kLanThreads), 0, st, dot_part, parts, joined);
      dots = joined;
      n_dot = 1;
    }
    hipLaunchKernelGGL(lanczos_update_kernel, dim3(nb), dim3(kLanThreads), 0, st, n, y, v, s, w, u, dots, n_dot,
                       norm_part, alpha + k);
  }
  hipLaunchKernelGGL(lanczos_eig_kernel, dim3(1), dim3(kLanThreads), 0, st, steps, alpha, beta, norm_part, nb, out);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

int vector_blocks(int64_t n) { return int(std::min<int64_t>(2048, (n + 255) / 256)); }

}  // namespace

extern "C" int64_t fne_lanczos_work_len(int32_t n, int32_t precision) {
  int lpr = (precision >> 8) & 0xff;
  if (lpr == 0) lpr = 8;
  if (n < 0 || lpr > 64) return -1;
  return 6 * int64_t(n) + kLanBlocks + 2 * kLanSteps + 8 + lanczos_parts(n, lpr);
}

extern "C" int fne_lanczos_max(int32_t n, const int32_t* indptr, const int32_t* indices, const void* vals,
                               int32_t precision, const int64_t* diag, const double* v0, int32_t steps, double* dinv,
                               double* work, int64_t work_len, double* out, fne_stream_t stream) {
  if (n <= 0 || steps < 1 || steps > kLanSteps) {
    fne_set_error("fne_lanczos_max: need n > 0 and 1 to 64 steps");
    return FNE_EINVAL;
  }
  if (!indptr || !indices || !vals || !diag || !v0 || !dinv || !work || !out) {
    fne_set_error("fne_lanczos_max: null pointer");
    return FNE_EINVAL;
  }
  int lpr, form;
  if (!csr_code(precision, indices, vals, lpr, form) || work_len < fne_lanczos_work_len(n, precision)) {
    fne_set_error("fne_lanczos_max: lanes per row must be a power of two <= 64, work fne_lanczos_work_len");
    return FNE_EINVAL;
  }
  const int prec = precision & 0xff;
  hipStream_t s = (hipStream_t)stream;
  if (prec == FNE_FP64)
    return lanczos_run<double>(n, indptr, indices, (const double*)vals, lpr, form, diag, v0, steps, dinv, work, out, s);
  if (prec == FNE_FP32)
    return lanczos_run<float>(n, indptr, indices, (const float*)vals, lpr, form, diag, v0, steps, dinv, work, out, s);
  fne_set_error("fne_lanczos_max: precision must be FNE_FP64 or FNE_FP32");
  return FNE_EINVAL;
}

extern "C" int fne_smoother_weights(int32_t n, const double* dinv, const double* lam, double wd_factor,
                                    const double* cheb_factors, int32_t n_cheb, double* wd, double* wcheb,
                                    fne_stream_t stream) {
  if (n < 0 || n_cheb < 0 || n_cheb > 8 || (n_cheb > 0 && (!cheb_factors || !wcheb))) {
    fne_set_error("fne_smoother_weights: need n >= 0 and at most 8 Chebyshev factors");
    return FNE_EINVAL;
  }
  if (n == 0) return FNE_OK;
  if (!dinv || !lam || !wd) {
    fne_set_error("fne_smoother_weights: null pointer");
    return FNE_EINVAL;
  }
  SmootherFactors f{};
  f.wd = wd_factor;
  f.n = n_cheb;
  for (int k = 0; k < n_cheb; ++k) f.cheb[k] = cheb_factors[k];
  hipLaunchKernelGGL(smoother_weights_kernel, dim3(vector_blocks(n)), dim3(kLanThreads), 0, (hipStream_t)stream, n,
                     dinv, lam, f, wd, wcheb);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

extern "C" int fne_amg_transfers(int32_t nnz, const double* p, const int64_t* perm, double* r, void* p_cycle,
                                 void* r_cycle, int32_t precision, fne_stream_t stream) {
  if (nnz < 0 || (precision != FNE_FP64 && precision != FNE_FP32)) {
    fne_set_error("fne_amg_transfers: invalid size or precision");
    return FNE_EINVAL;
  }
  if (nnz == 0) return FNE_OK;
  if (!p || !perm || !r || !p_cycle || !r_cycle) {
    fne_set_error("fne_amg_transfers: null pointer");
    return FNE_EINVAL;
  }
  const dim3 grid(vector_blocks(nnz));
  if (precision == FNE_FP64)
    hipLaunchKernelGGL(transfers_kernel<double>, grid, dim3(256), 0, (hipStream_t)stream, nnz, p, perm, r,
                       (double*)p_cycle, (double*)r_cycle);
  else
    hipLaunchKernelGGL(transfers_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, nnz, p, perm, r,
                       (float*)p_cycle, (float*)r_cycle);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

extern "C" int fne_amg_symmetrise(int32_t nnz, const double* c, const int64_t* perm, double* a, void* a_cycle,
                                  int32_t precision, fne_stream_t stream) {
  if (nnz < 0 || (precision != FNE_FP64 && precision != FNE_FP32)) {
    fne_set_error("fne_amg_symmetrise: invalid size or precision");
    return FNE_EINVAL;
  }
  if (nnz == 0) return FNE_OK;
  if (!c || !perm || !a || a == c) {
    fne_set_error("fne_amg_symmetrise: null pointer, or the output is the input");
    return FNE_EINVAL;
  }
  const dim3 grid(vector_blocks(nnz));
  if (precision == FNE_FP64)
    hipLaunchKernelGGL(symmetrise_kernel<double>, grid, dim3(256), 0, (hipStream_t)stream, nnz, c, perm, a,
                       (double*)a_cycle);
  else
    hipLaunchKernelGGL(symmetrise_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, nnz, c, perm, a,
                       (float*)a_cycle);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

extern "C" int64_t fne_spd_inverse_work_len(int32_t n) {
  if (n < 0) return -1;
  const int64_t npad = (int64_t(n) + kTile - 1) / kTile * kTile;
  return 2 * npad * npad;
}

extern "C" int fne_spd_inverse(int32_t n, const int32_t* indptr, const int32_t* indices, const double* vals,
                               double* work, int64_t work_len, double* inv, double* status, fne_stream_t stream) {
  if (n < 0 || n > 46340) {  // n^2 entries with 32-bit offsets, as the cycle's dense operator has
    fne_set_error("fne_spd_inverse: need 0 <= n <= 46340");
    return FNE_EINVAL;
  }
  if (!status || (n > 0 && (!indptr || !indices || !vals || !work || !inv))) {
    fne_set_error("fne_spd_inverse: null pointer");
    return FNE_EINVAL;
  }
  if (work_len < fne_spd_inverse_work_len(n)) {
    fne_set_error("fne_spd_inverse: work needs fne_spd_inverse_work_len doubles");
    return FNE_EINVAL;
  }
  if (n == 0) return FNE_OK;
  hipStream_t s = (hipStream_t)stream;
  const int nt = (n + kTile - 1) / kTile, npad = nt * kTile;
  double* a = work;
  double* b = work + size_t(npad) * npad;
  hipLaunchKernelGGL(spd_rows_kernel, dim3(npad), dim3(256), 0, s, n, npad, indptr, indices, vals, b, status);
  hipLaunchKernelGGL(spd_symmetrise_kernel, dim3(nt, nt), dim3(256), 0, s, npad, b, a);
  for (int k = 0; k < nt; ++k)
    hipLaunchKernelGGL(spd_step_kernel, dim3(nt, nt - k), dim3(256), 0, s, npad, k, a, b, status);
  hipLaunchKernelGGL(spd_product_kernel, dim3(nt, nt), dim3(256), 0, s, n, npad, b, inv);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}
