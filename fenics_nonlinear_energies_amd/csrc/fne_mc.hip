// Plane-strain Mohr-Coulomb on P2/P4 triangles (rows A4/A5 of the hot path).
//
// Element energy (slope_stability/jax/jax_energy.py:45-142): per quadrature point q,
// eps = B_q u_e (engineering shear), sigma_tr = C eps, principal values s1,2 = m +- r with
// r = sqrt(d^2 + tau^2 + reg^2); elastic if alpha s1 - beta s2 - kappa <= 0, else a return
// to the yield line along z = A^-1 n (apex if s1 < s2 afterwards); sigma is rebuilt with the
// trial principal direction; psi = sigma.eps - 1/2 sigma.S sigma; E_e = sum_q w_q psi_q.
// The gradient is sum_q w_q B_q^T sigma_q and the Hessian sum_q w_q B_q^T D_q B_q with
// D = d sigma / d eps derived by hand (line return: chain rule through (m, r, theta); apex:
// zero), symmetrised.
//
// Two kernels per Newton-step assembly:
//   mc_elem_kernel         one wavefront evaluates 3 elements at a time: FP64 per quadrature point
//                          (strain, return mapping, energy, stress) on 3 x n_q lanes; the element
//                          gradients and Hessians by v_mfma 16x16x4 into a per-element scratch
//                          (element order of the plan).
//   mc_unit_gather_kernel  8 or 16 lanes per row, or pair of rows of a node: for each incident
//                          element (fixed ascending order) lane c adds the entries of node c into
//                          an LDS copy of the CSR rows at the precomputed byte positions; the rows
//                          are then written once.  No atomics: results are bitwise reproducible.
//                          Plans without row units: row_gather_kernel, the same row by row.
#include "fne_common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

constexpr int kMcMaxQ = 21;  // 3 elements x 21 points fill one wavefront
constexpr int kMcEpw = 3;    // elements per wavefront iteration
constexpr int kMcWaves = kBlock / 64;
// lanes per row group in the row gather: lane c < NL/2 carries element columns 2c and 2c+1, so
// 8 lanes cover a 12-column element row and 16 the 30 of P4
__host__ __device__ constexpr int mc_row_lanes(int nl) {
  return nl <= 16 ? 8 : 16;
}
constexpr unsigned char kPosNone = 255;

typedef float mc_f4 __attribute__((ext_vector_type(4)));
typedef double mc_d4 __attribute__((ext_vector_type(4)));

struct McConst {
  double C00, C01, C22;  // C = [[C00, C01, 0], [C01, C00, 0], [0, 0, C22]]
  double S00, S01, S22;  // S = C^-1 in plane strain
  double alpha, beta, kappa, reg;
  double z1, z2, inv_nz; // return direction z = A^-1 n, n = (alpha, -beta), and 1 / (n.z)
  // line return: d(mean) = am dm + ar dr and d(radius) = bm dm + br dr of the trial (m, r)
  double am, ar, bm, br;
  double s_apex;
  int mode;              // 0 full Mohr-Coulomb, 1 elastic
};

// evaluated on the host once per launch (a sine, a cosine and ten divisions per thread otherwise)
McConst mc_const(const double* prm, int mode) {
  McConst k;
  const double E = prm[0], nu = prm[1], phi_deg = prm[2], coh = prm[3];
  const double lam = E * nu / ((1.0 + nu) * (1.0 - 2.0 * nu));
  const double mu = E / (2.0 * (1.0 + nu));
  k.C00 = lam + 2.0 * mu;
  k.C01 = lam;
  k.C22 = mu;
  k.S00 = (1.0 - nu * nu) / E;
  k.S01 = -(nu * (1.0 + nu)) / E;
  k.S22 = 1.0 / mu;
  const double phi = phi_deg * (M_PI / 180.0);
  const double sphi = sin(phi), cphi = cos(phi);
  k.alpha = 1.0 + sphi;
  k.beta = 1.0 - sphi;
  k.kappa = 2.0 * coh * cphi;
  k.reg = prm[4];
  const double A11 = k.S00, A12 = k.S01, A22 = k.S00;
  const double n1 = k.alpha, n2 = -k.beta;
  const double det = A11 * A22 - A12 * A12;
  k.z1 = (A22 * n1 - A12 * n2) / det;
  k.z2 = (-A12 * n1 + A11 * n2) / det;
  const double nz = n1 * k.z1 + n2 * k.z2;
  k.inv_nz = 1.0 / nz;
  const double P11 = 1.0 - k.z1 * n1 / nz, P12 = -k.z1 * n2 / nz;
  const double P21 = -k.z2 * n1 / nz, P22 = 1.0 - k.z2 * n2 / nz;
  k.am = 0.5 * (P11 + P12 + P21 + P22);
  k.ar = 0.5 * (P11 - P12 + P21 - P22);
  k.bm = 0.5 * (P11 + P12 - P21 - P22);
  k.br = 0.5 * (P11 - P12 - P21 + P22);
  const double den = fabs(k.alpha - k.beta) > 1.0e-14 ? k.alpha - k.beta : 1.0;
  k.s_apex = k.kappa / den;
  k.mode = mode;
  return k;
}

// One quadrature point: energy density, stress and (optionally) the symmetric tangent
// D = [d00 d01 d02 d11 d12 d22] (Voigt, engineering shear).
template <bool WANT_D>
__device__ __forceinline__ double mc_point(const McConst& k, double e0, double e1, double e2, double sig[3],
                                           double D[6]) {
  const double st0 = k.C00 * e0 + k.C01 * e1;
  const double st1 = k.C01 * e0 + k.C00 * e1;
  const double st2 = k.C22 * e2;
  bool elastic = k.mode == 1;
  double m = 0.0, d = 0.0, r = 0.0, s1 = 0.0, s2 = 0.0;
  if (!elastic) {
    m = 0.5 * (st0 + st1);
    d = 0.5 * (st0 - st1);
    r = sqrt(d * d + st2 * st2 + k.reg * k.reg);
    s1 = m + r;
    s2 = m - r;
    elastic = k.alpha * s1 - k.beta * s2 - k.kappa <= 0.0;
  }
  if (elastic) {
    sig[0] = st0;
    sig[1] = st1;
    sig[2] = st2;
    if (WANT_D) {
      D[0] = k.C00;
      D[1] = k.C01;
      D[2] = 0.0;
      D[3] = k.C00;
      D[4] = 0.0;
      D[5] = k.C22;
    }
  } else {
    const double n1 = k.alpha, n2 = -k.beta;
    const double lam_mc = (n1 * s1 + n2 * s2 - k.kappa) * k.inv_nz;
    const double s1l = s1 - lam_mc * k.z1;
    const double s2l = s2 - lam_mc * k.z2;
    const bool line = s1l >= s2l;
    const double s1p = line ? s1l : k.s_apex;
    const double s2p = line ? s2l : k.s_apex;
    const double mp = 0.5 * (s1p + s2p);
    const double rp = 0.5 * (s1p - s2p);
    // 2 theta = atan2(2 tau, sxx - syy): cos/sin from the trial deviator (atan2(0,0) = 0)
    const double r0 = sqrt(d * d + st2 * st2);
    const double ir0 = r0 > 0.0 ? 1.0 / r0 : 0.0;
    const double c2 = r0 > 0.0 ? d * ir0 : 1.0;
    const double sn2 = r0 > 0.0 ? st2 * ir0 : 0.0;
    sig[0] = mp + rp * c2;
    sig[1] = mp - rp * c2;
    sig[2] = rp * sn2;
    if (WANT_D) {
      if (!line) {
#pragma unroll
        for (int i = 0; i < 6; ++i) D[i] = 0.0;
      } else {
        const double am = k.am, ar = k.ar, bm = k.bm, br = k.br;
        const double ir = r > 0.0 ? 1.0 / r : 0.0;
        // derivatives with respect to the trial stress (sxx, syy, txy)
        const double dr[3] = {0.5 * d * ir, -0.5 * d * ir, st2 * ir};
        const double dph[3] = {0.5 * sn2 * ir0, -0.5 * sn2 * ir0, -c2 * ir0};
        const double dm[3] = {0.5, 0.5, 0.0};
        double Ds[3][3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const double dmp = am * dm[j] + ar * dr[j];
          const double drp = bm * dm[j] + br * dr[j];
          Ds[0][j] = dmp + c2 * drp + rp * sn2 * dph[j];
          Ds[1][j] = dmp - c2 * drp - rp * sn2 * dph[j];
          Ds[2][j] = sn2 * drp - rp * c2 * dph[j];
        }
        // D = Ds * C, then symmetrise
        double Dm[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          Dm[i][0] = Ds[i][0] * k.C00 + Ds[i][1] * k.C01;
          Dm[i][1] = Ds[i][0] * k.C01 + Ds[i][1] * k.C00;
          Dm[i][2] = Ds[i][2] * k.C22;
        }
        D[0] = Dm[0][0];
        D[1] = 0.5 * (Dm[0][1] + Dm[1][0]);
        D[2] = 0.5 * (Dm[0][2] + Dm[2][0]);
        D[3] = Dm[1][1];
        D[4] = 0.5 * (Dm[1][2] + Dm[2][1]);
        D[5] = Dm[2][2];
      }
    }
  }
  const double Ss0 = k.S00 * sig[0] + k.S01 * sig[1];
  const double Ss1 = k.S01 * sig[0] + k.S00 * sig[1];
  const double Ss2 = k.S22 * sig[2];
  return sig[0] * e0 + sig[1] * e1 + sig[2] * e2 - 0.5 * (sig[0] * Ss0 + sig[1] * Ss1 + sig[2] * Ss2);
}

__device__ __forceinline__ mc_f4 mfma16(float a, float b, mc_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mc_d4 mfma16(double a, double b, mc_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// Result layout of the 16x16x4 products: lane l holds D[row][l % 16] in slot r, with
// row = 4 (l / 16) + r for the FP32 form and row = l / 16 + 4 r for the FP64 form.
template <typename T> struct Vec4;
template <> struct Vec4<float> {
  typedef mc_f4 type;
  static __device__ __forceinline__ int row(int kk, int r) { return 4 * kk + r; }
};
template <> struct Vec4<double> {
  typedef mc_d4 type;
  static __device__ __forceinline__ int row(int kk, int r) { return kk + 4 * r; }
};

template <typename T> struct Pair;
template <> struct Pair<float> {
  typedef float2 type;
  static __device__ __forceinline__ float2 zero() { return make_float2(0.f, 0.f); }
};
template <> struct Pair<double> {
  typedef double2 type;
  static __device__ __forceinline__ double2 zero() { return make_double2(0.0, 0.0); }
};

__device__ __forceinline__ float mc_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double mc_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// blocks of the element kernel, each with `rounds` rounds of consecutive elements
struct McBlocks {
  int rounds = 1, all = 1;
};

// LDS of one wavefront
// NQ: points of the matrix products' K range; those beyond n_q stay zero
template <int NQ, typename HT, bool WG, bool WH, bool HV>
struct McWaveLds {
  double u[kMcEpw][32];                    // element DOF values
  double v[HV ? kMcEpw : 1][32];           // direction of a Hessian product
  double geo[kMcEpw][8];                   // K00 K01 K10 K11 |detJ|
  double P[WG ? kMcEpw : 1][NQ][4];        // w sigma_{ia} K_ag of the points, i-major
  HT M[WH ? kMcEpw * NQ * 12 : 2];         // pulled-back tangents [t][q][g][xx, xy, yy][h]
};

// Values of an element matrix in the scratch, [n][m][j][i]: rows (n, i), columns (m, j).  The node rows
// of P4 have 16 columns: 256 B (FP32) or 512 B at multiples of that, so that the row gather reads two
// lines of 128 B for each instead of 2.75 (32,000 elements, assembly 140 -> 127 us).  Plans without
// row units store row (n, i) as kMcNodeRow / 2 values in the order of its columns instead (BY_ROWS: a
// branch at run time spills two registers more, 98,000 elements 370 -> 376 us).
template <int NN>
constexpr int kMcNodeRow = 4 * (NN == 15 ? 16 : NN);
template <int NN>
constexpr int kMcMatrix = NN * kMcNodeRow<NN>;

// Element energies, gradients and Hessians; NN nodes per element (6: P2, 15: P4).
//
// Bound by latency and issue (FP64 return mapping), then by the matrix units and the stores.  Per
// point the tangent is pulled back to the reference triangle in FP64 and rounded once,
//   M^{ij}_{gh} = sum_ab w K_ag D^{ij}_ab K_bh,
//   H^{ij}[n][m] = sum_{q,g} dphi_n,g(q) sum_h M^{ij}_{gh}(q) dphi_m,h(q),
// so the first factor is the same for all elements and the second is two multiply-adds.
//   P4: four 16x16 tiles (xx, xy, yx, yy) over K = (q, g); yx is the xy product with its factors
//       exchanged, so that a lane ends with all four components of node pairs.
//   P2: one 16x16 tile of the 12 DOFs over K = (q, i, g): n_q products instead of 4 n_q / 2.
// Both leave the element matrix as [n][m][j][i] (rows (n, i), columns (m, j)): the four values of a
// node pair side by side, written and read as one vector.
// K ranges padded with zeros make every LDS address a base plus a constant; clamped points cost 31
// registers and spills.  128 registers, four wavefronts per SIMD.  With gradient and energy: P4 FP32,
// 98,000 elements 221 -> 154 us (matrix units busy 60, VALU 60 of it, 376 MB stored); P2 FP64, 21,978
// elements, Hessian alone 65 -> 39 us, gradient alone 11.8 -> 10.8; product with a direction, P4,
// 32,000 elements 46 -> 22 us.
template <int NN, int NS, typename HT, bool WE, bool WG, bool WH, bool HV, bool BY_ROWS>
__global__ __launch_bounds__(kBlock, WH && sizeof(HT) == 8 && (WG || (NN == 15 && NS == 11)) ? 3 : 4) void mc_elem_kernel(
    fne_plan_desc d, McConst k, const double* __restrict__ x, const double* __restrict__ dvals,
    const double* __restrict__ f, const double* __restrict__ vin, EnergySum energy,
    double* __restrict__ eelem, double* __restrict__ gbuf, HT* __restrict__ hbuf, McBlocks B) {
  constexpr int NL = 2 * NN;
  constexpr bool kOneTile = NL <= 16;
  typedef typename Vec4<HT>::type V4;
  typedef typename Pair<HT>::type HT2;
  // reference gradients [q][n][g], zero beyond the last point
  constexpr int kCols = kOneTile ? 8 : 16, kPoints = 2 * NS;
  __shared__ __align__(16) double sTab[kPoints * NN * 2];
  // in the type of the element matrices, zero beyond the last node too
  __shared__ __align__(16) HT sTabH[WH ? kPoints * kCols * 2 : 2];
  __shared__ double sW[kMcMaxQ];
  __shared__ __align__(16) McWaveLds<kPoints, HT, WG, WH, HV> sWave[kMcWaves];
  const int nq = d.nq, ne = d.n_elem;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  McWaveLds<kPoints, HT, WG, WH, HV>& L = sWave[wave];
  const int block = blockIdx.x;
  constexpr int kRound = kMcWaves * kMcEpw;  // elements of a block's round
  const int first = block * B.rounds * kRound + wave * kMcEpw;
  const int end = min(ne, (block + 1) * B.rounds * kRound);
  double es = 0.0, ec = 0.0;
  // a round of a wavefront: three elements' DOF codes, then their values and geometry, loaded one
  // round ahead (the first under the table's load)
  constexpr int kVals = (kMcEpw * NL + 63) / 64;
  int code[kVals];
  double val[kVals], vdir[HV ? kVals : 1], geo = 0.0;
  auto load_codes = [&](int base) {
#pragma unroll
    for (int v = 0; v < kVals; ++v) {
      const int i = lane + 64 * v, t = i / NL, c = i - t * NL;
      code[v] = i < kMcEpw * NL && base + t < ne ? d.edof[size_t(c) * ne + base + t] : -1;
    }
  };
  auto load_values = [&](int base) {
#pragma unroll
    for (int v = 0; v < kVals; ++v) {
      val[v] = code[v] >= 0 ? gather_dof(code[v], d.n_free, x, dvals) : 0.0;
      if (HV) vdir[v] = code[v] >= 0 && code[v] < d.n_free ? vin[code[v]] : 0.0;  // zero on constrained DOFs
    }
    const int t = lane / 5, c = lane - 5 * t;
    if (lane < kMcEpw * 5) geo = base + t < ne ? d.egeo[size_t(c) * ne + base + t] : (c == 4 ? 0.0 : 1.0);
  };
  if (first < end) load_codes(first);
  for (int i = threadIdx.x; i < kPoints * NN * 2; i += kBlock) sTab[i] = i < nq * NN * 2 ? d.qdata[nq + i] : 0.0;
  if constexpr (WG) {
    for (int i = lane; i < kMcEpw * kPoints * 4; i += 64) (&L.P[0][0][0])[i] = 0.0;
  }
  if constexpr (WH) {
    for (int i = lane; i < kMcEpw * kPoints * 12; i += 64) L.M[i] = HT(0);
    for (int i = threadIdx.x; i < kPoints * kCols * 2; i += kBlock) {
      const int qs = i / (2 * kCols), n = (i >> 1) & (kCols - 1);
      sTabH[i] = qs < nq && n < NN ? HT(d.qdata[nq + (qs * NN + n) * 2 + (i & 1)]) : HT(0);
    }
  }
  for (int i = threadIdx.x; i < nq; i += kBlock) sW[i] = d.qdata[i];
  if (first < end) load_values(first);
  __syncthreads();
  const int c15 = lane & 15, kk = lane >> 4;
  const bool has_eps = d.n_geo >= 5 + 3 * nq;
  const int t = lane / nq, q = lane - t * nq;
  for (int base = first; base < end; base += kRound) {
#pragma unroll
    for (int v = 0; v < kVals; ++v) {
      const int i = lane + 64 * v, tv = i / NL;
      if (i < kMcEpw * NL) {
        L.u[tv][i - tv * NL] = val[v];
        if (HV) L.v[tv][i - tv * NL] = vdir[v];
      }
    }
    if (lane < kMcEpw * 5) L.geo[lane / 5][lane % 5] = geo;
    const int next = base + kRound;
    if (next < end) load_codes(next);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // ---- quadrature points: lanes t * nq + q
    const bool point = t < kMcEpw && base + t < ne;
    double wpsi = 0.0;
    if (point) {
      const int e = base + t;
      double U00 = 0.0, U01 = 0.0, U10 = 0.0, U11 = 0.0;  // U[i][g] = sum_n u_{n,i} dphi_n/dxi_g
      double V00 = 0.0, V01 = 0.0, V10 = 0.0, V11 = 0.0;
#pragma unroll 3
      for (int n = 0; n < NN; ++n) {
        const double2 gr = *reinterpret_cast<const double2*>(sTab + (q * NN + n) * 2);
        const double2 u = *reinterpret_cast<const double2*>(&L.u[t][2 * n]);
        U00 = fma(u.x, gr.x, U00);
        U01 = fma(u.x, gr.y, U01);
        U10 = fma(u.y, gr.x, U10);
        U11 = fma(u.y, gr.y, U11);
        if (HV) {
          const double2 v = *reinterpret_cast<const double2*>(&L.v[t][2 * n]);
          V00 = fma(v.x, gr.x, V00);
          V01 = fma(v.x, gr.y, V01);
          V10 = fma(v.y, gr.x, V10);
          V11 = fma(v.y, gr.y, V11);
        }
      }
      const double K00 = L.geo[t][0], K01 = L.geo[t][1], K10 = L.geo[t][2], K11 = L.geo[t][3];
      double e0 = K00 * U00 + K01 * U01;
      double e1 = K10 * U10 + K11 * U11;
      double e2 = (K10 * U00 + K11 * U01) + (K00 * U10 + K01 * U11);
      if (has_eps) {
        const size_t o = size_t(5 + 3 * q) * ne + e;
        e0 -= d.egeo[o];
        e1 -= d.egeo[o + ne];
        e2 -= d.egeo[o + 2 * size_t(ne)];
      }
      double sig[3], D[6];
      const double w = sW[q] * L.geo[t][4];
      wpsi = w * mc_point<WH || HV>(k, e0, e1, e2, sig, D);
      if (d.eweight) wpsi *= d.eweight[e];
      if (WE) acc_add(es, ec, wpsi);
      if (HV) {  // the stress of the direction
        const double v0 = K00 * V00 + K01 * V01;
        const double v1 = K10 * V10 + K11 * V11;
        const double v2 = (K10 * V00 + K11 * V01) + (K00 * V10 + K01 * V11);
        sig[0] = D[0] * v0 + D[1] * v1 + D[2] * v2;
        sig[1] = D[1] * v0 + D[3] * v1 + D[4] * v2;
        sig[2] = D[2] * v0 + D[4] * v1 + D[5] * v2;
      }
      if (WG) {
        const double sx0 = w * sig[0], sy1 = w * sig[1], sxy = w * sig[2];
        L.P[t][q][0] = sx0 * K00 + sxy * K10;  // i = x, g = 0
        L.P[t][q][1] = sx0 * K01 + sxy * K11;  // i = x, g = 1
        L.P[t][q][2] = sxy * K00 + sy1 * K10;  // i = y, g = 0
        L.P[t][q][3] = sxy * K01 + sy1 * K11;  // i = y, g = 1
      }
      if constexpr (WH) {
        // D^{xx} = [d00 d02; d02 d22], D^{xy} = [d02 d01; d22 d12], D^{yy} = [d22 d12; d12 d11] over
        // the physical derivatives of the row's and the column's shape function; M = w K^T D K
        const double Dij[3][4] = {{D[0], D[2], D[2], D[5]}, {D[2], D[1], D[5], D[4]}, {D[5], D[4], D[4], D[3]}};
        const double wK00 = w * K00, wK01 = w * K01, wK10 = w * K10, wK11 = w * K11;
#pragma unroll
        for (int ij = 0; ij < 3; ++ij) {
          const double x0 = fma(Dij[ij][1], K10, Dij[ij][0] * K00), x1 = fma(Dij[ij][1], K11, Dij[ij][0] * K01);
          const double y0 = fma(Dij[ij][3], K10, Dij[ij][2] * K00), y1 = fma(Dij[ij][3], K11, Dij[ij][2] * K01);
          HT* M = L.M + (t * kPoints + q) * 12 + 2 * ij;
          M[0] = HT(fma(wK10, y0, wK00 * x0));
          M[1] = HT(fma(wK10, y1, wK00 * x1));
          M[6] = HT(fma(wK11, y0, wK01 * x0));
          M[7] = HT(fma(wK11, y1, wK01 * x1));
        }
      }
    }
    if (eelem) {  // lane t sums element t's points in order
      double s = 0.0;
      for (int qq = 0; qq < nq; ++qq) s += __shfl(wpsi, min(lane * nq + qq, 63));
      if (lane < kMcEpw && base + lane < ne) eelem[base + lane] = s;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (next < end) load_values(next);
    if (WG) {
      // element gradients: [n][(q,g)] x [(q,g)][(t,i)] in FP64, the three elements' six columns at once
      // (columns beyond the three elements repeat the last one's and are not stored)
      const int tc = c15 >> 1;
      const bool col = tc < kMcEpw;
      // opaque, here and below: the table is read again for every element instead of being hoisted into
      // registers, which would spill
      int tcol = ((kk >> 1) * NN + min(c15, NN - 1)) * 2 + (kk & 1);
      asm volatile("" : "+v"(tcol));
      const double* Pk = &L.P[min(tc, kMcEpw - 1)][kk >> 1][2 * (c15 & 1) + (kk & 1)];
      mc_d4 ag = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < NS; ++s) {  // K rows 4 s + kk = 2 q + g
        const double a = sTab[s * NN * 4 + tcol];
        const double b = Pk[s * 8];
        ag = mfma16(a, b, ag);
      }
      if (col) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = Vec4<double>::row(kk, r);
          if (n < NN) gbuf[size_t(base + tc) * 32 + 2 * n + (c15 & 1)] = ag[r];
        }
      }
    }
    if constexpr (WH) {
#pragma unroll 1  // 154 us against 159 unrolled (12 registers spill)
      for (int te = 0; te < kMcEpw; ++te) {  // beyond the last element: into the scratch's padding
        HT* H = hbuf + size_t(base + te) * kMcMatrix<NN>;
        const HT* M = L.M + te * kPoints * 12;
        int tcol = (kOneTile ? c15 >> 1 : (kk >> 1) * kCols + c15) * 2;
        asm volatile("" : "+v"(tcol));
        if constexpr (kOneTile) {
          // lane: column (m, j) and K row (i, g) of point s; its row (n, i') of the first factor
          // has the same shape function, n = m, and i' = j
          const int m = c15 >> 1, j = c15 & 1, i = kk >> 1, g = kk & 1;
          const bool in = m < NN;
          // M^{ij}_{g0}, M^{ij}_{g1}; M^{yx}_{gh} = M^{xy}_{hg}
          const HT* M0 = M + (i > j ? 2 + g : 6 * g + 2 * (i + j));
          const int m1 = i > j ? 6 : 1;
          V4 acc = {0, 0, 0, 0};
#pragma unroll 4
          for (int qs = 0; qs < kPoints; ++qs) {
            const HT2 gr = *reinterpret_cast<const HT2*>(sTabH + qs * kCols * 2 + tcol);
            const HT b = mc_fma(M0[qs * 12 + m1], gr.y, M0[qs * 12] * gr.x);
            acc = mfma16(i == j ? (g ? gr.y : gr.x) : HT(0), b, acc);
          }
          if (in) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = Vec4<HT>::row(kk, r);  // 2 n + i
              const int to = BY_ROWS ? (row & 1) * (kMcNodeRow<NN> / 2) + c15 : c15 * 2 + (row & 1);
              if (row < NL) H[(row >> 1) * kMcNodeRow<NN> + to] = acc[r];
            }
          }
        } else {
          const HT* Mk = M + (kk >> 1) * 12 + 6 * (kk & 1);
          V4 axx = {0, 0, 0, 0}, axy = {0, 0, 0, 0}, ayx = {0, 0, 0, 0}, ayy = {0, 0, 0, 0};
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const HT2* Mq = reinterpret_cast<const HT2*>(Mk + s * 24);  // K row 4 s + kk = 2 q + g
            const HT2 mxx = Mq[0], mxy = Mq[1], myy = Mq[2];
            const HT2 gr = *reinterpret_cast<const HT2*>(sTabH + s * kCols * 4 + tcol);
            const HT h0 = gr.x, h1 = gr.y;
            const HT a = (kk & 1) ? h1 : h0;
            const HT bxy = mc_fma(mxy.y, h1, mxy.x * h0);
            axx = mfma16(a, mc_fma(mxx.y, h1, mxx.x * h0), axx);
            axy = mfma16(a, bxy, axy);
            ayx = mfma16(bxy, a, ayx);
            ayy = mfma16(a, mc_fma(myy.y, h1, myy.x * h0), ayy);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {  // column 15 is zero
            const int n = Vec4<HT>::row(kk, r);
            if (n < NN) {
              if constexpr (BY_ROWS) {
                HT2* to = reinterpret_cast<HT2*>(H + n * kMcNodeRow<NN>) + c15;
                to[0] = HT2{axx[r], axy[r]};
                to[kMcNodeRow<NN> / 4] = HT2{ayx[r], ayy[r]};
              } else {
                V4 v = {axx[r], ayx[r], axy[r], ayy[r]};
                *reinterpret_cast<V4*>(H + n * kMcNodeRow<NN> + c15 * 4) = v;
              }
            }
          }
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (WE) {
    if (f) {
      const int all = B.all * kBlock;
      for (int i = block * kBlock + threadIdx.x; i < d.n_free; i += all) acc_add(es, ec, -(f[i] * x[i]));
    }
    block_energy(energy, block, es, ec);
  }
}

// Row gather of element matrices stored row by row: tetrahedral plans without node patches and
// Mohr-Coulomb plans without row units.  A group of mc_row_lanes(NL) lanes owns kRB consecutive CSR rows;
// lane c < NL/2 handles the element columns 2c and 2c+1 (paired loads).  inc[it] = element * 32 + local row
// lists the incidences of every row (rows consecutive, elements ascending); pos[it*32 + c] is the
// position of the element's local column c inside the row (255 = constrained).  The incidences of the
// batch are read in one load (lane j holds item j), up to 8 items' element rows and positions are
// fetched together and then added in item order into LDS copies of the rows, which are written once.
// Every CSR entry therefore sums its contributions in a fixed order.  One row per group for 12 columns
// (320x16x16 beam: 0.335 ms; 0.37 with 2 rows, 0.40 with 4), two for the 30 of P4 (98,000 elements: 0.50 ms;
// 0.55 with 1, 0.52 with 4).
template <int NL>
constexpr int kRowStride = NL == 30 ? kMcNodeRow<15> / 2 : NL;  // of an element matrix
template <int NL>
constexpr int kRowBatch = NL == 30 ? 2 : 1;

template <int NL, typename HT, bool WG, bool WH>
__global__ __launch_bounds__(kBlock) void row_gather_kernel(fne_plan_desc d, const HT* __restrict__ hbuf,
                                                            const double* __restrict__ gbuf,
                                                            const double* __restrict__ f,
                                                            double* __restrict__ g, HT* __restrict__ vals) {
  extern __shared__ __align__(16) unsigned char mc_smem[];
  constexpr int kL = mc_row_lanes(NL), kRB = kRowBatch<NL>, kRowsBlk = (kBlock / kL) * kRB, kPf = 8;
  typedef typename Pair<HT>::type HT2;
  const int cap = (d.max_row_len + 1) & ~1;
  const int grp = threadIdx.x / kL;
  const int c = threadIdx.x & (kL - 1);
  HT* sRows = reinterpret_cast<HT*>(mc_smem) + size_t(grp) * kRB * cap;
  const int r0 = xcd_remap(blockIdx.x, gridDim.x) * kRowsBlk + grp * kRB;
  if (r0 >= d.n_free) return;  // uniform over the lane group; no block-level barrier below
  const int nr = min(kRB, d.n_free - r0);
  const unsigned char* pos = reinterpret_cast<const unsigned char*>(d.pitem);
  const unsigned int* inc = reinterpret_cast<const unsigned int*>(d.inc);
  const int ip_l = c <= nr && WH ? d.indptr[r0 + c] : 0;
  const int ic_l = c <= nr ? d.inc_ptr[r0 + c] : 0;
  int kb[kRB + 1], ib[kRB + 1];
#pragma unroll
  for (int t = 0; t <= kRB; ++t) {
    kb[t] = __shfl(ip_l, t < nr ? t : nr, kL);
    ib[t] = __shfl(ic_l, t < nr ? t : nr, kL);
  }
  if (WH) {
#pragma unroll
    for (int t = 0; t < kRB; ++t)
      if (t < nr)
        for (int j = c; j < kb[t + 1] - kb[t]; j += kL) sRows[t * cap + j] = HT(0);
  }
  __builtin_amdgcn_wave_barrier();
  double gacc = 0.0;  // lane t < nr: gradient of row r0 + t
  for (int base = ib[0]; base < ib[nr]; base += kL) {
    const int nb = min(kL, ib[nr] - base);
    const unsigned int mine = c < nb ? inc[base + c] : 0u;
    int myslot = 0;
#pragma unroll
    for (int t = 1; t < kRB; ++t)
      if (t < nr && base + c >= ib[t]) myslot = t;
    if (WG) {
      const double gv = c < nb ? gbuf[size_t(mine >> 5) * 32 + (mine & 31u)] : 0.0;
      for (int j = 0; j < nb; ++j) {
        const double v = __shfl(gv, j, kL);
        const int t = __shfl(myslot, j, kL);
        if (c == t) gacc += v;
      }
    }
    if (WH) {
      for (int j0 = 0; j0 < nb; j0 += kPf) {
        HT2 v[kPf];
        unsigned int pp[kPf];
        int sl[kPf];
#pragma unroll
        for (int jj = 0; jj < kPf; ++jj) {
          const int j = j0 + jj;
          const unsigned int item = __shfl(mine, j < nb ? j : 0, kL);
          sl[jj] = __shfl(myslot, j < nb ? j : 0, kL);
          v[jj] = Pair<HT>::zero();
          pp[jj] = 0xFFFFu;
          if (j < nb && c < NL / 2) {
            pp[jj] = *reinterpret_cast<const unsigned short*>(pos + size_t(base + j) * 32 + 2 * c);
            v[jj] = *reinterpret_cast<const HT2*>(hbuf + size_t(item >> 5) * (NL * kRowStride<NL>) +
                                                  (item & 31u) * kRowStride<NL> + 2 * c);
          }
        }
#pragma unroll
        for (int jj = 0; jj < kPf; ++jj) {
          const unsigned int p0 = pp[jj] & 0xFFu, p1 = pp[jj] >> 8;
          if (p0 != kPosNone) sRows[sl[jj] * cap + p0] += v[jj].x;
          if (p1 != kPosNone) sRows[sl[jj] * cap + p1] += v[jj].y;
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  if (WH) {
#pragma unroll
    for (int t = 0; t < kRB; ++t)
      if (t < nr)
        for (int j = c; j < kb[t + 1] - kb[t]; j += kL) vals[kb[t] + j] = sRows[t * cap + j];
  }
  if (WG && c < nr) g[r0 + c] = f ? gacc - f[r0 + c] : gacc;
}

template <int NL>
int launch_row_gather(fne_plan* plan, bool want_g, bool want_h, const FneCall& c) {
  const fne_plan_desc& d = plan->d;
  const bool fp32 = c.precision == FNE_FP32;
  const int rows_per_block = kBlock / mc_row_lanes(NL) * kRowBatch<NL>;
  const dim3 grid((d.n_free + rows_per_block - 1) / rows_per_block);
  const int cap = (d.max_row_len + 1) & ~1;
  const size_t shm = want_h ? size_t(rows_per_block) * cap * (fp32 ? 4 : 8) : 0;
  if (shm > plan->max_lds || d.max_row_len > 254) {
    fne_set_error("row gather: CSR rows too long for the LDS row copies");
    return FNE_EINVAL;
  }
  if (d.n_free == 0 || (!want_g && !want_h)) return FNE_OK;
#define RG(HT, G, H)                                                                                \
  hipLaunchKernelGGL((row_gather_kernel<NL, HT, G, H>), grid, dim3(kBlock), shm, c.stream, d,       \
                     (const HT*)plan->mc_h, plan->mc_g, c.f, c.g, (HT*)c.vals)
  if (!want_h) RG(double, true, false);
  else if (fp32) { if (want_g) RG(float, true, true); else RG(float, false, true); }
  else { if (want_g) RG(double, true, true); else RG(double, false, true); }
#undef RG
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

// ---------------------------------------------------------------------------------------------
// Mohr-Coulomb rows from element matrices stored as [n][m][j][i].  A unit is a CSR row, or the x and
// y rows of a node with the same columns and elements (FneRowUnits): positions and incidences are then
// read once for two rows, and a lane reads its node pair as one vector.  Plans without units take
// row_gather_kernel, whose rows lie together in memory: a unit of one row reads twice the bytes that it
// needs (32,000 P4 elements, Hessian with every row a unit of its own: FP64 272 us, FP32 125 to 146; row
// gather 195 and 109; pairs 198 and 101).
// mc_row_lanes lanes per unit; the contributions are added in item order into LDS copies of
// the rows, which are written once (storing rows of a single element straight from the registers
// measured the same).  Bound by memory traffic: P4 FP32, 98,000 elements: 376 MB of element matrices,
// 60 MB of positions and incidences, 314 MB of values, 231 us = 3.2 TB/s (before: rows one by one,
// 94 MB of positions, 244 us); P2 FP64, 21,978 elements 15.2 -> 12.9 us.  The loads of P4 FP32 bypass
// the caches (a row of a matrix is read once, 246 us against 258); those of P2, whose scratch stays in
// the last-level cache, do not (17.5 us against 12.9).  Fetching a unit's items while the one before is
// added, and cutting the elements into runs whose scratch fits the last-level cache, were slower (277
// us; 503 us for both kernels).
// ---------------------------------------------------------------------------------------------
struct McUnit {
  int k0, item0, row, len, items;
  bool two;
};
__device__ __forceinline__ McUnit mc_unit(const fne_plan_desc& d, const FneRowUnits& U, int u) {
  if (U.unit) {
    const int4 w = U.unit[u];
    return McUnit{w.x, w.y, w.z, w.w & 255, w.w >> 9, ((w.w >> 8) & 1) != 0};
  }
  const int k0 = d.indptr ? d.indptr[u] : 0, k1 = d.indptr ? d.indptr[u + 1] : 0;
  const int i0 = d.inc_ptr[u], i1 = d.inc_ptr[u + 1];
  return McUnit{k0, i0, u, k1 - k0, i1 - i0, false};  // items of d.inc / d.pitem
}

template <int NN, typename HT, bool WG>
__global__ __launch_bounds__(kBlock) void mc_unit_gather_kernel(fne_plan_desc d, FneRowUnits U,
                                                                int n_unit, const HT* __restrict__ hbuf,
                                                                const double* __restrict__ gbuf,
                                                                const double* __restrict__ f,
                                                                double* __restrict__ g, HT* __restrict__ vals) {
  extern __shared__ __align__(16) unsigned char mc_unit_smem[];
  constexpr int NL = 2 * NN, kL = mc_row_lanes(NL), kGroups = kBlock / kL, kPf = 4;
  typedef typename Vec4<HT>::type V4;
  typedef typename Pair<HT>::type HT2;
  const int grp = threadIdx.x / kL, c = threadIdx.x & (kL - 1);
  const int u = xcd_remap(blockIdx.x, gridDim.x) * kGroups + grp;
  if (u >= n_unit) return;  // uniform over the lane group; no block-level barrier below
  const McUnit w = mc_unit(d, U, u);
  const unsigned char* pos = U.pos + size_t(w.item0) * (2 * kL) + 2 * c;
  const unsigned int* inc = U.inc + w.item0;
  // both rows side by side; entry `none` takes what falls on constrained columns and idle lanes
  const unsigned none = d.max_row_len;
  HT2* buf = reinterpret_cast<HT2*>(mc_unit_smem) + size_t(grp) * (none + 1);
  const int my_row = w.row + (w.two ? c & 1 : 0);
  const double load = WG && f ? f[my_row] : 0.0;
  double gsum = 0.0;
  for (int i = c; i < w.len; i += kL) buf[i] = Pair<HT>::zero();
  for (int base = 0; base < w.items; base += kL) {
    const int nb = min(kL, w.items - base);
    const unsigned int mine = c < nb ? inc[base + c] : 0u;
    for (int j0 = 0; j0 < nb; j0 += kPf) {
      V4 v[kPf];
      unsigned pp[kPf];
      double gv[kPf];
#pragma unroll
      for (int jj = 0; jj < kPf; ++jj) {
        pp[jj] = 0xFFFFu;
        if (j0 + jj < nb && c < NN)
          pp[jj] = *reinterpret_cast<const unsigned short*>(pos + size_t(base + j0 + jj) * (2 * kL));
      }
#pragma unroll
      for (int jj = 0; jj < kPf; ++jj) {
        if (j0 + jj < nb) {
          const unsigned item = __shfl(mine, j0 + jj, kL);
          const unsigned e = item >> 5, n = (item & 31u) >> 1;
          if (c < NN) {
            const V4* from = reinterpret_cast<const V4*>(hbuf + size_t(e) * kMcMatrix<NN> + n * kMcNodeRow<NN> + c * 4);
            v[jj] = NN == 15 && sizeof(HT) == 4 ? __builtin_nontemporal_load(from) : *from;
          }
          if (!w.two && (item & 1u)) {  // the y row of a node by itself
            v[jj][0] = v[jj][1];
            v[jj][2] = v[jj][3];
          }
          if (WG && c < 2) gv[jj] = gbuf[size_t(e) * 32 + 2 * n + (w.two ? c : int(item & 1u))];
        }
      }
#pragma unroll
      for (int jj = 0; jj < kPf; ++jj) {
        if (j0 + jj < nb) {
          const unsigned p0 = pp[jj] & 0xFFu, p1 = pp[jj] >> 8;
          // both reads, then both writes: the two positions are distinct
          HT2* b0 = buf + min(p0, none);
          HT2* b1 = buf + min(p1, none);
          HT2 o0 = *b0, o1 = *b1;
          o0.x += v[jj][0];
          o0.y += v[jj][1];
          o1.x += v[jj][2];
          o1.y += v[jj][3];
          *b0 = o0;
          *b1 = o1;
          if (WG && c < 2) gsum += gv[jj];
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  // the rows of a node follow each other in the CSR arrays: one run, cut at multiples of kL entries
  // so that a store fills whole 64-byte pieces (FP32, 98,000 elements: 255 -> 240 us)
  HT* dst = vals + w.k0;
  const int n = w.two ? 2 * w.len : w.len;
  for (int i0 = c - (w.k0 & (kL - 1)); i0 < n; i0 += 4 * kL) {
    HT o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = max(min(i0 + j * kL, n - 1), 0);  // (a row without entries reads one and stores none)
      o[j] = i < w.len ? buf[i].x : buf[i - w.len].y;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = i0 + j * kL;
      if (i >= 0 && i < n) dst[i] = o[j];
    }
  }
  if (WG && c < (w.two ? 2 : 1)) g[my_row] = gsum - load;
}

// the gradient alone: one thread per unit, the same additions in the same order (98,000 elements: 23 us)
__global__ __launch_bounds__(kBlock) void mc_unit_grad_kernel(fne_plan_desc d, FneRowUnits U,
                                                              int n_unit, const double* __restrict__ gbuf,
                                                              const double* __restrict__ f,
                                                              double* __restrict__ g) {
  const int u = xcd_remap(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (u >= n_unit) return;
  const McUnit w = mc_unit(d, U, u);
  const unsigned int* inc = U.unit ? U.inc : reinterpret_cast<const unsigned int*>(d.inc);
  const double f0 = f ? f[w.row] : 0.0, f1 = f && w.two ? f[w.row + 1] : 0.0;
  double g0 = 0.0, g1 = 0.0;
  for (int i = 0; i < w.items; i += 4) {
    unsigned item[4];
    double2 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) item[j] = i + j < w.items ? inc[w.item0 + i + j] : 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i + j < w.items)
        v[j] = *reinterpret_cast<const double2*>(gbuf + size_t(item[j] >> 5) * 32 + (item[j] & 30u));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i + j < w.items) {
        g0 += !w.two && (item[j] & 1u) ? v[j].y : v[j].x;
        g1 += v[j].y;
      }
  }
  g[w.row] = g0 - f0;
  if (w.two) g[w.row + 1] = g1 - f1;
}

// Element outputs for fne_element_eval: scratch (element-major) -> SoA outputs.
template <int NN>
__global__ __launch_bounds__(kBlock) void mc_element_out_kernel(int ne, const double* __restrict__ gbuf,
                                                                const double* __restrict__ hbuf,
                                                                double* __restrict__ ge_out,
                                                                double* __restrict__ he_out) {
  constexpr int NL = 2 * NN;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  if (ge_out)
    for (int i = 0; i < NL; ++i) ge_out[size_t(i) * ne + e] = gbuf[size_t(e) * 32 + i];
  if (he_out) {
    const double* H = hbuf + size_t(e) * kMcMatrix<NN>;
    for (int r = 0; r < NL; ++r)
      for (int c = 0; c < NL; ++c)
        he_out[size_t(r * NL + c) * ne + e] = H[(r >> 1) * kMcNodeRow<NN> + (c >> 1) * 4 + (c & 1) * 2 + (r & 1)];
  }
}

// wavefront rounds spread evenly over at most kEnergyBlocks blocks
McBlocks mc_blocks(int ne) {
  constexpr int kRound = kMcWaves * kMcEpw;
  const int need = std::max(1, (ne + kRound - 1) / kRound);
  McBlocks b;
  b.rounds = (need + kEnergyBlocks - 1) / kEnergyBlocks;
  b.all = (need + b.rounds - 1) / b.rounds;
  return b;
}

// CSR values (HT) and / or the gradient from the element scratch
template <int NN>
int launch_mc_rows(fne_plan* plan, bool want_g, bool want_h, const FneCall& c) {
  const fne_plan_desc& d = plan->d;
  const int n_unit = plan->units.n_unit > 0 ? plan->units.n_unit : d.n_free;
  if (n_unit == 0) return FNE_OK;
  if (!want_h) {
    hipLaunchKernelGGL(mc_unit_grad_kernel, dim3((n_unit + kBlock - 1) / kBlock), dim3(kBlock), 0, c.stream, d,
                       plan->units, n_unit, plan->mc_g, c.f, c.g);
    FNE_LAUNCH_CHECK();
    return FNE_OK;
  }
  if (plan->units.n_unit == 0) return launch_row_gather<2 * NN>(plan, want_g, true, c);
  constexpr int kGroups = kBlock / mc_row_lanes(2 * NN);
  const bool fp32 = c.precision == FNE_FP32;
  const size_t shm = size_t(kGroups) * 2 * (d.max_row_len + 1) * (fp32 ? 4 : 8);
  if (shm > plan->max_lds) {
    fne_set_error("row gather LDS request exceeds the device limit");
    return FNE_EINVAL;
  }
  const dim3 grid((n_unit + kGroups - 1) / kGroups);
#define MC_ROWS(HT, G)                                                                                         \
  hipLaunchKernelGGL((mc_unit_gather_kernel<NN, HT, G>), grid, dim3(kBlock), shm, c.stream, d, plan->units, n_unit, \
                     (const HT*)plan->mc_h, plan->mc_g, c.f, c.g, (HT*)c.vals)
  if (fp32) {
    if (want_g) MC_ROWS(float, true);
    else MC_ROWS(float, false);
  } else {
    if (want_g) MC_ROWS(double, true);
    else MC_ROWS(double, false);
  }
#undef MC_ROWS
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

template <int NN>
int launch_mc(fne_plan* plan, FneOp op, const FneCall& c) {
  const fne_plan_desc& d = plan->d;
  const int ne = d.n_elem;
  const McBlocks B = mc_blocks(ne);
  const bool by_rows = plan->units.n_unit == 0;
  const int nb = B.all;
  if (nb > plan->n_partials) {
    fne_set_error("energy reduction scratch too small");
    return FNE_EINVAL;
  }
  const McConst k = mc_const(d.param, plan->mode);
  const bool want_e = op == kOpEnergy || (op == kOpFused && c.out);
  const bool want_g = op == kOpGradient || ((op == kOpHessian || op == kOpFused) && c.g);
  const bool want_h = op == kOpHessian || op == kOpFused;
  const EnergySum energy = fne_energy_sum(plan, op, nb, c.out);
  double* gb = plan->mc_g;
  void* hb = plan->mc_h;
#define MC_ELEM_GO(NS, HT, E, G, H, R, FV, EV)                                                                      \
  hipLaunchKernelGGL((mc_elem_kernel<NN, NS, HT, E, G, H, false, R>), dim3(nb), dim3(kBlock), 0, c.stream, d, k, c.x, \
                     c.dvals, FV, (const double*)nullptr, energy, EV, gb, (HT*)hb, B)
  // NS: products of four K rows that cover 2 n_q
#define MC_ELEM_R(HT, E, G, H, R, FV, EV)       \
  do {                                          \
    if (d.nq <= 20)                             \
      MC_ELEM_GO(10, HT, E, G, H, R, FV, EV);   \
    else                                        \
      MC_ELEM_GO(11, HT, E, G, H, R, FV, EV);   \
  } while (0)
  // (only matrices are stored in two ways)
#define MC_ELEM(HT, E, G, H, FV, EV)            \
  do {                                          \
    if (H && by_rows)                           \
      MC_ELEM_R(HT, E, G, H, H, FV, EV);        \
    else                                        \
      MC_ELEM_R(HT, E, G, H, false, FV, EV);    \
  } while (0)
  if (op == kOpElementEval) {
    MC_ELEM_R(double, false, true, true, false, (const double*)nullptr, c.e_out);
    FNE_LAUNCH_CHECK();
    if (c.ge_out || c.he_out) {
      hipLaunchKernelGGL(mc_element_out_kernel<NN>, dim3((ne + kBlock - 1) / kBlock), dim3(kBlock), 0, c.stream,
                         ne, gb, (const double*)hb, c.ge_out, c.he_out);
      FNE_LAUNCH_CHECK();
    }
    return FNE_OK;
  }
  if ((want_g || want_h) && (!d.inc_ptr || !d.inc || (want_h && !d.pitem))) {
    fne_set_error("row incidence arrays missing from the plan");
    return FNE_EINVAL;
  }
  if (want_h && d.max_row_len > 254) {
    fne_set_error("CSR rows longer than 254 entries are not supported");
    return FNE_EINVAL;
  }
  const bool fp32 = c.precision == FNE_FP32;
  double* const none = nullptr;
  if (want_h) {
    if (fp32) {
      if (want_e && want_g) MC_ELEM(float, true, true, true, c.f, none);
      else if (want_e) MC_ELEM(float, true, false, true, c.f, none);
      else if (want_g) MC_ELEM(float, false, true, true, c.f, none);
      else MC_ELEM(float, false, false, true, c.f, none);
    } else {
      if (want_e && want_g) MC_ELEM(double, true, true, true, c.f, none);
      else if (want_e) MC_ELEM(double, true, false, true, c.f, none);
      else if (want_g) MC_ELEM(double, false, true, true, c.f, none);
      else MC_ELEM(double, false, false, true, c.f, none);
    }
  } else if (want_g) {
    if (want_e) MC_ELEM(double, true, true, false, c.f, none);
    else MC_ELEM(double, false, true, false, c.f, none);
  } else {
    MC_ELEM(double, true, false, false, c.f, none);
  }
#undef MC_ELEM
#undef MC_ELEM_R
#undef MC_ELEM_GO
  FNE_LAUNCH_CHECK();
  if (want_e) {
    const int rc = fne_finalize_energy(plan, nb, c.out, c.stream);
    if (rc) return rc;
  }
  if (!want_g && !want_h) return FNE_OK;
  return launch_mc_rows<NN>(plan, want_g, want_h, c);
}

// ---------------------------------------------------------------------------------------------
// Matrix-free Hessian products (slope_stability/jax_petsc/reordered_element_assembler.py:313-562).
// Products: the element kernel with the stress of the direction, H_e v_e = sum_q w_q B_q^T D_q
// (B_q v_e) with D_q the tangent of the return mapping at the state x (the matrix that it
// assembles).  Diagonals diag(H_e)_a = sum_q w_q b_a^T D_q b_a have a kernel of their own.  Both go
// to the element-vector scratch and are summed per row like the gradient.  FP64 throughout.
// ---------------------------------------------------------------------------------------------
struct McDiagLds {
  double u[kMcEpw][32];
  double geo[kMcEpw][8];
  double D[kMcEpw][kMcMaxQ][6];  // w * D
};

template <int NN>
__global__ __launch_bounds__(kBlock) void mc_diag_kernel(fne_plan_desc d, McConst k, const double* __restrict__ x,
                                                         const double* __restrict__ dvals,
                                                         double* __restrict__ gbuf) {
  constexpr int NL = 2 * NN;
  __shared__ double sTab[kMcMaxQ * 16 * 2];
  __shared__ double sW[kMcMaxQ];
  __shared__ McDiagLds sWave[kMcWaves];
  const int nq = d.nq;
  for (int i = threadIdx.x; i < nq * NN * 2; i += blockDim.x) sTab[i] = d.qdata[nq + i];
  for (int i = threadIdx.x; i < nq; i += blockDim.x) sW[i] = d.qdata[i];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  McDiagLds& L = sWave[wave];
  const int ne = d.n_elem;
  const bool has_eps = d.n_geo >= 5 + 3 * nq;
  const int nwaves = gridDim.x * kMcWaves;
  for (int base = (blockIdx.x * kMcWaves + wave) * kMcEpw; base < ne; base += nwaves * kMcEpw) {
    for (int i = lane; i < kMcEpw * NL; i += 64) {
      const int t = i / NL, c = i - t * NL;
      const int e = base + t;
      L.u[t][c] = e < ne ? gather_dof(d.edof[size_t(c) * ne + e], d.n_free, x, dvals) : 0.0;
    }
    if (lane < kMcEpw * 5) {
      const int t = lane / 5, c = lane - 5 * t;
      const int e = base + t;
      L.geo[t][c] = e < ne ? d.egeo[size_t(c) * ne + e] : (c == 4 ? 0.0 : 1.0);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (lane < kMcEpw * nq) {
      const int t = lane / nq, q = lane - t * nq;
      const int e = base + t;
      if (e < ne) {
        double U00 = 0.0, U01 = 0.0, U10 = 0.0, U11 = 0.0;
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const double g0 = sTab[(q * NN + n) * 2 + 0], g1 = sTab[(q * NN + n) * 2 + 1];
          U00 += L.u[t][2 * n] * g0;
          U01 += L.u[t][2 * n] * g1;
          U10 += L.u[t][2 * n + 1] * g0;
          U11 += L.u[t][2 * n + 1] * g1;
        }
        const double K00 = L.geo[t][0], K01 = L.geo[t][1], K10 = L.geo[t][2], K11 = L.geo[t][3];
        double e0 = K00 * U00 + K01 * U01;
        double e1 = K10 * U10 + K11 * U11;
        double e2 = (K10 * U00 + K11 * U01) + (K00 * U10 + K01 * U11);
        if (has_eps) {
          const size_t o = size_t(5 + 3 * q) * ne + e;
          e0 -= d.egeo[o];
          e1 -= d.egeo[o + ne];
          e2 -= d.egeo[o + 2 * size_t(ne)];
        }
        double sig[3], D[6];
        mc_point<true>(k, e0, e1, e2, sig, D);
        const double w = sW[q] * L.geo[t][4];
#pragma unroll
        for (int i = 0; i < 6; ++i) L.D[t][q][i] = w * D[i];
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int i = lane; i < kMcEpw * NL; i += 64) {
      const int t = i / NL, rr = i - t * NL;
      const int e = base + t;
      if (e >= ne) continue;
      const int n = rr >> 1, comp = rr & 1;
      double s = 0.0;
      for (int q = 0; q < nq; ++q) {
        const double g0 = sTab[(q * NN + n) * 2 + 0], g1 = sTab[(q * NN + n) * 2 + 1];
        const double gx = L.geo[t][0] * g0 + L.geo[t][1] * g1;
        const double gy = L.geo[t][2] * g0 + L.geo[t][3] * g1;
        const double* Dq = L.D[t][q];
        // b = (gx, 0, gy) for an x component, (0, gy, gx) for a y component
        s += comp == 0 ? Dq[0] * gx * gx + 2.0 * Dq[2] * gx * gy + Dq[5] * gy * gy
                       : Dq[3] * gy * gy + 2.0 * Dq[4] * gx * gy + Dq[5] * gx * gx;
      }
      gbuf[size_t(e) * 32 + rr] = s;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
}

// v == nullptr: the diagonal
template <int NN>
int launch_mc_aux(fne_plan* plan, const double* x, const double* dvals, const double* v, double* out,
                  hipStream_t stream) {
  const fne_plan_desc& d = plan->d;
  const McBlocks B = mc_blocks(d.n_elem);
  const dim3 grid(B.all);
  const McConst k = mc_const(d.param, plan->mode);
  if (v) {
    const double* none = nullptr;
#define MC_HVP(NS)                                                                                                 \
  hipLaunchKernelGGL((mc_elem_kernel<NN, NS, double, false, true, false, true, false>), grid, dim3(kBlock), 0, stream, d, k, \
                     x, dvals, none, v, EnergySum{}, (double*)nullptr, plan->mc_g, (double*)nullptr, B)
    if (d.nq <= 20)
      MC_HVP(10);
    else
      MC_HVP(11);
#undef MC_HVP
  } else {
    hipLaunchKernelGGL((mc_diag_kernel<NN>), grid, dim3(kBlock), 0, stream, d, k, x, dvals, plan->mc_g);
  }
  FNE_LAUNCH_CHECK();
  FneCall c{};
  c.f = nullptr;
  c.g = out;
  c.precision = FNE_FP64;
  c.stream = stream;
  return launch_mc_rows<NN>(plan, true, false, c);
}

int mc_aux(fne_plan* plan, int aux, const double* x, const double* dvals, const double* v, double* out,
           fne_stream_t stream) {
  if (!plan || !x || !out || (aux == 1 && (!v || v == out))) {
    fne_set_error("invalid arguments");
    return FNE_EINVAL;
  }
  const fne_plan_desc& d = plan->d;
  if (d.kind != FNE_KIND_MOHR_COULOMB) {
    fne_set_error("the matrix-free Hessian diagonal is implemented for the Mohr-Coulomb family");
    return FNE_EUNSUPPORTED;
  }
  if (!plan->mc_g || !d.inc_ptr || !d.inc) {
    fne_set_error("the plan needs FNE_FLAG_ROW_GATHER (row incidences and element scratch)");
    return FNE_EINVAL;
  }
  if (d.n_total > 0 && !dvals) {
    fne_set_error("Dirichlet values missing");
    return FNE_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  if (d.n_loc == 12) return launch_mc_aux<6>(plan, x, dvals, aux == 1 ? v : nullptr, out, s);
  if (d.n_loc == 30) return launch_mc_aux<15>(plan, x, dvals, aux == 1 ? v : nullptr, out, s);
  fne_set_error("Mohr-Coulomb plans need n_loc = 12 (P2) or 30 (P4)");
  return FNE_EINVAL;
}

}  // namespace

extern "C" int fne_hvp(fne_plan* plan, const double* x, const double* dvals, const double* v, double* y,
                       fne_stream_t stream) {
  if (!plan || !x || !v || !y || v == y) {
    fne_set_error("fne_hvp: invalid arguments");
    return FNE_EINVAL;
  }
  const int kind = plan->d.kind;
  if (kind == FNE_KIND_MOHR_COULOMB) return mc_aux(plan, 1, x, dvals, v, y, stream);
  if (plan->d.n_total > 0 && !dvals) {
    fne_set_error("Dirichlet values missing");
    return FNE_EINVAL;
  }
  if (kind == FNE_KIND_PLAPLACE || kind == FNE_KIND_GINZBURG_LANDAU)
    return fne_hvp_p1(plan, x, dvals, v, y, (hipStream_t)stream);
  if (kind == FNE_KIND_NEOHOOKEAN) return fne_hvp_tet(plan, x, dvals, v, y, (hipStream_t)stream);
  fne_set_error("fne_hvp: unknown energy family");
  return FNE_EUNSUPPORTED;
}

extern "C" int fne_hessian_diag(fne_plan* plan, const double* x, const double* dvals, double* diag,
                                fne_stream_t stream) {
  return mc_aux(plan, 2, x, dvals, nullptr, diag, stream);
}

int fne_launch_row_gather(fne_plan* plan, bool want_g, bool want_h, const FneCall& c) {
  if (plan->d.n_loc != 12) {
    fne_set_error("row gather supports elements with 12 DOFs");
    return FNE_EINVAL;
  }
  return launch_row_gather<12>(plan, want_g, want_h, c);
}

size_t fne_mc_scratch_bytes(const fne_plan_desc& d, size_t* gbytes) {
  const size_t nl = size_t(d.n_loc);
  // padding: a wavefront stores all three elements of its last round
  const size_t ne = size_t(d.n_elem) + (d.kind == FNE_KIND_MOHR_COULOMB ? kMcEpw : 0);
  if (gbytes) *gbytes = ne * 32 * sizeof(double);
  const size_t values = d.kind != FNE_KIND_MOHR_COULOMB ? nl * nl : (nl == 30 ? kMcMatrix<15> : kMcMatrix<6>);
  return ne * values * sizeof(double);
}

int fne_launch_mc(fne_plan* plan, FneOp op, const FneCall& c) {
  if (!plan->mc_g || !plan->mc_h) {
    fne_set_error("Mohr-Coulomb element scratch missing");
    return FNE_EINVAL;
  }
  switch (plan->d.n_loc) {
    case 12:
      return launch_mc<6>(plan, op, c);
    case 30:
      return launch_mc<15>(plan, op, c);
    default:
      fne_set_error("Mohr-Coulomb plans need n_loc = 12 (P2) or 30 (P4)");
      return FNE_EINVAL;
  }
}
