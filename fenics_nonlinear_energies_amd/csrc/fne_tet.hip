// Compressible Neo-Hookean P1 tetrahedra (A3): energy, gradient, CSR Hessian.
//
// Element data (SoA): edof[(3a+i)*n_elem+e] (deformed position y_{a,i}, a=0..3, i=x,y,z),
// egeo[k*n_elem+e]: dphix[0..3], dphiy[0..3], dphiz[0..3], vol.
// Math (hand-derived; replaces jax.hessian of _he_energy_density,
// hyperelasticity/jax_petsc/parallel_hessian_dof.py:17-52):
//   F_ij = sum_a y_{a,i} D_{a,j}   (D_a = grad phi_a),  J = det F  (|det F| with FNE_FLAG_ABS_DET)
//   W = C1 (|F|^2 - 3 - 2 ln J) + D1 (J-1)^2,   E = W vol
//   G = F^{-T},  q_a = G D_a
//   dE/dy_{a,i} = vol [ 2 C1 (F D_a)_i + c q_{a,i} ],            c = -2 C1 + 2 D1 J (J-1)
//   H_{(a,i),(b,k)} = vol [ 2 C1 d_ik (D_a.D_b) + alpha q_{b,i} q_{a,k} + beta q_{a,i} q_{b,k} ]
//                     alpha = 2 C1 - 2 D1 J (J-1),  beta = 2 D1 J (2J-1)
#include "fne_common.h"

#include <algorithm>

namespace {

struct TetElem {
  double y[4][3];
  double D[4][3];
  double vol;
};

__device__ __forceinline__ void tet_load(const fne_plan_desc& d, int e, const double* __restrict__ x,
                                         const double* __restrict__ dvals, TetElem& t) {
  const int ne = d.n_elem;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
#pragma unroll
    for (int i = 0; i < 3; ++i) t.y[a][i] = gather_dof(d.edof[(3 * a + i) * ne + e], d.n_free, x, dvals);
    t.D[a][0] = d.egeo[a * ne + e];
    t.D[a][1] = d.egeo[(4 + a) * ne + e];
    t.D[a][2] = d.egeo[(8 + a) * ne + e];
  }
  t.vol = d.egeo[12 * ne + e];
}

struct TetKin {
  double F[3][3];
  double det, J;
};

__device__ __forceinline__ void tet_kinematics(const TetElem& t, bool absdet, TetKin& k) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      k.F[i][j] = t.y[0][i] * t.D[0][j] + t.y[1][i] * t.D[1][j] + t.y[2][i] * t.D[2][j] + t.y[3][i] * t.D[3][j];
  const double(&F)[3][3] = k.F;
  k.det = F[0][0] * (F[1][1] * F[2][2] - F[1][2] * F[2][1]) - F[0][1] * (F[1][0] * F[2][2] - F[1][2] * F[2][0]) +
          F[0][2] * (F[1][0] * F[2][1] - F[1][1] * F[2][0]);
  k.J = absdet ? fabs(k.det) : k.det;
}

__device__ __forceinline__ double dot3(const double a[3], const double b[3]) {
  return fma(a[2], b[2], fma(a[1], b[1], a[0] * b[0]));
}

// F, its cofactors and determinant, and the energy density from them: shared by fne_energy and the
// node-patch assembly, so that both round every element alike.  Near rest the energy is the small
// difference of terms of size C1; fused products keep its error 60 times below that of separate ones
// (160x8x8 beam, turned cross-sections: 1.2e-15 against 7.2e-14 of the energy).
__device__ __forceinline__ double tet_deformation(const double (&y)[4][3], const double (&D)[4][3], double (&F)[3][3],
                                                  double (&C)[3][3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      F[i][j] = fma(y[3][i], D[3][j], fma(y[2][i], D[2][j], fma(y[1][i], D[1][j], y[0][i] * D[0][j])));
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      C[i][j] = F[i1][j1] * F[i2][j2] - F[i1][j2] * F[i2][j1];  // cofactor
    }
  return fma(F[0][2], C[0][2], fma(F[0][1], C[0][1], F[0][0] * C[0][0]));
}

__device__ __forceinline__ double tet_density(const double (&F)[3][3], double J, double C1, double D1) {
  double I1 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) I1 += dot3(F[i], F[i]);
  return C1 * (I1 - 3.0 - 2.0 * log(J)) + D1 * ((J - 1.0) * (J - 1.0));
}

__device__ __forceinline__ double tet_energy(const TetElem& t, const double* prm, bool absdet) {
  double F[3][3], C[3][3];
  const double det = tet_deformation(t.y, t.D, F, C);
  return t.vol * tet_density(F, absdet ? fabs(det) : det, prm[0], prm[1]);
}

// compact per-element state: the Hessian is expanded from (coefs, q, D) where it is needed
struct TetState {
  double s0, s1, s2;  // vol*2C1, vol*alpha, vol*beta
  double q[4][3];
  double g[4][3];
};

__device__ __forceinline__ void tet_state(const TetElem& t, const double* prm, bool absdet, TetState& s) {
  TetKin k;
  tet_kinematics(t, absdet, k);
  const double(&F)[3][3] = k.F;
  const double C1 = prm[0], D1 = prm[1];
  const double J = k.J;
  // G = F^{-T} = cof(F) / det
  const double inv = 1.0 / k.det;
  double G[3][3];
  G[0][0] = (F[1][1] * F[2][2] - F[1][2] * F[2][1]) * inv;
  G[0][1] = -(F[1][0] * F[2][2] - F[1][2] * F[2][0]) * inv;
  G[0][2] = (F[1][0] * F[2][1] - F[1][1] * F[2][0]) * inv;
  G[1][0] = -(F[0][1] * F[2][2] - F[0][2] * F[2][1]) * inv;
  G[1][1] = (F[0][0] * F[2][2] - F[0][2] * F[2][0]) * inv;
  G[1][2] = -(F[0][0] * F[2][1] - F[0][1] * F[2][0]) * inv;
  G[2][0] = (F[0][1] * F[1][2] - F[0][2] * F[1][1]) * inv;
  G[2][1] = -(F[0][0] * F[1][2] - F[0][2] * F[1][0]) * inv;
  G[2][2] = (F[0][0] * F[1][1] - F[0][1] * F[1][0]) * inv;
  const double c = -2.0 * C1 + 2.0 * D1 * J * (J - 1.0);
  s.s0 = t.vol * 2.0 * C1;
  s.s1 = t.vol * (2.0 * C1 - 2.0 * D1 * J * (J - 1.0));
  s.s2 = t.vol * (2.0 * D1 * J * (2.0 * J - 1.0));
#pragma unroll
  for (int a = 0; a < 4; ++a) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double qa = G[i][0] * t.D[a][0] + G[i][1] * t.D[a][1] + G[i][2] * t.D[a][2];
      const double fa = F[i][0] * t.D[a][0] + F[i][1] * t.D[a][1] + F[i][2] * t.D[a][2];
      s.q[a][i] = qa;
      s.g[a][i] = t.vol * (2.0 * C1 * fa + c * qa);
    }
  }
}

// staged layout in LDS (FP64, [field][chunk]): 0..2 coefs, 3..14 q, 15..26 D, 27..38 g
constexpr int kTetStage = 39;

__global__ __launch_bounds__(kBlock) void tet_energy_kernel(fne_plan_desc d, const double* __restrict__ x,
                                                            const double* __restrict__ dvals,
                                                            const double* __restrict__ f,
                                                            EnergySum energy) {
  double s = 0.0, c = 0.0;
  const bool absdet = (d.flags & FNE_FLAG_ABS_DET) != 0;
  const int stride = gridDim.x * blockDim.x;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < d.n_elem; e += stride) {
    TetElem t;
    tet_load(d, e, x, dvals, t);
    double E = tet_energy(t, d.param, absdet);
    if (d.eweight) E *= d.eweight[e];
    acc_add(s, c, E);
  }
  if (f) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < d.n_free; i += stride) acc_add(s, c, -(f[i] * x[i]));
  }
  block_energy(energy, blockIdx.x, s, c);
}

// Patch kernel.  Rows come in node triples; thread t of the workgroup owns scalar row r0+t.
// Incidence lists are per node row: item (uint64) = slot[0:16) | a[16:18) | bpos_b[24+8b : 32+8b)
// (bpos = block column of element node b inside the node's block row, 255 = constrained node).
template <typename HT, bool WANT_G, bool WANT_H>
__global__ __launch_bounds__(kBlock) void tet_patch_kernel(fne_plan_desc d, const double* __restrict__ x,
                                                           const double* __restrict__ dvals,
                                                           const double* __restrict__ f,
                                                           double* __restrict__ g, HT* __restrict__ vals) {
  extern __shared__ double smem[];
  const int p = xcd_remap(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  const int chunk = d.chunk;
  const int r0 = d.prow[p], r1 = d.prow[p + 1];
  const int k0 = d.indptr[r0];
  const int nslice = WANT_H ? d.indptr[r1] - k0 : 0;
  const int eb = d.pelem_ptr[p];
  const int ne = d.pelem_ptr[p + 1] - eb;
  const bool absdet = (d.flags & FNE_FLAG_ABS_DET) != 0;

  HT* sVal = reinterpret_cast<HT*>(smem);
  double* sS = smem + (WANT_H ? (size_t(d.max_patch_nnz) * sizeof(HT) + 7) / 8 : 0);  // [39][chunk]
  if (WANT_H)
    for (int k = tid; k < nslice; k += blockDim.x) sVal[k] = HT(0);

  const int r = r0 + tid;
  const bool has_row = r < r1;
  const int node_row = r / 3;
  const int comp = r - 3 * node_row;
  const uint64_t* inc = reinterpret_cast<const uint64_t*>(d.inc);
  int ip = has_row ? d.inc_ptr[node_row] : 0;
  const int ie = has_row ? d.inc_ptr[node_row + 1] : 0;
  const int roff = has_row ? d.indptr[r] - k0 : 0;
  double gacc = 0.0;
  __syncthreads();

  for (int c0 = 0; c0 < ne; c0 += chunk) {
    const int nc = min(chunk, ne - c0);
    for (int sl = tid; sl < nc; sl += blockDim.x) {
      const int e = d.pelem[eb + c0 + sl];
      TetElem t;
      tet_load(d, e, x, dvals, t);
      TetState st;
      tet_state(t, d.param, absdet, st);
      if (WANT_H) {
        sS[0 * chunk + sl] = st.s0;
        sS[1 * chunk + sl] = st.s1;
        sS[2 * chunk + sl] = st.s2;
      }
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          if (WANT_H) {
            sS[(3 + 3 * a + i) * chunk + sl] = st.q[a][i];
            sS[(15 + 3 * a + i) * chunk + sl] = t.D[a][i];
          }
          if (WANT_G) sS[(27 + 3 * a + i) * chunk + sl] = st.g[a][i];
        }
    }
    __syncthreads();
    if (has_row) {
      while (ip < ie) {
        const uint64_t it = inc[ip];
        const int slot = int(it & 0xFFFFull);
        if (slot >= c0 + nc) break;
        const int sl = slot - c0;
        const int a = int((it >> 16) & 3ull);
        if (WANT_G) gacc += sS[(27 + 3 * a + comp) * chunk + sl];
        if (WANT_H) {
          const double s0 = sS[0 * chunk + sl], s1 = sS[1 * chunk + sl], s2 = sS[2 * chunk + sl];
          double qa[3], Da[3];
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            qa[i] = sS[(3 + 3 * a + i) * chunk + sl];
            Da[i] = sS[(15 + 3 * a + i) * chunk + sl];
          }
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const int bp = int((it >> (24 + 8 * b)) & 0xFFull);
            if (bp == 255) continue;
            double qb[3], Db[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              qb[i] = sS[(3 + 3 * b + i) * chunk + sl];
              Db[i] = sS[(15 + 3 * b + i) * chunk + sl];
            }
            const double dd = Da[0] * Db[0] + Da[1] * Db[1] + Da[2] * Db[2];
            const double qbi = qb[comp], qai = qa[comp];
            HT* dst = sVal + roff + 3 * bp;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              double h = s1 * qbi * qa[k] + s2 * qai * qb[k];
              if (k == comp) h += s0 * dd;
              dst[k] += HT(h);
            }
          }
        }
        ++ip;
      }
    }
    __syncthreads();
  }
  if (WANT_H)
    for (int k = tid; k < nslice; k += blockDim.x) vals[k0 + k] = sVal[k];
  if (WANT_G && has_row) g[r] = f ? gacc - f[r] : gacc;
}

__global__ __launch_bounds__(kBlock) void tet_element_kernel(fne_plan_desc d, const double* __restrict__ x,
                                                             const double* __restrict__ dvals,
                                                             double* __restrict__ e_out,
                                                             double* __restrict__ ge_out,
                                                             double* __restrict__ he_out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d.n_elem) return;
  const bool absdet = (d.flags & FNE_FLAG_ABS_DET) != 0;
  TetElem t;
  tet_load(d, e, x, dvals, t);
  const int ne = d.n_elem;
  if (e_out) e_out[e] = tet_energy(t, d.param, absdet);
  if (!ge_out && !he_out) return;
  TetState s;
  tet_state(t, d.param, absdet, s);
  if (ge_out)
    for (int a = 0; a < 4; ++a)
      for (int i = 0; i < 3; ++i) ge_out[(3 * a + i) * ne + e] = s.g[a][i];
  if (he_out)
    for (int a = 0; a < 4; ++a)
      for (int i = 0; i < 3; ++i)
        for (int b = 0; b < 4; ++b) {
          const double dd = t.D[a][0] * t.D[b][0] + t.D[a][1] * t.D[b][1] + t.D[a][2] * t.D[b][2];
          for (int k = 0; k < 3; ++k) {
            double h = s.s1 * s.q[b][i] * s.q[a][k] + s.s2 * s.q[a][i] * s.q[b][k];
            if (i == k) h += s.s0 * dd;
            he_out[((3 * a + i) * 12 + 3 * b + k) * ne + e] = h;
          }
        }
}

}  // namespace

// Row-gather form (FNE_FLAG_ROW_GATHER): one thread per element writes its gradient
// (gbuf[e][32], FP64) and 12x12 Hessian (hbuf[e][144], HT) element-major; the CSR rows then
// gather them (fne_launch_row_gather).
template <typename HT, bool WANT_G, bool WANT_H>
__global__ __launch_bounds__(kBlock) void tet_store_kernel(fne_plan_desc d, const double* __restrict__ x,
                                                           const double* __restrict__ dvals,
                                                           double* __restrict__ gbuf, HT* __restrict__ hbuf) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d.n_elem) return;
  const bool absdet = (d.flags & FNE_FLAG_ABS_DET) != 0;
  TetElem t;
  tet_load(d, e, x, dvals, t);
  TetState s;
  tet_state(t, d.param, absdet, s);
  if (WANT_G)
    for (int a = 0; a < 4; ++a)
      for (int i = 0; i < 3; ++i) gbuf[size_t(e) * 32 + 3 * a + i] = s.g[a][i];
  if (WANT_H) {
    HT* hb = hbuf + size_t(e) * 144;
    for (int a = 0; a < 4; ++a)
      for (int i = 0; i < 3; ++i)
        for (int b = 0; b < 4; ++b) {
          const double dd = t.D[a][0] * t.D[b][0] + t.D[a][1] * t.D[b][1] + t.D[a][2] * t.D[b][2];
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            double h = s.s1 * s.q[b][i] * s.q[a][k] + s.s2 * s.q[a][i] * s.q[b][k];
            if (i == k) h += s.s0 * dd;
            hb[(3 * a + i) * 12 + 3 * b + k] = HT(h);
          }
        }
  }
}

// Hessian-vector product, row-gather form: one thread per element writes y_e = H_e v_e (the
// 12x12 element Hessian at x applied to the element's v, zero on constrained DOFs) into the
// element gradient scratch; the gradient row gather then sums each row in its fixed order.
__global__ __launch_bounds__(kBlock) void tet_hvp_store_kernel(fne_plan_desc d, const double* __restrict__ x,
                                                               const double* __restrict__ dvals,
                                                               const double* __restrict__ v,
                                                               double* __restrict__ gbuf) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= d.n_elem) return;
  const bool absdet = (d.flags & FNE_FLAG_ABS_DET) != 0;
  TetElem t;
  tet_load(d, e, x, dvals, t);
  TetState s;
  tet_state(t, d.param, absdet, s);
  double ve[4][3];
  for (int b = 0; b < 4; ++b)
    for (int k = 0; k < 3; ++k) {
      const int code = d.edof[size_t(3 * b + k) * d.n_elem + e];
      ve[b][k] = code < d.n_free ? v[code] : 0.0;
    }
  for (int a = 0; a < 4; ++a)
    for (int i = 0; i < 3; ++i) {
      double acc = 0.0;
      for (int b = 0; b < 4; ++b) {
        const double dd = t.D[a][0] * t.D[b][0] + t.D[a][1] * t.D[b][1] + t.D[a][2] * t.D[b][2];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          double h = s.s1 * s.q[b][i] * s.q[a][k] + s.s2 * s.q[a][i] * s.q[b][k];
          if (i == k) h += s.s0 * dd;
          acc += h * ve[b][k];
        }
      }
      gbuf[size_t(e) * 32 + 3 * a + i] = acc;
    }
}

int fne_hvp_tet(fne_plan* plan, const double* x, const double* dvals, const double* v, double* y, hipStream_t stream) {
  const fne_plan_desc& d = plan->d;
  if (!(d.flags & FNE_FLAG_ROW_GATHER) || !plan->mc_g || !d.inc || !d.inc_ptr) {
    fne_set_error("tetrahedral Hessian-vector products need a row-gather plan (FNE_FLAG_ROW_GATHER)");
    return FNE_EUNSUPPORTED;
  }
  const int nb = (d.n_elem + kBlock - 1) / kBlock;
  if (nb > 0) {
    hipLaunchKernelGGL(tet_hvp_store_kernel, dim3(nb), dim3(kBlock), 0, stream, d, x, dvals, v, plan->mc_g);
    FNE_LAUNCH_CHECK();
  }
  FneCall c{};
  c.f = nullptr;
  c.g = y;
  c.precision = FNE_FP64;
  c.stream = stream;
  return fne_launch_row_gather(plan, true, false, c);
}

// ---------------------------------------------------------------------------------------------
// Node-patch assembly (FneNodePatches): energy, gradient and Hessian in one launch, nothing stored
// per element in memory.
//
// The row gather writes every 12x12 element matrix (576 B in FP32) and reads it back with 32 B of
// positions per row: on the 320x16x16 beam 850 MB against the 120 MB that the assembly cannot do
// without.  Here a workgroup evaluates the <= 240 elements around a run of ~20 free nodes, one per
// thread, and keeps their compact state in LDS (24 FP64: the four q_a, the two coefficients, the
// ten vol 2 C1 D_a.D_b).  Then each thread owns one 3x3 block of the CSR rows -- node i against
// neighbour j -- and sums the 4 to 8 elements around that edge in registers, in element order; where
// both nodes are in the patch it also writes the transposed block of (j, i).  Eight threads per node
// sum the diagonal block.  Every CSR value is written once, by one thread; no atomics, so results
// are bitwise reproducible.  Elements on patch borders are evaluated by every patch that touches
// them (2.2 times each on the 160x8x8 beam, 2.3 on 320x16x16), which costs less than a pass over memory.  The gradient goes
// through the same LDS before the states do.  Sums are FP64 in both precisions (an FP32 value is
// rounded once: 2.6e-8 from the exact Hessian, 6.4e-8 with the row gather's FP32 sums).
// What bounds it: latency.  A workgroup lives ~18k cycles, of which 6.6k are the element phase (two
// dependent gathers and ~350 FP64 operations), 6k the blocks (LDS reads at random slots), 2k the
// energy's compensated sum; HBM moves under 2 TB/s.
// Fused call, before (element matrices + row gather + separate energy) and after, us:
//   160x8x8 FP64 61.5 -> 16.7, 320x16x16 FP32 318 -> 62.4 (back to back, with the final sum).
// Slot stride 26 doubles (52 words): 16 consecutive slots start in 16 bank groups.
// ---------------------------------------------------------------------------------------------
namespace {

constexpr int kNpStride = 26;   // doubles per element state
constexpr int kNpGStride = 13;  // doubles per element gradient

// item k (16 bits) of a block of 8 or 4
__device__ __forceinline__ unsigned np_item(const uint4& w, int k) {
  const unsigned v = k < 2 ? w.x : (k < 4 ? w.y : (k < 6 ? w.z : w.w));
  return (k & 1) ? v >> 16 : v & 0xFFFFu;
}
__device__ __forceinline__ unsigned np_item(const uint2& w, int k) {
  const unsigned v = k < 2 ? w.x : w.y;
  return (k & 1) ? v >> 16 : v & 0xFFFFu;
}

// adds the 3x3 block of one element: H[i][k] += s1 qb[i] qa[k] + s2 qa[i] qb[k]; iso += vol 2 C1 D_a.D_b
__device__ __forceinline__ void np_add_block(const double* __restrict__ sS, unsigned it, double acc[9], double& iso) {
  const double* S = sS + int(it & 511u) * kNpStride;
  const double* qa = S + 3 * int((it >> 9) & 3u);
  const double* qb = S + 3 * int((it >> 11) & 3u);
  const double s1 = S[12], s2 = S[13];
  iso += S[18 + int(it >> 13)];
  const double a0 = qa[0], a1 = qa[1], a2 = qa[2], b0 = qb[0], b1 = qb[1], b2 = qb[2];
  const double u[3] = {s1 * b0, s1 * b1, s1 * b2}, v[3] = {s2 * a0, s2 * a1, s2 * a2};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    acc[3 * i + 0] = fma(u[i], a0, fma(v[i], b0, acc[3 * i + 0]));
    acc[3 * i + 1] = fma(u[i], a1, fma(v[i], b1, acc[3 * i + 1]));
    acc[3 * i + 2] = fma(u[i], a2, fma(v[i], b2, acc[3 * i + 2]));
  }
}

// adds the diagonal block of one element, h = 00 11 22 01 02 12
__device__ __forceinline__ void np_add_diag(const double* __restrict__ sS, unsigned it, double h[6]) {
  const int a = int(it >> 9);
  const double* S = sS + int(it & 511u) * kNpStride;
  const double q0 = S[3 * a], q1 = S[3 * a + 1], q2 = S[3 * a + 2], iso = S[14 + a];
  const double t = S[12] + S[13], t0 = t * q0, t1 = t * q1, t2 = t * q2;
  h[0] += fma(t0, q0, iso);
  h[1] += fma(t1, q1, iso);
  h[2] += fma(t2, q2, iso);
  h[3] = fma(t0, q1, h[3]);
  h[4] = fma(t0, q2, h[4]);
  h[5] = fma(t1, q2, h[5]);
}

template <typename HT>
__device__ __forceinline__ void np_store3(HT* dst, double a, double b, double c) {
  dst[0] = HT(a);
  dst[1] = HT(b);
  dst[2] = HT(c);
}

template <typename HT, bool WANT_E, bool WANT_G, bool WANT_H>
__global__ __launch_bounds__(kNodePatchThreads, 2) void tet_node_patch_kernel(
    fne_plan_desc d, FneNodePatches P, const double* __restrict__ x, const double* __restrict__ dvals,
    const double* __restrict__ f, double* __restrict__ g, HT* __restrict__ vals, EnergySum energy) {
  constexpr int kThreads = kNodePatchThreads;
  __shared__ double sS[(kNodePatchElems + 1) * (WANT_H ? kNpStride : kNpGStride)];
  __shared__ uint2 sDiag[kNodePatchNodes * 8];
  __shared__ uint32_t sInfo[kNodePatchNodes];
  __shared__ int2 sRow[kNodePatchNodes];  // first CSR entry and row length of the node's rows
  const int p = xcd_remap(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  const int node0 = P.pnode[p], nn = P.pnode[p + 1] - node0;
  const int eb = P.pelem_ptr[p], ne = P.pelem_ptr[p + 1] - eb;
  const int nown = WANT_E ? P.pown[p] : 0;
  const int pb = WANT_H ? P.pair_ptr[p] : 0, np = WANT_H ? P.pair_ptr[p + 1] - pb : 0;
  // everything the later phases index with is loaded under the element phase: the thread's first
  // block into registers, the nodes' diagonal items and rows into LDS
  int e = 0;
  int4 nc = make_int4(0, 0, 0, 0);
  const bool act = tid < ne;
  if (act) {
    e = P.pelem[eb + tid];
    nc = P.pelem_node[eb + tid];
  }
  uint2 pd = make_uint2(0, 0);
  uint4 items = make_uint4(0, 0, 0, 0);
  if (WANT_H && tid < np) {
    pd = P.pair[pb + tid];
    items = P.pair_items[pb + tid];
  }
  static_assert(8 * kNodePatchNodes <= kThreads, "one diagonal block of items per thread");
  uint2 ditems = make_uint2(0, 0);
  uint32_t info0 = 0;
  int row0 = 0, row1 = 0;
  if (tid < 8 * nn) ditems = P.diag_items[8 * node0 + tid];
  if (tid < nn) {
    info0 = P.diag[node0 + tid];
    if (WANT_H) {
      row0 = d.indptr[3 * (node0 + tid)];
      row1 = d.indptr[3 * (node0 + tid) + 1];
    }
  }
  double es = 0.0, ec = 0.0;
  if (WANT_E && f)
    for (int i = tid; i < 3 * nn; i += kThreads) acc_add(es, ec, -(f[3 * node0 + i] * x[3 * node0 + i]));
  double q[4][3], dd[10], s1 = 0.0, s2 = 0.0;
  if (act) {
    const int code[4] = {nc.x, nc.y, nc.z, nc.w};
    const int nfree = d.n_free / 3;
    const size_t n = d.n_elem;
    double y[4][3], D[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const double* src = code[a] < nfree ? x + 3 * size_t(code[a]) : dvals + 3 * size_t(code[a] - nfree);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        y[a][i] = src[i];
        D[a][i] = d.egeo[size_t(4 * i + a) * n + e];
      }
    }
    const double vol = d.egeo[12 * n + e];
    double F[3][3], C[3][3];
    const double det = tet_deformation(y, D, F, C);
    const double J = (d.flags & FNE_FLAG_ABS_DET) ? fabs(det) : det;
    const double C1 = d.param[0], D1 = d.param[1];
    if (WANT_E && tid < nown) {
      double E = vol * tet_density(F, J, C1, D1);
      if (d.eweight) E *= d.eweight[e];
      acc_add(es, ec, E);
    }
    if (WANT_G || WANT_H) {
      const double inv = 1.0 / det;
      const double c = 2.0 * D1 * J * (J - 1.0) - 2.0 * C1;
      s1 = -(vol * c);
      s2 = vol * (2.0 * D1 * J * (2.0 * J - 1.0));
      const double s0 = vol * 2.0 * C1;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) C[i][j] *= inv;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < 3; ++i) q[a][i] = dot3(C[i], D[a]);
      if (WANT_G) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int i = 0; i < 3; ++i) sS[tid * kNpGStride + 3 * a + i] = fma(s0, dot3(F[i], D[a]), -(s1 * q[a][i]));
      }
      if (WANT_H) {
#pragma unroll
        for (int a = 0; a < 4; ++a) dd[a] = s0 * dot3(D[a], D[a]);
        dd[4] = s0 * dot3(D[0], D[1]);
        dd[5] = s0 * dot3(D[0], D[2]);
        dd[6] = s0 * dot3(D[0], D[3]);
        dd[7] = s0 * dot3(D[1], D[2]);
        dd[8] = s0 * dot3(D[1], D[3]);
        dd[9] = s0 * dot3(D[2], D[3]);
      }
    }
  }
  // (stored only now: the loads above must not be waited for before the element's own)
  if (tid < 8 * nn) sDiag[tid] = ditems;
  if (tid < nn) {
    sInfo[tid] = info0;
    sRow[tid] = make_int2(row0, row1 - row0);
  }
  if (WANT_G) {
    if (tid < kNpGStride) sS[kNodePatchElems * kNpGStride + tid] = 0.0;
    __syncthreads();
    // eight threads per node
    for (int u = tid; u < 8 * nn; u += kThreads) {
      const int i = u >> 3, l = u & 7;
      double acc[3] = {0.0, 0.0, 0.0};
      auto add = [&](unsigned it) {
        const double* G = sS + int(it & 511u) * kNpGStride + 3 * int(it >> 9);
        acc[0] += G[0];
        acc[1] += G[1];
        acc[2] += G[2];
      };
      const uint2 w = sDiag[u];
#pragma unroll
      for (int k = 0; k < 4; ++k) add(np_item(w, k));
      const uint32_t info = sInfo[i];
      const int more = int((info >> 8) & 255u);
      if (more) {
        const uint4* xb = P.extra + P.extra_ptr[p] + int(info >> 16);
        for (int b = l; b < more; b += 8)
          for (int k = 0; k < 8; ++k) add(np_item(xb[b], k));
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        acc[c] += __shfl_xor(acc[c], 1, 8);
        acc[c] += __shfl_xor(acc[c], 2, 8);
        acc[c] += __shfl_xor(acc[c], 4, 8);
      }
      if (l < 3) {
        const int row = 3 * (node0 + i) + l;
        const double v = l == 0 ? acc[0] : (l == 1 ? acc[1] : acc[2]);
        g[row] = f ? v - f[row] : v;
      }
    }
    if (WANT_H) __syncthreads();
  }
  if (WANT_H) {
    if (tid < kNpStride) sS[kNodePatchElems * kNpStride + tid] = 0.0;
    if (act) {
      double* S = sS + tid * kNpStride;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < 3; ++i) S[3 * a + i] = q[a][i];
      S[12] = s1;
      S[13] = s2;
#pragma unroll
      for (int k = 0; k < 10; ++k) S[14 + k] = dd[k];
    }
    __syncthreads();
    const int np8 = (np + 7) & ~7;  // the diagonal blocks follow, eight threads each
    for (int u = tid; u < np8 + 8 * nn; u += kThreads) {
      if (u < np) {
        if (u != tid) {
          pd = P.pair[pb + u];
          items = P.pair_items[pb + u];
        }
        const int cnt = int((pd.x >> 14) & 15u);
        double acc[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, iso = 0.0;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
          if (k < cnt || k == 0) {  // two elements' loads in flight; an unused item adds zeros
            np_add_block(sS, np_item(items, k), acc, iso);
            np_add_block(sS, np_item(items, k + 1), acc, iso);
          }
        }
        const int more = int((pd.x >> 18) & 15u);
        if (more) {
          const uint4* xb = P.extra + P.extra_ptr[p] + int(pd.x >> 22);
          for (int b = 0; b < more; ++b)
            for (int k = 0; k < 8; ++k) np_add_block(sS, np_item(xb[b], k), acc, iso);
        }
        acc[0] += iso;
        acc[4] += iso;
        acc[8] += iso;
        const int2 row = sRow[pd.x & 63u];
        HT* dst = vals + row.x + 3 * int((pd.x >> 6) & 255u);
#pragma unroll
        for (int r = 0; r < 3; ++r) np_store3(dst + r * row.y, acc[3 * r], acc[3 * r + 1], acc[3 * r + 2]);
        if (pd.y != kNodePatchNone) {
          const int2 trow = sRow[pd.y & 63u];
          HT* tdst = vals + trow.x + 3 * int((pd.y >> 6) & 255u);
#pragma unroll
          for (int r = 0; r < 3; ++r) np_store3(tdst + r * trow.y, acc[r], acc[3 + r], acc[6 + r]);
        }
      } else if (u >= np8) {
        const int i = (u - np8) >> 3, l = (u - np8) & 7;
        double h[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // 00 11 22 01 02 12
        const uint2 w = sDiag[u - np8];
#pragma unroll
        for (int k = 0; k < 4; ++k) np_add_diag(sS, np_item(w, k), h);
        const uint32_t info = sInfo[i];
        const int more = int((info >> 8) & 255u);
        if (more) {
          const uint4* xb = P.extra + P.extra_ptr[p] + int(info >> 16);
          for (int b = l; b < more; b += 8)
            for (int k = 0; k < 8; ++k) np_add_diag(sS, np_item(xb[b], k), h);
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          h[k] += __shfl_xor(h[k], 1, 8);
          h[k] += __shfl_xor(h[k], 2, 8);
          h[k] += __shfl_xor(h[k], 4, 8);
        }
        const int2 row = sRow[i];
        HT* dst = vals + row.x + 3 * int(info & 255u);
        if (l == 0) np_store3(dst, h[0], h[3], h[4]);
        if (l == 1) np_store3(dst + row.y, h[3], h[1], h[5]);
        if (l == 2) np_store3(dst + 2 * row.y, h[4], h[5], h[2]);
      }
    }
  }
  if (WANT_E) {
    block_energy<kNodePatchThreads>(energy, p, es, ec);
  }
}

int launch_tet_node_patches(fne_plan* plan, bool want_e, bool want_g, bool want_h, const FneCall& c) {
  const FneNodePatches& P = plan->np;
  const dim3 grid(P.n_patch), block(kNodePatchThreads);
#define NP_GO(HT, E, G, H)                                                                                    \
  hipLaunchKernelGGL((tet_node_patch_kernel<HT, E, G, H>), grid, block, 0, c.stream, plan->d, P, c.x, c.dvals, c.f, \
                     c.g, (HT*)c.vals, fne_energy_sum(plan, kOpFused, P.n_patch, c.out))
  if (!want_h) {
    NP_GO(double, false, true, false);
  } else if (c.precision == FNE_FP32) {
    if (want_e && want_g) NP_GO(float, true, true, true);
    else if (want_e) NP_GO(float, true, false, true);
    else if (want_g) NP_GO(float, false, true, true);
    else NP_GO(float, false, false, true);
  } else {
    if (want_e && want_g) NP_GO(double, true, true, true);
    else if (want_e) NP_GO(double, true, false, true);
    else if (want_g) NP_GO(double, false, true, true);
    else NP_GO(double, false, false, true);
  }
#undef NP_GO
  FNE_LAUNCH_CHECK();
  if (want_e) return fne_finalize_energy(plan, P.n_patch, c.out, c.stream);
  return FNE_OK;
}

}  // namespace

int fne_launch_tet(fne_plan* plan, FneOp op, const FneCall& c) {
  const fne_plan_desc& d = plan->d;
  if (op == kOpEnergy) {
    // one element per thread, so that a small mesh is one pass of few blocks and few partial sums
    const int nb = std::max(1, std::min(plan->n_partials, (d.n_elem + kBlock - 1) / kBlock));
    hipLaunchKernelGGL(tet_energy_kernel, dim3(nb), dim3(kBlock), 0, c.stream, d, c.x, c.dvals, c.f,
                       fne_energy_sum(plan, kOpEnergy, nb, c.out));
    FNE_LAUNCH_CHECK();
    return fne_finalize_energy(plan, nb, c.out, c.stream);
  }
  if (plan->np.n_patch > 0 && (op == kOpFused || op == kOpHessian || op == kOpGradient)) {
    const bool want_h = op != kOpGradient;
    return launch_tet_node_patches(plan, op == kOpFused && c.out, c.g != nullptr, want_h, c);
  }
  if (op == kOpFused) {
    if (c.out) {
      const int rc = fne_launch_tet(plan, kOpEnergy, c);
      if (rc) return rc;
    }
    return fne_launch_tet(plan, kOpHessian, c);
  }
  if (op == kOpElementEval) {
    const int nb = (d.n_elem + kBlock - 1) / kBlock;
    if (nb > 0) {
      hipLaunchKernelGGL(tet_element_kernel, dim3(nb), dim3(kBlock), 0, c.stream, d, c.x, c.dvals, c.e_out,
                         c.ge_out, c.he_out);
      FNE_LAUNCH_CHECK();
    }
    return FNE_OK;
  }
  const bool want_h = (op == kOpHessian);
  const bool want_g = (op == kOpGradient) || (c.g != nullptr);
  if (d.flags & FNE_FLAG_ROW_GATHER) {
    if (!plan->mc_g || !plan->mc_h || !d.inc || !d.inc_ptr || (want_h && !d.pitem)) {
      fne_set_error("row-gather arrays missing from the tetrahedron plan");
      return FNE_EINVAL;
    }
    const int nb = (d.n_elem + kBlock - 1) / kBlock;
    if (nb > 0) {
      if (!want_h)
        hipLaunchKernelGGL((tet_store_kernel<double, true, false>), dim3(nb), dim3(kBlock), 0, c.stream, d, c.x,
                           c.dvals, plan->mc_g, (double*)plan->mc_h);
      else if (c.precision == FNE_FP32)
        hipLaunchKernelGGL((tet_store_kernel<float, true, true>), dim3(nb), dim3(kBlock), 0, c.stream, d, c.x,
                           c.dvals, plan->mc_g, (float*)plan->mc_h);
      else
        hipLaunchKernelGGL((tet_store_kernel<double, true, true>), dim3(nb), dim3(kBlock), 0, c.stream, d, c.x,
                           c.dvals, plan->mc_g, (double*)plan->mc_h);
      FNE_LAUNCH_CHECK();
    }
    return fne_launch_row_gather(plan, want_g, want_h, c);
  }
  if (d.n_patch <= 0) return FNE_OK;
  const size_t hsz = c.precision == FNE_FP32 ? 4 : 8;
  size_t shm = sizeof(double) * size_t(kTetStage) * size_t(d.chunk);
  if (want_h) shm += ((size_t(d.max_patch_nnz) * hsz + 7) / 8) * 8;
  if (shm > plan->max_lds) {
    fne_set_error("tet patch LDS request " + std::to_string(shm) + " B exceeds the device limit " +
                  std::to_string(plan->max_lds) + " B");
    return FNE_EINVAL;
  }
  const dim3 grid(d.n_patch), block(kBlock);
  if (!want_h) {
    hipLaunchKernelGGL((tet_patch_kernel<double, true, false>), grid, block, shm, c.stream, d, c.x, c.dvals,
                       c.f, c.g, (double*)nullptr);
  } else if (c.precision == FNE_FP32) {
    if (want_g)
      hipLaunchKernelGGL((tet_patch_kernel<float, true, true>), grid, block, shm, c.stream, d, c.x, c.dvals,
                         c.f, c.g, (float*)c.vals);
    else
      hipLaunchKernelGGL((tet_patch_kernel<float, false, true>), grid, block, shm, c.stream, d, c.x, c.dvals,
                         c.f, c.g, (float*)c.vals);
  } else {
    if (want_g)
      hipLaunchKernelGGL((tet_patch_kernel<double, true, true>), grid, block, shm, c.stream, d, c.x, c.dvals,
                         c.f, c.g, (double*)c.vals);
    else
      hipLaunchKernelGGL((tet_patch_kernel<double, false, true>), grid, block, shm, c.stream, d, c.x, c.dvals,
                         c.f, c.g, (double*)c.vals);
  }
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}
