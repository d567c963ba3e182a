// Per-node MLP for the learned warm start: BF16-MFMA forward, backward and Adam.
//
// Network: n_layers linear layers y = W x + b (W: [out][in] BF16, b: FP32), tanh after every
// layer but the last.  Activations, gradients and the optimiser state are FP32; every matrix
// product runs on v_mfma_f32_16x16x16bf16_1k with BF16 operands and FP32 accumulation.
//
// Networks of width <= 128 (every width of the nodal predictors) run in four launches: the whole
// forward pass, the whole chain of hidden gradients, every weight gradient, and the reduction of
// the partial sums (see "Narrow networks" below).  Wider ones take one GEMM launch per product:
// C[m][n] = sum_k A(m,k) B(k,n) with arbitrary element strides for A and B (so X W^T, dZ^T H and
// dZ W are the same kernel), a 64x64 block tile, 16-deep K steps staged through LDS as BF16, four
// wavefronts each owning a 32x32 sub-tile (2x2 MFMA tiles).  Long reductions (the weight and bias
// gradients sum over all nodes) are split into FP32 partials that a second kernel adds in a fixed
// order, so every result is bitwise reproducible.
#include "fne_common.h"

namespace {

typedef short mlp_s4 __attribute__((ext_vector_type(4)));
typedef float mlp_f4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float(unsigned(h) << 16); }

__device__ __forceinline__ unsigned short load_bf(const float* p, size_t i) { return f2bf(p[i]); }
__device__ __forceinline__ unsigned short load_bf(const unsigned short* p, size_t i) { return p[i]; }

enum MlpEpi : int { kEpiNone = 0, kEpiTanh = 1, kEpiDTanh = 2 };

struct GemmArgs {
  int M, N, K;
  const void* A;
  long sam, sak;
  const void* B;
  long sbk, sbn;
  float* C;       // [M][ldc] (final) or partials [splits][M][N]
  long ldc;
  const float* bias;  // [N] or null
  const float* H;     // kEpiDTanh: C *= (1 - H^2), H [M][ldh]
  long ldh;
  int epi;
  int kchunk;         // K range per grid.z slice
  int split;          // 1: write raw partials
};

constexpr int kT = 64;   // block tile
constexpr int kKs = 16;  // K step

template <typename TA, typename TB>
__global__ __launch_bounds__(256) void mlp_gemm_kernel(GemmArgs g) {
  __shared__ unsigned short As[kT][kKs + 4];
  __shared__ unsigned short Bs[kKs][kT + 4];
  const TA* A = reinterpret_cast<const TA*>(g.A);
  const TB* B = reinterpret_cast<const TB*>(g.B);
  const int m0 = blockIdx.y * kT, n0 = blockIdx.x * kT;
  const int kbeg = blockIdx.z * g.kchunk;
  const int kend = min(g.K, kbeg + g.kchunk);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wy = wave >> 1, wx = wave & 1;
  mlp_f4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = mlp_f4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = kbeg; k0 < kend; k0 += kKs) {
    // 64x16 A elements and 16x64 B elements, 4 of each per thread
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int idx = tid + 256 * r;
      const int am = idx / kKs, ak = idx % kKs;  // A tile [m][k]
      const int gm = m0 + am, gk = k0 + ak;
      As[am][ak] = (gm < g.M && gk < kend) ? load_bf(A, size_t(gm) * g.sam + size_t(gk) * g.sak) : 0;
      const int bk = idx / kT, bn = idx % kT;  // B tile [k][n]
      const int gk2 = k0 + bk, gn = n0 + bn;
      Bs[bk][bn] = (gn < g.N && gk2 < kend) ? load_bf(B, size_t(gk2) * g.sbk + size_t(gn) * g.sbn) : 0;
    }
    __syncthreads();
    const int kq = 4 * (lane >> 4);
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const int row = wy * 32 + ti * 16 + (lane & 15);
      mlp_s4 a;
      a[0] = (short)As[row][kq + 0];
      a[1] = (short)As[row][kq + 1];
      a[2] = (short)As[row][kq + 2];
      a[3] = (short)As[row][kq + 3];
#pragma unroll
      for (int tj = 0; tj < 2; ++tj) {
        const int col = wx * 32 + tj * 16 + (lane & 15);
        mlp_s4 b;
        b[0] = (short)Bs[kq + 0][col];
        b[1] = (short)Bs[kq + 1][col];
        b[2] = (short)Bs[kq + 2][col];
        b[3] = (short)Bs[kq + 3][col];
        acc[ti][tj] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[ti][tj], 0, 0, 0);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wy * 32 + ti * 16 + 4 * (lane >> 4) + r;
        const int gn = n0 + wx * 32 + tj * 16 + (lane & 15);
        if (gm >= g.M || gn >= g.N) continue;
        float v = acc[ti][tj][r];
        if (g.split) {
          g.C[(size_t(blockIdx.z) * g.M + gm) * g.N + gn] = v;
          continue;
        }
        if (g.bias) v += g.bias[gn];
        if (g.epi == kEpiTanh) v = tanhf(v);
        if (g.epi == kEpiDTanh) {
          const float h = g.H[size_t(gm) * g.ldh + gn];
          v *= 1.0f - h * h;
        }
        g.C[size_t(gm) * g.ldc + gn] = v;
      }
}

// out[i] = sum_s part[s][i] in split order
__global__ __launch_bounds__(256) void mlp_split_reduce_kernel(const float* __restrict__ part, int splits, long n,
                                                               float* __restrict__ out) {
  const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int k = 0; k < splits; ++k) s += part[size_t(k) * n + i];
  out[i] = s;
}

// column sums of X [rows][cols] over row chunks of kColsumRows -> part[chunk][cols].  A thread
// sums kColsumRows / 4 rows of one column (64 neighbouring columns per wavefront, so loads
// coalesce), the four wavefronts' sums are added in order.
constexpr int kColsumRows = 256;

__global__ __launch_bounds__(256) void mlp_colsum_kernel(const float* __restrict__ X, long rows, int cols,
                                                         float* __restrict__ part) {
  __shared__ float sums[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.y * 64 + lane;
  const long r0 = long(blockIdx.x) * kColsumRows;
  float s = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int r = wave; r < kColsumRows; r += 4)
      if (r0 + r < rows) s += X[size_t(r0 + r) * cols + c];
  }
  sums[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && c < cols)
    part[size_t(blockIdx.x) * cols + c] = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
}

__global__ __launch_bounds__(256) void mlp_adam_kernel(long n, float* __restrict__ w, unsigned short* __restrict__ wb,
                                                       const float* __restrict__ grad, float* __restrict__ m,
                                                       float* __restrict__ v, float lr, float b1, float b2,
                                                       float eps, float c1, float c2, float wd) {
  const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = grad[i] + wd * w[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ __launch_bounds__(256) void mlp_to_bf16_kernel(long n, const float* __restrict__ w,
                                                          unsigned short* __restrict__ wb) {
  const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) wb[i] = f2bf(w[i]);
}

// ---------------------------------------------------------------------------------------------
// Narrow networks (every width <= kNarrow = 128).
//
// A 10-128x4-3 network on 16,384 rows is 5 GFLOP and 8 MB per hidden activation: one launch per
// product (25 of them, 64x64 tiles read and written through memory, a bias-gradient column sum of
// 1,024 serial loads per thread) took 1,475 us on an MI355X for forward + backward, of which the
// arithmetic needs under 10.  Here a workgroup keeps its R rows in LDS (BF16) through all
// layers; a wavefront holds the weight fragments of its 32 columns in registers, so a layer costs
// one LDS read per 16x16 input tile and two MFMAs.  The order of every accumulation (16-deep
// steps, k ascending, then bias, tanh) is that of the GEMM kernel: activations and hidden
// gradients have the same bits in both forms.  Measured (forward + backward of 10-128x4-3, 16,384
// rows): 1,475 -> 113 us, of which forward 37.6 (tanhf and 34 MB of activations written), chain
// 34.3, weight gradients 34.2 (67 MB read at 2 TB/s), reduction 5.7.
// ---------------------------------------------------------------------------------------------
constexpr int kNarrow = 128;
constexpr int kNarrowStride = kNarrow + 8;  // LDS row of BF16: 272 B, so 16 rows start in 16 bank groups
static_assert(kNarrowStride * sizeof(unsigned short) % 8 == 0, "rows are read in vectors of 8 bytes");

typedef __bf16 mlp_b8 __attribute__((ext_vector_type(8)));
typedef unsigned short mlp_u8 __attribute__((ext_vector_type(8)));

// FP32 -> BF16 by the conversion instruction (round to nearest even, as f2bf; a NaN stays a NaN)
__device__ __forceinline__ unsigned short cvt_bf(float f) {
  return __builtin_bit_cast(unsigned short, static_cast<__bf16>(f));
}

// rows per workgroup: 32 put two workgroups on every CU at 16,384 rows (forward + chain 71.8 us;
// 16 rows 80.7: the weights are loaded twice as often; 64 rows 94.9: one workgroup per CU)
constexpr int kNarrowRows = 32;

// layer l's 16x16x16 products over the workgroup's rows: acc[mt][j] for column tiles 2 wave + j
template <int R>
__device__ __forceinline__ void narrow_products(const unsigned short (*sA)[kNarrowStride], const mlp_s4 (*bf)[8],
                                                int ksteps, int lane, mlp_f4 (*acc)[2]) {
#pragma unroll
  for (int mt = 0; mt < R / 16; ++mt) acc[mt][0] = acc[mt][1] = mlp_f4{0.f, 0.f, 0.f, 0.f};
  const int kq = 4 * (lane >> 4);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if (s < ksteps) {
#pragma unroll
      for (int mt = 0; mt < R / 16; ++mt) {
        const mlp_s4 a = *reinterpret_cast<const mlp_s4*>(&sA[mt * 16 + (lane & 15)][16 * s + kq]);
        acc[mt][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bf[0][s], acc[mt][0], 0, 0, 0);
        acc[mt][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bf[1][s], acc[mt][1], 0, 0, 0);
      }
    }
  }
}

// the workgroup's rows of X [n][cols] as BF16, columns padded with zeros to a multiple of 16
template <int R>
__device__ __forceinline__ void narrow_load_rows(const float* __restrict__ X, long n, long row0, int cols,
                                                 unsigned short (*sA)[kNarrowStride]) {
  const int kp = (cols + 15) & ~15;
  for (int i = threadIdx.x; i < R * kp; i += 256) {
    const int r = i / kp, k = i - r * kp;
    sA[r][k] = (row0 + r < n && k < cols) ? cvt_bf(X[size_t(row0 + r) * cols + k]) : 0;
  }
}

template <int R>
__global__ __launch_bounds__(256) void mlp_narrow_forward_kernel(fne_mlp_desc net, long n, const float* __restrict__ x,
                                                                 float* __restrict__ y, float* __restrict__ acts) {
  __shared__ __align__(16) unsigned short sA[R][kNarrowStride];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c15 = lane & 15, kq = 4 * (lane >> 4);
  const long row0 = long(blockIdx.x) * R;
  narrow_load_rows<R>(x, n, row0, net.dims[0], sA);
  size_t off = 0;
  for (int l = 0; l < net.n_layers; ++l) {
    const int din = net.dims[l], dout = net.dims[l + 1];
    const bool last = l == net.n_layers - 1;
    const unsigned short* W = net.w[l];
    const int ksteps = (din + 15) >> 4;
    const bool vec = (din & 3) == 0 && (reinterpret_cast<uintptr_t>(W) & 7u) == 0;  // 8-byte fragments
    mlp_s4 bf[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = (2 * wave + j) * 16 + c15;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        mlp_s4 b = {0, 0, 0, 0};
        const int k = 16 * s + kq;
        if (s < ksteps && col < dout) {
          const unsigned short* w = W + size_t(col) * din + k;  // B(k, col) = W[col][k]
          if (vec) {
            if (k < din) b = *reinterpret_cast<const mlp_s4*>(w);
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (k + q < din) b[q] = (short)w[q];
          }
        }
        bf[j][s] = b;
      }
    }
    __syncthreads();  // the rows are in LDS
    mlp_f4 acc[R / 16][2];
    narrow_products<R>(sA, bf, ksteps, lane, acc);
    __syncthreads();  // every read of the rows is done
    float* out = last ? y : acts + off;
    const float* bias = net.b[l];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = (2 * wave + j) * 16 + c15;
      if (col >= ((dout + 15) & ~15)) continue;
      const float bj = col < dout ? bias[col] : 0.f;
#pragma unroll
      for (int mt = 0; mt < R / 16; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = mt * 16 + kq + r;
          float v = 0.f;
          if (col < dout) {
            v = acc[mt][j][r] + bj;
            if (!last) v = tanhf(v);
            if (row0 + row < n) out[size_t(row0 + row) * dout + col] = v;
          }
          if (!last) sA[row][col] = cvt_bf(v);
        }
    }
    if (!last) off += size_t(n) * dout;
  }
}

// hidden gradients dz_{l-1} = (dz_l W_l) (1 - h_{l-1}^2) for l = L-1 .. 1, written back to back in
// acts' layout, and the column sums of every dz over the workgroup's rows (cpart [blocks][sum of
// widths], layer l at the sum of the widths before it)
template <int R>
__global__ __launch_bounds__(256) void mlp_narrow_chain_kernel(fne_mlp_desc net, long n,
                                                               const float* __restrict__ acts,
                                                               const float* __restrict__ dy, float* __restrict__ dz,
                                                               float* __restrict__ cpart, int widths) {
  __shared__ __align__(16) unsigned short sA[R][kNarrowStride];
  __shared__ __align__(16) unsigned short sW[kNarrow][kNarrowStride];  // W_l transposed: [input][output]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c15 = lane & 15, kq = 4 * (lane >> 4);
  const long row0 = long(blockIdx.x) * R;
  const int L = net.n_layers;
  float* cp = cpart + size_t(blockIdx.x) * widths;
  size_t off = 0;  // of dz_{L-2} in acts' layout
  int coff = widths - net.dims[L];
  for (int l = 0; l + 2 < L; ++l) off += size_t(n) * net.dims[l + 1];
  narrow_load_rows<R>(dy, n, row0, net.dims[L], sA);
  for (int c = threadIdx.x; c < net.dims[L]; c += 256) {
    float s = 0.f;
    for (int r = 0; r < R; ++r)
      if (row0 + r < n) s += dy[size_t(row0 + r) * net.dims[L] + c];
    cp[coff + c] = s;
  }
  for (int l = L - 1; l > 0; --l) {
    const int din = net.dims[l], dout = net.dims[l + 1];
    const unsigned short* W = net.w[l];
    const int ksteps = (dout + 15) >> 4;
    // four rows by eight columns of W at a time (16-byte loads where the rows allow), zero-padded
    // to whole K steps
    const int kp = 16 * ksteps;
    const bool vec = (din & 7) == 0 && (reinterpret_cast<uintptr_t>(W) & 15u) == 0;
    const int cg = (din + 7) >> 3;
    for (int u = threadIdx.x; u < (kp >> 2) * cg; u += 256) {
      const int k0 = (u / cg) * 4, col0 = (u % cg) * 8;
      mlp_u8 w[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        w[q] = mlp_u8{0, 0, 0, 0, 0, 0, 0, 0};
        if (k0 + q < dout) {
          const unsigned short* src = W + size_t(k0 + q) * din + col0;
          if (vec) {
            w[q] = *reinterpret_cast<const mlp_u8*>(src);
          } else {
#pragma unroll
            for (int t = 0; t < 8; ++t)
              if (col0 + t < din) w[q][t] = src[t];
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 8; ++t)
        *reinterpret_cast<mlp_s4*>(&sW[col0 + t][k0]) =
            mlp_s4{short(w[0][t]), short(w[1][t]), short(w[2][t]), short(w[3][t])};
    }
    const float* H = acts + off;
    float hv[2][R / 16][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mt = 0; mt < R / 16; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = (2 * wave + j) * 16 + c15;
          const long row = row0 + mt * 16 + kq + r;
          hv[j][mt][r] = (col < din && row < n) ? H[size_t(row) * din + col] : 0.f;
        }
    __syncthreads();  // rows and weights are in LDS
    mlp_s4 bf[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (s < ksteps) bf[j][s] = *reinterpret_cast<const mlp_s4*>(&sW[(2 * wave + j) * 16 + c15][16 * s + kq]);
    mlp_f4 acc[R / 16][2];
    narrow_products<R>(sA, bf, ksteps, lane, acc);
    __syncthreads();  // every read of the rows and weights is done
    coff -= din;
    float* out = dz + off;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = (2 * wave + j) * 16 + c15;
      if (col >= ((din + 15) & ~15)) continue;
      float s = 0.f;
#pragma unroll
      for (int mt = 0; mt < R / 16; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = mt * 16 + kq + r;
          float v = 0.f;
          if (col < din && row0 + row < n) {
            const float h = hv[j][mt][r];
            v = acc[mt][j][r] * (1.0f - h * h);
            out[size_t(row0 + row) * din + col] = v;
            s += v;
          }
          if (l > 1) sA[row][col] = cvt_bf(v);
        }
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (lane < 16 && col < din) cp[coff + col] = s;
    }
    if (l > 1) off -= size_t(n) * net.dims[l - 1];
  }
}

// weight gradients dW_l = dz_l^T h_{l-1}, all layers in one launch: blockIdx.y is the layer,
// blockIdx.x a chunk of rows; a workgroup reads its rows of both factors once and holds the whole
// dout x din product (four wavefronts of 64x64).  Rows are transposed into LDS as BF16, 32 at a
// time (one K step of the 16x16x32 MFMA), the next 32 being loaded meanwhile.
constexpr int kWgStride = 40;  // LDS row of 32 BF16: 80 B, 16-byte aligned fragments in 16 bank groups
static_assert(kWgStride * sizeof(unsigned short) % 16 == 0, "rows are written and read in vectors of 16 bytes");

struct MlpWgradArgs {
  const float* dz[FNE_MLP_MAX_LAYERS];  // [n][dims[l+1]]
  const float* h[FNE_MLP_MAX_LAYERS];   // [n][dims[l]]
  int dims[FNE_MLP_MAX_LAYERS + 1];
  long woff[FNE_MLP_MAX_LAYERS];  // layer l's weights within a slice of partials
  long weights;                   // length of a slice
};

__global__ __launch_bounds__(256) void mlp_narrow_wgrad_kernel(MlpWgradArgs g, long n, long chunk,
                                                               float* __restrict__ part) {
  __shared__ __align__(16) unsigned short sD[kNarrow][kWgStride];
  __shared__ __align__(16) unsigned short sH[kNarrow][kWgStride];
  const int l = blockIdx.y;
  const int M = g.dims[l + 1], N = g.dims[l];
  const float* D = g.dz[l];
  const float* H = g.h[l];
  const long r0 = long(blockIdx.x) * chunk, r1 = r0 + chunk < n ? r0 + chunk : n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const int c = tid & 127, rb = (tid >> 7) * 16;  // this thread's column and 16 of the 32 rows
  mlp_f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = mlp_f4{0.f, 0.f, 0.f, 0.f};
  float fd[16], fh[16];
  auto load = [&](long base) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const long r = base + rb + i;
      fd[i] = (r < r1 && c < M) ? D[size_t(r) * M + c] : 0.f;
      fh[i] = (r < r1 && c < N) ? H[size_t(r) * N + c] : 0.f;
    }
  };
  load(r0);
  for (long base = r0; base < r1; base += 32) {
    mlp_u8 d0, d1, h0, h1;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      d0[i] = cvt_bf(fd[i]);
      d1[i] = cvt_bf(fd[8 + i]);
      h0[i] = cvt_bf(fh[i]);
      h1[i] = cvt_bf(fh[8 + i]);
    }
    __syncthreads();  // the previous step's fragments have been read
    *reinterpret_cast<mlp_u8*>(&sD[c][rb]) = d0;
    *reinterpret_cast<mlp_u8*>(&sD[c][rb + 8]) = d1;
    *reinterpret_cast<mlp_u8*>(&sH[c][rb]) = h0;
    *reinterpret_cast<mlp_u8*>(&sH[c][rb + 8]) = h1;
    if (base + 32 < r1) load(base + 32);
    __syncthreads();
    mlp_b8 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (wm + 16 * i < M) a[i] = *reinterpret_cast<const mlp_b8*>(&sD[wm + 16 * i + (lane & 15)][8 * (lane >> 4)]);
      if (wn + 16 * i < N) b[i] = *reinterpret_cast<const mlp_b8*>(&sH[wn + 16 * i + (lane & 15)][8 * (lane >> 4)]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (wm + 16 * i < M && wn + 16 * j < N)  // uniform over the wavefront
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }
  float* out = part + size_t(blockIdx.x) * g.weights + g.woff[l];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = wm + 16 * i + 4 * (lane >> 4) + r, k = wn + 16 * j + (lane & 15);
        if (m < M && k < N) out[size_t(m) * N + k] = acc[i][j][r];
      }
}

// sums of the partial weight gradients over the row chunks (blocks [0, wblocks)) and of the partial
// column sums over the chain's workgroups (one wavefront per column), both in index order per thread
struct MlpGrads {
  float* dw[FNE_MLP_MAX_LAYERS];
  float* db[FNE_MLP_MAX_LAYERS];
};

__global__ __launch_bounds__(256) void mlp_narrow_reduce_kernel(MlpWgradArgs g, int layers, MlpGrads out, int wblocks,
                                                                const float* __restrict__ part, int splits,
                                                                const float* __restrict__ cpart, int cblocks,
                                                                int widths) {
  if (int(blockIdx.x) < wblocks) {
    const long i = long(blockIdx.x) * 256 + threadIdx.x;
    if (i >= g.weights) return;
    float s = 0.f;
#pragma unroll 8
    for (int k = 0; k < splits; ++k) s += part[size_t(k) * g.weights + i];
    int l = 0;
    while (l + 1 < layers && i >= g.woff[l + 1]) ++l;
    out.dw[l][i - g.woff[l]] = s;
    return;
  }
  const int col = (int(blockIdx.x) - wblocks) * 4 + int(threadIdx.x >> 6);
  if (col >= widths) return;
  const int lane = threadIdx.x & 63;
  float s = 0.f;
  for (int k = lane; k < cblocks; k += 64) s += cpart[size_t(k) * widths + col];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) {
    int l = 0, c = col;
    while (c >= g.dims[l + 1]) c -= g.dims[++l];
    out.db[l][c] = s;
  }
}

template <typename TA, typename TB>
int run_gemm(GemmArgs g, int splits, hipStream_t s, int* used_splits = nullptr) {
  if (g.M <= 0 || g.N <= 0) return FNE_OK;
  if (splits < 1) splits = 1;
  g.kchunk = ((g.K + splits - 1) / splits + kKs - 1) / kKs * kKs;
  if (g.kchunk < kKs) g.kchunk = kKs;
  splits = (g.K + g.kchunk - 1) / g.kchunk;
  if (splits < 1) splits = 1;
  g.split = splits > 1 ? 1 : g.split;
  if (used_splits) *used_splits = splits;
  dim3 grid((g.N + kT - 1) / kT, (g.M + kT - 1) / kT, splits);
  hipLaunchKernelGGL((mlp_gemm_kernel<TA, TB>), grid, dim3(256), 0, s, g);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

bool net_ok(const fne_mlp_desc* net) {
  if (!net || net->n_layers < 1 || net->n_layers > FNE_MLP_MAX_LAYERS) return false;
  for (int l = 0; l < net->n_layers; ++l)
    if (net->dims[l] < 1 || net->dims[l + 1] < 1 || !net->w[l] || !net->b[l]) return false;
  return true;
}

long max_width(const fne_mlp_desc* net) {
  long w = 0;
  for (int l = 0; l <= net->n_layers; ++l) w = net->dims[l] > w ? net->dims[l] : w;
  return w;
}

constexpr int kWgradSplits = 64;
constexpr int kWgradRows = 128;  // rows of a chunk at least (narrow networks)

bool narrow(const fne_mlp_desc* net) { return max_width(net) <= kNarrow; }

// widths of all layer outputs, weights of all layers, row chunks of the weight gradients
struct NarrowSizes {
  long hidden = 0, widths = 0, weights = 0, blocks = 0, chunk = 0, splits = 0;
};

NarrowSizes narrow_sizes(const fne_mlp_desc* net, int64_t n) {
  NarrowSizes z;
  for (int l = 0; l < net->n_layers; ++l) {
    z.widths += net->dims[l + 1];
    z.weights += long(net->dims[l]) * net->dims[l + 1];
  }
  z.hidden = z.widths - net->dims[net->n_layers];
  z.blocks = (n + kNarrowRows - 1) / kNarrowRows;
  // whole 32-row steps, at most kWgradSplits chunks of at least kWgradRows rows: 64 chunks x 5 layers give
  // every CU a workgroup (39.9 us with the reduction at 16,384 rows; 128 chunks 41.6: more partial
  // sums to reduce)
  z.chunk = ((n + kWgradSplits - 1) / kWgradSplits + 31) / 32 * 32;
  if (z.chunk < kWgradRows) z.chunk = kWgradRows;
  z.splits = (n + z.chunk - 1) / z.chunk;
  return z;
}

int narrow_backward(const fne_mlp_desc* net, long n, const float* x, const float* acts, const float* dy,
                    float* const* dw, float* const* db, void* workspace, hipStream_t s) {
  const NarrowSizes z = narrow_sizes(net, n);
  const int L = net->n_layers;
  float* dz = reinterpret_cast<float*>(workspace);
  float* part = dz + size_t(n) * z.hidden;
  float* cpart = part + size_t(z.splits) * z.weights;
  hipLaunchKernelGGL(mlp_narrow_chain_kernel<kNarrowRows>, dim3(z.blocks), dim3(256), 0, s, *net, n, acts, dy, dz,
                     cpart, int(z.widths));
  FNE_LAUNCH_CHECK();
  MlpWgradArgs g{};
  MlpGrads out{};
  size_t off = 0;
  for (int l = 0; l < L; ++l) {
    g.dims[l] = net->dims[l];
    g.h[l] = l == 0 ? x : acts + off - size_t(n) * net->dims[l];
    g.dz[l] = l == L - 1 ? dy : dz + off;
    g.woff[l] = g.weights;
    g.weights += long(net->dims[l]) * net->dims[l + 1];
    if (l < L - 1) off += size_t(n) * net->dims[l + 1];
    out.dw[l] = dw[l];
    out.db[l] = db[l];
  }
  g.dims[L] = net->dims[L];
  hipLaunchKernelGGL(mlp_narrow_wgrad_kernel, dim3(z.splits, L), dim3(256), 0, s, g, n, z.chunk, part);
  FNE_LAUNCH_CHECK();
  const int wblocks = int((z.weights + 255) / 256), cb = int((z.widths + 3) / 4);
  hipLaunchKernelGGL(mlp_narrow_reduce_kernel, dim3(wblocks + cb), dim3(256), 0, s, g, L, out, wblocks, part,
                     int(z.splits), cpart, int(z.blocks), int(z.widths));
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

}  // namespace

extern "C" {

int64_t fne_mlp_workspace_bytes(const fne_mlp_desc* net, int64_t n) {
  if (!net_ok(net) || n < 0) return FNE_EINVAL;
  if (narrow(net)) {
    // every hidden gradient, the weight gradients' partials, the column sums' partials.  Chunks grow in
    // steps of 32 rows, so their number falls again above 64 chunks of 128 rows: the most that any
    // smaller n has, so that a workspace serves every smaller batch too
    const NarrowSizes z = narrow_sizes(net, n);
    const long splits = n < kWgradSplits * kWgradRows ? (n + kWgradRows - 1) / kWgradRows : kWgradSplits;
    return int64_t(sizeof(float)) * (n * z.hidden + splits * z.weights + z.blocks * z.widths);
  }
  const long w = max_width(net);
  const long chunks = (n + kColsumRows - 1) / kColsumRows;
  // two dZ buffers, weight-gradient split partials, bias-gradient chunk partials
  return int64_t(sizeof(float)) * (2 * n * w + long(kWgradSplits) * w * w + chunks * w);
}

int fne_mlp_forward(const fne_mlp_desc* net, int64_t n, const float* x, float* y, float* acts,
                    fne_stream_t stream) {
  if (!net_ok(net) || n < 0 || !x || !y) {
    fne_set_error("fne_mlp_forward: invalid arguments");
    return FNE_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  if (narrow(net)) {
    if (net->n_layers > 1 && !acts) {
      fne_set_error("fne_mlp_forward: activation buffer required");
      return FNE_EINVAL;
    }
    if (n == 0) return FNE_OK;
    hipLaunchKernelGGL(mlp_narrow_forward_kernel<kNarrowRows>, dim3((n + kNarrowRows - 1) / kNarrowRows), dim3(256), 0,
                       s, *net, long(n), x, y, acts);
    FNE_LAUNCH_CHECK();
    return FNE_OK;
  }
  const float* in = x;
  size_t off = 0;
  for (int l = 0; l < net->n_layers; ++l) {
    const int din = net->dims[l], dout = net->dims[l + 1];
    const bool last = l == net->n_layers - 1;
    float* out = last ? y : acts + off;
    if (!last && !acts) {
      fne_set_error("fne_mlp_forward: activation buffer required");
      return FNE_EINVAL;
    }
    GemmArgs g{};
    g.M = int(n);
    g.N = dout;
    g.K = din;
    g.A = in;
    g.sam = din;
    g.sak = 1;
    g.B = net->w[l];  // B(k, n) = W[n][k]
    g.sbk = 1;
    g.sbn = din;
    g.C = out;
    g.ldc = dout;
    g.bias = net->b[l];
    g.epi = last ? kEpiNone : kEpiTanh;
    const int rc = run_gemm<float, unsigned short>(g, 1, s);
    if (rc) return rc;
    if (!last) off += size_t(n) * dout;
    in = out;
  }
  return FNE_OK;
}

int fne_mlp_backward(const fne_mlp_desc* net, int64_t n, const float* x, const float* acts, const float* dy,
                     float* const* dw, float* const* db, void* workspace, int64_t ws_bytes, fne_stream_t stream) {
  if (!net_ok(net) || n < 1 || !x || !dy || !dw || !db || !workspace) {
    fne_set_error("fne_mlp_backward: invalid arguments");
    return FNE_EINVAL;
  }
  if (ws_bytes < fne_mlp_workspace_bytes(net, n)) {
    fne_set_error("fne_mlp_backward: workspace too small");
    return FNE_EINVAL;
  }
  if (net->n_layers > 1 && !acts) {
    fne_set_error("fne_mlp_backward: activation buffer required");
    return FNE_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  if (narrow(net)) return narrow_backward(net, n, x, acts, dy, dw, db, workspace, s);
  const long w = max_width(net);
  float* dz0 = reinterpret_cast<float*>(workspace);
  float* dz1 = dz0 + size_t(n) * w;
  float* part = dz1 + size_t(n) * w;
  float* cpart = part + size_t(kWgradSplits) * w * w;
  const long chunks = (n + kColsumRows - 1) / kColsumRows;
  // offsets of each hidden activation in acts
  size_t offs[FNE_MLP_MAX_LAYERS + 1];
  offs[0] = 0;
  for (int l = 0; l + 1 < net->n_layers; ++l) offs[l + 1] = offs[l] + size_t(n) * net->dims[l + 1];
  const float* dz = dy;  // gradient w.r.t. the pre-activation of layer l
  float* bufs[2] = {dz0, dz1};
  for (int l = net->n_layers - 1; l >= 0; --l) {
    const int din = net->dims[l], dout = net->dims[l + 1];
    const float* hin = l == 0 ? x : acts + offs[l - 1];
    // dW[j][k] = sum_i dz[i][j] hin[i][k]  (M = dout, N = din, K = n): split over nodes
    GemmArgs g{};
    g.M = dout;
    g.N = din;
    g.K = int(n);
    g.A = dz;
    g.sam = 1;
    g.sak = dout;
    g.B = hin;
    g.sbk = din;
    g.sbn = 1;
    g.C = part;
    g.ldc = din;
    g.split = 1;
    int splits = 1;
    int rc = run_gemm<float, float>(g, kWgradSplits, s, &splits);
    if (rc) return rc;
    const long nw = long(dout) * din;
    hipLaunchKernelGGL(mlp_split_reduce_kernel, dim3((nw + 255) / 256), dim3(256), 0, s, part, splits, nw, dw[l]);
    FNE_LAUNCH_CHECK();
    // db[j] = sum_i dz[i][j]
    hipLaunchKernelGGL(mlp_colsum_kernel, dim3(chunks, (dout + 63) / 64), dim3(256), 0, s, dz, long(n), dout,
                       cpart);
    FNE_LAUNCH_CHECK();
    hipLaunchKernelGGL(mlp_split_reduce_kernel, dim3((dout + 255) / 256), dim3(256), 0, s, cpart, int(chunks),
                       long(dout), db[l]);
    FNE_LAUNCH_CHECK();
    if (l == 0) break;
    // dz_prev[i][k] = (sum_j dz[i][j] W[j][k]) * (1 - h[i][k]^2)
    float* out = bufs[l & 1];
    GemmArgs h{};
    h.M = int(n);
    h.N = din;
    h.K = dout;
    h.A = dz;
    h.sam = dout;
    h.sak = 1;
    h.B = net->w[l];  // B(k=j, n=k) = W[j][k]
    h.sbk = din;
    h.sbn = 1;
    h.C = out;
    h.ldc = din;
    h.H = hin;
    h.ldh = din;
    h.epi = kEpiDTanh;
    rc = run_gemm<float, unsigned short>(h, 1, s);
    if (rc) return rc;
    dz = out;
  }
  return FNE_OK;
}

int fne_mlp_adam(int64_t n, float* w, uint16_t* w_bf16, const float* grad, float* m, float* v, float lr,
                 float beta1, float beta2, float eps, float weight_decay, int32_t step, fne_stream_t stream) {
  if (n < 0 || !w || !grad || !m || !v || step < 1) {
    fne_set_error("fne_mlp_adam: invalid arguments");
    return FNE_EINVAL;
  }
  if (n == 0) return FNE_OK;
  const float c1 = 1.f - powf(beta1, float(step));
  const float c2 = 1.f - powf(beta2, float(step));
  hipLaunchKernelGGL(mlp_adam_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, long(n), w,
                     (unsigned short*)w_bf16, grad, m, v, lr, beta1, beta2, eps, c1, c2, weight_decay);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

int fne_mlp_to_bf16(int64_t n, const float* w, uint16_t* w_bf16, fne_stream_t stream) {
  if (n < 0 || !w || !w_bf16) return FNE_EINVAL;
  if (n == 0) return FNE_OK;
  hipLaunchKernelGGL(mlp_to_bf16_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, long(n), w,
                     (unsigned short*)w_bf16);
  FNE_LAUNCH_CHECK();
  return FNE_OK;
}

}  // extern "C"
