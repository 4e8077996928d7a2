// mlp.hip -- the per-vertex MLP surrogate: hand-written BF16 MFMA kernels
// (gfx950 v_mfma_f32_32x32x16_bf16) for training and inference, FP32
// accumulation, FP32 master weights and Adam.
//
// Network: x (n_in) -> [Linear(width) + GELU] x depth -> Linear(n_out).
// Weights are stored "out x in" (row n holds the weights of output n) in
// BF16 for the forward/backward kernels and in FP32 for the optimizer.
// The hidden width x width layers run on MFMA through one generic kernel
//   C[m][n] = sum_k A(m,k) B(k,n),  A(m,k) = A[m*sam + k*sak],
//                                   B(k,n) = B[k*sbk + n*sbn],
// which covers the forward product h W^T, the backward dh = dz W and the
// weight gradient dW = dz^T h (split over K = batch rows, partials reduced
// in a fixed order). Tiles of A and B are staged through LDS with k
// contiguous, so one 16-byte LDS read feeds each MFMA operand.
// The n_in -> width and width -> n_out layers (K = 8 or N = 2) are FP32
// dot products on the vector units. GELU is the tanh form
//   gelu(z) = z/2 (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))).
// Widths 64, 128 and 256 (n_in <= 32) take the fused kernels further down
// instead: one kernel for the whole network, one for all weight gradients.

#include <cmath>
#include <cstdint>
#include <limits>
#include <vector>

#include "kernels.hpp"
#include "mlp.hpp"

namespace nosh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 64, kBN = 128, kBK = 32, kPad = 8;
constexpr int kLds = kBK + kPad;  // bf16 per LDS row

// r = 1 / (exp(2u) + 1), u = sqrt(2/pi) (z + 0.044715 z^3), with the hardware
// exponential and reciprocal (relative error ~1e-6, far below the BF16 rounding
// the activations take next; exp(2u) = inf gives 0, 0 gives 1): tanh u = 1 - 2 r.
__device__ __forceinline__ float gelu_r(float z) {
  const float c = 0.7978845608028654f;  // sqrt(2/pi)
  return __builtin_amdgcn_rcpf(__expf(2.0f * c * (z + 0.044715f * z * z * z)) + 1.0f);
}

// z/2 (1 + tanh u), the halvings exact: the bits are those of
// 0.5f * z * (1.0f + (1.0f - 2.0f * r)) at one instruction less. Its nine
// ordinary and two quarter-rate instructions, not the matrix cores, set the
// pace of the fused network. (z (1 - r) would be one less yet, but does not
// round tanh u as the derivative does; those last bits flip BF16 roundings of
// the activations, 1e-4 of the outputs at depth 4.)
__device__ __forceinline__ float gelu(float z) { return z * (0.5f + (0.5f - gelu_r(z))); }

__device__ __forceinline__ float dgelu(float z) {
  const float c = 0.7978845608028654f;
  const float t = 1.0f - 2.0f * gelu_r(z);
  return 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * c * (1.0f + 3.0f * 0.044715f * z * z);
}

struct GemmArgs {
  const __bf16* A;
  int64_t sam, sak;
  const __bf16* B;
  int64_t sbk, sbn;
  int64_t M, N, K;     // K: per split
  int64_t kchunk;      // K range per split (grid.z)
  int epi;             // 0: z = acc + bias, h = gelu(z); 1: dz = acc * gelu'(zin); 2: store acc
  const float* bias;   // [N]
  const float* zin;    // [M][N] pre-activations (epi 1)
  float* outf;         // [M][N] fp32 (z for epi 0, partials for epi 2 at + z*M*N)
  __bf16* outb;        // [M][N] bf16 (h for epi 0, dz for epi 1)
};

// Loads a kBM x kBK tile of A (rows m0.., k0..) into As[m][k].
__device__ __forceinline__ void load_a(const GemmArgs& g, int64_t m0, int64_t k0, int64_t kend,
                                       __bf16 (*As)[kLds]) {
  const int t = threadIdx.x;
  if (g.sak == 1) {
    const int row = t >> 2, kq = (t & 3) * 8;
    const int64_t m = m0 + row, k = k0 + kq;
    bf16x8 v;
    if (m < g.M && k + 8 <= kend) {
      v = *reinterpret_cast<const bf16x8*>(g.A + m * g.sam + k);
    } else {
      for (int q = 0; q < 8; ++q)
        v[q] = (m < g.M && k + q < kend) ? g.A[m * g.sam + k + q] : __bf16(0.0f);
    }
    *reinterpret_cast<bf16x8*>(&As[row][kq]) = v;
  } else {
    // m contiguous: 8 consecutive m for one k.
    const int kk = t >> 3, mq = (t & 7) * 8;
    const int64_t k = k0 + kk;
    for (int q = 0; q < 8; ++q) {
      const int64_t m = m0 + mq + q;
      As[mq + q][kk] = (m < g.M && k < kend) ? g.A[m * g.sam + k * g.sak] : __bf16(0.0f);
    }
  }
}

// Loads a kBK x kBN tile of B (k0.., n0..) into Bs[n][k].
__device__ __forceinline__ void load_b(const GemmArgs& g, int64_t k0, int64_t n0, int64_t kend,
                                       __bf16 (*Bs)[kLds]) {
  const int t = threadIdx.x;
  if (g.sbk == 1) {
    const int n = t >> 1, kq = (t & 1) * 16;
    const int64_t nn = n0 + n;
    for (int h = 0; h < 2; ++h) {
      const int64_t k = k0 + kq + 8 * h;
      bf16x8 v;
      if (nn < g.N && k + 8 <= kend) {
        v = *reinterpret_cast<const bf16x8*>(g.B + nn * g.sbn + k);
      } else {
        for (int q = 0; q < 8; ++q)
          v[q] = (nn < g.N && k + q < kend) ? g.B[nn * g.sbn + k + q] : __bf16(0.0f);
      }
      *reinterpret_cast<bf16x8*>(&Bs[n][kq + 8 * h]) = v;
    }
  } else {
    const int kk = t >> 3, nq = (t & 7) * 16;
    const int64_t k = k0 + kk;
    for (int q = 0; q < 16; ++q) {
      const int64_t nn = n0 + nq + q;
      Bs[nq + q][kk] = (nn < g.N && k < kend) ? g.B[k * g.sbk + nn * g.sbn] : __bf16(0.0f);
    }
  }
}

// One block (4 waves, 2 x 2) computes a kBM x kBN tile; each wave 32 x 64 as
// two 32x32 MFMA accumulators. grid: (ceil(M/kBM), ceil(N/kBN), splits).
__global__ __launch_bounds__(256) void k_gemm_bf16(GemmArgs g) {
  __shared__ __bf16 As[kBM][kLds];
  __shared__ __bf16 Bs[kBN][kLds];
  const int64_t m0 = int64_t(blockIdx.x) * kBM, n0 = int64_t(blockIdx.y) * kBN;
  const int64_t kbeg = int64_t(blockIdx.z) * g.kchunk;
  const int64_t kend = min(g.K, kbeg + g.kchunk);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2];
  for (int t = 0; t < 2; ++t)
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
  for (int64_t k0 = kbeg; k0 < kend; k0 += kBK) {
    load_a(g, m0, k0, kend, As);
    load_b(g, k0, n0, kend, Bs);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      const int kk = ks * 16 + 8 * (lane >> 5);
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[wm * 32 + (lane & 31)][kk]);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16x8 b =
            *reinterpret_cast<const bf16x8*>(&Bs[wn * 64 + t * 32 + (lane & 31)][kk]);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // D[i][j], j = lane % 32, i = 8 (r/4) + 4 (lane/32) + r%4.
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t n = n0 + wn * 64 + t * 32 + (lane & 31);
    if (n >= g.N) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t m = m0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (m >= g.M) continue;
      const float v = acc[t][r];
      const int64_t o = m * g.N + n;
      if (g.epi == 0) {
        const float z = v + g.bias[n];
        if (g.outf) g.outf[o] = z;
        g.outb[o] = __bf16(gelu(z));
      } else if (g.epi == 1) {
        const float dz = v * dgelu(g.zin[o]);
        g.outb[o] = __bf16(dz);
        if (g.outf) g.outf[o] = dz;
      } else {
        g.outf[int64_t(blockIdx.z) * g.M * g.N + o] = v;
      }
    }
  }
}

// out[i] = sum_s part[s * len + i] (fixed order).
__global__ void k_sum_splits(const float* __restrict__ part, int splits, int64_t len,
                             float* __restrict__ out) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= len) return;
  float s = 0.0f;
  for (int z = 0; z < splits; ++z) s += part[int64_t(z) * len + i];
  out[i] = s;
}

// First layer: z[m][n] = sum_c x[m][c] w[n][c] + b[n]; h = gelu(z).
__global__ void k_layer_in(const float* __restrict__ X, int64_t M, int nin,
                           const __bf16* __restrict__ W, const float* __restrict__ b, int N,
                           float* __restrict__ z, __bf16* __restrict__ h) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  const int64_t m = i / N;
  const int n = int(i - m * N);
  float s = b[n];
  for (int c = 0; c < nin; ++c) s += X[m * nin + c] * float(W[n * nin + c]);
  if (z) z[i] = s;
  h[i] = __bf16(gelu(s));
}

// Last layer: y[m][o] = sum_k h[m][k] w[o][k] + b[o].
__global__ void k_layer_out(const __bf16* __restrict__ H, int64_t M, int K,
                            const __bf16* __restrict__ W, const float* __restrict__ b, int nout,
                            float* __restrict__ Y) {
  const int64_t m = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (m >= M) return;
  for (int o = 0; o < nout; ++o) {
    float s = b[o];
    for (int k = 0; k < K; ++k) s += float(H[m * K + k]) * float(W[o * K + k]);
    Y[m * nout + o] = s;
  }
}

// Loss (mean squared error over M x nout) partials and dy = 2 (y - t) / (M nout).
__global__ void k_loss(const float* __restrict__ Y, const float* __restrict__ T, int64_t len,
                       float scale, float* __restrict__ dY, double* __restrict__ partials) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double v[1] = {0.0};
  if (i < len) {
    const float d = Y[i] - T[i];
    dY[i] = 2.0f * d * scale;
    v[0] = double(d) * double(d);
  }
  block_partials<1>(v, partials);
}

__global__ void k_finalize1(const double* __restrict__ partials, int nb, double scale,
                            double* __restrict__ out) {
  double v[1];
  finalize_sum<1>(v, partials, nb);
  if (threadIdx.x == 0) *out = v[0] * scale;
}

// dz4[m][k] = (sum_o dy[m][o] w[o][k]) gelu'(z4[m][k]).
__global__ void k_back_out(const float* __restrict__ dY, int64_t M, int nout,
                           const __bf16* __restrict__ W, int K, const float* __restrict__ z,
                           __bf16* __restrict__ dz) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= M * K) return;
  const int64_t m = i / K;
  const int k = int(i - m * K);
  float s = 0.0f;
  for (int o = 0; o < nout; ++o) s += dY[m * nout + o] * float(W[o * K + k]);
  dz[i] = __bf16(s * dgelu(z[i]));
}

// Column sums over rows of a [M][N] matrix in row chunks: part[c][n] = sum over chunk c.
template <class T>
__global__ void k_colsum_chunks(const T* __restrict__ A, int64_t M, int N, int64_t chunk,
                                float* __restrict__ part) {
  const int n = blockIdx.y * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int64_t beg = int64_t(blockIdx.x) * chunk, end = min(M, beg + chunk);
  float s = 0.0f;
  for (int64_t m = beg; m < end; ++m) s += float(A[m * N + n]);
  part[int64_t(blockIdx.x) * N + n] = s;
}

// Small weight gradients: part[c][o][k] = sum over chunk c of dy[m][o] x[m][k] with
// x = FP32 (first layer inputs) or BF16 (last hidden layer).
template <class T>
__global__ void k_small_wgrad(const float* __restrict__ D, int no, const T* __restrict__ X,
                              int nk, int64_t M, int64_t chunk, float* __restrict__ part) {
  const int idx = blockIdx.y * blockDim.x + threadIdx.x;
  if (idx >= no * nk) return;
  const int o = idx / nk, k = idx - o * nk;
  const int64_t beg = int64_t(blockIdx.x) * chunk, end = min(M, beg + chunk);
  float s = 0.0f;
  for (int64_t m = beg; m < end; ++m) s += D[m * no + o] * float(X[m * nk + k]);
  part[int64_t(blockIdx.x) * no * nk + idx] = s;
}

__global__ void k_bf16_to_f32(const __bf16* __restrict__ a, int64_t n, float* __restrict__ b) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) b[i] = float(a[i]);
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ gr, float* __restrict__ m,
                       float* __restrict__ v, __bf16* __restrict__ wb, int64_t nwb, int64_t n,
                       float lr, float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = gr[i];
  const float mi = b1 * m[i] + (1.0f - b1) * g;
  const float vi = b2 * v[i] + (1.0f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (i < nwb) wb[i] = __bf16(wi);  // the weights; biases stay FP32
}

__global__ void k_f32_to_bf16(const float* __restrict__ a, int64_t n, __bf16* __restrict__ b) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) b[i] = __bf16(a[i]);
}

// ------------------------------------------------------- fused network
// Widths 64, 128 and 256 with n_in <= 32: the whole network for R = 128, 64 or
// 32 rows in one workgroup of 4 waves, the activations (BF16) in LDS between layers,
// all layers but the last on MFMA with FP32 accumulation; in training the same
// kernel goes on to the loss and back through the layers.
//
// Weights come as operand fragments: the 64 lanes' 8-element operands of one
// MFMA in lane order, 1 KB contiguous (make_fragments lays them out once
// per weight update). A wave owns 32 NT output columns for all rows, so no two
// waves of a workgroup read the same weight and none goes through LDS; the
// next four k-steps' fragments are loaded while the current four multiply,
// and the next layer's first ones before the GELU epilogue. The weights
// are the A operand: a lane then holds four consecutive outputs of one row
// and stores them as 8 bytes. LDS (68 KB at width 256) and registers (196)
// let two workgroups share a CU, so one's GELUs run beside the other's
// MFMAs. Before, every wave computed 32 rows x all columns with the weights
// staged through LDS (135 KB, one workgroup a CU): 1.5 LDS reads an MFMA
// where 1 read of 8 cycles in 32 is the limit of four waves.
// Measured (width 256, depth 4, n_in 7): inference of 912,673 rows 2310 ->
// 568 us (640 TFLOP/s; its 2.4e8 vector instructions of a wave are 0.5 ms of
// issue, the GELUs 0.4 of them), four Adam steps on 16,384 rows 5.95 -> 0.66 ms
// (1.06 with 128 rows a workgroup).
//
// Every value is, bit for bit, that of the layer-by-layer path: layer 0 runs on
// the FP32 matrix instruction (32x32x2, whose sums round like the chain of
// fmaf over the inputs, from the bias on), the hidden layers take the same
// k-steps, and the last layer is an FP32 chain over k again, as such or (beyond
// kChainOut outputs) on the 16x16x4 matrix instruction.
// In the weight gradients x and dy are split into three BF16 parts of 8 bits
// each (x = x1 + x2 + x3 exactly): exact products with the BF16 dz and h.
constexpr int kFusedMaxIn = 32;
constexpr int kMaxLayers = 18;
// Most outputs that the last layer takes as chains on the vector units: a wave
// of them costs 512 instructions, a wave of matrix tiles 64 dependent ones of 32
// cycles whatever the outputs. 300,000 rows of width 256 and depth 4, chains |
// tiles: 4 outputs 221 | 224 us, 8 outputs 244 | 228, 16 outputs 294 | 239; 912,673
// rows with 2 outputs 568 | 606.
constexpr int kChainOut = 4;
constexpr int kFrag = 512;  // bf16 per operand fragment

struct FusedArgs {
  const float* X;
  int64_t M;
  int nin, kx, kp, depth, nout;  // kx: nin rounded up to 2; kp: 3 nin + 1 up to 32
  const float* w0;           // layer 0's FP32 fragments
  const bf16x8* wf;          // forward fragments of the hidden layers
  const bf16x8* wb;          // transposed ones (training)
  const float* wlast;        // last layer, [nout][width]
  const float* wl;           // the same as FP32 fragments
  const float* bias;
  int64_t boff[kMaxLayers];
  float* Y;  // inference
  // Training.
  const float* T;
  float scale;     // 1 / (M nout)
  float4* z;       // pre-activations, in each thread's own order
  bf16x8* hT;      // [layer][16-row chunk][32-column tile] fragments of h
  bf16x8* dzT;     // same of dz
  bf16x8* xT;      // [chunk][tile of kp columns]: x1 | x2 | x3 | 1
  bf16x8* dyT;     // [chunk][tile of 3 nout columns]: dy1 | dy2 | dy3
  double* loss;    // one partial sum per workgroup
  int dy_lds;      // LDS offset of the rows' dy
};

// Fragments per layer (layer 0: 64 floats each, 32 outputs of 2 inputs).
__host__ __device__ inline int64_t frags_first(int width, int kx) {
  return int64_t(width / 32) * (kx / 2);
}
__host__ __device__ inline int64_t frags_hidden(int width) {
  return int64_t(width / 32) * (width / 16);
}

// The three BF16 parts of an FP32 value, by truncation (exact remainders;
// part 0 carries infinities and NaN alone).
__device__ __forceinline__ float top_part(float x) {
  return __uint_as_float(__float_as_uint(x) & 0xffff0000u);
}
__device__ __forceinline__ __bf16 split_part(float x, int part) {
  if ((__float_as_uint(x) & 0x7f800000u) == 0x7f800000u) return part == 0 ? __bf16(x) : __bf16(0.0f);
  const float x1 = top_part(x), r1 = x - x1, x2 = top_part(r1);
  return __bf16(part == 0 ? x1 : part == 1 ? x2 : r1 - x2);
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  union {
    __bf16 h[2];
    uint32_t u;
  } v;
  v.h[0] = __bf16(a);
  v.h[1] = __bf16(b);
  return v.u;
}

template <int W, int R>
struct Tiling {
  static constexpr int NT = W >= 256 ? 2 : 1;   // 32-column tiles per wave
  static constexpr int WN = W / (32 * NT);      // waves along the columns
  static constexpr int MT = R * WN / 128;       // 32-row tiles per wave
  static constexpr int LD = W + 8;              // padded LDS row (bf16): no bank conflicts
  static constexpr int KC = W / 16;             // k-steps of a hidden layer
  static constexpr int Q = MT * NT * 4;         // groups of 4 outputs per thread
  static_assert(MT >= 1, "a wave needs a row tile");
};

// Workgroups a CU holds by LDS: 2 at 128 rows of width 256, 4 below.
template <int W, int R, bool TRAIN>
__global__ __launch_bounds__(256, W * R >= 256 * 128 ? 2 : TRAIN && W * R >= 128 * 128 ? 3 : 4) void
k_mlp_fused(FusedArgs g) {
  using C = Tiling<W, R>;
  constexpr int kRows = R;
  constexpr int NT = C::NT, MT = C::MT, LD = C::LD, KC = C::KC, G = 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __bf16* act = reinterpret_cast<__bf16*>(lds);  // [kRows][LD]; first the split inputs
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int n0 = (wave % C::WN) * 32 * NT, m0 = (wave / C::WN) * 32 * MT;
  const int64_t blk = blockIdx.x, r0 = blk * kRows;
  const int rows = int(min<int64_t>(kRows, g.M - r0));
  const int64_t nchunk = int64_t(gridDim.x) * (kRows / 16);

  // Column-major fragments of an LDS matrix for the weight gradients.
  auto transpose_out = [&](const __bf16* src, int ld, int tiles, bf16x8* dst) {
    for (int f = wave; f < tiles * (kRows / 16); f += 4) {
      const int mc = f / tiles, t = f - mc * tiles;
      const __bf16* q = src + (mc * 16 + 8 * half) * ld + t * 32 + col;
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = q[j * ld];
      dst[((blk * (kRows / 16) + mc) * tiles + t) * 64 + lane] = v;
    }
  };

  f32x16 acc[MT][NT];
  auto clear = [&] {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][t][r] = 0.0f;
  };
  bf16x8 pre[G][NT];  // the first fragments of the next hidden product
  auto prefetch = [&](const bf16x8* w) {
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int t = 0; t < NT; ++t) pre[q][t] = w[((n0 / 32 + t) * KC + q) * 64 + lane];
  };
  // acc = fragments w (rows n0 ..) times the activations, from pre on.
  auto product = [&](const bf16x8* w) {
    clear();
    bf16x8 cur[G][NT];
#pragma unroll
    for (int k0 = 0; k0 < KC; k0 += G) {
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          cur[q][t] = pre[q][t];
          if (k0 + G < KC) pre[q][t] = w[((n0 / 32 + t) * KC + k0 + G + q) * 64 + lane];
        }
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const bf16x8 b = *reinterpret_cast<const bf16x8*>(
              act + (m0 + m * 32 + col) * LD + (k0 + q) * 16 + 8 * half);
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[m][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[q][t], b, acc[m][t], 0, 0, 0);
        }
    }
  };
  // Visits this thread's groups of 4 outputs: (group, row, column, values).
  auto each = [&](auto f) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          f((t * 4 + q) * MT + m, m0 + m * 32 + col, n0 + t * 32 + 8 * q + 4 * half,
            make_float4(acc[m][t][4 * q], acc[m][t][4 * q + 1], acc[m][t][4 * q + 2],
                        acc[m][t][4 * q + 3]));
  };
  auto put = [&](int r, int n, float a, float b, float c, float d) {
    *reinterpret_cast<uint2*>(act + r * LD + n) = make_uint2(pack2(a, b), pack2(c, d));
  };
  auto zslot = [&](int l, int i) { return ((blk * g.depth + l) * C::Q + i) * 256 + tid; };
  // z = acc + bias (layer 0 starts from it), h = gelu(z) into the activations.
  auto activate = [&](int l) {
    const float* bl = g.bias + g.boff[l];
    __syncthreads();  // every wave has read the previous activations
    each([&](int i, int r, int n, float4 v) {
      if (l > 0) {
        const float4 b = *reinterpret_cast<const float4*>(bl + n);
        v = make_float4(v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w);
      }
      if constexpr (TRAIN) g.z[zslot(l, i)] = v;
      put(r, n, gelu(v.x), gelu(v.y), gelu(v.z), gelu(v.w));
    });
    __syncthreads();
  };

  // Layer 0 (its inputs where the activations will be; an odd row pitch).
  float* xs = reinterpret_cast<float*>(lds);
  const int lx = g.kx + 1;
  for (int i = tid; i < kRows * g.kx; i += 256) {
    const int r = i / g.kx, c = i - r * g.kx;
    xs[r * lx + c] = r < rows && c < g.nin ? g.X[(r0 + r) * g.nin + c] : 0.0f;
  }
  if (g.depth > 1) prefetch(g.wf);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 b =
          *reinterpret_cast<const float4*>(g.bias + g.boff[0] + n0 + t * 32 + 8 * q + 4 * half);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        acc[m][t][4 * q] = b.x, acc[m][t][4 * q + 1] = b.y;
        acc[m][t][4 * q + 2] = b.z, acc[m][t][4 * q + 3] = b.w;
      }
    }
  for (int kc = 0; kc < g.kx / 2; ++kc) {
    float a[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) a[t] = g.w0[((n0 / 32 + t) * (g.kx / 2) + kc) * 64 + lane];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float b = xs[(m0 + m * 32 + col) * lx + 2 * kc + half];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[m][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b, acc[m][t], 0, 0, 0);
    }
  }
  if constexpr (TRAIN) {
    const int tiles = g.kp / 32;
    for (int f = wave; f < tiles * (kRows / 16); f += 4) {
      const int mc = f / tiles, k = (f - mc * tiles) * 32 + col;
      const int part = k / g.nin, c = k - part * g.nin;
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = part < 3 ? split_part(xs[(mc * 16 + 8 * half + j) * lx + c], part)
                        : __bf16(k == 3 * g.nin ? 1.0f : 0.0f);
      g.xT[((blk * (kRows / 16) + mc) * tiles + (f - mc * tiles)) * 64 + lane] = v;
    }
  }
  activate(0);
  const int64_t lstride = nchunk * (W / 32) * 64;  // one layer of hT / dzT
  for (int l = 1; l < g.depth; ++l) {
    if constexpr (TRAIN) transpose_out(act, LD, W / 32, g.hT + (l - 1) * lstride);
    product(g.wf + (l - 1) * frags_hidden(W) * 64);
    if (l + 1 < g.depth) prefetch(g.wf + l * frags_hidden(W) * 64);
    activate(l);
  }
  // Last layer: f(row, output, y) once for each. Up to kChainOut outputs go a
  // row and output per lane, weights in scalar registers, more of them through
  // the matrix cores, 16 rows a tile.
  constexpr int kTiles = (kRows + 63) / 64;  // of a wave, or groups of 64 rows
  auto last_layer = [&](auto f) {
    if (g.nout <= kChainOut) {
      for (int u = wave; u < kTiles * g.nout; u += 4) {
        const int o = uniform(u / kTiles), r = (u % kTiles) * 64 + lane;
        if (r >= kRows) continue;
#if __HIP_DEVICE_COMPILE__
        // Never written by this kernel, and the same for the whole wave.
        const auto w = (const __attribute__((address_space(4))) float*)(g.wlast + int64_t(o) * W);
#else
        const float* w = g.wlast + int64_t(o) * W;
#endif
        float s = g.bias[g.boff[g.depth] + o];
#pragma unroll 4
        for (int k = 0; k < W; k += 8) {
          const bf16x8 h = *reinterpret_cast<const bf16x8*>(act + r * LD + k);
#pragma unroll
          for (int e = 0; e < 8; ++e) s += float(h[e]) * w[k + e];
        }
        f(r, o, s);
      }
      return;
    }
    if (wave * 16 >= kRows) return;
    const int q = lane >> 4, r = wave * 16 + (lane & 15);
    f32x4 out[kTiles];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float b = 4 * q + e < g.nout ? g.bias[g.boff[g.depth] + 4 * q + e] : 0.0f;
#pragma unroll
      for (int t = 0; t < kTiles; ++t) out[t][e] = b;
    }
#pragma unroll 8
    for (int k = 0; k < W; k += 4) {
      const float a = g.wl[k * 16 + lane];
#pragma unroll
      for (int t = 0; t < kTiles; ++t)
        out[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, float(act[(r + 64 * t) * LD + k + q]),
                                                      out[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * q + e < g.nout) f(r + 64 * t, 4 * q + e, out[t][e]);
  };
  if constexpr (!TRAIN) {
    last_layer([&](int r, int o, float y) {
      if (r < rows) g.Y[(r0 + r) * g.nout + o] = y;
    });
    return;
  } else {
    float* dys = reinterpret_cast<float*>(lds + g.dy_lds);
    double sq[1] = {0.0};
    last_layer([&](int r, int o, float y) {
      const float d = r < rows ? y - g.T[(r0 + r) * g.nout + o] : 0.0f;
      dys[r * g.nout + o] = 2.0f * d * g.scale;
      sq[0] += double(d) * double(d);
    });
    transpose_out(act, LD, W / 32, g.hT + (g.depth - 1) * lstride);
    const bf16x8* wback = g.wb + (g.depth - 2) * frags_hidden(W) * 64;
    if (g.depth > 1) prefetch(wback);
    __shared__ double wsum[16];
    block_sum<1>(sq, wsum);  // its barriers also publish dys and end the reads of h
    if (tid == 0) g.loss[blk] = sq[0];
    {
      const int tiles = (3 * g.nout + 31) / 32;
      for (int f = wave; f < tiles * (kRows / 16); f += 4) {
        const int mc = f / tiles, i = (f - mc * tiles) * 32 + col;
        const int part = i / g.nout, o = i - part * g.nout;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[j] = part < 3 ? split_part(dys[(mc * 16 + 8 * half + j) * g.nout + o], part)
                          : __bf16(0.0f);
        g.dyT[((blk * (kRows / 16) + mc) * tiles + (f - mc * tiles)) * 64 + lane] = v;
      }
    }
    // dz of the last hidden layer: (dy W_out) gelu'(z).
    each([&](int i, int r, int n, float4) {
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int o = 0; o < g.nout; ++o) {
        const float d = dys[r * g.nout + o];
        const float4 w = *reinterpret_cast<const float4*>(g.wlast + int64_t(o) * W + n);
        s.x += d * w.x;
        s.y += d * w.y;
        s.z += d * w.z;
        s.w += d * w.w;
      }
      const float4 z = g.z[zslot(g.depth - 1, i)];
      put(r, n, s.x * dgelu(z.x), s.y * dgelu(z.y), s.z * dgelu(z.z), s.w * dgelu(z.w));
    });
    __syncthreads();
    for (int l = g.depth - 1; l >= 1; --l) {
      transpose_out(act, LD, W / 32, g.dzT + l * lstride);
      product(g.wb + (l - 1) * frags_hidden(W) * 64);
      if (l > 1) prefetch(g.wb + (l - 2) * frags_hidden(W) * 64);
      __syncthreads();
      each([&](int i, int r, int n, float4 v) {
        const float4 z = g.z[zslot(l - 1, i)];
        put(r, n, v.x * dgelu(z.x), v.y * dgelu(z.y), v.z * dgelu(z.z), v.w * dgelu(z.w));
      });
      __syncthreads();
    }
    transpose_out(act, LD, W / 32, g.dzT);
  }
}

// Operand fragments of the BF16 weights (see k_mlp_fused): element j of lane
// l in fragment (t, c) of a matrix A is A[32 t + l % 32][16 c + 8 (l / 32) + j];
// layer 0's are FP32, A[32 t + l % 32][2 c + l / 32], zero past the last input.
// The last layer is stored as FP32 rows and as FP32 fragments of 16 outputs and
// 4 inputs: A[l % 16][4 c + l / 16].
struct FragArgs {
  const __bf16* w;
  int nin, kx, width, depth, nout;
  int64_t woff[kMaxLayers];
  float *w0, *wlast, *wl;
  bf16x8 *wf, *wb;
};
__global__ void k_make_fragments(FragArgs g) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int lane = int(i & 63), row = lane & 31, k8 = 8 * (lane >> 5);
  const int W = g.width;
  const int64_t nh = frags_hidden(W), n0 = frags_first(W, g.kx), f = i >> 6;
  if (f < n0) {
    const int t = int(f / (g.kx / 2)), k = 2 * int(f % (g.kx / 2)) + (lane >> 5);
    g.w0[i] = k < g.nin ? float(g.w[g.woff[0] + int64_t(32 * t + row) * g.nin + k]) : 0.0f;
  }
  if (f < (g.depth - 1) * nh) {
    const int l = int(f / nh) + 1;
    const int q = int(f - (l - 1) * nh), t = q / (W / 16), c = q - t * (W / 16);
    const __bf16* w = g.w + g.woff[l];
    g.wf[i] = *reinterpret_cast<const bf16x8*>(w + int64_t(32 * t + row) * W + 16 * c + k8);
    bf16x8 v;
    for (int j = 0; j < 8; ++j) v[j] = w[int64_t(16 * c + k8 + j) * W + 32 * t + row];
    g.wb[i] = v;
  }
  if (i < int64_t(g.nout) * W) g.wlast[i] = float(g.w[g.woff[g.depth] + i]);
  if (i < 16 * int64_t(W)) {
    const int o = lane & 15, k = int(f) * 4 + (lane >> 4);
    g.wl[i] = o < g.nout ? float(g.w[g.woff[g.depth] + int64_t(o) * W + k]) : 0.0f;
  }
}

// All weight and bias gradients of a minibatch: products over the rows of the
// fragments k_mlp_fused wrote (each 1 KB load feeds an MFMA operand, nothing
// goes through LDS). One wave per output tile and row split:
//   64 x 64 tiles of dz_l^T h_{l-1} (hidden layers), then 32 x 32 tiles of
//   dz_l^T [x | 1] (layer 0's weights; the column of ones gives every
//   layer's bias gradient) and of dy^T [h | 1] (last layer).
// Split sums go to hpart / spart and are added in order by k_grad_sum. Splits
// of 512 rows: 16 k rows at width 256 and depth 4 give 2848 waves.
struct WgradArgs {
  int width, depth, kp, nin, nout, ptiles;  // ptiles: 32-column tiles of dyT
  int64_t nchunk, per_split;                // 16-row chunks, chunks per split
  const bf16x8 *hT, *dzT, *xT, *dyT;
  float* hpart;  // [split][l - 1][width][width]
  float* spart;  // [split][small tile][32][32]
};
__host__ __device__ inline int wgrad_big(int width, int depth) {
  return (depth - 1) * (width / 64) * (width / 64);
}
// Small tiles: (l = 0: width/32 x kp/32), (l >= 1: width/32), (dy: ptiles x
// width/32), (dy bias: ptiles).
__host__ __device__ inline int wgrad_small(int width, int depth, int kp, int ptiles) {
  return (width / 32) * (kp / 32) + (depth - 1) * (width / 32) + ptiles * (width / 32) + ptiles;
}

template <int TA, int TB>
__device__ __forceinline__ void wgrad_tile(const bf16x8* __restrict__ A, int64_t sa,
                                           const bf16x8* __restrict__ B, int64_t sb, int64_t c0,
                                           int64_t c1, int lane, float* __restrict__ out, int ld) {
  f32x16 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;
  for (int64_t c = c0; c < c1; ++c) {
    bf16x8 av[TA], bv[TB];
#pragma unroll
    for (int a = 0; a < TA; ++a) av[a] = A[(c * sa + a) * 64 + lane];
#pragma unroll
    for (int b = 0; b < TB; ++b) bv[b] = B[(c * sb + b) * 64 + lane];
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * a + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        out[int64_t(i) * ld + 32 * b + (lane & 31)] = acc[a][b][r];
      }
}

__global__ __launch_bounds__(256) void k_wgrad(WgradArgs g) {
  const int lane = threadIdx.x & 63;
  const int W = g.width, wt = W / 32;
  const int big = wgrad_big(W, g.depth), small = wgrad_small(W, g.depth, g.kp, g.ptiles);
  // One split's workgroups run on one XCD, whose L2 then reads its rows once
  // (spread over all eight, 16 k rows took 32 us; now 20). Loading four
  // chunks ahead measured slower (26 us, 202 registers).
  const int per_split_blocks = (big + small + 3) / 4;
  const int64_t logical = xcd_block(true);
  const int64_t split = logical / per_split_blocks;
  int job = int(logical - split * per_split_blocks) * 4 + (threadIdx.x >> 6);
  if (job >= big + small) return;
  const int64_t c0 = split * g.per_split, c1 = min(g.nchunk, c0 + g.per_split);
  const int64_t ls = g.nchunk * wt * 64;
  if (job < big) {
    const int per = (W / 64) * (W / 64);
    const int l = job / per + 1, q = job - (l - 1) * per, ti = q / (W / 64), tj = q - ti * (W / 64);
    float* out = g.hpart + ((split * (g.depth - 1) + l - 1) * W + 64 * ti) * W + 64 * tj;
    wgrad_tile<2, 2>(g.dzT + l * ls + 2 * ti * 64, wt, g.hT + (l - 1) * ls + 2 * tj * 64, wt, c0,
                     c1, lane, out, W);
    return;
  }
  job -= big;
  float* out = g.spart + (split * small + job) * 1024;
  const int xt = g.kp / 32, ones = 3 * g.nin / 32;
  const bf16x8 *A, *B;
  int64_t sa, sb;
  if (job < wt * xt) {
    A = g.dzT + (job / xt) * 64, sa = wt;
    B = g.xT + (job % xt) * 64, sb = xt;
  } else if ((job -= wt * xt) < (g.depth - 1) * wt) {
    A = g.dzT + (1 + job / wt) * ls + (job % wt) * 64, sa = wt;
    B = g.xT + ones * 64, sb = xt;
  } else if ((job -= (g.depth - 1) * wt) < g.ptiles * wt) {
    A = g.dyT + (job / wt) * 64, sa = g.ptiles;
    B = g.hT + (g.depth - 1) * ls + (job % wt) * 64, sb = wt;
  } else {
    job -= g.ptiles * wt;
    A = g.dyT + job * 64, sa = g.ptiles;
    B = g.xT + ones * 64, sb = xt;
  }
  wgrad_tile<1, 1>(A, sa, B, sb, c0, c1, lane, out, 32);
}

// Gradient of parameter i (layout of the parameter vector): the split sums
// of its tile in split order, the three parts of a split operand together.
struct GradSumArgs {
  WgradArgs w;
  int splits;
  int64_t nweights, nparams;
  int64_t woff[kMaxLayers], boff[kMaxLayers];
  float* grad;
  const double* loss_part;  // nloss partial sums; the last workgroup adds them
  int nloss;
  double loss_scale;
  double* loss;
};
__global__ void k_grad_sum(GradSumArgs g) {
  if (blockIdx.x + 1 == gridDim.x) {
    double v[1];
    finalize_sum<1>(v, g.loss_part, g.nloss);
    if (threadIdx.x == 0) *g.loss = v[0] * g.loss_scale;
    return;
  }
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= g.nparams) return;
  const int W = g.w.width, D = g.w.depth, wt = W / 32, xt = g.w.kp / 32, nin = g.w.nin,
            nout = g.w.nout, pt = g.w.ptiles;
  const int small = wgrad_small(W, D, g.w.kp, pt);
  const int j1 = wt * xt, j2 = j1 + (D - 1) * wt, j3 = j2 + pt * wt;
  const int ones = 3 * nin;
  const bool is_bias = i >= g.nweights;
  const int64_t q = is_bias ? i - g.nweights : i;
  const int64_t* off = is_bias ? g.boff : g.woff;
  int l = 0;
  while (l < D && q >= off[l + 1]) ++l;
  const int64_t e = q - off[l];
  float s = 0.0f;
  if (!is_bias && l > 0 && l < D) {
    const float* p = g.w.hpart + int64_t(l - 1) * W * W + e;
    const int64_t st = int64_t(D - 1) * W * W;
#pragma unroll 16
    for (int z = 0; z < g.splits; ++z) s += p[z * st];
  } else {
    // Up to three entries of the small tiles.
    int64_t at[3];
    int parts = 3;
    if (!is_bias && l == 0) {
      const int n = int(e / nin), c = int(e - int64_t(n) * nin);
      for (int p = 0; p < 3; ++p) {
        const int k = p * nin + c;
        at[p] = int64_t((n / 32) * xt + k / 32) * 1024 + (n % 32) * 32 + k % 32;
      }
    } else if (!is_bias) {
      const int o = int(e / W), k = int(e - int64_t(o) * W);
      for (int p = 0; p < 3; ++p) {
        const int r = p * nout + o;
        at[p] = int64_t(j2 + (r / 32) * wt + k / 32) * 1024 + (r % 32) * 32 + k % 32;
      }
    } else if (l < D) {
      const int n = int(e);
      const int job = l == 0 ? (n / 32) * xt + ones / 32 : j1 + (l - 1) * wt + n / 32;
      at[0] = int64_t(job) * 1024 + (n % 32) * 32 + ones % 32;
      parts = 1;
    } else {
      for (int p = 0; p < 3; ++p) {
        const int r = p * nout + int(e);
        at[p] = int64_t(j3 + r / 32) * 1024 + (r % 32) * 32 + ones % 32;
      }
    }
    if (parts == 1) at[1] = at[2] = at[0];
#pragma unroll 8
    for (int z = 0; z < g.splits; ++z) {
      const float* p = g.w.spart + int64_t(z) * small * 1024;
      const float v1 = p[at[0]], v2 = p[at[1]], v3 = p[at[2]];
      s += parts == 1 ? v1 : v1 + (v2 + v3);
    }
  }
  g.grad[i] = s;
}

unsigned g1(int64_t n, int b = 256) { return grid_for(n, b); }

}  // namespace

// ----------------------------------------------------------------- host
void Mlp::init(int nin_, int width_, int depth_, int nout_, uint64_t seed) {
  nin = nin_;
  width = width_;
  depth = depth_;
  nout = nout_;
  NOSH_CHECK(nin >= 1 && nin <= 64 && nout >= 1 && nout <= 16 && depth >= 1 && depth <= 16,
             kInvalid, "mlp: unsupported shape");
  NOSH_CHECK(width % 64 == 0 && width <= 2048, kInvalid, "mlp: width must be a multiple of 64");
  // Layer l maps dim[l] -> dim[l+1].
  dims.clear();
  dims.push_back(nin);
  for (int l = 0; l < depth; ++l) dims.push_back(width);
  dims.push_back(nout);
  woff.clear();
  boff.clear();
  int64_t nw = 0, nb = 0;
  for (size_t l = 0; l + 1 < dims.size(); ++l) {
    woff.push_back(nw);
    boff.push_back(nb);
    nw += int64_t(dims[l]) * dims[l + 1];
    nb += dims[l + 1];
  }
  nweights = nw;
  nparams = nw + nb;
  // He-style uniform init from a SplitMix64 stream (host), biases zero.
  std::vector<float> p(nparams, 0.0f);
  uint64_t st = seed;
  auto uni = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return double(z >> 11) * (1.0 / 9007199254740992.0);
  };
  for (size_t l = 0; l + 1 < dims.size(); ++l) {
    const double a = std::sqrt(6.0 / dims[l]) * (l + 2 == dims.size() ? 0.1 : 1.0);
    for (int64_t i = 0; i < int64_t(dims[l]) * dims[l + 1]; ++i)
      p[woff[l] + i] = float((2.0 * uni() - 1.0) * a);
  }
  hipStream_t s = default_stream();
  master.alloc(nparams);
  master.upload(p.data(), nparams, s);
  grad.alloc(nparams);
  grad.zero(s);
  m1.alloc(nparams);
  m1.zero(s);
  m2.alloc(nparams);
  m2.zero(s);
  wbf.alloc(nweights);
  sync_bf16(s);
  steps = 0;
  NOSH_HIP(hipStreamSynchronize(s));
}

void Mlp::ensure(int64_t M) {
  if (M <= cap) return;
  cap = M;
  const int L = int(dims.size()) - 1;
  zbuf.resize(L - 1);
  hbuf.resize(L - 1);
  for (int l = 0; l < L - 1; ++l) {
    zbuf[l].alloc(M * dims[l + 1]);
    hbuf[l].alloc(M * dims[l + 1]);
  }
  dzb.alloc(M * width);
  dza.alloc(M * width);
  y.alloc(M * nout);
  dy.alloc(M * nout);
  partials.alloc(g1(M * nout) + 64);
  loss.alloc(1);
}

const float* Mlp::bias(int l) const { return master.p + nweights + boff[l]; }

void Mlp::gemm(const __bf16* A, int64_t sam, int64_t sak, const __bf16* B, int64_t sbk,
               int64_t sbn, int64_t M, int64_t N, int64_t K, int epi, const float* bias_,
               const float* zin, float* outf, __bf16* outb, int splits, hipStream_t s) {
  GemmArgs g;
  g.A = A;
  g.sam = sam;
  g.sak = sak;
  g.B = B;
  g.sbk = sbk;
  g.sbn = sbn;
  g.M = M;
  g.N = N;
  g.K = K;
  const int64_t kc = ((K + splits - 1) / splits + kBK - 1) / kBK * kBK;
  g.kchunk = kc;
  g.epi = epi;
  g.bias = bias_;
  g.zin = zin;
  g.outf = outf;
  g.outb = outb;
  dim3 grid(unsigned((M + kBM - 1) / kBM), unsigned((N + kBN - 1) / kBN),
            unsigned((K + kc - 1) / kc));
  k_gemm_bf16<<<grid, 256, 0, s>>>(g);
}

// ------------------------------------------------ fused path (host side)
bool Mlp::fused() const {
  return (width == 64 || width == 128 || width == 256) && nin <= kFusedMaxIn;
}

namespace {

int even_cols(int nin) { return (nin + 1) / 2 * 2; }
int split_cols(int nin) { return (3 * nin + 1 + 31) / 32 * 32; }

template <int W, int R, bool TRAIN>
void launch_fused(FusedArgs g, hipStream_t s) {
  const size_t top = size_t(R) * Tiling<W, R>::LD * 2;  // the inputs need less
  static_assert(Tiling<W, R>::LD * 2 >= (kFusedMaxIn + 1) * 4, "room for the inputs");
  const size_t lds = top + (TRAIN ? size_t(R) * g.nout * 4 : 0);
  g.dy_lds = int(top);
  // More than the 64 KB a kernel may use by default at 128 rows of width 256.
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(k_mlp_fused<W, R, TRAIN>),
      hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  NOSH_HIP(attr);
  k_mlp_fused<W, R, TRAIN><<<unsigned((g.M + R - 1) / R), 256, lds, s>>>(g);
}

// Rows per workgroup: the largest that still gives every CU of the chip a
// workgroup (128-row ones read each weight half as often as 64-row ones, but
// leave CUs idle below 32 k rows: a training pass over 16,384 rows of width
// 256 took 146 us with 128 of them and 84 us with 256). A wave needs a
// 32-row tile of its own, which sets the least at width 64.
int fused_rows(int width, int64_t M) {
  const int64_t cus = 256;
  if ((M + 127) / 128 >= cus) return 128;
  if (width == 64 || (M + 63) / 64 >= cus) return 64;
  return 32;
}

template <int W, bool TRAIN>
void launch_fused_rows(int rows, const FusedArgs& g, hipStream_t s) {
  if (rows == 128)
    launch_fused<W, 128, TRAIN>(g, s);
  else if (rows == 64)
    launch_fused<W, 64, TRAIN>(g, s);
  else if constexpr (W > 64)
    launch_fused<W, 32, TRAIN>(g, s);
}

template <bool TRAIN>
void launch_fused_width(int width, int rows, const FusedArgs& g, hipStream_t s) {
  if (width == 256)
    launch_fused_rows<256, TRAIN>(rows, g, s);
  else if (width == 128)
    launch_fused_rows<128, TRAIN>(rows, g, s);
  else
    launch_fused_rows<64, TRAIN>(rows, g, s);
}

FusedArgs fused_args(const Mlp& n, const float* X, int64_t M) {
  FusedArgs g{};
  g.X = X;
  g.M = M;
  g.nin = n.nin;
  g.kx = even_cols(n.nin);
  g.kp = split_cols(n.nin);
  g.depth = n.depth;
  g.nout = n.nout;
  g.w0 = n.w32.p;
  g.wlast = n.w32.p + frags_first(n.width, g.kx) * 64;
  g.wl = g.wlast + int64_t(n.nout) * n.width;
  g.wf = reinterpret_cast<const bf16x8*>(n.wfrag.p);
  g.wb = reinterpret_cast<const bf16x8*>(n.wfrag_t.p);
  g.bias = n.master.p + n.nweights;
  for (int l = 0; l <= n.depth; ++l) g.boff[l] = n.boff[l];
  return g;
}

}  // namespace

void Mlp::make_fragments(hipStream_t s) {
  if (!fused()) return;
  const int kx = even_cols(nin);
  const int64_t n0 = frags_first(width, kx), nh = (depth - 1) * frags_hidden(width);
  if (!wfrag.p) {
    w32.alloc(n0 * 64 + int64_t(nout + 16) * width);
    wfrag.alloc(std::max<int64_t>(1, nh) * kFrag);
    wfrag_t.alloc(std::max<int64_t>(1, nh) * kFrag);
  }
  FragArgs g{};
  g.w = wbf.p;
  g.nin = nin;
  g.kx = kx;
  g.width = width;
  g.depth = depth;
  g.nout = nout;
  g.w0 = w32.p;
  g.wlast = w32.p + n0 * 64;
  g.wl = g.wlast + int64_t(nout) * width;
  for (int l = 0; l <= depth; ++l) g.woff[l] = woff[l];
  g.wf = reinterpret_cast<bf16x8*>(wfrag.p);
  g.wb = reinterpret_cast<bf16x8*>(wfrag_t.p);
  const int64_t threads = std::max({n0 * 64, nh * 64, int64_t(16) * width});
  k_make_fragments<<<g1(threads), 256, 0, s>>>(g);
}

void Mlp::ensure_fused(int64_t M) {
  if (M <= fcap) return;
  fcap = M;
  const int64_t mp = (M + 127) / 128 * 128;  // covers every rows-per-workgroup choice below M too
  const int64_t pt = (3 * nout + 31) / 32;
  zs.alloc(mp * width * depth);
  hT.alloc(mp * width * depth);
  dzT.alloc(mp * width * depth);
  xT.alloc(mp * split_cols(nin));
  dyT.alloc(mp * pt * 32);
  partials.alloc(mp / 32 + 64);
  if (!loss.p) loss.alloc(1);
}

void Mlp::gradients_fused(const float* X, const float* T, int64_t M, hipStream_t s) {
  ensure_fused(M);
  const int rows = fused_rows(width, M);
  const unsigned nb = unsigned((M + rows - 1) / rows);
  FusedArgs g = fused_args(*this, X, M);
  g.T = T;
  g.scale = 1.0f / float(M * nout);
  g.z = reinterpret_cast<float4*>(zs.p);
  g.hT = reinterpret_cast<bf16x8*>(hT.p);
  g.dzT = reinterpret_cast<bf16x8*>(dzT.p);
  g.xT = reinterpret_cast<bf16x8*>(xT.p);
  g.dyT = reinterpret_cast<bf16x8*>(dyT.p);
  g.loss = partials.p;
  launch_fused_width<true>(width, rows, g, s);
  GradSumArgs r{};
  WgradArgs& w = r.w;
  w.width = width;
  w.depth = depth;
  w.kp = g.kp;
  w.nin = nin;
  w.nout = nout;
  w.ptiles = (3 * nout + 31) / 32;
  w.nchunk = int64_t(nb) * (rows / 16);
  // 512 rows a split, at most 64 splits.
  w.per_split = std::max<int64_t>(32, (w.nchunk + 63) / 64);
  r.splits = int((w.nchunk + w.per_split - 1) / w.per_split);
  const int big = wgrad_big(width, depth), small = wgrad_small(width, depth, w.kp, w.ptiles);
  const size_t nh = size_t(r.splits) * (depth - 1) * width * width;
  const size_t need = nh + size_t(r.splits) * small * 1024;
  if (red.n < need) red.alloc(need);
  w.hT = g.hT;
  w.dzT = g.dzT;
  w.xT = g.xT;
  w.dyT = g.dyT;
  w.hpart = red.p;
  w.spart = red.p + nh;
  k_wgrad<<<unsigned((big + small + 3) / 4 * r.splits), 256, 0, s>>>(w);
  r.nweights = nweights;
  r.nparams = nparams;
  for (int l = 0; l <= depth; ++l) {
    r.woff[l] = woff[l];
    r.boff[l] = boff[l];
  }
  r.grad = grad.p;
  r.loss_part = partials.p;
  r.nloss = int(nb);
  r.loss_scale = 1.0 / double(M * nout);
  r.loss = loss.p;
  k_grad_sum<<<g1(nparams) + 1, 256, 0, s>>>(r);
}

void Mlp::forward(const float* X, int64_t M, float* Y, hipStream_t s, bool keep_pre) {
  if (fused() && !keep_pre) {
    FusedArgs g = fused_args(*this, X, M);
    g.Y = Y;
    launch_fused_width<false>(width, fused_rows(width, M), g, s);
    return;
  }
  ensure(M);
  const int L = int(dims.size()) - 1;
  k_layer_in<<<g1(M * dims[1]), 256, 0, s>>>(X, M, nin, wbf.p + woff[0], bias(0), dims[1],
                                             keep_pre ? zbuf[0].p : nullptr, hbuf[0].p);
  for (int l = 1; l < L - 1; ++l) {
    // z = h W^T: A = h [M][K], B(k,n) = W[n][k].
    gemm(hbuf[l - 1].p, dims[l], 1, wbf.p + woff[l], 1, dims[l], M, dims[l + 1], dims[l], 0,
         bias(l), nullptr, keep_pre ? zbuf[l].p : nullptr, hbuf[l].p, 1, s);
  }
  k_layer_out<<<g1(M), 256, 0, s>>>(hbuf[L - 2].p, M, dims[L - 1], wbf.p + woff[L - 1],
                                    bias(L - 1), nout, Y ? Y : y.p);
}

void Mlp::infer(const float* X, int64_t M, float* Y, hipStream_t s) {
  if (fused()) {
    forward(X, M, Y, s, false);
    return;
  }
  constexpr int64_t kChunk = 1 << 19;
  for (int64_t r0 = 0; r0 < M; r0 += kChunk)
    forward(X + r0 * nin, std::min(kChunk, M - r0), Y + r0 * nout, s, false);
}

double Mlp::last_loss(hipStream_t s) {
  double lh = 0.0;
  NOSH_HIP(hipMemcpyAsync(&lh, loss.p, sizeof(double), hipMemcpyDeviceToHost, s));
  NOSH_HIP(hipStreamSynchronize(s));
  return lh;
}

double Mlp::gradients(const float* X, const float* T, int64_t M, hipStream_t s, bool read_loss) {
  if (fused()) {
    gradients_fused(X, T, M, s);
    return read_loss ? last_loss(s) : std::numeric_limits<double>::quiet_NaN();
  }
  ensure(M);
  forward(X, M, y.p, s);
  const int L = int(dims.size()) - 1;
  const int64_t len = M * nout;
  const unsigned nbl = g1(len);
  k_loss<<<nbl, 256, 0, s>>>(y.p, T, len, 1.0f / float(len), dy.p, partials.p);
  k_finalize1<<<1, 256, 0, s>>>(partials.p, int(nbl), 1.0 / double(len), loss.p);
  // Row chunks for the deterministic reductions over the batch (column sums
  // and the small first/last-layer weight gradients): 32 rows (at most 4096
  // chunks), so that a batch of 8 k rows gives 256 chunks of parallel work
  // (1024-row chunks took 240 us per reduction at 8 k rows, 1.6 of the 2 ms
  // of an Adam step).
  const int64_t chunk = std::max<int64_t>(32, (M + 4095) / 4096);
  const int64_t nchunk = (M + chunk - 1) / chunk;
  // Split-K of the hidden layers' weight-gradient GEMMs: 1024 rows a split.
  const int64_t nsplit = (M + 1023) / 1024;
  // Scratch for the partial sums: split-K GEMM partials (<= 64 x width^2),
  // per-chunk column sums (nchunk x width) and small weight gradients
  // (nchunk x width x max(n_in, n_out)).
  const int64_t need = std::max<int64_t>(64 * int64_t(width) * width,
                                         nchunk * int64_t(width) * std::max(nin, nout));
  if (red.n < size_t(need)) red.alloc(need);
  auto wg = [&](int l) { return grad.p + woff[l]; };
  auto bg = [&](int l) { return grad.p + nweights + boff[l]; };
  // Last layer: dW = dy^T h, db = sum dy.
  {
    const int K = dims[L - 1];
    dim3 grid(unsigned(nchunk), unsigned(g1(int64_t(nout) * K)));
    k_small_wgrad<__bf16><<<grid, 256, 0, s>>>(dy.p, nout, hbuf[L - 2].p, K, M, chunk, red.p);
    k_sum_splits<<<g1(int64_t(nout) * K), 256, 0, s>>>(red.p, int(nchunk), int64_t(nout) * K,
                                                        wg(L - 1));
    dim3 gb(unsigned(nchunk), 1);
    k_colsum_chunks<float><<<gb, 256, 0, s>>>(dy.p, M, nout, chunk, red.p);
    k_sum_splits<<<1, 256, 0, s>>>(red.p, int(nchunk), nout, bg(L - 1));
    k_back_out<<<g1(M * K), 256, 0, s>>>(dy.p, M, nout, wbf.p + woff[L - 1], K, zbuf[L - 2].p,
                                        dzb.p);
  }
  // Hidden layers l = L-2 .. 1 (MFMA): dW_l = dz^T h_{l-1}, dh_{l-1} = dz W_l.
  __bf16* dz = dzb.p;
  __bf16* dzn = dza.p;
  for (int l = L - 2; l >= 1; --l) {
    const int64_t N = dims[l + 1], K = dims[l];
    const int splits = int(std::min<int64_t>(nsplit, 64));
    // C[n][k] = sum_m dz[m][n] h[m][k]: A(n,m) = dz[m*N + n], B(m,k) = h[m*K + k].
    gemm(dz, 1, N, hbuf[l - 1].p, K, 1, N, K, M, 2, nullptr, nullptr, red.p, nullptr, splits,
         s);
    const int64_t kc = ((M + splits - 1) / splits + kBK - 1) / kBK * kBK;
    const int used = int((M + kc - 1) / kc);
    k_sum_splits<<<g1(N * K), 256, 0, s>>>(red.p, used, N * K, wg(l));
    dim3 gb(unsigned(nchunk), unsigned(g1(N)));
    k_colsum_chunks<__bf16><<<gb, 256, 0, s>>>(dz, M, int(N), chunk, red.p);
    k_sum_splits<<<g1(N), 256, 0, s>>>(red.p, int(nchunk), N, bg(l));
    // dz_{l-1} = (dz W_l) * gelu'(z_{l-1}): A = dz [M][N], B(n,k) = W[n][k].
    gemm(dz, N, 1, wbf.p + woff[l], K, 1, M, K, N, 1, nullptr, zbuf[l - 1].p, nullptr, dzn, 1,
         s);
    std::swap(dz, dzn);
  }
  // First layer: dW = dz^T x, db = sum dz.
  {
    const int K = nin, N = dims[1];
    dim3 grid(unsigned(nchunk), unsigned(g1(int64_t(N) * K)));
    // part[c][n][k] = sum dz[m][n] x[m][k] with dz in BF16: convert to FP32 rows first.
    k_bf16_to_f32<<<g1(M * N), 256, 0, s>>>(dz, M * N, zbuf[0].p);
    k_small_wgrad<float><<<grid, 256, 0, s>>>(zbuf[0].p, N, X, K, M, chunk, red.p);
    k_sum_splits<<<g1(int64_t(N) * K), 256, 0, s>>>(red.p, int(nchunk), int64_t(N) * K, wg(0));
    dim3 gb(unsigned(nchunk), unsigned(g1(N)));
    k_colsum_chunks<float><<<gb, 256, 0, s>>>(zbuf[0].p, M, N, chunk, red.p);
    k_sum_splits<<<g1(N), 256, 0, s>>>(red.p, int(nchunk), N, bg(0));
  }
  return read_loss ? last_loss(s) : std::numeric_limits<double>::quiet_NaN();
}

void Mlp::adam(float lr, hipStream_t s) {
  ++steps;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.0f - std::pow(b1, float(steps)), c2 = 1.0f - std::pow(b2, float(steps));
  k_adam<<<g1(nparams), 256, 0, s>>>(master.p, grad.p, m1.p, m2.p, wbf.p, nweights, nparams, lr,
                                     b1, b2, eps, c1, c2);
  make_fragments(s);
}

void Mlp::sync_bf16(hipStream_t s) {
  k_f32_to_bf16<<<g1(nweights), 256, 0, s>>>(master.p, nweights, wbf.p);
  make_fragments(s);
}

namespace {
__global__ void k_gather_rows(const float* __restrict__ src, const int64_t* __restrict__ idx,
                              int64_t B, int w, float scale, float* __restrict__ dst) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= B * w) return;
  const int64_t r = i / w;
  dst[i] = src[idx[r] * w + (i - r * w)] * scale;
}

__global__ void k_sumsq_f32(const float* __restrict__ x, int64_t n, double* __restrict__ part) {
  double v[1] = {0.0};
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const double t = x[i];
    v[0] += t * t;
  }
  block_partials<1>(v, part);
}
}  // namespace

double rms_f32(const float* x, int64_t n, hipStream_t s) {
  if (n <= 0) return 0.0;
  const int nb = int(std::min<int64_t>(1024, grid_for(n, 256)));
  DBuf<double> part{size_t(nb)};
  k_sumsq_f32<<<nb, 256, 0, s>>>(x, n, part.p);
  std::vector<double> h(static_cast<size_t>(nb));
  part.download(h.data(), h.size(), s);
  NOSH_HIP(hipStreamSynchronize(s));
  double ss = 0.0;
  for (double v : h) ss += v;
  return std::sqrt(ss / double(n));
}

void launch_gather_rows(const float* src, const int64_t* idx, int64_t B, int w, float scale,
                        float* dst, hipStream_t s) {
  k_gather_rows<<<grid_for(B * w, 256), 256, 0, s>>>(src, idx, B, w, scale, dst);
}

}  // namespace nosh
