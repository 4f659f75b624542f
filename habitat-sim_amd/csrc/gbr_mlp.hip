// Chunk-visibility MLP (32 -> 256 -> 256 -> 1, ReLU) on gfx950 MFMA:
// BF16 operands, FP32 accumulation, FP32 master weights with Adam.
//
// A training step is four launches (it was nineteen):
//   k_train_forward  per 32 rows of the minibatch: the rows from the training
//                    set, both layers, the logits, the loss and its gradient
//                    by the logits, dH2 = [H2 > 0] dl w3
//   k_train_grads    dW2 = dH2^T H1, dH1 = (dH2 W2) o [H1 > 0] and the sums over
//                    the batch for w3, b2, b3 and the loss
//   k_train_grads1   dW1 = dH1^T X and the sums for b1
//   k_adam           the weights, and their bf16 copies
// Every product is an "NT" one, C[M][N] = sum_k A[M][K] * Bt[N][K], with the
// eight k of an MFMA fragment's lane contiguous in both operands.  The sums
// are reductions with one writer per output (no atomics), and every sum runs
// in a fixed order, whatever the launch geometry.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "gbr_mlp.h"

namespace gbr {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// float -> bf16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ int rows_of(int M, const uint32_t* M_dev) {
  return M_dev ? min(M, (int)*M_dev) : M;
}

// four bf16 in one 8-byte store
__device__ __forceinline__ void store4(uint16_t* dst, uint16_t a, uint16_t b, uint16_t c, uint16_t d) {
  *reinterpret_cast<uint2*>(dst) =
      make_uint2((uint32_t)a | ((uint32_t)b << 16), (uint32_t)c | ((uint32_t)d << 16));
}

// The batch matrices that a weight gradient contracts over the batch (X, H1,
// dH2, dH1 transposed) are kept in the order of MFMA fragments: for 32
// columns and 16 rows of the batch, lane l's eight values (column l%32, rows
// 8*(l/32) .. +8) one after the other, so that a wave's fragment is 1 KB in a
// row.  (As [column][batch] rows a load gathered 64 pieces of 16 bytes: with 32
// steps ahead k_train_grads took 21.5 us at 4096 rows, and takes 14.1 so; with 16
// ahead 24.9 and 17.2.)
__device__ __forceinline__ size_t frag_at(int column, int row, int batch) {
  return (((size_t)(column >> 5) * (size_t)(batch >> 4) + (size_t)(row >> 4)) * 64 +
          (size_t)((column & 31) + 32 * ((row >> 3) & 1))) * 8 + (size_t)(row & 7);
}

// --------------------------------------------------------------------------
// One 32x32 tile of an NT product by one wave (v_mfma_f32_32x32x16_bf16):
// lane l supplies A[m0 + l%32][k + 8*(l/32) .. +8] and Bt[n0 + l%32][same k],
// at ap and bp for k = 0 and a_step, b_step elements further per 16 k;
// accumulator v holds C[m0 + 8*(v/4) + 4*(l/32) + v%4][n0 + l%32].  The K
// steps run in order, k = 0, 16, ...
//
// A weight gradient is a chain of K / 16 = 256 such steps (4096 rows) in 64
// waves, so what bounds it is the latency of the fragments' loads: kAhead
// steps' fragments are in flight at any time.  One wave a SIMD is all there is
// to run, so they may take 256 registers (16 steps: 17.2 us; 32: 14.1).
// --------------------------------------------------------------------------
constexpr int kAhead = 32;

__device__ __forceinline__ floatx16 tile_product(const uint16_t* __restrict__ ap, size_t a_step,
                                                 const uint16_t* __restrict__ bp, size_t b_step,
                                                 int steps) {
  bf16x8 a[kAhead], b[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (u < steps) {
      a[u] = *reinterpret_cast<const bf16x8*>(ap + a_step * u);
      b[u] = *reinterpret_cast<const bf16x8*>(bp + b_step * u);
    }
  floatx16 acc = {};
  int s0 = 0;
  for (; s0 + 2 * kAhead <= steps; s0 += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u], b[u], acc, 0, 0, 0);
      a[u] = *reinterpret_cast<const bf16x8*>(ap + a_step * (size_t)(s0 + u + kAhead));
      b[u] = *reinterpret_cast<const bf16x8*>(bp + b_step * (size_t)(s0 + u + kAhead));
    }
  }
  for (; s0 < steps; s0 += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (s0 + u < steps) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u], b[u], acc, 0, 0, 0);
      if (s0 + u + kAhead < steps) {
        a[u] = *reinterpret_cast<const bf16x8*>(ap + a_step * (size_t)(s0 + u + kAhead));
        b[u] = *reinterpret_cast<const bf16x8*>(bp + b_step * (size_t)(s0 + u + kAhead));
      }
    }
  }
  return acc;
}

// the product over the batch of 32 columns m0 of A and 32 columns n0 of B,
// both in fragment order
__device__ __forceinline__ floatx16 batch_product(const uint16_t* __restrict__ A,
                                                  const uint16_t* __restrict__ B, int m0, int n0,
                                                  int batch, int lane) {
  return tile_product(A + frag_at(m0, 0, batch) + 8 * lane, 512, B + frag_at(n0, 0, batch) + 8 * lane, 512,
                      batch / 16);
}

__device__ __forceinline__ void store_tile(const floatx16& acc, float* __restrict__ C, int ldc, int m0,
                                           int n0, int lane) {
  const int n = n0 + (lane & 31);
#pragma unroll
  for (int v = 0; v < 16; ++v)
    C[(size_t)(m0 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4) * ldc + n] = acc[v];
}

// sum_r M[column][r] * (w ? w[r] : 1) over the batch by one wave, M in fragment
// order: lane l adds r = l, l + 64, ..., then a butterfly (sixteen loads in
// flight at a time; 64 rows on are four fragments on)
__device__ __forceinline__ float column_sum(const uint16_t* __restrict__ M, int column,
                                            const float* __restrict__ w, int batch, int lane) {
  const uint16_t* at = M + frag_at(column, lane, batch);
  float s = 0.0f;
  int r = lane;
  for (; r - lane + 1024 <= batch; r += 1024) {
    uint16_t x[16];
    float y[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      x[q] = at[2048 * (size_t)q];
      y[q] = w ? w[r + 64 * q] : 1.0f;
    }
    at += 2048 * 16;
#pragma unroll
    for (int q = 0; q < 16; ++q) s += w ? bf2f(x[q]) * y[q] : bf2f(x[q]);
  }
  for (; r < batch; r += 64, at += 2048) s += w ? bf2f(*at) * w[r] : bf2f(*at);
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  return s;
}

// sum of v[0..n) by one wave, as four partial sums of 256-strided elements
__device__ __forceinline__ float quarter_sums(const float* __restrict__ v, int n, int lane) {
  float part[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float s = 0.0f;
#pragma unroll 8
    for (int i = 64 * q + lane; i < n; i += 256) s += v[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    part[q] = s;
  }
  return (part[0] + part[1]) + (part[2] + part[3]);
}

// minibatch: row i of the batch = dataset row hash(seed, step, i) mod total
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

constexpr int kTrainRows = 32;                  // rows per workgroup of k_train_forward
constexpr int kTrainThreads = kMlpHidden / 32 * 64;
constexpr int kTrainStride = kMlpHidden + 8;    // padded LDS row of bf16
constexpr int kTrainPart = kMlpHidden + 4;      // padded LDS row of fp32

// A workgroup of 8 waves takes 32 rows through the forward pass, wave w the
// hidden columns [32w, 32w + 32) of both layers, and leaves behind what the
// gradients read: X, H1, H2 and dH2 transposed, and dH2.
//   loss_r = w_r [log(1 + e^-|z|) + max(z, 0) - z y],  dl_r = w_r (sigmoid(z) - y) / rows
// with w_r = pos_weight for visible rows, 1 otherwise; dH2 = [H2 > 0] dl[r] w3[k].
// The arithmetic and its order are the scorer's (k_mlp_score).  At 4096 rows it
// is 128 workgroups, half the CUs, and takes 15 us, most of it the latency of
// its loads, barriers and stores in turn.
__global__ __launch_bounds__(kTrainThreads) void k_train_forward(TrainArgs t) {
  __shared__ uint16_t s_h[kTrainRows * kTrainStride];  // H1, then dH2
  __shared__ float s_part[kTrainRows * kTrainPart];
  __shared__ uint64_t s_src[kTrainRows];
  __shared__ float s_dl[kTrainRows];
  __shared__ uint8_t s_y[kTrainRows];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 31, kh = 8 * (lane >> 5), hi = lane >> 5;
  const int n = wave * 32 + lr;  // this lane's hidden column
  const int row0 = blockIdx.x * kTrainRows;
  if (threadIdx.x < kTrainRows) {
    const uint64_t i = (uint64_t)(row0 + (int)threadIdx.x);
    // (total 0: the batch's rows as they are)
    const uint64_t src =
        t.total ? mix64(t.seed ^ mix64(t.step * 0x9e3779b97f4a7c15ull + i)) % t.total : i;
    s_src[threadIdx.x] = src;
    s_y[threadIdx.x] = t.Y[src];
  }
  bf16x8 w1f[2], w2f[kMlpHidden / 16];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    w1f[s] = *reinterpret_cast<const bf16x8*>(t.W1 + (size_t)n * kMlpIn + 16 * s + kh);
#pragma unroll
  for (int s = 0; s < kMlpHidden / 16; ++s)
    w2f[s] = *reinterpret_cast<const bf16x8*>(t.W2 + (size_t)n * kMlpHidden + 16 * s + kh);
  const float bias1 = t.b1[n], bias2 = t.b2[n], wn = bf2f(t.w3[n]), bias3 = *t.b3;
  __syncthreads();
  bf16x8 xa[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    xa[s] = *reinterpret_cast<const bf16x8*>(t.X + s_src[lr] * kMlpIn + 16 * s + kh);
  if (wave == 0) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const __bf16 x = xa[s][k];
        t.Xt[frag_at(16 * s + kh + k, row0 + lr, t.batch)] = __builtin_bit_cast(uint16_t, x);
      }
  }
  // layer 1
  floatx16 acc = {};
#pragma unroll
  for (int s = 0; s < 2; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[s], w1f[s], acc, 0, 0, 0);
  uint16_t h[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = 8 * (v / 4) + 4 * hi + (v % 4);
    float x = acc[v] + bias1;
    x = x > 0.0f ? x : 0.0f;
    h[v] = f2bf(x);
    s_h[m * kTrainStride + n] = h[v];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    store4(t.H1t + frag_at(n, row0 + 8 * q + 4 * hi, t.batch), h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]);
  __syncthreads();
  // layer 2
  acc = floatx16{};
#pragma unroll
  for (int s = 0; s < kMlpHidden / 16; ++s) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(s_h + lr * kTrainStride + 16 * s + kh);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w2f[s], acc, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = 8 * (v / 4) + 4 * hi + (v % 4);
    float x = acc[v] + bias2;
    x = x > 0.0f ? x : 0.0f;
    h[v] = f2bf(x);
    s_part[m * kTrainPart + n] = bf2f(h[v]) * wn;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    store4(t.H2t + frag_at(n, row0 + 8 * q + 4 * hi, t.batch), h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]);
  __syncthreads();
  // logits, loss and its gradient: wave w takes rows w, w + 8, ...; lane l
  // adds columns l, l + 64, l + 128, l + 192, then a butterfly
#pragma unroll
  for (int q = 0; q < kTrainRows / (kTrainThreads / 64); ++q) {
    const int m = wave + q * (kTrainThreads / 64);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kMlpHidden; k += 64) sum += s_part[m * kTrainPart + k + lane];
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) {
      const float z = sum + bias3;
      const float y = s_y[m] ? 1.0f : 0.0f;
      const float w = s_y[m] ? t.pos_weight : 1.0f;
      const float sig = 1.0f / (1.0f + expf(-z));
      const float d = w * (sig - y) / (float)t.batch;
      s_dl[m] = d;
      t.dl[row0 + m] = d;
      t.loss[row0 + m] = w * (log1pf(expf(-fabsf(z))) + fmaxf(z, 0.0f) - z * y);
    }
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = 8 * (v / 4) + 4 * hi + (v % 4);
    h[v] = bf2f(h[v]) > 0.0f ? f2bf(s_dl[m] * wn) : (uint16_t)0;
    s_h[m * kTrainStride + n] = h[v];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    store4(t.dH2t + frag_at(n, row0 + 8 * q + 4 * hi, t.batch), h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]);
  __syncthreads();
  // dH2 by rows, 32 bytes a thread
  static_assert(kTrainThreads * 16 == kTrainRows * kMlpHidden, "one pass");
  const int row = threadIdx.x / (kMlpHidden / 16), col = threadIdx.x % (kMlpHidden / 16) * 16;
  const uint4* src = reinterpret_cast<const uint4*>(s_h + row * kTrainStride + col);
  uint4* dst = reinterpret_cast<uint4*>(t.dH2 + (size_t)(row0 + row) * kMlpHidden + col);
  dst[0] = src[0];
  dst[1] = src[1];
}

// One wave per workgroup; by workgroup index: the 64 tiles of dW2 (the
// longest chains, first), the column sums for w3 and b2, the sums for b3 and the
// loss, then the tiles of dH1.
constexpr int kDw2Tiles = kMlpHidden / 32 * (kMlpHidden / 32);

__global__ __launch_bounds__(64) void k_train_grads(TrainArgs t) {
  const int lane = threadIdx.x;
  int i = (int)blockIdx.x;
  if (i < kDw2Tiles) {
    const int m0 = i / (kMlpHidden / 32) * 32, n0 = i % (kMlpHidden / 32) * 32;
    store_tile(batch_product(t.dH2t, t.H1t, m0, n0, t.batch, lane), t.gW2, kMlpHidden, m0, n0, lane);
    return;
  }
  i -= kDw2Tiles;
  if (i < 2 * kMlpHidden) {
    const bool w3 = i < kMlpHidden;
    const int j = w3 ? i : i - kMlpHidden;
    const float s = w3 ? column_sum(t.H2t, j, t.dl, t.batch, lane)
                       : column_sum(t.dH2t, j, nullptr, t.batch, lane);
    if (lane == 0) (w3 ? t.gw3 : t.gb2)[j] = s;
    return;
  }
  i -= 2 * kMlpHidden;
  if (i < 2) {
    const float s = quarter_sums(i ? t.dl : t.loss, t.batch, lane);
    if (lane == 0) *(i ? t.gb3 : t.loss_sum) = s;
    return;
  }
  i -= 2;
  const int m0 = i / (kMlpHidden / 32) * 32, n0 = i % (kMlpHidden / 32) * 32;
  const int kofs = 8 * (lane >> 5);
  const floatx16 acc = tile_product(t.dH2 + (size_t)(m0 + (lane & 31)) * kMlpHidden + kofs, 16,
                                    t.W2t + (size_t)(n0 + (lane & 31)) * kMlpHidden + kofs, 16,
                                    kMlpHidden / 16);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const size_t at = frag_at(n0 + (lane & 31), m0 + 8 * q + 4 * (lane >> 5), t.batch);
    const uint2 mask = *reinterpret_cast<const uint2*>(t.H1t + at);
    uint16_t d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint16_t hm = (uint16_t)((k < 2 ? mask.x : mask.y) >> (16 * (k & 1)));
      d[k] = f2bf(bf2f(hm) > 0.0f ? acc[4 * q + k] : 0.0f);
    }
    store4(t.dH1t + at, d[0], d[1], d[2], d[3]);
  }
}

// the 8 tiles of dW1, then the column sums for b1
__global__ __launch_bounds__(64) void k_train_grads1(TrainArgs t) {
  const int lane = threadIdx.x;
  const int i = (int)blockIdx.x;
  if (i < kMlpHidden / 32) {
    store_tile(batch_product(t.dH1t, t.Xt, 32 * i, 0, t.batch, lane), t.gW1, kMlpIn, 32 * i, 0, lane);
    return;
  }
  const int j = i - kMlpHidden / 32;
  const float s = column_sum(t.dH1t, j, nullptr, t.batch, lane);
  if (lane == 0) t.gb1[j] = s;
}

// float -> bf16 conversion (weights after the optimiser step), optionally
// also transposed ([rows][cols] -> [cols][rows])
__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ in, size_t n,
                                                 uint16_t* __restrict__ out,
                                                 uint16_t* __restrict__ out_t, int rows, int cols) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint16_t b = f2bf(in[i]);
  out[i] = b;
  if (out_t) out_t[(i % cols) * rows + i / cols] = b;
}

// Adam (Kingma & Ba 2015) on fp32 master weights; bc1/bc2 = bias corrections.
// Writes the new weights' bf16 copies as well.
__global__ __launch_bounds__(256) void k_adam(AdamArgs a) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const float gi = a.g[i];
  const float mi = a.b1 * a.m[i] + (1.0f - a.b1) * gi;
  const float vi = a.b2 * a.v[i] + (1.0f - a.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float w = a.w[i] - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
  a.w[i] = w;
  const uint16_t b = f2bf(w);
  if (i >= a.at_w1 && i < a.at_w1 + (size_t)kMlpHidden * kMlpIn) a.W1[i - a.at_w1] = b;
  if (i >= a.at_w2 && i < a.at_w2 + (size_t)kMlpHidden * kMlpHidden) {
    const size_t j = i - a.at_w2;
    a.W2[j] = b;
    a.W2t[j % kMlpHidden * kMlpHidden + j / kMlpHidden] = b;
  }
  if (i >= a.at_w3 && i < a.at_w3 + kMlpHidden) a.w3[i - a.at_w3] = b;
}

// ---- launchers --------------------------------------------------------------

static unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

hipError_t mlp_train(const TrainArgs& t, hipStream_t s) {
  // the batch is a multiple of 32 rows (checked by the callers)
  if (t.batch < kTrainRows || t.batch % kTrainRows) return hipErrorInvalidValue;
  const unsigned row_tiles = (unsigned)(t.batch / kTrainRows);
  hipLaunchKernelGGL(k_train_forward, dim3(row_tiles), dim3(kTrainThreads), 0, s, t);
  hipLaunchKernelGGL(k_train_grads, dim3(kDw2Tiles + 2 * kMlpHidden + 2 + row_tiles * (kMlpHidden / 32)),
                     dim3(64), 0, s, t);
  hipLaunchKernelGGL(k_train_grads1, dim3(kMlpHidden / 32 + kMlpHidden), dim3(64), 0, s, t);
  return hipGetLastError();
}

hipError_t mlp_to_bf16(const float* in, size_t n, uint16_t* out, uint16_t* out_t, int rows, int cols,
                       hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks_for(n)), dim3(256), 0, s, in, n, out, out_t, rows, cols);
  return hipGetLastError();
}

hipError_t mlp_adam(const AdamArgs& a, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(a.n)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace gbr

namespace gbr {

// --------------------------------------------------------------------------
// Fused scorer for rendering: logits of min(rows, *rows_dev) feature rows in
// one persistent pass with the weights in registers.  A workgroup of 8 waves
// holds the model: wave w owns hidden columns [32w, 32w + 32) of both layers,
// with its slices of W1 (2 MFMA B fragments) and W2 (16 fragments) in VGPRs
// for the whole kernel.  Per tile of 32 rows: layer 1 (K = 32, 2
// v_mfma_f32_32x32x16_bf16) -> bias, ReLU, bf16 -> the tile's H1 in LDS;
// layer 2 (K = 256, 16 MFMAs, A fragments from LDS) -> bias, ReLU, bf16,
// times w3 -> per-column products in LDS; then each row's logit is summed in
// k_train_forward's order (lane l: columns l, l+64, l+128, l+192, then a
// butterfly over 64 lanes).  The K loops run k = 0, 16, ... like its own, so
// H1, H2 and the logits equal the training forward's bit for bit.
// --------------------------------------------------------------------------

constexpr int kScoreRows = 32;                  // rows per tile
constexpr int kScoreWaves = kMlpHidden / 32;    // one wave per 32 hidden columns
constexpr int kScoreThreads = kScoreWaves * 64;
constexpr int kH1Stride = kMlpHidden + 8;       // padded LDS row of H1 (bf16)
constexpr int kPartStride = kMlpHidden + 4;     // padded LDS row of the products (fp32)
static_assert(kMlpIn == 32 && kMlpHidden % 32 == 0, "scorer tiling");
static_assert(kScoreRows % kScoreWaves == 0, "rows of the logit reduction per wave");

__global__ __launch_bounds__(kScoreThreads) void k_mlp_score(const uint16_t* __restrict__ X,
                                                             const uint16_t* __restrict__ W1,
                                                             const float* __restrict__ b1,
                                                             const uint16_t* __restrict__ W2,
                                                             const float* __restrict__ b2,
                                                             const uint16_t* __restrict__ w3,
                                                             const float* __restrict__ b3,
                                                             int rows,
                                                             const uint32_t* __restrict__ rows_dev,
                                                             float* __restrict__ logits) {
  __shared__ uint16_t s_h1[kScoreRows * kH1Stride];
  __shared__ float s_part[kScoreRows * kPartStride];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 31, kh = 8 * (lane >> 5);
  const int n = wave * 32 + lr;  // this lane's hidden column
  const int n_rows = rows_of(rows, rows_dev);
  const int n_tiles = (n_rows + kScoreRows - 1) / kScoreRows;
  if ((int)blockIdx.x >= n_tiles) return;  // (whole workgroup)
  // the wave's weight slices, loaded once
  bf16x8 w1f[2], w2f[kMlpHidden / 16];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    w1f[s] = *reinterpret_cast<const bf16x8*>(W1 + (size_t)n * kMlpIn + 16 * s + kh);
#pragma unroll
  for (int s = 0; s < kMlpHidden / 16; ++s)
    w2f[s] = *reinterpret_cast<const bf16x8*>(W2 + (size_t)n * kMlpHidden + 16 * s + kh);
  const float bias1 = b1[n], bias2 = b2[n], wn = bf2f(w3[n]), bias3 = *b3;
  // the A fragments of a tile's feature rows, fetched one tile ahead (rows
  // past the last read the last row; they are zeroed when used)
  bf16x8 xnext[2];
  auto load_x = [&](int tile, bf16x8 (&xa)[2]) {
    const int rr = min(tile * kScoreRows + lr, n_rows - 1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
      xa[s] = *reinterpret_cast<const bf16x8*>(X + (size_t)rr * kMlpIn + 16 * s + kh);
  };
  load_x(blockIdx.x, xnext);
  for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int row0 = tile * kScoreRows;
    bf16x8 xa[2] = {xnext[0], xnext[1]};
    if (row0 + lr >= n_rows) xa[0] = xa[1] = bf16x8{};
    if (tile + (int)gridDim.x < n_tiles) load_x(tile + gridDim.x, xnext);
    // layer 1: the tile's 32 rows (zero past the last row) x the wave's columns
    floatx16 acc = {};
#pragma unroll
    for (int s = 0; s < 2; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[s], w1f[s], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
      float x = acc[v] + bias1;
      x = x > 0.0f ? x : 0.0f;
      s_h1[m * kH1Stride + n] = f2bf(x);
    }
    __syncthreads();  // H1 complete (and the previous tile's products are consumed)
    // layer 2: A fragments of every row from LDS, the wave's W2 slice from VGPRs
    acc = floatx16{};
#pragma unroll
    for (int s = 0; s < kMlpHidden / 16; ++s) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(s_h1 + lr * kH1Stride + 16 * s + kh);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w2f[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
      float x = acc[v] + bias2;
      x = x > 0.0f ? x : 0.0f;
      s_part[m * kPartStride + n] = bf2f(f2bf(x)) * wn;
    }
    __syncthreads();  // products complete; H1 may be rewritten
    // logits: wave w sums rows w, w + 8, ... in k_train_forward's order
#pragma unroll
    for (int q = 0; q < kScoreRows / kScoreWaves; ++q) {
      const int m = wave + q * kScoreWaves;
      float sum = 0.0f;
#pragma unroll
      for (int k = 0; k < kMlpHidden; k += 64) sum += s_part[m * kPartStride + k + lane];
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
      if (lane == 0 && row0 + m < n_rows) logits[row0 + m] = sum + bias3;
    }
  }
}

hipError_t mlp_score(const uint16_t* X, const uint16_t* W1, const float* b1, const uint16_t* W2,
                     const float* b2, const uint16_t* w3, const float* b3, int rows,
                     const uint32_t* rows_dev, float* logits, int max_blocks, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  const int tiles = (rows + kScoreRows - 1) / kScoreRows;
  const int blocks = max_blocks > 0 ? std::min(tiles, max_blocks) : tiles;
  hipLaunchKernelGGL(k_mlp_score, dim3(blocks), dim3(kScoreThreads), 0, s, X, W1, b1, W2, b2, w3,
                     b3, rows, rows_dev, logits);
  return hipGetLastError();
}

}  // namespace gbr
