// pw_mlp_train.hip -- training of the far-field network (FP32 master
// weights, FP32 arithmetic) and the packing of its BF16 inference
// fragments.
//
// One block trains on tiles of 16 samples: forward through the four layers with
// the pre-activations kept in registers, then back-propagation of the squared
// error, the weight gradients accumulated in registers over the block's tiles
// and written to the block's own row of a partial buffer; a second kernel sums
// the rows in a fixed order (deterministic) and a third applies Adam.  Every
// product runs on the matrix cores in FP32 (v_mfma_f32_16x16x4: FP32 inputs,
// products and sums).  GELU is the tanh form x sigmoid(2 z), z = sqrt(2/pi)(x +
// 0.044715 x^3), the same function as the inference kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "pw_mlp.h"

namespace pw {
namespace {

constexpr int R = kTrainRows;
constexpr int H = kMlpHid;
constexpr int kLd = H + 4;    // row stride of the 128-wide LDS arrays
constexpr int kLdN = 16 + 4;  // of the 16-wide ones

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gelu_f(float x) {
  const float z2 = -2.0f * 0.7978845608f * fmaf(0.044715f * x * x, x, x);
  return x / (1.0f + __expf(z2));
}
__device__ __forceinline__ float gelu_d(float x) {
  const float z2 = -2.0f * 0.7978845608f * fmaf(0.044715f * x * x, x, x);
  const float sg = 1.0f / (1.0f + __expf(z2));
  const float dz = 0.7978845608f * fmaf(3.0f * 0.044715f, x * x, 1.0f);
  return sg + x * sg * (1.0f - sg) * 2.0f * dz;
}

struct TrainLds {
  float x[R][kLdN];
  float h1[R][kLd], h2[R][kLd], h3[R][kLd];
  float d[2][R][kLd];   // deltas of two neighbouring layers
  float o[R][kLdN];     // 2 (f - y)
  float part[4][R][16]; // the output layer's four K quarters
  float loss[4];
};

// Tiles.  A 16x16 tile D += A B of v_mfma_f32_16x16x4 (four k per instruction):
// lane l = 16 g + c holds A[c][k_g], B[k_g][c] and D[4 g + r][c], r = 0..3.  Which
// k goes to group g in step s is free as long as A and B agree; over K = 128
// group g takes k = 32 g + s, so that a lane's A values are contiguous in LDS.
__device__ __forceinline__ v4f mfma(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// This lane's 64 B values of a 128-long product, for the wave's two column
// tiles: value s of tile t.  Loaded a product ahead of their use, so that a
// wave, alone on its SIMD, does not wait for them (registers are there: 512).
struct Weights {
  float v[2][32];
};

// W[k][j] row-major 128 x 128: columns j of the forward product;
// w = W + 32 wave + c + 128 * 32 g
__device__ __forceinline__ void load_forward(const float* __restrict__ w, Weights& b) {
#pragma unroll
  for (int s = 0; s < 32; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t) b.v[t][s] = w[H * s + 16 * t];
}
// the transposed product: column n of W^T is row n of W;
// w = W + 128 (32 wave + c) + 32 g
__device__ __forceinline__ void load_backward(const float* __restrict__ w, Weights& b) {
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const v4f x = *reinterpret_cast<const v4f*>(w + 16 * H * t + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) b.v[t][4 * q + i] = x[i];
    }
}

// acc[t] += in (16 x 128, LDS) times B, for the wave's two column tiles
__device__ __forceinline__ void product128(const float (*in)[kLd], const Weights& b, v4f (&acc)[2]) {
  const int lane = static_cast<int>(threadIdx.x) & 63, c = lane & 15, g = lane >> 4;
  v4f a[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) a[q] = *reinterpret_cast<const v4f*>(&in[c][32 * g + 4 * q]);
#pragma unroll
  for (int s = 0; s < 32; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] = mfma(a[s >> 2][s & 3], b.v[t][s], acc[t]);
}

// acc[a][b] += in^T d over the tile's 16 samples: rows 16 (NA wave + a) of the
// weights, columns 16 b
template <int NA, int NB, int LDI, int LDD>
__device__ __forceinline__ void wgrad(const float (*in)[LDI], int row0, const float (*d)[LDD], int col0,
                                      v4f (&acc)[NA][NB]) {
  const int lane = static_cast<int>(threadIdx.x) & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < R / 4; ++s) {
    float a[NA], b[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) a[i] = in[4 * s + g][row0 + 16 * i + c];
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = d[4 * s + g][col0 + 16 * j + c];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
  }
}

// the wave's two column tiles to LDS, through f(pre-activation)
template <typename F>
__device__ __forceinline__ void store_tiles(const v4f (&a)[2], float (*out)[kLd], F f) {
  const int lane = static_cast<int>(threadIdx.x) & 63, c = lane & 15, g = lane >> 4, wave = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) out[4 * g + r][32 * wave + 16 * t + c] = f(a[t][r], t, r);
}

// Each wave owns 32 of the 128 units: forward and backward products write its
// columns, so its pre-activations stay in its registers for gelu'; activations
// and deltas pass to the other waves through LDS.  Weights are read straight
// from memory, each by the one wave that uses it, a phase ahead of their use:
// the block is nine phases between barriers, and with the loads inside them each
// waited for memory (42.6 us a batch of 4,096, now 32.3, of which the matrix
// cores work 6 and the partial rows take about 9 to write).
//
// The products were FP32 vector instructions fed one LDS read each, over 32
// samples per block: 144 us for a batch of 4,096 on 128 CUs (164 us a training
// step of 1,024 on 32).
__global__ __launch_bounds__(256) void k_mlp_grad(const float* __restrict__ params, const float* __restrict__ X,
                                                  const float* __restrict__ Y, const int* __restrict__ idx,
                                                  int n, float* __restrict__ gpart, float* __restrict__ lpart) {
  extern __shared__ __align__(16) unsigned char smem[];
  TrainLds& s = *reinterpret_cast<TrainLds*>(smem);
  const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int col = 32 * wave + c;  // this lane's first column
  v4f g1[1][2] = {}, g2[2][8] = {}, g3[2][8] = {}, g4[2][1] = {};
  float gb[3] = {0.0f, 0.0f, 0.0f}, gb4 = 0.0f, lsum = 0.0f;
  const auto sample = [&](int r) { return static_cast<size_t>(idx ? idx[r] : r); };
  const int tiles = (n + R - 1) / R;
  for (int tile = static_cast<int>(blockIdx.x); tile < tiles; tile += static_cast<int>(gridDim.x)) {
    const int row0 = tile * R;
    // the same weights for every tile: an opaque base keeps the compiler from
    // hoisting 147 KB of loads out of the loop into (spilled) registers
    const float* P = params;
    asm volatile("" : "+s"(P));
    // what the first phases read, in flight together: inputs (rows beyond n are
    // zero and carry zero error), biases, first and second layer
    const int er = tid >> 4, ej = tid & 15;  // this thread's input, and its output's error
    const bool has = row0 + er < n;
    const size_t at = sample(has ? row0 + er : row0);
    const float xin = X[at * kMlpIn + ej];
    v4f a1[2], a2[2], a3[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        a1[t][r] = P[kOffB1 + col + 16 * t];
        a2[t][r] = P[kOffB2 + col + 16 * t];
        a3[t][r] = P[kOffB3 + col + 16 * t];
      }
    static_assert(kMlpIn == 16 && R == 16, "one 16x16 tile of inputs");
    float w1[4][2];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int t = 0; t < 2; ++t) w1[q][t] = P[kOffW1 + H * (4 * q + g) + col + 16 * t];
    Weights wa, wb;
    load_forward(P + kOffW2 + 32 * H * g + col, wa);
    s.x[er][ej] = has ? xin : 0.0f;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int t = 0; t < 2; ++t) a1[t] = mfma(s.x[c][4 * q + g], w1[q][t], a1[t]);
    const auto act = [](float v, int, int) { return gelu_f(v); };
    store_tiles(a1, s.h1, act);
    load_forward(P + kOffW3 + 32 * H * g + col, wb);
    __syncthreads();
    product128(s.h1, wa, a2);
    store_tiles(a2, s.h2, act);
    load_backward(P + kOffW3 + H * col + 32 * g, wa);
    // the output layer's weights both ways, its bias and the target
    float w4[8], w4t[3][2];
#pragma unroll
    for (int q = 0; q < 8; ++q) w4[q] = c < kMlpOut ? P[kOffW4 + (32 * wave + 4 * q + g) * kMlpOut + c] : 0.0f;
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int t = 0; t < 2; ++t) w4t[q][t] = P[kOffW4 + (col + 16 * t) * kMlpOut + 4 * q + g];
    const bool out_on = ej < kMlpOut && has;
    const float b4 = out_on ? P[kOffB4 + ej] : 0.0f, target = out_on ? Y[at * kMlpOut + ej] : 0.0f;
    __syncthreads();
    product128(s.h2, wb, a3);
    store_tiles(a3, s.h3, act);
    __syncthreads();
    // output layer: 12 columns of one tile, a K quarter per wave
    {
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int q = 0; q < 8; ++q) acc = mfma(s.h3[c][32 * wave + 4 * q + g], w4[q], acc);
#pragma unroll
      for (int r = 0; r < 4; ++r) s.part[wave][4 * g + r][c] = acc[r];
    }
    __syncthreads();
    {
      float err = 0.0f;
      if (out_on)
        err = (((s.part[0][er][ej] + s.part[1][er][ej]) + (s.part[2][er][ej] + s.part[3][er][ej])) + b4) - target;
      s.o[er][ej] = 2.0f * err;
      lsum = fmaf(err, err, lsum);
    }
    __syncthreads();
    // delta3 = (o W4^T) gelu'(a3): 12 columns in three steps
    v4f d[2] = {};
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        d[t] = mfma(s.o[c][4 * q + g], w4t[q][t], d[t]);
    load_backward(P + kOffW2 + H * col + 32 * g, wb);
    store_tiles(d, s.d[0], [&](float v, int t, int r) { return v * gelu_d(a3[t][r]); });
    wgrad<2, 1>(s.h3, 32 * wave, s.o, 0, g4);
    if (tid < kMlpOut)
      for (int r = 0; r < R; ++r) gb4 += s.o[r][tid];
    __syncthreads();
    // delta2, and the third layer's gradient
    d[0] = d[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    product128(s.d[0], wa, d);
    store_tiles(d, s.d[1], [&](float v, int t, int r) { return v * gelu_d(a2[t][r]); });
    wgrad<2, 8>(s.h2, 32 * wave, s.d[0], 0, g3);
    if (tid < H)
      for (int r = 0; r < R; ++r) gb[2] += s.d[0][r][tid];
    __syncthreads();
    // delta1, and the second layer's
    d[0] = d[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    product128(s.d[1], wb, d);
    store_tiles(d, s.d[0], [&](float v, int t, int r) { return v * gelu_d(a1[t][r]); });
    wgrad<2, 8>(s.h1, 32 * wave, s.d[1], 0, g2);
    if (tid < H)
      for (int r = 0; r < R; ++r) gb[1] += s.d[1][r][tid];
    __syncthreads();
    wgrad<1, 2>(s.x, 0, s.d[0], 32 * wave, g1);
    if (tid < H)
      for (int r = 0; r < R; ++r) gb[0] += s.d[0][r][tid];
    __syncthreads();  // x and the deltas are free for the next tile
  }
  float* out = gpart + static_cast<size_t>(blockIdx.x) * kMlpParams;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 32 * wave + 16 * i + 4 * g + r;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        out[kOffW2 + H * row + 16 * j + c] = g2[i][j][r];
        out[kOffW3 + H * row + 16 * j + c] = g3[i][j][r];
      }
      if (c < kMlpOut) out[kOffW4 + kMlpOut * row + c] = g4[i][0][r];
      out[kOffW1 + H * (4 * g + r) + col + 16 * i] = g1[0][i][r];
    }
  }
  if (tid < H) {
    out[kOffB1 + tid] = gb[0];
    out[kOffB2 + tid] = gb[1];
    out[kOffB3 + tid] = gb[2];
  }
  if (tid < kMlpOut) out[kOffB4 + tid] = gb4;
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
  if (lane == 0) s.loss[wave] = lsum;
  __syncthreads();
  if (tid == 0) lpart[blockIdx.x] = (s.loss[0] + s.loss[1]) + (s.loss[2] + s.loss[3]);
}

// grad[p] = sum_b gpart[b][p] / n; loss likewise.  64 parameters per block, a
// quarter of the rows per wave (in order), the quarters added in order.
__global__ __launch_bounds__(256) void k_grad_reduce(const float* __restrict__ gpart, const float* __restrict__ lpart,
                                                     int blocks, int n, float* __restrict__ grad,
                                                     float* __restrict__ loss) {
  __shared__ float red[4][64];
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = static_cast<int>(threadIdx.x) & 63;
  const int p = static_cast<int>(blockIdx.x) * 64 + lane;
  const float inv = 1.0f / static_cast<float>(n);
  const int b0 = blocks * wave / 4, b1 = blocks * (wave + 1) / 4;
  float acc = 0.0f;
  if (p < kMlpParams) {
#pragma unroll 8
    for (int b = b0; b < b1; ++b) acc += gpart[static_cast<size_t>(b) * kMlpParams + p];
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && p < kMlpParams) grad[p] = ((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane])) * inv;
  if (blockIdx.x == 0 && wave == 1) {
    float l = 0.0f;
    for (int b = lane; b < blocks; b += 64) l += lpart[b];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
    if (lane == 0) *loss = l * inv;
  }
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ P, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, float lr,
                                              float b1, float b2, float eps, float c1, float c2) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= kMlpParams) return;
  const float gi = g[p];
  const float mi = b1 * m[p] + (1.0f - b1) * gi;
  const float vi = b2 * v[p] + (1.0f - b2) * gi * gi;
  m[p] = mi;
  v[p] = vi;
  P[p] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

}  // namespace

// One block per tile up to one per CU (413 registers: one wave per SIMD), then
// several tiles per block: the partial rows, 147 KB each, stay below 38 MB.
int train_blocks(int n) {
  const int tiles = (n + R - 1) / R;
  return std::min(tiles, 256);
}

hipError_t launch_mlp_grad(const float* params, const float* X, const float* Y, const int* idx, int n,
                           float* gpart, float* lpart, float* grad, float* loss_dev, hipStream_t st) {
  if (n <= 0) return hipErrorInvalidValue;
  const int blocks = train_blocks(n);
  static std::atomic<unsigned long long> lds_raised{0};
  hipError_t e = ensure_lds_limit(reinterpret_cast<const void*>(k_mlp_grad), sizeof(TrainLds), lds_raised);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mlp_grad, dim3(blocks), dim3(256), sizeof(TrainLds), st, params, X, Y, idx, n, gpart,
                     lpart);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_grad_reduce, dim3((kMlpParams + 63) / 64), dim3(256), 0, st, gpart, lpart, blocks,
                     n, grad, loss_dev);
  return hipGetLastError();
}

hipError_t launch_adam(float* params, const float* grad, float* m, float* v, float lr, float b1, float b2,
                       float eps, int step, hipStream_t st) {
  const float c1 = 1.0f / (1.0f - std::pow(b1, static_cast<float>(step)));
  const float c2 = 1.0f / (1.0f - std::pow(b2, static_cast<float>(step)));
  hipLaunchKernelGGL(k_adam, dim3((kMlpParams + 255) / 256), dim3(256), 0, st, params, grad, m, v, lr, b1, b2,
                     eps, c1, c2);
  return hipGetLastError();
}

uint16_t bf16_bits(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return 0x7fc0;  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

void pack_mlp(const float* P, std::vector<uint16_t>& frag, std::vector<float>& bias) {
  frag.assign(kMlpFragElems, 0);
  bias.assign(kMlpBiasLen, 0.0f);
  size_t o = 0;
  // layer 1: tile m, lane (c, g), slot j -> W1[4g + j][16m + c]
  for (int m = 0; m < 8; ++m)
    for (int lane = 0; lane < 64; ++lane)
      for (int j = 0; j < 4; ++j) {
        const int c = lane & 15, g = lane >> 4;
        frag[o++] = bf16_bits(P[kOffW1 + (4 * g + j) * H + 16 * m + c]);
      }
  // layers 2, 3: tile m, K block b, lane, slot j -> W[in][16m + c],
  // in = 32b + 4g + j (j < 4), 32b + 16 + 4g + j - 4 (j >= 4)
  for (int layer = 0; layer < 2; ++layer) {
    const float* W = P + (layer == 0 ? kOffW2 : kOffW3);
    for (int m = 0; m < 8; ++m)
      for (int b = 0; b < 4; ++b)
        for (int lane = 0; lane < 64; ++lane)
          for (int j = 0; j < 8; ++j) {
            const int c = lane & 15, g = lane >> 4;
            const int in = 32 * b + (j < 4 ? 4 * g + j : 16 + 4 * g + j - 4);
            frag[o++] = bf16_bits(W[in * H + 16 * m + c]);
          }
  }
  // layer 4: K block b, lane, slot j -> W4[in][c] (c < 12)
  for (int b = 0; b < 4; ++b)
    for (int lane = 0; lane < 64; ++lane)
      for (int j = 0; j < 8; ++j) {
        const int c = lane & 15, g = lane >> 4;
        const int in = 32 * b + (j < 4 ? 4 * g + j : 16 + 4 * g + j - 4);
        frag[o++] = c < kMlpOut ? bf16_bits(P[kOffW4 + in * kMlpOut + c]) : 0;
      }
  for (int j = 0; j < H; ++j) {
    bias[j] = P[kOffB1 + j];
    bias[H + j] = P[kOffB2 + j];
    bias[2 * H + j] = P[kOffB3 + j];
  }
  for (int j = 0; j < kMlpOut; ++j) bias[3 * H + j] = P[kOffB4 + j];
}

void init_mlp(uint64_t seed, float* P) {
  // weights and biases of a layer uniform in +-1/sqrt(fan_in); trains
  // markedly faster on the far-field samples than Glorot with zero biases
  uint64_t s = seed;
  auto fill = [&](int off, int count, int fan_in) {
    const double lim = 1.0 / std::sqrt(static_cast<double>(fan_in));
    for (int i = 0; i < count; ++i) {
      const double u = (splitmix(s) >> 11) * 0x1.0p-53;
      P[off + i] = static_cast<float>((2.0 * u - 1.0) * lim);
    }
  };
  fill(kOffW1, kMlpIn * H, kMlpIn);
  fill(kOffB1, H, kMlpIn);
  fill(kOffW2, H * H, H);
  fill(kOffB2, H, H);
  fill(kOffW3, H * H, H);
  fill(kOffB3, H, H);
  fill(kOffW4, H * kMlpOut, H);
  fill(kOffB4, kMlpOut, H);
}

}  // namespace pw
