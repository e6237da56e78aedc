// gfx950 kernels of the learned preconditioner: a 4-layer 3x3 convolutional
// network (4 -> 32 -> 32 -> 32 -> 3 channels, GELU after the first three
// layers, zero padding), FP32 weights and accumulation, BF16 activations.
// No reference counterpart: FwiFlow's plain method is L-BFGS on the raw
// gradient; this network maps (gradient of cp, cs, rho; illumination) to a
// search direction and is trained on the plain inversion's accepted updates.
//
// Layouts: feature maps are planar [channel][row][column] (rows = depth z,
// columns = x fastest), i.e. the row-major [NZ][NX] of the operator's
// gradients, one plane per channel.  Parameters are one flat FP32 vector:
// per layer W [Cout][Cin][3][3] then b [Cout].
//
// The layers are products on the FP32 matrix cores (weights x pixels).  An FP32
// MFMA adds its products to the accumulator one by one in the order of k, each
// a fused multiply-add, so every sum has a fixed order: channels, then taps
// (k = 9 ci + t) from the bias on; pixels of a 16x16 tile row by row; tiles.
//
// Kernels:
//   k_conv32     3x3 convolution to 32 channels (hidden layers; input gradients,
//                as the convolution with the transposed and flipped weights)
//   k_conv3      the output layer
//   k_wgrad      weight / bias gradient partial sums of one 16x16 tile
//   k_sum_rows   deterministic reduction of the per-tile partials
//   k_loss_grad  masked MSE and its gradient
//   k_adam       Adam update
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "cnn.hpp"

namespace fwiflow {
namespace {

#define TRY(expr)            \
  do {                       \
    Status s_ = (expr);      \
    if (!s_.ok()) return s_; \
  } while (0)

#define CNN_HIP(expr)                                                                        \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess)                                                                    \
      return Status::Err(FWIFLOW_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int kTile = 16;       // tile edge of the weight gradient
constexpr int kHalo = kTile + 2;
constexpr int kMaxC = 32;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;

// FP32 -> BF16, round to nearest even (finite inputs; NaN kept as NaN)
__device__ inline bf16_t to_bf16(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ inline float from_bf16(bf16_t h) { return __uint_as_float((unsigned)h << 16); }

__device__ inline float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
  const float cdf = 0.5f * (1.f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

template <typename T>
__device__ inline float load_act(const T* p, size_t i);
template <>
__device__ inline float load_act<float>(const float* p, size_t i) {
  return p[i];
}
template <>
__device__ inline float load_act<bf16_t>(const bf16_t* p, size_t i) {
  return from_bf16(p[i]);
}

// Pixels (xa .. xa + TX - 1, ya .. ya + TY - 1) of the first C of CIN channels
// into lds[CIN][CS] (rows of TX pixels), zero outside the map and beyond C.  A
// wave takes whole channels, so that a lane's pixels and their offsets are the
// same for all of them.
template <typename TIn, int CIN, int C, int TY, int TX, int CS, int NW>
__device__ __forceinline__ void stage(const TIn* __restrict__ in, int H, int W, int xa, int ya, float* lds) {
  constexpr int N = TX * TY, I = (N + 63) / 64;
  const size_t plane = (size_t)H * W;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  size_t off[I];
  bool ok[I];
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int r = min(lane + 64 * i, N - 1), yy = ya + r / TX, xx = xa + r % TX;
    ok[i] = yy >= 0 && yy < H && xx >= 0 && xx < W;
    off[i] = (size_t)min(max(yy, 0), H - 1) * W + min(max(xx, 0), W - 1);
  }
#pragma unroll 2
  for (int c = wave; c < CIN; c += NW) {
    const TIn* p = in + (size_t)min(c, C - 1) * plane;
    float v[I];
#pragma unroll
    for (int i = 0; i < I; ++i) v[i] = load_act<TIn>(p, off[i]);
#pragma unroll
    for (int i = 0; i < I; ++i)
      if (lane + 64 * i < N) lds[c * CS + lane + 64 * i] = ok[i] && c < C ? v[i] : 0.f;
  }
}

constexpr int kConvX = 32, kConvY = 8;  // pixels of a convolution's tile
constexpr int kConvS = kConvX + 2;      // and of its row with the halo
// Tiles of a map, along y and z of the grid in runs of kConvRun: 65536 workgroups,
// the most along y, would end at 524288 rows.
constexpr int kConvRun = 32768;
__device__ __forceinline__ int conv_row() { return (int)(blockIdx.z * kConvRun + blockIdx.y) * kConvY; }
dim3 conv_grid(int H, int W) {
  const int rows = (H + kConvY - 1) / kConvY;
  return dim3((W + kConvX - 1) / kConvX, std::min(rows, kConvRun), (rows + kConvRun - 1) / kConvRun);
}

enum Epilogue { kHidden = 0, kInputGrad = 1 };

// out[m][y][x] = b[m] + sum_{c,ky,kx} w(m, c, ky, kx) in[c][y+ky-1][x+kx-1] for
// 32 channels m; in has C channels (CIN, even, in LDS).  kHidden: w = W[m][c][t];
// kInputGrad: W is the layer above's [C][32][9] and w = W[c][m][8 - t].
//
// Eight waves of a row of 32 pixels each; input (+1 halo) and weights in LDS (80
// KB: two workgroups a compute unit), 9 matrix instructions per two channels:
// 32 channels x 32 pixels x 2 products.  A lane's pixel operand for products k,
// k + 1 differs between the wave's halves by one of three offsets.
// Bound by the matrix cores (1.85 GFLOP at 224x448: 11.8 us at the card's 157
// TFLOP/s, 15.4 with the last of 3.06 rows a SIMD), before and after them by the
// load of the tile and the GELU.  224x448, 32 -> 32 channels: 107 -> 33 us
// against one pixel a thread with weights as scalars and vector multiply-adds
// (4 -> 32: 25 -> 15 us); four waves of two rows 36, of one row 40, two waves 53.
template <typename TIn, int CIN, int C, int EPI>
__global__ __launch_bounds__(64 * kConvY) void k_conv32(const TIn* __restrict__ in, int H, int W,
                                                        const float* __restrict__ w,
                                                        const float* __restrict__ b,
                                                        float* __restrict__ out_f32,
                                                        bf16_t* __restrict__ z_bf16,
                                                        bf16_t* __restrict__ a_bf16,
                                                        const bf16_t* __restrict__ zin) {
  constexpr int NW = kConvY, K = CIN * 9, CH = (kConvY + 2) * kConvS, WS = 33;
  __shared__ float tile[CIN * CH];
  __shared__ float wk[K * WS];  // [k][channel]
  const int x0 = blockIdx.x * kConvX, y0 = conv_row();
  if (y0 >= H) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t plane = (size_t)H * W;
  stage<TIn, CIN, C, kConvY + 2, kConvS, CH, NW>(in, H, W, x0 - 1, y0 - 1, tile);
  {
    // a wave takes whole channels: of the output, or of the layer above
    constexpr int N = EPI == kInputGrad ? 288 : C * 9, M = EPI == kInputGrad ? C : 32, I = (N + 63) / 64;
    int to[I];
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int r = lane + 64 * i;
      to[i] = EPI == kInputGrad ? (8 - r % 9) * WS + r / 9 : r * WS;
    }
#pragma unroll 2
    for (int m = wave; m < M; m += NW) {
      float v[I];
#pragma unroll
      for (int i = 0; i < I; ++i) v[i] = w[m * N + min(lane + 64 * i, N - 1)];
#pragma unroll
      for (int i = 0; i < I; ++i)
        if (lane + 64 * i < N) wk[to[i] + m * (EPI == kInputGrad ? 9 * WS : 1)] = v[i];
    }
  }
  if (C < CIN)
    for (int i = threadIdx.x; i < (CIN - C) * 9 * 32; i += 64 * NW)
      wk[(C * 9 + i / 32) * WS + i % 32] = 0.f;
  __syncthreads();
  const int n = lane & 31, h = lane >> 5;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = b ? b[8 * (i / 4) + 4 * h + i % 4] : 0.f;
  const float* wp = wk + h * WS + n;
  const float* tp = tile + wave * kConvS + n;
#pragma unroll 2
  for (int c = 0; c < CIN; c += 2, wp += 18 * WS, tp += 2 * CH) {
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      constexpr auto off = [](int k) { return k / 9 * CH + k % 9 / 3 * kConvS + k % 3; };
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wp[2 * j * WS], tp[h ? off(2 * j + 1) : off(2 * j)], acc, 0, 0, 0);
    }
  }
  const int x = x0 + n, y = y0 + wave;
  if (x >= W || y >= H) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const size_t o = (size_t)(8 * (i / 4) + 4 * h + i % 4) * plane + (size_t)y * W + x;
    if (EPI == kHidden) {
      z_bf16[o] = to_bf16(acc[i]);
      a_bf16[o] = to_bf16(gelu(acc[i]));
    } else {  // gradient of the activation -> of its z
      out_f32[o] = acc[i] * gelu_grad(from_bf16(zin[o]));
    }
  }
}

// The output layer: 32 -> 3 channels, FP32 result.  Three rows would leave nine
// tenths of a matrix instruction idle: one pixel a thread, weights as scalars.
// 224x448: 28 -> 14 us with all channels of the tile loaded at once.
__global__ __launch_bounds__(256) void k_conv3(const bf16_t* __restrict__ in, int H, int W,
                                               const float* __restrict__ w,
                                               const float* __restrict__ b, float* __restrict__ out) {
  constexpr int CH = (kConvY + 2) * kConvS;
  __shared__ float tile[32 * CH];
  const int x0 = blockIdx.x * kConvX, y0 = conv_row();
  if (y0 >= H) return;
  stage<bf16_t, 32, 32, kConvY + 2, kConvS, CH, 4>(in, H, W, x0 - 1, y0 - 1, tile);
  __syncthreads();
  const int n = threadIdx.x & 31, x = x0 + n, y = y0 + (threadIdx.x >> 5);
  const float* t = tile + (threadIdx.x >> 5) * kConvS + n;
  float acc[3] = {b[0], b[1], b[2]};
#pragma unroll 2
  for (int c = 0; c < 32; ++c, t += CH)
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const float v = t[k / 3 * kConvS + k % 3];
#pragma unroll
      for (int co = 0; co < 3; ++co) acc[co] += w[co * 288 + c * 9 + k] * v;
    }
  if (x >= W || y >= H) return;
#pragma unroll
  for (int co = 0; co < 3; ++co) out[(size_t)co * H * W + (size_t)y * W + x] = acc[co];
}

// Partial weight and bias gradients of one 16x16 tile: column n = t CIN + ci of
// part[co][NCOL] sums in[ci][p + tap t] dz[co][p] over the tile's pixels p, the
// last column dz[co][p].  Both operands in LDS; one wave per 32 columns (COUT =
// 32: 32x32x2 products) or 64 (COUT = 3: sixteen 4x4x1 blocks, 3 of 4 rows
// used).  Bound by the matrix cores (17 us at 224x448 with the last workgroups)
// after the tile's load.  224x448: 32 x 32 channels 120 -> 39 us, 4 x 32 73 ->
// 15, 32 x 3 31 -> 17, against a thread per (ci, tap) with vector multiply-adds
// (49, 23 and 24 with the tile's pixels taken one by one).
template <int CIN>
constexpr int kCols = CIN * 9 + 1;
template <int CIN, int COUT>
constexpr int kWgradThreads = COUT == 32 ? (CIN == 32 ? 640 : 256) : 320;
template <typename TIn, int CIN, int COUT>
__global__ __launch_bounds__((kWgradThreads<CIN, COUT>)) void k_wgrad(const TIn* __restrict__ in, int H, int W,
                                                                    const float* __restrict__ dz,
                                                                    float* __restrict__ part) {
  constexpr int T = kWgradThreads<CIN, COUT>, CS = kHalo * kHalo + 1, DS = kTile * kTile + 1;
  constexpr int NCOL = kCols<CIN>;
  __shared__ float sin[CIN * CS];
  __shared__ float sdz[COUT * DS];
  const int x0 = blockIdx.x * kTile, y0 = blockIdx.y * kTile;
  stage<TIn, CIN, CIN, kHalo, kHalo, CS, T / 64>(in, H, W, x0 - 1, y0 - 1, sin);
  stage<float, COUT, COUT, kTile, kTile, DS, T / 64>(dz, H, W, x0, y0, sdz);
  __syncthreads();
  float* pw = part + (size_t)(blockIdx.y * gridDim.x + blockIdx.x) * COUT * NCOL;
  constexpr int COLS = COUT == 32 ? 32 : 64;  // of a wave
  const int lane = threadIdx.x & 63, col0 = ((int)threadIdx.x >> 6) * COLS;
  const int col = col0 + lane % COLS;
  if (col0 >= NCOL) return;
  const int cc = min(col, NCOL - 2), t = cc / CIN;  // the bias column reads any operand
  const float* sb = sin + cc % CIN * CS + t / 3 * kHalo + t % 3;
  const bool one = col == NCOL - 1;
  if (COUT == 32) {
    const int h = lane >> 5;
    const float* sa = sdz + (lane & 31) * DS + h;
    f32x16 acc{};
    for (int py = 0; py < kTile; ++py)
#pragma unroll
      for (int j = 0; j < kTile / 2; ++j) {
        const float v = sb[py * kHalo + 2 * j + h];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(sa[py * kTile + 2 * j], one ? 1.f : v, acc, 0, 0, 0);
      }
    if (col < NCOL)
#pragma unroll
      for (int i = 0; i < 16; ++i) pw[(8 * (i / 4) + 4 * h + i % 4) * NCOL + col] = acc[i];
  } else {
    const float* sa = sdz + min(lane & 3, COUT - 1) * DS;
    f32x4 acc{};
    for (int py = 0; py < kTile; ++py)
#pragma unroll
      for (int j = 0; j < kTile; ++j) {
        const float v = sb[py * kHalo + j];
        acc = __builtin_amdgcn_mfma_f32_4x4x1f32(sa[py * kTile + j], one ? 1.f : v, acc, 0, 0, 0);
      }
    if (col < NCOL)
#pragma unroll
      for (int i = 0; i < COUT; ++i) pw[i * NCOL + col] = acc[i];
  }
}

// grads of a layer from its partials [row][co][t CIN + ci, bias]: the rows are
// added in order.  32 columns a workgroup; 16 half waves fetch 256 rows at a
// time into LDS, one adds them up.  Bound by the reads' latency (224x448: 392
// rows): 93 -> 6.7 us against one thread a column and its loads in series.
constexpr int kSumRows = 256;
__global__ __launch_bounds__(512) void k_sum_rows(const float* __restrict__ rows, int nrows, int Cin,
                                                  int Cout, float* __restrict__ out) {
  __shared__ float s[kSumRows][32];
  const int ncol = Cin * 9 + 1, n = Cout * ncol;
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5, k = blockIdx.x * 32 + c;
  const int kc = min(k, n - 1);
  float sum = 0.f;
  for (int r0 = 0; r0 < nrows; r0 += kSumRows) {
    const int m = min(kSumRows, nrows - r0);
    float v[kSumRows / 16];
#pragma unroll
    for (int i = 0; i < kSumRows / 16; ++i)
      v[i] = rows[(size_t)(r0 + min(g + 16 * i, m - 1)) * n + kc];
    if (r0) __syncthreads();
#pragma unroll
    for (int i = 0; i < kSumRows / 16; ++i) s[g + 16 * i][c] = v[i];
    __syncthreads();
    if (g == 0) {
#pragma unroll 16
      for (int i = 0; i < m; ++i) sum += s[i][c];
    }
  }
  if (g || k >= n) return;
  const int co = k / ncol, q = k % ncol;
  out[q == ncol - 1 ? Cout * Cin * 9 + co : (co * Cin + q % Cin) * 9 + q / Cin] = sum;
}

// loss = 0.5 / count * sum mask (out - target)^2 over C planes; d out
__global__ void k_loss_grad(const float* __restrict__ out, const float* __restrict__ target,
                            const float* __restrict__ mask, int C, size_t plane, float inv_count,
                            float* __restrict__ dout, double* __restrict__ partial) {
  __shared__ double red[256];
  double acc = 0.0;
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < C * plane;
       k += (size_t)gridDim.x * blockDim.x) {
    const float m = mask[k % plane];
    const float r = (out[k] - target[k]) * m;
    dout[k] = r * m * inv_count;
    acc += 0.5 * (double)r * (double)r;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0] * (double)inv_count;
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const float gk = g[k];
  const float mk = b1 * m[k] + (1.f - b1) * gk;
  const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
  m[k] = mk;
  v[k] = vk;
  p[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

constexpr int kLayers = 4;
constexpr int kCin[kLayers] = {4, 32, 32, 32};
constexpr int kCout[kLayers] = {32, 32, 32, 3};

}  // namespace

struct CnnState {
  int dev = 0;
  hipStream_t stream = nullptr;
  hipStream_t side = nullptr;    // uploads beside the forward pass
  hipEvent_t uploaded = nullptr;
  int H = 0, W = 0;
  std::vector<void*> allocs;
  size_t off[kLayers] = {};  // start of each layer's W in the flat vector
  int nparams = 0;
  float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;
  float *x0 = nullptr;        // network input [4][H][W]
  bf16_t *z[3] = {}, *a[3] = {};  // hidden pre-activations and activations
  float *out = nullptr, *target = nullptr, *mask = nullptr;
  float *d0 = nullptr, *d1 = nullptr;  // gradients w.r.t. z of the current / lower layer
  float* part = nullptr;      // per-tile weight-gradient partials
  double* lpart = nullptr;
  int lblocks = 512;
  long step = 0;

  ~CnnState() {
    if (stream) (void)hipSetDevice(dev);
    for (void* p : allocs) (void)hipFree(p);
    if (uploaded) (void)hipEventDestroy(uploaded);
    if (side) (void)hipStreamDestroy(side);
    if (stream) (void)hipStreamDestroy(stream);
  }
  template <typename T>
  Status alloc(T** p, size_t count) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, count * sizeof(T) + 4);
    if (e != hipSuccess) return Status::Err(FWIFLOW_ERR_MEMORY, "hipMalloc failed in the network");
    allocs.push_back(q);
    *p = (T*)q;
    return Status::Ok();
  }
  dim3 tiles() const { return dim3((W + kTile - 1) / kTile, (H + kTile - 1) / kTile); }
};

namespace {

template <typename TIn, int CIN, int C, int EPI>
void conv32(CnnState& s, const TIn* in, const float* w, const float* bias, float* out_f32, bf16_t* zb,
            bf16_t* ab, const bf16_t* zin) {
  hipLaunchKernelGGL((k_conv32<TIn, CIN, C, EPI>),
                     conv_grid(s.H, s.W), dim3(64 * kConvY), 0, s.stream, in, s.H, s.W, w, bias, out_f32, zb, ab, zin);
}

template <typename TIn, int CIN, int COUT>
void wgrad(CnnState& s, const TIn* in, const float* dz, float* gw) {
  const dim3 grid = s.tiles();
  hipLaunchKernelGGL((k_wgrad<TIn, CIN, COUT>), grid, dim3(kWgradThreads<CIN, COUT>), 0, s.stream, in,
                     s.H, s.W, dz, s.part);
  hipLaunchKernelGGL(k_sum_rows, dim3((COUT * kCols<CIN> + 31) / 32), dim3(512), 0, s.stream, s.part,
                     (int)(grid.x * grid.y), CIN, COUT, gw);
}

Status forward(CnnState& s) {
  auto W = [&](int l) { return s.params + s.off[l]; };
  auto B = [&](int l) { return W(l) + kCout[l] * kCin[l] * 9; };
  conv32<float, 4, 4, kHidden>(s, s.x0, W(0), B(0), nullptr, s.z[0], s.a[0], nullptr);
  for (int l = 1; l < 3; ++l)
    conv32<bf16_t, 32, 32, kHidden>(s, s.a[l - 1], W(l), B(l), nullptr, s.z[l], s.a[l], nullptr);
  hipLaunchKernelGGL(k_conv3, conv_grid(s.H, s.W), dim3(32 * kConvY), 0, s.stream,
                     s.a[2], s.H, s.W, W(3), B(3), s.out);
  CNN_HIP(hipGetLastError());
  return Status::Ok();
}

// loss and parameter gradients for the staged input / target / mask
Status backward(CnnState& s, const float* target, const float* mask, double* loss, float* grad) {
  const size_t plane = (size_t)s.H * s.W;
  // Target and mask go to the device beside the forward pass (every earlier use
  // of theirs was waited for), the mask's population for the mean is counted
  // here: a gradient at 224x448 takes 507 us with these uploads before the
  // forward pass, 475 so; in the same stream after it 533.  The second stream
  // adds 0.05 ms to the 2.1 ms of making a network.
  CNN_HIP(hipMemcpyAsync(s.target, target, 3 * plane * sizeof(float), hipMemcpyHostToDevice, s.side));
  CNN_HIP(hipMemcpyAsync(s.mask, mask, plane * sizeof(float), hipMemcpyHostToDevice, s.side));
  CNN_HIP(hipEventRecord(s.uploaded, s.side));
  CNN_HIP(hipStreamWaitEvent(s.stream, s.uploaded, 0));
  size_t cnt = 0;
  for (size_t k = 0; k < plane; ++k) cnt += mask[k] != 0.f;
  const float inv = cnt > 0 ? (float)(1.0 / ((double)cnt * kCout[3])) : 0.f;
  hipLaunchKernelGGL(k_loss_grad, dim3(s.lblocks), dim3(256), 0, s.stream, s.out, s.target,
                     s.mask, kCout[3], plane, inv, s.d0, s.lpart);
  // per layer: weight gradient from dz, then dz of the layer below
  auto W = [&](int l) { return s.params + s.off[l]; };
  auto G = [&](int l) { return s.grads + s.off[l]; };
  wgrad<bf16_t, 32, 3>(s, s.a[2], s.d0, G(3));
  conv32<float, 4, 3, kInputGrad>(s, s.d0, W(3), nullptr, s.d1, nullptr, nullptr, s.z[2]);
  wgrad<bf16_t, 32, 32>(s, s.a[1], s.d1, G(2));
  conv32<float, 32, 32, kInputGrad>(s, s.d1, W(2), nullptr, s.d0, nullptr, nullptr, s.z[1]);
  wgrad<bf16_t, 32, 32>(s, s.a[0], s.d0, G(1));
  conv32<float, 32, 32, kInputGrad>(s, s.d0, W(1), nullptr, s.d1, nullptr, nullptr, s.z[0]);
  wgrad<float, 4, 32>(s, s.x0, s.d1, G(0));
  CNN_HIP(hipGetLastError());
  std::vector<double> lp(s.lblocks);
  CNN_HIP(hipMemcpyAsync(lp.data(), s.lpart, lp.size() * sizeof(double), hipMemcpyDeviceToHost,
                         s.stream));
  if (grad)
    CNN_HIP(hipMemcpyAsync(grad, s.grads, s.nparams * sizeof(float), hipMemcpyDeviceToHost, s.stream));
  CNN_HIP(hipStreamSynchronize(s.stream));
  double L = 0;
  for (double v : lp) L += v;
  if (loss) *loss = L;
  return Status::Ok();
}

}  // namespace

Cnn::Cnn() = default;
Cnn::~Cnn() = default;

Status Cnn::create(int gpu, int height, int width, unsigned seed) {
  if (height < 1 || width < 1) return Status::Err(FWIFLOW_ERR_ARG, "network grid must be >= 1x1");
  int ndev = 0;
  CNN_HIP(hipGetDeviceCount(&ndev));
  if (gpu < 0 || gpu >= ndev) return Status::Err(FWIFLOW_ERR_HIP, "gpu_id not present");
  s_.reset(new CnnState());
  CnnState& s = *s_;
  s.dev = gpu;
  s.H = height;
  s.W = width;
  CNN_HIP(hipSetDevice(gpu));
  CNN_HIP(hipStreamCreate(&s.stream));
  CNN_HIP(hipStreamCreate(&s.side));
  CNN_HIP(hipEventCreateWithFlags(&s.uploaded, hipEventDisableTiming));
  size_t o = 0;
  for (int l = 0; l < kLayers; ++l) {
    s.off[l] = o;
    o += (size_t)kCout[l] * kCin[l] * 9 + kCout[l];
  }
  s.nparams = (int)o;
  // He-normal weights for the GELU layers, smaller for the linear output
  // layer, zero biases; deterministic in `seed`
  std::vector<float> h(o, 0.f);
  std::mt19937 rng(seed);
  for (int l = 0; l < kLayers; ++l) {
    const double fan_in = 9.0 * kCin[l];
    const double sd = (l < kLayers - 1 ? std::sqrt(2.0 / fan_in) : 0.1 * std::sqrt(1.0 / fan_in));
    std::normal_distribution<double> nd(0.0, sd);
    for (int k = 0; k < kCout[l] * kCin[l] * 9; ++k) h[s.off[l] + k] = (float)nd(rng);
  }
  const size_t plane = (size_t)height * width;
  const dim3 t = s.tiles();
  TRY(s.alloc(&s.params, o));
  TRY(s.alloc(&s.grads, o));
  TRY(s.alloc(&s.m1, o));
  TRY(s.alloc(&s.m2, o));
  TRY(s.alloc(&s.x0, 4 * plane));
  for (int l = 0; l < 3; ++l) {
    TRY(s.alloc(&s.z[l], (size_t)kMaxC * plane));
    TRY(s.alloc(&s.a[l], (size_t)kMaxC * plane));
  }
  TRY(s.alloc(&s.out, 3 * plane));
  TRY(s.alloc(&s.target, 3 * plane));
  TRY(s.alloc(&s.mask, plane));
  TRY(s.alloc(&s.d0, (size_t)kMaxC * plane));
  TRY(s.alloc(&s.d1, (size_t)kMaxC * plane));
  TRY(s.alloc(&s.part, (size_t)t.x * t.y * (kMaxC * kMaxC * 9 + kMaxC)));
  TRY(s.alloc(&s.lpart, (size_t)s.lblocks));
  CNN_HIP(hipMemcpy(s.params, h.data(), o * sizeof(float), hipMemcpyHostToDevice));
  CNN_HIP(hipMemset(s.m1, 0, o * sizeof(float)));
  CNN_HIP(hipMemset(s.m2, 0, o * sizeof(float)));
  return Status::Ok();
}

int Cnn::num_params() const { return s_ ? s_->nparams : 0; }

Status Cnn::get_params(float* out) const {
  if (!s_ || !out) return Status::Err(FWIFLOW_ERR_ARG, "null network or output");
  CNN_HIP(hipSetDevice(s_->dev));
  CNN_HIP(hipMemcpy(out, s_->params, s_->nparams * sizeof(float), hipMemcpyDeviceToHost));
  return Status::Ok();
}

Status Cnn::set_params(const float* in) {
  if (!s_ || !in) return Status::Err(FWIFLOW_ERR_ARG, "null network or input");
  CNN_HIP(hipSetDevice(s_->dev));
  CNN_HIP(hipMemcpy(s_->params, in, s_->nparams * sizeof(float), hipMemcpyHostToDevice));
  CNN_HIP(hipMemset(s_->m1, 0, s_->nparams * sizeof(float)));
  CNN_HIP(hipMemset(s_->m2, 0, s_->nparams * sizeof(float)));
  s_->step = 0;
  return Status::Ok();
}

Status Cnn::forward(const float* input, float* output) {
  if (!s_ || !input || !output) return Status::Err(FWIFLOW_ERR_ARG, "null network or buffer");
  CnnState& s = *s_;
  CNN_HIP(hipSetDevice(s.dev));
  CNN_HIP(hipMemcpyAsync(s.x0, input, 4 * (size_t)s.H * s.W * sizeof(float), hipMemcpyHostToDevice, s.stream));
  TRY(fwiflow::forward(s));
  CNN_HIP(hipMemcpyAsync(output, s.out, 3 * (size_t)s.H * s.W * sizeof(float),
                         hipMemcpyDeviceToHost, s.stream));
  CNN_HIP(hipStreamSynchronize(s.stream));
  return Status::Ok();
}

Status Cnn::gradients(const float* input, const float* target, const float* mask, double* loss,
                      float* grad) {
  if (!s_ || !input || !target || !mask)
    return Status::Err(FWIFLOW_ERR_ARG, "null network or buffer");
  CnnState& s = *s_;
  CNN_HIP(hipSetDevice(s.dev));
  CNN_HIP(hipMemcpyAsync(s.x0, input, 4 * (size_t)s.H * s.W * sizeof(float), hipMemcpyHostToDevice, s.stream));
  TRY(fwiflow::forward(s));
  return backward(s, target, mask, loss, grad);
}

Status Cnn::train_step(const float* input, const float* target, const float* mask, float lr,
                       double* loss) {
  TRY(gradients(input, target, mask, loss, nullptr));
  CnnState& s = *s_;
  s.step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)s.step), c2 = 1.f - std::pow(b2, (float)s.step);
  hipLaunchKernelGGL(k_adam, dim3((s.nparams + 255) / 256), dim3(256), 0, s.stream, s.params,
                     s.grads, s.m1, s.m2, s.nparams, lr, b1, b2, 1e-8f, c1, c2);
  CNN_HIP(hipGetLastError());
  CNN_HIP(hipStreamSynchronize(s.stream));
  return Status::Ok();
}

}  // namespace fwiflow
