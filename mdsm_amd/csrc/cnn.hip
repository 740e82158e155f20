// cnn.hip -- BF16 MFMA kernels of the event-triage CNN (forward, backward,
// optimiser).
//
// The 3x3 convolutions run as implicit products on v_mfma_f32_16x16x32_bf16
// and v_mfma_f32_16x16x16_bf16 with BF16 operands and FP32 accumulation, each
// fused with what follows or precedes it (forward with bias, ReLU and pool;
// the first layer's weight gradient with the pool's backward), reading NHWC
// activations without an im2col buffer.  The two linear layers run through
// one GEMM kernel, C[m][n] = sum_k A(m,k) B(k,n):
//
//   tile 64 (m) x 64 (n) x 32 (k), 256 threads = 4 waves in 2 x 2, each wave
//   a 32 x 32 block = 2 x 2 MFMA 16x16 tiles.  A is staged as As[m][k] and B
//   as Bt[n][k] in LDS (row pitch 36 halves: 8-byte aligned lane reads, no
//   bank conflicts between the 16-lane groups), so each lane's MFMA operand
//   is one 8-byte LDS read of 4 consecutive k.
//   MFMA 16x16x16 bf16 lane layout: A row = lane%16, k = 4*(lane/16)+j;
//   B column = lane%16, same k; D column = lane%16, rows 4*(lane/16)+j.
//   Split-K: grid.z slices the reduction; slices write FP32 partials that
//   epilogue_kernel sums in slice order (deterministic), adds the bias,
//   applies ReLU or a ReLU mask and stores FP32 and/or BF16.
//
// Element-wise kernels: backward of the pool with the bias gradients, softmax
// cross-entropy, Adam, NCHW -> NHWC input transpose, parameter layouts.  BF16 conversion is round-to-nearest-even.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cnn_internal.h"

namespace mdsm {
namespace cnn {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 64, BN = 64, BK = 32, PITCH = BK + 4, NT = 256;

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ------------------------------------------------------------ loaders
// Each loader fills 8 consecutive k of one operand row: fetchA(m, k, ...)
// gives A(m, k..k+7), fetchB(n, k, ...) gives B(k..k+7, n); k is a multiple
// of 8 and elements at or past kend are 0.  Index arithmetic is 32-bit
// (every operand here has fewer than 2^31 elements) and a run of 8 elements
// that is contiguous and 16-byte aligned in memory is one 16-byte load.
__device__ __forceinline__ bool aligned16(const uint16_t *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}
__device__ __forceinline__ void load8(const uint16_t *p, uint16_t v[8]) {
  const uint4 q = *reinterpret_cast<const uint4 *>(p);
  v[0] = (uint16_t)q.x; v[1] = (uint16_t)(q.x >> 16);
  v[2] = (uint16_t)q.y; v[3] = (uint16_t)(q.y >> 16);
  v[4] = (uint16_t)q.z; v[5] = (uint16_t)(q.z >> 16);
  v[6] = (uint16_t)q.w; v[7] = (uint16_t)(q.w >> 16);
}
__device__ __forceinline__ void zero8(uint16_t v[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0;
}

struct Dense {  // (r, c) at p[r*sr + c*sc]
  const uint16_t *p;
  int64_t sr, sc;
  __device__ __forceinline__ void fetchA(int64_t m, int64_t k, int64_t kend, uint16_t v[8]) const {
    const uint16_t *q = p + m * sr + k * sc;
    if (sc == 1 && k + 8 <= kend && aligned16(q)) {
      load8(q, v);
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = k + e < kend ? q[e * sc] : (uint16_t)0;
  }
  __device__ __forceinline__ void fetchB(int64_t n, int64_t k, int64_t kend, uint16_t v[8]) const {
    const uint16_t *q = p + k * sr + n * sc;
    if (sr == 1 && k + 8 <= kend && aligned16(q)) {
      load8(q, v);
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = k + e < kend ? q[e * sr] : (uint16_t)0;
  }
};

template <typename LA, typename LB>
__global__ __launch_bounds__(NT) void gemm_kernel(LA A, LB B, int64_t M, int64_t N, int64_t K,
                                                  int64_t kchunk, float *__restrict__ C,
                                                  int64_t ldc) {
  __shared__ __align__(16) uint16_t As[BM * PITCH];
  __shared__ __align__(16) uint16_t Bt[BN * PITCH];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.x * BM, n0 = (int64_t)blockIdx.y * BN;
  const int64_t kbeg = (int64_t)blockIdx.z * kchunk;
  const int64_t kend = kbeg + kchunk < K ? kbeg + kchunk : K;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lr = t >> 2, lk = (t & 3) * 8;  // loader: row (m or n) and first k of 8
  for (int64_t k0 = kbeg; k0 < kend; k0 += BK) {
    {
      const int64_t m = m0 + lr;
      uint16_t v[8];
      if (m < M) A.fetchA(m, k0 + lk, kend, v);
      else zero8(v);
      uint16_t *dst = As + lr * PITCH + lk;
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[e] = v[e];
    }
    {
      const int64_t n = n0 + lr;
      uint16_t v[8];
      if (n < N) B.fetchB(n, k0 + lk, kend, v);
      else zero8(v);
      uint16_t *dst = Bt + lr * PITCH + lk;
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[e] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < BK; ks += 16) {
      bf16x4 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x4 *>(As + (wm * 32 + i * 16 + (lane & 15)) * PITCH + ks +
                                                 4 * (lane >> 4));
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = *reinterpret_cast<const bf16x4 *>(Bt + (wn * 32 + j * 16 + (lane & 15)) * PITCH + ks +
                                                 4 * (lane >> 4));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  float *Cz = C + (int64_t)blockIdx.z * M * ldc;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + wm * 32 + i * 16 + 4 * (lane >> 4) + r;
        const int64_t n = n0 + wn * 32 + j * 16 + (lane & 15);
        if (m < M && n < N) Cz[m * ldc + n] = acc[i][j][r];
      }
}

// sum of split partials [splits][M][N] + bias[n]; out_f32 = value; then
// mask (mask[m*N+n] > 0) and/or ReLU; out_bf16 = value
__global__ void epilogue_kernel(const float *__restrict__ part, int splits, int64_t M, int64_t N,
                                const float *__restrict__ bias, float *__restrict__ out_f32,
                                const float *__restrict__ mask, int relu,
                                uint16_t *__restrict__ out_bf16) {
  const int64_t MN = M * N;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < MN;
       i += (int64_t)gridDim.x * blockDim.x) {
    // slices in order, 16 loads ahead of their adds (one at a time, 128
    // slices of 16384 values took 31 us; 9 us so)
    float v = part[i];
    int z = 1;
    for (; z + 16 <= splits; z += 16) {
      float t[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) t[u] = part[(int64_t)(z + u) * MN + i];
#pragma unroll
      for (int u = 0; u < 16; ++u) v += t[u];
    }
    for (; z < splits; ++z) v += part[(int64_t)z * MN + i];
    if (bias) v += bias[i % N];
    if (out_f32) out_f32[i] = v;
    if (mask && !(mask[i] > 0.f)) v = 0.f;
    if (relu) v = v > 0.f ? v : 0.f;
    if (out_bf16) out_bf16[i] = to_bf16(v);
  }
}

// ------------------------------------------------------------ convolutions
// Walks NHWC pixels: (b, h, w) of a linear index, stepped without division.
struct Pixel {
  int w, h;
  int64_t b;
  __device__ __forceinline__ void set(int64_t i, int H, int W) {
    const int64_t bh = i / W;
    w = (int)(i - bh * W);
    b = bh / H;
    h = (int)(bh - b * H);
  }
  __device__ __forceinline__ void advance(int n, int H, int W) {
    for (w += n; w >= W; w -= W)
      if (++h == H) {
        h = 0;
        ++b;
      }
  }
};

// Four pixels of one channel per lane from pixel-major LDS rows: in each group
// of 16 lanes, lane j names 4 channels (j % 4) of pixel j / 4 and lane n gets
// channel n of the four pixels.
__device__ __forceinline__ bf16x4 load_transposed(const uint16_t *p) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4 *)p);
}
__device__ __forceinline__ uint4 load8(const uint16_t *p) { return *reinterpret_cast<const uint4 *>(p); }
__device__ __forceinline__ f32x4 mfma32(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 3x3 convolution (pad 1) + bias + ReLU + 2x2 max pool in one pass, NHWC BF16
// in and out, FP32 accumulation over k = (ky*3 + kx)*CI + ci in order, on
// v_mfma_f32_16x16x32_bf16 (CI = 2, k to 18: v_mfma_f32_16x16x16_bf16).
//   A (16 x 16): rows are 4 pooled pixels x the 4 positions of their window,
//   so a lane's four results of one output channel (D rows 4*(lane/16)+r) are
//   one pool window and bias, ReLU and maximum need no exchange; a lane's
//   operand is one 16-byte load of 8 channels (two 4-byte loads for CI = 2),
//   straight from the activations (each is read 9 times, from L1/L2).
//   B: the layer's weights, held in registers for the wave's whole run of
//   tiles; NB output-channel tiles per wave.
// a[pooled][CO] = BF16 of the maximum, idx = argmax (0..3, first maximum) | 4
// when the maximum is positive.  Storing the FP32 pre-activations and pooling
// them in a second pass moved 8 bytes per pixel and channel: 256 snippets of
// 64 x 256, three layers: 320 + 117 + 57 us, now 46 + 33 + 29 (45 and 41 with
// 16-deep steps and 8-byte loads).  Bound by the activation loads (9 per
// element, L1 and L2).
template <int CI, int CO, int NB>
__global__ __launch_bounds__(NT) void conv_pool_kernel(const uint16_t *__restrict__ x,
                                                       const uint16_t *__restrict__ wt,
                                                       const float *__restrict__ bias, int64_t P, int H,
                                                       int W, int run, uint16_t *__restrict__ a,
                                                       uint8_t *__restrict__ idx) {
  constexpr int DEPTH = CI == 2 ? 16 : 32;             // k values per step, DEPTH / 4 per lane
  constexpr int KC = (9 * CI + DEPTH - 1) / DEPTH;
  using Operand = std::conditional_t<CI == 2, bf16x4, uint4>;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int Ho = H / 2, Wo = W / 2;
  const int n0 = blockIdx.y * NB * 16;
  Operand bw[KC][NB];
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int k = DEPTH * c + DEPTH / 4 * g;
      const uint16_t *q = wt + (int64_t)(n0 + 16 * j + n) * (9 * CI) + k;
      if constexpr (CI == 2) {  // rows of 18, 4-byte aligned
        const uint32_t lo = k < 18 ? *reinterpret_cast<const uint32_t *>(q) : 0u;
        const uint32_t hi = k + 2 < 18 ? *reinterpret_cast<const uint32_t *>(q + 2) : 0u;
        bw[c][j] = __builtin_bit_cast(bf16x4, ((uint64_t)hi << 32) | lo);
      } else {
        bw[c][j] = k < 9 * CI ? load8(q) : make_uint4(0u, 0u, 0u, 0u);
      }
    }
  // CI = 16: a step holds two taps, the lanes of g < 2 the first; this lane's
  // tap of each step (9 past the last: outside everywhere)
  int dy[KC], dx[KC];
  if constexpr (CI != 2) {
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int t = CI == 16 ? 2 * c + (g >> 1) : c * 32 / CI;
      dy[c] = t < 9 ? t / 3 - 1 : H;
      dx[c] = t % 3 - 1;
    }
  }
  float bs[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) bs[j] = bias[n0 + 16 * j + n];
  const int64_t wave = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  int64_t p = wave * run * 4;  // first pooled pixel of the wave's run
  const int64_t pend = p + (int64_t)run * 4 < P ? p + (int64_t)run * 4 : P;
  if (p >= pend) return;
  // this lane's A row: pooled pixel p + n/4, window position n%4
  Pixel px;
  px.set(p + (n >> 2) < P ? p + (n >> 2) : P - 1, Ho, Wo);
  for (; p < pend; p += 4) {
    const int h = 2 * px.h + ((n >> 1) & 1), w = 2 * px.w + (n & 1);
    const uint16_t *q = x + ((px.b * H + h) * W + w) * CI;
    f32x4 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (CI == 2) {
      // step 0: taps 2g and 2g + 1; step 1: tap 8 (g = 0), zeros
      uint32_t v[2];
      const int ty = (2 * g) / 3, tx = 2 * g - 3 * ty, uy = (2 * g + 1) / 3, ux = 2 * g + 1 - 3 * uy;
      const int dy[2] = {ty - 1, uy - 1}, dx[2] = {tx - 1, ux - 1};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int hh = h + dy[e], ww = w + dx[e];
        const bool ok = hh >= 0 && hh < H && ww >= 0 && ww < W;
        const uint32_t u = *reinterpret_cast<const uint32_t *>(q + (ok ? (dy[e] * W + dx[e]) * 2 : 0));
        v[e] = ok ? u : 0u;
      }
      const bool ok8 = g == 0 && h < H - 1 && w < W - 1;
      const uint32_t u8 = *reinterpret_cast<const uint32_t *>(q + (ok8 ? (W + 1) * 2 : 0));
      const bf16x4 a0 = __builtin_bit_cast(bf16x4, ((uint64_t)v[1] << 32) | v[0]);
      const bf16x4 a1 = __builtin_bit_cast(bf16x4, (uint64_t)(ok8 ? u8 : 0u));
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0, bw[0][j], acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, bw[1][j], acc[j], 0, 0, 0);
      }
    } else {
      uint4 av[KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const int hh = h + dy[c], ww = w + dx[c];
        const bool ok = (unsigned)hh < (unsigned)H && (unsigned)ww < (unsigned)W;
        av[c] = load8(q + (ok ? (dy[c] * W + dx[c]) * CI : 0) + (8 * g) % CI);
        if (!ok) av[c] = make_uint4(0u, 0u, 0u, 0u);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j] = mfma32(av[c], bw[c][j], acc[j]);
    }
    if (p + g < P) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        float best = -1.f;
        int arg = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float v = acc[j][k] + bs[j];
          v = v > 0.f ? v : 0.f;
          if (v > best) {
            best = v;
            arg = k;
          }
        }
        const int64_t o = (p + g) * CO + n0 + 16 * j + n;
        a[o] = to_bf16(best);
        idx[o] = (uint8_t)(arg | (best > 0.f ? 4 : 0));
      }
    }
    px.advance(4, Ho, Wo);
    if (p + 4 + (n >> 2) >= P) px.set(P - 1, Ho, Wo);  // rows past the end repeat the last pixel
  }
}

// Input gradient of a 3x3 convolution: dx[pix][ci] = sum over
// k = (ky*3 + kx)*CO + co, in order, of dz[pix moved back by the tap][co] *
// w[co][tap][ci], FP32.  As the forward kernel, with 16 consecutive pixels as
// rows; wf: the weights as [ci][(ky*3 + kx)*CO + co] (weights_flip_kernel).
// Bound by its gradient loads; every input-channel tile in one wave reads
// them once.  256 snippets: 64 -> 32 channels 43 us (98 with 8-byte loads and
// the weights in 144 registers of every wave instead of 36 KB of LDS), 32 -> 16
// 48 us (78 with 8-byte loads, 148 as an im2col product).
template <int CO, int CI, int NB>
__global__ __launch_bounds__(NT) void conv_dx_kernel(const uint16_t *__restrict__ dz,
                                                     const uint16_t *__restrict__ wf, int64_t P, int H,
                                                     int W, int run, float *__restrict__ dx) {
  constexpr int KC = 9 * CO / 32;
  constexpr bool LW = KC * NB > 18;  // weights in LDS
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.y * NB * 16;
  __shared__ uint4 ws[LW ? KC * NB * 64 : 1];
  uint4 bw[LW ? 1 : KC][NB];
  auto weight = [&](int c, int j) { return load8(wf + (int64_t)(n0 + 16 * j + n) * (9 * CO) + 32 * c + 8 * g); };
  if constexpr (LW) {
    for (int i = threadIdx.x >> 6; i < KC * NB; i += NT / 64) ws[i * 64 + lane] = weight(i / NB, i % NB);
    __syncthreads();
  } else {
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int j = 0; j < NB; ++j) bw[c][j] = weight(c, j);
  }
  const int64_t wave = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  int64_t p = wave * run * 16;
  const int64_t pend = p + (int64_t)run * 16 < P ? p + (int64_t)run * 16 : P;
  if (p >= pend) return;
  Pixel px;
  px.set(p + n < P ? p + n : P - 1, H, W);
  for (; p < pend; p += 16) {
    const uint16_t *q = dz + ((px.b * H + px.h) * W + px.w) * CO;
    f32x4 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 av[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int t = c / (CO / 32), cc = c % (CO / 32);
      const int ky = t / 3, kx = t - 3 * ky;  // reads (h - ky + 1, w - kx + 1)
      const bool ok = (ky != 2 || px.h > 0) && (ky != 0 || px.h < H - 1) && (kx != 2 || px.w > 0) &&
                      (kx != 0 || px.w < W - 1);
      av[c] = load8(q + (ok ? ((1 - ky) * W + (1 - kx)) * CO : 0) + 32 * cc + 8 * g);
      if (!ok) av[c] = make_uint4(0u, 0u, 0u, 0u);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j] = mfma32(av[c], LW ? ws[(c * NB + j) * 64 + lane] : bw[LW ? 0 : c][j], acc[j]);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t o = p + 4 * g + r;
        if (o < P) dx[o * CI + n0 + 16 * j + n] = acc[j][r];
      }
    px.advance(16, H, W);
    if (p + 16 + n >= P) px.set(P - 1, H, W);
  }
}

// w[co][tap*CI + ci] -> wf[ci][tap*CO + co]
__global__ void weights_flip_kernel(const uint16_t *__restrict__ w, int CI, int CO, uint16_t *__restrict__ wf) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 9 * CI * CO) return;
  const int ci = i / (9 * CO), r = i - ci * 9 * CO, t = r / CO, co = r - t * CO;
  wf[i] = w[co * 9 * CI + t * CI + ci];
}

// Weight gradient of a 3x3 convolution, dw[co][tap*CI + ci] = sum over pixels
// of dz[pix][co] * x[pix moved by the tap][ci]: a product with the pixels as
// the reduction, so both operands need 4 consecutive pixels of one channel
// per lane while the activations are stored channel by channel of a pixel.
// A workgroup stages WR rows x WC columns of dz and of x (with a border) in
// LDS and its lanes read them transposed (ds_read_b64_tr_b16).  The pixel pitch
// is 8 bytes more than the channels take, which spreads a group's four pixels
// over the banks.  A wave owns CT output-channel tiles x 9*CI/16
// column tiles (72 accumulator registers); with CO > 16 CT the waves split the
// output channels, and otherwise the workgroup's pixels (their sums are added
// in LDS).  Each workgroup writes one partial; sum_rows_kernel adds them.
// An item's loads are in registers while the products of the one before run.
// 256 snippets: 35 + 5 us (32 channels) and 30 + 13 us (64); 73 and 46 with the
// loads between the barriers and 2-byte LDS reads (transposed reads alone: 70
// and 42), 377 and 187 as split im2col products.
constexpr int WR = 2, WC = 64;
template <int CI, int CO, int CT>
__global__ __launch_bounds__(NT) void conv_dw_kernel(const uint16_t *__restrict__ dz,
                                                     const uint16_t *__restrict__ x, int64_t B, int H,
                                                     int W, float *__restrict__ part) {
  constexpr int PZ = CO + 4, PX = CI + 4;      // pixel pitch (elements)
  constexpr int NTILE = 9 * CI / 16, CS = CO / (16 * CT);  // column tiles; waves over co
  constexpr int KS = (NT / 64) / CS;           // waves over pixels
  constexpr int XW = WC + 2;
  __shared__ __align__(16) uint16_t sz[WR * WC * PZ];
  __shared__ __align__(16) uint16_t sx[(WR + 2) * XW * PX];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  const int ws = wave % CS, kw = wave / CS;
  f32x4 acc[CT][NTILE];
#pragma unroll
  for (int i = 0; i < CT; ++i)
#pragma unroll
    for (int j = 0; j < NTILE; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nh = (H + WR - 1) / WR, nw = (W + WC - 1) / WC;
  const int64_t items = B * nh * nw;
  constexpr int NZ = WR * WC * (CO / 4), NX = (WR + 2) * XW * (CI / 4);  // 8-byte pieces of an item
  constexpr int RZ = (NZ + NT - 1) / NT, RX = (NX + NT - 1) / NT;
  uint2 vz[RZ], vx[RX];
  auto fetch = [&](int64_t it) {
    const int iw = (int)(it % nw);
    const int64_t r0 = it / nw;
    const int h0 = (int)(r0 % nh) * WR, w0 = iw * WC;
    const int64_t b = r0 / nh;
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
      const int i = threadIdx.x + r * NT, c = i % (CO / 4), q = i / (CO / 4), hs = h0 + q / WC, wsrc = w0 + q % WC;
      vz[r] = make_uint2(0u, 0u);
      if (i < NZ && hs < H && wsrc < W)
        vz[r] = *reinterpret_cast<const uint2 *>(dz + ((b * H + hs) * W + wsrc) * CO + 4 * c);
    }
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      const int i = threadIdx.x + r * NT, c = i % (CI / 4), q = i / (CI / 4);
      const int hs = h0 + q / XW - 1, wsrc = w0 + q % XW - 1;
      vx[r] = make_uint2(0u, 0u);
      if (i < NX && hs >= 0 && hs < H && wsrc >= 0 && wsrc < W)
        vx[r] = *reinterpret_cast<const uint2 *>(x + ((b * H + hs) * W + wsrc) * CI + 4 * c);
    }
  };
  if (blockIdx.x < items) fetch(blockIdx.x);
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
      const int i = threadIdx.x + r * NT, c = i % (CO / 4), q = i / (CO / 4);
      if (i < NZ) *reinterpret_cast<uint2 *>(sz + q * PZ + 4 * c) = vz[r];
    }
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      const int i = threadIdx.x + r * NT, c = i % (CI / 4), q = i / (CI / 4);
      if (i < NX) *reinterpret_cast<uint2 *>(sx + q * PX + 4 * c) = vx[r];
    }
    __syncthreads();
    if (it + gridDim.x < items) fetch(it + gridDim.x);  // under this item's products
    for (int ks = kw; ks < WR * WC / 16; ks += KS) {
      const int hh = ks / (WC / 16), wb = (ks % (WC / 16)) * 16 + 4 * g;  // this lane's first pixel
      bf16x4 av[CT];
#pragma unroll
      for (int i = 0; i < CT; ++i) {
        av[i] = load_transposed(sz + (hh * WC + wb + n / 4) * PZ + (ws * CT + i) * 16 + 4 * (n & 3));
      }
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
#pragma unroll
        for (int cc = 0; cc < CI / 16; ++cc) {
          const uint16_t *q = sx + ((hh + ky) * XW + wb + n / 4) * PX + 16 * cc + 4 * (n & 3);
#pragma unroll
          for (int kx = 0; kx < 3; ++kx) {
            const bf16x4 bv = load_transposed(q + kx * PX);
            const int j = (ky * 3 + kx) * (CI / 16) + cc;
#pragma unroll
            for (int i = 0; i < CT; ++i)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[i], bv, acc[i][j], 0, 0, 0);
          }
        }
    }
  }
  // D: column n = (tap, ci) of tile j, rows 4g + r = co of tile i
  float *o = part + (int64_t)blockIdx.x * (CO * 9 * CI);
  auto at = [&](int i, int j, int r) { return ((ws * CT + i) * 16 + 4 * g + r) * 9 * CI + 16 * j + n; };
  if constexpr (KS == 1) {
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
      for (int j = 0; j < NTILE; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[at(i, j, r)] = acc[i][j][r];
  } else {
    __shared__ float sum[KS == 1 ? 1 : CO * 9 * CI];
    for (int w = 0; w < KS; ++w) {
      __syncthreads();
      if (kw == w) {
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
          for (int j = 0; j < NTILE; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float *q = sum + at(i, j, r);
              *q = w ? *q + acc[i][j][r] : acc[i][j][r];
            }
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < CO * 9 * CI; i += NT) o[i] = sum[i];
  }
}

// First layer (2 input channels, no input gradient): weight and bias gradients
// straight from the pooled gradient.  Only the argmax pixel of a pool window
// has a gradient, so each (pooled pixel, output channel) is 18 multiply-adds
// with the 3x3 neighbourhood of that pixel, and neither the full-resolution
// gradient (134 MB for 256 snippets) nor a product over all pixels is formed.
// Thread t: channel t % 16, every 16th pooled pixel of a row chunk whose
// input pixels (both channels in one word) are staged with a border in LDS.
// Products of BF16 values, FP32 sums; part[block][288 weights, 16 biases].
// A chunk's loads are in registers while the sums of the one before run.  256
// snippets: 40 us (75 with the loads between the barriers and one pooled pixel
// at a time), against 670 for the pool's backward, its column sums and the
// product over all pixels.
constexpr int W1C = 128;  // pooled columns per chunk
__global__ __launch_bounds__(NT) void conv1_dw_kernel(const float *__restrict__ da,
                                                      const uint8_t *__restrict__ idx,
                                                      const uint32_t *__restrict__ x, int64_t B, int H,
                                                      int W, float *__restrict__ part) {
  constexpr int XW = 2 * W1C + 2;
  __shared__ uint32_t sx[4 * XW];
  __shared__ float red[4][16][19];
  const int co = threadIdx.x & 15, slot = threadIdx.x >> 4;
  const int Ho = H / 2, Wo = W / 2, nc = (Wo + W1C - 1) / W1C;
  float acc[18], bsum = 0.f;
#pragma unroll
  for (int k = 0; k < 18; ++k) acc[k] = 0.f;
  const int64_t items = B * Ho * nc;
  constexpr int RC = W1C / 16, RX = (4 * XW + NT - 1) / NT;
  uint8_t vq[RC];
  float vd[RC];
  uint32_t vx[RX];
  auto fetch = [&](int64_t it) {
    const int ic = (int)(it % nc);
    const int64_t bh = it / nc, b = bh / Ho;  // bh = b * Ho + ho
    const int ho = (int)(bh % Ho), c0 = ic * W1C;
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      const int i = threadIdx.x + r * NT, hh = i / XW;
      const int h = 2 * ho - 1 + hh, w = 2 * c0 - 1 + (i - hh * XW);
      vx[r] = (hh < 4 && h >= 0 && h < H && w >= 0 && w < W) ? x[(b * H + h) * W + w] : 0u;
    }
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const int c = c0 + slot + 16 * r;
      const int64_t o = (bh * Wo + (c < Wo ? c : Wo - 1)) * 16 + co;
      vq[r] = idx[o];
      vd[r] = da[o];
    }
  };
  if (blockIdx.x < items) fetch(blockIdx.x);
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    const int c0 = (int)(it % nc) * W1C, cols = Wo - c0 < W1C ? Wo - c0 : W1C;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      const int i = threadIdx.x + r * NT;
      if (i < 4 * XW) sx[i] = vx[r];
    }
    uint8_t cq[RC];
    float cd[RC];
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      cq[r] = vq[r];
      cd[r] = vd[r];
    }
    __syncthreads();
    if (it + gridDim.x < items) fetch(it + gridDim.x);  // under this item's sums
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const int c = slot + 16 * r;
      if (c >= cols) break;
      const uint8_t q = cq[r];
      const float gr = (q & 4) ? from_bf16(to_bf16(cd[r])) : 0.f;
      const uint32_t *s = sx + ((q >> 1) & 1) * XW + 2 * c + (q & 1);
      bsum += gr;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const uint32_t v = s[(t / 3) * XW + t % 3];
        acc[2 * t] = __builtin_fmaf(gr, __uint_as_float(v << 16), acc[2 * t]);
        acc[2 * t + 1] = __builtin_fmaf(gr, __uint_as_float(v & 0xFFFF0000u), acc[2 * t + 1]);
      }
    }
  }
  // lanes 16 and 32 apart hold the same channel, then the four waves
#pragma unroll
  for (int k = 0; k < 19; ++k) {
    float v = k < 18 ? acc[k] : bsum;
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if ((threadIdx.x & 63) < 16) red[threadIdx.x >> 6][co][k] = v;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * 19; i += NT) {
    const int c = i / 19, k = i - c * 19;
    const float v = (red[0][c][k] + red[1][c][k]) + (red[2][c][k] + red[3][c][k]);
    part[(int64_t)blockIdx.x * 304 + (k < 18 ? c * 18 + k : 288 + c)] = v;
  }
}

// Backward of ReLU + pool with the bias gradient: da[B][H/2][W/2][C] (FP32)
// -> dz[B][H][W][C] (BF16, the gradient at the argmax when it was positive,
// zeros elsewhere) and per-workgroup sums of the BF16 gradients per channel.
// A thread takes 8 channels of a pooled pixel (16-byte stores).
template <int C>
__global__ __launch_bounds__(NT) void pool_bwd_kernel(const float *__restrict__ da,
                                                      const uint8_t *__restrict__ idx, int64_t P, int H,
                                                      int W, uint16_t *__restrict__ dz,
                                                      float *__restrict__ part) {
  constexpr int G = C / 8;  // channel groups
  __shared__ float s[NT * 8];
  const int Ho = H / 2, Wo = W / 2;
  const int cg = threadIdx.x % G;
  float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int64_t p = (int64_t)blockIdx.x * (NT / G) + threadIdx.x / G; p < P;
       p += (int64_t)gridDim.x * (NT / G)) {
    const float4 v0 = *reinterpret_cast<const float4 *>(da + p * C + 8 * cg);
    const float4 v1 = *reinterpret_cast<const float4 *>(da + p * C + 8 * cg + 4);
    const uint2 qq = *reinterpret_cast<const uint2 *>(idx + p * C + 8 * cg);
    const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    uint32_t gr[8], q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[e] = ((e < 4 ? qq.x : qq.y) >> (8 * (e & 3))) & 7u;
      gr[e] = (q[e] & 4u) ? (uint32_t)to_bf16(v[e]) : 0u;
      sum[e] += from_bf16((uint16_t)gr[e]);
    }
    const int64_t bh = p / Wo;
    const int wo = (int)(p - bh * Wo);
    const int64_t b = bh / Ho;
    const int ho = (int)(bh - b * Ho);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = ((q[2 * e] & 3u) == k ? gr[2 * e] : 0u) | ((q[2 * e + 1] & 3u) == k ? gr[2 * e + 1] << 16 : 0u);
      *reinterpret_cast<uint4 *>(dz + ((b * H + 2 * ho + (k >> 1)) * W + 2 * wo + (k & 1)) * C + 8 * cg) =
          make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s[(threadIdx.x / G) * C + 8 * cg + e] = sum[e];
  __syncthreads();
  for (int c = threadIdx.x; c < C; c += NT) {
    float v = 0.f;
    for (int r = 0; r < NT / G; ++r) v += s[r * C + c];
    part[(int64_t)blockIdx.x * C + c] = v;
  }
}

// out[j] = sum over rows of part[row][j]: 16 columns per workgroup, 16 rows at
// a time, 8 loads in flight per thread
__global__ __launch_bounds__(NT) void sum_rows_kernel(const float *__restrict__ part, int rows, int n,
                                                      float *__restrict__ out) {
  __shared__ float s[16][17];
  const int c = threadIdx.x & 15, r0 = threadIdx.x >> 4;
  const int j = blockIdx.x * 16 + c;
  float v = 0.f;
  if (j < n) {
    int r = r0;
    for (; r + 7 * 16 < rows; r += 8 * 16) {
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = part[(int64_t)(r + 16 * u) * n + j];
#pragma unroll
      for (int u = 0; u < 8; ++u) v += t[u];
    }
    for (; r < rows; r += 16) v += part[(int64_t)r * n + j];
  }
  s[r0][c] = v;
  __syncthreads();
  if (r0 == 0 && j < n) {
    float t = 0.f;
    for (int r = 0; r < 16; ++r) t += s[r][c];
    out[j] = t;
  }
}

// column sums of a BF16 matrix x[rows][C] (C <= 256): per-block partials
__global__ void colsum_kernel(const uint16_t *__restrict__ x, int64_t rows, int C,
                              int64_t rows_per_block, float *__restrict__ part) {
  __shared__ float s[NT];
  const int groups = NT / C;  // thread (g, c): rows g, g + groups, ...
  const int g = threadIdx.x / C, c = threadIdx.x - g * C;
  float acc = 0.f;
  if (g < groups) {
    const int64_t r0 = blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;
    for (int64_t r = r0 + g; r < r1; r += groups) acc += from_bf16(x[r * C + c]);
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x < C) {
    float v = 0.f;
    for (int k = 0; k < groups; ++k) v += s[k * C + threadIdx.x];
    part[(int64_t)blockIdx.x * C + threadIdx.x] = v;
  }
}

// one workgroup per channel: thread t sums parts t, t + NT, ... in order,
// then a fixed binary tree (deterministic for a given nparts)
__global__ __launch_bounds__(NT) void sum_parts_kernel(const float *__restrict__ part, int nparts,
                                                       int C, float *__restrict__ out) {
  __shared__ float s[NT];
  const int c = blockIdx.x;
  float v = 0.f;
  for (int p = threadIdx.x; p < nparts; p += NT) v += part[(int64_t)p * C + c];
  s[threadIdx.x] = v;
  __syncthreads();
#pragma unroll
  for (int h = NT / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = s[0];
}

// mean softmax cross-entropy over B rows of 2 logits; dl = (p - onehot)/B (BF16)
__global__ void softmax_ce_kernel(const float *__restrict__ logits, const int32_t *__restrict__ y,
                                  int B, uint16_t *__restrict__ dl, float *__restrict__ loss) {
  __shared__ float s[NT];
  float acc = 0.f;
  for (int b = threadIdx.x; b < B; b += NT) {
    const float l0 = logits[2 * b], l1 = logits[2 * b + 1];
    const float m = fmaxf(l0, l1);
    const float e0 = expf(l0 - m), e1 = expf(l1 - m), sum = e0 + e1;
    const int lab = y[b] != 0;
    acc += -((lab ? l1 : l0) - m - logf(sum));
    dl[2 * b] = to_bf16((e0 / sum - (lab == 0 ? 1.f : 0.f)) / (float)B);
    dl[2 * b + 1] = to_bf16((e1 / sum - (lab == 1 ? 1.f : 0.f)) / (float)B);
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = NT / 2; w >= 1; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = s[0] / (float)B;
}

__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, uint16_t *__restrict__ pb, int64_t n, float lr,
                            float b1, float b2, float eps, float c1, float c2, float wd) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i] + wd * p[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    pb[i] = to_bf16(pi);
  }
}

__global__ void to_bf16_kernel(const float *__restrict__ x, uint16_t *__restrict__ y, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = to_bf16(x[i]);
}

// x[B][2][HW] -> y[B][HW][2], four pixels per thread (HW is a multiple of 64)
__global__ void nchw2_to_nhwc_kernel(const uint16_t *__restrict__ x, int64_t n4, int64_t HW4,
                                     uint16_t *__restrict__ y) {
  typedef uint16_t u16x4 __attribute__((ext_vector_type(4), aligned(2)));
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / HW4, r = i - b * HW4;
    const uint16_t *p = x + (b * 2 * HW4 + r) * 4;
    const u16x4 u = *reinterpret_cast<const u16x4 *>(p), v = *reinterpret_cast<const u16x4 *>(p + HW4 * 4);
    reinterpret_cast<uint4 *>(y)[i] =
        make_uint4(u[0] | (uint32_t)v[0] << 16, u[1] | (uint32_t)v[1] << 16, u[2] | (uint32_t)v[2] << 16,
                   u[3] | (uint32_t)v[3] << 16);
  }
}

// Parameters or gradients from the device layout to the canonical one: conv
// weights [co][ci][tap] from [co][tap][ci] and fc1 columns [c][y][x] from
// [y][x][c].  Segments: L.w[k] and L.fw1 as offsets, everything else in place.
__global__ void canonical_kernel(const float *__restrict__ src, CanonicalLayout L, float *__restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < L.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    int64_t j = i;
    for (int k = 0; k < 3; ++k) {
      const int64_t r = i - L.w[k];
      if (r >= 0 && r < (int64_t)9 * L.ci[k] * L.co[k]) {
        const int t = (int)(r % 9), ci = (int)(r / 9 % L.ci[k]);
        j = L.w[k] + r / (9 * L.ci[k]) * 9 * L.ci[k] + t * L.ci[k] + ci;
      }
    }
    const int64_t r = i - L.fw1;
    if (r >= 0 && r < (int64_t)L.fin * L.hid) {
      const int64_t o = r / L.fin, e = r - o * L.fin;
      j = L.fw1 + o * L.fin + e % L.pix * L.chan + e / L.pix;
    }
    out[i] = src[j];
  }
}

inline unsigned grid1d(int64_t n) {
  const int64_t g = (n + NT - 1) / NT;
  return (unsigned)(g < 65536 ? (g > 0 ? g : 1) : 65536);
}

inline int64_t kchunk_of(int64_t K, int splits) {
  return ((K + splits - 1) / splits + BK - 1) / BK * BK;
}

template <typename LA, typename LB>
int gemm(LA A, LB B, int64_t M, int64_t N, int64_t K, int splits, float *C, hipStream_t s) {
  const int64_t kchunk = kchunk_of(K, splits);
  const int z = (int)((K + kchunk - 1) / kchunk);
  const dim3 grid((unsigned)((M + BM - 1) / BM), (unsigned)((N + BN - 1) / BN), (unsigned)z);
  hipLaunchKernelGGL((gemm_kernel<LA, LB>), grid, dim3(NT), 0, s, A, B, M, N, K, kchunk, C, N);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

}  // namespace

int splits_used(int64_t K, int splits) {
  const int64_t kchunk = kchunk_of(K, splits);
  return (int)((K + kchunk - 1) / kchunk);
}

int gemm_dense(const uint16_t *a, int64_t asr, int64_t asc, const uint16_t *b, int64_t bsr,
               int64_t bsc, int64_t M, int64_t N, int64_t K, int splits, float *C, hipStream_t s) {
  return gemm(Dense{a, asr, asc}, Dense{b, bsr, bsc}, M, N, K, splits, C, s);
}

namespace {

// tiles per wave: runs of up to `most` while 4096 waves remain
int run_of(int64_t tiles, int most) {
  const int64_t r = tiles / 4096;
  return (int)(r < 1 ? 1 : (r > most ? most : r));
}

int sum_rows(const float *part, int rows, int n, float *out, hipStream_t s) {
  hipLaunchKernelGGL(sum_rows_kernel, dim3((n + 15) / 16), dim3(NT), 0, s, part, rows, n, out);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

}  // namespace

int conv_pool(int layer, const uint16_t *x, int64_t B, int H, int W, const uint16_t *w, const float *bias,
              uint16_t *a, uint8_t *idx, hipStream_t s) {
  const int64_t P = B * (H / 2) * (W / 2), tiles = (P + 3) / 4;
  const int run = run_of(tiles, 8);
  const unsigned gx = (unsigned)((tiles + (int64_t)run * 4 - 1) / ((int64_t)run * 4));
  switch (layer) {
    case 0: hipLaunchKernelGGL((conv_pool_kernel<2, 16, 1>), dim3(gx, 1), dim3(NT), 0, s, x, w, bias, P, H, W, run, a, idx); break;
    case 1: hipLaunchKernelGGL((conv_pool_kernel<16, 32, 2>), dim3(gx, 1), dim3(NT), 0, s, x, w, bias, P, H, W, run, a, idx); break;
    default:
      // all four output tiles in one wave read the activations once (256
      // snippets of 64 x 256: 29 us, more with two waves of two tiles); with
      // few tiles the second wave is worth more (24 snippets: 7 us)
      if (tiles >= 8192)
        hipLaunchKernelGGL((conv_pool_kernel<32, 64, 4>), dim3(gx, 1), dim3(NT), 0, s, x, w, bias, P, H, W, run, a, idx);
      else
        hipLaunchKernelGGL((conv_pool_kernel<32, 64, 2>), dim3(gx, 2), dim3(NT), 0, s, x, w, bias, P, H, W, run, a, idx);
      break;
  }
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int conv_dx(int layer, const uint16_t *dz, int64_t B, int H, int W, const uint16_t *w, uint16_t *wf, float *dx,
            hipStream_t s) {
  const int CI = layer == 1 ? 16 : 32, CO = 2 * CI;
  hipLaunchKernelGGL(weights_flip_kernel, dim3((9 * CI * CO + NT - 1) / NT), dim3(NT), 0, s, w, CI, CO, wf);
  MDSM_HIP(hipGetLastError());
  const int64_t P = B * H * W, tiles = (P + 15) / 16;
  const int run = run_of(tiles, 8);
  const unsigned gx = (unsigned)((tiles + (int64_t)run * 4 - 1) / ((int64_t)run * 4));
  if (layer == 1) hipLaunchKernelGGL((conv_dx_kernel<32, 16, 1>), dim3(gx, 1), dim3(NT), 0, s, dz, wf, P, H, W, run, dx);
  else hipLaunchKernelGGL((conv_dx_kernel<64, 32, 2>), dim3(gx, 1), dim3(NT), 0, s, dz, wf, P, H, W, run, dx);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int64_t conv_dw_floats() { return (int64_t)DW_BLOCKS * 64 * 288; }

int conv_dw(int layer, const uint16_t *dz, const uint16_t *x, int64_t B, int H, int W, float *part, float *dw,
            hipStream_t s) {
  const int64_t items = B * ((H + WR - 1) / WR) * ((W + WC - 1) / WC);
  const int blocks = (int)(items < DW_BLOCKS ? items : DW_BLOCKS);
  if (layer == 1) hipLaunchKernelGGL((conv_dw_kernel<16, 32, 2>), dim3(blocks), dim3(NT), 0, s, dz, x, B, H, W, part);
  else hipLaunchKernelGGL((conv_dw_kernel<32, 64, 1>), dim3(blocks), dim3(NT), 0, s, dz, x, B, H, W, part);
  MDSM_HIP(hipGetLastError());
  return sum_rows(part, blocks, layer == 1 ? 32 * 144 : 64 * 288, dw, s);
}

int conv1_dw(const float *da, const uint8_t *idx, const uint16_t *x, int64_t B, int H, int W, float *part,
             float *dwb, hipStream_t s) {
  const int64_t items = B * (H / 2) * ((W / 2 + W1C - 1) / W1C);
  const int blocks = (int)(items < 1024 ? items : 1024);
  hipLaunchKernelGGL(conv1_dw_kernel, dim3(blocks), dim3(NT), 0, s, da, idx,
                     reinterpret_cast<const uint32_t *>(x), B, H, W, part);
  MDSM_HIP(hipGetLastError());
  return sum_rows(part, blocks, 304, dwb, s);
}

int pool_backward(const float *da, const uint8_t *idx, int64_t B, int H, int W, int C, uint16_t *dz, float *part,
                  float *db, hipStream_t s) {
  const int64_t P = B * (H / 2) * (W / 2), per = NT / (C / 8), want = (P + per - 1) / per;
  const int blocks = (int)(want < 1024 ? want : 1024);
  if (C == 32) hipLaunchKernelGGL(pool_bwd_kernel<32>, dim3(blocks), dim3(NT), 0, s, da, idx, P, H, W, dz, part);
  else hipLaunchKernelGGL(pool_bwd_kernel<64>, dim3(blocks), dim3(NT), 0, s, da, idx, P, H, W, dz, part);
  MDSM_HIP(hipGetLastError());
  return sum_rows(part, blocks, C, db, s);
}

int to_canonical(const float *src, const CanonicalLayout &L, float *out, hipStream_t s) {
  hipLaunchKernelGGL(canonical_kernel, dim3(grid1d(L.n)), dim3(NT), 0, s, src, L, out);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int epilogue(const float *part, int splits, int64_t M, int64_t N, const float *bias, float *out_f32,
             const float *mask, int relu, uint16_t *out_bf16, hipStream_t s) {
  hipLaunchKernelGGL(epilogue_kernel, dim3(grid1d(M * N)), dim3(NT), 0, s, part, splits, M, N, bias,
                     out_f32, mask, relu, out_bf16);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int column_sums(const uint16_t *x, int64_t rows, int C, float *part, int max_parts, float *out,
                hipStream_t s) {
  int64_t per = (rows + max_parts - 1) / max_parts;
  if (per < 1) per = 1;
  const int nparts = (int)((rows + per - 1) / per);
  hipLaunchKernelGGL(colsum_kernel, dim3(nparts > 0 ? nparts : 1), dim3(NT), 0, s, x, rows, C, per,
                     part);
  MDSM_HIP(hipGetLastError());
  hipLaunchKernelGGL(sum_parts_kernel, dim3(C), dim3(NT), 0, s, part, nparts > 0 ? nparts : 1, C,
                     out);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int softmax_ce(const float *logits, const int32_t *y, int B, uint16_t *dl, float *loss,
               hipStream_t s) {
  hipLaunchKernelGGL(softmax_ce_kernel, dim3(1), dim3(NT), 0, s, logits, y, B, dl, loss);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int adam(float *p, const float *g, float *m, float *v, uint16_t *pb, int64_t n, float lr, float b1,
         float b2, float eps, int step, float wd, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3(grid1d(n)), dim3(NT), 0, s, p, g, m, v, pb, n, lr, b1, b2,
                     eps, c1, c2, wd);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int to_bf16(const float *x, uint16_t *y, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid1d(n)), dim3(NT), 0, s, x, y, n);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

int nchw2_to_nhwc(const uint16_t *x, int64_t B, int64_t HW, uint16_t *y, hipStream_t s) {
  const int64_t n4 = B * HW / 4;
  hipLaunchKernelGGL(nchw2_to_nhwc_kernel, dim3(grid1d(n4)), dim3(NT), 0, s, x, n4, HW / 4, y);
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

}  // namespace cnn
}  // namespace mdsm
