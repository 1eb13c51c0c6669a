// A layer whose sublayers are normed on both sides: x <- x + norm_b(sublayer(norm_a(x))) on a float stream x.
// nhv_sandwich_step is the one launch between two sublayers: it norms the result y of the sublayer before it
// (y / sqrt(mean(y^2) + eps) * wb), adds that to the stream, and norms the new stream for the sublayer after it
// (x / sqrt(mean(x^2) + eps) * wa, given as rows of the model's element type). Either half may be absent: the first
// launch of a model only reads, the last only adds. One block a token whose size depends on the width alone, so the
// order of a row's sums, and with it a token's result, does not depend on the batch. Statistics, weights and the
// stream are float.
#include "nhv_common.h"
#include <math.h>

template <typename TY, typename TH, int BLOCK>
__global__ __launch_bounds__(BLOCK) void sandwich_step_kernel(float* __restrict__ x, const TY* __restrict__ y,
                                                              const float* __restrict__ wb, float eps_b,
                                                              const float* __restrict__ wa, float eps_a,
                                                              TH* __restrict__ h, int W) {
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * W;
  float* xr = x + base;
  if (y) {
    const TY* yr = y + base;
    float ss = 0.f;
    for (int i = threadIdx.x; i < W; i += BLOCK) {
      const float v = to_f32(yr[i]);
      ss = fmaf(v, v, ss);
    }
    const float r = 1.0f / sqrtf(block_sum(ss, scratch) / (float)W + eps_b);
    if (!wa) {
      for (int i = threadIdx.x; i < W; i += BLOCK) xr[i] += to_f32(yr[i]) * r * wb[i];
      return;
    }
    float sx = 0.f;
    for (int i = threadIdx.x; i < W; i += BLOCK) {
      const float v = xr[i] + to_f32(yr[i]) * r * wb[i];
      xr[i] = v;                               // (a thread reads back only what it wrote itself)
      sx = fmaf(v, v, sx);
    }
    const float rx = 1.0f / sqrtf(block_sum(sx, scratch) / (float)W + eps_a);
    TH* hr = h + base;
    for (int i = threadIdx.x; i < W; i += BLOCK) hr[i] = from_f32<TH>(xr[i] * rx * wa[i]);
    return;
  }
  float sx = 0.f;
  for (int i = threadIdx.x; i < W; i += BLOCK) {
    const float v = xr[i];
    sx = fmaf(v, v, sx);
  }
  const float rx = 1.0f / sqrtf(block_sum(sx, scratch) / (float)W + eps_a);
  TH* hr = h + base;
  for (int i = threadIdx.x; i < W; i += BLOCK) hr[i] = from_f32<TH>(xr[i] * rx * wa[i]);
}

// The same for widths that are a multiple of 4 (up to 16,384), four entries at a time: a thread has PASSES fours of the row in registers from
// the first load to the last store, everything that either half needs is asked for before the first sum, and a sum's parts meet
// over one barrier. Bound by the trips to memory and over the barriers for few rows, by the reads and writes for many. In a recorded graph
// 16 rows of 2,048: 4.0 -> 2.6 us, 1,925 rows: 11.8 -> 8.4; 8 of 8,192: 6.2 -> 3.8.
template <typename T>
struct alignas(4 * sizeof(T)) SandwichFour {
  T e[4];
};

template <int BLOCK>
__device__ __forceinline__ float sandwich_sum(float v, float* parts /* BLOCK / 64 floats of this sum alone */) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) parts[threadIdx.x >> 6] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < BLOCK / 64; ++i) total += parts[i];
  return total;
}

template <typename TY, typename TH, int BLOCK, int PASSES, bool ADD, bool READ>
__global__ __launch_bounds__(BLOCK) void sandwich_step_wide_kernel(float* __restrict__ x, const TY* __restrict__ y,
                                                                   const float* __restrict__ wb, float eps_b,
                                                                   const float* __restrict__ wa, float eps_a,
                                                                   TH* __restrict__ h, int W) {
  __shared__ float parts_y[BLOCK / 64], parts_x[BLOCK / 64];
  const size_t base = (size_t)blockIdx.x * W;
  SandwichFour<float> xv[PASSES], av[PASSES], bv[PASSES];
  SandwichFour<TY> yv[PASSES];
  int at[PASSES];
  bool in[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int i = (p * BLOCK + threadIdx.x) * 4;
    in[p] = i < W;
    at[p] = in[p] ? i : W - 4;
    if (ADD) yv[p] = *reinterpret_cast<const SandwichFour<TY>*>(y + base + at[p]);
    xv[p] = *reinterpret_cast<const SandwichFour<float>*>(x + base + at[p]);
  }
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    if (ADD) bv[p] = *reinterpret_cast<const SandwichFour<float>*>(wb + at[p]);
    if (READ) av[p] = *reinterpret_cast<const SandwichFour<float>*>(wa + at[p]);
  }
  if (ADD) {
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = in[p] ? to_f32(yv[p].e[k]) : 0.f;
        ss = fmaf(v, v, ss);
      }
    const float r = 1.0f / sqrtf(sandwich_sum<BLOCK>(ss, parts_y) / (float)W + eps_b);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
#pragma unroll
      for (int k = 0; k < 4; ++k) xv[p].e[k] += to_f32(yv[p].e[k]) * r * bv[p].e[k];
      if (in[p]) *reinterpret_cast<SandwichFour<float>*>(x + base + at[p]) = xv[p];
    }
  }
  if (READ) {
    float sx = 0.f;
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = in[p] ? xv[p].e[k] : 0.f;
        sx = fmaf(v, v, sx);
      }
    const float rx = 1.0f / sqrtf(sandwich_sum<BLOCK>(sx, parts_x) / (float)W + eps_a);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      SandwichFour<TH> out;
#pragma unroll
      for (int k = 0; k < 4; ++k) out.e[k] = from_f32<TH>(xv[p].e[k] * rx * av[p].e[k]);
      if (in[p]) *reinterpret_cast<SandwichFour<TH>*>(h + base + at[p]) = out;
    }
  }
}

template <typename TY, typename TH>
static void sandwich_launch(hipStream_t s, int T, int W, float* x, const void* y, const float* wb, float eps_b,
                            const float* wa, float eps_a, void* h) {
  // (a row's sums have the order of its width, whichever of its halves are there and whatever the addresses: one kernel a width,
  // but for what cannot be read four at a time)
  const bool fours = (((uintptr_t)x | (uintptr_t)wb | (uintptr_t)wa) & 15) == 0 && ((uintptr_t)y & (4 * sizeof(TY) - 1)) == 0 &&
                     ((uintptr_t)h & (4 * sizeof(TH) - 1)) == 0;
  if (W % 4 == 0 && W <= 16384 && fours) {
#define LAUNCH_HALVES(B, P, ADD, READ)                                                                                               \
  hipLaunchKernelGGL((sandwich_step_wide_kernel<TY, TH, B, P, ADD, READ>), dim3(T), dim3(B), 0, s, x, (const TY*)y, wb, eps_b, wa, eps_a, (TH*)h, W)
#define LAUNCH_WIDE(B, P)                                    \
  do {                                                       \
    if (y && wa) LAUNCH_HALVES(B, P, true, true);            \
    else if (y) LAUNCH_HALVES(B, P, true, false);            \
    else LAUNCH_HALVES(B, P, false, true);                   \
  } while (0)
    if (W <= 1024) LAUNCH_WIDE(256, 1);
    else if (W <= 2048) LAUNCH_WIDE(512, 1);
    else if (W <= 4096) LAUNCH_WIDE(512, 2);
    else if (W <= 8192) LAUNCH_WIDE(1024, 2);
    else LAUNCH_WIDE(1024, 4);
#undef LAUNCH_WIDE
#undef LAUNCH_HALVES
    return;
  }
#define LAUNCH(B) hipLaunchKernelGGL((sandwich_step_kernel<TY, TH, B>), dim3(T), dim3(B), 0, s, x, (const TY*)y, wb, eps_b, wa, eps_a, (TH*)h, W)
  if (W <= 1024) LAUNCH(256);
  else if (W <= 4096) LAUNCH(512);
  else LAUNCH(1024);
#undef LAUNCH
}

// x [T, W] float, rewritten if y is given. y [T, W] of y_dtype with wb [W] float, or null. wa [W] float with h [T, W] of
// h_dtype, or null.
extern "C" int nhv_sandwich_step(void* x, const void* y, int y_dtype, const void* wb, float eps_b, const void* wa,
                                 float eps_a, void* h, int h_dtype, int T, int W, void* stream) {
  NHV_REQUIRE(T > 0 && W > 0 && x, "sandwich_step: bad sizes T=%d W=%d", T, W);
  NHV_REQUIRE(y || wa, "sandwich_step: nothing to add and nothing to read");
  NHV_REQUIRE(!y || wb, "sandwich_step: a result without the weight of its norm");
  NHV_REQUIRE(!wa || h, "sandwich_step: a norm to read through without rows for it");
  NHV_REQUIRE(eps_a >= 0.f && eps_b >= 0.f, "sandwich_step: eps %g, %g", (double)eps_a, (double)eps_b);
  hipStream_t s = (hipStream_t)stream;
  const bool yf = !y || y_dtype == NHV_F32, hf = !wa || h_dtype == NHV_F32;
  NHV_REQUIRE((yf || y_dtype == NHV_BF16) && (hf || h_dtype == NHV_BF16), "sandwich_step: unknown dtypes %d, %d", y_dtype, h_dtype);
  if (yf && hf) sandwich_launch<float, float>(s, T, W, (float*)x, y, (const float*)wb, eps_b, (const float*)wa, eps_a, h);
  else if (yf) sandwich_launch<float, bf16_t>(s, T, W, (float*)x, y, (const float*)wb, eps_b, (const float*)wa, eps_a, h);
  else if (hf) sandwich_launch<bf16_t, float>(s, T, W, (float*)x, y, (const float*)wb, eps_b, (const float*)wa, eps_a, h);
  else sandwich_launch<bf16_t, bf16_t>(s, T, W, (float*)x, y, (const float*)wb, eps_b, (const float*)wa, eps_a, h);
  NHV_LAUNCH_CHECK("sandwich_step");
  return 0;
}
