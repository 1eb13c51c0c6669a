// Eight entries of a row at a time, in float; and what a head of queries or keys passes between its projection and the cache.
#pragma once
#include "nhv_common.h"
#include <type_traits>

template <typename V>
__device__ __forceinline__ void load8f(const V* p, float* out) {
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = to_f32(p[e]);
}
template <>
__device__ __forceinline__ void load8f<bf16_t>(const bf16_t* p, float* out) {
  typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 v8;
  const v8 v = *reinterpret_cast<const v8*>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = (float)v[e];
}
template <>
__device__ __forceinline__ void load8f<float>(const float* p, float* out) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w; out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
}
template <typename V>
__device__ __forceinline__ void store8f(V* p, const float* in) {
#pragma unroll
  for (int e = 0; e < 8; ++e) p[e] = from_f32<V>(in[e]);
}
template <>
__device__ __forceinline__ void store8f<bf16_t>(bf16_t* p, const float* in) {
  typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 v8;
  v8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (__bf16)in[e];
  *reinterpret_cast<v8*>(p) = v;
}
template <>
__device__ __forceinline__ void store8f<float>(float* p, const float* in) {
  *reinterpret_cast<float4*>(p) = make_float4(in[0], in[1], in[2], in[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(in[4], in[5], in[6], in[7]);
}

// Row ids[t] of a table times scale, as TO, by the whole block in pieces of eight entries (H a multiple of 8, table and rows 16 bytes aligned). An
// id out of range gives a row of zeros. One trip to memory after the id's; entry by entry, a row of 4,096 in bfloat16 takes 256 threads 16
// trips: 8 rows 8.9 us, so 3.8, 2,048 rows 16.6 and 11.5; 16 rows of 2,048 as floats 7.3 and 3.1.
template <typename T, typename TO>
__device__ __forceinline__ void embed_row(const int* ids, const T* table, TO* out, int H, int V, float scale) {
  const int t = blockIdx.x, id = ids[t];
  const bool ok = id >= 0 && id < V;
  for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
    const T* from = table + (size_t)(ok ? id : 0) * H + i;
    TO* to = out + (size_t)t * H + i;
    if (std::is_same<T, TO>::value && scale == 1.0f) {   // (the bytes)
#pragma unroll
      for (int p = 0; p < (int)sizeof(T) / 2; ++p) {
        const uint4 v = reinterpret_cast<const uint4*>(from)[p];
        reinterpret_cast<uint4*>(to)[p] = ok ? v : uint4{0, 0, 0, 0};
      }
    } else {
      float v[8];
      load8f<T>(from, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = ok ? v[e] * scale : 0.f;
      store8f<TO>(to, v);
    }
  }
}
inline bool embeds_by_pieces(const void* table, const void* out, int H) { return H % 8 == 0 && (((uintptr_t)table | (uintptr_t)out) & 15) == 0; }
inline unsigned embed_threads(int H) { return H >= 8192 ? 1024 : (unsigned)((H / 8 + 63) / 64 * 64); }

// Eight entries of a product that comes as float parts (gemm_lines_bf16.hip), `stride` entries apart, added in their order; all
// parts are asked for before the first is used.
template <int SPLITS>
__device__ __forceinline__ void add_parts8(const float* p, size_t stride, float* out) {
  float part[SPLITS][8];
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) load8f<float>(p + s * stride, part[s]);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    out[e] = part[0][e];
#pragma unroll
    for (int s = 1; s < SPLITS; ++s) out[e] += part[s][e];
  }
}
__device__ __forceinline__ void add_parts8(const float* p, size_t stride, int splits, float* out) {
  if (splits == 8) add_parts8<8>(p, stride, out);
  else if (splits == 4) add_parts8<4>(p, stride, out);
  else if (splits == 2) add_parts8<2>(p, stride, out);
  else add_parts8<1>(p, stride, out);
}

// A head of 8 CH entries in CH lanes, lane c of it with v = entries 8 c ...: the norm's sum and the rotation's partner come by shuffles, so the
// lanes of a head come here together.
// Divided by its root mean square and multiplied by its weight, each rounded.
template <typename T, typename W, int CH>
__device__ __forceinline__ void normed_head(float* v, const W* nw, float eps, int c) {
  constexpr int D = CH * 8;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
#pragma unroll
  for (int off = 1; off < CH; off <<= 1) ss += __shfl_xor(ss, off, NHV_WAVE);
  const float r = 1.0f / sqrtf(ss / (float)D + eps);
  float wv[8];
  load8f<W>(nw + c * 8, wv);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = to_f32(from_f32<T>(to_f32(from_f32<T>(v[e] * r)) * wv[e]));
}

// Turned by halves: cs, sn are the cosines and sines of entries 8 c ... modulo the half.
template <int CH>
__device__ __forceinline__ void turned_head(const float* v, const float* cs, const float* sn, int c, float* o) {
  constexpr int HALF_LANES = CH / 2 > 0 ? CH / 2 : 1;
  const bool first_half = c < HALF_LANES;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float partner = __shfl_xor(v[e], HALF_LANES, NHV_WAVE);
    o[e] = first_half ? v[e] * cs[e] - partner * sn[e] : v[e] * cs[e] + partner * sn[e];
  }
}
