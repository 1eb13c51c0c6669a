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

// E entries of a row (16 bytes of floats or of the type itself), in float
template <int E, typename V>
__device__ __forceinline__ void load_entries(const V* p, float* out) {
  if constexpr (E == 8) {
    load8f<V>(p, out);
  } else if constexpr (sizeof(V) == 4) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    out[0] = a.x, out[1] = a.y, out[2] = a.z, out[3] = a.w;
  } else {
    typedef V four __attribute__((ext_vector_type(4)));
    const four a = *reinterpret_cast<const four*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = (float)a[i];
  }
}
template <int E, typename V>
__device__ __forceinline__ void store_entries(V* p, const float* in) {
  if constexpr (E == 8) store8f<V>(p, in);
  else *reinterpret_cast<float4*>(p) = make_float4(in[0], in[1], in[2], in[3]);
}

// Row ids[t] of a table times scale, as TO, by the whole block, eight entries a thread at a time (H a multiple of 8, table and rows 16
// bytes aligned), in pieces of 16 bytes of the result, neighbours' side by side: what a wave stores is in a row. (Eight floats a thread
// side by side: 2,048 rows of 4,096 floats 12.0 us, so 10.7, entry by entry 11.4.) An id out of range gives a row of zeros. One trip to
// memory after the id's; entry by entry, a row of 4,096 in bfloat16 takes 256 threads 16 trips: 8 rows 8.9 us, so 3.8, 2,048 rows 16.6 and
// 11.5; 16 rows of 2,048 as floats 7.3 and 3.1.
template <typename T, typename TO>
__device__ __forceinline__ void embed_row(const int* ids, const T* table, TO* out, int H, int V, float scale) {
  constexpr int E = 16 / sizeof(TO), P = 8 / E;
  const int t = blockIdx.x, id = ids[t];
  const bool ok = id >= 0 && id < V;
  const T* row = table + (size_t)(ok ? id : 0) * H;
  TO* to = out + (size_t)t * H;
  for (int first = threadIdx.x * E; first < H; first += blockDim.x * 8) {
    int at[P];
#pragma unroll
    for (int p = 0; p < P; ++p) at[p] = min(first + p * (int)blockDim.x * E, H - E);   // (behind the end: the last piece once more)
    if (std::is_same<T, TO>::value && scale == 1.0f) {   // (the bytes)
      uint4 v[P];
#pragma unroll
      for (int p = 0; p < P; ++p) v[p] = *reinterpret_cast<const uint4*>(row + at[p]);
#pragma unroll
      for (int p = 0; p < P; ++p) *reinterpret_cast<uint4*>(to + at[p]) = ok ? v[p] : uint4{0, 0, 0, 0};
    } else {
      float v[P][E];
#pragma unroll
      for (int p = 0; p < P; ++p) load_entries<E, T>(row + at[p], v[p]);
#pragma unroll
      for (int p = 0; p < P; ++p) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[p][e] = ok ? v[p][e] * scale : 0.f;
        store_entries<E, TO>(to + at[p], v[p]);
      }
    }
  }
}
inline bool embeds_by_pieces(const void* table, const void* out, int H) { return H % 8 == 0 && (((uintptr_t)table | (uintptr_t)out) & 15) == 0; }
inline unsigned embed_threads(int H) {       // (as many trips as 1,024 threads need, all of them full)
  const int trips = (H / 8 + 1023) / 1024;
  return (unsigned)((H / 8 + 64 * trips - 1) / (64 * trips) * 64);
}

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
