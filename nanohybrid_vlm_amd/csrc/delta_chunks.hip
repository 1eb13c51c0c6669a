// The gated delta rule over portions of prompts, 16 tokens at a time (what the recurrence is, and the kernels for single
// tokens and for 32-bit runs: delta_rule.hip). With l_t the running sums of the decays' base-2 logarithms within a chunk
// (the token's own included) and E_t = 2^l_t per key channel,
//   S_t = E_t S_0 + sum_(j <= t) (E_t / E_j) k_j u_j^T,     u_t = beta_t (v_t - (E_t k_t)^T S_0 - sum_(j < t) A'[t, j] u_j),
//   A'[t, j] = sum_d k_t k_j 2^(l_t - l_j),   B[t, j] = sum_d q_t k_j 2^(l_t - l_j)  (j <= t),
// so with U the chunk's u, A = beta A' strictly below the diagonal and (I + A) solved forwards for every column:
//   W = (I + A)^-1 beta E k,   V' = (I + A)^-1 beta v,   U = V' - W S_0,   O = E q S_0 + B U = R S_0 + B V',
//   S_16 = E_16 S_0 + K^T U,   K_j = k_j 2^(l_16 - l_j).
// Only differences of logarithms that are never positive are raised: a strong decay gives zeros, not overflows. A sum of
// logarithms is kept as a float and what its additions rounded off, and a token's logarithm is no lower than -256 (whose power
// is 0 all the same): the difference of two sums is then as exact as a sum over the tokens between them, whatever decays came
// before, and never inf - inf. (One float alone: after three tokens of -300 a state off by 3e-5 of its largest entry, and NaN
// after an infinite one. Token by token and with both parts 1e-7.)
// Two kernels:
//  - nhv_delta_chunks_prepare: all chunks at once, a block per (chunk, head, request), from the projection's rows to W, R - B W,
//    K, V', B V' and the chunk's decay (a token's sum of B V' takes the tokens up to it and no others: as a product of whole
//    matrices an infinite value would come back to the tokens before it as 0 times infinity): convolutions, SiLU, unit vectors, decays, products and the solution without a trip to
//    memory between them (the rows are read once and a fifth over; the separate kernel that wrote q, k, v, beta and decays
//    took 101 us for 2,201 tokens of 16 heads of 128);
//  - nhv_delta_chunks: a request's chunks in order, as float matrix products (v_mfma_f32_16x16x4_f32).
// The second is a chain of chunks, and what it lasts is what a chunk waits for (two rows of dependent matrix instructions and
// one exchange between the waves: 0.82 us a chunk), not its arithmetic; the token-by-token kernel takes 0.36 us a token. Eight
// waves a block, a tile each, wait longer for each other (99 us where four took 91).
// us of the chain, before its loads were whole kilobytes in the preparation's order, its results were stored without a branch and R was
// multiplied while the shares come back, and now: portions of 1,500 and 764 tokens, 16 heads of 128, 88, 77; of 64 55, 49; 8 heads of 256 on
// 128 171, 140; 24 of 80 tokens, 16 heads of 128, 69, 54; 8,000 tokens 446, 389.
// The preparation is bound by its vector instructions (80 % of the clocks of all SIMDs). It took 4,230 a wave, of which 1,520 were the
// decays (a division to find token and channel, log1pf, expf), 720 the inputs' SiLU and 280 moved scalar values to vector
// registers and back; with the functions below, rows dealt to waves, and nothing worked out ahead that a wave cannot keep, half of
// that: the same sizes 77, 61; 56, 43; 114, 82; 69, 51; 274, 179 us, 40 and 17 tokens 22, 15. Results are as far from 64 bits as before (1.7e-7 to
// 2.8e-7 of their size, by how slowly they decay).
// Portions of 1,500 and 701 tokens, 16 heads of 128, with the update of the kept inputs and the read-out's norm: 198 us where the
// separate kernels take 638; one of 8,000 770 against 3,204. The blocks of the preparation are requests by the longest portion:
// for 2,000 tokens beside 60 decoded ones 98 of 100 are empty, which is 16 us of 290 (a search for each place's request gave
// them back there and cost 11 of 174 us for 24 portions of 80). Everything is float, and the state is as far from 64 bits as
// token by token.
// The method, triangular systems in place of products of Householder-like steps (a WY representation; Bischof and Van Loan,
// "The WY representation for products of Householder matrices", 1987), is that of Yang, Wang, Zhang, Shen and Kim,
// "Parallelizing Linear Transformers with the Delta Rule over Sequence Length", 2024, here with a decay a key channel.
#include "nhv_common.h"
#include <float.h>
#include <math.h>

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define NHV_LOG2E 1.4426950408889634f
#define NHV_CHUNK 16
#define NHV_MAX_TAPS 16

__device__ __forceinline__ float exp2_of(float x) { return __builtin_amdgcn_exp2f(x); }   // (x <= 0; tiny results may become 0)
// e^x for |x| up to 110, the part of x log2(e) behind the whole number in two pieces of log2(e)
__device__ __forceinline__ float exp_of(float x) {
  const float whole = __builtin_rintf(x * 1.44269502f);
  return ldexpf(exp2_of(fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502f, -whole))), (int)whole);
}
// z / (1 + e^-z): the quotient by the reciprocal, put right by what it leaves of z (off by 3.7e-8 on average, as the division is, in half
// the instructions)
__device__ __forceinline__ float silu_of(float z) {
  const float d = 1.0f + exp_of(__builtin_amdgcn_fmed3f(-z, -110.f, 110.f)), r = __builtin_amdgcn_rcpf(d), q = z * r;
  const float y = fmaf(fmaf(-d, q, z), r, q);
  return y == y ? y : q;                     // (an infinite d or z leaves no number)
}
// rate log2(1 + e^z), rate log2(e) in two pieces: max(z, 0) log2(e) and log2(w), w = 1 + e^-|z|, of which w's own rounding c is the part c / w.
// Off by 2.5e-8 (z > 1) to 5.1e-8 (z down to -12; below, where nothing decays, 7e-8) on average; -log2(e) rate log1p(e^z) by the
// library's functions 4.6e-8 to 5.3e-8, and 190 instructions with its addresses where this is 40.
// Where the first part alone is beyond what counts (512; the logarithm ends at -256) it is the result: of an infinite or huge z the second, whose sign is
// that of log2(e) rate's rounding, would be as infinite, against it.
__device__ __forceinline__ float softplus_bits(float z, float rate, float bits, float rest) {
  const float a = fabsf(z), u = exp_of(a > 110.f ? -110.f : -a), w = 1.0f + u, c = u - (w - 1.0f), m = fmaxf(z, 0.f), first = bits * m;
  const float sum = fmaf(bits, m, fmaf(rest, m, fmaf(rate, __builtin_amdgcn_logf(w), c * __builtin_amdgcn_rcpf(w) * bits)));
  return first > 512.f ? first : sum;
}
#define NHV_LOWEST_LOG (-256.f)

struct DeltaIn {
  const void* proj;                          // [T, ld]: q (G D) | k (G D) | v (H E) | beta (H)
  long long ld;
  const float* taps;                         // [C, n], last column for the token itself
  int n_taps;
  const float* kept;                         // [slots, C, n - 1]
  const float* a_lin;                        // [T, a_ld]: the decays' linear part, H Dd columns
  long long a_ld;
  const float *dt_bias, *a_log;              // [H Dd], [H]
  const int *positions, *cu, *state_slots;
  int H, G, D, E, Dd;
};

struct DeltaChunks {                         // per (place, head); a chunk's place: cu[req] / 16 + req + its number in the request
  float *w, *r;                              // [Dp / 16][4][16][4]: of a tile of 16 channels, four channels, their tokens
  float *k;                                  // [Dp][16]
  float *v;                                  // [E][16]
  float *o;                                  // [E][16]: B V'
  float *decay;                              // [Dp]
};

// A channel's sixteen convolved inputs, through SiLU; zeros for tokens beyond n. TAPS 0: any number.
template <typename TI, int TAPS>
__device__ __forceinline__ void convolved(const DeltaIn& in, int c, int first, int i0, int pos0, const float* mine, int n, float* y) {
  // (taken anew at each call: worked out ahead for all calls, rows' places and conditions would be kept in parts of vector registers)
  asm volatile("" : "+s"(first), "+s"(i0), "+s"(n), "+s"(pos0));
  const TI* col = (const TI*)in.proj + (size_t)first * in.ld + c;
  const int taps = TAPS ? TAPS : in.n_taps;
  const float* tap = in.taps + (size_t)c * taps;
  auto input = [&](int i) -> float {         // the request's i-th token of the step, counted from the chunk's first
    if (i >= n || pos0 + i < 0) return 0.f;
    const int at = i0 + i;
    return at >= 0 ? to_f32(col[(size_t)at * in.ld]) : mine[(size_t)c * (taps - 1) + (taps - 1) + at];
  };
  if (TAPS) {
    float x[NHV_CHUNK + (TAPS ? TAPS : 1) - 1], m[TAPS ? TAPS : 1];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) m[j] = tap[TAPS - 1 - j];
    if (i0 > 0 && n == NHV_CHUNK) {          // (all of it lies among the step's rows: loads without conditions; TAPS <= 16 <= i0)
#pragma unroll
      for (int i = 0; i < NHV_CHUNK + TAPS - 1; ++i) x[i] = to_f32(col[(size_t)(i0 + i - (TAPS - 1)) * in.ld]);
    } else {
#pragma unroll
      for (int i = 0; i < NHV_CHUNK + TAPS - 1; ++i) x[i] = input(i - (TAPS - 1));
    }
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) sum = fmaf(m[j], x[t + TAPS - 1 - j], sum);
      y[t] = silu_of(sum);
    }
  } else {
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) {
      float sum = 0.f;
      for (int j = 0; j < taps; ++j) sum = fmaf(tap[taps - 1 - j], input(t - j), sum);
      y[t] = silu_of(sum);
    }
  }
  if (n < NHV_CHUNK) {                       // (one branch, not one a token)
    asm volatile("");
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) y[t] = t < n ? y[t] : 0.f;
  }
}

template <typename TI, int TAPS>
__global__ __launch_bounds__(256, 4) void delta_chunks_prepare_kernel(const DeltaIn in, const DeltaChunks to, int Dp) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ __attribute__((aligned(16))) float A[NHV_CHUNK][NHV_CHUNK], B[NHV_CHUNK][NHV_CHUNK];
  __shared__ float beta[NHV_CHUNK];
  __shared__ float2 last[256];               // a channel's sum over the chunk
  const int h = blockIdx.x, req = blockIdx.z;
  const int first = in.cu[req], i0 = blockIdx.y * NHV_CHUNK, t0 = first + i0, end = in.cu[req + 1];
  if (t0 >= end) return;                     // (the same for the whole block)
  const int n = min(NHV_CHUNK, end - t0), pos0 = in.positions[t0];
  const size_t place = ((size_t)(first / NHV_CHUNK) + req + blockIdx.y) * in.H + h;
  const int H = in.H, G = in.G, D = in.D, E = in.E, Dd = in.Dd, C = 2 * G * D + H * E, g = h / (H / G);
  const int tid = threadIdx.x, LD = Dp + 4;  // (rows of an odd number of fours)
  float* qs = lds;
  float* ks = qs + NHV_CHUNK * LD;
  float2* ls = reinterpret_cast<float2*>(ks + NHV_CHUNK * LD);       // the sums of logarithms and what they are short of
  const float* mine = in.kept + (size_t)in.state_slots[req] * C * (in.n_taps - 1);

  // queries and keys, a channel a thread; the decays' logarithms; beta
  for (int x = tid; x < 2 * Dp; x += 256) {
    const int d = x < Dp ? x : x - Dp;
    float* to_row = (x < Dp ? qs : ks) + d;
    float y[NHV_CHUNK];
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) y[t] = 0.f;
    if (d < D) convolved<TI, TAPS>(in, (x < Dp ? 0 : G * D) + g * D + d, first, i0, pos0, mine, n, y);
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) to_row[t * LD] = y[t];
  }
  // (four rows a wave, channels on its lanes: no division, and a row's address is the wave's)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // (finite pieces, so that they leave nothing of what does not decay; what is no number stays none)
  const float asked = expf(in.a_log[h]), rate = asked > FLT_MAX ? FLT_MAX : asked;
  const float bits = rate > FLT_MAX / 1.5f ? FLT_MAX : rate * 1.44269502f, rest = fmaf(rate, 1.92596299e-8f, fmaf(rate, 1.44269502f, -bits));
  for (int d = lane; d < Dp; d += 64) {
    const int at = h * Dd + (Dd == 1 ? 0 : min(d, D - 1));
    const float bias = in.dt_bias[at];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = wave + 4 * i;
      const float l = -softplus_bits(in.a_lin[(size_t)(t0 + min(t, n - 1)) * in.a_ld + at] + bias, rate, bits, rest);
      ls[t * LD + d].x = t < n && d < D ? (l < NHV_LOWEST_LOG ? NHV_LOWEST_LOG : l) : 0.f;      // (what is no number stays none)
    }
  }
  if (tid < NHV_CHUNK)
    beta[tid] = tid < n ? 1.0f / (1.0f + expf(-to_f32(((const TI*)in.proj)[(size_t)(t0 + tid) * in.ld + C + h]))) : 0.f;
  __syncthreads();
  for (int d = tid; d < Dp; d += 256) {
    float sum = 0.f, rest = 0.f;
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) {
      const float l = ls[t * LD + d].x, next = sum + l, part = next - sum;
      rest += (sum - (next - part)) + (l - part);        // (what the addition rounded off, exactly)
      sum = next;
      ls[t * LD + d] = make_float2(sum, rest);
    }
    last[d] = make_float2(sum, rest);        // (a row beyond the request's end adds 0)
  }
  {                                          // unit length (the sum of squares plus 1e-6 under the root), q also times D^(-1/2)
    const int t = (tid >> 3) & 15;
    float* row = (tid < 128 ? qs : ks) + t * LD;
    float ss = 0.f;
    for (int d = (tid & 7) * 4; d < Dp; d += 32) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(row + d);
      ss += x[0] * x[0] + x[1] * x[1] + (x[2] * x[2] + x[3] * x[3]);
    }
    ss += __shfl_xor(ss, 1, NHV_WAVE);
    ss += __shfl_xor(ss, 2, NHV_WAVE);
    ss += __shfl_xor(ss, 4, NHV_WAVE);
    const float r = (tid < 128 ? 1.0f / sqrtf((float)D) : 1.0f) / sqrtf(ss + 1e-6f);
    for (int d = (tid & 7) * 4; d < Dp; d += 32) *reinterpret_cast<floatx4*>(row + d) *= r;
  }
  __syncthreads();
  // the products of the chunk's tokens: two threads a pair j < t (120 pairs), sixteen threads for j = t
  if (tid < 240) {
    const int p = tid >> 1;
    int t = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)p)) * 0.5f);
    t = t * (t - 1) / 2 > p ? t - 1 : ((t + 1) * t / 2 <= p ? t + 1 : t);
    const int j = p - t * (t - 1) / 2, d0 = (tid & 1) * 4;
    const float *qt = qs + t * LD, *kt = ks + t * LD, *kj = ks + j * LD;
    const float2 *lt = ls + t * LD, *lj = ls + j * LD;
    floatx4 kk = {0.f, 0.f, 0.f, 0.f}, qk = {0.f, 0.f, 0.f, 0.f};
    if (Dd == 1) {
      for (int d = d0; d < Dp; d += 8) {
        const floatx4 x = *reinterpret_cast<const floatx4*>(kj + d);
        kk += *reinterpret_cast<const floatx4*>(kt + d) * x;
        qk += *reinterpret_cast<const floatx4*>(qt + d) * x;
      }
      const float e = exp2_of((lt[0].x - lj[0].x) + (lt[0].y - lj[0].y));
      kk *= e;
      qk *= e;
    } else {
#pragma unroll 2
      for (int d = d0; d < Dp; d += 8) {
        floatx4 x;
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const floatx4 l = *reinterpret_cast<const floatx4*>(lt + d + i) - *reinterpret_cast<const floatx4*>(lj + d + i);
          x[i] = exp2_of(l[0] + l[1]);
          x[i + 1] = exp2_of(l[2] + l[3]);
        }
        x *= *reinterpret_cast<const floatx4*>(kj + d);
        kk += *reinterpret_cast<const floatx4*>(kt + d) * x;
        qk += *reinterpret_cast<const floatx4*>(qt + d) * x;
      }
    }
    float a = (kk[0] + kk[1]) + (kk[2] + kk[3]), b = (qk[0] + qk[1]) + (qk[2] + qk[3]);
    a += __shfl_xor(a, 1, NHV_WAVE);
    b += __shfl_xor(b, 1, NHV_WAVE);
    if ((tid & 1) == 0) {
      A[t][j] = beta[t] * a;
      B[t][j] = b;
    }
  } else {
    const int t = tid - 240;
    floatx4 qk = {0.f, 0.f, 0.f, 0.f};
    for (int d = 0; d < Dp; d += 4) qk += *reinterpret_cast<const floatx4*>(qs + t * LD + d) * *reinterpret_cast<const floatx4*>(ks + t * LD + d);
    B[t][t] = (qk[0] + qk[1]) + (qk[2] + qk[3]);
  }
  __syncthreads();
  // E_t q_t, E_t k_t and, in the sums' place, k_t 2^(l_16 - l_t) (rows beyond n are zeros)
  for (int d = lane; d < Dp; d += 64) {
    const float2 all = last[d];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = (wave + 4 * i) * LD + d;
      const float2 l = ls[at];
      const float e = exp2_of(l.x + l.y), k = ks[at];
      qs[at] *= e;
      ks[at] = e * k;
      ls[at].x = k * exp2_of((all.x - l.x) + (all.y - l.y));
    }
  }
  __syncthreads();
  // a column a thread: W's Dp, then V''s E
  for (int c = tid; c < Dp + E; c += 256) {
    const bool key = c < Dp;
    float x[NHV_CHUNK];
    if (key) {
#pragma unroll
      for (int t = 0; t < NHV_CHUNK; ++t) x[t] = ks[t * LD + c];
    } else {
      convolved<TI, TAPS>(in, 2 * G * D + h * E + c - Dp, first, i0, pos0, mine, n, x);
    }
#pragma unroll
    for (int t = 0; t < NHV_CHUNK; ++t) {
      asm volatile("" ::: "memory");         // (a row of A at a time: all of A and B in registers would leave one wave a SIMD)
      x[t] *= beta[t];
#pragma unroll
      for (int j = 0; j < t; ++j) x[t] = fmaf(-A[t][j], x[j], x[t]);
    }
    if (key) {
      float* k = to.k + (place * Dp + c) * NHV_CHUNK;
#pragma unroll
      for (int t = 0; t < NHV_CHUNK; ++t) {
        asm volatile("" ::: "memory");
        ks[t * LD + c] = x[t];
        float y = qs[t * LD + c];
#pragma unroll
        for (int j = 0; j <= t; ++j) y = fmaf(-B[t][j], x[j], y);
        qs[t * LD + c] = y;
      }
#pragma unroll
      for (int t = 0; t < NHV_CHUNK; t += 4) {
        floatx4 kk;
#pragma unroll
        for (int j = 0; j < 4; ++j) kk[j] = ls[(t + j) * LD + c].x;
        *reinterpret_cast<floatx4*>(k + t) = kk;
      }
      to.decay[place * Dp + c] = exp2_of(last[c].x + last[c].y);
    } else {
      float* v = to.v + (place * E + c - Dp) * NHV_CHUNK;
      float* o = to.o + (place * E + c - Dp) * NHV_CHUNK;
#pragma unroll
      for (int t = 0; t < NHV_CHUNK; t += 4) {
        floatx4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          asm volatile("" ::: "memory");
          y[i] = 0.f;
#pragma unroll
          for (int j = 0; j <= t + i; ++j) y[i] = fmaf(B[t + i][j], x[j], y[i]);
        }
        *reinterpret_cast<floatx4*>(o + t) = y;
      }
#pragma unroll
      for (int t = 0; t < NHV_CHUNK; t += 4) *reinterpret_cast<floatx4*>(v + t) = floatx4{x[t], x[t + 1], x[t + 2], x[t + 3]};
    }
  }
  __syncthreads();
  // W and R as the second kernel's lanes take them: a load of a tile is a kilobyte in a row (with rows of Dp entries, sixteen times
  // 64 bytes, which come to a compute unit half as fast)
  for (int x = tid; x < 4 * Dp; x += 256) {
    const int at = (x & 15) * LD + (x >> 4) * 4;
    const size_t out = place * NHV_CHUNK * Dp + 4 * x;
    *reinterpret_cast<floatx4*>(to.w + out) = *reinterpret_cast<const floatx4*>(ks + at);
    *reinterpret_cast<floatx4*>(to.r + out) = *reinterpret_cast<const floatx4*>(qs + at);
  }
}

extern "C" int nhv_delta_chunks_prepare(const void* proj, int proj_dtype, long long ld, const void* taps, int n_taps, const void* kept,
                                        const void* a_lin, long long a_ld, const void* dt_bias, const void* a_log, const void* positions,
                                        const void* cu, const void* state_slots, void* w, void* r, void* k, void* v, void* o,
                                        void* decay, int B, int H, int G, int D, int E, int decay_dim, int max_q_len, void* stream) {
  NHV_REQUIRE(B > 0 && H > 0 && G > 0 && D > 0 && E > 0 && H % G == 0, "delta_chunks: bad sizes B=%d H=%d G=%d D=%d E=%d", B, H, G, D, E);
  NHV_REQUIRE(D <= 256 && E <= 1024 && B <= 65535 && max_q_len > 0 && max_q_len <= 65535 * NHV_CHUNK,
              "delta_chunks: D=%d (up to 256), E=%d (up to 1024), %d requests, portions of %d", D, E, B, max_q_len);
  NHV_REQUIRE(decay_dim == D || decay_dim == 1, "delta_chunks: %d decays a head (one, or one per key channel: %d)", decay_dim, D);
  NHV_REQUIRE(n_taps >= 1 && n_taps <= NHV_MAX_TAPS, "delta_chunks: %d taps (1 to %d are taken)", n_taps, NHV_MAX_TAPS);
  NHV_REQUIRE(ld >= 2ll * G * D + (long long)H * E + H && a_ld >= (long long)H * decay_dim, "delta_chunks: rows of %lld and %lld entries", ld, a_ld);
  const DeltaIn in = {proj, ld, (const float*)taps, n_taps, (const float*)kept, (const float*)a_lin, a_ld, (const float*)dt_bias,
                      (const float*)a_log, (const int*)positions, (const int*)cu, (const int*)state_slots, H, G, D, E, decay_dim};
  const DeltaChunks to = {(float*)w, (float*)r, (float*)k, (float*)v, (float*)o, (float*)decay};
  const int Dp = (D + 15) & ~15;
  const size_t lds = 4 * (size_t)NHV_CHUNK * (Dp + 4) * sizeof(float);   // (67 KB at most)
  const dim3 grid(H, (max_q_len + NHV_CHUNK - 1) / NHV_CHUNK, B);
  hipStream_t s = (hipStream_t)stream;
#define LAUNCH(TI, TAPS)                                                                                                          \
  do {                                       /* (more than 64 KB of LDS is to be allowed once per kernel) */                        \
    static const hipError_t allowed = hipFuncSetAttribute((const void*)delta_chunks_prepare_kernel<TI, TAPS>,                        \
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, 4 * NHV_CHUNK * 260 * 4);      \
    if (allowed != hipSuccess) return nhv_fail("delta_chunks: %zu bytes of LDS are refused: %s", lds, hipGetErrorString(allowed));   \
    hipLaunchKernelGGL((delta_chunks_prepare_kernel<TI, TAPS>), grid, dim3(256), lds, s, in, to, Dp);                               \
  } while (0)
  if (proj_dtype == NHV_F32) {
    if (n_taps == 4) LAUNCH(float, 4);
    else LAUNCH(float, 0);
  } else if (proj_dtype == NHV_BF16) {
    if (n_taps == 4) LAUNCH(bf16_t, 4);
    else LAUNCH(bf16_t, 0);
  } else {
    return nhv_fail("delta_chunks: unknown dtype %d", proj_dtype);
  }
#undef LAUNCH
  NHV_LAUNCH_CHECK("delta_chunks_prepare");
  return 0;
}

// ---------------------------------------------------------------- a request's chunks in order
// A block owns 16 columns of S (value channels) of one head of one request; its four waves share D in tiles of 16 rows, TPW
// tiles a wave, which stay in registers as the result of the matrix cores' products (lane l holds S[16 tile + 4 (l / 16) + i,
// column l % 16]) and are the right-hand operand of W S and R S as they stand. The waves' shares of W S meet in LDS, one
// barrier a chunk; every wave adds them up in the waves' order, and what it has then, U, lies in its registers as K^T U needs
// it. The shares of O, which begin with a quarter of B V' each, are added up and written a chunk
// later, behind that chunk's barrier. What a chunk needs is
// asked for AHEAD chunks before it is used. EVEN: every wave has TPW tiles.
template <int TPW>
struct DeltaOperands {
  floatx4 w[TPW], r[TPW], g[TPW], kk[TPW], v;
  float o;                                   // of token 4 grp + wave
};

template <int TPW, bool EVEN>
__global__ __launch_bounds__(256, TPW <= 2 ? 2 : 1) void delta_chunks_kernel(const DeltaChunks from, float* __restrict__ state, float* __restrict__ out,
                                                           const int* __restrict__ positions, const int* __restrict__ cu,
                                                           const int* __restrict__ state_slots, int H, int D, int Dp, int E) {
  constexpr int AHEAD = TPW <= 2 ? 3 : 2;
  __shared__ __attribute__((aligned(16))) float share[2][4][64 * 4];
  __shared__ __attribute__((aligned(16))) float red[2][4][64 * 4];
  const int req = blockIdx.z, h = blockIdx.x, e0 = blockIdx.y * 16;
  const int first = cu[req], end = cu[req + 1];
  if (end <= first) return;                  // (the same for the whole block)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int tiles = Dp / 16, tile0 = wave * TPW;
  const bool column = e0 + col < E;
  const int e_mine = column ? e0 + col : 0;  // (a lane beyond E works on a column that it does not write)
  float* mine = state + (((size_t)state_slots[req] * H + h) * E + e_mine) * D;
  const bool fresh = positions[first] == 0;
  floatx4 S[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = (tile0 + i) * 16 + grp * 4 + j;
      S[i][j] = (!fresh && column && d < D) ? mine[d] : 0.f;
    }
  const int chunks = (end - first + NHV_CHUNK - 1) / NHV_CHUNK;
  const size_t place0 = (size_t)(first / NHV_CHUNK) + req;
  const int r_at = tile0 * 256 + lane * 4, k_at = (tile0 * 16 + col) * NHV_CHUNK + grp * 4, g_at = tile0 * 16 + grp * 4;
  const int v_at = e_mine * NHV_CHUNK + grp * 4;
  const int spare = (EVEN ? 0 : tiles) - 1;  // (a wave without a tile reads the last one's and leaves it unused)
  DeltaOperands<TPW> ops[AHEAD];
  const size_t place = place0 * H + h;
  const float *wb = from.w + place * NHV_CHUNK * Dp, *rb = from.r + place * NHV_CHUNK * Dp, *kb = from.k + place * NHV_CHUNK * Dp;
  const float *gb = from.decay + place * Dp, *vb = from.v + place * NHV_CHUNK * E, *ob = from.o + place * NHV_CHUNK * E;
  int asked = 0;
  auto ask = [&](DeltaOperands<TPW>& x) {    // (behind the last chunk: it again, so that the waits count the same loads on every way)
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int back = EVEN ? 0 : max(tile0 + i - spare, 0);
      x.w[i] = *reinterpret_cast<const floatx4*>(wb + (uint32_t)(r_at + (i - back) * 256));
      x.r[i] = *reinterpret_cast<const floatx4*>(rb + (uint32_t)(r_at + (i - back) * 256));
      x.g[i] = *reinterpret_cast<const floatx4*>(gb + (uint32_t)(g_at + (i - back) * 16));
      x.kk[i] = *reinterpret_cast<const floatx4*>(kb + (uint32_t)(k_at + (i - back) * 16 * NHV_CHUNK));
    }
    x.v = *reinterpret_cast<const floatx4*>(vb + (uint32_t)v_at);
    x.o = ob[(uint32_t)(v_at + wave)];
    const bool more = ++asked < chunks;
    const size_t rows = more ? (size_t)H * NHV_CHUNK * Dp : 0, columns = more ? (size_t)H * NHV_CHUNK * E : 0;
    wb += rows, rb += rows, kb += rows, gb += more ? (size_t)H * Dp : 0, vb += columns, ob += columns;
  };
  // wave w writes tokens 4 grp + w of a chunk, the sum of the four waves' shares. Tokens behind the request's last one and columns behind E lie
  // behind the end of what is described here, and are not written: without a branch the products go on beside it.
  const uint32_t o_at = column ? (uint32_t)((grp * 4 + wave) * H * E + col) * 4 : 0x80000000u;
  auto emit = [&](const float* part, int c) {
    const int t = first + c * NHV_CHUNK;
    const int bytes = (min(NHV_CHUNK, end - t) * H * E - h * E - e0) * 4;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, ((part[0] + part[1]) + part[2]) + part[3]),
                                          __builtin_amdgcn_make_buffer_rsrc(out + ((size_t)t * H + h) * E + e0, 0, bytes, 0x00020000), o_at, 0, 0);
  };
  auto parts = [&](int c, float* part) {
#pragma unroll
    for (int w = 0; w < 4; ++w) part[w] = red[c & 1][w][lane * 4 + wave];
  };
  auto step = [&](DeltaOperands<TPW>& x, int c) {
    floatx4 p = {0.f, 0.f, 0.f, 0.f}, p2 = p, o2 = p;
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      if (!EVEN && tile0 + i >= tiles) continue;      // (the same for the whole wave)
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][0], S[i][0], p, 0, 0, 0);
      p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][1], S[i][1], p2, 0, 0, 0);
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][2], S[i][2], p, 0, 0, 0);
      p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][3], S[i][3], p2, 0, 0, 0);
    }
    *reinterpret_cast<floatx4*>(&share[c & 1][wave][lane * 4]) = p + p2;
    // a barrier for LDS alone: __syncthreads would also wait for the loads that were asked for ahead. A buffer of shares is
    // read right behind its barrier and written again only behind the next one.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    floatx4 u = x.v, got[4];
    float part[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) got[w] = *reinterpret_cast<const floatx4*>(&share[c & 1][w][lane * 4]);
    if (c > 0) parts(c - 1, part);
    __builtin_amdgcn_sched_barrier(0);
    // (while the shares come; R holds - B W already: what is left of B U is B V')
    floatx4 o = {wave == 0 ? x.o : 0.f, wave == 1 ? x.o : 0.f, wave == 2 ? x.o : 0.f, wave == 3 ? x.o : 0.f};
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      if (!EVEN && tile0 + i >= tiles) continue;
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[i][0], S[i][0], o, 0, 0, 0);
      o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[i][1], S[i][1], o2, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[i][2], S[i][2], o, 0, 0, 0);
      o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[i][3], S[i][3], o2, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TPW; ++i) S[i] *= x.g[i];
    u -= ((got[0] + got[1]) + got[2]) + got[3];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < TPW; ++i)
        if (EVEN || tile0 + i < tiles) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kk[i][j], u[j], S[i], 0, 0, 0);
    ask(x);
    if (c > 0) emit(part, c - 1);            // (while the products are under way; written behind the last barrier but one)
    *reinterpret_cast<floatx4*>(&red[c & 1][wave][lane * 4]) = o + o2;
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) ask(ops[i]);
  int c = 0;
  for (; c + AHEAD <= chunks; c += AHEAD) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) step(ops[i], c + i);
  }
#pragma unroll
  for (int i = 0; i < AHEAD - 1; ++i)
    if (c + i < chunks) step(ops[i], c + i);
  __syncthreads();
  float part[4];
  parts(chunks - 1, part);
  emit(part, chunks - 1);
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = (tile0 + i) * 16 + grp * 4 + j;
      if (column && d < D) mine[d] = S[i][j];
    }
}

extern "C" int nhv_delta_chunks(const void* w, const void* r, const void* k, const void* v, const void* o, const void* decay, void* state,
                                void* out, const void* positions, const void* cu, const void* state_slots, int B, int H, int D, int E,
                                void* stream) {
  NHV_REQUIRE(B > 0 && H > 0 && D > 0 && E > 0 && D <= 256 && B <= 65535 && (E + 15) / 16 <= 65535, "delta_chunks: bad sizes B=%d H=%d D=%d E=%d",
              B, H, D, E);
  const DeltaChunks from = {(float*)w, (float*)r, (float*)k, (float*)v, (float*)o, (float*)decay};
  const int Dp = (D + 15) & ~15, tiles = Dp / 16, tpw = (tiles + 3) / 4;
  const dim3 grid(H, (E + 15) / 16, B);
  hipStream_t s = (hipStream_t)stream;
#define LAUNCH(TPW, EVEN)                                                                                               \
  hipLaunchKernelGGL((delta_chunks_kernel<TPW, EVEN>), grid, dim3(256), 0, s, from, (float*)state, (float*)out,           \
                     (const int*)positions, (const int*)cu, (const int*)state_slots, H, D, Dp, E)
#define BY_EVEN(TPW)                            \
  do {                                          \
    if (tiles == 4 * (TPW)) LAUNCH(TPW, true);  \
    else LAUNCH(TPW, false);                    \
  } while (0)
  if (tpw == 1) BY_EVEN(1);
  else if (tpw == 2) BY_EVEN(2);
  else if (tpw == 3) BY_EVEN(3);
  else BY_EVEN(4);
#undef BY_EVEN
#undef LAUNCH
  NHV_LAUNCH_CHECK("delta_chunks");
  return 0;
}
