// y[M, N] = x[M, K] . w[N, K]^T (+ bias[N]) in float, or a gate of two such products (w[2 N, K]: N gate rows, then N up rows), on the
// bfloat16 matrix cores, to float's precision.
//
// A float (times 2^16) is the sum of three bfloat16 numbers, exactly: what rounding to 8 bits gives, what that leaves rounded to
// 8 bits, and the rest (nhv_split_float.h). A product of two floats is then nine products of 8 bits by 8, each exact in float; six
// of them are summed. The three left out (middle x rest, rest x middle, rest x rest) are at most about 2^-24 of the product
// together, what rounding one float product may cost: a middle is at most 2^-8 of a number's power of two, a rest 2^-17 (1 + 2^-8 -
// 2^-17 times itself: 0.99 x 2^-24). One v_mfma_f32_16x16x32_bf16 sums 32 products in 16 clocks where the float
// instruction sums 4 in 32: six of them take 96 clocks for what took 256. The products of the largest parts and the five small ones
// have an accumulator each, which meet at a segment's end.
// Off from 64 bits, 2-norm over 2-norm, normal entries, K = 64, 1024, 2048, 3072, 6144: 4.8e-8, 8.6e-8, 1.06e-7, 1.23e-7, 1.69e-7
// (float matrix instructions: 8.4e-8, 2.11e-7, 2.93e-7, 3.56e-7, 5.0e-7).
//
// A row's result does not depend on how many rows there are: K is cut into 8 segments by K alone (a multiple of 32 long), a
// segment is summed in blocks of 32 k, and the segments are added in rising order. Which tile an output lies in changes
// nothing of that, so the tile may be chosen by the shape.
//
// What the factors 2^16 cost: one multiplication an entry taken apart, 3 % of a prompt of 517 tokens (0.6B shape), 1 % of decoding.
//
// The parts of an infinity are infinity and no numbers, and so are those of a number beyond 2^112. So an output that comes out
// infinite (sums beyond 2^96 do) or as no number is summed once more by plain float multiply-adds: that is what it is then.
// (Such inputs make every output of their row or column such a one.)
//
// Three kernels. Few rows, or few columns: a block is 8 waves and owns 16 RT rows by 16 CT columns, wave s sums segment s, and
// LDS adds the segments up. Both operands come straight from memory (a lane: 16 bytes of each half of a row's 128); all loads
// of a stage of U blocks of 32 k are asked for one stage ahead. What bounds it is what a compute unit takes in: a tile's time
// grows by 5.6 us a 3,072 k with every 16 rows of x or w that it reads (35 GB/s), whatever their product. Many rows: a block is
// 4 waves that share their operands' parts through LDS, 32 or 64 rows of x a block, see below. And where a product has few outputs and its
// reader adds parts up (a norm does), the segments go to blocks of their own and the sums over segments are left to that reader.
// The blocks of one column tile follow each other on one XCD, whose L2 then reads those rows of w once.
// A gated product takes tiles of gate rows and of their up rows in turn (two a wave), and a lane that has finished both writes
// the gate of them: what a kernel of its own made of the packed rows before (6 rows of 3,072: 4.1 us, 517: 5.5).
#include "nhv_common.h"
#include "nhv_gates.h"
#include "nhv_split_float.h"

#define SEGMENTS 8

__host__ __device__ static inline int segment_length(int K) { return ((K + SEGMENTS - 1) / SEGMENTS + 31) & ~31; }
__host__ __device__ static inline int segments(int K) { return (K + segment_length(K) - 1) / segment_length(K); }

// four entries of a row from column k on. WIDE: rows of a multiple of four entries on 16-byte boundaries; beyond K the row's
// last four (the caller puts zeros in their place), so that no load hangs on a condition: with conditions the compiler
// waits for all loads under way, and a stage is no longer asked for ahead.
template <bool WIDE>
__device__ __forceinline__ f32x4 four_of(const float* __restrict__ row, int k, int K) {
  if (WIDE) return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));
  f32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float e = row[min(k + j, K - 1)];
    v[j] = k + j < K ? e : 0.f;
  }
  return v;
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }

// Outputs (m, n), one a lane, of which the ``odd`` ones are made once more by plain float multiply-adds (see above): the wave takes one
// after the other, lane l the columns l, l + 64, ..., and stops where a lane's sum is no number. A row of x or of w with an entry that is no
// number settles all of the wave's outputs of that row. The order hangs on K alone. us, without such outputs, with one entry
// of x that is no number, with one column of sums beyond 2^96, with nothing but infinities, with nothing but sums beyond 2^96: 517 x 4096 . 1024
// 50, 50, 87, 697, 1,706; 6 x 1024 . 3072 11, 12, 24, 44, 222 (by one lane an output: 204 and 230 with one such entry, 5,600 and 283 with infinities).
__device__ __attribute__((noinline)) float plain_products(const float* __restrict__ x, const float* __restrict__ w, int K, float v, int m, int n, bool odd) {
  const int lane = threadIdx.x & 63;
  for (unsigned long long left = __ballot(odd); left;) {
    const int from = __ffsll(left) - 1, row = __shfl(m, from, NHV_WAVE), column = __shfl(n, from, NHV_WAVE);
    const float *xr = x + (size_t)row * K, *wr = w + (size_t)column * K;
    float sum = 0.f;
    bool x_none = false, w_none = false;
    for (int k0 = lane; k0 - lane < K; k0 += 4 * 64) {
      float a[4], b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = min(k0 + 64 * j, K - 1);
        a[j] = xr[k], b[j] = wr[k];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x_none |= a[j] != a[j], w_none |= b[j] != b[j];
        if (k0 + 64 * j < K) sum = fmaf(a[j], b[j], sum);
      }
      if (__any(sum != sum)) break;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, NHV_WAVE);
    x_none = __any(x_none), w_none = __any(w_none);
    const bool settled = lane == from || (x_none && m == row) || (w_none && n == column);
    if (odd && settled) v = sum;
    left &= ~__ballot(settled);
  }
  return v;
}

// PARTS: two waves a block, each with a segment of its own, whose sums are the result (times 2^32, [segment][M][N]).
template <int RT, int CT, int U, bool GATED, bool PARTS, bool WIDE>
__global__ __launch_bounds__(PARTS ? 128 : 64 * SEGMENTS) void gemm_float32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                     const float* __restrict__ bias, float* __restrict__ y,
                                                                     int M, int N, int K, int m_tiles, int n_tiles, NhvGate gate) {
  static_assert(!GATED || CT == 2, "a gate tile and its up tile");
  constexpr int COLS = GATED ? 16 : 16 * CT;             // outputs of a row
  __shared__ __attribute__((aligned(16))) float part[PARTS ? 1 : SEGMENTS][PARTS ? 1 : CT * 256];
  const int total = m_tiles * n_tiles, share = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);        // (consecutive blocks go round the 8 XCDs)
  if (tile >= total) return;
  const int m0 = (tile % m_tiles) * 16 * RT, n0 = (tile / m_tiles) * COLS;
  const int s = (threadIdx.x >> 6) + (PARTS ? 2 * blockIdx.y : 0), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int length = segment_length(K);
  const int begin = s * length, end = min(K, begin + length);
  const int active = segments(K);

  f32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (begin < end) {
    f32x4 low[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) low[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *xp[RT], *wp[CT];                        // (rows beyond the last are the last one: their results are dropped)
#pragma unroll
    for (int r = 0; r < RT; ++r) xp[r] = x + (size_t)min(m0 + 16 * r + r16, M - 1) * K;
#pragma unroll
    for (int c = 0; c < CT; ++c) wp[c] = w + (GATED ? (size_t)c * N + min(n0 + r16, N - 1) : (size_t)min(n0 + 16 * c + r16, N - 1)) * K;
    f32x4 a[2][U][RT][2], b[2][U][CT][2];
    auto ask = [&](int buf, int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int h = 0; h < 2; ++h) b[buf][u][c][h] = four_of<WIDE>(wp[c], k0 + 32 * u + 4 * g + 16 * h, K);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int h = 0; h < 2; ++h) a[buf][u][r][h] = four_of<WIDE>(xp[r], k0 + 32 * u + 4 * g + 16 * h, K);
      }
    };
    auto sum = [&](int buf, int u) {
      SplitFloats8 xs[RT], ws[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) ws[c] = split_floats<true>(b[buf][u][c][0], b[buf][u][c][1]);
#pragma unroll
      for (int r = 0; r < RT; ++r) xs[r] = split_floats<true>(a[buf][u][r][0], a[buf][u][r][1]);
#pragma unroll
      for (int step = 0; step < 6; ++step)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) split_product(step, xs[r], ws[c], acc[r][c], low[r][c]);
    };
    // the last stage: what lies beyond the segment is left out, or counts as zeros
    auto sum_last = [&](int buf, int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + 32 * u >= end) break;
        if (WIDE && k0 + 32 * u + 32 > end) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const bool in = k0 + 32 * u + 4 * g + 16 * h < end;      // (end is a multiple of four)
#pragma unroll
            for (int c = 0; c < CT; ++c)
              if (!in) b[buf][u][c][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < RT; ++r)
              if (!in) a[buf][u][r][h] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
        sum(buf, u);
      }
    };
    ask(0, begin);
    for (int k0 = begin;;) {
      if (k0 + 32 * U >= end) {
        sum_last(0, k0);
        break;
      }
      ask(1, k0 + 32 * U);
#pragma unroll
      for (int u = 0; u < U; ++u) sum(0, u);
      k0 += 32 * U;
      if (k0 + 32 * U >= end) {
        sum_last(1, k0);
        break;
      }
      ask(0, k0 + 32 * U);
#pragma unroll
      for (int u = 0; u < U; ++u) sum(1, u);
      k0 += 32 * U;
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[r][c] += low[r][c];
  }
  if (PARTS) {
    if (begin < end)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = m0 + 16 * r + 4 * g + i, n = n0 + 16 * c + r16;
            if (m < M && n < N) y[((size_t)s * M + m) * N + n] = acc[r][c][i];
          }
    return;
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (m0 + 16 * r >= M) break;                         // (the same for the whole block)
    if (r) __syncthreads();
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4*>(&part[s][(c * 64 + lane) * 4]) = acc[r][c];
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * COLS; i += 64 * SEGMENTS) {
      // (lane 16 g + n of a tile holds rows 4 g .. 4 g + 3 of column n)
      const int c = i % COLS, row = i / COLS, m = m0 + 16 * r + row, n = n0 + c;
      float v[GATED ? 2 : 1];
#pragma unroll
      for (int both = 0; both < (GATED ? 2 : 1); ++both) {
        const int at = (((c >> 4) + both) * 64 + (row >> 2) * 16 + (c & 15)) * 4 + (row & 3);
        v[both] = part[0][at];
        for (int p = 1; p < active; ++p) v[both] += part[p][at];
      }
      const bool in = m < M && n < N;
#pragma unroll
      for (int both = 0; both < (GATED ? 2 : 1); ++both) {
        const bool odd = in && !finite(v[both]);
        v[both] *= SPLIT_UNSCALE;
        if (__any(odd)) v[both] = plain_products(x, w, K, v[both], m, both * N + n, odd);
      }
      if (in) {
        if (bias) {
#pragma unroll
          for (int both = 0; both < (GATED ? 2 : 1); ++both) v[both] += bias[both * N + n];
        }
        y[(size_t)m * N + n] = GATED ? nhv_gated(v[0], v[GATED], gate) : v[0];
      }
    }
  }
}

template <int RT, int CT, int U, bool GATED, bool PARTS = false>
static void launch(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, const NhvGate& gate, hipStream_t s) {
  constexpr int COLS = GATED ? 16 : 16 * CT;
  const int m_tiles = (M + 16 * RT - 1) / (16 * RT), n_tiles = (N + COLS - 1) / COLS;
  const dim3 grid(8u * (unsigned)(((long long)m_tiles * n_tiles + 7) / 8), PARTS ? (segments(K) + 1) / 2 : 1), block(PARTS ? 128 : 64 * SEGMENTS);
  if (PARTS || (K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0))
    hipLaunchKernelGGL((gemm_float32_kernel<RT, CT, U, GATED, PARTS, true>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles, gate);
  else if constexpr (!PARTS)
    hipLaunchKernelGGL((gemm_float32_kernel<RT, CT, U, GATED, false, false>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles, gate);
}

// ---------------------------------------------------------------- many rows
// 4 waves, 2 x 2, a wave RT x CT tiles of 16 x 16; the parts of both operands through LDS in pieces of 32 k, two buffers, two
// pieces under way in registers: an entry is taken apart once a block. A wave takes every segment in turn and adds it to the
// total: the same sums in the same order as above. What bounds it is a block's chain of pieces (0.4 us each at 32 x 32). 32 x 32: for the
// middling numbers of rows and outputs whose larger tiles would leave units idle. 64 x 64: for more of them in rows that are not whole pieces of
// 32 columns on 16-byte boundaries, which the kernel below does not take: made to, it took 1,024 x 3072 . 1001 in 140 us and 517 x
// 4096 . 1176 in 55 (gated 104) where this one takes 85 and 56 (95).
#define PIECE 32
#define AHEAD 2
template <int RT, int CT, bool GATED, bool WIDE>
__global__ __launch_bounds__(256, RT * CT > 2 ? 3 : 4) void gemm_float32_tiles_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                                 int K, int m_tiles, int n_tiles, NhvGate gate) {
  static_assert(!GATED || CT == 2, "a gate tile and its up tile");
  constexpr int BM = 32 * RT, BN = 32 * CT, LOADS = (BM + BN) * PIECE / 4 / 256, PLANE = (BM + BN) * PIECE;
  __shared__ __attribute__((aligned(16))) bf16_t rows[2][3 * PLANE];
  const int total_tiles = m_tiles * n_tiles, share = (total_tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
  if (tile >= total_tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * (GATED ? BN / 2 : BN);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int mw = (wave >> 1) * 16 * RT, nw = (wave & 1) * 16 * CT;
  const int length = segment_length(K), at = (g ^ (r16 >> 2)) << 3;
  // what this thread brings of a piece: 16 bytes of rows x (first BM) and w
  const float* src[LOADS];
  const int col = (threadIdx.x & 7) * 4;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (threadIdx.x >> 3) + 32 * i;
    // (gated: 16 gate rows and their 16 up rows in turn)
    const int n = GATED ? n0 + ((r - BM) >> 5) * 16 + (r & 15) : n0 + r - BM, up = GATED ? (r >> 4) & 1 : 0;
    src[i] = r < BM ? x + (size_t)min(m0 + r, M - 1) * K : w + ((size_t)up * N + min(n, N - 1)) * K;
  }
  // where they go: lane group g of a product takes k = 4 g .. and 16 + 4 g .., 16 bytes together, whose place in the row's 64
  // turns with the row so that 16 rows lie in different banks
  const int r8 = threadIdx.x >> 3, to_row = r8 * PIECE + (((threadIdx.x & 3) ^ (r8 >> 2 & 3)) << 3) + ((threadIdx.x >> 2 & 1) << 2);
  f32x4 hold[AHEAD][LOADS];
  auto ask = [&](int i_hold, int k0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) hold[i_hold][i] = four_of<WIDE>(src[i], k0 + col, K);
  };
  auto put = [&](int buf, int i_hold, int k0) {
    if (WIDE && k0 + PIECE > K) {                        // (the same for the whole grid)
      asm volatile("");                                  // a real branch: not a selection in every piece
      if (k0 + col >= K)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) hold[i_hold][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const SplitFloats4 p = split_floats<true>(hold[i_hold][i]);
      bf16_t* to = &rows[buf][32 * i * PIECE + to_row];
      *reinterpret_cast<bf16x4*>(to) = p.high;
      *reinterpret_cast<bf16x4*>(to + PLANE) = p.middle;
      *reinterpret_cast<bf16x4*>(to + 2 * PLANE) = p.rest;
    }
  };
  f32x4 acc[RT][CT], low[RT][CT], total[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[r][c] = low[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      total[r][c] = f32x4{-0.f, -0.f, -0.f, -0.f};
    }
  auto close = [&] {                                     // a segment's end
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        total[r][c] += acc[r][c] + low[r][c];
        acc[r][c] = low[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  int left = length;                                     // of the segment
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) ask(d, d * PIECE);
  put(0, 0, 0);
  ask(0, AHEAD * PIECE);
  __syncthreads();
  for (int k0 = 0; k0 < K; k0 += AHEAD * PIECE) {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {                    // (piece d lies in buffer d)
      const int k = k0 + d * PIECE, buf = d;
      if (k >= K) break;
      SplitFloats8 a[RT], b[CT];
#pragma unroll
      for (int r = 0; r < RT; ++r) a[r] = split_at<PLANE>(&rows[buf][(mw + 16 * r + r16) * PIECE + at]);
#pragma unroll
      for (int c = 0; c < CT; ++c) b[c] = split_at<PLANE>(&rows[buf][(BM + nw + 16 * c + r16) * PIECE + at]);
#pragma unroll
      for (int step = 0; step < 6; ++step)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) split_product(step, a[r], b[c], acc[r][c], low[r][c]);
      left -= PIECE;
      if (left == 0) {
        left = length;
        asm volatile("");                                // (a real branch)
        close();
      }
      put(buf ^ 1, d ^ 1, k + PIECE);
      ask(d ^ 1, k + (1 + AHEAD) * PIECE);
      __syncthreads();
    }
  }
  if (left != length) close();                           // (the last segment is shorter and not added yet)
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; c += GATED ? 2 : 1) {
      const int n = n0 + (GATED ? nw / 2 : nw + 16 * c) + r16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + mw + 16 * r + 4 * g + i;
        const bool in = m < M && n < N;
        float v[GATED ? 2 : 1];
#pragma unroll
        for (int both = 0; both < (GATED ? 2 : 1); ++both) {
          const bool odd = in && !finite(total[r][c + both][i]);
          v[both] = total[r][c + both][i] * SPLIT_UNSCALE;
          if (__any(odd)) v[both] = plain_products(x, w, K, v[both], m, both * N + n, odd);
        }
        if (in) {
          if (bias) {
#pragma unroll
            for (int both = 0; both < (GATED ? 2 : 1); ++both) v[both] += bias[both * N + n];
          }
          y[(size_t)m * N + n] = GATED ? nhv_gated(v[0], v[GATED], gate) : v[0];
        }
      }
    }
}

template <int RT, int CT, bool GATED>
static void launch_tiles(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, const NhvGate& gate, hipStream_t s) {
  constexpr int COLS = GATED ? 16 * CT : 32 * CT;
  const int m_tiles = (M + 32 * RT - 1) / (32 * RT), n_tiles = (N + COLS - 1) / COLS;
  const dim3 grid(8u * (unsigned)(((long long)m_tiles * n_tiles + 7) / 8)), block(256);
  if (K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0)
    hipLaunchKernelGGL((gemm_float32_tiles_kernel<RT, CT, GATED, true>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles, gate);
  else
    hipLaunchKernelGGL((gemm_float32_tiles_kernel<RT, CT, GATED, false>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles, gate);
}

// The same with 32 x 32 outputs a matrix instruction, CT of them a wave: 64 rows by 64 CT columns a block. A 32x32x16 instruction leaves
// vector instructions three quarters of its 32 clocks, a 16x16x32 one next to nothing of its 16 (two waves of a SIMD, ns for two matrix
// and twelve vector instructions: 31 where 27 and 22 apart; 39 for as many products of the smaller kind). Two of them in a
// row sum eight k after eight k as one of the other kind does: the same bits.
// PARTS: a block sums one segment, whose sums are the result (times 2^32, [segment][M][N]): K over blocks where there are few outputs.
// What bounds it: a piece takes a block 0.8 us (24 matrix instructions a wave are 0.37, its 190 others as much), and two blocks on
// a unit hardly less each. Rows of LDS turn by their number / 4: 16-byte reads go in quarters of lanes 0-3, 12-15, 20-23, 24-27 and
// the like (by / 2: 8 % slower). Asked for LDS one piece ahead, with two barriers or a third buffer, it was no faster.
// us, tiles of 64 x 64 of 16x16x32 instructions in brackets: 517 x 4096 . 1024 47 (53), gated 517 x 3072 . 1024 56 (67), 300 x 6144 . 2048 106 (140),
// 1,500 x 12,288 . 2048 454 (550).
// Rows are whole pieces of 32 columns on 16-byte boundaries (whole_pieces).
//
// WAVES 8: 128 x 128 outputs, a wave 32 by 64. Half the loads and half the parts taken from floats a product, but what is read from LDS for
// it is the same, and eight waves that have all met wait for it: 1,125 clocks a piece, beside which nothing ran. So the middle parts
// of the next piece are read among this one's last products, behind a barrier that stands between its third and its fourth kind of
// product. Taken where its rounds of blocks are half of what the smaller tiles need (big_tiles). us, 64 x 128 and 128 x 128: 517 x 3072 . 1024 gated 60, 52 (read all at
// once 56), 416 rows 50, 45, 1,000 x 4096 . 1024 58, 52, 1,049 x 3,072 . 1024 56, 54; without the matrix instructions 46 for the 56, without loads 44, matrix
// instructions alone 34. Three pieces under way in registers: the same; 4 waves of 64 x 64, whose accumulators move between register files, 70.
template <int CT, bool GATED, bool PARTS, int WAVES>
__global__ __launch_bounds__(64 * WAVES, CT == 2 ? 2 : 3) void gemm_float32_blocks_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                                   const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                                                   int K, int m_tiles, int n_tiles, NhvGate gate) {
  static_assert(!GATED || (CT == 2 && !PARTS), "a gate tile and its up tile");
  static_assert(WAVES == 4 || !PARTS, "parts come from the smaller tiles");
  constexpr int BM = 16 * WAVES, BN = 64 * CT, LOADS = (BM + BN) / BM, PLANE = (BM + BN) * PIECE, OUT = GATED ? BN / 2 : BN, TOTALS = PARTS ? 1 : CT;
  __shared__ __attribute__((aligned(16))) bf16_t rows[2][3 * PLANE];
  const int total_tiles = m_tiles * n_tiles, share = (total_tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
  if (tile >= total_tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * OUT;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5;
  const int mw = (wave >> 1) * 32, nw = (wave & 1) * 32 * CT;
  const int length = segment_length(K), begin = PARTS ? blockIdx.y * length : 0, end = PARTS ? min(K, begin + length) : K;
  // what this thread brings of a piece: 16 bytes of each half of the 128 of rows row, row + BM, ...: an address that the wave shares, and
  // an offset (of less than 128 rows of less than 2^22 entries: 32 bits)
  const int col = (threadIdx.x & 3) * 4, row = threadIdx.x >> 2;
  const float* base[LOADS];
  uint32_t offset[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    // (gated: 32 gate rows and their 32 up rows in turn)
    const int b = row + BM * (i - 1), n = GATED ? n0 + (b >> 6) * 32 + (b & 31) : n0 + b;
    const int up = GATED ? __builtin_amdgcn_readfirstlane((b >> 5) & 1) : 0;
    base[i] = i == 0 ? x + (size_t)m0 * K : w + ((size_t)up * N + n0) * K;
    offset[i] = (uint32_t)(i == 0 ? min(row, M - 1 - m0) : min(n, N - 1) - n0) * (uint32_t)K;
  }
  const int to_row = row * PIECE + (((threadIdx.x & 3) ^ (row >> 2 & 3)) << 3);
  f32x4 hold[AHEAD][LOADS][2];
  auto ask = [&](int i_hold, int k0) {
    const int at = min(k0, K - PIECE);                     // (beyond the last piece it again, into registers that nobody reads)
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) hold[i_hold][i][h] = *reinterpret_cast<const f32x4*>(base[i] + at + (offset[i] + col + 16 * h));
  };
  auto put = [&](int buf, int i_hold, int i) {
    const SplitFloats8 p = split_floats<false>(hold[i_hold][i][0], hold[i_hold][i][1]);
    bf16_t* to = &rows[buf][BM * i * PIECE + to_row];
    *reinterpret_cast<bf16x8*>(to) = p.high;
    *reinterpret_cast<bf16x8*>(to + PLANE) = p.middle;
    *reinterpret_cast<bf16x8*>(to + 2 * PLANE) = p.rest;
  };
  f32x16 acc[CT], low[CT], total[TOTALS];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc[c][i] = low[c][i] = 0.f;
      if (!PARTS) total[c % TOTALS][i] = -0.f;
    }
  auto close = [&] {                                     // a segment's end
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      total[c % TOTALS] += acc[c] + low[c];
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[c][i] = low[c][i] = 0.f;
    }
  };
  // (a lane holds rows 8 (i / 4) + 4 half + i % 4 of column r32 of a tile)
  auto row_of = [&](int i) { return m0 + mw + 8 * (i >> 2) + 4 * half + (i & 3); };
  int left = length;                                     // of the segment
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) ask(d, begin + d * PIECE);
#pragma unroll
  for (int i = 0; i < LOADS; ++i) put(0, 0, i);
  ask(0, begin + AHEAD * PIECE);
  __syncthreads();
  int a_at[2], b_at[2];                                  // of 16 k: lane groups' 8 k are pieces 2 s and 2 s + 1
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_at[s] = (mw + r32) * PIECE + (((2 * s + half) ^ (r32 >> 2 & 3)) << 3);
    b_at[s] = (BM + nw + r32) * PIECE + (((2 * s + half) ^ (r32 >> 2 & 3)) << 3);
  }
  constexpr bool EARLY = WAVES == 8;                     // the middle parts are read a piece ahead
  auto part_of = [&](int buf, int at, int plane) { return *reinterpret_cast<const bf16x8*>(&rows[buf][at + plane * PLANE]); };
  SplitFloats8 a[2], b[2][CT];
  bf16x8 a_next[2], b_next[2][CT];
  auto read_middle = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      a_next[s] = part_of(buf, a_at[s], 1);
#pragma unroll
      for (int c = 0; c < CT; ++c) b_next[s][c] = part_of(buf, b_at[s] + 32 * c * PIECE, 1);
    }
  };
  if (EARLY) read_middle(0);
  for (int k0 = begin; k0 < end; k0 += AHEAD * PIECE) {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {                    // (piece d lies in buffer d)
      const int k = k0 + d * PIECE, buf = d;
      if (k >= end) break;
      // the parts in the order in which the products need them
      auto part = [&](int at, int plane) { return part_of(buf, at, plane); };
      if (EARLY) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          a[s].middle = a_next[s];
#pragma unroll
          for (int c = 0; c < CT; ++c) b[s][c].middle = b_next[s][c];
        }
      } else {
#pragma unroll
        for (int s = 0; s < 2; ++s) a[s].middle = part(a_at[s], 1);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int c = 0; c < CT; ++c) b[s][c].middle = part(b_at[s] + 32 * c * PIECE, 1);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) a[s].rest = part(a_at[s], 2);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < CT; ++c) b[s][c].high = part(b_at[s] + 32 * c * PIECE, 0);
#pragma unroll
      for (int s = 0; s < 2; ++s) a[s].high = part(a_at[s], 0);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < CT; ++c) b[s][c].rest = part(b_at[s] + 32 * c * PIECE, 2);
#pragma unroll
      for (int step = 0; step < 6; ++step) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int c = 0; c < CT; ++c) split_product(step, a[s], b[s][c], acc[c], low[c]);
        if (step < LOADS) put(buf ^ 1, d ^ 1, step);
        if (EARLY && step == LOADS - 1) ask(d ^ 1, k + (1 + AHEAD) * PIECE);
        if (EARLY && step == 2) {
          __syncthreads();
          read_middle(buf ^ 1);
        }
      }
      if (!EARLY) ask(d ^ 1, k + (1 + AHEAD) * PIECE);
      left -= PIECE;
      if (!PARTS && left == 0) {
        left = length;
        asm volatile("");                                // (a real branch)
        close();
      }
      if (!EARLY) __syncthreads();
    }
  }
  if (PARTS) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int n = n0 + nw + 32 * c + r32;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = row_of(i);
        if (m < M && n < N) y[((size_t)blockIdx.y * M + m) * N + n] = acc[c][i] + low[c][i];
      }
    }
    return;
  }
  if (left != length) close();                           // (the last segment is shorter and not added yet)
#pragma unroll
  for (int c = 0; c < CT; c += GATED ? 2 : 1) {
    const int n = n0 + (GATED ? nw / 2 : nw + 32 * c) + r32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = row_of(i);
      const bool in = m < M && n < N;
      float v[GATED ? 2 : 1];
#pragma unroll
      for (int both = 0; both < (GATED ? 2 : 1); ++both) {
        const float t = total[(c + both) % TOTALS][i];
        const bool odd = in && !finite(t);
        v[both] = t * SPLIT_UNSCALE;
        if (__any(odd)) v[both] = plain_products(x, w, K, v[both], m, both * N + n, odd);
      }
      if (in) {
        if (bias) {
#pragma unroll
          for (int both = 0; both < (GATED ? 2 : 1); ++both) v[both] += bias[both * N + n];
        }
        y[(size_t)m * N + n] = GATED ? nhv_gated(v[0], v[GATED], gate) : v[0];
      }
    }
  }
}

template <int CT, bool GATED, bool PARTS = false, int WAVES = 4>
static void launch_blocks(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, const NhvGate& gate, hipStream_t s) {
  constexpr int COLS = GATED ? 32 * CT : 64 * CT;
  const int m_tiles = (M + 16 * WAVES - 1) / (16 * WAVES), n_tiles = (N + COLS - 1) / COLS;
  const dim3 grid(8u * (unsigned)(((long long)m_tiles * n_tiles + 7) / 8), PARTS ? segments(K) : 1), block(64 * WAVES);
  hipLaunchKernelGGL((gemm_float32_blocks_kernel<CT, GATED, PARTS, WAVES>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles, gate);
}

static bool whole_pieces(const void* x, const void* w, int K) {
  return K % PIECE == 0 && K < (1 << 22) && (((uintptr_t)x | (uintptr_t)w) & 15) == 0;
}

// Every tile's time in units of what a compute unit needs for 16 rows of an operand, from the times of all tiles at 1 to 1,500
// rows of the 0.6B and 1.7B shapes' products. Tiles of 8 waves: rounds of 256 blocks times 16-row operands; the tiles through
// LDS: a floor (one block's chain of pieces) and what a block a compute unit adds (64 x 128: whole rounds). E.g. 17 x 6144 . 1024: 32 x 32 10.1 us,
// 16 x 32 14.0, 16 x 16 13.9; 130 x 2048 . 2048: 48 x 32 21.9 us, 32 x 32 33.7, 64 x 64 42.4; 517 x 4096 . 1024: 64 x 64 46, 64 x 128 50, 32 x 32
// through LDS 56; 1,500 x 4096 . 1024: 98, 90 and 147. Up to 16 rows LDS has nothing to share and is left out (6 x 151,936 . 1024: 116 us with 16 x 32,
// 135 through LDS). Not whole pieces: 64 x 64 of 16x16x32 instructions in place of both.
// 32 x 16, whose second 16 rows are few different ones at 17 rows and 16 at 32: 17 x 4096 . 4096 24.2 us, 16 x 32 27.4; 32 rows 29.2 and 28.1.
struct Choice {
  int tile;
  double cost;
};
// 64 x 64 of whole pieces: one block a unit, two, three; beyond, what a block adds (1,000 x 1024 . 3072 62 us, 32 x 32 through LDS 76; 256 x 4096 .
// 4096 83 and 102; 130 x 6144 . 2048 58 and 53; 700 x 2048 . 2048 59, 64 x 128 55).
static double square_tiles(long long blocks) {
  const double a_unit = blocks / 256.0;
  return a_unit <= 1 ? 11.2 : a_unit <= 2 ? 12.0 + 2.75 * a_unit : a_unit <= 3 ? 13.5 + 3.8 * a_unit : 1.8 + 7.7 * a_unit;
}
static double wide_tiles(long long blocks) { return fmax(15.2, 13.3 * (blocks <= 2048 ? (double)((blocks + 255) / 256) : blocks / 256.0) - 1.5); }
static Choice plain_tile(long long M, long long N, bool whole) {
  auto blocks = [&](long long m, long long n) { return ((M + m - 1) / m) * ((N + n - 1) / n); };
  auto rounds = [&](int rt, int ct) { return (double)((blocks(16 * rt, 16 * ct) + 255) / 256 * (rt + ct)); };
  const double none = 1e300;
  const double cost[8] = {rounds(1, 1), rounds(1, 2), M > 16 ? rounds(2, 2) : none, M > 32 ? rounds(3, 2) : none,
                          M > 16 ? fmax(9.0, 1.5 + 2.9 / 256 * blocks(32, 32)) : none,
                          M <= 16 ? none : whole ? square_tiles(blocks(64, 64)) : fmax(11.5, 4.5 + 7.7 / 256 * blocks(64, 64)),
                          M > 16 && M <= 32 ? rounds(2, 1) / 3 * (2.05 + 0.035 * M) : none,
                          M > 16 && whole ? wide_tiles(blocks(64, 128)) : none};
  Choice best = {0, cost[0]};
  for (int i = 1; i < 8; ++i)
    if (cost[i] < best.cost) best = {i, cost[i]};
  return best;
}
// a gate of two products: a column counting for two rows of w; through LDS only tiles with a pair a wave
static Choice gated_tile(long long M, long long N, bool whole) {
  auto blocks = [&](long long m, long long n) { return ((M + m - 1) / m) * ((N + n - 1) / n); };
  auto rounds = [&](int rt) { return (double)((blocks(16 * rt, 16) + 255) / 256 * (rt + 2)); };
  const double none = 1e300;
  const double cost[5] = {rounds(1), M > 16 ? rounds(2) : none, M > 32 ? rounds(3) : none,
                          M > 16 ? fmax(9.5, 3.0 + 4.9 / 256 * blocks(32, 32)) : none,
                          M <= 16 ? none : whole ? wide_tiles(blocks(64, 64)) : fmax(11.5, 4.5 + 7.7 / 256 * blocks(64, 32))};
  Choice best = {0, cost[0]};
  for (int i = 1; i < 5; ++i)
    if (cost[i] < best.cost) best = {i, cost[i]};
  return best;
}

// Whether tiles of 128 x 128 rows of x and of w (gated: 64 outputs) are the faster ones: where tiles of 64 x 128 need twice the rounds of
// 256 blocks that these do. Measured over 9,700 sizes (90 to 2,048 rows, 700 to 8,200 outputs of 256 to 4,096 columns; time over that of
// the choice without them): 1 round 0.86 and 0.88 gated, the worst 1.01 and 1.03; 2 rounds 0.87 and 0.91, 1.01; 3 0.89 and 0.91, 1.0; 4 and
// more 0.92, 1.08. Elsewhere 0.9 to 1.57 (2 rounds where the others need 2). A second round of smaller ones that is hardly begun is little
// to save: of 257 to 300 blocks up to 1.17. And of few columns a tile's first pieces and its sums are most of its time: 192 columns 0.97,
// 224 0.89, but 128 1.05, the worst 1.07 (1,004 x 2,592 12.2, 13.1 us).
constexpr int BEGUN = 44, BIG_COLUMNS = 192;
static bool big_tiles(long long M, long long N, int K, bool whole, bool gated) {
  const long long columns = gated ? 64 : 128, n = (N + columns - 1) / columns, blocks = (M + 127) / 128 * n, smaller = (M + 63) / 64 * n;
  const long long rounds = (blocks + 255) / 256;
  return whole && K >= BIG_COLUMNS && M > 64 && smaller > (2 * rounds - 1) * 256 + (rounds == 1 ? BEGUN : 0);
}

// The same for operands on 16-byte boundaries.
extern "C" int nhv_gemm_float32_big_tiles(int M, int N, int K, int gated) {
  return M > 0 && N > 0 && K > 0 && big_tiles(M, N, K, whole_pieces(nullptr, nullptr, K), gated != 0);
}

extern "C" int nhv_gemm_float32(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, void* stream) {
  NHV_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  NHV_REQUIRE(K < (1 << 30) && (((long long)M + 15) / 16) * (((long long)N + 15) / 16) < (1ll << 30), "gemm: too many rows (%d) for %d columns", M, N);
  hipStream_t s = (hipStream_t)stream;
  const float *xf = (const float*)x, *wf = (const float*)w, *bf = (const float*)bias;
  float* yf = (float*)y;
  const bool whole = whole_pieces(x, w, K);
  switch (big_tiles(M, N, K, whole, false) ? 8 : plain_tile(M, N, whole).tile) {
    case 0: launch<1, 1, 2, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 1: launch<1, 2, 1, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 2: launch<2, 2, 1, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 3: launch<3, 2, 1, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 4: launch_tiles<1, 1, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 5:
      if (whole) launch_blocks<1, false>(xf, wf, bf, yf, M, N, K, {}, s);
      else launch_tiles<2, 2, false>(xf, wf, bf, yf, M, N, K, {}, s);
      break;
    case 7: launch_blocks<2, false>(xf, wf, bf, yf, M, N, K, {}, s); break;
    case 8: launch_blocks<2, false, false, 8>(xf, wf, bf, yf, M, N, K, {}, s); break;
    default: launch<2, 1, 2, false>(xf, wf, bf, yf, M, N, K, {}, s);
  }
  NHV_LAUNCH_CHECK("gemm_float32");
  return 0;
}

// ---------------------------------------------------------------- parts that their reader adds up
// Which tiles make the parts of more than 16 rows: 64 x 64, or 64 x 128, which read x half as often, where few tiles of rows leave w the larger part of
// what is read (130 x 4096 . 2048 32.2 and 28.4 us, 517 x 1024 . 3072 33 and 38).
static bool wide_parts(long long M, long long N, int K) {
  return ((M + 63) / 64) * ((N + 63) / 64) * segments(K) > 3000 || (M > 64 && M <= 192 && N >= 2048);
}

// Whether a product is best left in parts for a norm that adds them up. What K over more blocks saves grows with K and is little where outputs alone
// make blocks enough; what it costs are the parts' way to memory and back, 8 entries for one, and the tiles' first pieces. Measured over 4,600 sizes (cold
// weights, product and norm; time in parts over finished). Up to 16 rows, 1 and 16: 1,024 outputs of 512 columns 0.96, 0.91, 2,048 of 512 1.09, 1.09, of 768 0.99, 0.92, of
// 3,072 0.85, 0.79; 2,560 of 1,536 1.14, 1.14, of 2,048 0.97, 1.02, of 3,072 0.92, 0.94; 4,096 of 3,072 1.03, 1.1. More rows: 512 columns 1.0 to 1.6
// everywhere, 2,048 and more 0.6 to 1.0 but for few rows of many outputs (17 rows, 4,096 outputs of 4,096 1.13, 5,120 of 8,192 1.04, 32 rows, 4,096 of 2,048 1.12, of 4,096 0.96, 40
// rows, 8,192 of 2,048 1.18). In between it hangs on how the tiles fill the chip either way (1,024 columns: 256 x 1536 0.81, 257 x 1280 1.2; 1,536 columns: 256 x
// 1536 0.68, 96 x 2304 1.14), for which both ways' times are estimated: the finished one's by its tile's cost, the parts' by a block's pieces and how many
// blocks a unit has, both with the norm that reads them (mean error 4 and 6 %). Of those sizes 3 % are now more than 3 % slower than by the better way, the worst 16 %.
static bool parts_pay(int M, int N, int K) {
  if (M <= 16) return N <= (K < 768 ? 1024 : K < 3072 ? 2048 : 2560);
  if ((long long)M * N > 1200000 || K < 768) return false;
  if (M <= 48 && N > 2560 && (N > 5120 || K < 1280 || (M <= 32 && (long long)M * K < 28ll * N))) return false;
  if (K >= 2048 || (K >= 1280 && N < 2304)) return true;
  const bool wide = wide_parts(M, N, K);
  if (wide ? K < 1024 : M <= 48 && N >= 2304) return false;
  const Choice tile = plain_tile(M, N, true);
  const double outputs = 1e-6 * M * N, finished = 5.2 + 5.5 / 3072 * tile.cost * K + (tile.tile == 4 ? 1.5 : 0.0) + 9.5 * outputs;
  const int count = segments(K), pieces = segment_length(K) / PIECE, columns = wide ? 128 : 64;
  const double a_unit = fmax(1.0, (double)((M + 63) / 64) * ((N + columns - 1) / columns) * count / 256);
  return (wide ? 8.9 + pieces * (0.76 * a_unit + 0.15) + 2.0 * a_unit + 1.0 * count * outputs : 7.1 + pieces * (0.43 * a_unit + 0.15) + 2.25 * count * outputs) < finished;
}

// How many parts (the segments of K) that are; 0: the product is best finished here.
extern "C" int nhv_gemm_float32_parts_count(const void* x, const void* w, int M, int N, int K) {
  return M > 0 && N > 0 && K >= 512 && whole_pieces(x, w, K) && parts_pay(M, N, K) ? segments(K) : 0;
}

// y[segments][M][N], times 2^32. Up to 16 rows two waves a block, each with all of a segment under way (one with half of it: 8.1 us where 7.0
// are kept at 1024 . 3072).
extern "C" int nhv_gemm_float32_parts(const void* x, const void* w, void* y, int M, int N, int K, void* stream) {
  NHV_REQUIRE(M > 0 && N > 0 && K > 0 && K % PIECE == 0 && K < (1 << 22), "gemm in parts: bad sizes M=%d N=%d K=%d (a multiple of %d)", M, N, K, PIECE);
  NHV_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "gemm in parts: rows off 16-byte boundaries");
  NHV_REQUIRE((((long long)M + 15) / 16) * (((long long)N + 15) / 16) < (1ll << 27), "gemm in parts: too many rows (%d) for %d columns", M, N);
  hipStream_t s = (hipStream_t)stream;
  const float *xf = (const float*)x, *wf = (const float*)w;
  float* yf = (float*)y;
  if (M <= 16) launch<1, 1, 4, false, true>(xf, wf, nullptr, yf, M, N, K, {}, s);
  else if (wide_parts(M, N, K)) launch_blocks<2, false, true>(xf, wf, nullptr, yf, M, N, K, {}, s);
  else launch_blocks<1, false, true>(xf, wf, nullptr, yf, M, N, K, {}, s);
  NHV_LAUNCH_CHECK("gemm_float32_parts");
  return 0;
}

// Eight neighbouring outputs of row m from their parts: the finished product's bits. The whole wave comes here; `in`: the lane has outputs.
__device__ __forceinline__ void finish_parts8(const float* __restrict__ parts, int count, size_t stride, const float* __restrict__ x,
                                              const float* __restrict__ w, int K, int m, int n, size_t at, bool in, float* v) {
  f32x4 part[SEGMENTS][2];
#pragma unroll
  for (int p = 0; p < SEGMENTS; ++p)                       // (all are asked for before the first is used; those beyond the last are it again)
#pragma unroll
    for (int h = 0; h < 2; ++h) part[p][h] = *reinterpret_cast<const f32x4*>(parts + (in ? min(p, count - 1) * stride + at : 0) + 4 * h);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float sum = part[0][e >> 2][e & 3];
#pragma unroll
    for (int p = 1; p < SEGMENTS; ++p)
      if (p < count) sum += part[p][e >> 2][e & 3];
    const bool odd = in && !finite(sum);
    v[e] = sum * SPLIT_UNSCALE;
    if (__any(odd)) v[e] = plain_products(x, w, K, v[e], m, n + e, odd);
  }
}

// residual += the product whose parts these are; y = the norm of the sum: what rmsnorm does with mode 1, bit for bit.
// 6 rows of 1,024 take 4.5 us in a recorded step, of the finished product 4.6; 517 rows 6.4 and 5.1.
template <int MAXC>
__global__ __launch_bounds__(1024) void add_parts_norm_float32_kernel(const float* __restrict__ parts, int count, const float* __restrict__ x,
                                                                      const float* __restrict__ xw, int K, float* __restrict__ residual,
                                                                      const float* __restrict__ w, float* __restrict__ y, int H, float eps) {
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * H, stride = (size_t)gridDim.x * H;
  const int nch = H / 8;
  float v[MAXC][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = threadIdx.x + c * blockDim.x;
    const bool in = ch < nch;
    f32x4 r[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) r[h] = *reinterpret_cast<const f32x4*>(residual + base + (in ? ch * 8 : 0) + 4 * h);
    finish_parts8(parts, count, stride, x, xw, K, blockIdx.x, ch * 8, base + ch * 8, in, v[c]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[c][e] = in ? v[c][e] + r[e >> 2][e & 3] : 0.f;
  }
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = threadIdx.x + c * blockDim.x;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (ch < nch) *reinterpret_cast<f32x4*>(residual + base + ch * 8 + 4 * h) = f32x4{v[c][4 * h], v[c][4 * h + 1], v[c][4 * h + 2], v[c][4 * h + 3]};
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += v[c][e] * v[c][e];
  }
  const float total = block_sum(ss, scratch);
  const float r = 1.0f / sqrtf(total / (float)H + eps);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = threadIdx.x + c * blockDim.x;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (ch < nch) {
        const f32x4 g = *reinterpret_cast<const f32x4*>(w + ch * 8 + 4 * h);
        *reinterpret_cast<f32x4*>(y + base + ch * 8 + 4 * h) =
            f32x4{v[c][4 * h] * r * g[0], v[c][4 * h + 1] * r * g[1], v[c][4 * h + 2] * r * g[2], v[c][4 * h + 3] * r * g[3]};
      }
  }
}

// x[T, K] and xw[H, K]: the product's operands, from which outputs that are not finite are made once more
extern "C" int nhv_add_parts_norm_float32(const void* parts, int count, const void* x, const void* xw, int K, void* residual, const void* w, void* y,
                                          int T, int H, float eps, void* stream) {
  NHV_REQUIRE(T > 0 && H > 0 && H % 8 == 0 && H <= 16384 && K > 0, "add_parts_norm: bad sizes T=%d H=%d K=%d", T, H, K);
  NHV_REQUIRE(count == segments(K), "add_parts_norm: %d parts of a product over %d", count, K);
  NHV_REQUIRE((((uintptr_t)parts | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)y) & 15) == 0, "add_parts_norm: rows off 16-byte boundaries");
  const int nch = H / 8, threads = nch <= 1024 ? (nch + 63) / 64 * 64 : 1024;
  auto kernel = nch <= 1024 ? add_parts_norm_float32_kernel<1> : add_parts_norm_float32_kernel<2>;
  hipLaunchKernelGGL(kernel, dim3(T), dim3(threads), 0, (hipStream_t)stream, (const float*)parts, count, (const float*)x, (const float*)xw, K,
                     (float*)residual, (const float*)w, (float*)y, H, eps);
  NHV_LAUNCH_CHECK("add_parts_norm_float32");
  return 0;
}

// y[M, N] = the product whose parts these are, one output a lane, a row's lanes in whole waves
__global__ __launch_bounds__(256) void sum_parts_float32_kernel(const float* __restrict__ parts, int count, const float* __restrict__ x,
                                                                const float* __restrict__ w, int K, float* __restrict__ y, int M, int N) {
  const int n = blockIdx.y * 256 + threadIdx.x;
  for (int m = blockIdx.x; m < M; m += gridDim.x) {
    const bool in = n < N;
    float v = 0.f;
    if (in) {
      v = parts[(size_t)m * N + n];
      for (int p = 1; p < count; ++p) v += parts[((size_t)p * M + m) * N + n];
    }
    const bool odd = in && !finite(v);
    v *= SPLIT_UNSCALE;
    if (__any(odd)) v = plain_products(x, w, K, v, m, n, odd);
    if (in) y[(size_t)m * N + n] = v;
  }
}

extern "C" int nhv_sum_parts_float32(const void* parts, int count, const void* x, const void* w, int K, void* y, int M, int N, void* stream) {
  NHV_REQUIRE(M > 0 && N > 0 && N < (1 << 23) && K > 0 && count == segments(K), "sum_parts: %d parts of a product M=%d N=%d K=%d", count, M, N, K);
  hipLaunchKernelGGL(sum_parts_float32_kernel, dim3(M < 4096 ? M : 4096, (N + 255) / 256), dim3(256), 0, (hipStream_t)stream, (const float*)parts, count,
                     (const float*)x, (const float*)w, K, (float*)y, M, N);
  NHV_LAUNCH_CHECK("sum_parts_float32");
  return 0;
}

// Gates of whole pieces whose 64 x 64 tiles (64 x 128 of w) are best halved, by the kernel of 16x16x32 instructions: a block of the larger ones takes 4 us more
// before its first product, which short rows do not make up where half of the last round's units have nothing to do. us, larger and halved: 200 x
// 6144 of 256, 512, 1,024, 2,048 and 4,096 columns 22.4, 32.6, 53.9, 96.5, 183 and 19.7, 29.9, 50.9, 93.6, 178; 700 x 3072 34.5, 48.4, 81.9, 151, 281 and
// 28.9, 45.7, 80.1, 151, 287; in one round, 200 x 3072 16.6, 22.4, 35.0 and 14.0, 21.4, 36.2, 256 x 2048 of
// 768 and 1,024 25.1, 29.3 and 22.4, 27.4 (of 256 columns 32 x 32 are the faster ones with fewer halves than 1.4 a unit: 600 x 1024 13.2, halved 15.3).
static bool halved(long long M, long long N, int K) {
  const long long m = (M + 63) / 64, rounds = (m * ((N + 63) / 64) + 255) / 256, halves = m * ((N + 31) / 32);
  return K <= 1024 && (rounds == 1 ? (K < 512 ? halves > 358 : halves <= 256) : rounds <= 3 && halves <= 256 * (2 * rounds - 1));
}

// Whether the gate is best made in the product's kernel (1), or of the packed product's rows by a kernel of its own (0). A block takes both
// rows of w of an output, so a gated product of few outputs has half the packed one's blocks and as many more units idle: us at 1 and
// 17 rows, here and packed (before this kernel was there): 512 of 8,192 columns 38.1, 47.3 and 25.8, 35.8 (25.4, 35.5); 1,024 of 3,072 18.6,
// 21.8 and 15.0, 19.0 (14.2, 18.5); 2,048 of 6,144 32.8, 38.6 and 25.4, 40.8 (24.9, 36.7); 2,560 of 9,728 48.2, 62.8 and 50.8, 64.6 (59.1, 80.5);
// 3,072 of 1,024 10.8, 13.4 and 12.5, 15.1 (13.0, 16.4). A unit of the costs above takes 5.6 us a 3,072 columns, five times that where rows come
// entry by entry (1,000 of 1,001 at 1 row 20.8 and 13.4), the gate's kernel 2 and more (in a recorded step 4).
extern "C" int nhv_gemm_float32_gated_pays(const void* x, const void* w, int M, int N, int K) {
  const bool wide = K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
  const bool whole = whole_pieces(x, w, K);
  if (big_tiles(M, N, K, whole, true)) return 1;              // (as many blocks as the packed product)
  const bool halves = whole && halved(M, N, K);
  const Choice gated = gated_tile(M, N, whole && !halves);
  if (halves && gated.tile == 4) return 1;                 // (the packed product's larger blocks cost the same 4 us more: 1,000 x 1024 of 256 15.6 here, packed 21.2)
  return (gated.cost - plain_tile(M, 2ll * N, whole).cost) * (wide ? 5.6 : 28.0) * K / 3072 <= 2.0;
}

extern "C" int nhv_gemm_float32_gated(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int act, float limit,
                                      float alpha, float offset, void* stream) {
  NHV_REQUIRE(M > 0 && N > 0 && K > 0, "gated gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  NHV_REQUIRE(K < (1 << 30) && N < (1 << 30) && (((long long)M + 15) / 16) * (((long long)N + 15) / 16) < (1ll << 30),
              "gated gemm: too many rows (%d) for %d columns", M, N);
  NHV_REQUIRE(act >= 0 && act <= 2, "gated gemm: unknown gate %d", act);
  hipStream_t s = (hipStream_t)stream;
  const NhvGate gate = {act, limit, alpha, offset};
  const float *xf = (const float*)x, *wf = (const float*)w, *bf = (const float*)bias;
  float* yf = (float*)y;
  const bool big = big_tiles(M, N, K, whole_pieces(x, w, K), true), whole = whole_pieces(x, w, K) && !halved(M, N, K);
  switch (big ? 5 : gated_tile(M, N, whole).tile) {
    case 0: launch<1, 2, 1, true>(xf, wf, bf, yf, M, N, K, gate, s); break;
    case 1: launch<2, 2, 1, true>(xf, wf, bf, yf, M, N, K, gate, s); break;
    case 2: launch<3, 2, 1, true>(xf, wf, bf, yf, M, N, K, gate, s); break;
    case 3: launch_tiles<1, 2, true>(xf, wf, bf, yf, M, N, K, gate, s); break;
    case 5: launch_blocks<2, true, false, 8>(xf, wf, bf, yf, M, N, K, gate, s); break;
    default:
      if (whole) launch_blocks<2, true>(xf, wf, bf, yf, M, N, K, gate, s);
      else launch_tiles<2, 2, true>(xf, wf, bf, yf, M, N, K, gate, s);
  }
  NHV_LAUNCH_CHECK("gemm_float32_gated");
  return 0;
}
