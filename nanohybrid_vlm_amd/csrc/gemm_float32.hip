// y[M, N] = x[M, K] . w[N, K]^T (+ bias[N]) in float on the float matrix cores (v_mfma_f32_16x16x4_f32: every product and
// sum in 32 bits).
//
// A row's result does not depend on how many rows there are: K is cut into 8 segments by K alone (a multiple of 16 long), a
// segment is summed in blocks of 16 k, four matrix instructions a block (instruction j takes k = 4 g + j, g = 0..3), and the
// segments are added in rising order. Which tile an output lies in changes nothing of that, so the tile may be chosen by
// the shape.
//
// Two kernels. Up to some tens of rows, or few columns: a block is 8 waves and owns 16 RT rows by 16 CT columns, wave s sums
// segment s, and LDS adds the segments up. Both operands come straight from memory in the instructions' own layout (a lane:
// 16 bytes of one row), each row of x and w read once per block and by one wave only, so there is nothing for LDS to share;
// all loads of a stage of U blocks are asked for one stage ahead. Few rows are bound by the read of w (one row: 1024 x 151,936
// 113 us, 5.5 TB/s; 1024 x 4096 5.4 us) and, where the matrix is small, by the way there and back. Many rows: a block is 4
// waves that share their operands through LDS, see below; bound by the matrix cores and the last round of blocks (2,048 x
// 1024 . 4096: 160 us, 107 TFLOP/s; 517 rows 57 us). The kernel before this one (64 x 64 tiles, no matrix cores) took 197 us
// for one row and 248 for 517 on the mean of the 0.6B shape's layers.
// The blocks of one column tile follow each other on one XCD, whose L2 then reads those rows of w once.
#include "nhv_common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SEGMENTS 8

__host__ __device__ static inline int segment_length(int K) { return ((K + SEGMENTS - 1) / SEGMENTS + 15) & ~15; }

// four entries of a row from column k on. WIDE: rows of a multiple of four entries on 16-byte boundaries; beyond K the row's
// last four (the caller puts zeros in their place), so that no load hangs on a condition: with conditions the compiler
// waits for all loads under way, and a stage is no longer asked for ahead (47 us in place of 13 for 40 x 3072 . 1024).
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

template <int RT, int CT, int U, bool WIDE>
__global__ __launch_bounds__(64 * SEGMENTS) void gemm_float32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                     const float* __restrict__ bias, float* __restrict__ y,
                                                                     int M, int N, int K, int m_tiles, int n_tiles) {
  __shared__ __attribute__((aligned(16))) float part[SEGMENTS][CT * 256];
  const int total = m_tiles * n_tiles, share = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);        // (consecutive blocks go round the 8 XCDs)
  if (tile >= total) return;
  const int m0 = (tile % m_tiles) * 16 * RT, n0 = (tile / m_tiles) * 16 * CT;
  const int s = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int length = segment_length(K);
  const int begin = s * length, end = min(K, begin + length);
  const int active = (K + length - 1) / length;

  f32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (begin < end) {
    const float *xp[RT], *wp[CT];                        // (rows beyond the last are the last one: their results are dropped)
#pragma unroll
    for (int r = 0; r < RT; ++r) xp[r] = x + (size_t)min(m0 + 16 * r + r16, M - 1) * K;
#pragma unroll
    for (int c = 0; c < CT; ++c) wp[c] = w + (size_t)min(n0 + 16 * c + r16, N - 1) * K;
    f32x4 a[2][U][RT], b[2][U][CT];
    auto ask = [&](int buf, int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int c = 0; c < CT; ++c) b[buf][u][c] = four_of<WIDE>(wp[c], k0 + 16 * u + 4 * g, K);
#pragma unroll
        for (int r = 0; r < RT; ++r) a[buf][u][r] = four_of<WIDE>(xp[r], k0 + 16 * u + 4 * g, K);
      }
    };
    auto sum = [&](int buf) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c)
              acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[buf][u][r][j], b[buf][u][c][j], acc[r][c], 0, 0, 0);
    };
    // the last stage: what lies beyond the segment counts as zeros (which change no sum)
    auto sum_last = [&](int buf, int k0) {
      if (k0 + 16 * U > end) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool in = k0 + 16 * u + 4 * g < end;      // (WIDE: end is a multiple of four)
          if (WIDE || k0 + 16 * u >= end) {
#pragma unroll
            for (int c = 0; c < CT; ++c)
              if (!in) b[buf][u][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < RT; ++r)
              if (!in) a[buf][u][r] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
      sum(buf);
    };
    ask(0, begin);
    for (int k0 = begin;;) {
      if (k0 + 16 * U >= end) {
        sum_last(0, k0);
        break;
      }
      ask(1, k0 + 16 * U);
      sum(0);
      k0 += 16 * U;
      if (k0 + 16 * U >= end) {
        sum_last(1, k0);
        break;
      }
      ask(0, k0 + 16 * U);
      sum(1);
      k0 += 16 * U;
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (m0 + 16 * r >= M) break;                         // (the same for the whole block)
    if (r) __syncthreads();
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4*>(&part[s][(c * 64 + lane) * 4]) = acc[r][c];
    __syncthreads();
    for (int i = threadIdx.x; i < CT * 256; i += 64 * SEGMENTS) {
      // (lane 16 g + n of a tile holds rows 4 g .. 4 g + 3 of column n)
      const int c = i % (CT * 16), row = i / (CT * 16);
      const int at = ((c >> 4) * 64 + (row >> 2) * 16 + (c & 15)) * 4 + (row & 3);
      float v = part[0][at];
      for (int p = 1; p < active; ++p) v += part[p][at];
      const int m = m0 + 16 * r + row, n = n0 + c;
      if (m < M && n < N) y[(size_t)m * N + n] = bias ? v + bias[n] : v;
    }
  }
}

template <int RT, int CT, int U>
static void launch(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, hipStream_t s) {
  const int m_tiles = (M + 16 * RT - 1) / (16 * RT), n_tiles = (N + 16 * CT - 1) / (16 * CT);
  const dim3 grid(8u * (unsigned)(((long long)m_tiles * n_tiles + 7) / 8)), block(64 * SEGMENTS);
  if (K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0)
    hipLaunchKernelGGL((gemm_float32_kernel<RT, CT, U, true>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles);
  else
    hipLaunchKernelGGL((gemm_float32_kernel<RT, CT, U, false>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles);
}

// ---------------------------------------------------------------- many rows
// 4 waves, 2 x 2, a wave RT x CT tiles of 16 x 16; both operands through LDS in pieces of 32 k, two buffers, the next
// piece under way in registers while this one is summed. A wave takes every segment in turn and adds it to the total: the
// same sums in the same order as above.
#define PIECE 32
template <int RT, int CT, bool WIDE>
__global__ __launch_bounds__(256) void gemm_float32_tiles_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                                 int K, int m_tiles, int n_tiles) {
  constexpr int BM = 32 * RT, BN = 32 * CT, STRIDE = PIECE + 4, LOADS = (BM + BN) * PIECE / 4 / 256;
  __shared__ __attribute__((aligned(16))) float rows[2][(BM + BN) * STRIDE];
  const int total_tiles = m_tiles * n_tiles, share = (total_tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
  if (tile >= total_tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int mw = (wave >> 1) * 16 * RT, nw = (wave & 1) * 16 * CT;
  const int length = segment_length(K);
  // what this thread brings of a piece: 16 bytes of rows x (first BM) and w
  const float* src[LOADS];
  const int col = (threadIdx.x & 7) * 4;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (threadIdx.x >> 3) + 32 * i;
    src[i] = r < BM ? x + (size_t)min(m0 + r, M - 1) * K : w + (size_t)min(n0 + r - BM, N - 1) * K;
  }
  f32x4 hold[LOADS];
  auto ask = [&](int k0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) hold[i] = four_of<WIDE>(src[i], k0 + col, K);
  };
  auto put = [&](int buf, int k0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (WIDE && k0 + col >= K) hold[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(&rows[buf][((threadIdx.x >> 3) + 32 * i) * STRIDE + col]) = hold[i];
    }
  };
  f32x4 acc[RT][CT], total[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      total[r][c] = f32x4{-0.f, -0.f, -0.f, -0.f};
    }
  int left = length;                                     // of the segment
  ask(0);
  put(0, 0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += PIECE) {
    ask(k0 + PIECE);
#pragma unroll
    for (int h = 0; h < PIECE; h += 16) {
      f32x4 a[RT], b[CT];
#pragma unroll
      for (int r = 0; r < RT; ++r) a[r] = *reinterpret_cast<const f32x4*>(&rows[buf][(mw + 16 * r + r16) * STRIDE + h + 4 * g]);
#pragma unroll
      for (int c = 0; c < CT; ++c) b[c] = *reinterpret_cast<const f32x4*>(&rows[buf][(BM + nw + 16 * c + r16) * STRIDE + h + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r][j], b[c][j], acc[r][c], 0, 0, 0);
      left -= 16;
      if (left == 0) {
        left = length;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            total[r][c] += acc[r][c];
            acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
    put(buf ^ 1, k0 + PIECE);
    __syncthreads();
    buf ^= 1;
  }
  const bool rest = (K + 15) / 16 * 16 % length != 0;    // (the last segment is shorter and not added yet)
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      if (rest) total[r][c] += acc[r][c];
      const int n = n0 + nw + 16 * c + r16;
      const float add = bias && n < N ? bias[n] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + mw + 16 * r + 4 * g + i;
        if (m < M && n < N) y[(size_t)m * N + n] = bias ? total[r][c][i] + add : total[r][c][i];
      }
    }
}

template <int RT, int CT>
static void launch_tiles(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, hipStream_t s) {
  const int m_tiles = (M + 32 * RT - 1) / (32 * RT), n_tiles = (N + 32 * CT - 1) / (32 * CT);
  const dim3 grid(8u * (unsigned)(((long long)m_tiles * n_tiles + 7) / 8)), block(256);
  if (K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0)
    hipLaunchKernelGGL((gemm_float32_tiles_kernel<RT, CT, true>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles);
  else
    hipLaunchKernelGGL((gemm_float32_tiles_kernel<RT, CT, false>), grid, block, 0, s, x, w, bias, y, M, N, K, m_tiles, n_tiles);
}

extern "C" int nhv_gemm_float32(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, void* stream) {
  NHV_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  NHV_REQUIRE(K < (1 << 30) && (((long long)M + 15) / 16) * (((long long)N + 15) / 16) < (1ll << 30), "gemm: too many rows (%d) for %d columns", M, N);
  hipStream_t s = (hipStream_t)stream;
  const float *xf = (const float*)x, *wf = (const float*)w, *bf = (const float*)bias;
  float* yf = (float*)y;
  // Blocks that a tile of m rows and n columns gives. The largest tile that still fills the chip is the fastest (per output it
  // reads the least); the lines lie where the times of the 0.6B and 1.7B shapes' products cross (1 to 2,048 rows, every tile
  // timed): e.g. 517 x 1024 . 4096 64.5 us with 64 x 64 tiles (576 blocks), 57.5 with 32 x 64; 260 x 6144 . 2048 164 us with
  // 32 x 64 (288 blocks), 138 with 8 waves on 32 x 32; 40 x 3072 . 1024 25 us with 32 x 32, 19 with 32 x 16, 14 with 16 x 16.
  auto blocks = [&](long long m, long long n) { return ((M + m - 1) / m) * ((N + n - 1) / n); };
  if (M <= 16) launch<1, 1, 4>(xf, wf, bf, yf, M, N, K, s);
  else if (blocks(64, 64) >= 640) launch_tiles<2, 2>(xf, wf, bf, yf, M, N, K, s);
  else if (blocks(32, 64) >= 400) launch_tiles<1, 2>(xf, wf, bf, yf, M, N, K, s);
  else if (blocks(32, 32) >= 150) launch<2, 2, 2>(xf, wf, bf, yf, M, N, K, s);
  else if (blocks(32, 16) >= 150) launch<2, 1, 4>(xf, wf, bf, yf, M, N, K, s);
  else launch<1, 1, 4>(xf, wf, bf, yf, M, N, K, s);
  NHV_LAUNCH_CHECK("gemm_float32");
  return 0;
}
