// y[M, N] = x[M, K] . w[N, K]^T in bfloat16 for 17 to 128 rows: as float parts whose sum is the product, or as a gate of two
// products (w[2 N, K]: N gate rows, then N up rows).
//
// With so many rows a compute unit takes in as much of x as of w, and what bounds a product is how fast it takes them in: lines of
// 16 rows by 64 bytes, as the matrix instructions want their operands, come at 17 GB/s a unit, pieces of 256 bytes a row at 27
// to 35. So both operands go through LDS (global_load_lds, no registers) in chunks of 128 columns, in a ring of three or two
// chunks; a block is 8 waves, of which four share a chunk's 128 columns and two the tiles of w, and a chunk costs one barrier.
// Every byte in LDS is read once or twice. And K is cut over blocks where N gives too few of them or too little of w to each: a
// block then writes a float part, and who reads the product adds the parts up (a norm, the rotation: gemm parts in
// elementwise.hip). Parts are [splits][M][N], in rising order of K.
// Bank conflicts: a row's piece p of 16 bytes lies at place p ^ (row & 15), which costs nothing, since a lane chooses what it brings.
// us, and what the vendor's library takes by its best algorithm (with the gate's own kernel for gated products), cold weights: 64
// rows, 8B shape: qkv 15.5, 18.1; o 11.5, 14.0; gated 41.0, 50.0; down 25.6, 33.1; 79 rows, 4B shape: 13.5, 15.1; 10.8, 12.8; 31.1,
// 32.1; 18.1, 24.8; 32 rows, 0.6B shape: 4.5, 5.7; 3.9, 5.6; 6.4, 8.7; 4.3, 6.4.
#include "nhv_common.h"
#include "nhv_gates.h"
#include "nhv_lines.h"

namespace lines {

typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CHUNK = 128, PIECES = CHUNK / 8, ROWS_A_LOAD = 64 / PIECES;        // columns; 16-byte pieces and rows a wave's load

constexpr int lds_rows(int mt, int nt) { return (16 * (mt + nt) + 8 * ROWS_A_LOAD - 1) / (8 * ROWS_A_LOAD) * (8 * ROWS_A_LOAD); }
constexpr int stage_bytes(int mt, int nt) { return lds_rows(mt, nt) * CHUNK * 2; }
constexpr int stages(int mt, int nt) { return 3 * stage_bytes(mt, nt) <= 160 * 1024 ? 3 : 2; }

// MT tiles of 16 rows of x, NT of w (gated: NT / 2 gate tiles, then their up tiles).
template <int MT, int NT, bool GATED>
__global__ __launch_bounds__(512) void gemm_lines_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                                         void* __restrict__ y, int M, int N, int K, int splits, NhvGate gate) {
  constexpr int OUT = GATED ? NT / 2 : NT, BOTH = GATED ? 2 : 1, ROWS = lds_rows(MT, NT), LOADS = ROWS / ROWS_A_LOAD / 8, NB = stages(MT, NT);
  constexpr int MINE = (NT + 1) / 2;                                 // tiles of w a wave
  extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * OUT, split = blockIdx.y;
  const int chunks = K / CHUNK, c0 = (int)((long long)chunks * split / splits), c1 = (int)((long long)chunks * (split + 1) / splits);
  // what this lane brings of a chunk. Rows beyond the matrices are their last ones (their results are dropped).
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (i * 8 + wave) * ROWS_A_LOAD + lane / PIECES, tile = row >> 4;
    const bf16_t* from = tile < NT ? w + ((size_t)(GATED && tile >= OUT ? N : 0) + min(n0 + 16 * (tile % OUT) + (row & 15), N - 1)) * K
                                   : x + (size_t)min(row - 16 * NT, M - 1) * K;
    src[i] = from + ((lane % PIECES) ^ (row & 15)) * 8;
  }
  const uint32_t ring_at = nhv_lds_address(ring);
  const int first = c1 - c0 < 16 ? 0 : nhv_first_chunk(blockIdx.x, c1 - c0, K);       // (short splits lie apart already: 11.5 us against 12.0)
  auto ask = [&](int buf, int c) {
    const size_t k = (size_t)(c0 + nhv_chunk(first, c - c0, c1 - c0)) * CHUNK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const uint32_t to = ring_at + buf * stage_bytes(MT, NT) + (i * 8 + wave) * 1024;
      if (GATED && (i + 1) * 8 * ROWS_A_LOAD <= 16 * NT) nhv_load_to_lds<true>(to, src[i] + k);
      else nhv_load_to_lds<false>(to, src[i] + k);
    }
  };
  f32x4 acc[MINE][MT];
#pragma unroll
  for (int t = 0; t < MINE; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ks = wave & 3, half = wave >> 2, at = (((ks * 4 + g) ^ r16) << 3) + r16 * CHUNK;
#pragma unroll
  for (int i = 0; i < NB - 1; ++i) ask(i, c0 + i);
  int buf = 0;
  for (int c = c0; c < c1; ++c) {
    // this wave's loads of chunk c have arrived; behind the barrier everyone's have, and everyone has read chunk c - 1, whose
    // place the next load takes
    nhv_wait_and_meet<(NB - 2) * LOADS>();
    ask(buf == 0 ? NB - 1 : buf - 1, c + NB - 1);
    const bf16_t* now = ring + buf * (ROWS * CHUNK) + at;
    bf16x8 a[MINE], b[MT];
#pragma unroll
    for (int t = 0; t < MINE; ++t) a[t] = *reinterpret_cast<const bf16x8*>(now + min(half * MINE + t, NT - 1) * 16 * CHUNK);
#pragma unroll
    for (int m = 0; m < MT; ++m) b[m] = *reinterpret_cast<const bf16x8*>(now + (NT + m) * 16 * CHUNK);
#pragma unroll
    for (int t = 0; t < MINE; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[m], a[t], acc[t][m], 0, 0, 0);
    buf = buf == NB - 1 ? 0 : buf + 1;
  }
  nhv_wait_and_meet<0>();                                            // (the ring becomes room for the sums)
  // the sums of the four waves that share a tile's columns, in their order
  float* part = reinterpret_cast<float*>(ring);                      // [gate, up][MT][4][256]
#pragma unroll
  for (int p = 0; p < OUT; ++p) {
    if (p) __syncthreads();
#pragma unroll
    for (int both = 0; both < BOTH; ++both)
#pragma unroll
      for (int t = 0; t < MINE; ++t)
        if (half * MINE + t == p + both * OUT)
#pragma unroll
          for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&part[((both * MT + m) * 4 + ks) * 256 + lane * 4]) = acc[t][m];
    __syncthreads();
    for (int i = threadIdx.x; i < 256 * MT; i += 512) {
      // (lane 16 g + n of a tile holds rows 4 g .. 4 g + 3 of column n)
      const int row = i >> 4, col = i & 15, n = n0 + 16 * p + col, e = ((row & 15) >> 2) * 64 + col * 4 + (row & 3);
      if (row >= M || n >= N) continue;
      float v[BOTH];
#pragma unroll
      for (int both = 0; both < BOTH; ++both) {
        const float* from = &part[(both * MT + (row >> 4)) * 1024 + e];
        v[both] = ((from[0] + from[256]) + from[512]) + from[768];
        if (GATED && bias) v[both] += (float)bias[(size_t)both * N + n];
      }
      if (GATED) ((bf16_t*)y)[(size_t)row * N + n] = (bf16_t)nhv_gated(v[0], v[BOTH - 1], gate);
      else ((float*)y)[((size_t)split * M + row) * N + n] = v[0];
    }
  }
}

struct Plan {
  int mt, nt, splits;                                                // mt == 0: not for these kernels
  long long blocks;
  double taken_in;                                                   // us that a compute unit's share takes to come in
};

// The tile and the splits that take the least time by what was measured (17 to 128 rows of the 0.6B to 8B shapes' products): a
// launch's ends, what a compute unit takes in at 32 GB/s or the whole chip of w at 5.3 TB/s, whichever is longer, the parts' way
// to memory and back at 3.5 TB/s, and what a norm's block, which has a whole row to read, takes longer for them.
static Plan plan(int M, int N, int K, bool gated) {
  Plan best = {0, 0, 0, 0, 0.0};
  // (gated products of 128 rows 62.7 us at the 8B shape, the library's product and the gate's kernel 54; of 96 rows 44.5 against 47.5
  // there, and inside a step of the 4B shape 31.0 against 34.6. Of 128 rows wide products are slower too, 6,144 of 4,096 21.9
  // against 21.4, narrow ones not: 4,096 of 12,288 34 against 44.)
  if (M < 17 || M > (gated ? 96 : 128) || (M > 96 && N > K) || K % CHUNK || N < 64) return best;
  const int tiles = (M + 15) / 16, mt = tiles == 7 ? 8 : tiles;
  double least = 1e300;
  for (int nt : {2, 3, 4, 6}) {
    if (gated && nt == 3) continue;
    for (int splits : {1, 2, 4, 8}) {
      if ((gated && splits > 1) || splits * 2 > K / CHUNK) break;
      const int out = 16 * (gated ? nt / 2 : nt);
      const long long blocks = (long long)((N + out - 1) / out) * splits, rounds = (blocks + 255) / 256;
      const double taken_in = (double)rounds * (mt + nt) * 32 * ((K / CHUNK + splits - 1) / splits * CHUNK) / 32e3;
      const double of_w = 2.0 * (gated ? 2 : 1) * N * K / 5.3e6;
      const double time = (taken_in > of_w ? taken_in : of_w) + (gated ? 0.0 : 8.0 * splits * M * N / 3.5e6 + 4.0 * splits * N / 40e3);
      if (time < least) least = time, best = {mt, nt, splits, blocks, taken_in};
    }
  }
  return best;
}

// Where these kernels are the faster way: by 17, 32, 48, 64, 79, 96, 112 and 128 rows of 259 products, the 0.6B to 32B shapes and random
// ones of 64 to 36,864 outputs and 256 to 28,672 columns, each beside the fastest of the library's algorithms (gated: and the gate's
// kernel; plain: both with the norm that follows), cold weights; time by lines over the library's in brackets.
// Gated: one round of blocks. Where a second one begins the units that have none wait (17,408 outputs of 5,120 columns 1.08 to 1.27,
// 25,600 of 5,120 1.04 to 1.46, 13,824 of 5,120 from 48 rows on 1.07 to 1.17); where less than 144 blocks walk over many columns the others
// are idle from the start, K being whole (2,048 of 16,384 1.19 to 1.47, 960 of 9,856 up to 1.3, 1,024 of 4,096 1.2), unless the walk
// is a short one. 425 of the 726 are taken, 0.77 on average, the worst 1.04.
// Plain: up to 12,288 outputs (16,384 of 16,384 up to 1.22, 20,480 of 5,120 up to 1.10), two rounds of blocks (13,840 of 15,744 in eight parts up
// to 1.38, 8,192 of 28,672 at 112 rows 1.19), of more than 96 rows up to 8,192 outputs (10,256 of 14,464 1.06), and of more than 64 not the
// smallest products (376 of 384 up to 1.12, a microsecond). 890 of the 1,028 are taken, 0.75 on average, the
// worst 1.08 (112 rows of 300 outputs, 1.3 us). Sizes drawn after the rules were set, 827 measurements with these: gated 0.75, worst 1.09 (0.8 us),
// plain 0.76, worst 1.07.
static bool pays(const Plan& p, int M, int N, int K, bool gated) {
  if (gated) return p.blocks <= 256 && K <= 12288 && (p.blocks >= 144 || p.taken_in <= 10.0);
  return p.blocks <= 512 && N <= 12288 && K <= 32768 && (M <= 96 || N <= 8192) && (M <= 64 || (long long)N * K >= 1 << 18);
}

template <int MT, int NT, bool GATED>
static int launch(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int splits, const NhvGate& gate, hipStream_t s) {
  constexpr int OUT = 16 * (GATED ? NT / 2 : NT), ring = stages(MT, NT) * stage_bytes(MT, NT), sums = (GATED ? 2 : 1) * MT * 4096;
  constexpr int lds = ring > sums ? ring : sums;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = gemm_lines_kernel<MT, NT, GATED>;
  // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
  static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (allowed != hipSuccess) return nhv_fail("gemm by lines: %s", hipGetErrorString(allowed));
  hipLaunchKernelGGL(kernel, dim3((N + OUT - 1) / OUT, splits), dim3(512), lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, y, M, N, K,
                     splits, gate);
  NHV_LAUNCH_CHECK("gemm_lines_bf16");
  return 0;
}

template <int MT>
static int launch_rows(const Plan& p, bool gated, const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const NhvGate& gate,
                       hipStream_t s) {
  switch (p.nt * 2 + gated) {
    case 5: return launch<MT, 2, true>(x, w, bias, y, M, N, K, 1, gate, s);
    case 9: return launch<MT, 4, true>(x, w, bias, y, M, N, K, 1, gate, s);
    case 13: return launch<MT, 6, true>(x, w, bias, y, M, N, K, 1, gate, s);
    case 4: return launch<MT, 2, false>(x, w, bias, y, M, N, K, p.splits, gate, s);
    case 6: return launch<MT, 3, false>(x, w, bias, y, M, N, K, p.splits, gate, s);
    case 8: return launch<MT, 4, false>(x, w, bias, y, M, N, K, p.splits, gate, s);
    default: return launch<MT, 6, false>(x, w, bias, y, M, N, K, p.splits, gate, s);
  }
}

}  // namespace lines

// How many parts these kernels make of a product (1: a gated one's finished rows); ``whenever`` 0: 0 where another way is the faster one.
extern "C" int nhv_gemm_lines_splits(int M, int N, int K, int gated, int whenever) {
  const lines::Plan p = lines::plan(M, N, K, gated != 0);
  return p.mt > 0 && (whenever || lines::pays(p, M, N, K, gated != 0)) ? p.splits : 0;
}

// gated: y[M, N] in bfloat16; else y[splits][M][N] in float, whose sum over the splits is the product.
extern "C" int nhv_gemm_lines_bf16(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int gated, int act, float limit,
                                   float alpha, float offset, void* stream) {
  const lines::Plan p = lines::plan(M, N, K, gated != 0);
  NHV_REQUIRE(p.mt > 0, "gemm by lines: M=%d (17 to 128), N=%d (64 and more), K=%d (a multiple of %d)", M, N, K, lines::CHUNK);
  NHV_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) == 0, "gemm by lines: rows off 16-byte boundaries");
  NHV_REQUIRE(gated || bias == nullptr, "gemm by lines: parts have no bias");
  NHV_REQUIRE(act >= 0 && act <= 2, "gemm by lines: unknown gate %d", act);
  const NhvGate gate = {act, limit, alpha, offset};
  hipStream_t s = (hipStream_t)stream;
  switch (p.mt) {
    case 2: return lines::launch_rows<2>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
    case 3: return lines::launch_rows<3>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
    case 4: return lines::launch_rows<4>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
    case 5: return lines::launch_rows<5>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
    case 6: return lines::launch_rows<6>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
    default: return lines::launch_rows<8>(p, gated != 0, x, w, bias, y, M, N, K, gate, s);
  }
}
