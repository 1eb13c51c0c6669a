// A gate of two products of many rows in bfloat16, y[M, N] = gate(x[M, K] . wg[N, K]^T + bg, x . wu^T + bu) with w = [wg; wu], or
// one product and what its result passes, y = act(x . w^T).
//
// The product alone is no faster than the vendor's library's (0.96 to 1.1 of its time where tiles fill the chip); what is gained is that its rows need not exist:
// at 2,048 rows of 12,288 gates of 4,096 columns 100 MB that are written and read again, 30 us of 311. The library's product with the gate's
// kernel behind it, and this one, us: 2,048 x 12288 of 4,096 columns 311, 284; 1,866 rows 300, 276;
// 2,048 x 9728 of 2,560 214, 173; x 6144 of 2,048 104, 93; x 3072 of 1,024 37.6, 27.9; x 17408 of 5,120 618, 545; 8,192 x 12288 of 4,096
// 1,157, 1,093; activated, 1,925 x 6144 of 2,048 57.7, 48.3. (Gates are taken of float sums so, not of sums rounded to bfloat16.)
//
// A block is 8 waves, 2 x 4, and has 256 rows of x by 256 of w, a wave 128 by 64. The more both are, the less comes in for a
// product: at this size a compute unit takes in 64 KB for 512 matrix instructions, 45 bytes a ns, which the L2s give. Both
// operands go through LDS in pieces of 64 columns (whole lines of the caches), two pieces of 64 KB; a piece is four units, and a
// unit's place is loaded again as soon as every wave has read it, so that six of the eight units that fit are always under way:
// loads arrive 1.5 pieces after they are asked for (with whole pieces, one after they are asked for, 323 us for the 284). A
// wave reads the next quarter's operands while it multiplies this one's. Of LDS' 128 bytes a clock the reads take 96 and the
// loads 32, as long as the matrix instructions take. A block takes tile after tile (as many blocks as there are units), and the last quarters of one
// ask for the first pieces of the next.
// What bounds it is power: the matrix instructions take 74 % of the clocks, at 1.82 to 1.94 of 2.4 GHz (the library's 77 % at 1.93 or 82 % at 1.69); of
// zeros it is 222 us. That is why they are 16x16x32 ones: alone they run at 1,950 TFLOP/s, those of 32x32x16 at 1,720.
// Measured and not kept: four waves of 128 x 128 (369 us; accumulators move between register files), a barrier a quarter (the same), loads
// asked for at other places among the matrix instructions (the same), blocks at columns of their own (the same or up to 10 % more).
//
// Tiles are dealt out so that an XCD's 32 blocks have 8 tiles of rows of x and 4 of w at a time.
#include "nhv_common.h"
#include "nhv_gates.h"
#include "nhv_lines.h"

namespace phases {

typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 256, PIECE = 64;                    // rows of x and of w a block; columns of a piece of K
constexpr int UNIT = 128 * PIECE * 2, LDS = 8 * UNIT;    // bytes of 128 rows of a piece; two pieces of both operands

// 16 bytes a lane to LDS at `to` + 16 lane, from `lane_at` + `at` bytes behind the start of `rows`. What lies behind the end of `rows` is
// not read, also where `at` alone lies behind it: a lane's offset is compared with what the scalar offset leaves of the size, so that
// one is cut off at the size, which leaves nothing. (Written as an instruction, see nhv_lines.h; the one between gives m0 its wait.)
__device__ __forceinline__ void load_to_lds(uint32_t to, uint32_t lane_at, i32x4 rows, uint32_t at) {
  uint32_t cut;
  asm volatile("s_mov_b32 m0, %1\n\ts_min_u32 %0, %4, %5\n\tbuffer_load_dwordx4 %2, %3, %0 offen lds"
               : "=&s"(cut) : "s"(to), "v"(lane_at), "s"(rows), "s"(at), "s"(rows[2]) : "memory", "m0", "scc");
}
__device__ __forceinline__ i32x4 rows_from(const bf16_t* first, long long bytes) {
  const uint64_t at = (uint64_t)first;
  i32x4 r = {(int)(uint32_t)at, (int)((uint32_t)(at >> 32) & 0xffffu), (int)(bytes > 0xffffffffll ? 0xffffffffu : (uint32_t)bytes), 0x00020000};
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
  return r;
}

// z sigmoid(v) by the exponential and the reciprocal instruction (each within a unit in the last place or two of a float)
__device__ __forceinline__ float by_sigmoid(float z, float v) { return z * __builtin_amdgcn_rcpf(1.f + __expf(-v)); }
__device__ __forceinline__ float tanh_gelu(float z) { return by_sigmoid(z, 1.5957691216057308f * (z + 0.044715f * z * z * z)); }   // (1 + tanh v) / 2 is sigmoid(2 v)

template <int ACT>                                       // of NhvGate
__device__ __forceinline__ float gated(float g, float u, const NhvGate& p) {
  if (ACT == 2) {
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
    return by_sigmoid(g, p.alpha * g) * (u + p.offset);
  }
  return (ACT == 1 ? tanh_gelu(g) : by_sigmoid(g, g)) * u;
}
template <int ACT>                                       // 0 SiLU, 1 the tanh form of GELU, 2 the square of max(z, 0)
__device__ __forceinline__ float activated(float z) {
  if (ACT == 2) return fmaxf(z, 0.f) * fmaxf(z, 0.f);
  return ACT == 1 ? tanh_gelu(z) : by_sigmoid(z, z);
}

template <bool GATED, int ACT>
__global__ __launch_bounds__(512, 2) void gemm_phases_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                                             bf16_t* __restrict__ y, int M, int N, int K, NhvGate gate) {
  constexpr int COLUMNS = GATED ? TILE / 2 : TILE;       // outputs of a row
  extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int mt = (M + TILE - 1) / TILE, nt = (N + COLUMNS - 1) / COLUMNS;
  const int share = (mt * nt + 7) / 8, end = min((int)(blockIdx.x & 7) * share + share, mt * nt), stride = gridDim.x / 8;
  int tile = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
  if (tile >= end) return;
  const int pieces = K / PIECE;
  struct Place { int m0, n0; };
  auto place = [&](int i) {
    const int band = i / (8 * nt), in_band = i % (8 * nt), high = min(8, mt - 8 * band);
    return Place{(8 * band + in_band % high) * TILE, in_band / high * COLUMNS};
  };
  i32x4 x_rows, w_rows, u_rows;                          // of the tile that is being loaded
  auto turn_to = [&](const Place& p) {
    x_rows = rows_from(x + (size_t)p.m0 * K, (long long)(M - p.m0) * K * 2);
    w_rows = rows_from(w + (size_t)p.n0 * K, (long long)(N - p.n0) * K * 2);
    if (GATED) u_rows = rows_from(w + (size_t)(N + p.n0) * K, (long long)(N - p.n0) * K * 2);
  };
  // A wave brings 8 rows of 128 bytes a load. A row's 16 bytes p lie at place p ^ (row & 7): no bank conflicts.
  const uint32_t row = K * 2, lane_at = (lane >> 3) * row + ((lane & 7) ^ (lane >> 3)) * 16;
  const uint32_t ring_at = __builtin_amdgcn_readfirstlane(nhv_lds_address(ring)) + wave * 1024;
  const uint32_t x_at = wave * 8 * row, w_at = GATED ? x_at : ((wave >> 2) * 64 + (wave & 3) * 8) * row;
  enum { X0, X1, W0, W1 };                               // units of a piece: each wave's first and last 64 rows of x, first and last 32 of w (gated: gates, ups)
  auto load = [&](int slot, int unit, int piece) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t to = ring_at + ((unit >> 1) * 4 + slot * 2 + (unit & 1)) * UNIT + i * (UNIT / 2), at = piece * (PIECE * 2);
      if (unit <= X1) load_to_lds(to, lane_at, x_rows, x_at + (i * 128 + unit * 64) * row + at);
      else if (GATED) load_to_lds(to, lane_at, unit == W0 ? w_rows : u_rows, w_at + i * 64 * row + at);
      else load_to_lds(to, lane_at, w_rows, w_at + (i * 128 + (unit - W0) * 32) * row + at);
    }
  };
  const int wm = wave >> 2, wn = wave & 3;
  const bf16_t *a_at[2], *b_at[2];                       // of a piece's first and last 32 columns
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = r16 * PIECE + ((g + 4 * h) ^ (r16 & 7)) * 8;
    a_at[h] = ring + wm * 64 * PIECE + at;
    b_at[h] = ring + 2 * UNIT + wn * 32 * PIECE + at;
  }
  f32x4 acc[8][4];
  bf16x8 a[2][2][4], b[2][2][2];
  auto read_a = [&](int slot, int h, int q) { a[h][q >> 2][q & 3] = *reinterpret_cast<const bf16x8*>(a_at[q >> 2] + (slot * 2 + h) * (UNIT / 2) + (q & 3) * 16 * PIECE); };
  auto read_b = [&](int slot, int h, int q) { b[h][q >> 1][q & 1] = *reinterpret_cast<const bf16x8*>(b_at[q >> 1] + (slot * 2 + h) * (UNIT / 2) + (q & 1) * 16 * PIECE); };
  // A quarter of a piece: half `ha` of the wave's rows of x times half `hb` of its rows of w, 16 matrix instructions, among which
  // the unit that the next quarter needs is read.
  auto quarter = [&](int ha, int hb, int slot, int unit, auto between) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
#pragma unroll
      for (int n = 2 * q; n < 2 * q + 2; ++n) {
        const int h = n >> 3, i = (n & 7) >> 1, j = n & 1;
        acc[4 * ha + i][2 * hb + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[hb][h][j], a[ha][h][i], acc[4 * ha + i][2 * hb + j], 0, 0, 0);
      }
      if (unit <= X1) read_a(slot, unit, q);
      else if (q < 4) read_b(slot, unit - W0, q);
      between(q);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // Two quarters. Behind the barrier everyone's loads of the units that are read here have arrived (those of the two pairs before are
  // under way still), and everyone has read the two units of the pair before, whose places the next loads take.
  auto pair = [&](int ha0, int hb0, int slot0, int unit0, int ha1, int hb1, int slot1, int unit1, int to_slot, int to_unit0, int to_unit1, int piece) {
    nhv_wait_and_meet<8>();
    quarter(ha0, hb0, slot0, unit0, [&](int q) {
      if (q == 1) load(to_slot, to_unit0, piece);
      if (q == 4) load(to_slot, to_unit1, piece);
    });
    quarter(ha1, hb1, slot1, unit1, [](int) {});
  };

  Place now = place(tile);
  turn_to(now);
  load(0, X0, 0), load(0, W0, 0), load(0, W1, 0), load(0, X1, 0);
  load(1, X0, 1), load(1, W1, 1), load(1, W0, 1), load(1, X1, 1);
  nhv_wait_and_meet<12>();
#pragma unroll
  for (int q = 0; q < 8; ++q) read_a(0, 0, q);
#pragma unroll
  for (int q = 0; q < 4; ++q) read_b(0, 0, q);
  for (;;) {
    // (behind the last tile: its first pieces again, which nobody reads)
    const Place next = place(tile + stride < end ? tile + stride : tile);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int ahead = 2;
    for (int t = 0; t < pieces; t += 2, ahead += 2) {    // (a piece in either slot)
      if (t + 2 == pieces) {
        turn_to(next);
        ahead = 0;
      }
      pair(0, 0, 0, W1, 0, 1, 0, X1, 0, X0, W0, ahead);
      pair(1, 1, 1, X0, 1, 0, 1, W1, 0, W1, X1, ahead);
      pair(0, 1, 1, W0, 0, 0, 1, X1, 1, X0, W1, ahead + 1);
      pair(1, 0, 0, X0, 1, 1, 0, W0, 1, W0, X1, ahead + 1);
    }
    // lane 16 g + r of a tile holds outputs 4 g .. 4 g + 3 of row r
#pragma unroll
    for (int j = 0; j < (GATED ? 2 : 4); ++j) {
      const int n = now.n0 + wn * (COLUMNS / 4) + 16 * j + 4 * g;
      if (n >= N) continue;
      bf16x4 bg = {}, bu = {};
      if (GATED && bias) {
        bg = *reinterpret_cast<const bf16x4*>(bias + n);
        bu = *reinterpret_cast<const bf16x4*>(bias + N + n);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = now.m0 + wm * 128 + 16 * i + r16;
        if (m >= M) continue;
        bf16x4 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (GATED) out[e] = (bf16_t)gated<ACT>(acc[i][j][e] + (float)bg[e], acc[i][(j + 2) % 4][e] + (float)bu[e], gate);
          else out[e] = (bf16_t)activated<ACT>(acc[i][j][e]);
        }
        *reinterpret_cast<bf16x4*>(y + (size_t)m * N + n) = out;
      }
    }
    tile += stride;
    if (tile >= end) break;
    now = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (no load may come into LDS that is another block's by then)
}

template <bool GATED, int ACT>
static int launch(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const NhvGate& gate, hipStream_t s) {
  auto kernel = gemm_phases_kernel<GATED, ACT>;
  // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
  static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (allowed != hipSuccess) return nhv_fail("gemm by phases: %s", hipGetErrorString(allowed));
  constexpr int COLUMNS = GATED ? TILE / 2 : TILE;
  const long long tiles = (long long)((M + TILE - 1) / TILE) * ((N + COLUMNS - 1) / COLUMNS);
  hipLaunchKernelGGL(kernel, dim3(tiles < 256 ? (unsigned)((tiles + 7) / 8 * 8) : 256u), dim3(512), LDS, s, (const bf16_t*)x, (const bf16_t*)w,
                     (const bf16_t*)bias, (bf16_t*)y, M, N, K, gate);
  NHV_LAUNCH_CHECK("gemm_phases_bf16");
  return 0;
}

static bool takes(int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % (2 * PIECE) == 0 && K < (1 << 22) && ((long long)M + TILE) / TILE * (((long long)N + TILE) / TILE) < (1ll << 28);
}

}  // namespace phases

// Whether this is the faster way: where tiles' outputs are at least six tenths of what the rounds of 256 blocks could make. Measured over 459
// sizes (128 to 5,800 rows, 1,024 to 17,400 outputs, 256 to 6,200 columns, cold weights; time here over the library's product and the kernel that follows it): gated,
// 122 sizes at 0.6 and more, 0.78 on average, the worst 1.02 (543 rows, 9,728 outputs of 2,560); from 0.5 on 0.79, the worst 1.14 (793, 12,288 of 4,096); 0.4 to 0.5 0.99, up to
// 1.26. Activated, 54 sizes at 0.6 and more 0.79, the worst 1.05 (4,610 rows, 4,480 of 5,888), 0.5 to 0.6 0.87, up to 1.10.
extern "C" int nhv_gemm_phases_pays(int M, int N, int K, int gated) {
  if (!phases::takes(M, N, K)) return 0;
  const long long columns = gated ? phases::TILE / 2 : phases::TILE;
  const long long tiles = ((long long)M + phases::TILE - 1) / phases::TILE * ((N + columns - 1) / columns), rounds = (tiles + 255) / 256;
  return 10ll * M * N >= 6 * rounds * 256 * phases::TILE * columns;
}

extern "C" int nhv_gemm_phases_bf16(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int gated, int act, float limit,
                                    float alpha, float offset, void* stream) {
  NHV_REQUIRE(phases::takes(M, N, K), "gemm by phases: M=%d, N=%d (a multiple of 8), K=%d (a multiple of %d)", M, N, K, 2 * phases::PIECE);
  NHV_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0 && (((uintptr_t)y | (uintptr_t)bias) & 7) == 0, "gemm by phases: rows off their boundaries");
  NHV_REQUIRE(gated || bias == nullptr, "gemm by phases: a bias goes with a gate");
  NHV_REQUIRE(act >= 0 && act <= 2, "gemm by phases: unknown activation %d", act);
  const NhvGate gate = {act, limit, alpha, offset};
  hipStream_t s = (hipStream_t)stream;
  switch (act * 2 + (gated != 0)) {
    case 0: return phases::launch<false, 0>(x, w, bias, y, M, N, K, gate, s);
    case 1: return phases::launch<true, 0>(x, w, bias, y, M, N, K, gate, s);
    case 2: return phases::launch<false, 1>(x, w, bias, y, M, N, K, gate, s);
    case 3: return phases::launch<true, 1>(x, w, bias, y, M, N, K, gate, s);
    case 4: return phases::launch<false, 2>(x, w, bias, y, M, N, K, gate, s);
    default: return phases::launch<true, 2>(x, w, bias, y, M, N, K, gate, s);
  }
}
