// y[M, N] = x[M, K] . w[N, K]^T (+ bias), or a gate of x . wg^T and x . wu^T (nhv_gates.h), in bfloat16 for up to 16
// rows of x: the matrix products of a decoding step, whose time is the time to stream w from memory once.
//
// A block owns NT tiles of 16 rows of w (with GLU also their partners in the second matrix) and all
// of K; its waves take equal, contiguous shares of K, whole cache lines each, and a wave's lanes load
// 16 bytes each straight into the MFMA operand layout (v_mfma_f32_16x16x32_bf16: the w tile as the
// 16 x 32 operand, the rows of x as the 32 x 16 one), several loads in flight before the first is used.
// The waves' sums meet in LDS and are added in the order of the waves, so the result does not depend
// on timing. Rows of x beyond M and columns beyond K read as zero.
//
// Rows of a multiple of 256 columns and 2,048 and more, with outputs enough to fill the chip in tiles of 16, take a kernel that brings w and
// x through LDS by lines of 512 bytes (gemm_fewrows_lines_kernel, lines_plan() below): nearly all layer shapes and heads from the
// 1.7B widths on. Most of the others take one of two kernels in whose tiles nothing waits (tiles_plan() below). What neither takes:
// where all rows of x fit into LDS beside the sums (M (K + 8) 2 bytes of the 160 KB) a block copies x into LDS once (straight from
// memory, global_load_lds) and then walks over tiles of w, tile after tile, one or two blocks per compute unit for the whole matrix.
// The rows of x then cross from L2 to a compute unit once per call instead of once per tile: 5 to 25 % less time than by the kernel
// described above at every size measured, most where N is large. Where x does not fit at once and w has at most 256 tiles, a further
// kernel gives every block one tile and takes x through LDS in pieces (4,096 outputs of 12,288 columns from 7 rows on: 2 to 6 % less time,
// 12 % with 2,048 outputs). With more tiles than that, and x fitting in two pieces, another one walks over all of a block's tiles once for
// each piece and keeps the tiles' sums in LDS between the two (16 rows of 5,120 columns: 13 % less time for gate_up). (Sizes that are quoted
// here and at those kernels were measured before the kernel by lines was there, which takes those of 256 columns' multiples now; the
// rules hold for the others.)
//
// How many tiles a block takes, how many waves share K and how many loads a wave keeps in flight is
// chosen per call from M, N and K (plan() below): blocks that spread evenly over the compute units
// matter most, two tiles per block halve the reads of x when it has more than a few rows. (Splitting
// K over several blocks, with the last one to arrive adding the parts in order, was measured and never
// won: the fences cost more than the balance gains.)
#include "nhv_common.h"
#include "nhv_gemm_fusion.h"
#include "nhv_lines.h"
#include <type_traits>

namespace fewrows {

typedef NhvGemmFusion Fusion;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

__device__ __forceinline__ bf16x8 load8(const bf16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.f;
  return z;
}

// The scales of the rows of an x whose norm is still due (nhv_gemm_fusion.h), in two steps, so that the wait for
// the shares falls where other loads are under way. ask_row_scales: wave w asks for the shares of rows w, w + WAVES,
// ... (M <= 16: SCALE_ROWS<WAVES> rows at most), SCALE_SHARES of them per lane and row. set_row_scales: adds them up
// in a fixed order and leaves the scales in r_s[0..M); the caller's next barrier makes them visible.
constexpr int SCALE_SHARES = 4;              // up to 256 tiles (rows of 4,096) in one go; what is beyond is read when the sums are made
template <int WAVES>
constexpr int SCALE_ROWS = (16 + WAVES - 1) / WAVES;
template <int WAVES>
__device__ __forceinline__ void ask_row_scales(const Fusion& f, float (&share)[SCALE_ROWS<WAVES>][SCALE_SHARES], int M, int wave, int lane) {
  if (f.ss_in == nullptr) return;
#pragma unroll
  for (int i = 0; i < SCALE_ROWS<WAVES>; ++i) {
    const int m = wave + i * WAVES;
#pragma unroll
    for (int j = 0; j < SCALE_SHARES; ++j) {
      const int t = lane + j * 64;
      share[i][j] = (m < M && t < f.tiles_in) ? f.ss_in[(size_t)m * f.tiles_in + t] : 0.f;
    }
  }
}
template <int WAVES>
__device__ __forceinline__ void set_row_scales(const Fusion& f, const float (&share)[SCALE_ROWS<WAVES>][SCALE_SHARES], float* r_s, int M, int K,
                                               int wave, int lane) {
  if (f.ss_in == nullptr) return;
#pragma unroll
  for (int i = 0; i < SCALE_ROWS<WAVES>; ++i) {
    const int m = wave + i * WAVES;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < SCALE_SHARES; ++j) sum += share[i][j];
    if (m < M)
      for (int t = lane + SCALE_SHARES * 64; t < f.tiles_in; t += 64) sum += f.ss_in[(size_t)m * f.tiles_in + t];
    sum = wave_sum(sum);
    if (m < M && lane == 0) r_s[m] = 1.0f / sqrtf(sum / (float)K + f.eps);
  }
}

// A gated product's two finished sums (the first with its bias in): the second one's bias lies N further.
__device__ __forceinline__ float finish_gated(float g, float u, const bf16_t* bias, int n, int N, const NhvGate& gate) {
  if (bias && n < N) u += (float)bias[N + n];
  return nhv_gated(g, u, gate);
}

// What the wave that writes a tile adds to and multiplies with, asked for before the tile's weights: the residual's
// entries and the next norm's weights of the lane's four outputs.
__device__ __forceinline__ void read_residual(const Fusion& f, float (&ahead)[8], int col, int grp, int n0, int M, int N) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + grp * 4 + j;
    ahead[4 + j] = 1.0f;
    if (col < M && n < N) {
      const size_t at = (size_t)col * N + n;
      ahead[j] = f.residual_f32 ? reinterpret_cast<const float*>(f.residual)[at] : (float)reinterpret_cast<const bf16_t*>(f.residual)[at];
      if (f.next_w) ahead[4 + j] = f.next_w_f32 ? reinterpret_cast<const float*>(f.next_w)[n] : (float)reinterpret_cast<const bf16_t*>(f.next_w)[n];
    }
  }
}

// A finished tile goes out: lane (col, grp) holds outputs n0 + 4 grp + (0..3) of row col of x. Plain: stored as they
// are. With a residual stream (nhv_gemm_fusion.h): added to it in float, the sum kept there and, times the next
// norm's weight and rounded, in sum_out, and the tile's share of the row's sum of squares (over its 16 outputs, the
// lanes' shares added in a fixed order) in ss_out. `tile` and `tiles` count tiles of 16 outputs over all of N.
// `ahead`: the residual's entries and the next norm's weights where the caller has read them already (read_residual), else null.
template <bool FUSED, typename TOut>
__device__ __forceinline__ void emit_tile(const Fusion& f, const float (&r)[4], TOut* __restrict__ y, int col, int grp, int n0,
                                          int tile, int tiles, int M, int N, const float* ahead = nullptr) {
  if (!FUSED || f.residual == nullptr) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + grp * 4 + j;
      if (col < M && n < N) y[(size_t)col * N + n] = (TOut)r[j];
    }
    return;
  }
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + grp * 4 + j;
    if (col < M && n < N) {
      const size_t at = (size_t)col * N + n;
      float sum;
      if (f.residual_f32) {
        float* res = reinterpret_cast<float*>(f.residual);
        sum = r[j] + (ahead ? ahead[j] : res[at]);
        res[at] = sum;
      } else {
        bf16_t* res = reinterpret_cast<bf16_t*>(f.residual);
        sum = r[j] + (ahead ? ahead[j] : (float)res[at]);
        res[at] = (bf16_t)sum;
      }
      float weight = 1.0f;
      if (ahead) weight = ahead[4 + j];
      else if (f.next_w) weight = f.next_w_f32 ? reinterpret_cast<const float*>(f.next_w)[n] : (float)reinterpret_cast<const bf16_t*>(f.next_w)[n];
      f.sum_out[at] = (bf16_t)(sum * weight);
      sq += sum * sum;
    }
  }
  sq += __shfl_xor(sq, 16, 64);
  sq += __shfl_xor(sq, 32, 64);
  if (grp == 0 && col < M) f.ss_out[(size_t)col * tiles + tile] = sq;
}

// NT: tiles of 16 rows of w per block; WAVES: waves that share the block's part of K; UNROLL: loads in
// flight per wave and operand. A step is 32 columns of K (64 bytes of a row).
template <int NT, int WAVES, int UNROLL, bool GLU, bool FUSED, typename TOut>
__global__ __launch_bounds__(64 * WAVES) void gemm_fewrows_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                  const bf16_t* __restrict__ bias, TOut* __restrict__ y,
                                                                  int M, int N, int K, int steps_per_wave, const Fusion f) {
  constexpr int NA = GLU ? 2 : 1;
  constexpr int TILES = NA * NT;
  static_assert(NT <= WAVES, "wave nt finishes tile nt");
  __shared__ float red[WAVES][TILES][4][64];
  __shared__ float r_s[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT;
  float share[SCALE_ROWS<WAVES>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<WAVES>(f, share, M, wave, lane);

  const bf16_t* wrow[TILES];
  bool n_ok[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = n0 + nt * 16 + col;
    n_ok[nt] = n < N;
#pragma unroll
    for (int na = 0; na < NA; ++na) wrow[na * NT + nt] = w + ((size_t)na * N + (n_ok[nt] ? n : 0)) * K;
  }
  const bool m_ok = col < M;
  if (f.band_rows) x += (size_t)min(n0 / f.band_rows, f.bands - 1) * M * K;
  const bf16_t* xrow = x + (size_t)(m_ok ? col : 0) * K;

  floatx4 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int ksteps = (K + 31) / 32;
  const int first = wave * steps_per_wave;
  const int last = min(first + steps_per_wave, ksteps);
  // a run: UNROLL steps loaded, then multiplied. (Issuing the next run's loads before this run's products was
  // measured too and changed nothing: enough other waves have loads in flight meanwhile.)
  for (int s0 = first; s0 < last; s0 += UNROLL) {
    bf16x8 a[UNROLL][TILES], b[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int k = (s0 + u) * 32 + grp * 8;
      const bool k_ok = (s0 + u < last) && k < K;      // K is a multiple of 8: a piece is inside or outside as a whole
#pragma unroll
      for (int t = 0; t < TILES; ++t) a[u][t] = (n_ok[t % NT] && k_ok) ? load8(wrow[t] + k) : zero8();
      b[u] = (m_ok && k_ok) ? load8(xrow + k) : zero8();
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int t = 0; t < TILES; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][t], b[u], acc[t], 0, 0, 0);
  }
  if constexpr (FUSED) set_row_scales<WAVES>(f, share, r_s, M, K, wave, lane);
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave][t][j][lane] = acc[t][j];
  __syncthreads();
  if (wave >= NT) return;

  // wave nt adds the waves' sums of tile nt (and of its partner) in the order of the waves
  const int nt = wave;
  float v[NA][4];
#pragma unroll
  for (int na = 0; na < NA; ++na)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float sum = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) sum += red[wv][na * NT + nt][j][lane];
      v[na][j] = sum;
    }

  const float rs = (FUSED && f.ss_in) ? r_s[col] : 1.0f;           // the row's scale, where x is a sum whose norm is due
  float out[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + nt * 16 + grp * 4 + j;           // the tile's row 4 grp + j is output n, its column is row col of x
    float r = v[0][j] * rs;
    if (bias && n < N) r += (float)bias[n];
    if (GLU) r = finish_gated(r, v[NA - 1][j] * rs, bias, n, N, f.gate);
    else if (f.plain_act) r = nhv_plain_act(r, f.plain_act);
    out[j] = r;
  }
  emit_tile<FUSED, TOut>(f, out, y, col, grp, n0 + nt * 16, blockIdx.x * NT + nt, (N + 15) / 16, M, N);
}

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef const __attribute__((address_space(1))) void* global_ptr;

// The kernel with x resident in LDS: x_s[m][K + 8] (the 16 bytes between rows spread the rows over the
// banks), then for tile = blockIdx.x, + gridDim.x, ...: waves split K as above, sums meet in one of two
// LDS buffers (one barrier a tile), and the waves take turns in adding them up and writing the result.
// The first weights of a block's first tile are asked for right after x and the wait before the first product is for
// x alone (0.2 to 0.5 us less per call at every shape; asked for before x they made every shape slower, by 0.5 to
// 3 us).
template <int WAVES, int UNROLL, bool GLU, bool FUSED, typename TOut>
__global__ __launch_bounds__(64 * WAVES) void gemm_fewrows_resident_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                           const bf16_t* __restrict__ bias, TOut* __restrict__ y,
                                                                           int M, int N, int K, int tiles, int steps_per_wave,
                                                                           const Fusion f) {
  constexpr int NA = GLU ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  float(*red)[NA][4][64] = reinterpret_cast<float(*)[NA][4][64]>(lds_raw);      // [2 WAVES][NA][4][64]
  bf16_t* x_s = reinterpret_cast<bf16_t*>(lds_raw + 2 * WAVES * NA * 4 * 64 * sizeof(float));
  const int pitch = K + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  __shared__ float r_s[16];
  // (the rows' scales are wanted when the first tile goes out: their shares are asked for first of all, and the
  // barrier before the tile's sums are added up makes the scales visible)
  float share[SCALE_ROWS<WAVES>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<WAVES>(f, share, M, wave, lane);
  // x into LDS: a wave's load brings 64 consecutive 16-byte pieces of one row
  const int pieces_per_row = K / 8;
  const int loads_per_row = (pieces_per_row + 63) / 64;
  for (int job = wave; job < M * loads_per_row; job += WAVES) {
    const int m = job / loads_per_row, part = job % loads_per_row;
    const int piece = part * 64 + lane;
    if (piece < pieces_per_row)
      __builtin_amdgcn_global_load_lds((global_ptr)(x + (size_t)m * K + piece * 8), (lds_ptr)(x_s + m * pitch + part * 512), 16, 0, 0);
  }
  const int ksteps = (K + 31) / 32;
  const int first = wave * steps_per_wave;
  const int last = min(first + steps_per_wave, ksteps);
  // The first weights of the block's first tile are asked for while x is still on its way: every lane asks (from an
  // address moved into the matrix where it would lie outside), so that exactly UNROLL NA loads are younger than
  // those of x, and the wait below is for x alone.
  asm volatile("" ::: "memory");
  bf16x8 a_first[UNROLL][NA];
  {
    const int n0 = blockIdx.x * 16;
    const bool n_ok = n0 + col < N;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int k = (first + u) * 32 + grp * 8;
      const int k_in = k + 8 <= K ? k : 0;
#pragma unroll
      for (int na = 0; na < NA; ++na) a_first[u][na] = load8(w + ((size_t)na * N + (n_ok ? n0 + col : 0)) * K + k_in);
    }
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(UNROLL * NA) : "memory");
  __syncthreads();

  const bool m_ok = col < M;
  const bf16_t* xrow_s = x_s + (m_ok ? col : 0) * pitch;
  int parity = 0, turn = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, parity ^= 1, turn = turn + 1 == WAVES ? 0 : turn + 1) {
    const int n0 = tile * 16;
    const bool n_ok = n0 + col < N;
    // the wave that will write this tile asks for the residual's entries it adds to before the tile's weights
    // (the gated product is never added to a residual stream)
    float res_ahead[8] = {0.f, 0.f, 0.f, 0.f, 1.f, 1.f, 1.f, 1.f};
    if constexpr (FUSED && !GLU) if (f.residual != nullptr && wave == turn) read_residual(f, res_ahead, col, grp, n0, M, N);
    const bf16_t* wrow[NA];
#pragma unroll
    for (int na = 0; na < NA; ++na) wrow[na] = w + ((size_t)na * N + (n_ok ? n0 + col : 0)) * K;
    floatx4 acc[NA];
#pragma unroll
    for (int na = 0; na < NA; ++na) acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = first; s0 < last; s0 += UNROLL) {
      bf16x8 a[UNROLL][NA];
      const bool asked = tile == (int)blockIdx.x && s0 == first;
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int k = (s0 + u) * 32 + grp * 8;
        const bool k_ok = (s0 + u < last) && k < K;
#pragma unroll
        for (int na = 0; na < NA; ++na) {
          if (asked) a[u][na] = (n_ok && k_ok) ? a_first[u][na] : zero8();
          else a[u][na] = (n_ok && k_ok) ? load8(wrow[na] + k) : zero8();
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int k = (s0 + u) * 32 + grp * 8;
        const bool k_ok = (s0 + u < last) && k < K;
        const bf16x8 b = (m_ok && k_ok) ? *reinterpret_cast<const bf16x8*>(xrow_s + k) : zero8();
#pragma unroll
        for (int na = 0; na < NA; ++na) acc[na] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][na], b, acc[na], 0, 0, 0);
      }
    }
    if constexpr (FUSED) if (tile == (int)blockIdx.x) set_row_scales<WAVES>(f, share, r_s, M, K, wave, lane);
    float(*my_red)[NA][4][64] = red + parity * WAVES;
#pragma unroll
    for (int na = 0; na < NA; ++na)
#pragma unroll
      for (int j = 0; j < 4; ++j) my_red[wave][na][j][lane] = acc[na][j];
    __syncthreads();                          // the other buffer is the one written in the next tile
    if (wave != turn) continue;
    float v[NA][4];
#pragma unroll
    for (int na = 0; na < NA; ++na)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float sum = 0.f;
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) sum += my_red[wv][na][j][lane];
        v[na][j] = sum;
      }
    const float rs = (FUSED && f.ss_in) ? r_s[col] : 1.0f;         // the row's scale, where x is a sum whose norm is due
    float out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + grp * 4 + j;
      float r = v[0][j] * rs;
      if (bias && n < N) r += (float)bias[n];
      if (GLU) r = finish_gated(r, v[NA - 1][j] * rs, bias, n, N, f.gate);
      else if (f.plain_act) r = nhv_plain_act(r, f.plain_act);
      out[j] = r;
    }
    emit_tile<FUSED && !GLU, TOut>(f, out, y, col, grp, n0, tile, tiles, M, N, res_ahead);
  }
}

// Where all of x is too much for LDS: the same with one tile a block and x coming in `nchunks` pieces of
// `chunk_steps` steps of 32 columns, one after the other; the sums run on over the pieces. (A kernel of its own:
// as an option of the one above it cost that one 4 % of its speed.)
template <int WAVES, int UNROLL, bool FUSED, typename TOut>
__global__ __launch_bounds__(64 * WAVES) void gemm_fewrows_pieces_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                           const bf16_t* __restrict__ bias, TOut* __restrict__ y,
                                                                           int M, int N, int K, int tiles, int nchunks,
                                                                           int chunk_steps, int steps_per_wave, const Fusion f) {
  constexpr int NA = 1;
  constexpr bool GLU = false;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  float(*red)[NA][4][64] = reinterpret_cast<float(*)[NA][4][64]>(lds_raw);      // [2 WAVES][NA][4][64]
  bf16_t* x_s = reinterpret_cast<bf16_t*>(lds_raw + 2 * WAVES * NA * 4 * 64 * sizeof(float));
  const int pitch = min(K, chunk_steps * 32) + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  __shared__ float r_s[16];
  float share[SCALE_ROWS<WAVES>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<WAVES>(f, share, M, wave, lane);
  const int ksteps = (K + 31) / 32;
  const bool m_ok = col < M;
  const bf16_t* xrow_s = x_s + (m_ok ? col : 0) * pitch;
  // columns [32 c0, 32 c_end) of x into LDS: a wave's load brings 64 consecutive 16-byte pieces of one row
  auto load_x = [&](int c0, int c_end) {
    const int col0 = c0 * 32;
    const int pieces_per_row = (min(K, c_end * 32) - col0) / 8;
    const int loads_per_row = (pieces_per_row + 63) / 64;
    for (int job = wave; job < M * loads_per_row; job += WAVES) {
      const int m = job / loads_per_row, part = job % loads_per_row;
      const int piece = part * 64 + lane;
      if (piece < pieces_per_row)
        __builtin_amdgcn_global_load_lds((global_ptr)(x + (size_t)m * K + col0 + piece * 8),
                                         (lds_ptr)(x_s + m * pitch + part * 512), 16, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  int parity = 0, turn = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, parity ^= 1, turn = turn + 1 == WAVES ? 0 : turn + 1) {
    const int n0 = tile * 16;
    const bool n_ok = n0 + col < N;
    const bf16_t* wrow[NA];
#pragma unroll
    for (int na = 0; na < NA; ++na) wrow[na] = w + ((size_t)na * N + (n_ok ? n0 + col : 0)) * K;
    floatx4 acc[NA];
#pragma unroll
    for (int na = 0; na < NA; ++na) acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < nchunks; ++c) {
      const int c0 = c * chunk_steps, c_end = min(c0 + chunk_steps, ksteps);
      if (c > 0) __syncthreads();                        // the piece before has been read by every wave
      load_x(c0, c_end);
      const int first = c0 + wave * steps_per_wave;
      const int last = min(first + steps_per_wave, c_end);
      for (int s0 = first; s0 < last; s0 += UNROLL) {
        bf16x8 a[UNROLL][NA];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const int k = (s0 + u) * 32 + grp * 8;
          const bool k_ok = (s0 + u < last) && k < K;
#pragma unroll
          for (int na = 0; na < NA; ++na) a[u][na] = (n_ok && k_ok) ? load8(wrow[na] + k) : zero8();
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const int k = (s0 + u) * 32 + grp * 8;
          const bool k_ok = (s0 + u < last) && k < K;
          const bf16x8 b = (m_ok && k_ok) ? *reinterpret_cast<const bf16x8*>(xrow_s + (k - c0 * 32)) : zero8();
#pragma unroll
          for (int na = 0; na < NA; ++na) acc[na] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][na], b, acc[na], 0, 0, 0);
        }
      }
    }
    if constexpr (FUSED) if (tile == (int)blockIdx.x) set_row_scales<WAVES>(f, share, r_s, M, K, wave, lane);
    float(*my_red)[NA][4][64] = red + parity * WAVES;
#pragma unroll
    for (int na = 0; na < NA; ++na)
#pragma unroll
      for (int j = 0; j < 4; ++j) my_red[wave][na][j][lane] = acc[na][j];
    __syncthreads();                          // the other buffer is the one written in the next tile
    if (wave != turn) continue;
    float v[NA][4];
#pragma unroll
    for (int na = 0; na < NA; ++na)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float sum = 0.f;
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) sum += my_red[wv][na][j][lane];
        v[na][j] = sum;
      }
    const float rs = (FUSED && f.ss_in) ? r_s[col] : 1.0f;         // the row's scale, where x is a sum whose norm is due
    float out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + grp * 4 + j;
      float r = v[0][j] * rs;
      if (bias && n < N) r += (float)bias[n];
      if (GLU) r = finish_gated(r, v[NA - 1][j] * rs, bias, n, N, f.gate);
      else if (f.plain_act) r = nhv_plain_act(r, f.plain_act);
      out[j] = r;
    }
    emit_tile<FUSED, TOut>(f, out, y, col, grp, n0, tile, tiles, M, N);
  }
}

// Where all of x is too much for LDS and a block has several tiles: x comes in `npasses` pieces of `pass_steps`
// steps of 32 columns; for every piece the block walks over all of its tiles, and a tile's sums over the pieces so
// far wait in LDS (part_s, 1 KB a tile and matrix) for the next piece. The weights are still read once. The
// wave that adds up a tile's sums is the same in every pass, so what it left in part_s it finds again itself.
template <int WAVES, int UNROLL, bool GLU, bool FUSED, typename TOut>
__global__ __launch_bounds__(64 * WAVES) void gemm_fewrows_passes_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                           const bf16_t* __restrict__ bias, TOut* __restrict__ y,
                                                                           int M, int N, int K, int tiles, int npasses,
                                                                           int pass_steps, int steps_per_wave, int tiles_per_block,
                                                                           const Fusion f) {
  constexpr int NA = GLU ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  float(*red)[NA][4][64] = reinterpret_cast<float(*)[NA][4][64]>(lds_raw);      // [2 WAVES][NA][4][64]
  float(*part_s)[NA][4][64] = red + 2 * WAVES;                                   // [tiles_per_block][NA][4][64]
  bf16_t* x_s = reinterpret_cast<bf16_t*>(lds_raw + (size_t)(2 * WAVES + tiles_per_block) * NA * 4 * 64 * sizeof(float));
  const int pitch = min(K, pass_steps * 32) + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  __shared__ float r_s[16];
  float share[SCALE_ROWS<WAVES>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<WAVES>(f, share, M, wave, lane);
  const int ksteps = (K + 31) / 32;
  const bool m_ok = col < M;
  const bf16_t* xrow_s = x_s + (m_ok ? col : 0) * pitch;
  int parity = 0;
  for (int p = 0; p < npasses; ++p) {
    const int c0 = p * pass_steps, c_end = min(c0 + pass_steps, ksteps);
    // this piece of x into LDS: a wave's load brings 64 consecutive 16-byte pieces of one row
    if (p > 0) __syncthreads();                          // the piece before has been read by every wave
    {
      const int col0 = c0 * 32;
      const int pieces_per_row = (min(K, c_end * 32) - col0) / 8;
      const int loads_per_row = (pieces_per_row + 63) / 64;
      for (int job = wave; job < M * loads_per_row; job += WAVES) {
        const int m = job / loads_per_row, part = job % loads_per_row;
        const int piece = part * 64 + lane;
        if (piece < pieces_per_row)
          __builtin_amdgcn_global_load_lds((global_ptr)(x + (size_t)m * K + col0 + piece * 8),
                                           (lds_ptr)(x_s + m * pitch + part * 512), 16, 0, 0);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    const int first = c0 + wave * steps_per_wave;
    const int last = min(first + steps_per_wave, c_end);
    int ti = 0, turn = 0;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, ++ti, parity ^= 1, turn = turn + 1 == WAVES ? 0 : turn + 1) {
      const int n0 = tile * 16;
      const bool n_ok = n0 + col < N;
      const bf16_t* wrow[NA];
#pragma unroll
      for (int na = 0; na < NA; ++na) wrow[na] = w + ((size_t)na * N + (n_ok ? n0 + col : 0)) * K;
      floatx4 acc[NA];
#pragma unroll
      for (int na = 0; na < NA; ++na) acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
      for (int s0 = first; s0 < last; s0 += UNROLL) {
        bf16x8 a[UNROLL][NA];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const int k = (s0 + u) * 32 + grp * 8;
          const bool k_ok = (s0 + u < last) && k < K;
#pragma unroll
          for (int na = 0; na < NA; ++na) a[u][na] = (n_ok && k_ok) ? load8(wrow[na] + k) : zero8();
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const int k = (s0 + u) * 32 + grp * 8;
          const bool k_ok = (s0 + u < last) && k < K;
          const bf16x8 b = (m_ok && k_ok) ? *reinterpret_cast<const bf16x8*>(xrow_s + (k - c0 * 32)) : zero8();
#pragma unroll
          for (int na = 0; na < NA; ++na) acc[na] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][na], b, acc[na], 0, 0, 0);
        }
      }
      if constexpr (FUSED) if (p == 0 && ti == 0) set_row_scales<WAVES>(f, share, r_s, M, K, wave, lane);
      float(*my_red)[NA][4][64] = red + parity * WAVES;
#pragma unroll
      for (int na = 0; na < NA; ++na)
#pragma unroll
        for (int j = 0; j < 4; ++j) my_red[wave][na][j][lane] = acc[na][j];
      __syncthreads();                        // the other buffer is the one written for the next tile
      if (wave != turn) continue;
      float v[NA][4];
#pragma unroll
      for (int na = 0; na < NA; ++na)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float sum = p > 0 ? part_s[ti][na][j][lane] : 0.f;
#pragma unroll
          for (int wv = 0; wv < WAVES; ++wv) sum += my_red[wv][na][j][lane];
          v[na][j] = sum;
        }
      if (p + 1 < npasses) {
#pragma unroll
        for (int na = 0; na < NA; ++na)
#pragma unroll
          for (int j = 0; j < 4; ++j) part_s[ti][na][j][lane] = v[na][j];
        continue;
      }
      const float rs = (FUSED && f.ss_in) ? r_s[col] : 1.0f;       // the row's scale, where x is a sum whose norm is due
      float out[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + grp * 4 + j;
        float r = v[0][j] * rs;
        if (bias && n < N) r += (float)bias[n];
        if (GLU) r = finish_gated(r, v[NA - 1][j] * rs, bias, n, N, f.gate);
        else if (f.plain_act) r = nhv_plain_act(r, f.plain_act);
        out[j] = r;
      }
      emit_tile<FUSED, TOut>(f, out, y, col, grp, n0, tile, tiles, M, N);
    }
  }
}

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned uint4v;
typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned uint2v;

// Four neighbouring numbers as they lie in memory, in float32 or bfloat16 (a conversion where they are asked for would wait for
// them, and so would a branch on the type): two loads of 8 bytes, which for bfloat16 are the same one. Without a pointer:
// `some` is read and not used.
struct Four {
  uint2v lo, hi;
  __device__ __forceinline__ void ask(const void* p, size_t at, int is_f32, const void* some) {
    const char* from = p ? (const char*)p + at * (is_f32 ? 4 : 2) : (const char*)some;
    lo = *reinterpret_cast<const uint2v*>(from);
    hi = *reinterpret_cast<const uint2v*>(from + (is_f32 ? 8 : 0));
  }
  __device__ __forceinline__ float at(int j, int is_f32) const {
    return __uint_as_float(is_f32 ? (j < 2 ? lo[j] : hi[j - 2]) : j % 2 ? lo[j / 2] & 0xffff0000u : lo[j / 2] << 16);
  }
};
__device__ __forceinline__ void store4(bf16_t* p, const float (&v)[4]) {
  bf16x4 y;
#pragma unroll
  for (int j = 0; j < 4; ++j) y[j] = (__bf16)v[j];
  *reinterpret_cast<bf16x4*>(p) = y;
}
__device__ __forceinline__ void store4(float* p, const float (&v)[4]) { *reinterpret_cast<floatx4*>(p) = floatx4{v[0], v[1], v[2], v[3]}; }

// A barrier for LDS alone: loads from memory stay under way.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// What the two kernels below share. They are bound by the latency of a product's few loads where it is small and by the stream of
// w where it is large: a tile is up to 16 rows of w (a multiple of 4, so that all 256 compute units have one); 16 waves share
// K; a wave has AHEAD steps of 32 columns under way, AHEAD KB and matrix, which for most layers is its whole share. No load hangs
// on a condition, a conversion or another load (each makes the compiler wait for all that are under way): rows and columns
// beyond the matrix are read from the last ones inside, and columns are multiplied as zeros. Against the kernels further
// down, which ask for two steps at a time and wait for the residual before the weights: 1,024 outputs of 2,048 and 3,072 columns
// added to a residual at 1 row 6.4 -> 4.9 us and 8.5 -> 6.3, at 16 rows 8.0 -> 6.0 and 11.1 -> 8.0; 4,096 of 4,096 at 8 rows
// 12.4 -> 10.4; 6,144 of 4,096 13.7 -> 12.2 and 15.4 -> 13.0 at 1 and 8; gated 9,728 of 2,560 26.3 -> 23.3, 3,072 of 1,024 at
// 16 rows 9.9 -> 6.8, with biases 6,144 of 2,048 at 5 rows 16.9 -> 13.8.
constexpr int TW = 16;                       // waves

// x into LDS, [M][K + 8] (the 16 bytes between rows spread the rows over the banks): a wave's load brings 64 consecutive
// 16-byte pieces of one row
__device__ __forceinline__ void ask_x(const bf16_t* __restrict__ x, bf16_t* x_s, int M, int K, int wave, int lane) {
  const int pieces_per_row = K / 8, loads_per_row = (pieces_per_row + 63) / 64;
  for (int job = wave; job < M * loads_per_row; job += TW) {
    const int m = job / loads_per_row, part = job % loads_per_row;
    if (part * 64 + lane < pieces_per_row)
      __builtin_amdgcn_global_load_lds((global_ptr)(x + (size_t)m * K + (part * 64 + lane) * 8), (lds_ptr)(x_s + m * (K + 8) + part * 512), 16, 0, 0);
  }
}
// The wait for x alone, when YOUNGER loads have been asked for since (a fence would wait for all). It holds only while exactly
// these loads, the weights' first ones, stand between x's and the wait, so the two kernels' w is no __restrict__ pointer: loads
// through one may legally cross an asm that clobbers memory, loads of memory that the asm may have written may not, neither this
// one nor the one in front of the first of them. (A test counts the loads in what the compiler makes of each kernel.)
template <int YOUNGER>
__device__ __forceinline__ void wait_for_x() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ bf16x8 masked(bf16x8 v, unsigned mask) { return (bf16x8)((uint4v)v & mask); }

// A tile's sums of the waves (red[wave][matrix][lane]), added in the order of the waves; then the rows' scales, the biases, the gate.
template <bool GLU, bool FUSED>
__device__ __forceinline__ void add_waves(const Fusion& f, const floatx4 (*red)[GLU ? 2 : 1][64], const float* r_s, bool biased, const float (&bias)[GLU ? 2 : 1][4],
                                          float (&out)[4], int lane) {
  constexpr int NA = GLU ? 2 : 1, SIDE = 8 / NA;                     // (so many at once: the registers that are left)
  floatx4 v[NA];
#pragma unroll
  for (int na = 0; na < NA; ++na) v[na] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int wv = 0; wv < TW; wv += SIDE) {
    floatx4 part[SIDE][NA];
#pragma unroll
    for (int i = 0; i < SIDE; ++i)
#pragma unroll
      for (int na = 0; na < NA; ++na) part[i][na] = red[wv + i][na][lane];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SIDE; ++i)
#pragma unroll
      for (int na = 0; na < NA; ++na) v[na] += part[i][na];
  }
  const float rs = (FUSED && f.ss_in) ? r_s[lane & 15] : 1.0f;       // the row's scale, where x is a sum whose norm is due
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float r = v[0][j] * rs, up = v[NA - 1][j] * rs;
    if (biased) r += bias[0][j], up += bias[NA - 1][j];
    if (GLU) r = nhv_gated(r, up, f.gate);
    else if (f.plain_act) r = nhv_plain_act(r, f.plain_act);
    out[j] = r;
  }
}

// One tile a block. XLDS: x is brought to LDS, its loads before the first weights', and the wait before the first product is
// for x alone; without, x comes from memory step by step beside w.
template <int AHEAD, bool GLU, bool XLDS, bool FUSED, typename TOut>
__global__ __launch_bounds__(64 * TW) void gemm_fewrows_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* w,
                                                                    const bf16_t* __restrict__ bias, TOut* __restrict__ y, int M, int N, int K,
                                                                    int rows, int groups, const Fusion f) {
  constexpr int NA = GLU ? 2 : 1;
  asm volatile("" ::"s"(w));               // (fetched with the other arguments, not where it is first used)
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  floatx4(*red)[NA][64] = reinterpret_cast<floatx4(*)[NA][64]>(lds_raw);       // [TW][NA][64]
  bf16_t* x_s = reinterpret_cast<bf16_t*>(lds_raw + TW * NA * sizeof(floatx4) * 64);
  __shared__ float r_s[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int n0 = blockIdx.x * rows, n = n0 + grp * 4;
  float share[SCALE_ROWS<TW>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<TW>(f, share, M, wave, lane);
  Four res, next_w, bias4[NA];               // what the wave that writes the tile needs beside the sums
  if (wave == 0) {
    const int n_in = min(n, N - 4);
    if constexpr (FUSED && !GLU) {
      res.ask(f.residual, (size_t)min(col, M - 1) * N + n_in, f.residual && f.residual_f32, w);
      next_w.ask(f.next_w, n_in, f.next_w && f.next_w_f32, w);
    }
#pragma unroll
    for (int na = 0; na < NA; ++na) bias4[na].ask(bias, (size_t)na * N + n_in, 0, w);
  }
  if constexpr (XLDS) ask_x(x, x_s, M, K, wave, lane);
  const int k0 = wave * groups * AHEAD * 32 + grp * 8, k_end = min((wave + 1) * groups * AHEAD * 32, K);
  const char *xb = reinterpret_cast<const char*>(x), *wb[2] = {reinterpret_cast<const char*>(w), reinterpret_cast<const char*>(w + (size_t)N * K)};
  const unsigned xrow = (unsigned)min(col, M - 1) * K * 2, wrow = (unsigned)min(n0 + min(col, rows - 1), N - 1) * K * 2;
  const bf16_t* xrow_s = x_s + min(col, M - 1) * (K + 8);
  bf16x8 a[AHEAD][NA], b[AHEAD];
  auto ask = [&](int u, int s) {
    const unsigned k = (unsigned)min(k0 + s * 32, K - 8) * 2;
#pragma unroll
    for (int na = 0; na < NA; ++na) a[u][na] = *reinterpret_cast<const bf16x8*>(wb[na] + (wrow + k));
    if constexpr (!XLDS) b[u] = *reinterpret_cast<const bf16x8*>(xb + (xrow + k));
  };
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) ask(u, u);
  if constexpr (XLDS) wait_for_x<AHEAD * NA>();
  floatx4 acc[NA];
#pragma unroll
  for (int na = 0; na < NA; ++na) acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int u, int s) {
    const int k = k0 + s * 32;
    const unsigned in = k < k_end ? ~0u : 0u;
    bf16x8 bu = b[u];
    if constexpr (XLDS) bu = *reinterpret_cast<const bf16x8*>(xrow_s + min(k, K - 8));
    bu = masked(bu, in);
#pragma unroll
    for (int na = 0; na < NA; ++na) {
      asm volatile("" : "+v"(a[u][na]));                             // (nothing of it is done before it is this step's turn)
      acc[na] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(masked(a[u][na], in), bu, acc[na], 0, 0, 0);
    }
  };
  int s = 0;
  for (int g = 1; g < groups; ++g, s += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      multiply(u, s + u);
      ask(u, s + AHEAD + u);
    }
  }
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) multiply(u, s + u);
  if constexpr (FUSED) set_row_scales<TW>(f, share, r_s, M, K, wave, lane);
#pragma unroll
  for (int na = 0; na < NA; ++na) red[wave][na][lane] = acc[na];
  lds_barrier();
  if (wave > 0) return;

  float out[4], bias_here[NA][4];
#pragma unroll
  for (int na = 0; na < NA; ++na)
#pragma unroll
    for (int j = 0; j < 4; ++j) bias_here[na][j] = bias4[na].at(j, 0);
  add_waves<GLU, FUSED>(f, red, r_s, bias != nullptr, bias_here, out, lane);
  const bool mine = col < M && grp * 4 < rows && n < N;
  const size_t at = (size_t)col * N + n;
  if (!FUSED || GLU || f.residual == nullptr) {
    if (mine) store4(y + at, out);
    return;
  }
  float sum[4], weighted[4], sq = 0.f;                               // (see emit_tile)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sum[j] = out[j] + res.at(j, f.residual_f32);
    weighted[j] = sum[j] * (f.next_w ? next_w.at(j, f.next_w_f32) : 1.0f);
    sq += mine ? sum[j] * sum[j] : 0.f;
  }
  if (mine) {
    if (f.residual_f32) store4((float*)f.residual + at, sum);
    else store4((bf16_t*)f.residual + at, sum);
    store4(f.sum_out + at, weighted);
  }
  sq += __shfl_xor(sq, 16, 64);
  sq += __shfl_xor(sq, 32, 64);
  if (grp == 0 && col < M) f.ss_out[(size_t)col * gridDim.x + blockIdx.x] = sq;
}

// `rows` rows of w a block, in tiles of `height`, without a residual: the next tile's weights are under way while a tile is
// finished, whose biases lie in LDS from the start (asked for tile by tile they would be waited for behind the weights). (After the last one each lane asks for the matrix's first bytes instead: with a branch there the compiler
// waits for all loads before it uses one.)
template <int AHEAD, bool GLU, bool FUSED, bool BIASED, typename TOut>
__global__ __launch_bounds__(64 * TW) void gemm_fewrows_walk_kernel(const bf16_t* __restrict__ x, const bf16_t* w,
                                                                    const bf16_t* __restrict__ bias, TOut* __restrict__ y, int M, int N, int K, int rows, int height, int groups, const Fusion f) {
  constexpr int NA = GLU ? 2 : 1;
  asm volatile("" ::"s"(w));               // (fetched with the other arguments, not where it is first used)
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  floatx4(*red)[NA][64] = reinterpret_cast<floatx4(*)[NA][64]>(lds_raw);       // [2 TW][NA][64]: one tile's and the next one's
  bf16_t* x_s = reinterpret_cast<bf16_t*>(lds_raw + 2 * TW * NA * sizeof(floatx4) * 64);
  float* bias_s = reinterpret_cast<float*>(x_s + M * (K + 8));                 // [NA][rows] and what a lane beyond the last tile reads
  __shared__ float r_s[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  float share[SCALE_ROWS<TW>][SCALE_SHARES];
  if constexpr (FUSED) ask_row_scales<TW>(f, share, M, wave, lane);
  const int k0 = wave * groups * AHEAD * 32 + grp * 8, k_end = min((wave + 1) * groups * AHEAD * 32, K);
  const char* wb[2] = {reinterpret_cast<const char*>(w), reinterpret_cast<const char*>(w + (size_t)N * K)};
  const bf16_t* xrow_s = x_s + min(col, M - 1) * (K + 8);
  // (blocks side by side have tiles side by side: 2 % less time than with all of a block's rows in one place)
  const int tiles = (rows + height - 1) / height;
  auto height_of = [&](int tile) { return tile + 1 < tiles ? height : rows - (tiles - 1) * height; };
  auto first_of = [&](int tile) { return tile * (int)gridDim.x * height + (int)blockIdx.x * height_of(tile); };
  auto row_of = [&](int tile) { return (unsigned)min(first_of(tile) + min(col, height_of(tile) - 1), N - 1) * K * 2; };
  int tile = 0, turn = 0, parity = 0, g = 0;
  unsigned bias_bits = 0;                                            // one a thread: NA rows are no more than the block's threads
  if constexpr (BIASED) {
    const int mine = min((int)threadIdx.x, NA * rows - 1), my_row = mine % rows;
    bias_bits = reinterpret_cast<const unsigned short*>(bias)[(size_t)(mine / rows) * N + min(first_of(my_row / height) + my_row % height, N - 1)];
  }
  ask_x(x, x_s, M, K, wave, lane);
  bf16x8 a[AHEAD][NA];
  auto ask = [&](int u, unsigned at) {
#pragma unroll
    for (int na = 0; na < NA; ++na) a[u][na] = *reinterpret_cast<const bf16x8*>(wb[na] + at);
  };
  auto k_of = [&](int s) { return (unsigned)min(k0 + s * 32, K - 8) * 2; };
  unsigned row = row_of(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) ask(u, row + k_of(u));
  wait_for_x<AHEAD * NA>();
  if constexpr (BIASED) if ((int)threadIdx.x < NA * rows) bias_s[threadIdx.x] = __uint_as_float(bias_bits << 16);
  if constexpr (FUSED) set_row_scales<TW>(f, share, r_s, M, K, wave, lane);
  floatx4 acc[NA];
#pragma unroll
  for (int na = 0; na < NA; ++na) acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
  while (true) {
    const bool last = g + 1 == groups, more = !last || (tile + 1 < tiles && first_of(tile + 1) < N);
    const unsigned row_next = last ? row_of(tile + 1) : row;
    const int s_next = last ? 0 : (g + 1) * AHEAD;
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int k = k0 + (g * AHEAD + u) * 32;
      const unsigned in = k < k_end ? ~0u : 0u;
      const bf16x8 bu = masked(*reinterpret_cast<const bf16x8*>(xrow_s + min(k, K - 8)), in);
#pragma unroll
      for (int na = 0; na < NA; ++na) {
        asm volatile("" : "+v"(a[u][na]));                           // (nothing of it is done before it is this step's turn)
        acc[na] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(masked(a[u][na], in), bu, acc[na], 0, 0, 0);
      }
      ask(u, more ? row_next + k_of(s_next + u) : 0u);
    }
    ++g;
    if (!last) continue;
    floatx4(*my_red)[NA][64] = red + parity * TW;
#pragma unroll
    for (int na = 0; na < NA; ++na) {
      my_red[wave][na][lane] = acc[na];
      acc[na] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    lds_barrier();
    if (wave == turn) {
      float out[4], bias_here[NA][4];
#pragma unroll
      for (int na = 0; na < NA; ++na)
#pragma unroll
        for (int j = 0; j < 4; ++j) bias_here[na][j] = BIASED ? bias_s[na * rows + tile * height + grp * 4 + j] : 0.f;
      add_waves<GLU, FUSED>(f, my_red, r_s, BIASED, bias_here, out, lane);
      const int n = first_of(tile) + grp * 4;
      if (col < M && grp * 4 < height_of(tile) && n < N) store4(y + (size_t)col * N + n, out);
    }
    if (!more) break;
    ++tile, row = row_next, g = 0, parity ^= 1, turn = turn + 1 == TW ? 0 : turn + 1;
  }
}

constexpr size_t LDS_BYTES = 160 * 1024 - 64;      // (64 bytes are the rows' scales, which every kernel keeps beside)
// How the kernels above are launched; ahead == 0 where they are not the ones to take.
static int even_rows(int N) { return 4 * ((N + 4 * 256 - 1) / (4 * 256)); }
struct TilesPlan {
  int ahead;
  bool x_in_lds;
  int rows, height, groups;                                 // rows of w a block and a tile
  size_t lds;
};
// square_rows: outputs whose squares go out together, which are then a block's (0: no residual).
static TilesPlan tiles_plan(bool glu, int square_rows, bool biased, int M, int N, int K) {
  const bool squares = square_rows > 0;
  TilesPlan p = {};
  if (N % 4 || (size_t)N * K * sizeof(bf16_t) >> 32) return p;       // (four outputs a store; places in w are 32 bits)
  // as many rows a block as give each of the 256 compute units the same
  p.rows = squares ? square_rows : even_rows(N);
  const int tiles = (p.rows + 15) / 16;
  p.height = 4 * ((p.rows + 4 * tiles - 1) / (4 * tiles));
  const size_t sums = (size_t)(tiles > 1 ? 2 : 1) * TW * (glu ? 2 : 1) * 64 * sizeof(floatx4), x_bytes = (size_t)M * (K + 8) * 2;
  const size_t biases = tiles > 1 && biased ? ((glu ? 2 : 1) * p.rows + 16) * sizeof(float) : 0;
  p.x_in_lds = sums + x_bytes + biases <= LDS_BYTES;
  // (Of the sizes quoted here, those of a multiple of 256 columns go by lines now, but for what lines_plan() leaves.)
  // The kernels below it is where a product of several tiles a block has more biases than threads, and where x does not fit into LDS,
  // but for up to 8 rows on the whole chip (4,096 outputs of 12,288 columns at 8 rows 25.2 against 26.8 us; 3,584 of 18,944 on
  // 224 units, where x beside w is too much for a unit, 36.4 against 33.9; 4,096 of 12,288 at 16 rows 31.4 against 30.7).
  if (tiles > 1 && biases > (64 * TW + 16) * sizeof(float)) return p;
  if (!p.x_in_lds && (glu || tiles > 1 || M > 8 || N <= 240 * p.rows)) return p;
  // With a residual and more than 4,096 outputs a unit has a block or two. These kernels are the faster ones then too (5,120 outputs of 5,120
  // columns at 1 and 8 rows 17.3 against 19.8 us and 21.1 against 24.3; 5,120 of 17,408 at 4 rows 49.9 against 54.7; 8,192 of
  // 28,672 at 1 row 91.7 against 93.8), except where x does not fit into LDS (5,120 of 17,408 at 8 rows 65.0 against 58.6; of 25,600
  // 95.2 against 79.5; the only ones slower below it: 12,288 at 6 rows, 42.5 against 44.5) and for one row of many columns
  // that some units take twice (5,120 of 20,480 57.4 against 56.7, of 22,528 62.3 against 58.4, of 25,600 72.2 against 66.2).
  if (squares && N > 256 * p.rows && (!p.x_in_lds || (M == 1 && K > 20480 && N < 512 * p.rows))) return p;
  p.lds = sums + (p.x_in_lds ? x_bytes + biases : 0);
  const int steps = ((K + 31) / 32 + 15) / 16;
  int slots = 1 << 30;
  for (int u : {2, 3, 4, 5, 6, 7, 8}) {            // the fewest steps in all, and as many at once as can be
    if (u > (glu ? 5 : p.x_in_lds ? 8 : 6)) continue;
    const int groups = (steps + u - 1) / u;
    if (groups * u <= slots) p.ahead = u, p.groups = groups, slots = groups * u;
  }
  // So it is where a gated product walks over three tiles and more that come out even anyway (12,288 outputs of 4,096 columns at
  // 4 rows: 38.0 against 39.1 us) or whose steps do not come out even here (18,944 of 3,584 at 8 rows: 53.3 against 54.6).
  if (glu && tiles > 2 && (p.rows % 16 == 0 || slots != steps)) p.ahead = 0;
  return p;
}

template <int AHEAD, bool GLU, bool XLDS, bool FUSED, typename TOut>
static int launch_tiles(const TilesPlan& p, hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const Fusion& f) {
  // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
  auto once = gemm_fewrows_tile_kernel<AHEAD, GLU, XLDS, FUSED, TOut>;
  static const hipError_t allowed = hipFuncSetAttribute((const void*)once, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
  if (allowed != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(allowed));
  const dim3 grid((N + p.rows - 1) / p.rows);
  if (p.rows == p.height) {
    hipLaunchKernelGGL(once, grid, dim3(64 * TW), p.lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (TOut*)y, M, N, K,
                       p.rows, p.groups, f);
  } else if constexpr (XLDS) {
    // (the biases' reads cost a product without any 1 % as a condition)
    auto without = gemm_fewrows_walk_kernel<AHEAD, GLU, FUSED, false, TOut>, with = gemm_fewrows_walk_kernel<AHEAD, GLU, FUSED, true, TOut>;
    static const hipError_t allowed_too[2] = {hipFuncSetAttribute((const void*)without, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES),
                                              hipFuncSetAttribute((const void*)with, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES)};
    for (hipError_t e : allowed_too)
      if (e != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(e));
    hipLaunchKernelGGL(bias ? with : without, grid, dim3(64 * TW), p.lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (TOut*)y, M, N, K, p.rows, p.height,
                       p.groups, f);
  }
  return 0;
}

// The kernel for rows of w that fill the chip in tiles of 16 (see lines_plan): w and x through LDS in chunks of 256 columns, a row's
// 512 bytes in one piece, in a ring of NB chunks; a block is 8 waves, each with 32 of a chunk's columns, and a chunk costs one
// barrier. The kernels above and below bring 16 rows of 64 bytes a load, of which a compute unit takes in 17 to 20 GB/s; pieces of
// 512 bytes come at the memory's own rate. Their places are turned by the row, so that 16 rows lie in different banks. NT tiles of w a
// block (gated: one and its partner). us at 1, 8 and 16 rows, before and now: 6,144 outputs of 4,096 columns 12.6, 13.7, 17.7 and 11.7,
// 12.1, 12.6; 4,096 of 4,096 10.2, 10.6, 11.8 and 8.4, 8.6, 8.9; gated 12,288 of 4,096 42.8, 43.3, 48.6 and 36.3, 35.9, 36.5 (a kernel that only
// reads: 32.5); 4,096 of 12,288 23.0, 28.2, 31.0 and 19.7, 20.2, 22.1; 151,936 of 4,096 204, 216, 270 and 196, 198, 201 (201);
// gated 9,728 of 2,560 25.5, 26.0, 26.3 and 22.5, 22.9, 23.6.
// SKIPS: up to 8 rows, whose waves without rows of x bring none (in their place the others bring the last one: 2,560 outputs of 4,096 columns at 1 and
// 4 rows 7.5 and 7.6 us, with it 6.9 and 7.1; 2,560 of 9,728 15.2 and 15.3, 14.0 and 14.7; 3,584 of 18,944 25.9 and 26.1, 24.9 and 25.6). Not for
// gated products (12,288 of 4,096 at 1 and 8 rows 33.7 and 33.1 us, with it 35.5 and 34.2) nor for float results, whose stretches are summed apart.
// HALF: 8 rows of w a block, where 16 leave units idle: the lower half of the waves brings them, all of them bring x.
template <int NT, int NB, bool GATED, typename TOut, bool SKIPS, bool HALF>
__global__ __launch_bounds__(512) void gemm_fewrows_lines_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                                                 TOut* __restrict__ y, int M, int N, int K, const Fusion f) {
  constexpr int OUT = GATED ? 1 : NT, BOTH = GATED ? 2 : 1, CHUNK = 256, LOADS = NT + 1, STAGE = (NT + 1) * 16 * CHUNK, ROWS_W = HALF ? 8 : 16;
  static_assert(!HALF || (NT == 1 && !GATED && !SKIPS), "half tiles are a block's only ones");
  // (a name of its own: an array of this alignment under the others' name would cost the kernels around their last 1,024 bytes)
  extern __shared__ __attribute__((aligned(1024))) bf16_t line_ring[];
  const bf16_t* ring = line_ring;
  __shared__ float r_s[16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * ROWS_W * OUT, chunks = K / CHUNK;
  if (f.band_rows) x += (size_t)min(n0 / f.band_rows, f.bands - 1) * M * K;      // (a block's tiles lie in one band)
  // what the thread that finishes output (row, n) needs beside the sums, asked for before the weights
  const int row = (threadIdx.x >> 4) & 15, tile = threadIdx.x >> 8, n = n0 + 16 * tile + (threadIdx.x & 15);
  const bool mine = tile < OUT && row < M && n < N && (int)(threadIdx.x & 15) < ROWS_W;
  float share[SCALE_ROWS<8>][SCALE_SHARES];
  ask_row_scales<8>(f, share, M, wave, lane);
  float res = 0.f, next_w = 1.f, add[2] = {0.f, 0.f};
  if (mine) {
    if (f.residual) res = f.residual_f32 ? ((const float*)f.residual)[(size_t)row * N + n] : (float)((const bf16_t*)f.residual)[(size_t)row * N + n];
    if (f.next_w) next_w = f.next_w_f32 ? ((const float*)f.next_w)[n] : (float)((const bf16_t*)f.next_w)[n];
    if (bias) {
      add[0] = (float)bias[n];
      if (GATED) add[1] = (float)bias[N + n];
    }
  }
  // what this lane brings of a chunk: 16 bytes of row 2 wave + lane / 32 of every tile, the last tile x's. Rows beyond the matrices are their last
  // ones (their results are dropped).
  const bf16_t* src[LOADS];
  const int my_row = 2 * wave + (lane >> 5), piece = (lane & 31) ^ my_row;
#pragma unroll
  for (int t = 0; t < LOADS; ++t)
    src[t] = (t < NT ? w + ((size_t)(GATED ? t * N : 0) + min(n0 + (GATED ? 0 : 16 * t) + my_row, N - 1)) * K : x + (size_t)min(my_row, M - 1) * K) + piece * 8;
  const uint32_t ring_at = nhv_lds_address(ring) + wave * 1024;
  // Float results are logits, and equal rows of w (unused tokens' embeddings) have to give equal ones, or rounding would choose
  // between them: there the sums do not begin where the block does. The columns are STRETCHES stretches, a block begins with one
  // of them, and each is summed by itself and added to the others in their order. us at 1 and 16 rows without the turning, with
  // it, with it and two, four and eight stretches: 151,936 outputs of 4,096 columns 246 and 252, 187 and 192, 196 and 199, 187
  // and 191, 198 and 205; 151,936 of 2,048 120 and 128, 97 and 113, 98 and 115, 97 and 114, 132 and 140 (an eighth is one chunk).
  constexpr int STRETCHES = sizeof(TOut) == 4 ? 4 : 1;
  const bool stretches = STRETCHES > 1 && K % 2048 == 0;
  const int length = stretches ? chunks / STRETCHES : chunks + 1, place = nhv_first_chunk(blockIdx.x, chunks, K), first = stretches ? place / length * length : place;
  auto ask = [&](auto brings_w, auto brings_x, int buf, int c) {
    const size_t k = (size_t)nhv_chunk(first, c, chunks) * CHUNK;
#pragma unroll
    for (int t = decltype(brings_w)::value ? 0 : NT; t < (decltype(brings_x)::value ? LOADS : NT); ++t) {
      if (t < NT) nhv_load_to_lds<true>(ring_at + (buf * STAGE + t * 16 * CHUNK) * 2, src[t] + k);
      else nhv_load_to_lds<false>(ring_at + (buf * STAGE + t * 16 * CHUNK) * 2, src[t] + k);
    }
  };
  floatx4 acc[NT], done[STRETCHES][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < STRETCHES; ++i) done[i][t] = acc[t];
  }
  const int at = r16 * CHUNK + (((wave * 4 + g) ^ r16) << 3);
  if constexpr (!SKIPS && !HALF) {
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) ask(std::true_type{}, std::true_type{}, i, i);
    int buf = 0, now = first / length, left = length;
    for (int c = 0; c < chunks; ++c) {
      nhv_wait_and_meet<(NB - 2) * LOADS>();                            // chunk c is there, chunk c - 1 has been read
      ask(std::true_type{}, std::true_type{}, buf == 0 ? NB - 1 : buf - 1, c + NB - 1);
      const bf16_t* from = ring + buf * STAGE + at;
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(from + NT * 16 * CHUNK);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, *reinterpret_cast<const bf16x8*>(from + t * 16 * CHUNK), acc[t], 0, 0, 0);
      buf = buf == NB - 1 ? 0 : buf + 1;
      if (STRETCHES > 1 && --left == 0) {                               // (the same for the whole block)
#pragma unroll
        for (int i = 0; i < STRETCHES; ++i)
          if (i == now) {
#pragma unroll
            for (int t = 0; t < NT; ++t) done[i][t] = acc[t];
          }
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
        now = now == STRETCHES - 1 ? 0 : now + 1;
        left = length;
      }
    }
  } else {
    // a wave whose rows of x (HALF: of w) are not there brings none (what lies in LDS in their place comes into rows or columns whose
    // results are dropped)
    auto walk = [&](auto brings_w, auto brings_x) {
#pragma unroll
      for (int i = 0; i < NB - 1; ++i) ask(brings_w, brings_x, i, i);
      int buf = 0;
      for (int c = 0; c < chunks; ++c) {
        nhv_wait_and_meet<(NB - 2) * ((decltype(brings_w)::value ? NT : 0) + (decltype(brings_x)::value ? 1 : 0))>();
        ask(brings_w, brings_x, buf == 0 ? NB - 1 : buf - 1, c + NB - 1);
        const bf16_t* from = ring + buf * STAGE + at;
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(from + NT * 16 * CHUNK);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, *reinterpret_cast<const bf16x8*>(from + t * 16 * CHUNK), acc[t], 0, 0, 0);
        buf = buf == NB - 1 ? 0 : buf + 1;
      }
    };
    if (HALF ? wave < 4 : 2 * wave < M) walk(std::true_type{}, std::true_type{});
    else if constexpr (HALF) walk(std::false_type{}, std::true_type{});
    else walk(std::true_type{}, std::false_type{});
  }
  if (stretches) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      acc[t] = done[0][t];
#pragma unroll
      for (int i = 1; i < STRETCHES; ++i) acc[t] += done[i][t];
    }
  }
  nhv_wait_and_meet<0>();                                             // (the ring becomes room for the sums)
  float* part = reinterpret_cast<float*>(line_ring);                    // [tile][wave][256]
#pragma unroll
  for (int t = 0; t < NT; ++t) *reinterpret_cast<floatx4*>(&part[(t * 8 + wave) * 256 + lane * 4]) = acc[t];
  set_row_scales<8>(f, share, r_s, M, K, wave, lane);
  __syncthreads();
  if (tile >= OUT) return;                                            // (whole waves)
  // (lane 16 g + c of a tile holds rows 4 g .. 4 g + 3 of column c; the waves' sums in their order)
  float v[BOTH];
#pragma unroll
  for (int both = 0; both < BOTH; ++both) {
    const float* from = &part[(GATED ? both : tile) * 2048 + (row >> 2) * 64 + (threadIdx.x & 15) * 4 + (row & 3)];
    v[both] = 0.f;
#pragma unroll
    for (int wv = 0; wv < 8; ++wv) v[both] += from[wv * 256];
    if (f.ss_in) v[both] *= r_s[row];                                 // (r_s of rows beyond M is not set, nor used below)
    v[both] += add[both];
  }
  float out = GATED ? nhv_gated(v[0], v[BOTH - 1], f.gate) : f.plain_act ? nhv_plain_act(v[0], f.plain_act) : v[0];
  if (GATED || f.residual == nullptr) {
    if (mine) y[(size_t)row * N + n] = (TOut)out;
    return;
  }
  out += res;                                                         // (see emit_tile)
  if (mine) {
    if (f.residual_f32) ((float*)f.residual)[(size_t)row * N + n] = out;
    else ((bf16_t*)f.residual)[(size_t)row * N + n] = (bf16_t)out;
    f.sum_out[(size_t)row * N + n] = (bf16_t)(out * next_w);
  }
  float sq = mine ? out * out : 0.f;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) sq += __shfl_xor(sq, o, 64);
  const int tiles = (N + 15) / 16, my_tile = blockIdx.x * OUT + tile;
  if ((threadIdx.x & 15) == 0 && row < M && my_tile < tiles) f.ss_out[(size_t)row * tiles + my_tile] = sq;
}

// What else a product is, beside its sizes.
struct Form {
  bool glu, residual, banded;
  bool scaled;                                              // x is a sum whose rows lack their norm's scales
  bool floats;                                              // a float result
};

// Blocks of 8 outputs, by lines, for a bfloat16 result of 1,025 to 2,048 outputs without residual, where the tiles above have 8 rows of w a block
// as well: they differ by a block's fixed cost and by how x comes. Measured over nine numbers of outputs by twelve of columns (2,048 to 8,192)
// at ten numbers of rows; time by blocks of 8 over the tiles': from 9 rows on 0.55 to 1.0 nearly everywhere; up to 2,304 columns 0.91 to 1.01 from 4 rows on;
// with more, from where w has 2,048 x 2,816 entries, 0.90 to 1.0 at 6 and 7 rows (below that 0.95 to 1.0 for 2,816 and 3,072 columns, up to 1.07 for others: 1,536 of 3,584 1.05, 1,040 of 5,120 1.07), 0.90
// to 1.0 at 8 (below 0.98 to 1.07 beyond 3,072 columns). At 4 and 5 rows 2,048 of 3,072 0.99 and 0.98, of 4,096 0.97 and 0.95, but 1,280 of 3,584 1.05 and
// 1.04, 1,536 of 5,120 1.02 and 1.0. us: 2,048 of 2,048 at 4 and 16 rows 4.9, 5.2 and 4.8, 4.9; of 4,096 at 4 and 7 6.9, 7.2 and 6.6, 6.8; of 12,288 at 8 and 16 16.9,
// 17.5 and 14.7, 15.2. ``scaled``: such a block takes 0.5 us more and the tiles 0.1: below those 2,048 x 2,816 entries 1.0 to 1.13 at 6 to 8 rows (2,048 of 2,560 1.08,
// 1,040 of 5,120 1.13), from there on 0.95 to 1.02; at 12 and 16 rows 0.83 to 1.03 for 2,816 to 4,096 columns (2,304: 0.96 to 1.0 and 0.92 to 0.98), up to 1.09 for others, but 0.57 to 0.71 where x
// no longer fits beside w in the tiles' LDS (16 rows of 4,608 columns, 12 of 6,144).
static bool half_plan(bool scaled, int M, int N, int K) {
  if (N <= 1024 || N > 2048) return false;
  const bool many = (long long)N * K >= 2048 * 2816;
  if (scaled) return (M >= 6 && many && (K <= 5120 || M >= 8)) || (M >= 12 && K > (M >= 14 ? 2048 : 2560) && K <= 4096) || (M >= 8 && M * K >= 16 * 4608);
  if (M >= 9 || K <= 2304 || (M >= 8 && K <= 3072) || (M >= 6 && K > 2560 && K <= 3072)) return M >= 4;
  if (!many || M < 4 || (K > 5120 && M < 8)) return false;
  return M >= 6 || (K <= 4096 && N >= 1920) || (M == 5 && K >= 4096);
}

// Fewer than 8 rows and 2,560 to 4,095 outputs: where the tiles above are the faster ones all the same, of 2,048 columns above all, which are a
// ring's two fillings. Time by lines over theirs at 1, 2, 4 and 7 rows: rows to scale, 2,560 outputs of 2,048 columns 1.09, 1.09, 1.05, 1.07, 2,816 1.06, 1.07, 1.02,
// 1.02, 3,072 1.0, 1.03, 0.99, 0.98; 2,560 of 3,072 1.03, 1.04, 0.99, 0.96, of 2,304 0.98, 0.97, 0.96, 0.94; added to the residual stream as well, 2,560 of 2,048 1.06,
// 1.07, 1.0, 1.0, 2,816 1.04, 1.01, 0.97, 0.96. (Neither: 2,560 of 2,048 1.04, 1.05, 0.97, 1.0, which is left by lines, 2,816 0.99, 0.99, 0.92, 0.96; the
// addition alone never above 1.0.) In bands, whose other way is the kernel that takes x from memory: 2,560 outputs 1.08, 1.05, 1.02, 1.01, 2,816 1.04, 1.02, 0.99, 0.95,
// 3,584 1.02, 0.98, 0.96, 0.89; of 2,304 0.88 to 0.8. Float results are summed in stretches where K is a multiple of 2,048: 2,560
// outputs of 4,096 columns 7.1 us by the tiles and 7.8 at 1 row, 7.4 and 7.9 at 4; 3,072 of 2,048 1.02, 1.03, 0.96, 0.99, of 6,144 9.9 and 9.8, 10.5 and 9.9.
static bool lines_lose(const Form& p, int M, int N, int K) {
  if (p.banded) return K == 2048 && (N < 2816 || M == 1);
  if (p.floats) return K % 2048 == 0 && N < (K > 2048 ? 3072 : M <= 2 ? 3200 : 2944);
  if (p.residual) return p.scaled && K == 2048 && N < 2944 && M < 4;
  return p.scaled && (K == 2048 ? N < (M < 4 ? 3072 : 2944) : N < 2944 && M <= 2 && K > 2304 && K <= 3072);
}

// Where the rows of w are enough for it, by what was measured at 1, 4, 8, 12 and 16 rows (us before and with it): not for 4,096 outputs
// of 1,024 columns (4.2, 4.9 at 1 row) or a gated 3,072 of 1,024 (5.5, 5.7); with fewer than 2,560 outputs a tile of 16 leaves units idle,
// which the smaller tiles above do not, until there are so many rows that these are slower: 2,560 of 4,096 7.7, 6.9 at 1 row and 7.8, 7.1 at 4;
// 2,560 of 9,728 14.6, 14.0 and 15.3, 14.7; 3,584 of 3,584 8.5, 7.6 and 8.7, 7.8; 3,072 of 8,192 12.9, 12.0 and 13.6, 12.2; 2,048 of 6,144 8.3, 11
// at 1 and 9.5, 11.1 at 8, but 14.3, 11.5 at 12; 2,048 of 2,048 never (all by blocks of 16 outputs).
// ``even`` (in the rule): the tiles above would take the product and give every unit the same rows of w (with a residual they do so for fewer than 4,096 outputs
// alone, see nhv_gemm_fewrows_square_rows; with bands never). They stay the faster ones where the blocks of 32 outputs are a round and a bit (time by lines over theirs, K = 2,048
// to 12,288, at 1 to 8 rows: 8,448 outputs 1.07 to 1.18, 9,216 1.07 to 1.17, 10,240 1.00 to 1.11 and at K = 2,048 0.95, 11,264 0.96 to 1.07, 12,288 0.88 to
// 1.04; 16 rows: K = 3,072 1.05 to 1.15, from 4,096 on 0.62 to 0.88), and with rows 16 KB apart on some of the units (K = 8,192: 4,224
// to 6,144 outputs 1.06 to 1.22 at 1 to 4 rows, 0.81 to 0.99 at 8; 7,168 outputs 0.80 to 0.87), as long as all of x fits beside w.
static bool lines_plan(const Form& p, int M, int N, int K) {
  if (K % 256 != 0 || K < 2048) return false;
  if (p.glu) return N >= 4096;
  const bool even = !p.residual && !p.banded;
  if (even && N > 8192 && N <= (K > 2048 ? 11264 : 9216) && (long long)M * K <= 57344) return false;
  if (even && N > 4096 && N < 7168 && K % 8192 == 0 && (long long)M * K <= 32768) return false;
  if (even && !p.floats && half_plan(p.scaled, M, N, K)) return true;
  if (M < 8 && N < 4096 && lines_lose(p, M, N, K)) return false;
  return N >= 2560 || (N >= 2048 && K >= 4096 && M >= 12);
}

template <int NT, int NB, bool GATED, typename TOut, bool SKIPS, bool HALF = false>
static int launch_lines_as(hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const Fusion& f) {
  constexpr int OUT = HALF ? 8 : GATED ? 16 : 16 * NT, ring = NB * (NT + 1) * 16 * 512, sums = NT * 8192, lds = ring > sums ? ring : sums;
  auto kernel = gemm_fewrows_lines_kernel<NT, NB, GATED, TOut, SKIPS, HALF>;
  // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
  static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (allowed != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(allowed));
  hipLaunchKernelGGL(kernel, dim3((N + OUT - 1) / OUT), dim3(512), lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (TOut*)y, M, N, K, f);
  return 0;
}
// One block a compute unit: four chunks in the ring; several: three.
template <bool GATED, bool SKIPS, typename TOut>
static int launch_lines_of(hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const Fusion& f) {
  if constexpr (GATED) {
    return N <= 256 * 16 ? launch_lines_as<2, 4, true, TOut, false>(s, x, w, bias, y, M, N, K, f)
                         : launch_lines_as<2, 3, true, TOut, false>(s, x, w, bias, y, M, N, K, f);
  } else {
    if (N <= 256 * 16) return launch_lines_as<1, 4, false, TOut, SKIPS>(s, x, w, bias, y, M, N, K, f);
    return N <= 256 * 32 ? launch_lines_as<2, 4, false, TOut, SKIPS>(s, x, w, bias, y, M, N, K, f) : launch_lines_as<2, 3, false, TOut, SKIPS>(s, x, w, bias, y, M, N, K, f);
  }
}
template <bool GATED, typename TOut>
static int launch_lines(hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N, int K, const Fusion& f) {
  if constexpr (!GATED && sizeof(TOut) == 2) {
    if (N <= 128 * 16 && !f.residual) return launch_lines_as<1, 4, false, TOut, false, true>(s, x, w, bias, y, M, N, K, f);
    if (M <= 8) return launch_lines_of<false, true, TOut>(s, x, w, bias, y, M, N, K, f);
  }
  return launch_lines_of<GATED, false, TOut>(s, x, w, bias, y, M, N, K, f);
}

// The resident kernel's shape: waves, loads in flight and blocks per compute unit, from the best variants measured
// (same shapes as below), and in how many pieces x comes; waves == 0 when this kernel is not the one to take.
struct ResidentPlan {
  int waves, unroll, blocks_per_cu, nchunks, chunk_steps;
  size_t lds;
};
static ResidentPlan resident_plan(bool glu, int M, int N, int K) {
  const int tiles = (N + 15) / 16, ksteps = (K + 31) / 32;
  auto lds_of = [&](int waves, int steps) {
    const int columns = steps * 32 < K ? steps * 32 : K;
    return (size_t)2 * waves * (glu ? 2 : 1) * 4 * 64 * sizeof(float) + (size_t)M * (columns + 8) * 2;
  };
  int waves, unroll;
  if (glu) {
    waves = M <= 12 ? 8 : 4;
    unroll = M <= 12 ? 2 : 8;
  } else if (M >= 13) {
    waves = 8, unroll = 8;
  } else if (tiles <= 256 || M > 4 || tiles > 2048) {
    waves = 16, unroll = 2;
  } else {
    waves = 8, unroll = 2;
  }
  int nchunks = 1, chunk_steps = ksteps;
  if (lds_of(waves, ksteps) > LDS_BYTES) {      // fewer waves need less room for their sums
    const int fewer = glu ? 4 : 8;
    if (lds_of(fewer, ksteps) <= LDS_BYTES) {
      waves = fewer, unroll = 8;
    } else {
      // x in pieces: only where every block has one tile (the pieces would come again for every tile) and all
      // blocks are on the chip at once, one a compute unit (with 320 tiles it was measured slower by a quarter)
      if (glu || tiles > 256) return {0, 0, 0, 0, 0, 0};
      for (nchunks = 2; nchunks <= 16; ++nchunks) {
        chunk_steps = 2 * waves * ((ksteps + 2 * waves * nchunks - 1) / (2 * waves * nchunks));   // every wave whole lines
        if (lds_of(waves, chunk_steps) <= LDS_BYTES) break;
      }
      if (nchunks > 16) return {0, 0, 0, 0, 0, 0};
      nchunks = (ksteps + chunk_steps - 1) / chunk_steps;
    }
  }
  if (!glu && waves == 8 && unroll == 2 && 2 * lds_of(8, chunk_steps) > LDS_BYTES) {
    // one block a compute unit: eight waves with two loads each are too little in flight
    if (lds_of(16, chunk_steps) <= LDS_BYTES) waves = 16;
    else unroll = 8;
  }
  const size_t lds = lds_of(waves, chunk_steps);
  const int by_lds = (int)(LDS_BYTES / lds), by_waves = 32 / waves;
  const int bpc = by_lds < by_waves ? by_lds : by_waves;
  return {waves, unroll, bpc < 2 ? 1 : 2, nchunks, chunk_steps, lds};
}

template <int WAVES, int UNROLL, bool GLU, bool PIECES, bool FUSED, typename TOut>
static int launch_resident(const ResidentPlan& p, hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M,
                           int N, int K, const Fusion& f) {
  static_assert(!(GLU && PIECES), "x in pieces is not built for the gated kernel");
  const int steps_per_wave = 2 * ((p.chunk_steps + 2 * WAVES - 1) / (2 * WAVES));
  const int tiles = (N + 15) / 16;
  if constexpr (PIECES) {
    auto kernel = gemm_fewrows_pieces_kernel<WAVES, UNROLL, FUSED, TOut>;
    // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
    static const hipError_t allowed =
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
    if (allowed != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(allowed));
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(64 * WAVES), p.lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias,
                       (TOut*)y, M, N, K, tiles, p.nchunks, p.chunk_steps, steps_per_wave, f);
  } else {
    auto kernel = gemm_fewrows_resident_kernel<WAVES, UNROLL, GLU, FUSED, TOut>;
    static const hipError_t allowed =
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
    if (allowed != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(allowed));
    const int grid = tiles < 256 * p.blocks_per_cu ? tiles : 256 * p.blocks_per_cu;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * WAVES), p.lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias,
                       (TOut*)y, M, N, K, tiles, steps_per_wave, f);
  }
  return 0;
}

// The shape of the kernel that takes x in pieces and walks over all of a block's tiles for every piece: one
// block a compute unit; waves == 0 when it does not fit.
struct PassesPlan {
  int waves, unroll, npasses, pass_steps, tiles_per_block, grid;
  size_t lds;
};
static PassesPlan passes_plan(bool glu, int M, int N, int K) {
  const int tiles = (N + 15) / 16, ksteps = (K + 31) / 32;
  const int grid = tiles < 256 ? tiles : 256;
  const int tpb = (tiles + grid - 1) / grid;
  int waves, unroll;
  if (glu) waves = M <= 12 ? 8 : 4, unroll = M <= 12 ? 2 : 8;
  else waves = M >= 13 ? 8 : 16, unroll = M >= 13 ? 8 : 2;
  const int na = glu ? 2 : 1;
  for (int npasses = 2; npasses <= 8; ++npasses) {
    const int pass_steps = 2 * waves * ((ksteps + 2 * waves * npasses - 1) / (2 * waves * npasses));   // every wave whole lines
    const int columns = pass_steps * 32 < K ? pass_steps * 32 : K;
    const size_t lds = (size_t)(2 * waves + tpb) * na * 4 * 64 * sizeof(float) + (size_t)M * (columns + 8) * 2;
    if (lds <= LDS_BYTES) return {waves, unroll, (ksteps + pass_steps - 1) / pass_steps, pass_steps, tpb, grid, lds};
  }
  return {0, 0, 0, 0, 0, 0, 0};
}

template <int WAVES, int UNROLL, bool GLU, bool FUSED, typename TOut>
static int launch_passes(const PassesPlan& p, hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N,
                         int K, const Fusion& f) {
  auto kernel = gemm_fewrows_passes_kernel<WAVES, UNROLL, GLU, FUSED, TOut>;
  // more than 64 KB of dynamic LDS has to be allowed once per kernel (and per process)
  static const hipError_t allowed =
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
  if (allowed != hipSuccess) return nhv_fail("few-rows gemm: %s", hipGetErrorString(allowed));
  const int steps_per_wave = 2 * ((p.pass_steps + 2 * WAVES - 1) / (2 * WAVES));
  hipLaunchKernelGGL(kernel, dim3(p.grid), dim3(64 * WAVES), p.lds, s, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias,
                     (TOut*)y, M, N, K, (N + 15) / 16, p.npasses, p.pass_steps, steps_per_wave, p.tiles_per_block, f);
  return 0;
}

struct Plan {
  int nt, waves, unroll;
};

// Chosen from measurements on an MI355X at the layer and head shapes of the 8B, 14B and 32B models
// (N from 4096 to 151936, K from 4096 to 25600, M = 1, 2, 4, 8, 12, 16). The time of a variant followed
//     (1 + M / (16 NT)) * penalty(NT) / evenness(blocks)
// closely: the rows of x are read once per block, so their share falls with NT; two tiles per block cost
// about an eighth for the parallelism they give up; and `evenness` is how full the last of the rounds of
// 256 blocks (one per compute unit) is. Waves and loads in flight were then taken from the best variants.
static Plan plan(bool glu, int M, int N, int K) {
  const int tiles = (N + 15) / 16;
  auto cost = [&](int nt) {
    const int blocks = (tiles + nt - 1) / nt;
    const int rounds = (blocks + 255) / 256;
    const double evenness = (double)blocks / (256.0 * rounds);
    return (1.0 + M / (16.0 * nt)) * (nt == 2 ? 1.13 : 1.0) / evenness;
  };
  const int nt = cost(2) < cost(1) ? 2 : 1;
  if (glu) {
    if (nt == 2) return {2, 8, 4};
    return tiles <= 1024 ? Plan{1, 4, 4} : Plan{1, 8, 4};
  }
  if (nt == 2) return M <= 8 ? Plan{2, 8, 2} : Plan{2, 4, 4};
  if (tiles > 256 && tiles < 512) return M <= 2 ? Plan{1, 4, 8} : Plan{1, 4, 4};
  return {1, 8, 8};
}

template <int NT, int WAVES, int UNROLL, bool GLU>
static void launch(hipStream_t s, const void* x, const void* w, const void* bias, void* y, int M, int N, int K,
                   int out_dtype, bool fused, const Fusion& f) {
  const int ksteps = (K + 31) / 32;
  const int steps_per_wave = 2 * ((ksteps + 2 * WAVES - 1) / (2 * WAVES));     // even: whole cache lines of 128 bytes
  const unsigned blocks = (unsigned)((N + 16 * NT - 1) / (16 * NT));
  if (fused)
    hipLaunchKernelGGL((gemm_fewrows_kernel<NT, WAVES, UNROLL, GLU, true, bf16_t>), dim3(blocks), dim3(64 * WAVES), 0, s,
                       (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (bf16_t*)y, M, N, K, steps_per_wave, f);
  else if (out_dtype == NHV_BF16)
    hipLaunchKernelGGL((gemm_fewrows_kernel<NT, WAVES, UNROLL, GLU, false, bf16_t>), dim3(blocks), dim3(64 * WAVES), 0, s,
                       (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (bf16_t*)y, M, N, K, steps_per_wave, f);
  else
    hipLaunchKernelGGL((gemm_fewrows_kernel<NT, WAVES, UNROLL, GLU, false, float>), dim3(blocks), dim3(64 * WAVES), 0, s,
                       (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (float*)y, M, N, K, steps_per_wave, f);
}

}  // namespace fewrows

// Outputs whose squares a product that is added to the residual stream best sends out together: those of a block. With tiles of 16 the
// products of fewer than 4,096 outputs leave units idle, three quarters of the chip with 1,024 of them. (`aligned`: biases, residual
// and norm weights on 16-byte boundaries.) us at 1, 4, 8 and 16 rows by 16 and by
// even blocks: 1,024 of 2,048 4.9, 5.3, 5.5, 5.8 and 4.3, 4.6, 4.7, 5.1; 1,024 of 3,072 5.8, 6.4, 6.6, 7.2 and 4.8, 5.2, 5.6, 6.1; 2,048 of
// 2,048 5.4, 5.9, 6.0, 6.5 and 5.1, 5.3, 5.6, 6.0; 2,048 of 6,144 11.5, 11.1, 12.0 (10.8 by lines) and 8.5, 9.0, 10.0. The reader then
// adds up 256 shares a row where it added 64. (Of fewer than 1,024 columns a block is over before that matters.)
extern "C" int nhv_gemm_fewrows_square_rows(int M, int N, int K, int biased, int aligned) {
  using namespace fewrows;
  if (!aligned || K < 1024 || N >= 4096 || even_rows(N) >= 16 || lines_plan({.residual = true}, M, N, K)) return 16;
  return tiles_plan(false, even_rows(N), biased != 0, M, N, K).ahead ? even_rows(N) : 16;
}

// The caller has checked sizes, alignment and types (1 <= M <= 16, K a multiple of 8). Returns 0, or 1 with the
// error message set.
int nhv_gemm_fewrows_launch(bool glu, const void* x, const void* w, const void* bias, void* y, int M, int N, int K,
                            int out_dtype, hipStream_t s, const NhvGemmFusion& f) {
  using namespace fewrows;
  // a product that takes over work of its neighbours is a kernel of its own kind (more registers): bfloat16 results only
  const bool fused = f.residual != nullptr || f.ss_in != nullptr;
  if (f.band_rows) {
    // (a block's tiles lie in one band)
    if (glu || fused || f.band_rows % 16 != 0) return nhv_fail("few-rows gemm: bands of %d rows (multiples of 16, no gate, no fusion)", f.band_rows);
    // (8,224 outputs of 2,048 columns at 16 rows in five bands, in a trace: 14.9 us by the kernel that takes x
    // from memory, 11.9 by lines)
    if (f.band_rows % 32 == 0 && lines_plan({.banded = true, .floats = out_dtype != NHV_BF16}, M, N, K))
      return out_dtype == NHV_BF16 ? launch_lines<false, bf16_t>(s, x, w, bias, y, M, N, K, f) : launch_lines<false, float>(s, x, w, bias, y, M, N, K, f);
    const Plan p = plan(false, M, N, K);
    if (f.band_rows % 32 == 0 && p.nt == 2) launch<2, 8, 2, false>(s, x, w, bias, y, M, N, K, out_dtype, false, f);
    else launch<1, 8, 8, false>(s, x, w, bias, y, M, N, K, out_dtype, false, f);
    return 0;
  }
  if (fused && out_dtype != NHV_BF16) return nhv_fail("few-rows gemm: a product that takes over its neighbours' work gives bfloat16");
  const Form form = {.glu = glu, .residual = f.residual != nullptr, .scaled = f.ss_in != nullptr, .floats = out_dtype != NHV_BF16};
  if (lines_plan(form, M, N, K) && !(glu && out_dtype != NHV_BF16) && !(f.residual && f.square_rows != 16)) {
    if (glu) return launch_lines<true, bf16_t>(s, x, w, bias, y, M, N, K, f);
    return out_dtype == NHV_BF16 ? launch_lines<false, bf16_t>(s, x, w, bias, y, M, N, K, f) : launch_lines<false, float>(s, x, w, bias, y, M, N, K, f);
  }
  const TilesPlan tp = tiles_plan(glu, f.residual ? f.square_rows : 0, bias != nullptr, M, N, K);
  const bool on_16 = (((uintptr_t)y | (uintptr_t)bias | (uintptr_t)f.residual | (uintptr_t)f.sum_out | (uintptr_t)f.next_w) & 15) == 0;
#define NHV_TILES_CASE(AHEAD_, GLU_, XLDS_)                                                                            \
  if (tp.ahead == AHEAD_ && glu == GLU_ && tp.x_in_lds == XLDS_ && on_16)                                             \
    return fused                   ? launch_tiles<AHEAD_, GLU_, XLDS_, true, bf16_t>(tp, s, x, w, bias, y, M, N, K, f)   \
           : out_dtype == NHV_BF16 ? launch_tiles<AHEAD_, GLU_, XLDS_, false, bf16_t>(tp, s, x, w, bias, y, M, N, K, f) \
                                   : launch_tiles<AHEAD_, GLU_, XLDS_, false, float>(tp, s, x, w, bias, y, M, N, K, f);
  NHV_TILES_CASE(2, true, true) NHV_TILES_CASE(3, true, true) NHV_TILES_CASE(4, true, true) NHV_TILES_CASE(5, true, true)
  NHV_TILES_CASE(2, false, true) NHV_TILES_CASE(3, false, true) NHV_TILES_CASE(4, false, true) NHV_TILES_CASE(5, false, true)
  NHV_TILES_CASE(6, false, true) NHV_TILES_CASE(7, false, true) NHV_TILES_CASE(8, false, true)
  NHV_TILES_CASE(2, false, false) NHV_TILES_CASE(3, false, false) NHV_TILES_CASE(4, false, false) NHV_TILES_CASE(5, false, false)
  NHV_TILES_CASE(6, false, false)
#undef NHV_TILES_CASE
  if (f.residual && f.square_rows != 16) return nhv_fail("few-rows gemm: squares by %d outputs of M=%d N=%d K=%d", f.square_rows, M, N, K);
  const ResidentPlan rp = resident_plan(glu, M, N, K);
#define NHV_RESIDENT_CASE(WV_, UN_, GLU_, PIECES_)                                                                     \
  if (rp.waves == WV_ && rp.unroll == UN_ && glu == GLU_ && (rp.nchunks > 1) == PIECES_)                              \
    return fused                   ? launch_resident<WV_, UN_, GLU_, PIECES_, true, bf16_t>(rp, s, x, w, bias, y, M, N, K, f)  \
           : out_dtype == NHV_BF16 ? launch_resident<WV_, UN_, GLU_, PIECES_, false, bf16_t>(rp, s, x, w, bias, y, M, N, K, f) \
                                   : launch_resident<WV_, UN_, GLU_, PIECES_, false, float>(rp, s, x, w, bias, y, M, N, K, f);
  NHV_RESIDENT_CASE(8, 2, true, false)
  NHV_RESIDENT_CASE(4, 8, true, false)
  NHV_RESIDENT_CASE(16, 2, false, false)
  NHV_RESIDENT_CASE(8, 2, false, false)
  NHV_RESIDENT_CASE(8, 8, false, false)
  NHV_RESIDENT_CASE(4, 8, false, false)
  NHV_RESIDENT_CASE(16, 2, false, true)
  NHV_RESIDENT_CASE(8, 2, false, true)
  NHV_RESIDENT_CASE(8, 8, false, true)
#undef NHV_RESIDENT_CASE
  if (rp.waves == 0) {
    // two pieces of x were faster than the kernel below in all cases but one tie (gate_up at 16 rows of 5,120
    // columns: 97 against 112 us for 17,408 outputs), three and more pieces slower in most
    const PassesPlan pp = passes_plan(glu, M, N, K);
#define NHV_PASSES_CASE(WV_, UN_, GLU_)                                                                  \
  if (pp.npasses == 2 && pp.waves == WV_ && pp.unroll == UN_ && glu == GLU_)                             \
    return fused                   ? launch_passes<WV_, UN_, GLU_, true, bf16_t>(pp, s, x, w, bias, y, M, N, K, f)  \
           : out_dtype == NHV_BF16 ? launch_passes<WV_, UN_, GLU_, false, bf16_t>(pp, s, x, w, bias, y, M, N, K, f) \
                                   : launch_passes<WV_, UN_, GLU_, false, float>(pp, s, x, w, bias, y, M, N, K, f);
    NHV_PASSES_CASE(8, 2, true)
    NHV_PASSES_CASE(4, 8, true)
    NHV_PASSES_CASE(16, 2, false)
    NHV_PASSES_CASE(8, 8, false)
#undef NHV_PASSES_CASE
  }
  const Plan p = plan(glu, M, N, K);
#define NHV_FEWROWS_CASE(NT_, WV_, UN_, GLU_)                                              \
  if (p.nt == NT_ && p.waves == WV_ && p.unroll == UN_ && glu == GLU_) {                   \
    launch<NT_, WV_, UN_, GLU_>(s, x, w, bias, y, M, N, K, out_dtype, fused, f);           \
    return 0;                                                                              \
  }
  NHV_FEWROWS_CASE(1, 8, 8, false)
  NHV_FEWROWS_CASE(1, 4, 8, false)
  NHV_FEWROWS_CASE(1, 4, 4, false)
  NHV_FEWROWS_CASE(2, 8, 2, false)
  NHV_FEWROWS_CASE(2, 4, 4, false)
  NHV_FEWROWS_CASE(1, 4, 4, true)
  NHV_FEWROWS_CASE(1, 8, 4, true)
  NHV_FEWROWS_CASE(2, 8, 4, true)
#undef NHV_FEWROWS_CASE
  return nhv_fail("few-rows gemm: no kernel for the plan (%d, %d, %d)", p.nt, p.waves, p.unroll);
}
