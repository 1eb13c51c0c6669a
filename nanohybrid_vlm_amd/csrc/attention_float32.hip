// Attention over the paged cache in float on the float matrix cores (v_mfma_f32_16x16x4_f32: every product and sum in 32 bits),
// for key heads of a multiple of 16 entries and value heads of 64, 128, 192 or 256; masks and options are those of
// attention_generic.hip, which takes the other sizes.
//
// Keys are taken in blocks of 32 aligned to absolute positions, of which wave w of a block's 8 takes numbers w, w + 8, ... in
// turn, with a running maximum, sum and weighted values of its own; the 8 waves' results are merged in their order. Masked
// keys count as nothing and a row's numbers hang on its own keys alone, so a position's result depends neither on the batch nor
// on the portion.
//
// A block owns 16 rows, a row being (token, one of the query heads that read one key/value head), of one request: 8 tokens of
// a prompt where two heads share a key head, or one decoded token. Scores come as S^T = K Q^T, whose layout is that of the
// second product's right operand (O^T = V^T P^T), so the weights never leave their registers; neither do the sums: the waves
// meet in LDS once, at the end (before, after every eight blocks of keys, with a barrier on either side). What bounds it: a
// wave's blocks are 128 matrix instructions of 32 clocks each and two waves share a SIMD; registers allow one block a compute
// unit. 16 heads on 8 key heads of 128, us, before and now: a prompt of 517 tokens 54.6, 41.6; 500 tokens after 1,500 179, 122.
// Not faster there: a block's keys all asked for at once and the next block's before the values are worked on (44.8, 119), four
// waves a block (39.2, 114).
//
// AT_ONCE, where a request's rows are one tile (a decoded token, a portion of up to 16 rows) and heads are 64 or 128 entries for
// keys and values: what a few blocks of keys take is the way to them, four trips to memory for a wave's 32 keys after three
// for the positions and the table. So a block is asked for as a whole, keys and values, the first one while the
// queries are on their way and, where keys begin with the request's, at a place looked up before the positions are known; the
// next one's keys follow this one's scores. The sums and their order are the same, so are the bits. us where keys come from
// memory, the other order first: six tokens after 100 10.5, 8.5; one after 300 16.1, 15.0; eight after 3,000 112, 90; 64 after
// 500 59, 54; two after 200, 32 heads of 64 on 2, 9.0, 8.1. Where they lie in the L2: 8.1, 7.6; 14.4, 14.5; 90, 78.
#include "nhv_common.h"
#include "nhv_head_pieces.h"
#include <math.h>

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define WAVES 8
#define ROWS 16
#define KEYS 32
#define TILES (KEYS / 16)
#define MAX_E 256
#define MAX_D 256

struct FloatAttention {
  const float *q, *k, *v;
  float* out;
  const int *positions, *cu, *block_tables;
  int max_blocks, Hq, Hkv, D, E, page_size;
  float scale;
  int window, chunk;
  float cap;
  int has_sink;
  float sink;
  const float *sinks, *slopes, *gate;
  long long gate_ld;
};

// ROTATED (one token a request): queries and the token's own key and value come as their projection left them; a block norms and
// turns its heads while its first keys are on their way, stores the key and the value, and takes these from LDS. us a step of 14
// layers of the 0.6B shape, two launches and one: 1 request after 100 keys 762, 751, after 2,000 1,475, 1,472, 6 after 50 to 150
// 827, 811, 32 after 300 1,207, 1,190.
struct FloatRotated {
  const float *qkv, *bias, *q_norm, *k_norm;
  float eps;
  const float* cos_sin;                                  // null: nothing is turned
  const int *positions, *slots;
};

template <int CHUNKS, bool AT_ONCE, bool ROTATED>        // of 64 value entries
__global__ __launch_bounds__(64 * WAVES) void attention_float32_kernel(FloatAttention a, FloatRotated from_rows) {
  extern __shared__ __attribute__((aligned(16))) float shared[];
  constexpr int E = 64 * CHUNKS, UNITS = AT_ONCE ? E / 16 : 4;   // (blocks of 16 key entries that have registers)
  const int D = AT_ONCE ? E : a.D, group = a.Hq / a.Hkv;
  float* qs = shared;                                    // [ROWS][D + 4]
  float* part = qs + ROWS * (D + 4);                     // [WAVES][ROWS][E + 4]
  float* stats = part + WAVES * ROWS * (E + 4);          // [WAVES][ROWS][2]: maximum and sum
  float *own_k = stats + WAVES * ROWS * 2, *own_v = own_k + E;           // ROTATED: the token's own key and value
  const int kvh = blockIdx.y, req = blockIdx.z;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int* table = a.block_tables + (size_t)req * a.max_blocks;
  // where this lane's key of the wave's first block lies if the keys that are read begin with the request's
  int page = 0;
  if constexpr (AT_ONCE) page = table[min((wave * KEYS + lane % KEYS) / a.page_size, a.max_blocks - 1)];
  const int first = a.cu[req], rows = (a.cu[req + 1] - first) * group;
  const int row0 = (gridDim.x - 1 - blockIdx.x) * ROWS;  // (the tiles with the longest chains of keys first)
  if (row0 >= rows) return;                              // (the same for the whole block)

  f32x4 mine_q = {0.f, 0.f, 0.f, 0.f};                   // (AT_ONCE: what this thread brings of the queries)
  const int q_row = (int)threadIdx.x * 4 / D, q_at = (int)threadIdx.x * 4 % D;
  auto query = [&](int r, int d) {
    return *reinterpret_cast<const f32x4*>(a.q + ((size_t)(first + (row0 + r) / group) * a.Hq + kvh * group + (row0 + r) % group) * D + d);
  };
  if (AT_ONCE && !ROTATED && q_row < ROWS && row0 + q_row < rows) mine_q = query(q_row, q_at);
  // (ROTATED: threads take eight entries of a head, heads the group's queries, then the key and the value)
  constexpr int LANES = E / 8;
  const int item = threadIdx.x / LANES, lane8 = threadIdx.x % LANES;
  const bool of_v = item == group + 1, mine_item = ROTATED && item < group + 2;
  float piece[8];
  const int item_head = item < group ? kvh * group + item : a.Hq + (of_v ? a.Hkv : 0) + kvh;
  int store_at = -1;
  if constexpr (ROTATED) {
    if (mine_item) load8f<float>(from_rows.qkv + ((size_t)first * (a.Hq + 2 * a.Hkv) + item_head) * D + lane8 * 8, piece);
    store_at = from_rows.slots[first];
  }

  // this lane's row: what it may read
  const int row = row0 + r16;
  const bool live = row < rows;
  const int head = kvh * group + (live ? row % group : 0);
  const int pos = live ? a.positions[first + row / group] : -1;
  const int lo = !live ? 0x7fffffff : a.chunk > 0 ? pos - pos % a.chunk : a.window > 0 ? max(0, pos - a.window + 1) : 0;
  int tile_lo = lo, tile_hi = pos;                       // the same in every lane afterwards
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    tile_lo = min(tile_lo, __shfl_xor(tile_lo, o, NHV_WAVE));
    tile_hi = max(tile_hi, __shfl_xor(tile_hi, o, NHV_WAVE));
  }
  const float slope = a.slopes && live ? a.slopes[head] : 0.f;

  // lane l's own key of a block from kb on, and where it lies. A key that no row reads is taken for the tile's last: its score
  // is masked, and every load is without a condition (with one the compiler waits for all that are under way).
  auto slot_in = [&](int kb) {
    const int mine = kb + lane % KEYS;
    // (ROTATED: the tile's last key may be under way to its place, so a key before the first is taken for the first)
    const int own = ROTATED ? min(max(mine, tile_lo), tile_hi) : mine >= tile_lo && mine <= tile_hi ? mine : tile_hi;
    return table[own / a.page_size] * a.page_size + own % a.page_size;
  };
  // (the first block of this wave's from the tile's first key on)
  const int from = (tile_lo / KEYS + ((wave - tile_lo / KEYS) & (WAVES - 1))) * KEYS;
  int slot = 0;
  f32x4 kf[UNITS][TILES];
  const float* kr[TILES];
  auto keys_at = [&]() {
#pragma unroll
    for (int t = 0; t < TILES; ++t) kr[t] = a.k + ((size_t)__shfl(slot, 16 * t + r16, NHV_WAVE) * a.Hkv + kvh) * D + 4 * g;
  };
  auto ask = [&](int unit, int d) {                      // (the last 16 entries again where there are no more)
#pragma unroll
    for (int t = 0; t < TILES; ++t) kf[unit][t] = *reinterpret_cast<const f32x4*>(kr[t] + (AT_ONCE ? d : min(d, D - 16)));
  };
  if constexpr (AT_ONCE) {
    if (from <= tile_hi) {
      if (tile_lo == 0) {
        // (a key that no row reads is taken for the block's first here, whose page is known too)
        const int mine = from + lane % KEYS, own = mine <= tile_hi ? mine : from;
        const int first_page = __shfl(page, 0, NHV_WAVE);
        slot = (mine <= tile_hi ? page : first_page) * a.page_size + own % a.page_size;
      } else {
        slot = slot_in(from);
      }
      keys_at();
#pragma unroll
      for (int u = 0; u < UNITS; ++u) ask(u, 16 * u);
    }
    if constexpr (ROTATED) {
      if (mine_item) {
        float y[8], cs[8], sn[8];
        const bool turns = from_rows.cos_sin != nullptr && !of_v;
        if (turns) {
          const float* row = from_rows.cos_sin + (size_t)from_rows.positions[first] * D + lane8 % (LANES / 2) * 8;
          load8f<float>(row, cs);
          load8f<float>(row + D / 2, sn);
        }
        if (from_rows.bias) {
          float b[8];
          load8f<float>(from_rows.bias + (size_t)item_head * D + lane8 * 8, b);
#pragma unroll
          for (int e = 0; e < 8; ++e) piece[e] += b[e];
        }
        const float* norm = item < group ? from_rows.q_norm : from_rows.k_norm;
        if (norm && !of_v) normed_head<float, float, LANES>(piece, norm, from_rows.eps, lane8);
        if (turns) {
          turned_head<LANES>(piece, cs, sn, lane8, y);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = piece[e];
        }
        store8f<float>(item < group ? qs + item * (D + 4) + lane8 * 8 : (of_v ? own_v : own_k) + lane8 * 8, y);
        if (item >= group && store_at >= 0)
          store8f<float>(const_cast<float*>(of_v ? a.v : a.k) + ((size_t)store_at * a.Hkv + kvh) * D + lane8 * 8, y);
      } else if (item < ROWS + 2) {                      // (rows of the tile that no head has)
        float y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        store8f<float>(qs + (item - 2) * (D + 4) + lane8 * 8, y);
      }
    } else if (q_row < ROWS) {
      *reinterpret_cast<f32x4*>(&qs[q_row * (D + 4) + q_at]) = mine_q;
    }
  } else {
    for (int i = threadIdx.x * 4; i < ROWS * D; i += 64 * WAVES * 4) {
      const int r = i / D, d = i % D;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (row0 + r < rows) v = query(r, d);
      *reinterpret_cast<f32x4*>(&qs[r * (D + 4) + d]) = v;
    }
  }

  // of row r16: the maximum, this lane's share of the sum (lanes r16, 16 + r16, ... together have all) and values so far
  float M = -INFINITY, L = 0.f;
  f32x4 o[CHUNKS][4];
#pragma unroll
  for (int h = 0; h < CHUNKS; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) o[h][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // what is read at the token's position is what it stores
  bool own = false;
  if constexpr (ROTATED) own = store_at >= 0 && store_at == table[tile_hi / a.page_size] * a.page_size + tile_hi % a.page_size;
  __syncthreads();                                       // (the queries are in LDS)
  for (int kb = from; kb <= tile_hi; kb += KEYS * WAVES) {
    const int next = kb + KEYS * WAVES;
    int next_slot = 0;
    if constexpr (!AT_ONCE) {
      slot = slot_in(kb);
      keys_at();
    }
    f32x4 s[TILES], vf[AT_ONCE ? CHUNKS : 1][TILES][4];
    const float* vr[TILES][4];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) vr[t][i] = a.v + ((size_t)__shfl(slot, 16 * t + 4 * g + i, NHV_WAVE) * a.Hkv + kvh) * E + 4 * r16;
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto values = [&](int h) {
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) vf[AT_ONCE ? h : 0][t][i] = *reinterpret_cast<const f32x4*>(vr[t][i] + 64 * h);
    };
    auto score = [&](int unit, int d) {
      const f32x4 qf = *reinterpret_cast<const f32x4*>(&qs[r16 * (D + 4) + d + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < TILES; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[unit][t][j], qf[j], s[t], 0, 0, 0);
    };
    if constexpr (AT_ONCE) {
      // all of the block is under way before the first product; the next block's keys follow behind this one's scores
      next_slot = slot_in(next);                         // (before the values: it is waited for with the keys)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < CHUNKS; ++h) values(h);
      const bool newest = ROTATED && own && kb + KEYS > tile_hi;          // (keys beyond the last stand for it here, too)
      if (newest)
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
          const f32x4 k = *reinterpret_cast<const f32x4*>(&own_k[16 * u + 4 * g]);
#pragma unroll
          for (int t = 0; t < TILES; ++t)
            if (kb + 16 * t + r16 >= tile_hi) kf[u][t] = k;
          __builtin_amdgcn_sched_barrier(0);             // (one piece at a time: registers)
        }
#pragma unroll
      for (int u = 0; u < UNITS; ++u) score(u, 16 * u);
      if (newest)
#pragma unroll
        for (int h = 0; h < CHUNKS; ++h) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(&own_v[64 * h + 4 * r16]);
#pragma unroll
          for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (kb + 16 * t + 4 * g + i >= tile_hi) vf[h][t][i] = v;
          __builtin_amdgcn_sched_barrier(0);
        }
      if (next <= tile_hi) {
        slot = next_slot;
        keys_at();
#pragma unroll
        for (int u = 0; u < UNITS; ++u) ask(u, 16 * u);
      }
    } else {
      // keys two blocks of 16 entries ahead; the first 64 value entries at once
      ask(0, 0);
      ask(1, 16);
      values(0);
      int d = 0;
      for (; d + 64 <= D; d += 64) {
        ask(2, d + 32);
        ask(3, d + 48);
        score(0, d);
        score(1, d + 16);
        ask(0, d + 64);
        ask(1, d + 80);
        score(2, d + 32);
        score(3, d + 48);
      }
      if (d < D) {                                       // 16, 32 or 48 entries more
        ask(2, d + 32);
        ask(3, d + 48);
        score(0, d);
        if (d + 16 < D) score(1, d + 16);
        if (d + 32 < D) score(2, d + 32);
      }
    }
    // s[t][i]: key kb + 16 t + 4 g + i against row r16
    float m = -INFINITY;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb + 16 * t + 4 * g + i;
        float z = s[t][i] * a.scale;
        if (a.cap > 0.f) z = a.cap * tanhf(z / a.cap);
        if (a.slopes) z = fmaf(-slope, (float)(pos - key), z);
        s[t][i] = key >= lo && key <= pos ? z : -INFINITY;
        m = fmaxf(m, s[t][i]);
      }
    m = fmaxf(m, __shfl_xor(m, 16, NHV_WAVE));
    m = fmaxf(m, __shfl_xor(m, 32, NHV_WAVE));
    m = fmaxf(m, M);
    const float base = m == -INFINITY ? 0.f : m;       // (no visible key so far: every weight is 0)
    const float old = expf(M - base);
    M = m;
    L *= old;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[t][i] = expf(s[t][i] - base);
        L += s[t][i];
      }
    // value entry 64 h + 4 r + j is row r of matrix tile j: one load of 16 bytes a key feeds four tiles. The next chunk is
    // asked for as this one is used up.
#pragma unroll
    for (int h = 0; h < CHUNKS; ++h) {
      f32x4 now[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) now[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      float odd = 0.f;                                 // not a number as soon as some value is infinite or none
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            odd = fmaf(vf[AT_ONCE ? h : 0][t][i][j], 0.f, odd);
            now[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[AT_ONCE ? h : 0][t][i][j], s[t][i], now[j], 0, 0, 0);
          }
          if (!AT_ONCE && h + 1 < CHUNKS) vf[0][t][i] = *reinterpret_cast<const f32x4*>(vr[t][i] + 64 * (h + 1));
        }
      // now[j][i]: row r16, entry 64 h + 16 g + 4 i + j
      if (__any(odd != 0.f)) {
        // a value that is no finite number: it must not reach the rows that do not read it (0 times it is not 0)
#pragma unroll
        for (int j = 0; j < 4; ++j) now[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            for (int gk = 0; gk < 4; ++gk) {
              const float p = __shfl(s[t][i], 16 * gk + r16, NHV_WAVE);
              if constexpr (AT_ONCE) {                   // (the lanes of group gk hold the key's entries)
#pragma unroll
                for (int ii = 0; ii < 4; ++ii)
#pragma unroll
                  for (int j = 0; j < 4; ++j) {
                    const float value = __shfl(vf[h][t][i][j], 16 * gk + 4 * g + ii, NHV_WAVE);
                    if (p != 0.f) now[j][ii] = fmaf(p, value, now[j][ii]);
                  }
              } else {
                const int at = __shfl(slot, 16 * t + 4 * gk + i, NHV_WAVE);
                if (p != 0.f) {
                  const float* row_v = a.v + ((size_t)at * a.Hkv + kvh) * E + 64 * h + 16 * g;
#pragma unroll
                  for (int ii = 0; ii < 4; ++ii)
#pragma unroll
                    for (int j = 0; j < 4; ++j) now[j][ii] = fmaf(p, row_v[4 * ii + j], now[j][ii]);
                }
              }
            }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[h][j][i] = fmaf(o[h][j][i], old, now[j][i]);
    }
  }
  L += __shfl_xor(L, 16, NHV_WAVE);
  L += __shfl_xor(L, 32, NHV_WAVE);
  if (g == 0) {
    stats[(wave * ROWS + r16) * 2] = M;
    stats[(wave * ROWS + r16) * 2 + 1] = L;
  }
  if (from <= tile_hi) {
#pragma unroll
    for (int h = 0; h < CHUNKS; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(&part[(wave * ROWS + r16) * (E + 4) + 64 * h + 16 * g + 4 * i]) = f32x4{o[h][0][i], o[h][1][i], o[h][2][i], o[h][3][i]};
  }
  __syncthreads();

  // what a thread merges: 32 threads a row, entries c + 32 i
  const int my_row = threadIdx.x / (4 * WAVES), c = threadIdx.x % (4 * WAVES);
  if (row0 + my_row >= rows) return;
  float top = -INFINITY, sum = 0.f, total[2 * CHUNKS];
#pragma unroll
  for (int p = 0; p < WAVES; ++p) top = fmaxf(top, stats[(p * ROWS + my_row) * 2]);
#pragma unroll
  for (int i = 0; i < 2 * CHUNKS; ++i) total[i] = 0.f;
#pragma unroll
  for (int p = 0; p < WAVES; ++p) {
    const float m = stats[(p * ROWS + my_row) * 2], l = stats[(p * ROWS + my_row) * 2 + 1];
    // a wave of whose keys this row reads none, or none with a weight. (The maximum alone does not say that: fmaxf passes over a
    // score that is no number, and where all are such the sum of the weights tells.)
    if (m == -INFINITY && l == 0.f) continue;
    const float now = m == -INFINITY ? l : expf(m - top);  // (a sum that is no number makes all of the row none)
    sum += l * now;
#pragma unroll
    for (int i = 0; i < 2 * CHUNKS; ++i) total[i] = fmaf(part[(p * ROWS + my_row) * (E + 4) + c + 32 * i], now, total[i]);
  }

  const int t = first + (row0 + my_row) / group, h = kvh * group + (row0 + my_row) % group;
  float after = 1.f;
  if (a.has_sink || a.sinks) {                           // one more term of the denominator, without a value
    const float z = a.sinks ? a.sinks[h] : a.sink;
    const float most = fmaxf(top, z);
    after = expf(top - most);
    sum = sum * after + expf(z - most);
  }
  float inv = after / sum;
  if (a.gate) inv /= 1.0f + expf(-a.gate[(size_t)t * a.gate_ld + h]);
  float* out = a.out + ((size_t)t * a.Hq + h) * E;
#pragma unroll
  for (int i = 0; i < 2 * CHUNKS; ++i) out[c + 32 * i] = total[i] * inv;
}

template <int CHUNKS, bool AT_ONCE = false, bool ROTATED = false>
static int launch(const FloatAttention& a, dim3 grid, size_t lds, hipStream_t s, const FloatRotated& from_rows = {}) {
  static const hipError_t allowed = hipFuncSetAttribute((const void*)attention_float32_kernel<CHUNKS, AT_ONCE, ROTATED>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                        (int)((ROWS * (MAX_D + 4) + WAVES * ROWS * (64 * CHUNKS + 4) + WAVES * ROWS * 2 + 128 * CHUNKS) * sizeof(float)));
  if (allowed != hipSuccess) return nhv_fail("attention: %zu bytes of LDS are refused: %s", lds, hipGetErrorString(allowed));
  hipLaunchKernelGGL((attention_float32_kernel<CHUNKS, AT_ONCE, ROTATED>), grid, dim3(64 * WAVES), lds, s, a, from_rows);
  NHV_LAUNCH_CHECK("attention_float32");
  return 0;
}

extern "C" int nhv_attention_float32(const void* q, const void* k_cache, const void* v_cache, void* out, const void* positions,
                                     const void* cu_seqlens_q, const void* block_tables, int max_blocks, int B, int max_q_len, int Hq,
                                     int Hkv, int D, int E, int page_size, float scale, int window, int chunk, float cap,
                                     int has_sink, float sink, const void* sinks, const void* slopes, const void* gate, long long gate_ld,
                                     void* stream) {
  NHV_REQUIRE(cap >= 0.f && (!gate || gate_ld >= Hq), "attention: cap %g, gate rows %lld apart for %d heads", (double)cap, gate_ld, Hq);
  NHV_REQUIRE(B > 0 && max_q_len > 0 && Hq > 0 && Hkv > 0 && page_size > 0 && max_blocks > 0,
              "attention: bad sizes B=%d portion=%d Hq=%d Hkv=%d page=%d blocks=%d", B, max_q_len, Hq, Hkv, page_size, max_blocks);
  NHV_REQUIRE(Hq % Hkv == 0, "attention: %d query heads are not a multiple of %d key heads", Hq, Hkv);
  NHV_REQUIRE(D > 0 && D % 16 == 0 && D <= MAX_D && E > 0 && E % 64 == 0 && E <= MAX_E, "attention: head sizes %d and %d are not for this kernel", D, E);
  NHV_REQUIRE(window >= 0 && chunk >= 0 && !(window > 0 && chunk > 0), "attention: window %d and chunk %d", window, chunk);
  const long long tiles = ((long long)max_q_len * (Hq / Hkv) + ROWS - 1) / ROWS;
  NHV_REQUIRE(B <= 65535 && Hkv <= 65535 && tiles < (1ll << 31), "attention: %d requests, %d key heads, portions of %d", B, Hkv, max_q_len);
  const FloatAttention a = {(const float*)q, (const float*)k_cache, (const float*)v_cache, (float*)out, (const int*)positions,
                            (const int*)cu_seqlens_q, (const int*)block_tables, max_blocks, Hq, Hkv, D, E, page_size, scale, window, chunk,
                            cap, has_sink, sink, (const float*)sinks, (const float*)slopes, (const float*)gate, gate_ld};
  const size_t lds = (ROWS * (D + 4) + WAVES * ROWS * (E + 4) + WAVES * ROWS * 2) * sizeof(float);
  // (sizes whose registers and addresses are known when this is compiled: with any D up to 128 two tokens of 64 after 200 took 9.9)
  if (tiles == 1 && D == E && E == 64) return launch<1, true>(a, dim3(1, Hkv, B), lds, (hipStream_t)stream);
  if (tiles == 1 && D == E && E == 128) return launch<2, true>(a, dim3(1, Hkv, B), lds, (hipStream_t)stream);
  switch (E / 64) {
    case 1: return launch<1>(a, dim3((unsigned)tiles, Hkv, B), lds, (hipStream_t)stream);
    case 2: return launch<2>(a, dim3((unsigned)tiles, Hkv, B), lds, (hipStream_t)stream);
    case 3: return launch<3>(a, dim3((unsigned)tiles, Hkv, B), lds, (hipStream_t)stream);
    default: return launch<4>(a, dim3((unsigned)tiles, Hkv, B), lds, (hipStream_t)stream);
  }
}

// One token a request (max_q_len 1), heads of 64 or 128 entries, up to 16 query heads a key head: the same with queries, keys and
// values as their projection left them, ``qkv`` [T, (Hq + 2 Hkv) D]: the kernel adds the bias (null: none), divides every head of
// queries and keys by its root mean square and multiplies by its weight (null: not), turns it by its position's angles (cos_sin
// [positions, D]; null: not) and stores keys and values at slot_mapping[t] (negative: nowhere). Every token is of another request
// and reads no slot that another one of the call stores to.
extern "C" int nhv_attention_float32_rotated(const void* qkv, const void* bias, const void* q_norm_w, const void* k_norm_w, float eps,
                                             const void* cos_sin, const void* rotation_positions, const void* slot_mapping, void* k_cache,
                                             void* v_cache, void* out, const void* positions, const void* cu_seqlens_q,
                                             const void* block_tables, int max_blocks, int B, int Hq, int Hkv, int D, int page_size,
                                             float scale, int window, void* stream) {
  NHV_REQUIRE(B > 0 && B <= 65535 && Hq > 0 && Hkv > 0 && Hkv <= 65535 && page_size > 0 && max_blocks > 0,
              "attention: bad sizes B=%d Hq=%d Hkv=%d page=%d blocks=%d", B, Hq, Hkv, page_size, max_blocks);
  NHV_REQUIRE(Hq % Hkv == 0 && Hq / Hkv <= ROWS && (D == 64 || D == 128) && window >= 0,
              "attention: %d query heads of %d on %d key heads are not turned here", Hq, D, Hkv);
  NHV_REQUIRE((q_norm_w == nullptr) == (k_norm_w == nullptr), "attention: q and k norm weights come together");
  NHV_REQUIRE(slot_mapping && k_cache && v_cache && (!cos_sin || rotation_positions), "attention: keys and values without a place");
  const uintptr_t starts = (uintptr_t)qkv | (uintptr_t)bias | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w | (uintptr_t)cos_sin |
                           (uintptr_t)k_cache | (uintptr_t)v_cache;
  NHV_REQUIRE(starts % 16 == 0, "attention: rows off 16-byte boundaries");
  FloatAttention a = {};
  a.k = (const float*)k_cache, a.v = (const float*)v_cache, a.out = (float*)out;
  a.positions = (const int*)positions, a.cu = (const int*)cu_seqlens_q, a.block_tables = (const int*)block_tables;
  a.max_blocks = max_blocks, a.Hq = Hq, a.Hkv = Hkv, a.D = D, a.E = D, a.page_size = page_size, a.scale = scale, a.window = window;
  const FloatRotated from_rows = {(const float*)qkv, (const float*)bias, (const float*)q_norm_w, (const float*)k_norm_w, eps,
                                  (const float*)cos_sin, (const int*)rotation_positions, (const int*)slot_mapping};
  const size_t lds = (ROWS * (D + 4) + WAVES * ROWS * (D + 4) + WAVES * ROWS * 2 + 2 * D) * sizeof(float);
  const dim3 grid(1, Hkv, B);
  return D == 64 ? launch<1, true, true>(a, grid, lds, (hipStream_t)stream, from_rows) : launch<2, true, true>(a, grid, lds, (hipStream_t)stream, from_rows);
}
