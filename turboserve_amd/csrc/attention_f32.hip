// Paged attention of the true 32-bit path on the matrix cores' 32-bit instructions
// (v_mfma_f32_16x16x4_f32: a chain of fused multiply-adds, nothing narrower than 32 bits): what
// attention_generic.hip computes (the same keys, scores, sinks, caps and biases), for head sizes of 16, 32, 48, 64, 80,
// 96, 128 and 256, values as wide in pages of their own, and pages of 16 keys or more.
//
// A wavefront owns 16 rows of queries: 16 consecutive tokens of one head (prompts), or up to 16 query
// heads of one KV head for one token.  It walks the keys in tiles of 64, from multiples of 64, a block of 16 keys
// at a time: S^T = K Q^T (a lane holds the scores of query row lane % 16 for keys 4 (lane / 16) + i), the tile's own
// maximum, weights and sum, then O^T = V^T P^T with the scores' registers as they are.  Both products take
// their 16 elements (of the head, of the block's keys) in the order 0 4 8 12 1 5 ...: what a lane's 16-byte loads
// hold is an operand without any exchange between lanes.  A tile's (maximum, sum, accumulator) is folded into the row's by
// `fold`, tile after tile; a tile a row sees nothing of changes nothing, bit for bit.  So a row's result is a
// function of (its position, the lowest key it sees, its request's keys) alone: of neither the batch, nor the cutting,
// nor of who folds: a prompt's wavefront folds its tiles itself, for single tokens each tile is a wavefront's
// of its own and attention_f32_combine_kernel folds them in the same order.
//
// Bound by the matrix cores over a prompt (64 keys are 256 instructions of 32 cycles for 128-wide heads), by its
// start and the trip to memory for single tokens.  28 heads of 128 on 4 KV heads, us a layer, the generic kernel
// (a wavefront per token and head, vector multiply-adds) -> this one: 8 requests of one token at 1,024 keys 489 -> 12.8 and 4.7 to
// combine (33.6 MB of keys and values); a prompt of 500 tokens 1,947 -> 71 (1.8 GFLOP: the last block of rows walks 8 tiles one
// after the other, about 8 us each).
#include "common.hpp"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int F32_TILE = 64, F32_BLOCK = 16, F32_BLOCKS = F32_TILE / F32_BLOCK;

struct F32Rule {
  float scale, softcap;
  int window, chunk, keep_first, bias_len;
  float sinks;
  const float* slopes;
  const float* sink_scores;
  const float* distance_bias;
};

__device__ __forceinline__ int lowest_key(int p, const F32Rule& rule) {
  int lo = (rule.window > 0 && p - rule.window + 1 > 0) ? p - rule.window + 1 : 0;
  if (rule.chunk > 0 && (p / rule.chunk) * rule.chunk > lo) lo = (p / rule.chunk) * rule.chunk;
  return lo;
}

// The tiles a stretch of rows walks: 0 .. kept_tiles - 1 (the kept first keys), then from .. last.
struct F32Walk {
  int kept_tiles, from, last;
  __device__ __forceinline__ int count() const { return kept_tiles + last - from + 1; }
  __device__ __forceinline__ int tile(int ordinal) const { return ordinal < kept_tiles ? ordinal : from + ordinal - kept_tiles; }
};

// lo_first, p_last: the lowest key the first row sees, the last row's position; a row behind the first keeps no fewer keys.
__device__ __forceinline__ F32Walk walk_of(int lo_first, int lo_last, int p_last, int keep_first) {
  F32Walk w;
  w.from = lo_first / F32_TILE;
  w.last = p_last / F32_TILE;
  const int kept = min(keep_first, lo_last);
  w.kept_tiles = min((kept + F32_TILE - 1) / F32_TILE, w.from);
  return w;
}

// What a tile (or a row's tiles so far) and the next tile become together: scales of the two accumulators.
__device__ __forceinline__ void fold(float& m, float& l, float mt, float lt, float& a, float& b) {
  const float both = fmaxf(m, mt);
  const float base = both == -INFINITY ? 0.f : both;
  a = expf(m - base);
  b = expf(mt - base);
  l = fmaf(lt, b, l * a);
  m = both;
}

// Over the four lanes that hold a query row (lane % 16): every lane gets the result.
template <bool MAX>
__device__ __forceinline__ float over_row(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float x = __uint_as_float(s[0]), y = __uint_as_float(s[1]);
  v = MAX ? fmaxf(x, y) : x + y;
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float z = __uint_as_float(t[0]), u = __uint_as_float(t[1]);
  return MAX ? fmaxf(z, u) : z + u;
}

__device__ __forceinline__ bool finite4(f32x4 v) {
  return fabsf(v[0]) < INFINITY && fabsf(v[1]) < INFINITY && fabsf(v[2]) < INFINITY && fabsf(v[3]) < INFINITY;
}

// NC: 16-wide pieces of a head and of a value.  RING: blocks of keys or
// values in registers, one being used, the others on their way (a divisor of 8).  TILES: a workgroup is one
// wavefront, its rows are query heads of the token, and it leaves what the tiles blockIdx.x, + gridDim.x .. come to in `partial`
// [token, head, max_tiles, head size] and `ml` [.., 2]; else rows are tokens (rows_are_heads 0) or heads and are folded here.
template <int NC, int RING, bool TILES>
__global__ void __launch_bounds__(256, NC <= 8 && !TILES ? 2 : 1)
attention_f32_kernel(float* __restrict__ out, long out_stride, float out_scale, float* __restrict__ partial,
                     float* __restrict__ ml, int max_tiles, const float* __restrict__ q, long q_stride,
                     const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                     const int* __restrict__ block_table, int table_width, const int* __restrict__ token_seq,
                     const int* __restrict__ positions, int first_token, int tokens, int heads, int kv_heads,
                     int page_size, int rows_are_heads, F32Rule rule) {
  constexpr int dim = 16 * NC;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int group = heads / kv_heads;
  // Which 16 rows: (token0 + r, head0) or (token0, head0 + r), `rows` of them.
  int token0, head0, rows, kvh;
  if (TILES || rows_are_heads) {
    const int per = (group + 15) / 16;  // 16-row tiles of a KV head's query heads
    token0 = blockIdx.z;
    kvh = blockIdx.y / per;
    head0 = kvh * group + (blockIdx.y % per) * 16;
    rows = min(16, (kvh + 1) * group - head0);
    if (token0 >= tokens) return;
  } else {
    const int per = (group + waves - 1) / waves;
    token0 = (gridDim.x - 1 - blockIdx.x) * 16;  // the blocks with most keys first
    kvh = blockIdx.y / per;
    const int h = (blockIdx.y % per) * waves + wave;
    if (h >= group) return;  // no barrier below
    head0 = kvh * group + h;
    rows = min(16, tokens - token0);
  }
  const bool by_head = TILES || rows_are_heads;
  const bool row_valid = r < rows;
  const int row_token = first_token + token0 + (by_head ? 0 : min(r, rows - 1));
  const int row_head = head0 + (by_head ? min(r, rows - 1) : 0);
  const int row_seq = token_seq[row_token], row_p = positions[row_token];
  const float slope = rule.slopes ? rule.slopes[row_head] : 0.f;
  const float* bias_row = rule.distance_bias ? rule.distance_bias + (size_t)row_head * rule.bias_len : nullptr;

  f32x4 qf[NC];
  const float* qrow = q + (size_t)row_token * q_stride + (size_t)row_head * dim + 4 * g;
#pragma unroll
  for (int c = 0; c < NC; ++c) qf[c] = *reinterpret_cast<const f32x4*>(qrow + 16 * c) * rule.scale;

  f32x4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A sink is a key that is always there: the row starts from its score.
  float m_run = rule.sinks > 0.f ? (rule.sink_scores ? rule.sink_scores[row_head] : 0.f) : -INFINITY;
  float l_run = rule.sinks > 0.f ? rule.sinks : 0.f;

  // Stretches of rows of one request (heads: one stretch).  Rows that are tokens: the workgroups of blockIdx.z take them in turn.
  bool row_walked = by_head;
  int turn = by_head ? 0 : blockIdx.z;
  for (int first = 0; first < rows;) {
    const int seq = __builtin_amdgcn_readlane(row_seq, first);
    int last_row = rows - 1;
    if (!by_head) {
      const unsigned same = (unsigned)__ballot(row_seq == seq && row_valid) & 0xffffu;
      last_row = 31 - __builtin_clz(same);  // a request's tokens follow one another
    }
    if (!by_head) {
      const bool taken = turn == 0;
      turn = turn == 0 ? gridDim.z - 1 : turn - 1;
      if (!taken) {
        first = last_row + 1;
        continue;
      }
      row_walked = row_walked || (r >= first && r <= last_row);
    }
    const int p_first = __builtin_amdgcn_readlane(row_p, first), p_last = __builtin_amdgcn_readlane(row_p, last_row);
    const int lo_first = lowest_key(p_first, rule), lo_last = lowest_key(p_last, rule);
    const int kept_last = min(rule.keep_first, lo_last);  // of the stretch's rows the last keeps most
    const F32Walk walk = walk_of(lo_first, lo_last, p_last, rule.keep_first);
    const bool in_stretch = r >= first && r <= last_row;
    const int p = in_stretch ? row_p : -1;
    const int lo = lowest_key(row_p, rule);
    const int kept = min(rule.keep_first, lo);
    const bool whole_rows = first == 0 && last_row == 15;
    const int* table = block_table + (size_t)seq * table_width;
    first = last_row + 1;

    const int tiles = TILES ? min(walk.count(), max_tiles) : walk.count();  // never past a token's share of the scratch
    const int step = TILES ? gridDim.x : 1;
    int ordinal = TILES ? blockIdx.x : 0;
    if (ordinal >= tiles) continue;
    // A block's first key; what no row sees of a tile is read from the last block that some row sees instead (and masked).
    auto block_key = [&](int tile, int b) __attribute__((always_inline)) {
      const int key = tile * F32_TILE + b * F32_BLOCK;
      const bool seen = key <= p_last && (key + F32_BLOCK > lo_first || key < kept_last);
      return seen ? key : (p_last / F32_BLOCK) * F32_BLOCK;
    };
    int pages[F32_BLOCKS], next_pages[F32_BLOCKS];
    auto look_up = [&](int (&to)[F32_BLOCKS], int tile) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < F32_BLOCKS; ++b) to[b] = table[block_key(tile, b) / page_size];
    };
    f32x4 ring[RING][NC];
    auto fetch_keys = [&](f32x4 (&to)[NC], int page, int tile, int b) __attribute__((always_inline)) {
      const int off = block_key(tile, b) & (page_size - 1);
      const float* at = k_pages + (((size_t)page * kv_heads + kvh) * page_size + off) * dim + (r * dim + 4 * g);
#pragma unroll
      for (int c = 0; c < NC; ++c) to[c] = *reinterpret_cast<const f32x4*>(at + 16 * c);
    };
    auto fetch_values = [&](f32x4 (&to)[NC], int page, int tile, int b) __attribute__((always_inline)) {
      const int off = block_key(tile, b) & (page_size - 1);
      const float* at = v_pages + ((size_t)page * kv_heads + kvh) * page_size * dim + off + (r * page_size + 4 * g);
#pragma unroll
      for (int c = 0; c < NC; ++c) to[c] = *reinterpret_cast<const f32x4*>(at + (size_t)16 * c * page_size);
    };
    // Stage s of a tile: keys of block s (s < 4), values of block s - 4.  Stage s lies in slot s % RING.
    int tile = walk.tile(ordinal);
    look_up(pages, tile);
#pragma unroll
    for (int s = 0; s < RING - 1; ++s)
      s < F32_BLOCKS ? fetch_keys(ring[s], pages[s & 3], tile, s & 3) : fetch_values(ring[s], pages[s & 3], tile, s & 3);
    for (; ordinal < tiles; ordinal += step) {
      const int next_tile = walk.tile(min(ordinal + step, tiles - 1));  // past the end: the last one again, not used
      look_up(next_pages, next_tile);
      auto ahead = [&](int s) __attribute__((always_inline)) {  // the stage RING - 1 behind s goes on its way
        const int n = s + RING - 1, b = n & 3;
        if (n < 4) fetch_keys(ring[n % RING], pages[b], tile, b);
        else if (n < 8) fetch_values(ring[n % RING], pages[b], tile, b);
        else if (n < 12) fetch_keys(ring[n % RING], next_pages[b], next_tile, b);
        else fetch_values(ring[n % RING], next_pages[b], next_tile, b);
      };
      f32x4 s4[F32_BLOCKS];
      float mt = -INFINITY;
#pragma unroll
      for (int b = 0; b < F32_BLOCKS; ++b) {
        ahead(b);
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
          for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_16x16x4f32(ring[b % RING][c][i], qf[c][i], s, 0, 0, 0);
        }
        const int key0 = tile * F32_TILE + b * F32_BLOCK + 4 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = s[i];
          const int key = key0 + i;
          if (rule.softcap > 0.f) v = rule.softcap * tanhf(v / rule.softcap);
          if (rule.slopes) v = fmaf(slope, (float)(key - row_p), v);
          if (bias_row) v += bias_row[max(0, min(row_p - key, rule.bias_len - 1))];
          const bool seen = key <= p && (key >= lo || key < kept);
          s[i] = seen ? v : -INFINITY;
          mt = fmaxf(mt, s[i]);
        }
        s4[b] = s;
      }
      mt = over_row<true>(mt);
      const float base = mt == -INFINITY ? 0.f : mt;
      float lt = 0.f;
#pragma unroll
      for (int b = 0; b < F32_BLOCKS; ++b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float w = expf(s4[b][i] - base);
          s4[b][i] = w;
          lt += w;
        }
      }
      lt = over_row<false>(lt);

      f32x4 at_tile[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) at_tile[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < F32_BLOCKS; ++b) {
        ahead(F32_BLOCKS + b);
        f32x4 (&v)[NC] = ring[(F32_BLOCKS + b) % RING];
        const int key0 = tile * F32_TILE + b * F32_BLOCK;
        // Rows that do not see all of a block give some of its keys the weight 0; what lies there must not turn that
        // into something else: keys no row sees (not written yet, or another request's) count as zeros ...
        if (key0 + F32_BLOCK - 1 > p_last || key0 < lo_first) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 4 * g + i;
            const bool seen = key <= p_last && (key >= lo_first || key < kept_last);
#pragma unroll
            for (int c = 0; c < NC; ++c) v[c][i] = seen ? v[c][i] : 0.f;
          }
        }
        // ... and a value that is no finite number reaches the rows that see it and no other.
        bool apart = false;
        if (!by_head && (!whole_rows || key0 + F32_BLOCK - 1 > p_first || key0 < lo_last)) {
          bool fine = true;
#pragma unroll
          for (int c = 0; c < NC; ++c) fine = fine && finite4(v[c]);
          apart = __any(!fine);
        }
        if (!apart) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
              at_tile[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c][i], s4[b][i], at_tile[c], 0, 0, 0);
          }
        } else {
          // The same chains a key at a time, each taken by the rows that see it: -0 times 0 adds nothing to any sum.  (Gathered by
          // exchanges between lanes this stretch was so long that the compiler left the loops around it as loops at 256-wide
          // heads, and the ring in scratch memory: prompts of 2 / 16 tokens, 8 heads, 53 / 51 us a layer, now 21 / 21.)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
#pragma unroll 1
            for (int from = 0; from < 4; ++from) {
              const int key = key0 + 4 * from + i;
              const bool seen = key <= p && (key >= lo || key < kept), mine = g == from;
              const float w = mine ? s4[b][i] : 0.f;
#pragma unroll
              for (int c = 0; c < NC; ++c) {
                const f32x4 next = __builtin_amdgcn_mfma_f32_16x16x4f32(mine ? v[c][i] : -0.f, w, at_tile[c], 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) at_tile[c][e] = seen ? next[e] : at_tile[c][e];
              }
            }
          }
        }
      }
      if (TILES) {
        if (row_valid) {
          const size_t slot = ((size_t)token0 * heads + row_head) * max_tiles + ordinal;
#pragma unroll
          for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4*>(partial + slot * dim + 16 * c + 4 * g) = at_tile[c];
          if (g == 0) *reinterpret_cast<float2*>(ml + 2 * slot) = make_float2(mt, lt);
        }
      } else {
        float a, w;
        fold(m_run, l_run, mt, lt, a, w);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[c][e] = fmaf(at_tile[c][e], w, acc[c][e] * a);
        }
      }
      tile = next_tile;
#pragma unroll
      for (int b = 0; b < F32_BLOCKS; ++b) pages[b] = next_pages[b];
    }
  }
  if (TILES || !row_valid || !row_walked) return;
  const float inv = out_scale / l_run;
  float* to = out + (size_t)row_token * out_stride + (size_t)row_head * dim + 4 * g;
#pragma unroll
  for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4*>(to + 16 * c) = acc[c] * inv;
}

// A row's tiles in their order, as a prompt's wavefront folds them: a workgroup per (token, head), a thread per element.
__global__ void __launch_bounds__(256)
attention_f32_combine_kernel(float* __restrict__ out, long out_stride, float out_scale, const float* __restrict__ partial,
                             const float* __restrict__ ml, int max_tiles, const int* __restrict__ positions,
                             int first_token, int heads, int dim, F32Rule rule) {
  const int t = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  const int p = positions[first_token + t];
  const int lo = lowest_key(p, rule);
  const int tiles = min(walk_of(lo, lo, p, rule.keep_first).count(), max_tiles);
  if (d >= dim) return;
  float m = rule.sinks > 0.f ? (rule.sink_scores ? rule.sink_scores[h] : 0.f) : -INFINITY;
  float l = rule.sinks > 0.f ? rule.sinks : 0.f;
  const size_t slot = ((size_t)t * heads + h) * max_tiles;
  float acc = 0.f;
#pragma unroll 4
  for (int i = 0; i < tiles; ++i) {
    const float2 tile = *reinterpret_cast<const float2*>(ml + 2 * (slot + i));
    const float v = partial[(slot + i) * dim + d];
    float a, b;
    fold(m, l, tile.x, tile.y, a, b);
    acc = fmaf(v, b, acc * a);
  }
  out[(size_t)(first_token + t) * out_stride + (size_t)h * dim + d] = acc * (out_scale / l);
}

}  // namespace

// The arguments of ts_paged_attention_generic for `tokens` tokens from first_token on (q, out, token_seq and positions are
// the whole step's).  mode 0: rows are 16 consecutive tokens of a head, whose requests max_tiles (0: one) wavefronts walk
// side by side; 1: the heads of one token, folded in place; 2: the
// heads of one token, the tiles side by side: partial [tokens, heads, max_tiles, dim] and ml [tokens, heads, max_tiles, 2]
// (32-bit), max_tiles no smaller than any token's tiles: ceil((keys it can see, kept first ones apart) / 64) + 1 + ceil(keep_first / 64)
// (a token that has more is cut there: nothing is read or written outside the scratch).
extern "C" int ts_attention_f32(void* out, const void* q, long q_stride, const void* k_pages, const void* v_pages,
                                const int* block_table, int table_width, const int* token_seq, const int* positions,
                                int first_token, int tokens, int heads, int kv_heads, int dim, int block_size,
                                float scale, float softcap, int window, const float* slopes, int chunk, float sinks,
                                const float* sink_scores, const float* distance_bias, int bias_len, int keep_first,
                                long out_stride, float out_scale, int mode, float* partial, float* ml, int max_tiles,
                                hipStream_t stream) {
  if (tokens == 0) return TS_OK;
  if (keep_first < 0 || (keep_first > 0 && chunk > 0) || first_token < 0 || tokens < 0 || mode < 0 || mode > 2) return TS_ERR_ARG;
  if (!out || !q || !k_pages || !v_pages || !block_table || !token_seq || !positions) return TS_ERR_ARG;
  if (chunk < 0 || window < 0 || !(sinks >= 0.f)) return TS_ERR_ARG;
  if ((sink_scores && !(sinks > 0.f)) || (distance_bias && bias_len < 1)) return TS_ERR_ARG;
  if (mode == 2 && (!partial || !ml || max_tiles < 1)) return TS_ERR_ARG;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || heads > 65535 || table_width < 1) return TS_ERR_SHAPE;
  if (block_size < F32_BLOCK || (block_size & (block_size - 1)) != 0) return TS_ERR_SHAPE;
  if (q_stride % 4 != 0 || out_stride % 4 != 0 || out_stride < (long)heads * dim || (uintptr_t)q % 16 != 0 ||
      (uintptr_t)out % 16 != 0 || (uintptr_t)k_pages % 16 != 0 || (uintptr_t)v_pages % 16 != 0)
    return TS_ERR_SHAPE;
  const F32Rule rule = {scale, softcap, window, chunk, keep_first, bias_len, sinks, slopes, sink_scores, distance_bias};
  const int group = heads / kv_heads, per = (group + 15) / 16;
  dim3 grid, block(64);
  if (mode == 0) {
    const int waves = group < 4 ? group : 4;  // heads of one KV head side by side: they read the same keys
    block = dim3(64 * waves);
    grid = dim3((tokens + 15) / 16, kv_heads * ((group + waves - 1) / waves), max_tiles < 1 ? 1 : max_tiles > 16 ? 16 : max_tiles);
  } else {
    // Single tokens: no more workgroups than some thousands; one whose first tile lies past the end leaves.
    long side = mode == 2 ? max_tiles : 1;
    const long most = 8192 / ((long)tokens * kv_heads * per);
    if (side > most) side = most < 1 ? 1 : most;
    grid = dim3((unsigned)side, kv_heads * per, tokens);
  }
  if (grid.y > 65535 || grid.z > 65535) return TS_ERR_SHAPE;
#define TS_F32_SIZE(NC)                                                                                                    \
  case 16 * NC:                                                                                                            \
    if (mode == 2) TS_F32_LAUNCH(NC, (NC <= 8 ? 4 : 2), true);                                                             \
    else TS_F32_LAUNCH(NC, 2, false);                                                                                      \
    break
#define TS_F32_LAUNCH(NC, RING, TILES)                                                                                     \
  hipLaunchKernelGGL((attention_f32_kernel<NC, RING, TILES>), grid, block, 0, stream, (float*)out, out_stride,              \
                     out_scale, partial, ml, max_tiles, (const float*)q, q_stride, (const float*)k_pages,                   \
                     (const float*)v_pages, block_table, table_width, token_seq, positions, first_token, tokens, heads,     \
                     kv_heads, block_size, mode == 1 ? 1 : 0, rule)
  switch (dim) {
    TS_F32_SIZE(1);
    TS_F32_SIZE(2);
    TS_F32_SIZE(3);
    TS_F32_SIZE(4);
    TS_F32_SIZE(5);
    TS_F32_SIZE(6);
    TS_F32_SIZE(8);
    TS_F32_SIZE(16);
    default:
      return TS_ERR_SHAPE;
  }
#undef TS_F32_SIZE
#undef TS_F32_LAUNCH
  if (mode == 2)
    hipLaunchKernelGGL(attention_f32_combine_kernel, dim3(tokens, heads), dim3(((dim + 63) / 64) * 64), 0, stream, (float*)out,
                       out_stride, out_scale, partial, ml, max_tiles, positions, first_token, heads, dim, rule);
  return ts_launch_status();
}
