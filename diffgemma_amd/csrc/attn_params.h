// Kernel-side argument block and mask arithmetic shared by every attention kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace dg {

enum : uint32_t { DT_BF16 = 0, DT_F16 = 1, DT_F32 = 2 };

constexpr uint32_t kMaxSplits = 64;   // key-range splits per launch: the merge gives each a lane
constexpr int kBlockM = 128;   // stacked query rows per workgroup (4 waves x 32)
constexpr int kBlockN = 32;    // keys per tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Row tiles with split counts of their own (causal rows: a row tile sees as many key tiles as lie before it, and with one
// count for all the launch is as long as the last row tile's share).  The counts do not fall with the row tile, so they
// are given by where each begins: row tile mt has more than i splits from mt = first[i] on.  The units of a KV head are
// ordered by split, then row tile: split i of row tile mt is unit cum[i] + mt - first[i], which also numbers its partial rows.
// The workgroups may go by row tile, then split, instead (units_by_row_tile): the row tiles of i + 1 splits begin with
// workgroup at[i].
constexpr uint32_t kMapSplits = 8;
struct SplitMap {
  uint32_t n;                     // most splits of a row tile; 0: every row tile has n_splits
  uint32_t units;                 // of a KV head
  uint32_t first[kMapSplits], cum[kMapSplits], at[kMapSplits];   // past n: no row tile, no unit
};
__host__ __device__ __forceinline__ uint32_t map_splits(const SplitMap& m, uint32_t mt) {
  uint32_t s = 0;
#pragma unroll
  for (uint32_t i = 0; i < kMapSplits; ++i) s += mt >= m.first[i] ? 1u : 0u;
  return s;
}
// split of unit u of a KV head; its row tile is first[split] + u - cum[split]
__host__ __device__ __forceinline__ uint32_t map_split_of(const SplitMap& m, uint32_t u) {
  uint32_t s = 0;
#pragma unroll
  for (uint32_t i = 1; i < kMapSplits; ++i) s = u >= m.cum[i] ? i : s;
  return s;
}
// The map for row tiles that see tiles(mt) key tiles (not falling with mt), none of whose shares is longer than `len`;
// false where one needs more than kMapSplits.
template <typename Tiles>
inline bool make_split_map(uint32_t n_mtiles, uint32_t len, Tiles&& tiles, SplitMap* m) {
  m->n = m->units = 0;
  for (uint32_t i = 0; i < kMapSplits; ++i) m->first[i] = m->cum[i] = m->at[i] = 0xffffffffu;
  for (uint32_t mt = 0; mt < n_mtiles; ++mt) {
    const uint32_t s = (tiles(mt) + len - 1) / len;
    if (s > kMapSplits) return false;
    while (m->n < s) m->first[m->n++] = mt;
  }
  for (uint32_t i = 0; i < m->n; ++i) {
    m->cum[i] = m->units;
    m->units += n_mtiles - m->first[i];
    m->at[i] = i == 0 ? 0u : m->at[i - 1] + i * (m->first[i] - m->first[i - 1]);
  }
  return true;
}

// Stacked row r of a KV head = tok * group + g: the `group` query heads that share one KV
// head sit next to each other, so a 128-row tile covers 128/group consecutive canvas rows.
struct AttnParams {
  const void* q;       // [canvas][hq][D], element type = KV element type unless q_is_bf16
  const void* k;       // layer region + K offset (element type E)
  const void* v;       // layer region + V offset
  void* out;           // [canvas][hq][D]
  float* lse;          // [canvas][hq] or null
  float* part_o;       // [split][hkv][rows_pad][D]: unnormalised fp32 accumulators, or (part_half) the same
                       // index space in f16 holding accumulators divided by the split's row sum
  float* part_ml;      // [split][hkv][rows_pad][2] (m in log2 units, l)
  uint32_t* dbg;       // 4 words, first-writer-wins, or null
  const uint32_t* step_dev;   // device copy of the reference's StepParams, or null: when set, kv_len is read from its
                              // first word when the kernel runs (resolve_step) and the kv_len below is the largest
                              // prefix the launch was planned for
  int64_t k_tok_stride, k_head_stride, v_tok_stride, v_head_stride;  // elements
  uint32_t canvas, hq, hkv, group;
  uint32_t kv_len, t_all;   // (t_all: of a key range, the keys up to its end; keys_of_range)
  uint32_t causal_rows;
  uint32_t win_m1;       // window-1, or 0xffffffff when unwindowed
  uint32_t lo_nc;        // first visible key of a non-causal row
  uint32_t extra_lo;     // causal rows also see keys >= extra_lo (t_all = none)
  uint32_t ring_mask;
  uint32_t t_clip_lo, t_clip_hi;   // only keys in [t_clip_lo, t_clip_hi) count (a key-range partial); the whole range: 0, t_all
  uint32_t rows_total, rows_pad, n_mtiles;
  uint32_t n_splits, tile_first, tiles_per_split, tile_end;
  uint32_t q_is_bf16;    // Q holds bf16 although E is f16 (reference: bf16 activations, f16 cache)
  uint32_t out_dtype, out_trunc;
  uint32_t part_half;    // split partials are normalised f16 rows instead of unnormalised fp32 ones
  uint32_t touch_ahead;  // the rows will come from HBM: at head_dim 512 key/value tiles are touched into the L2 some tiles
                         // before they are loaded, in the one-launch kernel the key range at its start
  uint32_t lo_explicit;  // lo_nc was given by the caller (not the window rule)
  uint32_t cus;          // compute units of the device
  uint32_t sees_masked;  // causal rows also see the canvas keys behind the causal rows
  float scale_log2;      // softmax_scale * log2(e)
};

// Division of n < 2^31 by a divisor the host knows: q = (mulhi(n, mul) + n) >> shift (the round-up method: mul =
// floor(2^32 (2^shift - d) / d) + 1 with shift = ceil(log2 d)).  Three scalar instructions where a run-time division is
// two dozen on the vector unit.
struct FastDiv {
  uint32_t mul, shift;
};
inline FastDiv make_fast_div(uint32_t d) {
  uint32_t shift = 0;
  while ((1ull << shift) < d) ++shift;
  return FastDiv{(uint32_t)((((1ull << shift) - d) << 32) / d + 1u), shift};
}
__host__ __device__ __forceinline__ uint32_t fast_div(uint32_t n, FastDiv d) {
  return ((uint32_t)(((uint64_t)n * d.mul) >> 32) + n) >> d.shift;
}

// Workgroup u of a KV head in the order by row tile, then split; by[i] divides by i + 1.
struct MapUnit {
  uint32_t mt, split, splits;
};
__host__ __device__ __forceinline__ MapUnit map_unit_by_rows(const SplitMap& m, const FastDiv* by, uint32_t u) {
  uint32_t i = 0;
#pragma unroll
  for (uint32_t j = 1; j < kMapSplits; ++j) i = u >= m.at[j] ? j : i;
  const uint32_t v = u - m.at[i], tiles = fast_div(v, by[i]);
  return MapUnit{m.first[i] + tiles, v - tiles * (i + 1u), i + 1u};
}

// The map of the shortest length in [len, limit] that gives a KV head no more than `budget` units (and no row tile more than
// kMapSplits); false where even `limit` gives more.  Units do not grow with the length, so it is found by bisection, and rows
// behind a long prefix, all of which see about as many key tiles, are told by the first of them (each length in turn, with a map
// built for each, took 140 us of host time for 1024 rows behind 32768 keys).
template <typename Tiles>
inline bool shortest_split_map(uint32_t n_mtiles, uint32_t len, uint32_t limit, uint32_t budget, Tiles&& tiles, SplitMap* m) {
  if (len == 0u || len > limit || (uint64_t)n_mtiles * ((tiles(0u) + limit - 1) / limit) > budget) return false;
  auto fits = [&](uint32_t l) {
    const FastDiv by = make_fast_div(l);
    uint32_t units = 0;
    for (uint32_t mt = 0; mt < n_mtiles && units <= budget; ++mt) {
      const uint32_t s = fast_div(tiles(mt) + l - 1, by);
      units += s > kMapSplits ? budget + 1u : s;
    }
    return units <= budget;
  };
  if (fits(len)) limit = len;
  else if (!fits(limit)) return false;
  while (len < limit) {
    const uint32_t mid = len + (limit - len) / 2u;
    if (fits(mid)) limit = mid;
    else len = mid + 1u;
  }
  return make_split_map(n_mtiles, len, tiles, m);
}

// Key-range splits of a launch of `base` row tiles whose workgroups take a compute unit each: between `least` and `most`, the count
// whose rounds of the chip are shortest, in key tiles, where starting a workgroup costs `start` of them.  (One more workgroup than a
// whole round is a second round: with `cus` / `base` rounded up, 144 rows x 16 heads over 30k keys, 5 row tiles x 2, were 260 workgroups,
// and the filter kernel took twice as long: layer step 226.8 -> 164.4 us, where 128 rows take 140; 224 rows 297.9 -> 216.2, 192 over 5k
// keys 94.6 -> 75.5.)
// Looked at: the last count of each round, and none from where full rounds without a ragged share would cost more than the best so far
// (planning a top-k call, 256 | 1024 rows over 33k keys, with every count looked at 1.33 | 2.10 us, now 1.02 | 1.14).  `looked`: how many.
inline uint32_t splits_in_rounds(uint32_t base, uint32_t tiles, uint32_t least, uint32_t most, uint32_t cus, uint32_t start,
                                 uint32_t* looked = nullptr) {
  uint32_t best = least, n = 0;
  uint64_t best_cost = UINT64_MAX;
  for (uint32_t s = least; s <= most; ++s) {
    if (n != 0 && (uint64_t)base * (tiles + (uint64_t)s * start) >= best_cost * cus) break;
    const uint64_t rounds = ((uint64_t)base * s + cus - 1) / cus;
    s = (uint32_t)std::min<uint64_t>(most, rounds * cus / base);
    const uint64_t cost = rounds * ((tiles + s - 1) / s + start);
    ++n;
    if (cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  if (looked) *looked = n;
  const uint32_t share = std::max(1u, (tiles + best - 1) / best);
  return std::min(best, std::max(least, (tiles + share - 1) / share));      // (the fewest splits with these shares)
}

// In which order the split kernel's workgroups take their units.  Each of the 8 XCDs gets a run of them and reads what its run
// needs through an L2 of its own: by split, then row tile, a share of the keys and all query rows of a KV head; by row tile, then
// split, its own query rows alone, which no workgroup can begin without, and all keys.  And a row tile's partial rows are then
// written on one XCD, where the merge may take them up again (merge_on_xcd, whose gain is another and is not in these figures unless said).
// 16 heads over 2, us, splits first | rows first, rows merged in turn, keys in a cache.  Layer step: 64 rows over 841 keys 21.0 | 20.7, 1564
// 24.8 | 23.3, 3064 28.8 | 26.5, 6064 34.3 | 36.5; 128 rows over 905 26.1 | 26.0, 1628 29.6 | 27.4, 3128 32.4 | 31.9; 256 rows over 556 30.3 | 29.4, 1033
// 29.8 | 29.6, 1756 33.5 | 32.8, 3256 42.4 | 41.2, 6256 61.1 | 60.3, 24256 172.9 | 173.4; 512 rows over 612 33.4 | 33.3 (f16 33.8 | 36.6, and 32.3 merged in
// runs), 1289 43.0 | 39.8, 3512 69.9 | 67.5; 1024 causal rows behind 0 46.6 | 46.1, 300 57.2 | 55.4, 1000 78.4 | 75.7; 700 behind 700 48.9 | 47.1.
// Attention call: 64 rows over 2564 24.6 | 22.3, 4064 26.8 | 26.0; 128 over 2628 27.7 | 27.0, 5128 35.5 | 35.1; 1024 behind 8000 240.9 | 238.3,
// 32768 849 | 847.  Call with keys from HBM (rows merged in runs where merge_on_xcd says so, the first alone): 64 rows over 1564 22.1 | 19.3, 2564 25.9 |
// 26.0; 128 over 2628 29.0 | 28.5, 5128 37.7 | 37.4; 256 over 3256 40.5 | 40.3, 6256 59.2 | 60.3; 512 over 4512 78.7 | 77.2, 8512 129.2 | 130.5; 1024
// behind 3000 123.5 | 121.8, 8000 243.3 | 244.3, 32768 860 | 868.  The line lies where calls from HBM stop to gain; it turns away cached
// ones that do (64 rows over 3064, 6064 being a loss).  Row tiles that do not come in eights end in the middle of an XCD's run (call, merged in runs where that is
// taken): 72 rows over 972 keys 19.2 | 18.1, over 1672 22.7 | 23.1; 96 over 1696 24.4 | 21.7, 2496 26.1 | 25.4; 200 over 2600 33.2 | 32.3.
inline bool rows_before_splits(uint32_t hkv, uint32_t n_mtiles, uint32_t key_tiles) {
  return key_tiles <= std::min((hkv * n_mtiles % 8u == 0u ? 20u : 10u) * n_mtiles, 72u + 2u * n_mtiles);
}
// Whether a call takes that order.  With fewer than eight row tiles the splits of one are on several XCDs in either order; taken there
// where every XCD has a run of the same length out of one row tile (4 row tiles: 32 rows over 432 keys in 14 splits 14.9 -> 14.2; 8
// heads over 1, 64 rows over 364 keys 14.4 -> 13.8), and not where the ends of runs cut them (6 row tiles, 40 rows over 440 keys in 7 splits
// 14.8 -> 15.0; 4, 32 rows over 92 keys in 3 splits 15.1 -> 15.3, over 532 in 9 14.65 -> 14.64; turned away with them: 2, 16 rows over 316
// keys in 5 splits, 18.9 either way, f16 19.3 -> 18.9).
// With rows from HBM the gain ends sooner: 256 peaked rows over 3256 keys, 102 tiles, of an f16 cache 54.1 -> 54.7 (bf16 40.5 -> 40.3), and
// the line there leaves that form out and 128 rows over 2628 (83 tiles, 29.0 -> 28.5) and 1024 causal ones behind 3000 (126, 123.5 -> 121.8) in.
// With KV heads in eights an XCD has whole heads in either order: nothing to gain (8 over 8, 256 rows over 556 keys 20.2 | 20.2, 1256 24.1 |
// 24.1; 32 over 8, 64 rows over 364 17.8 | 17.8).  head_dim 256: 256 rows over 3256 keys 32.9 | 29.3; below it there are no times.
inline bool units_by_row_tile(const AttnParams& p, const SplitMap& map, uint32_t head_dim) {
  if (head_dim < 256u || p.hkv % 8u == 0u) return false;
  const uint32_t tiles = p.hkv * p.n_mtiles;
  if (tiles < 8u && (map.n || 8u % tiles != 0u || tiles * p.n_splits % 8u != 0u)) return false;
  const uint32_t key_tiles = p.tile_end - p.tile_first;
  if (p.touch_ahead && key_tiles > 72u + 3u * p.n_mtiles / 2u) return false;
  return rows_before_splits(p.hkv, p.n_mtiles, key_tiles);
}

// One pass of top-k sparse attention over canvas rows [tok0, tok0 + ntok).
constexpr int kTopkMaxK = 1024;   // most keys a row may keep
struct TopkParams {
  AttnParams a;          // tensors, strides and mask constants of the whole call
  float* s_plane;        // scores [hq][ntok][t_pad], fp32
  uint32_t tok0, ntok;
  uint32_t t_pad;        // floats per score row, a multiple of the key tile
  uint32_t n_mtiles;     // 128-row tiles of stacked rows in this pass
  uint32_t n_splits;     // key-range splits of the score kernel (no merge needed)
  uint32_t tile_first, tile_end;
  uint32_t k_cfg[4];     // (fixed k | chunk grid, divisor, k_min, k_max)
  float scale;
  // Filtered path (launch_topk_filter): n_mtiles counts 256-row tiles there.
  uint32_t sample_stride;   // every sample_stride-th key is a sampled one
  uint32_t sample_n;
  uint32_t sample_splits;   // key-range splits of the sampled launch, at most its key tiles and kTopkSampleSplits
  float* sample_max;     // [row of the pass][sample_splits * 32]: the largest score of each group of sampled keys
  float* tau;            // [hkv][n_mtiles * 256]: a row's threshold
  uint32_t* cand_n;      // [hkv][n_mtiles][n_splits][4 waves][kTopkSegs]: entries in a segment
  void* cand;            // the same index space, kTopkSegAlloc entries of 8 bytes each
  void* kept;            // [row of the pass][kept_pad]: (weight, byte offset of the key's V row), in order of position
  uint32_t kept_pad;
  uint32_t* fail_rows;   // [canvas][hq]: rows the filtered path has left over (null: every row takes the general path)
  uint32_t* fail_block;  // rows left over per block of canvas rows (general path: of this block)
  uint32_t fail_block_tok;   // canvas rows per block
  FastDiv div_mtiles, div_splits, div_group, div_rows;   // by n_mtiles, n_splits, the GQA group, ntok * group (set at the launch)
};
// A segment holds the candidates that one lane finds for one query row: half of the row's in a key-range split.  The spare
// places behind the limit take what one more key tile may bring before the count is looked at.
constexpr uint32_t kTopkSegs = 128;         // per wave of the filter kernel and split: two blocks of 32 rows, two lanes per row
constexpr uint32_t kTopkSegCap = 80, kTopkSegAlloc = kTopkSegCap + 16;
constexpr uint32_t kTopkFilterRows = 256;   // stacked rows per workgroup of the filter kernel
constexpr uint32_t kTopkSampleRows = 128;   // and of its instance for sampled keys
constexpr uint32_t kTopkListMax = 512;      // most keys kept on the filtered path
constexpr uint32_t kTopkListAlign = 8;      // a row's list of kept keys takes a multiple of this
constexpr uint32_t kTopkSampleMax = 8192;   // most sampled keys per row
constexpr uint32_t kTopkSampleSplits = 128; // most splits of the sampled keys: 4096 groups, what the threshold kernel holds
// head_dim slices the gather deals out, by the stacked rows of a pass (topk_gather_kernel has the times)
inline uint32_t topk_gather_slices(uint32_t rows) { return rows > 2048u ? 1u : rows > 1024u ? 2u : 4u; }

// Merging attention states of key-range partials (dg_attn_merge).  A state holds, per row
// (row = canvas row * n_q_heads + query head), m and l in two planes of `rows` floats and then, from
// the next 16-byte boundary, head_dim accumulators `acc` per row, with
//   output row = acc / l,   log-sum-exp of the row's scores = m + ln l   (natural log; l = 0: no key seen).
constexpr uint32_t kMaxStates = 16;
__host__ __device__ inline size_t state_acc_offset(size_t rows) { return (2 * rows + 3) & ~(size_t)3; }   // floats
struct StateMergeParams {
  const float* states[kMaxStates];
  uint32_t n, rows, hd, hq;
  void* out;            // [rows][head_dim] of out_dtype, or null
  float* lse;           // [rows] or null
  float* state_out;     // a state, or null; may be one of `states` (a row is read before it is written)
  uint32_t out_dtype, out_trunc;
  uint32_t* dbg;
};

// The reference binds StepParams as a device buffer (src/metal/step_kernel/enc.rs:2177-2220, buffer 4), so the
// prefix length a recorded command sequence works on is read when it runs.  With step_dev set, the same here:
// kv_len comes from device memory (clamped to the prefix the launch was planned for: grid, split count and
// workspace follow that maximum) and everything derived from it is worked out again, the way the host does it
// in make_plan.  The key range is the whole one (a key-range partial takes kv_len from the host).
__device__ __forceinline__ AttnParams resolve_step(const AttnParams& in) {
  AttnParams p = in;
  if (in.step_dev == nullptr) return p;
  const uint32_t kv = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(in.step_dev[0], in.kv_len));
  p.kv_len = kv;
  p.t_all = kv + p.canvas;
  const bool windowed = p.win_m1 != 0xffffffffu;
  if (!p.lo_explicit) p.lo_nc = (windowed && kv > p.win_m1) ? kv - p.win_m1 : 0u;
  p.lo_nc = min(p.lo_nc, p.t_all);
  p.extra_lo = p.sees_masked ? min(kv + p.causal_rows, p.t_all) : p.t_all;
  uint32_t lo_all = 0xffffffffu;
  if (p.causal_rows < p.canvas) lo_all = min(lo_all, p.lo_nc);
  if (p.causal_rows > 0u) lo_all = min(lo_all, (windowed && kv > p.win_m1) ? kv - p.win_m1 : 0u);
  lo_all = min(lo_all, p.t_all);
  p.t_clip_lo = 0u;
  p.t_clip_hi = p.t_all;
  p.tile_first = lo_all / (uint32_t)kBlockN;
  p.tile_end = max(p.tile_first, (p.t_all + (uint32_t)kBlockN - 1u) / (uint32_t)kBlockN);
  return p;
}

struct RowBounds {
  uint32_t lo, hi, extra;  // visible iff (lo <= t < hi) or (extra <= t), and t < t_all
};

// Reference rules: causal rows see [max(0,qpos-(window-1)), qpos]; the other rows see
// [lo_nc, t_all) where lo_nc = max(0, kv_len-(window-1)) unless the caller set it.
__device__ __forceinline__ RowBounds row_bounds(const AttnParams& p, uint32_t tok) {
  RowBounds b;
  const bool causal = tok < p.causal_rows;
  const uint32_t qpos = p.kv_len + tok;
  if (causal) {
    b.hi = min(p.t_all, qpos + 1u);
    b.lo = (p.win_m1 != 0xffffffffu && qpos > p.win_m1) ? qpos - p.win_m1 : 0u;
    b.extra = p.extra_lo;
  } else {
    b.hi = p.t_all;
    b.lo = p.lo_nc;
    b.extra = p.t_all;
  }
  b.lo = max(b.lo, p.t_clip_lo);
  b.hi = min(b.hi, p.t_clip_hi);
  b.extra = max(b.extra, p.t_clip_lo);   // (keys at or past t_clip_hi are cut by key_visible's last argument)
  return b;
}

__device__ __forceinline__ bool key_visible(const RowBounds& b, uint32_t t, uint32_t t_all) {
  return t < t_all && ((t >= b.lo && t < b.hi) || t >= b.extra);
}

// Rows of the key tile at position t0 that the kernels may read, as row numbers in the tile: [first, last].  Any other
// row is replaced by the nearest of these.  Past the last key there may be no memory; before `lo`, the first key a row of
// the workgroup sees, a dead ring slot may hold anything, and a holder of a key range (dg_attn_partial) who passes a
// shifted base has no memory there either.
struct TileRows {
  uint32_t first, last;
};
__host__ __device__ __forceinline__ TileRows tile_rows(uint32_t t0, uint32_t lo, uint32_t t_all) {
  const uint32_t left = t_all - 1u - t0;
  TileRows r;
  r.last = left < (uint32_t)kBlockN - 1u ? left : (uint32_t)kBlockN - 1u;
  // (a first visible key at or past t_all, i.e. rows that see nothing, must not move the clamp past the last key)
  r.first = lo <= t0 ? 0u : lo - t0 < r.last ? lo - t0 : r.last;
  return r;
}
// The number of keys a kernel is told of (AttnParams.t_all), for a launch over the key tiles [first, end): of a key range no more
// than its tiles, so that no kernel needs another bound to stay within what a holder of that range has in memory.
__host__ __device__ __forceinline__ uint32_t keys_of_range(uint32_t first, uint32_t end, uint32_t t_all) {
  return end > first && end * (uint32_t)kBlockN < t_all ? end * (uint32_t)kBlockN : t_all;
}
// Where loads and touches issued for tiles behind a row tile's last one (at t_last) go, so that the tile loop need not branch
// around them: the last tile again, its rows clamped at the end alone.  Where that tile begins before `lo` (it is then the only
// one), the rows from `lo` on instead; a ring has memory for every slot, and 32 rows from an arbitrary slot could run past its end.
__host__ __device__ __forceinline__ uint32_t past_end_pos(uint32_t t_last, uint32_t lo, uint32_t t_all, uint32_t ring_mask) {
  const uint32_t see = lo < t_all ? lo : t_all - 1u;
  return ring_mask == 0u && see > t_last ? see : t_last;
}
// The one-launch kernel touches a range of keys [pos0, pos1), `per` of them to a touch: position of key `i` of touch u.
__host__ __device__ __forceinline__ uint32_t touched_pos(uint32_t pos0, uint32_t pos1, uint32_t per, uint32_t u, uint32_t i) {
  const uint32_t pos = pos0 + u * per + i, last = pos1 - 1u;
  return pos < last ? pos : last;
}
// whether some row of the tile may not be read
__host__ __device__ __forceinline__ bool tile_is_edge(uint32_t t0, uint32_t lo, uint32_t t_all) {
  return t0 < lo || t0 + (uint32_t)kBlockN > t_all;
}

__device__ __forceinline__ uint32_t kv_slot(uint32_t ring_mask, uint32_t t) {
  return ring_mask ? (t & ring_mask) : t;
}

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
  return __uint_as_float((uint32_t)b << 16);
}

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f, bool trunc) {
  uint32_t u = __float_as_uint(f);
  if (!trunc) {
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
  }
  return (uint16_t)(u >> 16);
}

// The reference's DebugStatus vocabulary (src/shaders/include/debug_status.metal:8-19 error codes,
// src/shaders/include/dgq_kernels.metal:33-34 kernel ids), decoded on the host by
// src/metal/debug_status.rs:33-75.  include/dg_attn.h carries the same numbers as DG_DBG_*.
enum : uint32_t {
  DBG_ERR_SOFTMAX_NORM_ZERO = 3u,   // a row's softmax denominator was not > 0; value = (tok << 16) | query head
  DBG_ERR_NONFINITE = 4u,           // a result was NaN or infinite; value = element index (attention) / canvas row (producer)
  DBG_ERR_BAD_DIM = 8u,
  DBG_KERNEL_QK_ROPE_KV = 25u,
  DBG_KERNEL_ATTENTION = 26u,
};

// first-writer-wins status record, like the reference's debug_set_error (debug_status.metal:38-52).
// tg is (tok << 16) | query head of the row at fault (the reference's call sites pass 0 there).
__device__ __forceinline__ void dbg_report(uint32_t* dbg, uint32_t code, uint32_t kernel_id, uint32_t tg,
                                           uint32_t value) {
  if (dbg == nullptr) return;
  if (atomicCAS(dbg, 0u, code) == 0u) {
    dbg[1] = kernel_id;
    dbg[2] = tg;
    dbg[3] = value;
  }
}

// Where the merge that asks for all of a row's 16-bit partial rows at once beats the one that looks at the weights first, four
// rows at a time: up to 8 splits while they are less than 32 MiB in all; up to 16 where they are few bytes.  Attention call, us,
// weights first | at once, peaked rows (of which the first fetches a part) and flat ones: 64 rows over 841 keys in 9 splits 19.2 | 18.4,
// 20.5 | 18.4, over 1264 in 14 20.2 | 20.6, 23.5 | 20.7, over 2064 in 13 23.4 | 23.1, 25.7 | 23.1, over 5064 in 16 30.6 | 29.7, 32.7 | 29.8; 16 rows over 3300 in
// 15 25.3 | 22.5, 25.4 | 22.5.  With more rows peaked ones lose what flat ones gain: 96 rows in 10 splits, 15 MiB, 22.0 | 24.0, 25.3 | 24.0 (head_dim 256,
// rows half as long, 96 rows in 14 24.7 | 22.6, 24.8 | 22.6); past 17 MiB 128 rows over 428 keys in 14 splits 20.4 | 27.1 on peaked rows.
constexpr uint32_t kMergeFewSplits = 16;
inline bool merge_at_once(uint32_t n_splits, size_t bytes) {
  return n_splits <= 8 ? bytes < ((size_t)32 << 20) : n_splits <= kMergeFewSplits && bytes <= ((size_t)17 << 20);
}

// Whether the merge that asks for all rows at once takes a row on the XCD that wrote its partial rows (merge_runs): where these,
// `part_bytes` in all, and the keys that an XCD has read, `head_bytes` for each of its KV heads, are no more than 6 MiB.  An XCD's L2 is 4,
// and not all of it is wanted again; the line is a fit to times at head_dim 512 and 256, not worked out.  (Reading there and writing rows of which no other L2
// holds a copy are not told apart: under the profiler, 256 rows over 556 keys, rows in turn | in runs, the attention kernel took
// 20.0 | 17.4 us and the merge 6.0 | 5.8.)  Layer step, 16 heads over 2, us, units by row tile and rows in turn | in runs: 256 rows over 356 keys 26.8 |
// 25.0, 556 (3.2 MiB) 29.4 | 26.0, 1033 (5.1) 29.6 | 28.2, 1756 (7.5) 32.8 | 32.5; 128 rows over 905 (4.1) 26.0 | 23.0; 64 rows over 841 20.7 | 19.3,
// 1564 (4.7) 23.3 | 22.0; 512 over 612 33.3 | 32.7, f16 36.6 | 32.3; call alone, 64 over 2564 (7) 22.3 | 22.5, over 4064 26.0 | 26.3.  Other heads,
// call alone: 8 over 8, 256 rows over 556 20.2 | 18.1, over 1256 24.1 | 21.8; 32 over 8, 64 rows over 1064 24.1 | 21.2; 16 over 1, 64 rows
// over 1064 19.8 | 17.2; the one-launch kernel's shared row tiles, 64 rows over a window of 8 KV heads x 256 (1.6), 15.3 | 14.7 (step).
// Heads are rounded up: 12 KV heads are one and a half to an XCD, and it reads the keys of two.
inline bool merge_on_xcd(uint32_t hkv, size_t head_bytes, size_t part_bytes) {
  return head_bytes * ((hkv + 7u) / 8u) + part_bytes / 8 <= ((size_t)6 << 20);
}

// Rows of the merge that asks for all at once, four to a workgroup.  In turn: run = 0, span the rows of a KV head.  In runs, one of
// `run` workgroups for each XCD, that follow the split kernel's run of units there (one 8th of them, by row tile, then split), so they are
// counted with the padding of the last row tile; with KV heads in eights an XCD has whole heads in either order and in the one-launch
// kernel, and only the last workgroup of a head is padded.  A row tile that the end of a run cuts is merged by both sides in the
// share each wrote.  (Rows counted without the padding drift from the tiles: with 49 rows, 16 heads over 2, XCD 3 wrote the
// tile of rows 384 to 391 and merged rows 294 to 391.)
struct MergeRuns {
  uint32_t span, run;
};
inline MergeRuns merge_runs(uint32_t hkv, uint32_t rows_total, uint32_t n_mtiles, uint32_t n_splits) {
  if (hkv % 8u == 0u) {
    const uint32_t wgs = (rows_total + 3u) / 4u;
    return MergeRuns{wgs * 4u, hkv / 8u * wgs};
  }
  const uint32_t units = (hkv * n_mtiles * n_splits + 7u) / 8u;
  return MergeRuns{n_mtiles * (uint32_t)kBlockM, (units * (uint32_t)(kBlockM / 4) + n_splits - 1u) / n_splits};
}
// row of a wave, counted over KV heads of `span` rows each
__host__ __device__ __forceinline__ uint32_t merge_row(uint32_t block, uint32_t wave, uint32_t run) {
  return (run ? (block & 7u) * run + (block >> 3) : block) * 4u + wave;
}

// How the partial rows of a call are merged: by the kernel that asks for all of a row's at once or the one that looks at
// the weights first; and by the first in runs or in turn.  (shared_tiles: the partial rows are the one-launch kernel's, whose workgroups go by
// split, then row tile.  With a split map the rows without a merge would leave some XCDs idle: 1024 causal rows behind 0 keys
// 46.1 -> 51.5 us.)
struct MergePlan {
  bool at_once;
  MergeRuns rows;
};
inline MergePlan plan_merge(const AttnParams& p, const SplitMap& map, uint32_t head_dim, bool streamed, bool shared_tiles) {
  const uint32_t key_tiles = p.tile_end - p.tile_first;
  const size_t part_bytes = (size_t)p.n_splits * p.hkv * p.rows_pad * head_dim * (p.part_half ? 2 : 4);
  const bool at_once = map.n || (!streamed && (p.part_half || p.n_splits <= 8) && head_dim % 8 == 0 && head_dim <= 512 &&
                                 merge_at_once(p.n_splits, part_bytes));
  const bool one_xcd = map.n == 0 && head_dim >= 256 && (p.hkv % 8 == 0 || (!shared_tiles && units_by_row_tile(p, map, head_dim)));
  if (at_once && one_xcd && merge_on_xcd(p.hkv, (size_t)key_tiles * kBlockN * head_dim * 4, part_bytes))
    return MergePlan{true, merge_runs(p.hkv, p.rows_total, p.n_mtiles, p.n_splits)};
  return MergePlan{at_once, MergeRuns{p.rows_total, 0u}};
}

// host-side launchers (defined next to their kernels)
hipError_t launch_attn_scalar(const AttnParams& p, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s);
// (map: row tiles with split counts of their own, head_dim 512; n = 0 for none. It stands behind AttnParams in the
// arguments of these two and not inside it: its bytes, then 72 and now 104, pushed what the one-launch kernel reads first to a further
// line of the arguments, and a call with 64 canvas rows on a sliding layer took 9.77 us for 9.52.)
hipError_t launch_attn_mfma(const AttnParams& p, const SplitMap& map, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s);
hipError_t launch_attn_wsplit(const AttnParams& p, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s);
// (shared_tiles: see plan_merge)
hipError_t launch_attn_merge(const AttnParams& p, const SplitMap& map, uint32_t head_dim, bool streamed, bool shared_tiles, hipStream_t s);
hipError_t launch_state_merge(const StateMergeParams& p, hipStream_t s);
// l[row] = 1 where m[row] is finite, else 0: completes a state whose rows are already normalised
hipError_t launch_state_unit_l(float* m_plane, float* l_plane, uint32_t rows, hipStream_t s);
hipError_t launch_convert(const void* src, uint32_t src_dtype, void* dst, uint32_t dst_dtype, size_t n, hipStream_t s);
// gathers keys [0,t_all) of a strided (possibly ring) cache into planes [hkv][t_all][D] of dst_dtype
hipError_t launch_kv_gather(const void* src, uint32_t src_dtype, void* dst, uint32_t dst_dtype, uint32_t hkv,
                            uint32_t t_all, uint32_t head_dim, int64_t tok_stride, int64_t head_stride,
                            uint32_t ring_mask, hipStream_t s);

// The filtered path over rows [tok0, tok0 + ntok): thresholds and lists, then selection out of the lists.
hipError_t launch_topk_filter(const TopkParams& tp, uint32_t kv_dtype, hipStream_t s);
hipError_t launch_topk_list_select(const TopkParams& tp, uint32_t k_most, uint32_t kv_dtype, hipStream_t s);
hipError_t launch_topk_scores(const TopkParams& tp, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s);
hipError_t launch_topk_select(const TopkParams& tp, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s);

hipError_t launch_calib_copy(void* dst, const void* src, size_t bytes, hipStream_t s);
hipError_t launch_calib_mfma(float* sink, uint32_t workgroups, uint32_t iters, uint32_t operand_mode, hipStream_t s);

}  // namespace dg
