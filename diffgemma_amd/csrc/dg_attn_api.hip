// extern "C" boundary of libdg_attn_hip.so: descriptor validation, launch planning, and the
// reference-shaped dispatch entry.  No allocation, no host synchronisation, no exceptions.
#include "../../include/dg_attn.h"
#include "../../include/dg_attn_bench.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "attn_params.h"

namespace {

using dg::kMaxSplits;
constexpr size_t kAlign = 256;
// most key tiles (of 32 keys) a row tile may see for the one-launch kernel to be chosen.  Step time in us,
// one launch | split kernel + merge, 256-row canvas, 8 KV heads: head_dim 256: 40 tiles 19.8 | 23.4,
// 72 tiles 28.5 | 27.5, 104 tiles 37.8 | 28.7; head_dim 128: 40 tiles 12.7 | 15.1, 72 tiles 18.9 | 19.3,
// 104 tiles 25.0 | 21.4; head_dim 64: 40 tiles 11.6 | 13.4, 72 tiles 18.0 | 16.4.
#ifndef DG_WSPLIT_MAX_TILES
#define DG_WSPLIT_MAX_TILES 64
#endif
constexpr uint32_t kWsplitMaxTiles = DG_WSPLIT_MAX_TILES;
static_assert(kWsplitMaxTiles <= 64, "attn_wsplit.hip's leading reference for f16 probabilities is sized for at most 2048 keys per row");

inline size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }
inline uint32_t elem_size(uint32_t dt) { return dt == DG_F32 ? 4u : 2u; }
inline bool is_pow2(uint64_t x) { return x && !(x & (x - 1)); }

struct DeviceInfo {
  int checked = 0;  // 0 unknown, 1 ok, -1 wrong arch
  int cus = 256;
};

// Device memory of dg_attn_forward_static, the entry point that may not allocate: what
// dg_attn_forward takes as its workspace argument (split partial rows, converted copies of f32
// inputs) lives here instead.  Every device the library runs on holds its own copy at its own
// address until the process ends; the name below is only a host-side handle, the device address
// is looked up once per device (static_scratch_ptr) and that pointer is what kernels are given.
constexpr size_t kStaticScratchBytes = DG_ATTN_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
void* g_scratch_ptr[64] = {};
DeviceInfo g_dev[64];
thread_local uint32_t* g_tls_dbg = nullptr;
std::mutex g_dev_mu;

// Which caches this thread's calls streamed lately, to tell whether a call's key/value rows can still be in the
// memory-side cache (256 MB on MI355X): a cache is taken to be cold when other caches of more than 200 MiB in total
// were streamed since its last use, or on its first use when it is large (head_dim 512, where touching rows that were
// cached after all costs 3 %) or of any size (below, where it costs nothing that can be measured).  Decides only whether
// the kernels touch keys and values into the L2 ahead of their loads: same bits, other timing; under graph capture the
// decision recorded is the one made at capture.  64 entries: a loop over a model's layers (30 caches) has to find each of
// them again.
struct CacheMemo {
  const void* region = nullptr;
  uint64_t streamed_at_last_use = 0;
};
constexpr int kMemoEntries = 64;
thread_local CacheMemo g_memo[kMemoEntries];
thread_local uint64_t g_streamed = 0;

bool cache_is_cold(const void* region, uint64_t bytes, bool large_only) {
  int idx = -1, oldest = 0;
  for (int i = 0; i < kMemoEntries; ++i) {
    if (g_memo[i].region == region) idx = i;
    if (g_memo[i].streamed_at_last_use < g_memo[oldest].streamed_at_last_use) oldest = i;
  }
  bool cold;
  if (idx < 0) {
    cold = !large_only || bytes >= (32ull << 20);
    idx = oldest;
    g_memo[idx].region = region;
  } else {
    cold = g_streamed - g_memo[idx].streamed_at_last_use > (200ull << 20);
  }
  g_streamed += bytes;
  g_memo[idx].streamed_at_last_use = g_streamed;
  return cold;
}

struct ProfState {
  std::vector<hipEvent_t> ev;
  uint32_t used = 0;
  bool active = false;
};
thread_local ProfState g_prof;

int device_info(DeviceInfo* out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return DG_ERR_DEVICE;
  std::lock_guard<std::mutex> lock(g_dev_mu);
  DeviceInfo& di = g_dev[dev];
  if (di.checked == 0) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return DG_ERR_DEVICE;
    di.checked = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : -1;
    di.cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  }
  if (di.checked < 0) return DG_ERR_DEVICE;
  *out = di;
  return DG_OK;
}

// Compute units the launch plans are made for: those of the current device when it is a
// gfx950 part, else (no device: host-side sizing and tests) the 256 of an MI355X.  Sizing calls
// and launches use the same number, so a workspace sized by the library always fits its launch.
int plan_cus() {
  DeviceInfo di;
  return device_info(&di) == DG_OK ? di.cus : 256;
}

// Address of `scratch` on the current device, looked up the first time the device is seen.
int static_scratch_ptr(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return DG_ERR_DEVICE;
  std::lock_guard<std::mutex> lock(g_dev_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) return DG_ERR_DEVICE;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return DG_OK;
}

// Everything the launch needs that can be derived on the host without a device.
struct Plan {
  uint32_t group = 0, rows_total = 0, n_mtiles = 0, rows_pad = 0;
  uint32_t t_all = 0, lo_nc = 0, extra_lo = 0, win_m1 = 0xffffffffu;
  uint32_t clip_lo = 0, clip_hi = 0;   // keys that count: [clip_lo, clip_hi); the whole range unless a partial is asked for
  uint32_t cus = 256;
  uint32_t span_tiles = 0;      // most key tiles a 32-row tile sees
  uint32_t tile_first = 0, tile_end = 0, tiles_per_split = 0, n_splits = 1;
  uint32_t e_dtype = DG_BF16;   // element type the kernels compute in (bf16 or f16)
  bool convert_q = false, gather_kv = false, q_is_bf16 = false;
  bool scalar = false;
  bool wsplit = false;          // short key range, head_dim <= 256: keys split over the waves of a workgroup, one launch
  bool part_half = false;       // split partial rows travel as normalised f16 rows
  size_t off_q = 0, off_kv = 0, off_part_o = 0, off_part_ml = 0, total = 0;
  dg::SplitMap map = {};        // row tiles with split counts of their own (n = 0: none)
  float scale = 1.0f;
};

// Key tiles per split of the split kernel where the library chooses.  `base` = workgroups of one split, `room` = splits that
// keep it one round of the chip.
//
// head_dim 512: a tile takes c = 1.3 to 1.6 us, and a split what its partial rows take, written and read back, about 9 c / room:
// c n / s + 9 c s / room is least at s = sqrt(n room / 9).  The curve is flat around it; where it leads past the splits that
// are merged at once, fewer are taken as long as that makes a share at most three tiles longer, or 8 in all (32 rows over 3700 keys, 29 |
// 15 splits: peaked rows 25.0 | 24.8, flat 29.5 | 24.8; to 9 tiles, 48 rows over 4500, 29 | 16: 27.1 | 28.3, 30.3 | 28.5).  Attention call, us, splits
// of 6 tiles and more | this rule: 64 rows (room 32) over 841 keys 21.0 | 18.3, 2064 25.9 | 23.7,
// 5064 31.2 | 29.4; 128 rows (16) over 428 keys 21.7 | 18.6, 905 23.8 | 22.9, 2128 28.7 | 28.1; 256 rows (8) over 556 24.4 | 24.5, 1033 26.7 | 27.0.
//
// Once the merge has more workgroups than the chip has compute units (four rows each: past 64 rows of 16 heads), more than 8 rows at
// once cost it what they save the shares: 8 splits where that makes a share one tile longer.  More | 8 at most: 72 rows over 1000 keys,
// 11 splits, peaked 21.0 | 19.8, flat 21.1 | 20.1; 80 over 841, 9, 20.4 | 19.4, 20.4 | 19.5; 96 over 1264, 10, 24.0 | 23.1, 24.0 | 23.4; by
// two tiles, 96 over 1700, 11, 24.9 | 25.2, 25.0 | 25.5; 72 over 1500, 12, 23.1 | 22.0, 23.2 | 22.3.
//
// Other head counts (8 over 1 and 8, 16 over 1, 4 and 16, 32 over 4 and 8; 64 and 256 rows over 104 to 4256 keys), against the kernels and
// counts as they were before this rule: 2 to 75 % faster; slower for flat rows in 30 splits and more alone, 64 of 8 heads over 1 over 4200
// keys 30.1 | 31.6 (peaked 28.0 | 25.3).
//
// Fewer than kF32PartTiles tiles were one split as long as none was shorter than 6, and its rows fp32 until they are rounded for the
// output: where these are split, the partial rows are fp32 too.  They cost twice as much, so sqrt(n room / 18), and one split
// where that is small.  One split | this rule: 64 rows over 86 keys (n room 96) 14.2 | 16.0, over 184 (192) 18.4 | 17.1, over 314 (320)
// 23.6 | 18.1; 128 rows over 150 (80) 17.1 | 18.5, 228 (128) 21.0 | 20.0; 256 over 346 (88) 25.1 | 26.2; 200 causal rows behind 150
// (110) 25.9 | 25.7.
//
// Smaller head_dim: no split shorter than 6 tiles (a sliding layer's 40 tiles, step in us: 4 splits 25.7, 5 splits 24.8,
// 6 and 7 splits 23.7, 8 splits 24.5, 10 splits 33.4).
constexpr uint32_t kF32PartTiles = 12;
uint32_t tiles_of_split(uint32_t ntiles, uint32_t base, uint32_t cus, uint32_t hd, bool long_splits) {
  const uint32_t room = std::max(1u, std::min(cus / std::max(1u, base), kMaxSplits));
  if (hd != 512 || long_splits) {
    const uint32_t s = std::min(room, std::max(1u, ntiles / 6u));
    return (ntiles + s - 1) / s;
  }
  auto of = [&](uint32_t splits) { return (ntiles + splits - 1) / splits; };
  const bool f32_parts = ntiles < kF32PartTiles;
  if (f32_parts && ntiles * room < 108u) return ntiles;
  const double s = std::sqrt((double)ntiles * room / (f32_parts ? 18.0 : 9.0));
  const uint32_t t = std::max(std::max(1u, (uint32_t)(ntiles / s + 0.5)), of(room));
  const size_t split_bytes = (size_t)base * dg::kBlockM * hd * (f32_parts ? 4 : 2);
  auto at_once = [&](uint32_t splits) { return dg::merge_at_once(splits, splits * split_bytes); };
  if (at_once(of(t))) return of(t) > 8u && base * (dg::kBlockM / 4) > cus && of(8) <= t + 1u ? of(8) : t;
  for (uint32_t few = dg::kMergeFewSplits; few >= 8u; few -= 8u)
    if (at_once(of(of(few)))) return of(few) > t && of(few) <= std::max(t + 3u, few / 2u) ? of(few) : t;
  return t;
}

// Key tiles per workgroup of the one-launch kernel: all that a 32-row tile sees, or, where a few canvas rows over most of a
// window leave three quarters of the chip idle, a share of them, the rows merged as the split kernel's are (fp32 partial rows: in one
// launch nothing of a row is narrower; a workgroup's run is cut over its four waves again).  In tiles of a wave (1.07 us; a fifth
// more over an f16 cache, where peaked rows rescale) a number of shares costs the tiles of its longest run, and where it is not one, 2
// for the second launch and 1 for every 55 row tiles of partial rows.  Attention call, us, in 1 | 2 | 3 | 4 | 5 shares, 16 heads over
// 8: 16 rows over 36 tiles 15.5 in one, 10.9 in 5 (5 taken); 64 over 36 15.7 | 14.7 | 13.3 | 13.5 | 12.9 (3); 64 over 28 13.6 | 13.5 | 12.5 | 12.4 |
// 12.5 (4); 96 over 30 14.4 | 14.2 | 13.9 | 14.1 | 15.1 (4); 112 over 28 13.6 | 14.4 | 13.6 | 14.9 (1); over an f16 cache, peaked rows and flat ones,
// 64 over 30 18.7 | 15.7 | 14.4 | 13.3 | 13.8 and 14.7 | 13.7 | 12.9 | 12.6 | 13.1 (4).  Over 780 forms (1, 2 and 8 KV heads, 8 to 56 row tiles, 16 to 36
// key tiles, both caches) at most 3 % behind one launch; always 5 shares, as many as fit, was up to 14 % behind.
uint32_t share_of_short_range(const dg_attn_desc* d, const Plan& pl, uint32_t cus, uint32_t ntiles) {
  const uint32_t base = d->n_kv_heads * ((pl.rows_total + 31u) / 32u);
  if (d->head_dim != 256 || base * 9u > cus * 2u || pl.span_tiles < 17u + base / 6u) return ntiles;
  const double row_tiles = d->n_kv_heads * (pl.rows_total / 32.0), tile = pl.e_dtype == DG_F16 ? 1.2 : 1.0;
  auto cost = [&](uint32_t s) {
    const uint32_t share = (pl.span_tiles + s - 1) / s;
    return tile * ((share + 3u) / 4u) + (s > 1 ? 2.0 + s * row_tiles / 55.0 : 0.0);
  };
  uint32_t s = 1;
  for (uint32_t more = 2; more <= std::min(cus / base, 5u); ++more)
    if (cost(more) < cost(s)) s = more;
  return (ntiles + s - 1) / s;
}

// Row tiles that see different numbers of key tiles (causal rows of a global layer): split counts of their own, so that no
// share is longer than the smallest length that leaves one round of the chip.  With 16-bit partial rows (what the merge for
// them reads) and a prefix the host knows.  Taken where that shortens the longest share by a tenth and by two key tiles: attention
// call, us, one count for all | split map: 1024 causal rows behind 0 keys 50.7 | 45.1 (shares of 16 tiles become 12), behind 300
// 60.4 | 55.8, 901 behind 0 43.4 | 38.7, 700 behind 0 36.0 | 31.8, behind 700 51.5 | 45.6; by one tile: 512 behind 0 26.0 | 26.5,
// 300 20.5 | 19.9, 200 17.2 | 18.0, 256 rows, 128 of them causal, behind 300 23.9 | 25.0.
bool plan_split_map(const dg_attn_desc* d, const Plan& pl, int cus, uint32_t ntiles, dg::SplitMap* out) {
  if (d->head_dim != 512 || d->causal_rows == 0 || d->window != 0 || (d->flags & DG_ATTN_F_T_LO_EXPLICIT) || !pl.part_half) return false;
  const uint32_t budget = (uint32_t)cus / d->n_kv_heads;
  if (pl.tiles_per_split >= ntiles || budget < pl.n_mtiles || ntiles >= 65536u) return false;
  const dg::FastDiv by_group = dg::make_fast_div(pl.group);
  auto tiles = [&](uint32_t mt) -> uint32_t {   // as the kernel cuts them
    const uint32_t b = dg::fast_div(std::min((mt + 1) * dg::kBlockM, pl.rows_total) - 1, by_group);
    uint32_t hi = b < d->causal_rows ? std::min(pl.t_all, d->kv_len + b + 1) : pl.t_all;
    if (pl.extra_lo < pl.t_all && dg::fast_div(mt * dg::kBlockM, by_group) < d->causal_rows) hi = pl.t_all;
    return (hi + dg::kBlockN - 1) / dg::kBlockN;
  };
  // No length below the one where the partial rows of all row tiles cost what shorter shares save.  Down to four fifths of it the
  // longest share is shorter (layer step: 1024 rows behind 0 keys 46.4 -> 45.7 us, 12 -> 11 tiles; 700 behind 0 36.3 -> 35.1; 600 behind 200
  // 48.2 -> 42.4), but row tiles of one share, whose rows are fp32 until the output, would be two with 16-bit partial rows (rows 352
  // to 383 of the 1024).
  const double s = std::sqrt((double)ntiles * budget / pl.n_mtiles / 9.0);
  const uint32_t len = std::max(1u, (uint32_t)(ntiles / std::max(1.0, s))), tps = pl.tiles_per_split;
  const uint32_t limit = tps < 3u ? 0u : std::min(tps - 2u, 9u * tps / 10u);
  return dg::shortest_split_map(pl.n_mtiles, len, limit, budget, tiles, out) && out->n > 1;
}

// Scratch a split count takes, and the count for a call that has `scratch` bytes of it: what the rule asks for, or, where
// that is more, splits of at least 6 tiles (a caller may hold what an earlier library asked for).
// `with_map`: the call may have a split map.  Not where the prefix length is read when the kernels run (every row tile then has
// the same count), nor where the plan is not that of a dense call.
int make_plan(const dg_attn_desc* d, int cus, Plan* pl, const uint32_t* key_range = nullptr, size_t scratch = SIZE_MAX,
              bool with_map = true) {
  if (!d) return DG_ERR_NULL;
  pl->cus = (uint32_t)cus;
  const uint32_t hd = d->head_dim;
  if (d->canvas == 0 || d->canvas > 65536 || d->n_q_heads == 0 || d->n_kv_heads == 0) return DG_ERR_SHAPE;
  if (d->n_q_heads % d->n_kv_heads != 0 || d->n_q_heads > 65535) return DG_ERR_SHAPE;
  if (d->kernel > DG_KERNEL_MFMA) return DG_ERR_UNSUPPORTED;
  pl->scalar = d->kernel == DG_KERNEL_SCALAR;
  if (pl->scalar) {
    if (hd == 0 || hd > 512 || hd % 8 != 0) return DG_ERR_SHAPE;
  } else if (hd != 32 && hd != 64 && hd != 128 && hd != 256 && hd != 512) {
    return DG_ERR_SHAPE;
  }
  if ((uint64_t)d->kv_len + d->canvas > 0x7fffffffull) return DG_ERR_SHAPE;
  // the kernels address query rows with 32-bit byte offsets
  if ((uint64_t)d->canvas * d->n_q_heads * hd * 2ull >= (1ull << 32)) return DG_ERR_SHAPE;
  if (d->q_dtype > DG_F32 || d->kv_dtype > DG_F32 || d->out_dtype > DG_F32) return DG_ERR_DTYPE;
  if (d->out_dtype == DG_F16) return DG_ERR_DTYPE;
  if (d->causal_rows > d->canvas) return DG_ERR_MASK;
  if (d->kv_ring_mask != 0) {
    if (!is_pow2((uint64_t)d->kv_ring_mask + 1) || d->kv_ring_mask + 1 < (uint32_t)dg::kBlockN) return DG_ERR_LAYOUT;
  }
  pl->t_all = d->kv_len + d->canvas;
  if ((d->flags & DG_ATTN_F_T_LO_EXPLICIT) && d->t_lo > pl->t_all) return DG_ERR_MASK;
  if (!(d->softmax_scale >= 0.0f)) return DG_ERR_MASK;
  pl->scale = d->softmax_scale == 0.0f ? 1.0f : d->softmax_scale;

  // element type: the cache decides; f32 anywhere is brought down to f16 first
  pl->e_dtype = d->kv_dtype == DG_BF16 ? DG_BF16 : DG_F16;
  pl->gather_kv = d->kv_dtype == DG_F32;
  if (d->q_dtype == DG_F32) {
    // f32 queries become bf16 by truncation, the reference wrapper's rounding of Q
    // (src/shaders/attn/attention/mod.rs:218-240), whatever the cache holds
    pl->convert_q = true;
    pl->q_is_bf16 = pl->e_dtype == DG_F16;
  } else if (d->q_dtype == DG_BF16 && pl->e_dtype == DG_F16) {
    pl->q_is_bf16 = true;  // bf16 activations over an f16 cache: the reference's own pairing
  } else if (d->q_dtype != pl->e_dtype) {
    return DG_ERR_DTYPE;   // f16 Q over a bf16 cache
  }

  if (!pl->gather_kv) {
    // rows must be 16-byte addressable for the direct-to-LDS loads
    const int64_t s[5] = {d->k_tok_stride, d->k_head_stride, d->v_base_off, d->v_tok_stride, d->v_head_stride};
    for (int64_t x : s)
      if (x < 0 || x % 8 != 0) return DG_ERR_LAYOUT;
    if (d->kv_region_bytes % 16 != 0) return DG_ERR_LAYOUT;
    if (d->k_tok_stride < (int64_t)hd || d->v_tok_stride < (int64_t)hd) return DG_ERR_LAYOUT;
    if (d->k_tok_stride * 2 * dg::kBlockN >= (1ll << 31) || d->v_tok_stride * 2 * dg::kBlockN >= (1ll << 31))
      return DG_ERR_LAYOUT;
  } else {
    if (d->k_tok_stride < 0 || d->k_head_stride < 0 || d->v_base_off < 0 || d->v_tok_stride < 0 ||
        d->v_head_stride < 0)
      return DG_ERR_LAYOUT;
  }

  pl->group = d->n_q_heads / d->n_kv_heads;
  pl->rows_total = d->canvas * pl->group;
  pl->n_mtiles = (pl->rows_total + dg::kBlockM - 1) / dg::kBlockM;
  pl->rows_pad = pl->n_mtiles * dg::kBlockM;

  // mask constants (reference rules, src/shaders/attn/attention/attention.metal:49-63)
  pl->win_m1 = d->window ? d->window - 1u : 0xffffffffu;
  pl->lo_nc = (d->window && d->kv_len > d->window - 1u) ? d->kv_len - (d->window - 1u) : 0u;
  if (d->flags & DG_ATTN_F_T_LO_EXPLICIT) pl->lo_nc = d->t_lo;
  pl->extra_lo = (d->flags & DG_ATTN_F_CAUSAL_SEES_MASKED) ? std::min(d->kv_len + d->causal_rows, pl->t_all) : pl->t_all;

  // key tiles any row can see
  uint32_t lo_all = 0xffffffffu;
  if (d->causal_rows < d->canvas) lo_all = std::min(lo_all, pl->lo_nc);
  if (d->causal_rows > 0) {
    const uint32_t qpos0 = d->kv_len;
    lo_all = std::min(lo_all, (d->window && qpos0 > d->window - 1u) ? qpos0 - (d->window - 1u) : 0u);
  }
  lo_all = std::min(lo_all, pl->t_all);
  // a ring must hold every visible position at once, or two of them share a slot
  if (d->kv_ring_mask != 0 && pl->t_all - lo_all > d->kv_ring_mask + 1u) return DG_ERR_LAYOUT;
  pl->clip_lo = 0;
  pl->clip_hi = pl->t_all;
  if (key_range) {
    if (key_range[0] > key_range[1]) return DG_ERR_MASK;
    pl->clip_lo = std::min(key_range[0], pl->t_all);
    pl->clip_hi = std::min(key_range[1], pl->t_all);
    lo_all = std::max(lo_all, pl->clip_lo);
  }
  pl->tile_first = lo_all / dg::kBlockN;
  pl->tile_end = std::max(pl->tile_first, (pl->clip_hi + dg::kBlockN - 1) / dg::kBlockN);
  const uint32_t ntiles = std::max(1u, pl->tile_end - pl->tile_first);

  // A short key range at head_dim <= 256 (a sliding-window layer) runs as one launch in which the four waves
  // of a workgroup split the keys and merge in LDS (attn_wsplit.hip): every workgroup then streams all keys
  // its rows see, which pays while that is a few thousand keys.  The span is what one 32-row tile sees, not
  // the union over the canvas (causal windowed rows each see window keys, the canvas window + canvas).
  {
    uint32_t span = 0;
    if (d->causal_rows < d->canvas) span = std::max(span, pl->t_all - std::min(pl->lo_nc, pl->t_all));
    if (d->causal_rows > 0) {
      uint32_t c = d->kv_len + d->causal_rows;
      if (d->window) c = std::min(c, d->window + dg::kBlockN);
      if (d->flags & DG_ATTN_F_CAUSAL_SEES_MASKED) c = pl->t_all;
      span = std::max(span, std::min(c, pl->t_all));
    }
    pl->span_tiles = std::min(ntiles, span / dg::kBlockN + 2u);
    pl->wsplit = !pl->scalar && hd <= 256 && d->n_splits == 0 && !(d->flags & DG_ATTN_F_SPLIT_OVER_WORKGROUPS) &&
                 pl->span_tiles <= kWsplitMaxTiles;
  }
  const uint32_t base = d->n_kv_heads * pl->n_mtiles;
  // workspace carve-up, with splits of `tps` key tiles; f32_parts: partial rows stay fp32 whatever the flags allow
  auto carve = [&](uint32_t tps, bool f32_parts) {
    pl->tiles_per_split = tps;
    pl->n_splits = (ntiles + tps - 1) / tps;
    size_t off = 0;
    if (pl->convert_q) {
      pl->off_q = off;
      off += align_up((size_t)d->canvas * d->n_q_heads * hd * 2);
    }
    if (pl->gather_kv) {
      pl->off_kv = off;
      off += align_up((size_t)2 * d->n_kv_heads * pl->t_all * hd * 2);
    }
    // f16 partial rows need |V| <= 65504: an f16 cache guarantees it, for a bf16 cache the caller says so
    pl->part_half = pl->n_splits > 1 && !f32_parts && d->out_dtype != DG_F32 && !(d->flags & DG_ATTN_F_F32_PARTIALS) &&
                    (pl->e_dtype == DG_F16 || (d->flags & DG_ATTN_F_F16_PARTIALS));
    if (pl->n_splits > 1) {
      pl->off_part_o = off;
      off += align_up((size_t)pl->n_splits * d->n_kv_heads * pl->rows_pad * hd * (pl->part_half ? 2 : 4));
      pl->off_part_ml = off;
      off += align_up((size_t)pl->n_splits * d->n_kv_heads * pl->rows_pad * 2 * 4);
    }
    pl->total = off;
  };
  if (pl->wsplit) {
    const uint32_t share = share_of_short_range(d, *pl, (uint32_t)cus, ntiles);
    carve(share, true);
    if (pl->total > scratch) carve(ntiles, true);
  } else if (pl->scalar) {
    carve(ntiles, false);
  } else if (d->n_splits != 0) {
    const uint32_t splits = std::min(std::min(d->n_splits, kMaxSplits), ntiles);
    carve((ntiles + splits - 1) / splits, false);
  } else {
    carve(tiles_of_split(ntiles, base, (uint32_t)cus, hd, false), hd == 512 && ntiles < kF32PartTiles);
    dg::SplitMap map;
    if (with_map && !key_range && plan_split_map(d, *pl, cus, ntiles, &map)) {
      // (sized for either, so that one workspace serves the entry points with and without a host-known prefix)
      const size_t rows = (size_t)d->n_kv_heads * map.units * dg::kBlockM, equal = pl->total;
      const size_t ml = pl->off_part_o + align_up(rows * hd * 2), both = std::max(equal, ml + align_up(rows * 8));
      if (both <= scratch) {
        pl->map = map;
        pl->n_splits = map.n;
        pl->off_part_ml = ml;
        pl->total = both;
      }
    }
    if (pl->total > scratch) carve(tiles_of_split(ntiles, base, (uint32_t)cus, hd, true), false);
  }
  return DG_OK;
}

}  // namespace

extern "C" {

uint32_t dg_attn_abi_version(void) { return DG_ATTN_ABI_VERSION; }

const char* dg_attn_strerror(int status) {
  switch (status) {
    case DG_OK: return "ok";
    case DG_ERR_NULL: return "required pointer is null";
    case DG_ERR_SHAPE: return "unsupported canvas / head count / head_dim";
    case DG_ERR_DTYPE: return "unsupported dtype tag or dtype combination";
    case DG_ERR_LAYOUT: return "KV strides or offsets not usable (16-byte alignment, ring mask, range)";
    case DG_ERR_WORKSPACE: return "workspace missing or too small";
    case DG_ERR_MASK: return "inconsistent mask description";
    case DG_ERR_LAUNCH: return "HIP launch failed";
    case DG_ERR_DEVICE: return "no gfx950 device current";
    case DG_ERR_UNSUPPORTED: return "request not implemented";
    case DG_ERR_SCRATCH_LIMIT:
      return "the call needs more scratch than dg_attn_forward_static holds (dg_attn_static_scratch_bytes); "
             "use dg_attn_forward with a workspace";
    default: return "unknown status";
  }
}

void dg_attn_desc_reference_layout(dg_attn_desc* d) {
  const int64_t row = (int64_t)d->n_kv_heads * d->head_dim;
  d->k_tok_stride = 2 * row;
  d->k_head_stride = d->head_dim;
  d->v_base_off = row;
  d->v_tok_stride = 2 * row;
  d->v_head_stride = d->head_dim;
}

void dg_attn_desc_head_major_layout(dg_attn_desc* d, uint64_t t_cap) {
  d->k_tok_stride = d->head_dim;
  d->k_head_stride = (int64_t)t_cap * d->head_dim;
  d->v_base_off = (int64_t)d->n_kv_heads * (int64_t)t_cap * d->head_dim;
  d->v_tok_stride = d->head_dim;
  d->v_head_stride = (int64_t)t_cap * d->head_dim;
}

int dg_attn_workspace_bytes(const dg_attn_desc* d, size_t* out_bytes) {
  if (!d || !out_bytes) return DG_ERR_NULL;
  Plan pl;
  const int rc = make_plan(d, plan_cus(), &pl);
  if (rc != DG_OK) return rc;
  *out_bytes = pl.total;
  return DG_OK;
}

int dg_attn_resolved_splits(const dg_attn_desc* d, uint32_t* out_splits) {
  if (!d || !out_splits) return DG_ERR_NULL;
  Plan pl;
  const int rc = make_plan(d, plan_cus(), &pl);
  if (rc != DG_OK) return rc;
  *out_splits = pl.n_splits;
  return DG_OK;
}

int dg_attn_visible_pairs(const dg_attn_desc* d, uint64_t* pairs, double* flops) {
  if (!d) return DG_ERR_NULL;
  Plan pl;
  const int rc = make_plan(d, plan_cus(), &pl, nullptr, SIZE_MAX, false);
  if (rc != DG_OK) return rc;
  uint64_t n = 0;
  for (uint32_t tok = 0; tok < d->canvas; ++tok) {
    const bool causal = tok < d->causal_rows;
    const uint32_t qpos = d->kv_len + tok;
    uint32_t lo, hi, extra;
    if (causal) {
      hi = std::min(pl.t_all, qpos + 1u);
      lo = (d->window && qpos > d->window - 1u) ? qpos - (d->window - 1u) : 0u;
      extra = pl.extra_lo;
    } else {
      hi = pl.t_all;
      lo = pl.lo_nc;
      extra = pl.t_all;
    }
    if (hi > lo) n += hi - lo;
    const uint32_t e = std::max(extra, std::max(hi, lo));
    if (pl.t_all > e) n += pl.t_all - e;
  }
  if (pairs) *pairs = n;
  if (flops) *flops = 4.0 * d->head_dim * d->n_q_heads * (double)n;
  return DG_OK;
}

namespace {
// Fills the kernel parameter block from a validated descriptor; runs the f32 -> f16 conversion
// passes into the workspace when the plan asks for them.
int fill_params(const dg_attn_desc* d, const Plan& pl, const void* q, const void* kv_base, void* out, float* lse,
                char* ws, hipStream_t s, dg::AttnParams* pp) {
  const uint32_t hd = d->head_dim;
  const uint32_t esz_kv = elem_size(d->kv_dtype);
  dg::AttnParams& p = *pp;
  std::memset(&p, 0, sizeof(p));
  const char* region = (const char*)kv_base + d->kv_region_bytes;
  p.q = q;
  p.ring_mask = d->kv_ring_mask;
  p.t_clip_lo = pl.clip_lo;
  p.t_clip_hi = pl.clip_hi;
  if (pl.convert_q) {
    if (dg::launch_convert(q, d->q_dtype, ws + pl.off_q, DG_BF16, (size_t)d->canvas * d->n_q_heads * hd, s) != hipSuccess)
      return DG_ERR_LAUNCH;
    p.q = ws + pl.off_q;
  }
  if (pl.gather_kv) {
    char* kp = ws + pl.off_kv;
    char* vp = kp + (size_t)d->n_kv_heads * pl.t_all * hd * 2;
    if (dg::launch_kv_gather(region, d->kv_dtype, kp, pl.e_dtype, d->n_kv_heads, pl.t_all, hd, d->k_tok_stride,
                             d->k_head_stride, d->kv_ring_mask, s) != hipSuccess)
      return DG_ERR_LAUNCH;
    if (dg::launch_kv_gather(region + d->v_base_off * (int64_t)esz_kv, d->kv_dtype, vp, pl.e_dtype, d->n_kv_heads,
                             pl.t_all, hd, d->v_tok_stride, d->v_head_stride, d->kv_ring_mask, s) != hipSuccess)
      return DG_ERR_LAUNCH;
    p.k = kp;
    p.v = vp;
    p.k_tok_stride = p.v_tok_stride = hd;
    p.k_head_stride = p.v_head_stride = (int64_t)pl.t_all * hd;
    p.ring_mask = 0;
  } else {
    p.k = region;
    p.v = region + d->v_base_off * 2;
    p.k_tok_stride = d->k_tok_stride;
    p.k_head_stride = d->k_head_stride;
    p.v_tok_stride = d->v_tok_stride;
    p.v_head_stride = d->v_head_stride;
  }
  p.out = out;
  p.lse = lse;
  p.dbg = nullptr;
  p.canvas = d->canvas;
  p.hq = d->n_q_heads;
  p.hkv = d->n_kv_heads;
  p.group = pl.group;
  p.kv_len = d->kv_len;
  p.t_all = dg::keys_of_range(pl.tile_first, pl.tile_end, pl.t_all);   // (the whole range ends with the last key)
  p.causal_rows = d->causal_rows;
  p.win_m1 = pl.win_m1;
  p.lo_nc = pl.lo_nc;
  p.extra_lo = pl.extra_lo;
  p.rows_total = pl.rows_total;
  p.rows_pad = pl.rows_pad;
  p.n_mtiles = pl.n_mtiles;
  p.n_splits = pl.n_splits;
  p.tile_first = pl.tile_first;
  p.tiles_per_split = pl.tiles_per_split;
  p.tile_end = pl.tile_end;
  p.q_is_bf16 = pl.q_is_bf16 ? 1u : 0u;
  p.out_dtype = d->out_dtype;
  p.out_trunc = (d->flags & DG_ATTN_F_OUT_TRUNCATE) ? 1u : 0u;
  p.part_half = pl.part_half ? 1u : 0u;
  p.cus = pl.cus;
  p.lo_explicit = (d->flags & DG_ATTN_F_T_LO_EXPLICIT) ? 1u : 0u;
  p.sees_masked = (d->flags & DG_ATTN_F_CAUSAL_SEES_MASKED) ? 1u : 0u;
  // key/value rows this call streams: more than the 256 MiB memory-side cache holds cannot have
  // stayed there from the previous call, whatever else runs in between (131072 keys: 0.933 -> 0.912 ms)
  const uint64_t kv_streamed = 2ull * d->n_kv_heads * (uint64_t)(pl.tile_end - pl.tile_first) * dg::kBlockN * d->head_dim * 2ull;
  // ... and a cache that other large caches were streamed after since its last use has been displaced
  // (cache_is_cold); DG_ATTN_F_KV_CACHED says the caller knows better
  const bool cold = cache_is_cold(region, kv_streamed, hd == 512);
  p.touch_ahead = ((d->flags & DG_ATTN_F_KV_FROM_HBM) || kv_streamed > (256ull << 20) ||
                   (cold && !(d->flags & DG_ATTN_F_KV_CACHED))) ? 1u : 0u;
  p.scale_log2 = pl.scale * dg::kLog2e;
  return DG_OK;
}

}  // namespace

namespace {
// One attention call with its plan made: validation of the pointers, parameter block, launches.
int forward_planned(const dg_attn_desc* d, const Plan& pl, const void* q, const void* kv_base, void* out, float* lse,
                    void* workspace, size_t workspace_bytes, void* stream, const uint32_t* step_dev = nullptr) {
  int rc = DG_OK;
  if (pl.total > 0 && (!workspace || workspace_bytes < pl.total)) return DG_ERR_WORKSPACE;
  if (pl.total > 0 && ((uintptr_t)workspace % 16) != 0) return DG_ERR_WORKSPACE;
  if (((uintptr_t)q % 16) != 0 || ((uintptr_t)kv_base % 16) != 0 || ((uintptr_t)out % 16) != 0) return DG_ERR_LAYOUT;
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const uint32_t hd = d->head_dim;

  dg::AttnParams p;
  rc = fill_params(d, pl, q, kv_base, out, lse, ws, s, &p);
  if (rc != DG_OK) return rc;
  if (pl.n_splits > 1) {
    p.part_o = (float*)(ws + pl.off_part_o);
    p.part_ml = (float*)(ws + pl.off_part_ml);
  }
  p.dbg = g_tls_dbg;  // set only while dg_attention_dispatch is on the stack
  p.step_dev = step_dev;
  if (step_dev && (pl.scalar || pl.gather_kv)) return DG_ERR_UNSUPPORTED;   // (the f32 cache copy is made for a host-known length)

  if (pl.scalar) {
    if (dg::launch_attn_scalar(p, hd, pl.e_dtype, s) != hipSuccess) return DG_ERR_LAUNCH;
    return DG_OK;
  }
  const bool prof = g_prof.active && 2 * (size_t)g_prof.used + 1 < g_prof.ev.size();
  if (prof) (void)hipEventRecord(g_prof.ev[2 * g_prof.used], s);
  if ((pl.wsplit ? dg::launch_attn_wsplit(p, hd, pl.e_dtype, s) : dg::launch_attn_mfma(p, pl.map, hd, pl.e_dtype, s)) != hipSuccess)
    return DG_ERR_LAUNCH;
  if (prof) {
    (void)hipEventRecord(g_prof.ev[2 * g_prof.used + 1], s);
    ++g_prof.used;
  }
  if (pl.n_splits > 1 && dg::launch_attn_merge(p, pl.map, hd, (d->flags & DG_ATTN_F_STREAMED_MERGE) != 0, pl.wsplit, s) != hipSuccess)
    return DG_ERR_LAUNCH;
  return DG_OK;
}
}  // namespace

int dg_attn_forward(const dg_attn_desc* d, const void* q, const void* kv_base, void* out, float* lse,
                    void* workspace, size_t workspace_bytes, void* stream) {
  if (!d || !q || !kv_base || !out) return DG_ERR_NULL;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  Plan pl;
  rc = make_plan(d, di.cus, &pl, nullptr, workspace ? workspace_bytes : 0);
  if (rc != DG_OK) return rc;
  return forward_planned(d, pl, q, kv_base, out, lse, workspace, workspace_bytes, stream);
}

int dg_attn_forward_dev(const dg_attn_desc* d, const dg_step_params* step_dev, const void* q, const void* kv_base, void* out,
                        float* lse, void* workspace, size_t workspace_bytes, void* stream) {
  if (!d || !step_dev || !q || !kv_base || !out) return DG_ERR_NULL;
  if (((uintptr_t)step_dev % 4) != 0) return DG_ERR_LAYOUT;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  Plan pl;
  rc = make_plan(d, di.cus, &pl, nullptr, workspace ? workspace_bytes : 0, false);
  if (rc != DG_OK) return rc;
  return forward_planned(d, pl, q, kv_base, out, lse, workspace, workspace_bytes, stream, (const uint32_t*)step_dev);
}

size_t dg_attn_static_scratch_bytes(void) { return kStaticScratchBytes; }

int dg_attn_forward_static(const dg_attn_desc* d, const void* q, const void* kv_base, void* out, float* lse,
                           void* stream) {
  if (!d || !q || !kv_base || !out) return DG_ERR_NULL;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  Plan pl;
  // Calls that can do without scratch do without it, whatever splitting their keys would save (64 rows over a window 16 us for
  // 13): they never touched it, and callers may have them overlap.
  rc = make_plan(d, di.cus, &pl, nullptr, 0);
  if (rc != DG_OK) return rc;
  if (pl.total > 0) {
    pl = Plan();
    rc = make_plan(d, di.cus, &pl, nullptr, kStaticScratchBytes);
    if (rc != DG_OK) return rc;
  }
  if (pl.total > kStaticScratchBytes) return DG_ERR_SCRATCH_LIMIT;
  void* ptr = nullptr;
  rc = static_scratch_ptr(&ptr);
  if (rc != DG_OK) return rc;
  // Nothing in the scratch has to start at zero: a launch writes every partial row and every
  // converted element it later reads.
  return forward_planned(d, pl, q, kv_base, out, lse, ptr, kStaticScratchBytes, stream);
}

// ---- key-range partials and their merge --------------------------------------------------------

namespace {
inline size_t state_bytes_of(const dg_attn_desc* d) {
  const size_t rows = (size_t)d->canvas * d->n_q_heads;
  return (dg::state_acc_offset(rows) + rows * d->head_dim) * sizeof(float);
}
// The descriptor of a partial: the caller's, with an fp32 result (the state's accumulators).
inline dg_attn_desc partial_desc(const dg_attn_desc* d) {
  dg_attn_desc pd = *d;
  pd.out_dtype = DG_F32;
  pd.flags &= ~(uint32_t)(DG_ATTN_F_OUT_TRUNCATE | DG_ATTN_F_F16_PARTIALS);
  return pd;
}
}  // namespace

int dg_attn_state_bytes(const dg_attn_desc* d, size_t* out_bytes) {
  if (!d || !out_bytes) return DG_ERR_NULL;
  Plan pl;
  const int rc = make_plan(d, plan_cus(), &pl, nullptr, SIZE_MAX, false);
  if (rc != DG_OK) return rc;
  *out_bytes = state_bytes_of(d);
  return DG_OK;
}

int dg_attn_partial_workspace_bytes(const dg_attn_desc* d, uint32_t t_begin, uint32_t t_end, size_t* out_bytes) {
  if (!d || !out_bytes) return DG_ERR_NULL;
  const dg_attn_desc pd = partial_desc(d);
  const uint32_t range[2] = {t_begin, t_end};
  Plan pl;
  const int rc = make_plan(&pd, plan_cus(), &pl, range);
  if (rc != DG_OK) return rc;
  *out_bytes = pl.total;
  return DG_OK;
}

int dg_attn_partial(const dg_attn_desc* d, uint32_t t_begin, uint32_t t_end, const void* q, const void* kv_base,
                    void* state, size_t state_bytes, void* workspace, size_t workspace_bytes, void* stream) {
  if (!d || !q || !kv_base || !state) return DG_ERR_NULL;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  const dg_attn_desc pd = partial_desc(d);
  const uint32_t range[2] = {t_begin, t_end};
  Plan pl;
  rc = make_plan(&pd, di.cus, &pl, range, workspace ? workspace_bytes : 0);
  if (rc != DG_OK) return rc;
  if (state_bytes < state_bytes_of(d) || ((uintptr_t)state % 16) != 0) return DG_ERR_WORKSPACE;
  // The attention kernels leave the row normalised (acc / l) and its log-sum-exp: the state's normal
  // form is exactly that, (m, l) = (lse, 1), or (-inf, 0) for a row that saw no key of the range.
  const size_t rows = (size_t)d->canvas * d->n_q_heads;
  float* const m_plane = (float*)state;
  float* const acc = m_plane + dg::state_acc_offset(rows);
  rc = forward_planned(&pd, pl, q, kv_base, acc, m_plane, workspace, workspace_bytes, stream);
  if (rc != DG_OK) return rc;
  return dg::launch_state_unit_l(m_plane, m_plane + rows, (uint32_t)rows, (hipStream_t)stream) == hipSuccess
             ? DG_OK
             : DG_ERR_LAUNCH;
}

int dg_attn_merge(const dg_attn_desc* d, const void* const* states, uint32_t n_states, void* out, float* lse,
                  void* state_out, void* stream) {
  if (!d || !states) return DG_ERR_NULL;
  if (!out && !state_out) return DG_ERR_NULL;
  if (n_states == 0 || n_states > dg::kMaxStates) return DG_ERR_SHAPE;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  Plan pl;
  rc = make_plan(d, di.cus, &pl, nullptr, SIZE_MAX, false);
  if (rc != DG_OK) return rc;
  dg::StateMergeParams p;
  std::memset(&p, 0, sizeof(p));
  for (uint32_t i = 0; i < n_states; ++i) {
    if (!states[i] || ((uintptr_t)states[i] % 16) != 0) return DG_ERR_NULL;
    p.states[i] = (const float*)states[i];
  }
  if ((out && ((uintptr_t)out % 16) != 0) || (state_out && ((uintptr_t)state_out % 16) != 0)) return DG_ERR_LAYOUT;
  p.n = n_states;
  p.rows = d->canvas * d->n_q_heads;
  p.hd = d->head_dim;
  p.hq = d->n_q_heads;
  p.out = out;
  p.lse = lse;
  p.state_out = (float*)state_out;
  p.out_dtype = d->out_dtype;
  p.out_trunc = (d->flags & DG_ATTN_F_OUT_TRUNCATE) ? 1u : 0u;
  p.dbg = g_tls_dbg;
  return dg::launch_state_merge(p, (hipStream_t)stream) == hipSuccess ? DG_OK : DG_ERR_LAUNCH;
}

namespace {
// Top-k sparse attention walks the canvas in row blocks so that the fp32 score plane of a block
// ([Hq][rows][t_pad]) stays within the memory-side cache between the kernel that writes it and
// the one that reads it.
#ifndef DG_TOPK_PLANE_MIB
#define DG_TOPK_PLANE_MIB 144
#endif
constexpr size_t kTopkPlaneBudget = (size_t)DG_TOPK_PLANE_MIB << 20;

struct TopkPlan {
  uint32_t t_pad = 0, block_tok = 0;
  size_t total = 0;
  size_t general = 0;      // what the general path alone needs: with less than `total` it is taken
  // filtered path (pass_tok = 0: not taken): canvas rows per pass and, within a pass, per block of the general path
  // behind it; sampled keys; key-range splits; byte offsets in the workspace
  uint32_t pass_tok = 0, redo_tok = 0, stride = 0, sample_n = 0, sample_splits = 0, splits = 0, k_most = 0;
  size_t off_block = 0, off_plane = 0, off_tau = 0, off_cand_n = 0, off_kept = 0, off_lists = 0;
  uint32_t kept_pad = 0;
};

// Where the filtered path is taken: what its kernels are made for (head_dim 512, linear cache, every row sees all keys
// up to its own or the last), at most 512 keys kept (what a wave holds of a row's list), prefixes long
// enough that a pass over 1/17 of the keys tells where the k-th score lies, and calls large enough.  Its seven and more
// launches take about 40 us however small they are; the general path, a workgroup per (row, head) in the end, takes 35 and its
// time grows with the rounds of the chip those workgroups need (four of them at once on a compute unit).  Measured, the
// attention call with 16 heads over a bf16 cache, general | filtered path: 16 rows (256 workgroups) over 24k keys 67.6 | 76.8 us;
// 32 rows over 17k 66.6 | 70.7, 24k 81.7 | 77.5; 48 rows over 9k 55.0 | 62.9, 12k 75.5 | 68.0; 64 rows (a whole round) over 9k
// 58.3 | 64.6, 12k 68.6 | 69.7, 17k 83.9 | 76.1; 96 rows over 2100 65.6 | 53.0, 6500 91.2 | 62.7; 128 rows over 2100
// 69.7 | 55.8 (f16 71.2 | 59.7), 6500 85.6 | 64.7; 256 rows over 2100 120 | 66, 24k 450 | 172.  Over the reference's f16 cache, layer
// step: 64 rows over 14k 77.1 | 85.6, 16k 85.7 | 88.7, 18.4k 101 | 95, 128 over 2100 73.3 | 61.8.  That is with 64 to 192 keys kept (the
// production rule); with a fixed 128, 256 and 512 the lines lie no higher: 65 rows over 2200 keys 67.0 | 55.1, 78.7 | 69.1, 100.9 | 92.5, 128 rows over
// 2200 76.8 | 60.8, 91.1 | 76.6, 120 | 107, over 8000 101 | 72, 119 | 83, 148 | 105; 64 rows over 18.5k 81.8 | 75.1, 97.6 | 82.7, 122 | 96; 32 rows over 24.6k
// 73.9 | 77.3, 84.0 | 81.9, 100.5 | 93.3.
// And for rows the lists hold.  A row they do not (thousands of equal scores) has its block of canvas rows scored again:
// the attention call alone, 256 rows over 33k keys, general | filtered: none such 603 | 228 us, one 676 | 408, one in every canvas row
// 919 | 1229, all of them 1046 | 2031; 64 rows over 33k: 144 | 100, 224 | 334, 227 | 342, 263 | 530, over 18.5k 86 | 78, 134 | 233, 134 | 235, 168 | 355; 128 over
// 2200 69 | 56, 77 | 107, 77 | 109, 110 | 205, over 8000 90 | 67, 107 | 158, 109 | 160, 179 | 340.  The host cannot tell.
constexpr uint32_t kTopkFilterMinPrefix = 2048;
constexpr uint32_t kTopkFilterMinKeys[3] = {24576, 18432, 0};   // up to half a round, one round, more

size_t filter_bytes(const dg_attn_desc* d, const Plan& pl, uint32_t cus, uint32_t ntok, TopkPlan* tk) {
  const uint32_t n_mtiles = (ntok * pl.group + dg::kTopkFilterRows - 1) / dg::kTopkFilterRows;
  const uint32_t base = d->n_kv_heads * n_mtiles;
  const uint32_t n_tiles = (pl.t_all + dg::kBlockN - 1) / dg::kBlockN;
  // Whole rounds of the chip, four key tiles each at least; and segments that hold what comes.
  // A row's list is about stride w long, w = k / stride + 5 sqrt(k / stride) + 3 the rank of the threshold among the sampled
  // scores, in two segments per split.  The threshold is as uncertain as w sampled keys are, 1 / sqrt(w) of the list's length:
  // a segment that expects m entries holds m' + 4 sqrt(m') with m' = (1 + 4 / sqrt(w)) m.  (Half of what it holds, whatever w:
  // at 64 keys kept, w = 16, 35 expected in segments of 80 left one row in 130 over: 1024 rows behind 5k keys 546 us, now 298.)
  const double mean = (double)tk->k_most / tk->stride, w = mean + 5.0 * std::sqrt(mean) + 3.0;
  const double root = std::sqrt(dg::kTopkSegCap + 4.0) - 2.0, most = root * root / (1.0 + 4.0 / std::sqrt(w));
  const uint32_t fit = std::min((uint32_t)(w * tk->stride / 2.0 / most) + 1, dg::kMaxSplits);
  tk->splits = dg::splits_in_rounds(base, n_tiles, fit, std::min(std::max(fit, n_tiles / 4), dg::kMaxSplits), cus, 3);
  const size_t segs = (size_t)base * tk->splits * 4 * dg::kTopkSegs;
  tk->off_block = align_up((size_t)d->canvas * d->n_q_heads * sizeof(uint32_t));
  tk->off_plane = tk->off_block + align_up((size_t)ntok * sizeof(uint32_t));
  tk->off_tau = tk->off_plane;
  tk->off_cand_n = tk->off_tau + align_up((size_t)base * dg::kTopkFilterRows * sizeof(float));
  tk->off_kept = tk->off_cand_n + align_up(segs * sizeof(uint32_t));
  tk->kept_pad = (tk->k_most + dg::kTopkListAlign - 1) / dg::kTopkListAlign * dg::kTopkListAlign;
  tk->off_lists = tk->off_kept + align_up((size_t)ntok * d->n_q_heads * tk->kept_pad * 8);
  // Sampled keys: two key tiles each at least.
  const uint32_t sample_tiles = (tk->sample_n + dg::kBlockN - 1) / dg::kBlockN;
  const uint32_t sample_base = d->n_kv_heads * ((ntok * pl.group + dg::kTopkSampleRows - 1) / dg::kTopkSampleRows);
  tk->sample_splits = dg::splits_in_rounds(sample_base, sample_tiles, 1, std::max(1u, std::min(sample_tiles / 2, dg::kTopkSampleSplits)), cus, 4);
  // (the lists lie where the sampled keys' largest scores were)
  const size_t sample = (size_t)ntok * d->n_q_heads * tk->sample_splits * dg::kBlockN * sizeof(float);
  return tk->off_lists + align_up(std::max(segs * dg::kTopkSegAlloc * 8, sample));
}

void plan_filtered(const dg_attn_desc* d, const uint32_t* k_cfg, const Plan& pl, uint32_t cus, TopkPlan* tk) {
  if (d->head_dim != 512 || pl.lo_nc != 0 || pl.win_m1 != 0xffffffffu || d->kv_ring_mask != 0) return;
  if (d->kv_len < kTopkFilterMinPrefix || !std::isfinite(pl.scale) || (d->flags & DG_ATTN_F_TOPK_SCORE_PLANE)) return;
  const uint64_t rows = (uint64_t)d->canvas * d->n_q_heads;
  const uint32_t min_keys = kTopkFilterMinKeys[rows <= 2ull * cus ? 0 : rows <= 4ull * cus ? 1 : 2];
  if (pl.t_all < min_keys && !(d->flags & DG_ATTN_F_TOPK_THRESHOLD)) return;
  if (k_cfg[1] != 0u) {
    const uint64_t gran = std::max(k_cfg[0], 1u);
    const uint64_t most = (pl.t_all + gran - 1) / gran * gran / k_cfg[1];
    tk->k_most = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(most, k_cfg[2]), k_cfg[3]);
  } else {
    tk->k_most = std::max(k_cfg[0], 1u);
  }
  if (tk->k_most == 0u || tk->k_most > dg::kTopkListMax) return;
  // (odd: sampled rows of a head-major cache, 1 KiB each, then fall on all memory channels)
  tk->stride = std::max(17u, (pl.t_all + dg::kTopkSampleMax - 1) / dg::kTopkSampleMax | 1u);
  if (tk->stride > 21u) return;       // (17 to 21: the list of a row that keeps 512 keys still fits)
  // key rows of the sampled launch are `stride` rows apart, a tile's offsets have 31 bits
  if ((uint64_t)d->k_tok_stride * 2 * tk->stride * dg::kBlockN >= (1ull << 31)) return;
  if ((uint64_t)d->v_tok_stride * 2 * pl.t_all + 1024 >= (1ull << 32)) return;      // V rows are gathered by 32-bit offsets
  tk->sample_n = (pl.t_all + tk->stride - 1) / tk->stride;
  uint32_t ntok = d->canvas;
  size_t need = filter_bytes(d, pl, cus, ntok, tk);
  while (need > kTopkPlaneBudget && ntok > 32) {
    ntok = ((ntok + 1) / 2 + 31) & ~31u;
    need = filter_bytes(d, pl, cus, ntok, tk);
  }
  if (need > kTopkPlaneBudget) return;
  const size_t per_tok = (size_t)d->n_q_heads * tk->t_pad * sizeof(float);
  size_t total = std::max(tk->total, need);
  if (tk->block_tok == d->canvas) total = std::max(total, tk->off_plane + align_up((size_t)ntok * per_tok));
  const size_t fit = (total - tk->off_plane) / per_tok;
  if (fit == 0) return;
  tk->total = total;
  tk->pass_tok = ntok;
  const uint32_t blocks = (uint32_t)((ntok + fit - 1) / fit);
  tk->redo_tok = (ntok + blocks - 1) / blocks;
}

int make_topk_plan(const dg_attn_desc* d, const uint32_t* k_cfg, const Plan& pl, uint32_t cus, TopkPlan* tk) {
  if (!k_cfg) return DG_ERR_NULL;
  if (pl.scalar || d->q_dtype == DG_F32 || d->kv_dtype == DG_F32) return DG_ERR_UNSUPPORTED;
  if (k_cfg[1] == 0u) {
    if (k_cfg[0] > (uint32_t)dg::kTopkMaxK) return DG_ERR_SHAPE;
  } else if (k_cfg[3] > (uint32_t)dg::kTopkMaxK || k_cfg[2] > k_cfg[3]) {
    return DG_ERR_SHAPE;
  }
  tk->t_pad = (pl.t_all + dg::kBlockN - 1) / dg::kBlockN * dg::kBlockN;
  const size_t per_tok = (size_t)d->n_q_heads * tk->t_pad * sizeof(float);
  size_t blk = std::max<size_t>(1, kTopkPlaneBudget / per_tok);
  if (blk >= 16) blk &= ~(size_t)15;
  tk->block_tok = (uint32_t)std::min<size_t>(blk, d->canvas);
  tk->total = align_up((size_t)tk->block_tok * per_tok);
  if (tk->total / sizeof(float) >= (1ull << 32)) return DG_ERR_SHAPE;   // score rows are addressed with 32-bit offsets
  tk->general = tk->total;
  plan_filtered(d, k_cfg, pl, cus, tk);
  return DG_OK;
}
}  // namespace

int dg_attn_topk_workspace_bytes(const dg_attn_desc* d, const uint32_t* k_cfg, size_t* out_bytes) {
  if (!d || !out_bytes) return DG_ERR_NULL;
  Plan pl;
  int rc = make_plan(d, plan_cus(), &pl, nullptr, SIZE_MAX, false);
  if (rc != DG_OK) return rc;
  TopkPlan tk;
  rc = make_topk_plan(d, k_cfg, pl, plan_cus(), &tk);
  if (rc != DG_OK) return rc;
  *out_bytes = tk.total;
  return DG_OK;
}

int dg_attn_topk_forward(const dg_attn_desc* d, const uint32_t* k_cfg, const void* q, const void* kv_base,
                         void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (!d || !q || !kv_base || !out) return DG_ERR_NULL;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != DG_OK) return rc;
  Plan pl;
  rc = make_plan(d, plan_cus(), &pl, nullptr, SIZE_MAX, false);
  if (rc != DG_OK) return rc;
  TopkPlan tk;
  rc = make_topk_plan(d, k_cfg, pl, plan_cus(), &tk);
  if (rc != DG_OK) return rc;
  if (workspace_bytes < tk.total) tk.pass_tok = 0;
  if (!workspace || workspace_bytes < tk.general || ((uintptr_t)workspace % 16) != 0) return DG_ERR_WORKSPACE;
  if (((uintptr_t)q % 16) != 0 || ((uintptr_t)kv_base % 16) != 0 || ((uintptr_t)out % 16) != 0) return DG_ERR_LAYOUT;
  hipStream_t s = (hipStream_t)stream;

  dg::TopkParams tp;
  std::memset(&tp, 0, sizeof(tp));
  rc = fill_params(d, pl, q, kv_base, out, nullptr, nullptr, s, &tp.a);   // no conversion passes: dtypes checked above
  if (rc != DG_OK) return rc;
  tp.a.dbg = g_tls_dbg;
  tp.s_plane = (float*)workspace;
  tp.t_pad = tk.t_pad;
  tp.tile_first = pl.tile_first;
  tp.tile_end = pl.tile_end;
  for (int i = 0; i < 4; ++i) tp.k_cfg[i] = k_cfg[i];
  tp.scale = pl.scale;
  const uint32_t ntiles = std::max(1u, pl.tile_end - pl.tile_first);
  // (timing aid: one event pair per stage, scores first)
  bool prof = false;
  auto mark = [&](uint32_t i) {
    if (prof) (void)hipEventRecord(g_prof.ev[2 * g_prof.used + i], s);
  };
  // the general path over canvas rows [tok0, tok0 + ntok)
  auto block = [&](uint32_t tok0, uint32_t ntok, bool marks) -> hipError_t {
    tp.tok0 = tok0;
    tp.ntok = ntok;
    tp.n_mtiles = (tp.ntok * pl.group + dg::kBlockM - 1) / dg::kBlockM;
    // enough workgroups for every CU, no split shorter than 8 key tiles; splits write disjoint
    // columns of the score plane, so there is nothing to merge
    const uint32_t base = d->n_kv_heads * tp.n_mtiles;
    uint32_t splits = std::max(1u, ((uint32_t)di.cus + base - 1u) / base);
    tp.n_splits = std::max(1u, std::min(splits, ntiles / 8u));
    if (marks) mark(0);
    hipError_t e = dg::launch_topk_scores(tp, d->head_dim, pl.e_dtype, s);
    if (marks) {
      mark(1);
      mark(2);
    }
    if (e == hipSuccess) e = dg::launch_topk_select(tp, d->head_dim, pl.e_dtype, s);
    return e;
  };
  const uint32_t step = tk.pass_tok ? tk.pass_tok : tk.block_tok;
  for (uint32_t tok0 = 0; tok0 < d->canvas; tok0 += step) {
    const uint32_t ntok = std::min(step, d->canvas - tok0);
    prof = g_prof.active && 2 * (size_t)g_prof.used + 3 < g_prof.ev.size();
    if (tk.pass_tok == 0) {
      if (block(tok0, ntok, true) != hipSuccess) return DG_ERR_LAUNCH;
    } else {
      char* const ws = (char*)workspace;
      dg::TopkParams fp = tp;
      fp.tok0 = tok0;
      fp.ntok = ntok;
      fp.n_mtiles = (ntok * pl.group + dg::kTopkFilterRows - 1) / dg::kTopkFilterRows;
      fp.n_splits = tk.splits;
      fp.sample_stride = tk.stride;
      fp.sample_n = tk.sample_n;
      fp.sample_splits = tk.sample_splits;
      fp.sample_max = (float*)(ws + tk.off_lists);
      fp.tau = (float*)(ws + tk.off_tau);
      fp.cand_n = (uint32_t*)(ws + tk.off_cand_n);
      fp.cand = ws + tk.off_lists;
      fp.kept = ws + tk.off_kept;
      fp.kept_pad = tk.kept_pad;
      fp.fail_rows = (uint32_t*)ws;
      fp.fail_block = (uint32_t*)(ws + tk.off_block);
      fp.fail_block_tok = tk.redo_tok;
      mark(0);
      if (dg::launch_topk_filter(fp, pl.e_dtype, s) != hipSuccess) return DG_ERR_LAUNCH;
      mark(1);
      mark(2);
      if (dg::launch_topk_list_select(fp, tk.k_most, pl.e_dtype, s) != hipSuccess) return DG_ERR_LAUNCH;
      tp.s_plane = (float*)(ws + tk.off_plane);
      tp.fail_rows = fp.fail_rows;
      for (uint32_t b = 0; b * tk.redo_tok < ntok; ++b) {
        tp.fail_block = fp.fail_block + b;
        const uint32_t at = b * tk.redo_tok;
        if (block(tok0 + at, std::min(tk.redo_tok, ntok - at), false) != hipSuccess) return DG_ERR_LAUNCH;
      }
    }
    mark(3);
    if (prof) g_prof.used += 2;
  }
  return DG_OK;
}

static void desc_from_reference(const dg_layer_offsets* L, const dg_attn_dims* dims, uint32_t kv_len,
                                dg_attn_desc* d) {
  std::memset(d, 0, sizeof(*d));
  d->canvas = dims->canvas;
  d->n_q_heads = dims->n_q_heads;
  d->n_kv_heads = L->n_kv_heads;
  d->head_dim = L->head_dim;
  d->kv_len = kv_len;
  d->causal_rows = dims->causal ? dims->canvas : 0u;
  d->window = dims->window;
  d->kv_ring_mask = L->kv_ring_mask;
  d->q_dtype = DG_BF16;
  d->kv_dtype = DG_F16;
  d->out_dtype = DG_BF16;
  d->flags = DG_ATTN_F_OUT_TRUNCATE;
  d->kv_region_bytes = L->kv_region;
  dg_attn_desc_reference_layout(d);
}

int dg_attention_state_bytes(const dg_layer_offsets* L, const dg_attn_dims* dims, uint32_t kv_len,
                             size_t* out_bytes) {
  if (!L || !dims || !out_bytes) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, kv_len, &d);
  return dg_attn_workspace_bytes(&d, out_bytes);
}

int dg_attention_dispatch(const void* q, const void* kvcache, void* out, const dg_layer_offsets* L,
                          const dg_step_params* P, const dg_attn_dims* dims, dg_debug_status* dbg,
                          void* attn_state, size_t attn_state_bytes, void* stream) {
  if (!L || !P || !dims) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, P->kv_len, &d);
  g_tls_dbg = (uint32_t*)dbg;
  const int rc = dg_attn_forward(&d, q, kvcache, out, nullptr, attn_state, attn_state_bytes, stream);
  g_tls_dbg = nullptr;
  return rc;
}

int dg_attention_dispatch_dev(const void* q, const void* kvcache, void* out, const dg_layer_offsets* L,
                              const dg_step_params* P_dev, uint32_t kv_len_max, const dg_attn_dims* dims,
                              dg_debug_status* dbg, void* attn_state, size_t attn_state_bytes, void* stream) {
  if (!L || !P_dev || !dims) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, kv_len_max, &d);
  g_tls_dbg = (uint32_t*)dbg;
  const int rc = dg_attn_forward_dev(&d, P_dev, q, kvcache, out, nullptr, attn_state, attn_state_bytes, stream);
  g_tls_dbg = nullptr;
  return rc;
}

int dg_attention_block_state_bytes(const dg_layer_offsets* L, const dg_attn_dims* dims, uint32_t kv_len,
                                   size_t* out_bytes) {
  if (!L || !dims || !out_bytes) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, kv_len, &d);
  size_t ws_full = 0;
  int rc = dg_attn_workspace_bytes(&d, &ws_full);
  if (rc != DG_OK) return rc;
  // The partial of a block [a, b) is split over workgroups like a whole call, and the number of splits a range resolves to
  // is not monotone in its length (ceil(n / ceil(n / s)) jumps up and down with n), so a shorter range can take more splits
  // than the whole one.  The partial workspace is sized for the most any range takes, with fp32 partial rows (a partial's
  // result is fp32 accumulators).  (`room` is reached within a few thousand tiles.)
  const dg_attn_desc pd = partial_desc(&d);
  Plan pl;
  const int cus = plan_cus();
  rc = make_plan(&pd, cus, &pl);
  if (rc != DG_OK) return rc;
  const uint32_t ntiles_full = std::max(1u, (pl.t_all + dg::kBlockN - 1) / dg::kBlockN);
  const uint32_t base = d.n_kv_heads * pl.n_mtiles, room = (uint32_t)cus / std::max(1u, base);
  uint32_t most = 1;
  for (uint32_t n = 1; n <= ntiles_full && most < std::min(room, kMaxSplits); ++n) {
    const uint32_t t = tiles_of_split(n, base, (uint32_t)cus, d.head_dim, false);
    most = std::max(most, (n + t - 1) / t);
  }
  size_t ws_part = 0;
  if (most > 1)
    ws_part = align_up((size_t)most * d.n_kv_heads * pl.rows_pad * d.head_dim * 4) +
              align_up((size_t)most * d.n_kv_heads * pl.rows_pad * 2 * 4);
  *out_bytes = 2 * align_up(state_bytes_of(&d)) + std::max(ws_full, ws_part);
  return DG_OK;
}

int dg_attention_dispatch_block(const void* q, const void* kvcache, void* out, const dg_layer_offsets* L,
                                const dg_step_params* P, const dg_attn_dims* dims, const dg_attn_block_range* blk,
                                dg_debug_status* dbg, void* attn_state, size_t attn_state_bytes, void* stream) {
  if (!L || !P || !dims || !blk) return DG_ERR_NULL;
  if (blk->is_first && blk->is_last)
    return dg_attention_dispatch(q, kvcache, out, L, P, dims, dbg, attn_state, attn_state_bytes, stream);
  if (!attn_state || ((uintptr_t)attn_state % 16) != 0) return DG_ERR_WORKSPACE;
  dg_attn_desc d;
  desc_from_reference(L, dims, P->kv_len, &d);
  const size_t sb = align_up(state_bytes_of(&d));
  if (attn_state_bytes < 2 * sb) return DG_ERR_WORKSPACE;
  char* const carried = (char*)attn_state;        // (m, l, acc) of the blocks so far
  char* const fresh = carried + sb;               // this block's own partial
  char* const ws = carried + 2 * sb;
  const size_t ws_bytes = attn_state_bytes - 2 * sb;
  // A block with no key for some rows (a causal row's range ends before it) leaves l = 0 there, and
  // the merge passes the carried state through, which is what the reference's early return does.
  int rc = dg_attn_partial(&d, blk->t_begin, blk->t_end, q, kvcache, blk->is_first ? carried : fresh, sb, ws, ws_bytes,
                           stream);
  if (rc != DG_OK || blk->is_first) return rc;
  const void* both[2] = {carried, fresh};
  if (!blk->is_last) return dg_attn_merge(&d, both, 2u, nullptr, nullptr, carried, stream);
  if (!out) return DG_ERR_NULL;
  g_tls_dbg = (uint32_t*)dbg;
  rc = dg_attn_merge(&d, both, 2u, out, nullptr, nullptr, stream);
  g_tls_dbg = nullptr;
  return rc;
}

int dg_attention_topk_state_bytes(const dg_layer_offsets* L, const dg_attn_dims* dims, uint32_t kv_len,
                                  const uint32_t* k_cfg, size_t* out_bytes) {
  if (!L || !dims || !out_bytes) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, kv_len, &d);
  return dg_attn_topk_workspace_bytes(&d, k_cfg, out_bytes);
}

int dg_attention_topk_dispatch(const void* q, const void* kvcache, void* out, const dg_layer_offsets* L,
                               const dg_step_params* P, const dg_attn_dims* dims, const uint32_t* k_cfg,
                               dg_debug_status* dbg, void* scratch, size_t scratch_bytes, void* stream) {
  if (!L || !P || !dims) return DG_ERR_NULL;
  dg_attn_desc d;
  desc_from_reference(L, dims, P->kv_len, &d);
  g_tls_dbg = (uint32_t*)dbg;
  const int rc = dg_attn_topk_forward(&d, k_cfg, q, kvcache, out, scratch, scratch_bytes, stream);
  g_tls_dbg = nullptr;
  return rc;
}

int dg_prof_begin(uint32_t max_launches) {
  if (g_prof.active) return DG_ERR_UNSUPPORTED;
  g_prof.ev.assign(2 * (size_t)max_launches, nullptr);
  for (auto& e : g_prof.ev)
    if (hipEventCreate(&e) != hipSuccess) return DG_ERR_LAUNCH;
  g_prof.used = 0;
  g_prof.active = true;
  return DG_OK;
}

int dg_prof_end_split(double* even_ms_total, double* odd_ms_total, uint32_t* n_pairs) {
  if (!g_prof.active) return DG_ERR_UNSUPPORTED;
  double total[2] = {0.0, 0.0};
  int rc = DG_OK;
  if (g_prof.used > 0 && hipEventSynchronize(g_prof.ev[2 * g_prof.used - 1]) != hipSuccess) rc = DG_ERR_LAUNCH;
  for (uint32_t i = 0; i < g_prof.used && rc == DG_OK; ++i) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, g_prof.ev[2 * i], g_prof.ev[2 * i + 1]) != hipSuccess) rc = DG_ERR_LAUNCH;
    total[i & 1u] += ms;
  }
  for (auto e : g_prof.ev)
    if (e) (void)hipEventDestroy(e);
  if (even_ms_total) *even_ms_total = total[0];
  if (odd_ms_total) *odd_ms_total = total[1];
  if (n_pairs) *n_pairs = g_prof.used;
  g_prof.ev.clear();
  g_prof.used = 0;
  g_prof.active = false;
  return rc;
}

int dg_prof_end(double* main_kernel_ms_total, uint32_t* n_launches) {
  double even = 0.0, odd = 0.0;
  const int rc = dg_prof_end_split(&even, &odd, n_launches);
  if (main_kernel_ms_total) *main_kernel_ms_total = even + odd;
  return rc;
}

int dg_calib_copy(void* dst, const void* src, size_t bytes, void* stream) {
  if (!dst || !src) return DG_ERR_NULL;
  if (bytes % 16 != 0 || ((uintptr_t)dst % 16) != 0 || ((uintptr_t)src % 16) != 0) return DG_ERR_LAYOUT;
  return dg::launch_calib_copy(dst, src, bytes, (hipStream_t)stream) == hipSuccess ? DG_OK : DG_ERR_LAUNCH;
}

int dg_calib_mfma(float* sink, size_t sink_bytes, uint32_t workgroups, uint32_t iters, uint32_t random_operands,
                  uint64_t* flops, void* stream) {
  if (!sink || !flops) return DG_ERR_NULL;
  if (random_operands > 3u) return DG_ERR_UNSUPPORTED;
  if (workgroups == 0 || iters == 0 || sink_bytes < (size_t)workgroups * 256 * sizeof(float)) return DG_ERR_WORKSPACE;
  // per workgroup: 4 waves x iters x 16 MFMAs x (32 x 32 x 16 multiply-adds)
  *flops = (uint64_t)workgroups * 4ull * iters * 16ull * (2ull * 32 * 32 * 16);
  return dg::launch_calib_mfma(sink, workgroups, iters, random_operands, (hipStream_t)stream) == hipSuccess
             ? DG_OK
             : DG_ERR_LAUNCH;
}

uint64_t dg_kv_row_bytes(uint32_t head_dim, uint32_t kv_dtype) { return (uint64_t)head_dim * elem_size(kv_dtype); }

uint64_t dg_kv_region_bytes(uint32_t n_kv_heads, uint32_t head_dim, uint64_t slots, uint32_t kv_dtype) {
  return slots * (uint64_t)n_kv_heads * 2ull * dg_kv_row_bytes(head_dim, kv_dtype);
}

uint64_t dg_kv_slot(uint32_t kv_ring_mask, uint64_t pos) { return kv_ring_mask ? (pos & kv_ring_mask) : pos; }

uint64_t dg_layer_kv_slots(int is_full, uint64_t max_seq, uint64_t ring_slots_cap) {
  if (is_full) return (max_seq + 8 + 7) / 8 * 8;
  uint64_t p2 = 1;
  while (p2 < max_seq) p2 <<= 1;
  return ring_slots_cap ? std::min(p2, ring_slots_cap) : p2;
}

}  // extern "C"
