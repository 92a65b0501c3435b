// Top-k sparse attention for gfx950 (MI355X): per (query row, head) only the k highest-scoring
// visible keys are kept, softmax is renormalised over them and their V rows are gathered
// (reference: src/shaders/attn/attention_topk/attention_topk.metal, CPU twin cpu.rs:41-120).
//
// Two kernels per pass over a block of canvas rows:
//   topk_scores_kernel  S = Q.K^T on MFMA, fp32, written to a score plane [Hq][rows][t_pad].  Same
//                       decomposition as the dense kernel (stacked GQA rows, K tiles by
//                       direct-to-LDS loads, Q resident in registers) without softmax or P.V,
//                       so key-range splits need no merge: every split writes its own columns.
//   topk_select_kernel  one workgroup per (row, head): exact top-k by fp32 score with a radix
//                       select on the order-preserving integer image of the scores (11 + 11 + 10
//                       bits).  Histogram levels run over the score row in memory only until the
//                       class that holds the k-th score fits an LDS candidate list (at most one
//                       level for model-sized rows, none for short ones); the remaining levels,
//                       the tie-break (equal scores: lower key position first, as the CPU twin)
//                       and the softmax run in LDS.  The kept keys are sorted by position, so the
//                       order of the P.V sum and with it every output bit is reproducible, then the
//                       V rows are gathered with one 16-byte load per lane and row (hd 512).
// The host walks the canvas in row blocks sized so that the score plane stays within the
// memory-side cache.
// Long rows at head_dim 512 take another way ("filtered path" below), without the plane.
#include "attn_params.h"
#include "mfma_tile.h"

namespace dg {
namespace {

constexpr int kCandCap = 2048;     // LDS candidate list of the select kernel (sized for 4 workgroups per CU)

// radix digits of the 32-bit key, most significant first: 11 + 11 + 10 bits
__device__ __forceinline__ uint32_t digit_shift(int level) { return level == 0 ? 21u : level == 1 ? 10u : 0u; }
__device__ __forceinline__ uint32_t digit_bits(int level) { return level == 2 ? 10u : 11u; }
constexpr int kMaxBins = 2048;

// ---------------------------------------------------------------------------------------------
// scores
// ---------------------------------------------------------------------------------------------

// wait until at most N vector-memory operations of this wave are outstanding, then the workgroup
// barrier, as one statement the compiler cannot move memory accesses across.  (A __syncthreads()
// would also wait for the score stores, and with them for every prefetched tile.)
template <int N>
__device__ __forceinline__ void wait_loads_then_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");
  constexpr int enc = 0x0F70 | (N & 15) | ((N >> 4) << 14);
  asm volatile("s_waitcnt %0\n\ts_barrier" ::"n"(enc) : "memory");
}

template <int D, bool F16>
__global__ void __launch_bounds__(256) topk_scores_kernel(const TopkParams tp) {
  const AttnParams& p = tp.a;
  if (tp.fail_block != nullptr && *tp.fail_block == 0u) return;   // no row of this block was left over
  using L = Lay<D>;
  constexpr int NSTEP = D / 16;
  constexpr int NLD = L::NLD;
  constexpr int PF = 3, NB = PF + 1;   // K tiles in flight ahead of the one being multiplied
  static_assert((PF - 1) * NLD < 64, "wait count");
  __shared__ __attribute__((aligned(1024))) char smem[NB * L::K_BYTES];

  // (KV head, split, row tile) units in 8 equal runs, one per XCD (ids go round-robin over them)
  const uint32_t n_units = p.hkv * tp.n_splits * tp.n_mtiles;
  const uint32_t per_xcd = (n_units + 7u) >> 3;
  const uint32_t wg = blockIdx.x;
  const uint32_t unit = (wg & 7u) * per_xcd + (wg >> 3);
  if (unit >= n_units) return;
  const uint32_t stream = fast_div(unit, tp.div_mtiles), mt = unit - stream * tp.n_mtiles;
  const uint32_t kvh = fast_div(stream, tp.div_splits), split = stream - kvh * tp.n_splits;

  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g2 = lane >> 5, l32 = lane & 31u;

  const uint32_t rows_total = tp.ntok * p.group;
  const uint32_t row0 = mt * kBlockM;
  const uint32_t r = row0 + wave * 32u + l32;
  const bool row_ok = r < rows_total;
  const uint32_t tok_l = row_ok ? fast_div(r, tp.div_group) : 0u;           // row within this pass
  const uint32_t tok = tp.tok0 + tok_l;
  const uint32_t qh = kvh * p.group + (row_ok ? r - tok_l * p.group : 0u);

  // key tiles some row of this row tile can see
  uint32_t lo_min, hi_max;
  {
    const uint32_t last_row = min(row0 + kBlockM, rows_total) - 1u;
    const uint32_t tok_a = tp.tok0 + fast_div(row0, tp.div_group), tok_b = tp.tok0 + fast_div(last_row, tp.div_group);
    const RowBounds ba = row_bounds(p, tok_a), bb = row_bounds(p, tok_b);
    lo_min = min(ba.lo, bb.lo);
    hi_max = max(ba.hi, bb.hi);
    if (tok_a < p.causal_rows && tok_b >= p.causal_rows) {
      const RowBounds bc = row_bounds(p, p.causal_rows - 1u), bd = row_bounds(p, p.causal_rows);
      lo_min = min(lo_min, min(bc.lo, bd.lo));
      hi_max = max(hi_max, max(bc.hi, bd.hi));
    }
    if (tok_a < p.causal_rows && p.extra_lo < p.t_all) hi_max = p.t_all;
    lo_min = __builtin_amdgcn_readfirstlane(lo_min);
    hi_max = __builtin_amdgcn_readfirstlane(hi_max);
  }
  const uint32_t mt_begin = max(lo_min / kBlockN, tp.tile_first);
  const uint32_t mt_end = max(min((hi_max + kBlockN - 1) / kBlockN, tp.tile_end), mt_begin);
  const uint32_t per_split = (mt_end - mt_begin + tp.n_splits - 1u) / tp.n_splits;
  const uint32_t tb = __builtin_amdgcn_readfirstlane(min(mt_begin + split * per_split, mt_end));
  const uint32_t te = __builtin_amdgcn_readfirstlane(min(tb + per_split, mt_end));
  if (te <= tb) return;

  // Q fragments: lane = row, 8 consecutive d per step
  u32x4 qf[NSTEP];
  const bool convert = F16 && p.q_is_bf16;
  auto to_frag = [&](u32x4 raw) -> u32x4 {
    if (convert) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        raw[e] = pack2<true>(__uint_as_float(raw[e] << 16), __uint_as_float(raw[e] & 0xffff0000u));
    }
    return raw;
  };
  if constexpr (D == 512) {   // through the K buffers' LDS
    static_assert(4 * 32 * kQRowLds <= NB * L::K_BYTES, "the tile buffers hold the query rows");
    lds_char* const qb = (lds_char*)smem + wave * (32u * kQRowLds);
    issue_q_rows((const char*)p.q + ((size_t)tp.tok0 * p.hq + kvh * p.group) * (2 * D), row0 + wave * 32u, rows_total, p.group,
                 (uint32_t)(size_t)qb, lane,
                 [&](uint32_t rq) { return (rq + fast_div(rq, tp.div_group) * (p.hq - p.group)) * (uint32_t)(2 * D); });
    wait_vmem_all();
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) qf[st] = *(lds_u32x4*)(qb + l32 * kQRowLds + g2 * 16u + 32 * st);
    __syncthreads();   // the first tiles may take the rows' place (converted behind their loads, below)
  } else {
    const size_t qoff = ((size_t)tok * p.hq + qh) * D + 8u * g2;
    const uint16_t* qp = (const uint16_t*)p.q + qoff;
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) qf[st] = to_frag(row_ok ? *(const u32x4*)(qp + 16 * st) : u32x4{0, 0, 0, 0});
  }

  const char* kbase = (const char*)p.k + (int64_t)kvh * p.k_head_stride * 2;
  const int64_t kstride_b = p.k_tok_stride * 2;
  const uint32_t k_lane_off = l32 * L::K_STRIDE + (L::PAD ? g2 * 16u : 0u);
  const uint32_t k_swz = L::swz_k(l32);
  const uint32_t t_last = (te - 1u) * kBlockN;
  // loads for a tile past the last one fetch the last tile again into a buffer nobody reads, so
  // that every iteration issues the same number of loads and the wait counts stay fixed
  auto k_desc = [&](uint32_t j) {
    lds_char* buf = (lds_char*)(smem + ((j - tb) % NB) * L::K_BYTES);
    return make_tile_load<D, false, false>(kbase, kstride_b, min(j * kBlockN, t_last), 0u, p.t_all, p.ring_mask, buf,
                                           wave, lane);
  };
  auto issue_k = [&](uint32_t j) { issue_tile<D, false>(k_desc(j), wave, lane); };
  // The product is taken as S = Q.K^T (A = Q, B = K): the output lane is then the key and
  // register e of the block is query row 8 (e >> 2) + 4 g2 + (e & 3) of this wave's 32, so one
  // store instruction writes 32 consecutive keys of two rows: whole 128-byte lines.  (With the
  // operands the other way round every store scatters 32-byte pieces over 32 rows and the
  // kernel is bound by the write path.)  Where each of the 16 rows lives, and whether it exists:
  uint32_t row_off[16];      // byte offset of this lane's key column in the row, in the first key tile
  uint32_t row_mask = 0;
  const bool full_tile = row0 + kBlockM <= rows_total;      // (the same in every lane)
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const uint32_t rr = row0 + wave * 32u + 8u * (e >> 2) + 4u * g2 + (e & 3);
    const bool ok = rr < rows_total;
    const uint32_t tl = ok ? fast_div(rr, tp.div_group) : 0u;
    const uint32_t hh = kvh * p.group + (ok ? rr - tl * p.group : 0u);
    row_off[e] = ((hh * tp.ntok + tl) * tp.t_pad + l32) * 4u;
    row_mask |= ok ? 1u << e : 0u;
  }
#pragma unroll
  for (int i = 0; i < PF; ++i) issue_k(tb + i);
  if constexpr (D == 512) {
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) qf[st] = to_frag(qf[st]);
  }
  // lane l32 holds key t0 + l32 of sixteen rows; element e of a tile's scores goes to
  // (uniform tile base) + (per-lane 32-bit offset)
  auto store_elem = [&](auto e_c, const f32x16& sc, uint32_t tile) {
    constexpr int e = decltype(e_c)::value;
    char* const base = (char*)tp.s_plane + (size_t)tile * (kBlockN * sizeof(float));
    if (full_tile || (row_mask & (1u << e))) *(float*)(base + row_off[e]) = sc[e] * tp.scale;
  };
  auto store_tile = [&](const f32x16& sc, uint32_t tile) {
    static_for<0, 16>([&](auto e_c) { store_elem(e_c, sc, tile); });
  };
  f32x16 s_prev;
#pragma unroll
  for (int e = 0; e < 16; ++e) s_prev[e] = 0.f;
  for (uint32_t j = tb; j < te; ++j) {
    // this wave's loads of K(j) have landed (the PF-1 tiles behind it may still be in flight);
    // after the barrier everybody's have, and everybody is done reading K(j-1), whose buffer
    // takes K(j+PF).  The scores of tile j-1 are stored only now, a tile late, between the
    // first half of this tile's MFMAs: stores count in the same counter as the loads, and issued
    // right before the wait they would have to drain first; issued here they are at least half
    // a tile old at the next wait, and their address arithmetic hides behind the matrix pipe.
    wait_loads_then_barrier<(PF - 1) * NLD>();
    const bool have_prev = j > tb;
    // (the loads of K(j+PF) are issued between the MFMAs below: back to back each of them holds
    // the wave's issue slot for about two MFMAs' worth of cycles)
    const TileLoad tl_next = k_desc(j + PF);
    lds_char* const kb = (lds_char*)(smem + ((j - tb) % NB) * L::K_BYTES);
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
    // K fragments in chunks of CH: the reads of chunk c+1 are issued before the MFMAs of chunk c
    // (left to itself the compiler reads two fragments, waits, multiplies, and the LDS latency
    // is paid sixteen times per tile)
    constexpr int CH = NSTEP < 8 ? NSTEP : 8;
    constexpr int NCHUNK = NSTEP / CH;
    constexpr int LPC = (NLD + NCHUNK - 1) / NCHUNK;      // tile loads issued per chunk
    constexpr int LGAP = CH / LPC;                         // MFMAs between two of them
    static_assert(LPC * NCHUNK >= NLD && LPC <= CH, "tile loads must fit between the MFMAs");
    constexpr int SHALF = NSTEP / 2 > 0 ? NSTEP / 2 : 1;   // MFMAs that carry stores of the previous tile
    constexpr int SPM = (16 + SHALF - 1) / SHALF;          // stores behind each of them
    u32x4 fr[2][CH];
    auto read_chunk = [&](int c, u32x4 (&dst)[CH]) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int st = c * CH + i;
        if constexpr (L::PAD) {
          dst[i] = *(lds_u32x4*)(kb + k_lane_off + 32 * st);
        } else {
          const uint32_t cc = (uint32_t)(2 * st) + g2;
          dst[i] = *(lds_u32x4*)(kb + k_lane_off + ((cc ^ k_swz) << 4));
        }
      }
    };
    read_chunk(0, fr[0]);
    static_for<0, NCHUNK>([&](auto c_c) {
      constexpr int c = decltype(c_c)::value;
      if constexpr (c + 1 < NCHUNK) read_chunk(c + 1, fr[(c + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, CH>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        s = mfma16<F16>(qf[c * CH + i], fr[c & 1][i], s);
        if constexpr (i % LGAP == LGAP / 2 && c * LPC + i / LGAP < NLD) {
          issue_tile_part<D, false, c * LPC + i / LGAP>(tl_next, wave, lane);
          __builtin_amdgcn_sched_barrier(0);
        }
        constexpr int m = c * CH + i;                 // MFMA index within the tile
        if constexpr (m < SHALF) {
          if (have_prev) static_for<m * SPM, (m + 1) * SPM < 16 ? (m + 1) * SPM : 16>([&](auto e_c) { store_elem(e_c, s_prev, j - 1u); });
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    s_prev = s;
  }
  store_tile(s_prev, te - 1u);
  wait_vmem_all();   // no direct-to-LDS load may outlive the workgroup's LDS
}

// ---------------------------------------------------------------------------------------------
// select + softmax + gathered P.V
// ---------------------------------------------------------------------------------------------

// order-preserving integer image of a score (larger float <-> larger key); NaN sorts lowest
__device__ __forceinline__ uint32_t score_key(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0u;
  return (u & 0x80000000u) ? ~u : (u ^ 0x80000000u);
}

// the score a key stands for (inverse of score_key for every non-NaN score)
__device__ __forceinline__ float key_score(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

// number of keys row bounds b let through
__device__ __forceinline__ uint32_t visible_count(const RowBounds& b, uint32_t t_all) {
  const uint32_t hi = min(b.hi, t_all);
  const uint32_t len_a = hi > b.lo ? hi - b.lo : 0u;
  if (b.extra >= t_all) return len_a;
  if (len_a == 0u) return t_all - b.extra;
  if (b.extra <= b.lo) return t_all - b.extra;
  if (b.extra < hi) return t_all - b.lo;
  return len_a + (t_all - b.extra);
}

// keys kept for a row (attention_topk.metal:160-182)
__device__ __forceinline__ uint32_t row_k(const TopkParams& tp, uint32_t tok, uint32_t n_valid) {
  uint32_t k_req;
  if (tp.k_cfg[1] != 0u) {
    const uint32_t gran = max(tp.k_cfg[0], 1u);
    const uint32_t t_equiv = tok < tp.a.causal_rows ? ((n_valid + gran - 1u) / gran) * gran : n_valid;
    k_req = min(max(t_equiv / tp.k_cfg[1], tp.k_cfg[2]), tp.k_cfg[3]);
  } else {
    k_req = max(tp.k_cfg[0], 1u);
  }
  return min(min(k_req, n_valid), (uint32_t)kTopkMaxK);
}

struct SelectShared {
  uint32_t hist[kMaxBins];
  uint32_t tot[256];
  uint32_t res[4];              // chosen bin, entries above it, entries in it
  uint32_t n_sel, n_cand, pad0, pad1;
  uint32_t cand_key[kCandCap];
  uint32_t cand_t[kCandCap];
  float sel_s[kTopkMaxK];
  uint32_t sel_t[kTopkMaxK];
};

// From hist[0 .. nbins): the bin that holds the `remaining`-th largest entry, counting from the
// top bin down.  Leaves {bin, entries in higher bins, entries in the bin} in sh.res.  All 256
// threads call it; it contains barriers.
__device__ __forceinline__ void pick_bin(SelectShared& sh, uint32_t nbins, uint32_t remaining, uint32_t tid) {
  const uint32_t per = nbins >> 8;          // bins per thread: 8 or 4
  const uint32_t lane = tid & 63u, wave = tid >> 6;
  uint32_t c[8];
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) {
    c[i] = i < per ? sh.hist[tid * per + i] : 0u;
    sum += c[i];
  }
  // entries in the bins of higher threads: suffix sum over the lanes of the wave, then the
  // totals of the higher waves
  uint32_t incl = sum;
#pragma unroll
  for (uint32_t off = 1; off < 64u; off <<= 1) {
    const uint32_t v = __shfl_down(incl, off, 64);
    if (lane + off < 64u) incl += v;
  }
  if (lane == 0) sh.tot[wave] = incl;
  __syncthreads();
  uint32_t above = incl - sum;
  for (uint32_t w = wave + 1; w < 4u; ++w) above += sh.tot[w];
  if (above < remaining && remaining <= above + sum) {
    uint32_t run = above;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      if ((uint32_t)i < per) {
        if (run < remaining && remaining <= run + c[i]) {
          sh.res[0] = tid * per + (uint32_t)i;
          sh.res[1] = run;
          sh.res[2] = c[i];
        }
        run += c[i];
      }
    }
  }
  __syncthreads();
}

// One more in `bin`, in a pass over a whole score row.  The lanes that agree with the first one add once, together: such passes
// are what rows with thousands of equal scores come to, and there every atomic would wait for the one before it.  Attention call,
// every row of equal scores, over 33k keys: 256 rows 1947 -> 1044 us, 64 rows 489 -> 253.  (Not in the passes over a few
// thousand sampled keys or candidates: 64 ordinary rows over 3k to 9k keys 49 -> 50, 59.6 -> 61.0.)
__device__ __forceinline__ void hist_add(uint32_t* hist, uint32_t bin) {
  const uint32_t b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)bin);
  const uint64_t same = __builtin_amdgcn_ballot_w64(bin == b0);
  if (bin != b0) atomicAdd(&hist[bin], 1u);
  else if (__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u)) == 0u)
    atomicAdd(&hist[b0], (uint32_t)__builtin_popcountll(same));
}

// The `need`-th largest of the keys key_of(i) yields for i in [0, n) (key_of returns false for
// entries that do not take part), by three histogram levels over LDS.  Returns the key; *n_equal
// = entries equal to it, *take_equal = how many of those belong to the `need` largest.  All 256
// threads call it with the same arguments; needs 1 <= need <= number of participating entries.
template <typename KeyOf>
__device__ __forceinline__ uint32_t lds_kth_largest(SelectShared& sh, uint32_t n, uint32_t need, uint32_t tid,
                                                    KeyOf&& key_of, uint32_t* take_equal, uint32_t* n_equal) {
  uint32_t prefix = 0, pbits = 0, remaining = need, cls = 0;
  for (int lv = 0; lv < 3; ++lv) {
    const uint32_t nbins = 1u << digit_bits(lv);
    for (uint32_t b = tid; b < nbins; b += 256u) sh.hist[b] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += 256u) {
      uint32_t key;
      if (key_of(i, key) && (pbits == 0u || (key >> (32u - pbits)) == prefix))
        atomicAdd(&sh.hist[(key >> digit_shift(lv)) & (nbins - 1u)], 1u);
    }
    __syncthreads();
    pick_bin(sh, nbins, remaining, tid);
    remaining -= sh.res[1];
    prefix = (prefix << digit_bits(lv)) | sh.res[0];
    pbits += digit_bits(lv);
    cls = sh.res[2];
    __syncthreads();
  }
  *take_equal = remaining;
  *n_equal = cls;
  return prefix;
}

template <int D, bool F16>
__global__ void __launch_bounds__(256) topk_select_kernel(const TopkParams tp) {
  const AttnParams& p = tp.a;
  __shared__ SelectShared sh;
  static_assert(4 * D * sizeof(float) <= sizeof(sh.cand_key), "the P.V partial sums reuse the candidate list");
  float (*const red)[D] = (float (*)[D])sh.cand_key;
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u, wave = tid >> 6;
  const uint32_t tok_l = blockIdx.x, qh = blockIdx.y;
  const uint32_t tok = tp.tok0 + tok_l;
  if (tp.fail_rows != nullptr && tp.fail_rows[(size_t)tok * p.hq + qh] == 0u) return;   // done by the filtered path
  const uint32_t kvh = qh / p.group;
  const RowBounds rb = row_bounds(p, tok);
  const uint32_t n_valid = visible_count(rb, p.t_all);

  const uint32_t k = row_k(tp, tok, n_valid);

  const size_t out_off = ((size_t)tok * p.hq + qh) * D;
  if (k == 0u) {   // a row that sees no key stores zeros, like the dense path
    for (uint32_t d = tid; d < (uint32_t)D; d += 256u) {
      if (p.out_dtype == 2u) ((float*)p.out)[out_off + d] = 0.f;
      else ((uint16_t*)p.out)[out_off + d] = 0;
    }
    return;
  }

  const float* srow = tp.s_plane + ((size_t)qh * tp.ntok + tok_l) * tp.t_pad;
  // positions to scan: the hull of the visible set, widened to whole float4s
  const uint32_t hull_lo = (rb.extra < p.t_all ? min(rb.lo, rb.extra) : rb.lo) & ~3u;
  const uint32_t hull_hi = rb.extra < p.t_all ? p.t_all : min(rb.hi, p.t_all);

  // f(position, score) for every visible key of the row; each thread takes one float4 out of
  // every 256 and has four of them in flight.  The plane is read once: non-temporal loads (here and
  // for the sample above), so that 135 MB of scores per block do not push the V rows, which every
  // row of a KV group gathers from, out of the L2s (whole call 0.715 -> 0.664 ms)
  auto scan_row = [&](auto&& f) {
    for (uint32_t t4 = hull_lo + 4u * tid; t4 < hull_hi; t4 += 4096u) {
      f32x4 v[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t a = t4 + 1024u * u;
        v[u] = a < hull_hi ? __builtin_nontemporal_load((const f32x4*)(srow + a)) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
          const uint32_t t = t4 + 1024u * u + i;
          if (t < hull_hi && key_visible(rb, t, p.t_all)) f(t, v[u][i]);
        }
      }
    }
  };
  if (tid == 0) {
    sh.n_sel = 0;
    sh.n_cand = 0;
    sh.res[0] = sh.res[1] = sh.res[2] = 0;
  }
  __syncthreads();   // (a short row's scan counts into the lists at once: a late wave 0 would reset what another has counted)

  uint32_t prefix = 0, pbits = 0, remaining = k, class_count = n_valid;
  int level = 0;
  bool have_cand = false;   // the candidate list already holds every key at or above a sampled threshold

  // ---- long rows: cut at a threshold taken from a sample, so that the row is read once ----
  // About 2048 keys at an even stride give the key tau below which ~2.5 k keys are expected;
  // one pass collects everything >= tau.  If that is at least k and fits the list, the exact
  // k-th key is found in LDS; otherwise (an unlucky or clustered sample) the exact histogram
  // levels below run instead.
  if (n_valid > (uint32_t)kCandCap) {
    const uint32_t stride = max(1u, (hull_hi - hull_lo + 2047u) / 2048u);
    const uint32_t m = (hull_hi - hull_lo + stride - 1u) / stride;     // sample slots, at most 2048
    {
      float sv[8];
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) {      // m <= 2048: eight samples per thread, all in flight
        const uint32_t i = tid + 256u * u;
        sv[u] = i < m ? __builtin_nontemporal_load(srow + hull_lo + i * stride) : 0.f;
      }
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) {
        const uint32_t i = tid + 256u * u;
        // (an invisible position takes part as the lowest key, which cannot reach the top ranks asked for)
        if (i < m) sh.cand_key[i] = key_visible(rb, hull_lo + i * stride, p.t_all) ? score_key(sv[u]) : 0u;
      }
    }
    __syncthreads();
    if (m > 0u) {
      // aim at ~2.5 k keys at or above tau, but never beyond 3/4 of the list
      const uint64_t want = min<uint64_t>(5ull * k / 2ull, 3ull * kCandCap / 4ull);
      const uint32_t r = min(m, (uint32_t)((want * m + n_valid - 1ull) / n_valid) + 8u);
      uint32_t te, ne;
      const uint32_t tau = lds_kth_largest(
          sh, m, r, tid, [&](uint32_t i, uint32_t& key) { key = sh.cand_key[i]; return true; }, &te, &ne);
      scan_row([&](uint32_t t, float sv) {
        const uint32_t key = score_key(sv);
        if (key >= tau) {
          const uint32_t slot = atomicAdd(&sh.n_cand, 1u);
          if (slot < (uint32_t)kCandCap) {
            sh.cand_key[slot] = key;
            sh.cand_t[slot] = t;
          }
        }
      });
      __syncthreads();
      const uint32_t got = sh.n_cand;
      have_cand = got >= k && got <= (uint32_t)kCandCap;
      if (have_cand) class_count = got;
      __syncthreads();
      if (!have_cand && tid == 0) sh.n_cand = 0;
    }
    __syncthreads();
  }

  // ---- exact levels over the score row in memory, until the class of the k-th score fits the list ----
  for (; !have_cand && level < 3 && class_count > (uint32_t)kCandCap; ++level) {
    const uint32_t nbins = 1u << digit_bits(level);
    for (uint32_t b = tid; b < nbins; b += 256u) sh.hist[b] = 0;
    __syncthreads();
    scan_row([&](uint32_t, float sv) {
      const uint32_t key = score_key(sv);
      if (pbits == 0u || (key >> (32u - pbits)) == prefix)
        hist_add(sh.hist, (key >> digit_shift(level)) & (nbins - 1u));
    });
    __syncthreads();
    pick_bin(sh, nbins, remaining, tid);
    remaining -= sh.res[1];
    prefix = (prefix << digit_bits(level)) | sh.res[0];
    pbits += digit_bits(level);
    class_count = sh.res[2];
    __syncthreads();
  }
  if (class_count > (uint32_t)kCandCap) {
    // More than a list's worth of bit-identical scores at the threshold (a degenerate row, e.g.
    // an all-zero query).  Keys above go in as they come; of the ties the first `remaining` by
    // position are taken by one wave walking the row in order.
    scan_row([&](uint32_t t, float sv) {
      if (score_key(sv) > prefix) {
        const uint32_t slot = atomicAdd(&sh.n_sel, 1u);
        if (slot < (uint32_t)kTopkMaxK) {
          sh.sel_s[slot] = sv;
          sh.sel_t[slot] = t;
        }
      }
    });
    __syncthreads();
    if (wave == 0) {
      const uint32_t first = k - remaining;
      uint32_t taken = 0;
      for (uint32_t t0 = hull_lo; t0 < hull_hi && taken < remaining; t0 += 64u) {
        const uint32_t t = t0 + lane;
        float sv = 0.f;
        bool tie = false;
        if (t < hull_hi && key_visible(rb, t, p.t_all)) {
          sv = srow[t];
          tie = score_key(sv) == prefix;
        }
        const unsigned long long m = __builtin_amdgcn_ballot_w64(tie);
        const uint32_t rank = taken + __builtin_popcountll(m & ((1ull << lane) - 1ull));
        if (tie && rank < remaining && first + rank < (uint32_t)kTopkMaxK) {
          sh.sel_s[first + rank] = sv;
          sh.sel_t[first + rank] = t;
        }
        taken += __builtin_popcountll(m);
      }
    }
    __syncthreads();
  } else {
    if (!have_cand) {
      // ---- one pass: keys above the class go straight to the kept list, the class to the candidates ----
      scan_row([&](uint32_t t, float sv) {
        const uint32_t key = score_key(sv);
        const uint32_t hi = pbits ? key >> (32u - pbits) : 0u;
        if (hi > prefix) {
          const uint32_t slot = atomicAdd(&sh.n_sel, 1u);
          if (slot < (uint32_t)kTopkMaxK) {
            sh.sel_s[slot] = sv;
            sh.sel_t[slot] = t;
          }
        } else if (hi == prefix) {
          const uint32_t slot = atomicAdd(&sh.n_cand, 1u);
          if (slot < (uint32_t)kCandCap) {
            sh.cand_key[slot] = key;
            sh.cand_t[slot] = t;
          }
        }
      });
      __syncthreads();
    }
    const uint32_t n_cand = min(sh.n_cand, (uint32_t)kCandCap);

    // ---- the k-th key among the candidates: the levels not yet done, over the list ----
    uint32_t thr = prefix, take_eq = remaining, n_eq = class_count;
    if (level < 3) {
      // (the list holds exactly the keys whose leading pbits bits equal prefix: rebuild the full
      // key of the threshold from the remaining levels)
      uint32_t lp = prefix, lb = pbits, rem = remaining, cls = class_count;
      for (int lv = level; lv < 3; ++lv) {
        const uint32_t nbins = 1u << digit_bits(lv);
        for (uint32_t b = tid; b < nbins; b += 256u) sh.hist[b] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n_cand; i += 256u) {
          const uint32_t key = sh.cand_key[i];
          if (lb == 0u || (key >> (32u - lb)) == lp) atomicAdd(&sh.hist[(key >> digit_shift(lv)) & (nbins - 1u)], 1u);
        }
        __syncthreads();
        pick_bin(sh, nbins, rem, tid);
        rem -= sh.res[1];
        lp = (lp << digit_bits(lv)) | sh.res[0];
        lb += digit_bits(lv);
        cls = sh.res[2];
        __syncthreads();
      }
      thr = lp;
      take_eq = rem;
      n_eq = cls;
    }
    // thr is the k-th largest key; take_eq of the n_eq keys equal to it are kept

    // ---- equal scores: the lower positions win.  Threshold on position by the same select ----
    uint32_t t_key_min = 0u;   // ties with ~t >= t_key_min are kept
    if (n_eq > take_eq) {
      uint32_t te, ne;
      t_key_min = lds_kth_largest(
          sh, n_cand, take_eq, tid,
          [&](uint32_t i, uint32_t& key) {
            key = ~sh.cand_t[i];
            return sh.cand_key[i] == thr;
          },
          &te, &ne);
    }
    for (uint32_t i = tid; i < n_cand; i += 256u) {
      const uint32_t key = sh.cand_key[i];
      const uint32_t t = sh.cand_t[i];
      if (key > thr || (key == thr && ~t >= t_key_min)) {
        const uint32_t slot = atomicAdd(&sh.n_sel, 1u);
        if (slot < (uint32_t)kTopkMaxK) {
          sh.sel_s[slot] = key_score(key);
          sh.sel_t[slot] = t;
        }
      }
    }
    __syncthreads();
  }
  // ---- sort the kept keys by position (bitonic, padded with +inf positions) ----
  uint32_t npow = 1;
  while (npow < k) npow <<= 1;
  for (uint32_t i = k + tid; i < npow; i += 256u) {
    sh.sel_t[i] = 0xffffffffu;
    sh.sel_s[i] = -INFINITY;
  }
  __syncthreads();
  for (uint32_t size = 2; size <= npow; size <<= 1) {
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t i = tid; i < (npow >> 1); i += 256u) {
        const uint32_t lo = 2u * i - (i & (stride - 1u));
        const uint32_t hi = lo + stride;
        const bool up = (lo & size) == 0u;
        const uint32_t a = sh.sel_t[lo], b = sh.sel_t[hi];
        if ((a > b) == up) {
          sh.sel_t[lo] = b;
          sh.sel_t[hi] = a;
          const float fa = sh.sel_s[lo];
          sh.sel_s[lo] = sh.sel_s[hi];
          sh.sel_s[hi] = fa;
        }
      }
      __syncthreads();
    }
  }
  // ---- softmax over the kept scores (cpu.rs:95-104) ----
  float* const fred = (float*)sh.hist;   // histogram storage is free now
  float m = -INFINITY;
  for (uint32_t j = tid; j < k; j += 256u) m = fmaxf(m, sh.sel_s[j]);
  fred[tid] = m;
  __syncthreads();
  for (uint32_t w = 128; w > 0; w >>= 1) {
    if (tid < w) fred[tid] = fmaxf(fred[tid], fred[tid + w]);
    __syncthreads();
  }
  const float mmax = fred[0];
  __syncthreads();
  float l = 0.f;
  for (uint32_t j = tid; j < k; j += 256u) {
    const float e = expf(sh.sel_s[j] - mmax);
    sh.sel_s[j] = e;
    l += e;
  }
  fred[tid] = l;
  __syncthreads();
  for (uint32_t w = 128; w > 0; w >>= 1) {
    if (tid < w) fred[tid] += fred[tid + w];
    __syncthreads();
  }
  const float lsum = fred[0];
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  // ---- gathered P.V: wave w takes kept keys w, w+4, ...; a lane owns PER consecutive d ----
  constexpr int PER = D >= 64 ? D / 64 : 1;
  const bool lane_on = lane * PER < (uint32_t)D;
  float acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.f;
  const char* vbase = (const char*)p.v + (int64_t)kvh * p.v_head_stride * 2 + (size_t)lane * PER * 2;
  const int64_t vstride_b = p.v_tok_stride * 2;
  // kept keys in groups of GU per wave (wave w takes groups w, w+4, ...): the GU row loads of a
  // group are issued before any of them is used, so a row's latency is paid once per group
  constexpr int GU = 8;
  auto load_row = [&](const uint16_t* vp, uint16_t (&raw)[PER]) {
    if constexpr (PER == 8) {
      const u32x4 x = *(const u32x4*)vp;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        raw[2 * i] = (uint16_t)(x[i] & 0xffffu);
        raw[2 * i + 1] = (uint16_t)(x[i] >> 16);
      }
    } else if constexpr (PER == 4) {
      const u32x2 x = *(const u32x2*)vp;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        raw[2 * i] = (uint16_t)(x[i] & 0xffffu);
        raw[2 * i + 1] = (uint16_t)(x[i] >> 16);
      }
    } else if constexpr (PER == 2) {
      const uint32_t x = *(const uint32_t*)vp;
      raw[0] = (uint16_t)(x & 0xffffu);
      raw[1] = (uint16_t)(x >> 16);
    } else {
      raw[0] = *vp;
    }
  };
  for (uint32_t j0 = wave * GU; j0 < k; j0 += 4u * GU) {
    float pj[GU];
    uint16_t raw[GU][PER];
#pragma unroll
    for (int u = 0; u < GU; ++u) {
      const uint32_t j = min(j0 + (uint32_t)u, k - 1u);          // past the end: the last key again, weight 0
      pj[u] = j0 + (uint32_t)u < k ? sh.sel_s[j] * inv : 0.f;
      const uint32_t tj = min(sh.sel_t[j], p.t_all - 1u);       // (kept positions are < t_all by construction)
      const uint16_t* vp = (const uint16_t*)(vbase + (int64_t)kv_slot(p.ring_mask, tj) * vstride_b);
      if (lane_on) load_row(vp, raw[u]);
    }
    if (lane_on) {
#pragma unroll
      for (int u = 0; u < GU; ++u) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const float v = F16 ? (float)__builtin_bit_cast(_Float16, raw[u][i]) : bf16_bits_to_f32(raw[u][i]);
          acc[i] = __builtin_fmaf(pj[u], v, acc[i]);
        }
      }
    }
  }
  if (lane_on) {
#pragma unroll
    for (int i = 0; i < PER; ++i) red[wave][lane * PER + i] = acc[i];
  }
  __syncthreads();
  for (uint32_t d = tid; d < (uint32_t)D; d += 256u) {
    const float o = ((red[0][d] + red[1][d]) + red[2][d]) + red[3][d];
    if (p.out_dtype == 2u) ((float*)p.out)[out_off + d] = o;
    else ((uint16_t*)p.out)[out_off + d] = f32_to_bf16_bits(o, p.out_trunc != 0u);
  }
}

// ---------------------------------------------------------------------------------------------
// filtered path: long rows at head_dim 512 without a score plane
// ---------------------------------------------------------------------------------------------
//
// A call of the general path writes every score (541 MB for 256 rows over 33k keys) and reads it back to keep one key
// in 128.  Here a row's threshold tau is guessed first, from the scores of every 17th key; the score kernel then
// stores only scores at or above tau, as (score, position) entries in lists, and the select kernel works on a list of
// two to four times k entries that one wave holds in registers.  Whatever tau is, the result is exact: a row whose
// list holds fewer than k entries, or more than fit, is marked, and the general path redoes the marked rows (its
// launches end at once where no row of the block is marked, 1.5 us each).
// 256 rows x 16 heads over 33024 keys, layer step: 646 -> 249 us.  Launches: sampled scores 15 us (was: scores and plane, 4 x 55),
// thresholds 6, filter 126 to 133 by box (1.0 - 1.1 PFLOP/s; the products alone, with their LDS reads and nothing else, 101), selection 24
// and gathered P.V 51 (both: was 4 x 94).

// scores through an ordinary-register accumulator, query fragment in accumulation registers (256 of them hold the 64
// query rows of a wave; a comparison cannot read that file)
template <bool F16, bool FIRST>
__device__ __forceinline__ void mfma_filter(f32x16& s, const u32x4& k, const u32x4& q) {
  if constexpr (FIRST) {
    if constexpr (F16) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
  } else {
    if constexpr (F16) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
  }
}
// the last product of both row blocks and the wait states a non-MFMA read of the scores needs, in one statement
template <bool F16>
__device__ __forceinline__ void mfma_filter_last(f32x16& s0, f32x16& s1, const u32x4& k, const u32x4& q0, const u32x4& q1) {
  if constexpr (F16)
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %2, %3, %0\n\tv_mfma_f32_32x32x16_f16 %1, %2, %4, %1\n\ts_nop 11"
                 : "+v"(s0), "+v"(s1) : "v"(k), "a"(q0), "a"(q1));
  else
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %2, %3, %0\n\tv_mfma_f32_32x32x16_bf16 %1, %2, %4, %1\n\ts_nop 11"
                 : "+v"(s0), "+v"(s1) : "v"(k), "a"(q0), "a"(q1));
}
template <bool F16>
__device__ __forceinline__ void mfma_filter_last(f32x16& s0, const u32x4& k, const u32x4& q0) {
  if constexpr (F16) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\ts_nop 11" : "+v"(s0) : "v"(k), "a"(q0));
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\ts_nop 11" : "+v"(s0) : "v"(k), "a"(q0));
}
// Four stores of the filter kernel, each by the lanes in its mask and by lane 0.
__device__ __forceinline__ void store4_masked(const uint64_t (&m)[4], const uint32_t (&at)[4], u32x2 e0, u32x2 e1, u32x2 e2,
                                              u32x2 e3, char* base) {
  asm volatile(
      "s_or_b64 exec, %0, 1\n\tglobal_store_dwordx2 %4, %8, %12\n\t"
      "s_or_b64 exec, %1, 1\n\tglobal_store_dwordx2 %5, %9, %12\n\t"
      "s_or_b64 exec, %2, 1\n\tglobal_store_dwordx2 %6, %10, %12\n\t"
      "s_or_b64 exec, %3, 1\n\tglobal_store_dwordx2 %7, %11, %12\n\t"
      "s_mov_b64 exec, -1" ::"s"(m[0]), "s"(m[1]), "s"(m[2]), "s"(m[3]), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]),
      "v"(e0), "v"(e1), "v"(e2), "v"(e3), "s"(base)
      : "memory", "scc");
}

// Reductions and scans over the wave by DPP moves (through LDS, as a shuffle, each step is a round trip of its own).
// step(x, v): x with v = the value of the lane 1, 2, 4, 8, then of the last lane of the row or half below; ends in lane 63
template <typename T, typename F>
__device__ __forceinline__ T wave_scan(T x, T none, F step) {
  auto moved = [&](auto ctrl_c, auto rows_c) -> T {
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, none), __builtin_bit_cast(int, x),
                                                             decltype(ctrl_c)::value, decltype(rows_c)::value, 0xf, false));
  };
  x = step(x, moved(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{}));     // row_shr:1
  x = step(x, moved(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{}));
  x = step(x, moved(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{}));
  x = step(x, moved(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{}));
  x = step(x, moved(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}));     // row_bcast:15, rows 1 and 3
  x = step(x, moved(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{}));     // row_bcast:31, rows 2 and 3
  return x;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(x, 0u, [](uint32_t a, uint32_t b) { return max(a, b); }), 63);
}
__device__ __forceinline__ float wave_sum(float x) {
  x = wave_scan(x, 0.f, [](float a, float b) { return a + b; });
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), 63));
}
__device__ __forceinline__ uint32_t rank_in(uint64_t mask) {   // set bits below this lane
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// LDS written by this wave is read by it next (a wave's LDS operations complete in order; this holds the compiler)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Threshold of a row, one wave each: with `mean` = the number of sampled keys expected among the k largest, tau is about the
// w-th largest sampled score, w = mean + 5 sqrt(mean) + 3, so that the k largest lie above it but for a five-sigma accident.
// What there is to choose from are the largest scores of n groups of the N sampled keys that the row sees; a group of N / n keys holds
// one of the w largest with the chance 1 - (1 - w / N)^(N / n), so they fall into n times that many (38 of 1942 keys into 37 of 512
// groups; as if drawn with replacement, n (1 - exp(-w / n)), 61 of 136 keys were said to fall into 39 of 64 groups, not 46: with 512 kept of
// 2300 keys one row in 700 had a list too short).  Every rank more is a list 2 % longer, and twice as many lists that a wave cannot hold:
// the bisection goes on to that very count.
template <int NV>
__global__ void __launch_bounds__(256) topk_tau_kernel(const TopkParams tp) {
  const AttnParams& p = tp.a;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t rid = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
  if (rid >= tp.ntok * p.hq) return;
  const uint32_t rows = tp.ntok * p.group;
  const uint32_t kvh = fast_div(rid, tp.div_rows), rr = rid - kvh * rows;
  const uint32_t tok_l = fast_div(rr, tp.div_group), qh = kvh * p.group + rr - tok_l * p.group;
  const uint32_t tok = tp.tok0 + tok_l;
  if (qh == 0u && tok_l % tp.fail_block_tok == 0u && lane == 0u) tp.fail_block[tok_l / tp.fail_block_tok] = 0u;
  const RowBounds rb = row_bounds(p, tok);
  const uint32_t n_valid = visible_count(rb, p.t_all);
  const uint32_t k = row_k(tp, tok, n_valid);
  const uint32_t n_groups = tp.sample_splits * kBlockN;
  const float* srow = tp.sample_max + (size_t)rid * n_groups;
  uint32_t key[NV], top = 0u;
#pragma unroll
  for (int u = 0; u < NV; ++u) key[u] = __float_as_uint(srow[min(64u * u + lane, n_groups - 1u)]);   // (all in flight)
#pragma unroll
  for (int u = 0; u < NV; ++u) key[u] = 64u * u + lane < n_groups ? score_key(__uint_as_float(key[u])) : 0u;
#pragma unroll
  for (int u = 0; u < NV; ++u) top = max(top, key[u]);
  const float mean = (float)k / (float)tp.sample_stride;
  const float groups = (float)n_groups, sampled = (float)n_valid / (float)tp.sample_stride;   // (a row of this path sees 2048 keys and more)
  const float above = fminf((mean + 5.f * __builtin_sqrtf(mean) + 3.f) / sampled, 1.f);
  const uint32_t want = (uint32_t)(groups - groups * expf(sampled / groups * logf(1.f - above)) + 0.5f);
  // a lower end first, from the lanes' largest keys alone: the want-th largest of those 64 has at least `want` above it
  // (one comparison a step instead of NV; `want` is below 64 at 512 keys kept)
  uint32_t lo = ~wave_max(~top), hi = wave_max(top) + 1u;      // count(>= lo) >= want, count(>= hi) < want
  for (uint32_t h = hi; h - lo > 1u;) {
    const uint32_t mid = lo + ((h - lo) >> 1);
    const uint32_t c = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(top >= mid));
    if (c >= want) lo = mid;
    else h = mid;
    if (c == want) break;
  }
  while (hi - lo > 1u) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    uint32_t c = 0u;
#pragma unroll
    for (int u = 0; u < NV; ++u) c += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(key[u] >= mid));
    if (c >= want) lo = mid;
    else hi = mid;
    if (c == want) break;
  }
  // (A row with fewer groups than wanted that hold a key other than NaN: tau is -inf, what groups without one have, every score
  // passes, and the row is left over where its lists run over.)
  if (lane == 0u) tp.tau[(size_t)kvh * tp.n_mtiles * kTopkFilterRows + rr] = key_score(lo);
}

// Scores against thresholds.  256 stacked rows per workgroup, 64 per wave: with 32 (topk_scores_kernel) the four waves
// together read the K tile from LDS as fast as the LDS can give it (128 bytes a cycle) and the matrix cores wait.
// Splits take every n_splits-th key tile, so that keys that score high side by side spread over the segments.
//
// SAMPLE: every sample_stride-th key, and instead of lists the largest score of each group of sampled keys: a register of the
// score block is a group, of the keys it holds from one of the split's tiles to the next (n_splits tiles apart, so that a group's
// keys are no neighbours).  The thresholds come from those (topk_tau_kernel).  256 groups a row at 256 rows over 33k keys, 4 MB
// between the two launches; as 1942 sampled scores in a plane it was 32 MB: both launches 38 -> 21 us under the profiler (21.4 -> 15.3
// and 16.5 -> 5.6), the layer step 257.3 -> 242.9 (replayed in a graph; 50k keys 428 -> 390, 64 rows over 50k 177 -> 165, 256 over 3k
// 78.4 -> 76.2).  32 rows per wave: with the filter's 64 the query rows come in two trips, and the step took 241.5 - 242.1
// where 252.4 - 252.9 was the old one, but 79.4 for 78.2 over 3k keys.
template <bool F16, bool SAMPLE>
__global__ void __launch_bounds__(256) topk_filter_kernel(const TopkParams tp) {
  constexpr int D = 512;
  const AttnParams& p = tp.a;
  using L = Lay<D>;
  constexpr int NSTEP = D / 16;
  constexpr int NLD = L::NLD;
  constexpr int PF = 3, NB = PF + 1;   // K tiles in flight ahead of the one being multiplied
  constexpr int RB = SAMPLE ? 1 : 2;   // blocks of 32 rows per wave
  __shared__ __attribute__((aligned(1024))) char smem[NB * L::K_BYTES];

  const uint32_t n_units = p.hkv * tp.n_splits * tp.n_mtiles;
  const uint32_t per_xcd = (n_units + 7u) >> 3;
  const uint32_t unit = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
  if (unit >= n_units) return;
  // row tiles of one (KV head, split) next to each other: they read the same keys through one L2
  const uint32_t stream = fast_div(unit, tp.div_mtiles), mt = unit - stream * tp.n_mtiles;
  const uint32_t kvh = fast_div(stream, tp.div_splits), split = stream - kvh * tp.n_splits;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g2 = lane >> 5, l32 = lane & 31u;
  const uint32_t rows_total = tp.ntok * p.group;
  const uint32_t row0 = (mt * 4u + wave) * (32u * RB);
  const uint32_t t_end = SAMPLE ? tp.sample_n : p.t_all;
  const uint32_t n_tiles_all = (t_end + kBlockN - 1u) / kBlockN;
  const uint32_t n_tiles = split < n_tiles_all ? fast_div(n_tiles_all - split + tp.n_splits - 1u, tp.div_splits) : 0u;
  const uint32_t seg = (((kvh * tp.n_mtiles + mt) * tp.n_splits + split) * 4u + wave) * kTopkSegs;   // this wave's first segment
  if constexpr (!SAMPLE) {      // (sampled: no more splits than tiles)
    if (n_tiles == 0u) {
      tp.cand_n[seg + lane] = tp.cand_n[seg + 64u + lane] = 0u;
      return;
    }
  }

  const char* kbase = (const char*)p.k + (int64_t)kvh * p.k_head_stride * 2;
  const int64_t kstride_b = p.k_tok_stride * 2 * (SAMPLE ? tp.sample_stride : 1u);
  const uint32_t k_lane_off = l32 * L::K_STRIDE + g2 * 16u;
  auto tile_t0 = [&](uint32_t i) { return (split + min(i, n_tiles - 1u) * tp.n_splits) * (uint32_t)kBlockN; };
  // (past the last tile: the last one again into a buffer nobody reads, so that the wait counts stay fixed)
  auto k_desc = [&](uint32_t i) {
    return make_tile_load<D, false, false>(kbase, kstride_b, tile_t0(i), 0u, t_end, 0u,
                                           (lds_char*)(smem + (i % NB) * L::K_BYTES), wave, lane);
  };
  // Query rows through the K buffers' LDS, a block of 32 at a time, into accumulation registers.
  u32x4 qf[RB][NSTEP];
  {
    static_assert(4 * 32 * kQRowLds <= NB * L::K_BYTES, "the tile buffers hold a block of every wave's query rows");
    lds_char* const qb = (lds_char*)smem + wave * (32u * kQRowLds);
    const char* const q_base = (const char*)p.q + ((size_t)tp.tok0 * p.hq + kvh * p.group) * (2 * D);
    auto row_off = [&](uint32_t rq) { return (rq + fast_div(rq, tp.div_group) * (p.hq - p.group)) * (uint32_t)(2 * D); };
    u32x4 raw[NSTEP];
    auto read_rows = [&]() {
      wait_vmem_all();
#pragma unroll
      for (int st = 0; st < NSTEP; ++st) raw[st] = *(lds_u32x4*)(qb + l32 * kQRowLds + g2 * 16u + 32 * st);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (before the next loads land there)
    };
    // (bf16 queries over an f16 cache: 384 conversions a block, while the next loads are on their way)
    auto to_frags = [&](auto b_c) {
#pragma unroll
      for (int st = 0; st < NSTEP; ++st) {
        if (F16 && p.q_is_bf16) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            raw[st][e] = pack2<true>(__uint_as_float(raw[st][e] << 16), __uint_as_float(raw[st][e] & 0xffff0000u));
        }
        qf[decltype(b_c)::value][st] = raw[st];
        asm volatile("" : "+a"(qf[decltype(b_c)::value][st]));
      }
    };
    issue_q_rows(q_base, row0, rows_total, p.group, (uint32_t)(size_t)qb, lane, row_off);
    read_rows();
    if constexpr (RB == 2) {
      issue_q_rows(q_base, row0 + 32u, rows_total, p.group, (uint32_t)(size_t)qb, lane, row_off);
      to_frags(std::integral_constant<int, 0>{});
      read_rows();
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PF; ++i) issue_tile<D, false>(k_desc((uint32_t)i), wave, lane);
    to_frags(std::integral_constant<int, RB - 1>{});
  }
  // S = K.Q^T: the lane is a query row of the block, register e is key 8 (e >> 2) + 4 g2 + (e & 3) of the tile.  Each lane
  // keeps lists of its own, one per block, so an entry's place is the lane's count and nothing is exchanged.
  float tau[RB];
  uint32_t lane_base[RB], count[RB] = {};
  float largest[16];          // SAMPLE: of the keys a register has held
  RowBounds rb;
  uint32_t hi_least = 0u;
  if constexpr (SAMPLE) {
    rb = row_bounds(p, tp.tok0 + fast_div(min(row0 + l32, rows_total - 1u), tp.div_group));
    hi_least = ~wave_max(~rb.hi);
#pragma unroll
    for (int e = 0; e < 16; ++e) largest[e] = -INFINITY;
  } else {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const uint32_t r = row0 + 32u * b + l32;
      tau[b] = r < rows_total ? tp.tau[(size_t)kvh * tp.n_mtiles * kTopkFilterRows + r] : INFINITY;
      lane_base[b] = (64u * b + lane) * (kTopkSegAlloc * 8u);
    }
  }
  char* const cbase = (char*)tp.cand + (size_t)seg * (kTopkSegAlloc * 8u);
  const float scale = tp.scale;
  // Comparison of the scores in four registers, in four parts (between the parts, products; side by side, because one wave
  // per SIMD hides no latency of another's).  No branch, and exactly one store per register whose mask is never empty:
  // lane 0 always writes, and where its score is too low, its next entry or nothing takes the place.  So a key tile
  // is always 32 stores and NLD loads of the one memory counter, and the wait at a tile's start can tell its own loads
  // from what was issued behind them.
  // (With query rows in the registers and keys in the lanes an entry's place took a rank among the lanes and a scalar
  // count per register, 15 instructions a score register instead of 8: 163 us instead of 141 for 256 rows over 33k keys.)
  uint64_t mask[4];
  uint32_t at[4];
  u32x2 entry[16];          // (score, position) of register e: positions move on by a tile step, shared by the blocks
  auto keep = [&](auto n_c, const f32x16 (&sc)[RB]) {
    constexpr int n0 = decltype(n_c)::value & ~3, part = decltype(n_c)::value & 3, b = n0 >> 4, e0 = n0 & 15;
    if constexpr (SAMPLE) {
      if constexpr (b == 0) largest[e0 + part] = __builtin_fmaxf(largest[e0 + part], sc[0][e0 + part] * scale);    // (NaN: passed over)
    } else if constexpr (part == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = sc[b][e0 + i] * scale;
        entry[e0 + i][0] = __float_as_uint(v);
        mask[i] = __builtin_amdgcn_ballot_w64(v >= tau[b]);
      }
    } else if constexpr (part == 1) {
      asm volatile("s_nop 1");       // a mask written by a comparison is a carry-in two wait states later at the earliest
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        at[i] = lane_base[b] + count[b] * 8u;
        asm volatile("v_addc_co_u32_e64 %0, vcc, %0, 0, %1" : "+v"(count[b]) : "s"(mask[i]) : "vcc");
      }
    } else if constexpr (part == 2) {
      store4_masked(mask, at, entry[e0], entry[e0 + 1], entry[e0 + 2], entry[e0 + 3], cbase);
    } else if constexpr (e0 == 12) {
      count[b] = min(count[b], kTopkSegCap);
    }
  };
  auto positions = [&](uint32_t t0) {
#pragma unroll
    for (int e = 0; e < 16; ++e) entry[e][1] = t0 + 8u * (e >> 2) + (e & 3) + 4u * g2;
  };

  constexpr int CH = 8, NCHUNK = NSTEP / CH, LPC = NLD / NCHUNK;
  // tile i: its products into s, the comparison of the tile before (sp) between them
  auto tile_step = [&](uint32_t i, f32x16 (&s)[RB], const f32x16 (&sp)[RB]) {
    if constexpr (!SAMPLE) positions(tile_t0(i - 1u));
    // this wave's loads of K(i) have landed: they were issued PF tiles ago (or waited for before the loop), in front of at
    // least two tiles' worth of loads and stores, which is more than the counter can hold back
    static_assert((PF - 1) * (NLD + 32) >= 63, "operations issued behind a tile's loads");
    // (SAMPLE stores nothing: exactly those loads may be outstanding)
    wait_loads_then_barrier<SAMPLE ? (PF - 1) * NLD : 63>();
    const TileLoad tl_next = k_desc(i + PF);
    lds_char* const kb = (lds_char*)(smem + (i % NB) * L::K_BYTES);
    u32x4 fr[2][CH];
    auto read_chunk = [&](int c, u32x4 (&dst)[CH]) {
#pragma unroll
      for (int x = 0; x < CH; ++x) dst[x] = *(lds_u32x4*)(kb + k_lane_off + 32 * (c * CH + x));
    };
    read_chunk(0, fr[0]);
    static_for<0, NCHUNK>([&](auto c_c) {
      constexpr int c = decltype(c_c)::value;
      if constexpr (c + 1 < NCHUNK) read_chunk(c + 1, fr[(c + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, CH>([&](auto i_c) {
        constexpr int x = decltype(i_c)::value, st = c * CH + x;
        if constexpr (st + 1 < NSTEP) {
          static_for<0, RB>([&](auto b_c) { mfma_filter<F16, st == 0>(s[decltype(b_c)::value], fr[c & 1][x], qf[decltype(b_c)::value][st]); });
        } else if constexpr (RB == 1) {
          mfma_filter_last<F16>(s[0], fr[c & 1][x], qf[0][st]);
        } else {
          mfma_filter_last<F16>(s[0], s[1], fr[c & 1][x], qf[0][st], qf[1][st]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (x % (CH / LPC) == 1) issue_tile_part<D, false, c * LPC + x / (CH / LPC)>(tl_next, wave, lane);
        keep(std::integral_constant<int, st>{}, sp);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    if constexpr (SAMPLE) {
      // keys that a row does not see (behind the prefix: a few of the last tiles) and repeats of the last key do not count
      const uint32_t t0 = tile_t0(i);
      if ((t0 + (kBlockN - 1u)) * tp.sample_stride >= hi_least) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const uint32_t t = t0 + 8u * (e >> 2) + (e & 3) + 4u * g2;
          if (!key_visible(rb, t * tp.sample_stride, p.t_all)) s[0][e] = __uint_as_float(0x7fc00000u);
        }
      }
    }
  };
  wait_vmem_all();      // the first PF tiles
  __builtin_amdgcn_s_waitcnt(0xC07F);     // (lgkmcnt(0): or scalar loads in flight here make the compiler wait for whole chunks below)
  f32x16 sa[RB], sb[RB];
#pragma unroll
  for (int e = 0; e < 16; ++e) sb[0][e] = sb[RB - 1][e] = __uint_as_float(0x7fc00000u);   // (in front of the first tile: NaN passes nowhere)
  for (uint32_t i = 0; i < n_tiles; i += 2) {
    tile_step(i, sa, sb);
    if (i + 1u < n_tiles) {
      tile_step(i + 1u, sb, sa);
    } else {
      if constexpr (!SAMPLE) positions(tile_t0(i));
      static_for<0, 32>([&](auto n_c) { keep(n_c, sa); });
    }
  }
  if ((n_tiles & 1u) == 0u) {
    if constexpr (!SAMPLE) positions(tile_t0(n_tiles - 1u));
    static_for<0, 32>([&](auto n_c) { keep(n_c, sb); });
  }
  if constexpr (SAMPLE) {
    const uint32_t r = row0 + l32;
    float* const to = tp.sample_max + ((size_t)kvh * rows_total + r) * (tp.n_splits * kBlockN) + split * kBlockN + 16u * g2;
    if (r < rows_total) {
#pragma unroll
      for (int e = 0; e < 16; e += 4) *(f32x4*)(to + e) = f32x4{largest[e], largest[e + 1], largest[e + 2], largest[e + 3]};
    }
  } else {
    tp.cand_n[seg + lane] = count[0];
    tp.cand_n[seg + 64u + lane] = count[RB - 1];
  }
  wait_vmem_all();   // no direct-to-LDS load may outlive the workgroup's LDS
}

// One wave per row: candidates from the row's segments, the k-th largest by bisection over registers (a ballot per 64
// candidates and step; no histogram, no barrier), the kept keys in position order by ranking them in a bitmap, softmax.
// As long as a wave's instructions, 1270 vector and 1160 scalar ones at 646 candidates for 258 kept (four waves a SIMD, in one round). The
// last dozen steps of the bisection look at the candidates still between its ends alone, one register; only the kept ones are ranked,
// packed once more (5 registers instead of 11); sums and scans by DPP, not through LDS: 1790 and 1260 before, without the spills,
// 31.3 -> 26.3 us under the profiler, layer step with 256 rows over 33k keys 237.7 -> 229.8, over 3k 75.7 -> 71.1, 64 rows over 50k 147.4 -> 138.3.
constexpr uint32_t kRankWords = 64 * 17;               // bitmap words, 17 per lane: an odd stride, no bank conflicts
constexpr uint32_t kRankWindow = kRankWords * 32;      // positions per pass
template <int NR>
__global__ void __launch_bounds__(256, NR <= 20 ? 4 : NR == 24 ? 3 : 2) topk_list_select_kernel(const TopkParams tp) {
  constexpr uint32_t CAP = 64u * NR;                   // candidates a wave can hold
  constexpr uint32_t SEL = NR == 16 ? 160u : NR == 20 ? 272u : NR == 24 ? 384u : 512u;   // most keys kept
  static_assert(CAP * 8u >= kRankWords * 6u + SEL * 8u, "bitmap, prefix counts and kept keys reuse the candidate list");
  const AttnParams& p = tp.a;
  __shared__ __attribute__((aligned(16))) u32x2 lists[4][CAP];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n_rows = tp.ntok * p.hq;
  const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);   // runs of rows, one per XCD
  const uint32_t rid = wg * 4u + wave;
  if (rid >= n_rows) return;
  const uint32_t rows = tp.ntok * p.group;
  const uint32_t kvh = fast_div(rid, tp.div_rows), rr = rid - kvh * rows;
  const uint32_t tok_l = fast_div(rr, tp.div_group), qh = kvh * p.group + rr - tok_l * p.group;
  const uint32_t tok = tp.tok0 + tok_l;
  const RowBounds rb = row_bounds(p, tok);
  const uint32_t k = row_k(tp, tok, visible_count(rb, p.t_all));
  u32x2* const list = lists[wave];

  // ---- this row's candidates, packed ----
  // (half a wave per segment: the two lanes that held the row in the filter kernel had a list each)
  const uint32_t seg0 = ((kvh * tp.n_mtiles + (rr >> 8)) * tp.n_splits * 4u + ((rr >> 6) & 3u)) * kTopkSegs +
                        ((rr >> 5) & 1u) * 64u + (rr & 31u) + (lane & 32u);
  constexpr uint32_t seg_step = 4u * kTopkSegs;
  const uint32_t l32 = lane & 31u;
  const u32x2* const cand = (const u32x2*)tp.cand;
  uint32_t n = 0u;
  bool over = false;
  auto take = [&](u32x2 v, bool in) {
    const bool own = in && key_visible(rb, v[1], p.t_all);
    const uint64_t m = __builtin_amdgcn_ballot_w64(own);
    const uint32_t to = n + rank_in(m);
    if (own && to < CAP) list[to] = u32x2{score_key(__uint_as_float(v[0])), v[1]};
    n += (uint32_t)__builtin_popcountll(m);
  };
  constexpr uint32_t SB = 8;       // splits in flight
  for (uint32_t s0 = 0; s0 < tp.n_splits; s0 += SB) {
    u32x2 v[SB];
    uint32_t c[SB];
#pragma unroll
    for (uint32_t i = 0; i < SB; ++i) {
      c[i] = s0 + i < tp.n_splits ? tp.cand_n[seg0 + (s0 + i) * seg_step] : 0u;
      // (the first 32 places of a segment exist whatever its count)
      v[i] = cand[(size_t)(seg0 + min(s0 + i, tp.n_splits - 1u) * seg_step) * kTopkSegAlloc + l32];
    }
#pragma unroll
    for (uint32_t i = 0; i < SB; ++i) {
      over |= c[i] >= kTopkSegCap;
      take(v[i], l32 < c[i]);
      for (uint32_t x = 32u; __builtin_amdgcn_ballot_w64(x < c[i]) != 0ull; x += 32u) {
        u32x2 w = {0u, 0u};
        if (l32 + x < c[i]) w = cand[(size_t)(seg0 + (s0 + i) * seg_step) * kTopkSegAlloc + l32 + x];
        take(w, l32 + x < c[i]);
      }
    }
  }
  const bool fail = __builtin_amdgcn_ballot_w64(over) != 0ull || n < k || n > CAP;
  if (lane == 0u) {
    tp.fail_rows[(size_t)tok * p.hq + qh] = fail ? 1u : 0u;
    if (fail) atomicAdd(&tp.fail_block[tok_l / tp.fail_block_tok], 1u);
  }
  if (fail) return;
  wave_lds_fence();
  const uint32_t nu = (n + 63u) >> 6;
  uint32_t key[NR], pos[NR];
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    key[u] = 0u;           // (below every candidate: NaN never passes a threshold)
    pos[u] = 0xffffffffu;
    if ((uint32_t)u < nu && 64u * u + lane < n) {
      const u32x2 v = list[64u * u + lane];
      key[u] = v[0];
      pos[u] = v[1];
    }
  }
  wave_lds_fence();

  // ---- the k-th largest ----
  uint32_t top = 0u, bot = 0xffffffffu;
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    top = max(top, key[u]);
    if (pos[u] != 0xffffffffu) bot = min(bot, key[u]);
  }
  top = wave_max(top);
  bot = ~wave_max(~bot);
  auto count_ge = [&](uint32_t x) {
    uint32_t c = 0u;
#pragma unroll
    for (int u = 0; u < NR; u += 4) {
      if ((uint32_t)u < nu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(key[u + i] >= x));
      }
    }
    return c;
  };
  // bisection over all registers until no more than a lane's worth of candidates is between the ends, then over those alone
  uint32_t lo = bot, hi = top + 1u, c_lo = n, c_hi = 0u;      // count(>= lo) = c_lo >= k > c_hi = count(>= hi)
  while (hi - lo > 1u && c_lo != k && c_lo - c_hi > 64u) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    const uint32_t c = count_ge(mid);
    if (c >= k) {
      lo = mid;
      c_lo = c;
    } else {
      hi = mid;
      c_hi = c;
    }
  }
  if (hi - lo > 1u && c_lo != k) {
    uint32_t* const few = (uint32_t*)list;
    uint32_t at = 0u;
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      if ((uint32_t)u < nu) {
        const bool own = key[u] >= lo && key[u] < hi;
        const uint64_t m = __builtin_amdgcn_ballot_w64(own);
        if (own) few[at + rank_in(m)] = key[u];
        at += (uint32_t)__builtin_popcountll(m);
      }
    }
    wave_lds_fence();
    const uint32_t x = lane < at ? few[lane] : 0u;
    wave_lds_fence();
    while (hi - lo > 1u && c_lo != k) {
      const uint32_t mid = lo + ((hi - lo) >> 1);
      const uint32_t c = c_hi + (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(x >= mid && x < hi));
      if (c >= k) {
        lo = mid;
        c_lo = c;
      } else {
        hi = mid;
        c_hi = c;
      }
    }
  }
  // equal scores at the threshold: the lower positions are kept, up to t_last
  uint32_t t_last = 0xfffffffeu;
  if (c_lo != k) {
    const uint32_t drop = c_lo - k;              // this many of the highest positions among the equal ones go
    uint32_t a = 0u, b = p.t_all;                // count(equal, position >= a) >= drop > ... >= b
    while (b - a > 1u) {
      const uint32_t mid = a + ((b - a) >> 1);
      uint32_t c = 0u;
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        if ((uint32_t)u < nu) c += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(key[u] == lo && pos[u] >= mid));
      }
      if (c >= drop) a = mid;
      else b = mid;
    }
    t_last = a - 1u;      // (position a is the last one dropped; a > 0 because at least one equal key stays)
  }
  // ---- the kept ones, packed: fewer registers to rank ----
  uint32_t* const bits = (uint32_t*)list;
  uint16_t* const before = (uint16_t*)(bits + kRankWords);
  u32x2* const sel = list + kRankWords * 6u / 8u;          // (key, position), then (weight, byte offset of the key's V row)
  constexpr int NK = (int)(SEL + 63u) / 64;
  uint32_t kkey[NK], kpos[NK];
  {
    uint32_t at = 0u;
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      if ((uint32_t)u < nu) {
        const bool own = key[u] > lo || (key[u] == lo && pos[u] <= t_last);
        const uint64_t m = __builtin_amdgcn_ballot_w64(own);
        const uint32_t to = at + rank_in(m);
        if (own && to < SEL) sel[to] = u32x2{key[u], pos[u]};
        at += (uint32_t)__builtin_popcountll(m);
      }
    }
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const u32x2 v = sel[min(64u * u + lane, k - 1u)];
      kkey[u] = v[0];
      kpos[u] = 64u * u + lane < k ? v[1] : 0xffffffffu;      // (in no window below)
    }
    wave_lds_fence();
  }

  // ---- softmax over the kept scores (cpu.rs:95-104), and their order by position ----
  const uint32_t v_step = (uint32_t)p.v_tok_stride * 2u;   // (offsets stay below 2^32: the host's rule)
  const float mmax = key_score(top);
  float l = 0.f;
  uint32_t ranked = 0u;
  for (uint32_t t0 = 0; t0 < p.t_all; t0 += kRankWindow) {
#pragma unroll
    for (uint32_t w = 0; w < 17u; ++w) bits[64u * w + lane] = 0u;
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      if (kpos[u] - t0 < kRankWindow) atomicOr(&bits[(kpos[u] - t0) >> 5], 1u << ((kpos[u] - t0) & 31u));
    }
    wave_lds_fence();
    uint32_t run = 0u;
#pragma unroll
    for (uint32_t w = 0; w < 17u; ++w) {
      before[17u * lane + w] = (uint16_t)run;
      run += (uint32_t)__builtin_popcount(bits[17u * lane + w]);
    }
    const uint32_t incl = wave_scan(run, 0u, [](uint32_t a, uint32_t b) { return a + b; });
    const uint32_t excl = incl - run;
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const bool in = kpos[u] - t0 < kRankWindow;
      const uint32_t w = in ? (kpos[u] - t0) >> 5 : 0u;
      const uint32_t base = (uint32_t)__shfl((int)excl, (int)(w / 17u), 64);
      if (in) {
        const uint32_t r = ranked + base + before[w] + (uint32_t)__builtin_popcount(bits[w] & ((1u << (kpos[u] & 31u)) - 1u));
        const float e = expf(key_score(kkey[u]) - mmax);
        l += e;
        if (r < SEL) sel[r] = u32x2{__float_as_uint(e), kpos[u] * v_step};
      }
    }
    ranked += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    wave_lds_fence();
  }
  l = wave_sum(l);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u32x2* const out = (u32x2*)tp.kept + (size_t)rid * tp.kept_pad;
  for (uint32_t j = lane; j < k; j += 64u) {
    const u32x2 v = sel[j];
    out[j] = u32x2{__float_as_uint(__uint_as_float(v[0]) * inv), v[1]};
  }
}

// Gathered P.V of the rows the selection has listed.  A launch of its own so that its waves begin together: all waves of an XCD
// sweep the keys in order, and a V row that several of its rows want should be fetched into its L2 once.
// One wave per (row, slice of head_dim), SL slices: a slice's lanes of SL keys stand side by side and their sums meet at the end.
// With more than 2048 rows whole rows (SL = 1), 512 rows of 256 x 16 to an XCD: bound by what the eight L2s fetch, 288 MB
// at 33k keys where 270 are the least (each V row once into each L2 whose rows want it), and 30 us of unpacking and
// multiplying.  Fewer loads ahead than four hide too little, more pull the sweeps apart: 1 row ahead 101 us, 2 rows 68, 4 rows 52,
// 8 rows 88.  Up to 2048 rows there are too few waves for that, and XCDs take one slice of more rows each: 128 rows over 30k keys, layer
// step, whole rows | halves | quarters 148.0 | 140.6 | 145.0 us, 64 rows 115.0 | 103.6 | 101.2, 64 over 50k 168.3 | 148.4 | 147.4, 16 over
// 100k 245.0 | 207.5 | 188.8.  With 256 rows over 33k slices lose, 239.6 | 249.0 | 260.5: a slice of every row
// lies on a part of an L2's channels, and although less is fetched (199 MB in halves), it comes slower.
template <bool F16, uint32_t SL>
__global__ void __launch_bounds__(256, 8) topk_gather_kernel(const TopkParams tp) {
  constexpr uint32_t D = 512, PER = 8, LPK = 64u / SL, GU = 4;     // LPK lanes per key, GU loads in flight
  static_assert(LPK * PER * SL == D, "a lane owns 8 consecutive d");
  const AttnParams& p = tp.a;
  __shared__ u32x2 lists[4][kTopkListMax];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t rows = tp.ntok * p.group;
  const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);   // runs of units, one per XCD
  const uint32_t unit = wg * 4u + wave;                                           // (KV head, row, slice)
  if (unit >= tp.ntok * p.hq * SL) return;
  const uint32_t stream = fast_div(unit, tp.div_rows), rr = unit - stream * rows;
  const uint32_t kvh = stream / SL, slice = stream % SL, rid = kvh * rows + rr;
  const uint32_t tok_l = fast_div(rr, tp.div_group), tok = tp.tok0 + tok_l, qh = kvh * p.group + rr - tok_l * p.group;
  if (tp.fail_rows[(size_t)tok * p.hq + qh] != 0u) return;       // (the general path's)
  const uint32_t k = row_k(tp, tok, visible_count(row_bounds(p, tok), p.t_all));
  u32x2* const list = lists[wave];
  {
    const u32x2* const kept = (const u32x2*)tp.kept + (size_t)rid * tp.kept_pad;
    for (uint32_t j = lane; j < k; j += 64u) list[j] = kept[j];
  }
  wave_lds_fence();
  float acc[PER];
#pragma unroll
  for (uint32_t i = 0; i < PER; ++i) acc[i] = 0.f;
  const char* const vbase = (const char*)p.v + (int64_t)kvh * p.v_head_stride * 2 + slice * (LPK * PER * 2u);
  const uint32_t lane_b = lane % LPK * (PER * 2u);
  const uint32_t own = lane / LPK;
  auto group = [&](uint32_t j0, auto tail_c) {      // keys j0 + own + SL u
    constexpr bool TAIL = decltype(tail_c)::value;
    float w[GU];
    u32x4 raw[GU];
#pragma unroll
    for (uint32_t u = 0; u < GU; ++u) {
      const uint32_t j = j0 + own + SL * u;
      const u32x2 v = list[TAIL ? min(j, k - 1u) : j];
      w[u] = __uint_as_float(v[0]);
      raw[u] = *(const u32x4*)(vbase + (v[1] + lane_b));
      if (TAIL && j >= k) raw[u] = u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (uint32_t u = 0; u < GU; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = __builtin_fmaf(w[u], unpack_lo<F16>(raw[u][i]), acc[2 * i]);
        acc[2 * i + 1] = __builtin_fmaf(w[u], unpack_hi<F16>(raw[u][i]), acc[2 * i + 1]);
      }
    }
  };
  uint32_t j0 = 0u;
  for (; j0 + SL * GU <= k; j0 += SL * GU) group(j0, std::false_type{});
  if (j0 < k) group(j0, std::true_type{});
#pragma unroll
  for (uint32_t i = 0; i < PER; ++i) {
#pragma unroll
    for (uint32_t off = LPK; off < 64u; off <<= 1) acc[i] += __shfl_xor(acc[i], (int)off, 64);
  }
  if (lane >= LPK) return;
  const size_t out_off = ((size_t)tok * p.hq + qh) * D + (slice * LPK + lane) * PER;
  if (p.out_dtype == 2u) {
    float* const o = (float*)p.out + out_off;
    *(f32x4*)o = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *(f32x4*)(o + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
  } else {
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = (uint32_t)f32_to_bf16_bits(acc[2 * i], p.out_trunc != 0u) |
             ((uint32_t)f32_to_bf16_bits(acc[2 * i + 1], p.out_trunc != 0u) << 16);
    *(u32x4*)((uint16_t*)p.out + out_off) = o;
  }
}

void set_dividers(TopkParams* tp) {
  tp->div_mtiles = make_fast_div(tp->n_mtiles);
  tp->div_splits = make_fast_div(tp->n_splits);
  tp->div_group = make_fast_div(tp->a.group);
  tp->div_rows = make_fast_div(tp->ntok * tp->a.group);
}

template <int D, bool F16>
hipError_t launch_stage(TopkParams tp, int stage, hipStream_t s) {
  set_dividers(&tp);
  if (stage == 0) {
    const uint32_t n_units = tp.a.hkv * tp.n_splits * tp.n_mtiles;
    const uint32_t grid = ((n_units + 7u) / 8u) * 8u;
    hipLaunchKernelGGL((topk_scores_kernel<D, F16>), dim3(grid), dim3(256), 0, s, tp);
  } else {
    hipLaunchKernelGGL((topk_select_kernel<D, F16>), dim3(tp.ntok, tp.a.hq), dim3(256), 0, s, tp);
  }
  return hipGetLastError();
}

template <bool F16>
hipError_t launch_by_dim(const TopkParams& tp, int stage, uint32_t head_dim, hipStream_t s) {
  switch (head_dim) {
    case 32: return launch_stage<32, F16>(tp, stage, s);
    case 64: return launch_stage<64, F16>(tp, stage, s);
    case 128: return launch_stage<128, F16>(tp, stage, s);
    case 256: return launch_stage<256, F16>(tp, stage, s);
    case 512: return launch_stage<512, F16>(tp, stage, s);
    default: return hipErrorInvalidValue;
  }
}

template <bool F16>
hipError_t launch_filter(TopkParams tp, hipStream_t s) {
  set_dividers(&tp);
  TopkParams sample = tp;
  sample.n_splits = tp.sample_splits;
  sample.n_mtiles = (tp.ntok * tp.a.group + kTopkSampleRows - 1u) / kTopkSampleRows;
  set_dividers(&sample);
  const uint32_t sample_units = tp.a.hkv * sample.n_mtiles * sample.n_splits;
  hipLaunchKernelGGL((topk_filter_kernel<F16, true>), dim3((sample_units + 7u) / 8u * 8u), dim3(256), 0, s, sample);
  hipError_t rc = hipGetLastError();
  if (rc != hipSuccess) return rc;
  const uint32_t rows = tp.ntok * tp.a.hq;
  const dim3 by_wave((rows + 3u) / 4u);
  const uint32_t n_groups = tp.sample_splits * kBlockN;
  if (n_groups <= 64u * 4u) hipLaunchKernelGGL((topk_tau_kernel<4>), by_wave, dim3(256), 0, s, tp);
  else if (n_groups <= 64u * 8u) hipLaunchKernelGGL((topk_tau_kernel<8>), by_wave, dim3(256), 0, s, tp);
  else if (n_groups <= 64u * 16u) hipLaunchKernelGGL((topk_tau_kernel<16>), by_wave, dim3(256), 0, s, tp);
  else if (n_groups <= 64u * 32u) hipLaunchKernelGGL((topk_tau_kernel<32>), by_wave, dim3(256), 0, s, tp);
  else hipLaunchKernelGGL((topk_tau_kernel<64>), by_wave, dim3(256), 0, s, tp);
  if ((rc = hipGetLastError()) != hipSuccess) return rc;
  hipLaunchKernelGGL((topk_filter_kernel<F16, false>), dim3((tp.a.hkv * tp.n_mtiles * tp.n_splits + 7u) / 8u * 8u), dim3(256), 0, s, tp);
  return hipGetLastError();
}
template <bool F16>
hipError_t launch_list_select(TopkParams tp, uint32_t k_most, hipStream_t s) {
  set_dividers(&tp);
  const dim3 sel((tp.ntok * tp.a.hq + 31u) / 32u * 8u);
  // Instances by what their waves hold of a list, 1024 to 2048 candidates.  Past 139k keys every 19th or 21st is sampled and a list is
  // longer and less certain: the next instance there.  (256 rows over 170k keys, where the smaller one cannot hold 1 to 2 rows in 10^4: with
  // 384 kept and two such rows 1674 -> 917 us; without one 847 -> 859 with 258 kept, 785 -> 788 with 128.)
  const uint32_t inst = (k_most <= 160u ? 0u : k_most <= 272u ? 1u : k_most <= 384u ? 2u : 3u) + (tp.sample_stride > 17u ? 1u : 0u);
  if (inst == 0u) hipLaunchKernelGGL((topk_list_select_kernel<16>), sel, dim3(256), 0, s, tp);
  else if (inst == 1u) hipLaunchKernelGGL((topk_list_select_kernel<20>), sel, dim3(256), 0, s, tp);
  else if (inst == 2u) hipLaunchKernelGGL((topk_list_select_kernel<24>), sel, dim3(256), 0, s, tp);
  else hipLaunchKernelGGL((topk_list_select_kernel<32>), sel, dim3(256), 0, s, tp);
  const hipError_t rc = hipGetLastError();
  if (rc != hipSuccess) return rc;
  const uint32_t n_rows = tp.ntok * tp.a.hq, slices = topk_gather_slices(n_rows);
  const dim3 gather((n_rows * slices + 31u) / 32u * 8u);
  if (slices == 1u) hipLaunchKernelGGL((topk_gather_kernel<F16, 1>), gather, dim3(256), 0, s, tp);
  else if (slices == 2u) hipLaunchKernelGGL((topk_gather_kernel<F16, 2>), gather, dim3(256), 0, s, tp);
  else hipLaunchKernelGGL((topk_gather_kernel<F16, 4>), gather, dim3(256), 0, s, tp);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_topk_filter(const TopkParams& tp, uint32_t kv_dtype, hipStream_t s) {
  return kv_dtype == 1u ? launch_filter<true>(tp, s) : launch_filter<false>(tp, s);
}
hipError_t launch_topk_list_select(const TopkParams& tp, uint32_t k_most, uint32_t kv_dtype, hipStream_t s) {
  return kv_dtype == 1u ? launch_list_select<true>(tp, k_most, s) : launch_list_select<false>(tp, k_most, s);
}
hipError_t launch_topk_scores(const TopkParams& tp, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s) {
  return kv_dtype == 1u ? launch_by_dim<true>(tp, 0, head_dim, s) : launch_by_dim<false>(tp, 0, head_dim, s);
}
hipError_t launch_topk_select(const TopkParams& tp, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s) {
  return kv_dtype == 1u ? launch_by_dim<true>(tp, 1, head_dim, s) : launch_by_dim<false>(tp, 1, head_dim, s);
}

}  // namespace dg
