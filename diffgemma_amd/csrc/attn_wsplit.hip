// Denoise-step attention for short key ranges (a sliding-window layer: ~1300 visible keys) in ONE launch.
//
// A sliding layer is a 5 GFLOP problem: split over workgroups along the keys (attn_mfma.hip), most of its
// time is what the split costs (partial rows written to memory, a second kernel that reads them back, two
// launches), not its tile loop.  Here the keys are split over the WAVES of a workgroup instead and the
// partial results meet in LDS:
//
//   workgroup = MR x 32 stacked query rows of one KV head (stacked row = canvas_row * group + head_in_group),
//   wave w    = a quarter of the key tiles those rows can see, all of the rows, the whole head_dim.
//
// A wave holds Q (B operand of S^T = K.Q^T) for its rows and the MR x 32 x head_dim accumulators O in registers, streams
// its own 32-key K and V tiles into its own piece of LDS with direct-to-LDS loads, and waits only for its own loads
// (vmcnt): the tile loop has no workgroup barrier.  The score accumulator holds, per lane, 16 keys of the lane's row in
// exactly the order the B operand of O^T += V^T.P^T wants them, so P never leaves the registers.  K and V have one buffer
// each per wave (two would not fit the LDS): per tile a wave runs softmax(j), with the loads of K(j+1) issued as soon as
// the tile's maximum has read the scores (the K buffer is free once the scores of tile j exist), then P.V(j), then the
// scores of tile j+1 with the loads of V(j+1) between its MFMAs (the V buffer is free after P.V).
// At the end the (m, l, O) of a row's shares are combined through LDS with the closed form
//   m = max m_i,  l = sum l_i 2^(m_i - m),  O = sum O_i 2^(m_i - m) / l,
// always in the same order (run-to-run bit-identical), and each output row is stored once, whole.
//
// What bounds it.  A tile is read by one wave only, so every workgroup streams all keys of its KV head through its compute
// unit's load path (64 B/clk: 32 KiB per wave and tile is 2048 cycles for four waves), and 16 row tiles of a head draw
// most of what an L2 delivers.  With 32 rows per wave that is twice the tile's MFMA time; with 64 (MR = 2) every loaded
// byte and every fragment read from LDS serves twice the MFMAs, at half as many workgroups.  Around the loop it is
// instructions: code that runs once per launch is fetched cold, about 10 cycles per instruction, so the prologue
// and the epilogue are written for few of them (LDS rows padded so that a tile needs one per-lane load offset instead of a
// table, scalar address arithmetic, divisions by multiplication, accumulators stored to LDS without passing through vector
// registers, the shares of a row exchanged in register order).
// A few canvas rows over most of a window leave three quarters of the chip idle: there several workgroups share a row tile's
// keys and leave fp32 rows for the split kernel's merge (SHARED; the rule with both sides measured: dg_attn_api.hip).
// Measured (GPU time of producer + attention, before and after these): a sliding layer over 1279 keys 23.1 -> 21.0 us, over
// an f16 cache 25.6 -> 22.4; 64 rows behind 22 keys 13.4 -> 9.5; 901 causal rows 50.2 -> 33.8; 64 rows over a window 18.8 -> 14.5.  Of a launch over 1279 keys
// 1.5 us go before the first scores, 1.6 into the first tile (cold code), 1.07 into each later one (the compute unit's load
// path alone takes 0.85), 2.1 into the shares of the four waves and the rows.
// Softmax arithmetic (lazy reference max, exponent offset under which negligible weights become exact zeros,
// row sum over the rounded probabilities) is that of attn_mfma.hip, without its explicit zeroing of weights
// far below the running max (a power device of the long kernel; here it would only cost instructions).
#include "attn_params.h"
#include "mfma_tile.h"
#include "wt_store.h"

#include <algorithm>

namespace dg {
namespace {

template <bool F16>
constexpr float kWsTau = F16 ? 15.9f : 120.0f;   // as attn_mfma.hip: how far a tile max may exceed the reference
template <bool F16>
constexpr float kWsPOff = F16 ? 0.0f : 86.0f;    // probabilities are stored as 2^(score - reference - offset)
// With f16 probabilities a raise puts the reference this many binades ABOVE the running max, so that the next
// raise needs a score 2^(15.9 + 4) over it: a wave of a sliding layer rescales O 3.3 times in its 10 tiles instead
// of 5.6 (a rescale is 128 accumulation registers read, multiplied and written: as long as a tile).  The price is
// f16's tail: a weight more than 2^(24 - 4) below the row's largest is stored with an absolute error of up to
// 2^-25 of the reference or dropped, i.e. up to 2^-21 of the largest weight per key; this kernel sees at most 2048
// keys per row (64 tiles, dg_attn_api.hip), so at most 2^-10 of a row's mass moves: under the rounding of a 16-bit
// output (tests/test_gpu_parity.py builds the worst case).  The kernel for long key ranges (attn_mfma.hip) keeps a
// reference that never leads: at 33 024 keys the same bound would be 2^-6.
template <bool F16>
constexpr float kWsLead = F16 ? 4.0f : 0.0f;

typedef __bf16 ws_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 ws_f16x2 __attribute__((ext_vector_type(2)));
template <bool F16>
__device__ __forceinline__ float ws_add_pair(uint32_t pk, float acc) {
  if constexpr (F16) {
    const ws_f16x2 ones = {(_Float16)1.f, (_Float16)1.f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(ws_f16x2, pk), ones, acc, false);
  } else {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ws_bf16x2, pk), __builtin_bit_cast(ws_bf16x2, 0x3f803f80u),
                                           acc, false);
  }
}

// A 32-key tile in LDS.  One direct-to-LDS instruction brings a KiB = RPK = 512 / D whole rows, and instruction i brings
// rows i, i + NBLK, i + 2 NBLK, ...: the lanes' offset from the tile's first row is then the same for every instruction
// of the tile, which only moves a scalar address by one row.  The KiB blocks are padded apart (K by 16 bytes, V by 64),
// which keeps the fragment reads free of bank conflicts at head_dim 256.
template <int D>
struct WsLay {
  static constexpr int NBLK = D / 16, RPK = 512 / D, ROWB = 2 * D;
  static constexpr int K_BLK = 1024 + 16, V_BLK = 1024 + 64;
  static constexpr int K_BYTES = NBLK * K_BLK, V_BYTES = NBLK * V_BLK;
  static constexpr int SLICE = K_BYTES + V_BYTES > 32 * (4 * D + 16) ? K_BYTES + V_BYTES : 32 * (4 * D + 16);
  // byte offset of row 8 n (+ a row below 8, whose offset is per lane) in a V tile
  static constexpr int v_row8(int n) {
    return NBLK == 16 ? (n & 1) * 8 * V_BLK + (n >> 1) * ROWB : n * (8 / NBLK) * ROWB;
  }
};

// lds_dma_group (mfma_tile.h) with an offset of its own for every block.
template <int G, int LDS_OFF, int BLK>
__device__ __forceinline__ void ws_issue_clamped(uint64_t base, const uint32_t (&voff)[4], uint32_t lds) {
  if constexpr (G == 1)
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff[0]), "s"(base), "n"(LDS_OFF)
                 : "memory", "scc");
  else if constexpr (G == 2)
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\t"
                 "global_load_lds_dwordx4 %2, %3 offset:%5" ::"s"(lds), "v"(voff[0]), "v"(voff[1]), "s"(base), "n"(LDS_OFF), "n"(BLK)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %0, %6\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %5\n\t"
                 "global_load_lds_dwordx4 %2, %5 offset:%7\n\tglobal_load_lds_dwordx4 %3, %5 offset:%8\n\t"
                 "global_load_lds_dwordx4 %4, %5 offset:%9" ::"s"(lds), "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(base),
                 "n"(LDS_OFF), "n"(BLK), "n"(2 * BLK), "n"(3 * BLK)
                 : "memory", "scc");
}

struct WsArgs {
  AttnParams p;
  FastDiv div_rt;        // by the number of row tiles
  FastDiv div_group;     // by the GQA group
  FastDiv div_splits;    // by the workgroups that share a row tile's keys (AttnParams.n_splits)
  uint32_t n_rt;
  uint32_t touch;        // the key range is touched into the L2 first
};

// SHARED: several workgroups to a row tile (an instance of its own: what it takes at the start and the end is 0.4 us of a
// launch of 7)
template <int D, bool F16, int MR, bool SHARED>
__global__ void __launch_bounds__(256) attn_wsplit_kernel(const WsArgs args) {
  const AttnParams p = resolve_step(args.p);
  using L = WsLay<D>;
  constexpr int NSTEP = D / 16, NDB = D / 32, NBLK = L::NBLK;
  constexpr int ROWS = 32 * MR;
  // K and V tile of wave w: slice w.  The query rows come in through LDS too: 32 of them in a piece of their own, 64 in
  // the V tiles of slices 0 and 1 (not in use yet).
  constexpr int OFF_ML = 4 * L::SLICE + (MR == 1 ? L::K_BYTES : 0), OFF_DUMP = OFF_ML + 4 * ROWS * 8, LDS_BYTES = OFF_DUMP + 4 * 256;
  auto off_q = [](uint32_t m) { return MR == 1 ? (uint32_t)(4 * L::SLICE) : m * (uint32_t)L::SLICE + (uint32_t)L::K_BYTES; };
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of one compute unit");
  __shared__ __attribute__((aligned(1024))) char smem[LDS_BYTES];

  // ---- which (KV head, row tile) this workgroup owns: ids go round-robin over the 8 XCDs (each has its
  // own L2); the units, KV head first, are cut into 8 equal runs, so the row tiles of a head, which stream
  // the same keys, sit behind one L2 ----
  const uint32_t n_units = p.hkv * (SHARED ? p.n_splits : 1u) * args.n_rt;
  const uint32_t per_xcd = (n_units + 7u) >> 3;
  const uint32_t unit = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
  if (unit >= n_units) return;
  const uint32_t stream = fast_div(unit, args.div_rt), rt = unit - stream * args.n_rt;
  const uint32_t kvh = SHARED ? fast_div(stream, args.div_splits) : stream, split = SHARED ? stream - kvh * p.n_splits : 0u;

  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g2 = lane >> 5, l32 = lane & 31u, h16 = (lane >> 4) & 1u, i16 = lane & 15u;

  // ---- bounds that hold for every row of the workgroup: which key tiles to visit, which need the mask ----
  const uint32_t row0 = rt * ROWS;
  uint32_t lo_min, lo_max, hi_min, hi_max;
  {
    const uint32_t last_row = min(row0 + ROWS, p.rows_total) - 1u;
    const uint32_t tok_a = fast_div(row0, args.div_group), tok_b = fast_div(last_row, args.div_group);
    const RowBounds ba = row_bounds(p, tok_a), bb = row_bounds(p, tok_b);
    lo_min = min(ba.lo, bb.lo);
    lo_max = max(ba.lo, bb.lo);
    hi_min = min(ba.hi, bb.hi);
    hi_max = max(ba.hi, bb.hi);
    if (tok_a < p.causal_rows && tok_b >= p.causal_rows) {  // both kinds of rows in the tile
      const RowBounds bc = row_bounds(p, p.causal_rows - 1u), bd = row_bounds(p, p.causal_rows);
      lo_min = min(lo_min, min(bc.lo, bd.lo));
      lo_max = max(lo_max, max(bc.lo, bd.lo));
      hi_min = min(hi_min, min(bc.hi, bd.hi));
      hi_max = max(hi_max, max(bc.hi, bd.hi));
    }
    if (tok_a < p.causal_rows && p.extra_lo < p.t_clip_hi) hi_max = p.t_clip_hi;
  }
  // the key tiles these rows can see (a run of them each for the workgroups that share a row tile), cut into four equal runs,
  // one per wave
  uint32_t mt_begin = max(lo_min / kBlockN, p.tile_first);
  uint32_t mt_end = max(min((hi_max + kBlockN - 1) / kBlockN, p.tile_end), mt_begin);
  if constexpr (SHARED) {
    const uint32_t end = mt_end, per_split = fast_div(end - mt_begin + p.n_splits - 1u, args.div_splits);
    mt_begin = min(mt_begin + split * per_split, end);
    mt_end = min(mt_begin + per_split, end);
  }
  const uint32_t per_run = (mt_end - mt_begin + 3u) >> 2;
  const uint32_t tb = min(mt_begin + wave * per_run, mt_end);
  const uint32_t te = min(tb + per_run, mt_end);
  const uint32_t ntile = te - tb;

  // ---- how tiles are loaded ----
  const char* kbase = (const char*)p.k + (int64_t)kvh * p.k_head_stride * 2;
  const char* vbase = (const char*)p.v + (int64_t)kvh * p.v_head_stride * 2;
  const int64_t kstride_b = p.k_tok_stride * 2, vstride_b = p.v_tok_stride * 2;
  const uint32_t lgrp = lane / (64u / L::RPK), lcol = (lane & (64u / L::RPK - 1u)) * 16u;
  const uint32_t koff = lgrp * (uint32_t)NBLK * (uint32_t)kstride_b + lcol;
  const uint32_t voff = lgrp * (uint32_t)NBLK * (uint32_t)vstride_b + lcol;
  const uint32_t lds0 = (uint32_t)(size_t)(lds_char*)smem;
  const uint32_t my_k = lds0 + wave * (uint32_t)L::SLICE, my_v = my_k + (uint32_t)L::K_BYTES;
  // a tile with rows that must not be read (tile_rows): of K as of V
  auto is_edge = [&](uint32_t tile) { return tile_is_edge(tile * kBlockN, lo_min, p.t_all); };
  auto tile_base = [&](auto is_v_c, uint32_t tile) __attribute__((always_inline)) -> uint64_t {
    constexpr bool IS_V = decltype(is_v_c)::value;
    return uniform_address((IS_V ? vbase : kbase) + (int64_t)kv_slot(p.ring_mask, tile * kBlockN) * (IS_V ? vstride_b : kstride_b));
  };
  // group g of G blocks of a tile at `base`
  auto issue_group = [&](auto is_v_c, auto size_c, auto g_c, uint64_t base) __attribute__((always_inline)) {
    constexpr bool IS_V = decltype(is_v_c)::value;
    constexpr int G = decltype(size_c)::value, g = decltype(g_c)::value, BLK = IS_V ? L::V_BLK : L::K_BLK;
    const uint64_t stride_b = IS_V ? vstride_b : kstride_b;
    lds_dma_group<G, g * G * BLK, BLK>(base + (uint64_t)(g * G) * stride_b, stride_b - BLK, IS_V ? voff : koff, IS_V ? my_v : my_k);
  };
  // The same for an edge tile: every row that must not be read is replaced by the nearest one that may.
  auto issue_edge = [&](auto is_v_c, uint32_t tile) __attribute__((always_inline)) {
    constexpr bool IS_V = decltype(is_v_c)::value;
    constexpr int BLK = IS_V ? L::V_BLK : L::K_BLK, G = NBLK >= 4 ? 4 : NBLK;
    constexpr uint32_t BIAS = 4096;   // keeps the compensated offsets positive
    const uint32_t stride_b = (uint32_t)(IS_V ? vstride_b : kstride_b);
    const uint64_t base = tile_base(is_v_c, tile) - BIAS;
    const TileRows rows = tile_rows(tile * kBlockN, lo_min, p.t_all);
    const uint32_t lo = rows.first * stride_b + lcol, hi = rows.last * stride_b + lcol;
    static_for<0, NBLK / G>([&](auto g_c) {
      constexpr int g = decltype(g_c)::value;
      uint32_t off[4];
#pragma unroll
      for (int i = 0; i < G; ++i)
        asm("v_med3_u32 %0, %1, %2, %3" : "=v"(off[i]) : "v"((IS_V ? voff : koff) + (uint32_t)(g * G + i) * stride_b), "v"(lo), "v"(hi));
#pragma unroll
      for (int i = 0; i < G; ++i) off[i] += BIAS - (uint32_t)(i * BLK);
      ws_issue_clamped<G, g * G * BLK, BLK>(base, off, IS_V ? my_v : my_k);
    });
  };
  constexpr int GK = NBLK >= 4 ? 4 : NBLK, GV = 2;
  auto issue_k = [&](uint32_t tile) __attribute__((always_inline)) {
    if (__builtin_expect(is_edge(tile), 0)) {
      issue_edge(std::false_type{}, tile);
    } else {
      const uint64_t base = tile_base(std::false_type{}, tile);
      static_for<0, NBLK / GK>([&](auto g_c) { issue_group(std::false_type{}, std::integral_constant<int, GK>{}, g_c, base); });
    }
  };
  // ---- rows that will come from HBM (AttnParams.touch_ahead says so): the key range is touched into the L2 first.  With
  // one buffer per matrix a tile's loads have half a tile's time to land, which covers the L2 and not HBM (a 30-layer loop,
  // 1.1 GB of caches: 1842 us an iteration without, 1768 with; at a 2k prefix 922 and 846).  The workgroups of a KV head
  // sit behind one L2 and stream the same keys, so they share the work: one instruction is 64 lines of 128 bytes, K's
  // first, then V's, dealt out to the waves; what does not fit NTOUCH rounds of them stays untouched.  A touch is a load
  // into a dump area nobody reads. ----
  constexpr int NTOUCH = 4;
  const uint32_t pos0 = max(mt_begin * kBlockN, lo_min), pos1 = min(mt_end * kBlockN, p.t_all);
  if (args.touch && pos0 < pos1) {   // (rows that see no key have none to touch: their range may begin past the last one)
    constexpr uint32_t LPRW = 2 * D >= 128 ? 2 * D / 128 : 1, RPT = 64 / LPRW;   // lines per row, rows per touch
    const uint32_t per_matrix = (pos1 - pos0 + RPT - 1u) / RPT;
    const uint32_t dump = lds0 + (uint32_t)OFF_DUMP + wave * 256u;
#pragma unroll 1
    for (uint32_t t = 0; t < (uint32_t)NTOUCH; ++t) {
      const uint32_t u = min(rt * 4u + wave + t * 4u * args.n_rt, 2u * per_matrix - 1u);   // (past the end: the last one again)
      const bool is_v = u >= per_matrix;
      const uint32_t pos = touched_pos(pos0, pos1, RPT, is_v ? u - per_matrix : u, lane / LPRW);
      const uint32_t first = p.ring_mask ? 0u : pos0;     // (32-bit offsets from the ring's first slot or the range's first key)
      const int64_t stride_b = is_v ? vstride_b : kstride_b;
      lds_dma_touch((is_v ? vbase : kbase) + (int64_t)first * stride_b,
                    (kv_slot(p.ring_mask, pos) - first) * (uint32_t)stride_b + (lane % LPRW) * 128u, dump);
    }
  }
  // ---- Q fragments: B operand of S^T = K.Q^T, lane = row, 8 consecutive d per step.  The rows come in
  // through LDS as whole rows, in the layout of a K tile, the KiB blocks dealt out to the waves; every wave
  // then reads its 32 rows the way it reads K fragments. ----
  u32x4 qf[MR][NSTEP];
  {
    constexpr int NQ = (MR * NBLK + 3) / 4;   // blocks per wave
    const char* qbase = (const char*)p.q + (size_t)kvh * p.group * (2 * D);
    const bool convert = F16 && p.q_is_bf16;
    u32x4 raw[NQ];
    static_for<0, NQ>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      const uint32_t b = wave * (uint32_t)NQ + i, m = b / NBLK, bm = b & (uint32_t)(NBLK - 1);   // block bm of row block m
      const uint32_t qr = min(row0 + m * 32u + bm + lgrp * (uint32_t)NBLK, p.rows_total - 1u);   // (past the last row: repeat it)
      const uint32_t off = (qr + fast_div(qr, args.div_group) * (p.hq - p.group)) * (uint32_t)(2 * D) + lcol;
      if (MR * NBLK >= 4 || b < (uint32_t)(MR * NBLK)) {
        if (convert) raw[i] = *(const u32x4*)(qbase + off);
        else lds_dma_16<0>(qbase, off, lds0 + off_q(m) + bm * (uint32_t)L::K_BLK);
      }
    });
    if (ntile > 0) issue_k(tb);   // the first K tile right behind the query rows
    if (convert) {   // bf16 queries over an f16 cache: converted once, on the way in
      static_for<0, NQ>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        const uint32_t b = wave * (uint32_t)NQ + i, m = b / NBLK, bm = b & (uint32_t)(NBLK - 1);
        u32x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = pack2<true>(__uint_as_float(raw[i][e] << 16), __uint_as_float(raw[i][e] & 0xffff0000u));
        if (MR * NBLK >= 4 || b < (uint32_t)(MR * NBLK))
          *(lds_u32x4*)((lds_char*)smem + off_q(m) + bm * (uint32_t)L::K_BLK + lane * 16u) = h;
      });
    }
  }
  // this lane's query rows and their key bounds (rows past the last one are copies of it that nobody stores)
  RowBounds rb[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) rb[m] = row_bounds(p, fast_div(min(row0 + 32u * m + l32, p.rows_total - 1u), args.div_group));
  // per-lane LDS byte offsets of the fragment reads; everything else is a compile-time offset
  const uint32_t k_lane_off = (l32 & (uint32_t)(NBLK - 1)) * L::K_BLK + l32 / NBLK * L::ROWB + g2 * 16u;
  const uint32_t v_row = 4u * g2 + (i16 >> 2);   // below 8
  const uint32_t v_lane_off = (v_row & (uint32_t)(NBLK - 1)) * L::V_BLK + v_row / NBLK * L::ROWB + (2u * h16 + ((i16 & 3u) >> 1)) * 16u +
                              (i16 & 1u) * 8u;
  // (Over a bf16 cache at head_dim 256 by MFMAs: the compiler put the 128 register writes between the first scores and the
  // first tile, 0.2 - 0.3 us of a launch.  Over an f16 cache its other choices with them cost 0.3, and 64 rows spill.)
  f32x16 o[MR][NDB];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
      if constexpr (D == 256 && MR == 1 && !F16) {
        mfma_zero(o[m][i]);
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) o[m][i][e] = 0.f;
      }
    }
  __builtin_amdgcn_sched_barrier(0);   // (all of the above while the loads are on their way)
  wait_vmem_all();
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) qf[m][st] = *(lds_u32x4*)((lds_char*)smem + off_q(m) + k_lane_off + 32 * st);
  if constexpr (MR > 1) __syncthreads();   // the query rows are read: the V tiles may take their place

  float m_ref[MR], m_run[MR];       // reference max of the row in use, log2 units (scale folded in), and running max itself
  float l_part[MR], l_part2[MR];    // this lane's share of the row sum (its 16 of every 32 keys)
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    m_ref[m] = m_run[m] = -INFINITY;
    l_part[m] = l_part2[m] = 0.f;
  }
  lds_char* const kb = (lds_char*)smem + wave * (uint32_t)L::SLICE + k_lane_off;   // this wave's tiles, plus the lane's offset
  lds_char* const vb = (lds_char*)smem + wave * (uint32_t)L::SLICE + L::K_BYTES + v_lane_off;
  // K fragment of MFMA step st: A operand, lane = key row l32, 8 consecutive d at 16 st + 8 g2
  auto k_frag = [&](int st) -> u32x4 { return *(lds_u32x4*)(kb + 32 * st); };
  // V^T fragment of k-step ks, d-block db: k-slot j of lane half g2 is key 16 ks + 8 (j>>2) + 4 g2 + (j&3),
  // the order in which the score accumulator holds a lane's keys
  auto v_frag = [&](int ks, int db) -> u32x4 {
    const u32x2 lo = __builtin_bit_cast(
        u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vb + L::v_row8(2 * ks) + 64 * db)));
    const u32x2 hi = __builtin_bit_cast(
        u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vb + L::v_row8(2 * ks + 1) + 64 * db)));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };

  // S^T = K.Q^T of the tile in the K buffer.  The score MFMAs are assembly with an ordinary register tuple as
  // accumulator: left to the compiler they accumulate in the same register class as O, and O then moves
  // between the classes around every tile.  Fragment reads run PFK steps ahead of the MFMA that consumes them
  // (the loads between the MFMAs are assembly the compiler will not move LDS reads across, so the distance is
  // spelled out).  `between(st)` is what follows MFMA st in program order.
  f32x16 s[MR];
  auto scores = [&](auto&& between) __attribute__((always_inline)) {
    constexpr int PFK = MR > 1 ? 2 : NSTEP < 4 ? NSTEP : 4;
    u32x4 kf[PFK];
#pragma unroll
    for (int i = 0; i < PFK; ++i) kf[i] = k_frag(i);
    static_for<0, NSTEP>([&](auto st_c) {
      constexpr int st = decltype(st_c)::value;
      static_for<0, MR>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value;
        if constexpr (st == 0) mfma_scores_first<F16>(s[m], kf[0], qf[m][0]);
        else if constexpr (st == NSTEP - 1 && m == MR - 1) mfma_scores_last<F16>(s[m], kf[st % PFK], qf[m][st]);
        else mfma_scores_acc<F16>(s[m], kf[st % PFK], qf[m][st]);
      });
      if constexpr (st + PFK < NSTEP) kf[st % PFK] = k_frag(st + PFK);
      between(st_c);
    });
    // every K fragment is in registers: the buffer may take the next tile
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // masks an edge tile's scores and returns the tile max of the row's half
  auto mask_and_max = [&](auto m_c, uint32_t t0) __attribute__((always_inline)) -> float {
    constexpr int m = decltype(m_c)::value;
    f32x16& sm = s[m];
    if (__builtin_expect(!(t0 >= lo_max && t0 + kBlockN <= hi_min), 0)) {
      // lane's keys are t0 + 4 g2 + c, c = 8 (e >> 2) + (e & 3): visible iff c - (lo - first) < hi - lo, unsigned
      const uint32_t first = t0 + 4u * g2, hi = min(rb[m].hi, p.t_clip_hi);
      const uint32_t from = rb[m].lo - first, len = hi > rb[m].lo ? hi - rb[m].lo : 0u;
      if (__builtin_expect(p.extra_lo < p.t_clip_hi, 0)) {   // some rows see a second range
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (!key_visible(rb[m], first + 8u * (e >> 2) + (e & 3), p.t_clip_hi)) sm[e] = -INFINITY;
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) sm[e] = 8u * (e >> 2) + (e & 3) - from < len ? sm[e] : -INFINITY;
      }
    }
    const float a0 = fmaxf(fmaxf(sm[0], sm[1]), sm[2]), a1 = fmaxf(fmaxf(sm[3], sm[4]), sm[5]);
    const float a2 = fmaxf(fmaxf(sm[6], sm[7]), sm[8]), a3 = fmaxf(fmaxf(sm[9], sm[10]), sm[11]);
    const float a4 = fmaxf(fmaxf(sm[12], sm[13]), sm[14]);
    return fmaxf(fmaxf(fmaxf(a0, a1), a2), fmaxf(fmaxf(a3, a4), sm[15]));
  };
  // ---- online softmax with a lazily raised reference max: the tile's probabilities in the MFMA's operand layout ----
  u32x4 pk[MR][2];
  auto raise_reference = [&](auto m_c, float tmax) __attribute__((always_inline)) {
    constexpr int m = decltype(m_c)::value;
    tmax = max_across_halves(tmax) * p.scale_log2;
    const bool raise = __builtin_amdgcn_ballot_w64(tmax > m_ref[m] + kWsTau<F16>) != 0ull;
    m_run[m] = fmaxf(m_run[m], tmax);
    if (__builtin_expect(raise, 0)) {
      // one row has to raise its reference: every row moves up to its running max (the block is rescaled
      // anyway, and the next raise is then as far away as it can be)
      const float m_new = fmaxf(m_ref[m], m_run[m] + kWsLead<F16>);
      const float corr = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m_ref[m] - m_new);
      const bool rescale = __builtin_amdgcn_ballot_w64(m_ref[m] != -INFINITY && corr != 1.f) != 0ull;
      l_part[m] *= corr;
      l_part2[m] *= corr;
      if (rescale) {   // O stays in the accumulation registers: spelled out, or the allocator moves all of it
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
          for (int e = 0; e < 16; e += 8) {
            float x0 = o[m][i][e], x1 = o[m][i][e + 1], x2 = o[m][i][e + 2], x3 = o[m][i][e + 3];
            float x4 = o[m][i][e + 4], x5 = o[m][i][e + 5], x6 = o[m][i][e + 6], x7 = o[m][i][e + 7];
            scale_acc8(x0, x1, x2, x3, x4, x5, x6, x7, corr);
            o[m][i][e] = x0;
            o[m][i][e + 1] = x1;
            o[m][i][e + 2] = x2;
            o[m][i][e + 3] = x3;
            o[m][i][e + 4] = x4;
            o[m][i][e + 5] = x5;
            o[m][i][e + 6] = x6;
            o[m][i][e + 7] = x7;
          }
        scale_acc_done();
      }
      m_ref[m] = m_new;
    }
  };
  // The probabilities are 2^(score - reference - offset): with bf16 the offset puts a weight 2^40 below the
  // reference (and so below the row's largest) under the smallest normal number, an exact zero.  Scores 4 q .. 4 q + 3.
  auto probs = [&](auto m_c, auto q_c) __attribute__((always_inline)) {
    constexpr int m = decltype(m_c)::value, q = decltype(q_c)::value;
    const float m_use = (m_ref[m] == -INFINITY) ? 0.f : m_ref[m] + kWsPOff<F16>;
    float ex[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ex[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[m][4 * q + i], p.scale_log2, -m_use));
    const uint32_t a = pack2<F16>(ex[0], ex[1]), b = pack2<F16>(ex[2], ex[3]);
    pk[m][q >> 1][(2 * q) & 3] = a;
    pk[m][q >> 1][(2 * q + 1) & 3] = b;
    // the row sum uses the rounded probabilities, the same numbers P.V multiplies
    l_part[m] = ws_add_pair<F16>(a, l_part[m]);
    l_part2[m] = ws_add_pair<F16>(b, l_part2[m]);
  };
  // O^T += V^T.P^T, a V fragment serving every row block
  auto pv = [&](auto ks_c, auto&& between) __attribute__((always_inline)) {
    constexpr int ks = decltype(ks_c)::value;
    static_for<0, NDB>([&](auto db_c) {
      constexpr int db = decltype(db_c)::value;
      const u32x4 vf = v_frag(ks, db);
#pragma unroll
      for (int m = 0; m < MR; ++m) o[m][db] = mfma16<F16>(vf, pk[m][ks], o[m][db]);
      between(db_c);
    });
  };
  // scores of `tile` (its K has landed) with the loads of its V, two at a time, between them: they have the rest of the
  // scores, the issue of the next K tile and the softmax to land
  auto scores_and_v = [&](uint32_t tile) __attribute__((always_inline)) {
    const bool edge = is_edge(tile);
    uint64_t base = 0;
    if (__builtin_expect(edge, 0)) issue_edge(std::true_type{}, tile);
    else base = tile_base(std::true_type{}, tile);
    scores([&](auto st_c) {
      constexpr int st = decltype(st_c)::value;
      if constexpr (st % 2 == 0 && st / 2 < NBLK / GV) {
        if (!edge) issue_group(std::true_type{}, std::integral_constant<int, GV>{}, std::integral_constant<int, st / 2>{}, base);
      }
    });
  };

  if (ntile > 0) scores_and_v(tb);
  for (uint32_t jj = 0; jj < ntile; ++jj) {
    const uint32_t tile = tb + jj;
    const bool more = jj + 1u < ntile;
    float tmax[MR];
    static_for<0, MR>([&](auto m_c) { tmax[decltype(m_c)::value] = mask_and_max(m_c, tile * kBlockN); });
    // The scores of this tile are read (the K buffer was free since they existed): the next K tile's loads, all of
    // them here, behind the tile max and ahead of everything that depends on it.  (Between the softmax and P.V
    // instructions, one at a time, they land too late for the next scores: 22.4 -> 24.3 us for a sliding layer's step.)
    if (more) issue_k(tile + 1u);
    static_for<0, MR>([&](auto m_c) { raise_reference(m_c, tmax[decltype(m_c)::value]); });
    static_for<0, MR>([&](auto m_c) {
      probs(m_c, std::integral_constant<int, 0>{});
      probs(m_c, std::integral_constant<int, 1>{});
    });
    // V(jj) has landed (the loads of K(jj+1), issued after it, may still be on their way)
    if (more) wait_vmem_but<NBLK>();
    else wait_vmem_all();
    // With 64 rows the probabilities of the last 16 keys are worked out between the products of the first 16 (901 causal rows 27.6
    // -> 26.7 us, 700 over an f16 cache 36.5 -> 35.1); with 32 rows the load path sets the pace, and the wave gets to the next
    // loads' wait that much earlier for nothing (256 rows 17.8 -> 18.1).
    constexpr int PIECES = 2 * MR, PER = NDB >= PIECES ? NDB / PIECES : 1;
    constexpr bool BETWEEN = MR > 1 && NDB >= PIECES;
    if constexpr (!BETWEEN)
      static_for<0, PIECES>([&](auto x_c) {
        probs(std::integral_constant<int, decltype(x_c)::value / 2>{}, std::integral_constant<int, 2 + decltype(x_c)::value % 2>{});
      });
    pv(std::integral_constant<int, 0>{}, [&](auto db_c) {
      constexpr int db = decltype(db_c)::value;
      if constexpr (BETWEEN && db % PER == 0 && db / PER < PIECES) {
        probs(std::integral_constant<int, db / PER / 2>{}, std::integral_constant<int, 2 + db / PER % 2>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    pv(std::integral_constant<int, 1>{}, [](auto) {});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the V buffer is free for the next tile's loads
    if (more) {
      wait_vmem_all();   // K(jj+1), the only load outstanding
      scores_and_v(tile + 1u);
    }
  }
  wait_vmem_all();   // (only when ntile == 0 is there nothing to wait for; cheap either way)

  // ---- the four waves' (m, l, O) of every row meet in LDS ----
  // The accumulators of a wave are D / 8 units of four registers per row block (unit u: d 8 u + 4 g2 .. + 3 of the lane's
  // row).  Every wave finishes a quarter of the units: it keeps its own, sends the others to their finishers (in register
  // order, a KiB per unit), and adds up what it is sent.  LDS writes run at half the rate of reads, so what is not written
  // is what counts.  One row block after the other.
  constexpr int NU = D / 8, UPW = NU / 4;
  constexpr int OFF_T = 3 * NU * 1024, T_ROW = 4 * D + 16;   // finished rows, on their way to whole-row stores
  static_assert(OFF_T + 32 * T_ROW <= 4 * L::SLICE, "the tiles' LDS holds both");
  const bool f32_out = SHARED || p.out_dtype == DT_F32;
  const uint32_t cpr = f32_out ? D / 4 : D / 8;            // 16-byte chunks per row (a power of two)
  const uint32_t tok0 = fast_div(row0, args.div_group);
  // Workgroups that share a row tile leave fp32 rows relative to their (m, l), as the split kernel does, for its merge.
  const size_t prow0 = ((size_t)split * p.hkv + kvh) * p.rows_pad + row0;
  const auto out_win = SHARED ? wt_window(p.part_o + prow0 * D)
                             : wt_window((const char*)p.out + ((size_t)tok0 * p.hq + kvh * p.group) * (f32_out ? 4u * D : 2u * D));
#pragma unroll 1   // (one copy of the code: what is fetched for the first row block serves the second)
  for (uint32_t mb = 0; mb < (uint32_t)MR; ++mb) {
  const uint32_t r = row0 + 32u * mb + l32;
  __syncthreads();   // every wave is done with its tiles (with the previous row block)
  f32x4 y[UPW];
  // (accumulators are registers: their numbers are compile-time constants, so this much is there once per row block)
  auto send = [&](auto m_c) __attribute__((always_inline)) {
  constexpr int m = decltype(m_c)::value;
  {
    const float l_tot = sum_across_halves(l_part[m] + l_part2[m]);
    const u32x2 ml = {__float_as_uint(m_ref[m] + kWsPOff<F16>), __float_as_uint(l_tot)};   // (the exponent the sums are relative to)
    if (g2 == 0) *(__attribute__((address_space(3))) u32x2*)((lds_char*)smem + OFF_ML + (wave * 32u + l32) * 8u) = ml;
  }
  static_for<0, 4>([&](auto d_c) {
    constexpr int dst = decltype(d_c)::value;
    auto unit = [&](auto u_c) -> f32x4 {
      constexpr int u = dst * UPW + decltype(u_c)::value, i = u / 4, e = 4 * (u % 4);
      return f32x4{o[m][i][e], o[m][i][e + 1], o[m][i][e + 2], o[m][i][e + 3]};
    };
    if (wave == (uint32_t)dst) {
      static_for<0, UPW>([&](auto u_c) {
        constexpr int u = dst * UPW + decltype(u_c)::value;
        y[u - dst * UPW] = acc_read4<true>(o[m][u / 4], 4 * (u % 4));   // (read here and not, all of O, at the loop's exit)
      });
    } else {
      lds_char* const to = (lds_char*)smem + ((uint32_t)(dst * 3) + (wave < (uint32_t)dst ? wave : wave - 1u)) * (uint32_t)(UPW * 1024) + lane * 16u;
      static_for<0, UPW>([&](auto u_c) { *(__attribute__((address_space(3))) f32x4*)(to + decltype(u_c)::value * 1024) = unit(u_c); });
    }
  });
  };
  if (MR == 1 || mb == 0u) send(std::integral_constant<int, 0>{});
  else send(std::integral_constant<int, MR - 1>{});
  __syncthreads();
  {
    // weights of the lane's row: 2^(m_i - m) / l for the waves that saw a key of it
    float mi[4], li[4], w[4];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x2 ml = *(__attribute__((address_space(3))) u32x2*)((lds_char*)smem + OFF_ML + (i * 32u + l32) * 8u);
      mi[i] = __uint_as_float(ml[0]);
      li[i] = __uint_as_float(ml[1]);
      mx = li[i] > 0.f ? fmaxf(mx, mi[i]) : mx;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = li[i] > 0.f ? __builtin_amdgcn_exp2f(mi[i] - mx) : 0.f;
    const float den = (w[0] * li[0] + w[1] * li[1]) + (w[2] * li[2] + w[3] * li[3]);
    const bool den_ok = den > 0.f;
    const float inv = SHARED ? 1.f : den_ok ? __builtin_amdgcn_rcpf(den) : 0.f;
    if constexpr (SHARED) {
      if (wave == 0 && g2 == 0) wt_store8(wt_window(p.part_ml + prow0 * 2), l32 * 8u, u32x2{__float_as_uint(mx), __float_as_uint(den)});
    } else if ((p.lse || p.dbg) && wave == 0 && g2 == 0 && r < p.rows_total) {
      const uint32_t tok = fast_div(r, args.div_group), qh = kvh * p.group + r - tok * p.group;
      if (p.lse) p.lse[(size_t)tok * p.hq + qh] = den_ok ? mx * kLn2 + __logf(den) : -INFINITY;
      if (p.dbg && !den_ok) dbg_report(p.dbg, DBG_ERR_SOFTMAX_NORM_ZERO, DBG_KERNEL_ATTENTION, (tok << 16) | qh, (tok << 16) | qh);
    }
    // (a wave that saw no key of the row holds exact zeros there and gets weight zero)
    const float w_own = wave == 0 ? w[0] : wave == 1 ? w[1] : wave == 2 ? w[2] : w[3];
#pragma unroll
    for (int u = 0; u < UPW; ++u) y[u] *= w_own * inv;
#pragma unroll
    for (int j = 0; j < 3; ++j) {   // the other waves, in order
      const float wj = (wave <= (uint32_t)j ? w[j + 1] : w[j]) * inv;
      lds_char* const from = (lds_char*)smem + (wave * 3u + (uint32_t)j) * (uint32_t)(UPW * 1024) + lane * 16u;
#pragma unroll
      for (int u = 0; u < UPW; ++u) {
        const f32x4 x = *(__attribute__((address_space(3))) f32x4*)(from + u * 1024);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[u][e] = __builtin_fmaf(wj, x[e], y[u][e]);
      }
    }
  }
  {
    lds_char* const to = (lds_char*)smem + OFF_T + l32 * (uint32_t)T_ROW;
    const uint32_t d0 = wave * (uint32_t)(UPW * 8) + g2 * 4u;
    if (f32_out) {
#pragma unroll
      for (int u = 0; u < UPW; ++u) *(__attribute__((address_space(3))) f32x4*)(to + (d0 + u * 8u) * 4u) = y[u];
    } else if (p.out_trunc) {
#pragma unroll
      for (int u = 0; u < UPW; ++u) {
        const u32x2 h = {(__float_as_uint(y[u][0]) >> 16) | (__float_as_uint(y[u][1]) & 0xffff0000u),
                         (__float_as_uint(y[u][2]) >> 16) | (__float_as_uint(y[u][3]) & 0xffff0000u)};
        *(__attribute__((address_space(3))) u32x2*)(to + (d0 + u * 8u) * 2u) = h;
      }
    } else {
#pragma unroll
      for (int u = 0; u < UPW; ++u)
        *(__attribute__((address_space(3))) u32x2*)(to + (d0 + u * 8u) * 2u) = u32x2{pack2<false>(y[u][0], y[u][1]), pack2<false>(y[u][2], y[u][3])};
    }
  }
  __syncthreads();
  // ---- whole rows out, 16 bytes per lane, written through (wt_store.h): the next kernel reads these rows, and a kernel
  // does not end before the lines it left dirty in its L2 are written back ----
#pragma unroll 4
  for (uint32_t c = threadIdx.x; c < 32u * cpr; c += 256u) {
    const uint32_t rl = c / cpr, ch = c & (cpr - 1u);
    const u32x4 h = *(lds_u32x4*)((lds_char*)smem + OFF_T + rl * (uint32_t)T_ROW + ch * 16u);
    const uint32_t rr = row0 + 32u * mb + rl;
    if constexpr (SHARED) {
      wt_store16(out_win, (rl * cpr + ch) * 16u, h);
      continue;
    }
    if (rr >= p.rows_total) break;
    const uint32_t tok = fast_div(rr, args.div_group), g = rr - tok * p.group;
    if (p.dbg) {   // a NaN or infinity among the chunk's elements: an all-ones exponent carries into the top bit
      uint32_t t[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        t[e] = f32_out ? ((h[e] & 0x7fffffffu) + 0x00800000u) & 0x80000000u : ((h[e] & 0x7fff7fffu) + 0x00800080u) & 0x80008000u;
      if ((t[0] | t[1]) | (t[2] | t[3]))   // (named by fours, as an accumulator holds them: a chunk of 16-bit elements is two)
        dbg_report(p.dbg, DBG_ERR_NONFINITE, DBG_KERNEL_ATTENTION, (tok << 16) | (kvh * p.group + g),
                   f32_out ? ch * 4u : ch * 8u + (t[0] | t[1] ? 0u : 4u));
    }
    wt_store16(out_win, (((tok - tok0) * p.hq + g) * cpr + ch) * 16u, h);
  }
  }
}

template <int D, bool F16, int MR, bool SHARED = false>
hipError_t launch_rows(const AttnParams& p, hipStream_t s) {
  WsArgs a;
  a.p = p;
  a.n_rt = (p.rows_total + 32 * MR - 1) / (32 * MR);
  a.div_rt = make_fast_div(a.n_rt);
  a.div_group = make_fast_div(p.group);
  a.div_splits = make_fast_div(p.n_splits);
  // (touches use 32-bit byte offsets: a range or ring whose rows span 4 GiB goes without)
  const uint64_t rows = p.ring_mask ? (uint64_t)p.ring_mask + 1u : (uint64_t)(p.tile_end - p.tile_first + 2u) * kBlockN;
  a.touch = p.touch_ahead && rows * 2u * (uint64_t)std::max(p.k_tok_stride, p.v_tok_stride) < (1ull << 32) ? 1u : 0u;
  const uint32_t grid = ((p.hkv * p.n_splits * a.n_rt + 7u) / 8u) * 8u;
  hipLaunchKernelGGL((attn_wsplit_kernel<D, F16, MR, SHARED>), dim3(grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <int D, bool F16>
hipError_t launch_ws(const AttnParams& p, hipStream_t s) {
  // 32 rows per workgroup while they are one round of the chip's compute units (one workgroup each: LDS); past that 64
  // rows, whose workgroups take 1.6 x as long for twice the rows, where that is fewer rounds' time.  (Sliding layer, step
  // in us, 32 | 64 rows: 256 canvas rows = 128 workgroups of 32: 21.0 | 31.0; 901 rows = 456: 40.3 | 33.8.)
  const uint32_t cus = p.cus, r1 = (p.hkv * ((p.rows_total + 31u) / 32u) + cus - 1u) / cus;
  const uint32_t r2 = (p.hkv * ((p.rows_total + 63u) / 64u) + cus - 1u) / cus;
  if constexpr (D == 256) {
    if (p.n_splits > 1u) return launch_rows<D, F16, 1, true>(p, s);
  }
  if (8u * r2 < 5u * r1) return launch_rows<D, F16, 2>(p, s);
  return launch_rows<D, F16, 1>(p, s);
}

}  // namespace

hipError_t launch_attn_wsplit(const AttnParams& p, uint32_t head_dim, uint32_t kv_dtype, hipStream_t s) {
  const bool f16 = kv_dtype == DT_F16;
  switch (head_dim) {
    case 32: return f16 ? launch_ws<32, true>(p, s) : launch_ws<32, false>(p, s);
    case 64: return f16 ? launch_ws<64, true>(p, s) : launch_ws<64, false>(p, s);
    case 128: return f16 ? launch_ws<128, true>(p, s) : launch_ws<128, false>(p, s);
    case 256: return f16 ? launch_ws<256, true>(p, s) : launch_ws<256, false>(p, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dg
