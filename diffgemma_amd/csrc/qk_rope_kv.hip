// The producer of the cache rows attention reads: per-head RMSNorm + RoPE + KV-cache write for
// the canvas rows of one layer (reference: src/shaders/attn/qk_rope_kv/qk_rope_kv.metal:29-149,
// CPU twin src/shaders/attn/cpu.rs:78-145).
//
// A wave owns NR rows (canvas row, head), heads = Hq query heads, then Hkv key heads, then Hkv value heads as in the
// reference's grid (enc.rs:1794-1804); the four waves of a workgroup share the canvas row and with it one table of cos
// and sin.  A row (at most 1 KiB) is read once with up to 16-byte loads, normalised and rotated in registers (the
// partner of element d, hd/2 + d, sits in the lane 32 away), and written once: Q (and K, unless V aliases it) back in
// place as bf16, K and V into the cache at slot(pos) in the cache's element type.  Every byte moves once.  At 256 canvas
// rows (9 MB) the launch is one wave's chain: launch, arguments, row, sum, rotation, store; 3.4 - 3.6 us where an empty
// kernel takes 1.8.  At 1024 rows it is HBM-bound: 7.4 us for the 42 MB of a global layer, 8.0 for the 38 MB of a sliding
// one.  Half of what it took before (5.1 us and 12 - 15 us) was instructions: rows staged through LDS for the rotation,
// shuffles for the row sum, storage rounding in integer arithmetic, a correctly rounded root and quotient.
#include "attn_params.h"
#include "mfma_tile.h"
#include "wt_store.h"
#include "../../include/dg_attn.h"

namespace dg {
namespace {

struct RopeParams {
  uint16_t* q;           // [canvas][hq][hd] bf16, in place
  uint16_t* k;           // [canvas][hkv][hd] bf16, in place unless v_from_k
  const uint16_t* v;     // [canvas][hkv][hd] bf16 (unused when v_from_k)
  void* kc;              // cache region + K offset
  void* vc;              // cache region + V offset
  const uint16_t* qw;    // [hd] bf16 norm weights
  const uint16_t* kw;
  uint32_t* dbg;
  const uint32_t* step_dev;   // device copy of the reference's StepParams, or null: kv_len (word 0) and kv_write_end
                              // (word 11) are then read from it when the kernel runs
  int64_t k_tok_stride, k_head_stride, v_tok_stride, v_head_stride;  // elements
  uint32_t canvas, hq, hkv, hd;
  uint32_t kv_len, kv_write_end, ring_mask;
  uint32_t is_full, v_from_k, kv_dtype, qk_trunc;
};

// theta^(-2 d / hd), the angle of pair d per position.  -2 d / hd is a multiple of 1/256 for every head_dim, so one table
// per theta serves them all (entry d * 512 / hd).  Worked out in double precision and rounded once, which is what the C
// library's powf of the reference's CPU twin returns (cpu.rs:35,57): the angle pos * inv_freq is an fp32 product, and at
// pos ~ 1e5 one unit in the last place of inv_freq moves it by a hundredth of a radian, so it must not depend on the
// device's pow.  A constant of the code object and not a kernel argument: 1 KiB of arguments per launch is read by every
// workgroup from host-visible memory.
struct InvFreq {
  float split[256];          // theta 1e4: whole head
  float proportional[64];    // theta 1e6: first quarter of the head
};
constexpr double const_sqrt(double x) {
  double r = x > 1.0 ? x : 1.0;
  for (int i = 0; i < 64; ++i) r = 0.5 * (r + x / r);
  return r;
}
constexpr InvFreq make_inv_freq() {
  double r128 = 10.0;                                     // 10^(1/128)
  for (int i = 0; i < 7; ++i) r128 = const_sqrt(r128);
  const double r64 = r128 * r128, r3 = r128 * r128 * r128;   // theta^(1/256): 1e4 -> 10^(4/256), 1e6 -> 10^(6/256)
  InvFreq t{};
  double x = 1.0;
  for (int d = 0; d < 256; ++d, x *= r64) t.split[d] = (float)(1.0 / x);
  x = 1.0;
  for (int d = 0; d < 64; ++d, x *= r3) t.proportional[d] = (float)(1.0 / x);
  return t;
}
__constant__ constexpr InvFreq kInvFreq = make_inv_freq();

// Sum over the wave, in every lane.  Lane exchanges on the vector unit (DPP, permlane swaps): six dependent steps of a few
// cycles each, where the LDS crossbar (shuffles) takes a round trip per step.
template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) {
  const int u = __builtin_bit_cast(int, v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(u, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
  v = add_dpp<0xB1>(v);    // quad_perm 1,0,3,2
  v = add_dpp<0x4E>(v);    // quad_perm 2,3,0,1
  v = add_dpp<0x141>(v);   // row_half_mirror
  v = add_dpp<0x140>(v);   // row_mirror
  uint32_t u = __float_as_uint(v);
  auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  u = __float_as_uint(v);
  auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// 1 / sqrt(a), the hardware estimate and one Newton step in fused arithmetic: within an ulp, like a correctly rounded
// root followed by a correctly rounded quotient, in a fifth of the instructions.  a = inf gives 0.
__device__ __forceinline__ float inv_sqrt(float a) {
  const float r = __builtin_amdgcn_rsqf(a);
  const float e = __builtin_fmaf(-a * r, r, 1.0f);
  return a < INFINITY ? __builtin_fmaf(0.5f * r, e, r) : r;
}

constexpr float kRmsEps = 1e-6f;   // cpu.rs:3, attention_device.metal:10

// One row of `hd` bf16 elements, `per` = hd/64 consecutive ones per lane, moved with the widest access the count allows
// (16 bytes at hd 512).  Load and conversion are apart so that several rows' loads can be in flight before the first
// is looked at.
template <int PER>
struct RawRow {
  uint32_t w[PER >= 2 ? PER / 2 : 1];
};
template <int PER>
__device__ __forceinline__ RawRow<PER> load_raw(const uint16_t* src) {
  RawRow<PER> r;
  if constexpr (PER == 8) {
    const uint4 v = *(const uint4*)src;
    r.w[0] = v.x;
    r.w[1] = v.y;
    r.w[2] = v.z;
    r.w[3] = v.w;
  } else if constexpr (PER == 4) {
    const uint2 v = *(const uint2*)src;
    r.w[0] = v.x;
    r.w[1] = v.y;
  } else if constexpr (PER == 2) {
    r.w[0] = *(const uint32_t*)src;
  } else {
    r.w[0] = src[0];
  }
  return r;
}
template <int PER>
__device__ __forceinline__ float raw_elem(const RawRow<PER>& r, int i) {
  return __uint_as_float(i & 1 ? r.w[i / 2] & 0xffff0000u : r.w[i / 2] << 16);
}

// The same for results: `per` consecutive elements as 16-bit storage values (the conversions are the hardware's packed
// ones; spelled out with integer arithmetic they were half of the kernel's instructions) ...
enum RowFormat { ROW_BF16, ROW_BF16_TRUNC, ROW_F16 };
template <int PER>
__device__ __forceinline__ RawRow<PER> pack_row(const float (&y)[PER], RowFormat f) {
  constexpr int NW = PER >= 2 ? PER / 2 : 1, LAST = PER >= 2 ? 1 : 0;
  RawRow<PER> r;
  if (f == ROW_F16) {   // kv_store: half(v), round to nearest
#pragma unroll
    for (int i = 0; i < NW; ++i) r.w[i] = pack2<true>(y[2 * i], y[2 * i + LAST]);
  } else if (f == ROW_BF16) {
#pragma unroll
    for (int i = 0; i < NW; ++i) r.w[i] = pack2<false>(y[2 * i], y[2 * i + LAST]);
  } else {
#pragma unroll
    for (int i = 0; i < NW; ++i)
      r.w[i] = (__float_as_uint(y[2 * i]) >> 16) | (__float_as_uint(y[2 * i + LAST]) & 0xffff0000u);
  }
  return r;
}
// ... and one store of them, at element `d0` of the row that starts at `row` (the same row for the whole wave).
// Written through: the attention kernel that follows reads these rows from every XCD (wt_store.h).
template <int PER>
__device__ __forceinline__ void store_row(uint16_t* row, uint32_t d0, const RawRow<PER>& r) {
  const auto win = wt_window_wave(row);
  if constexpr (PER == 8) wt_store16(win, d0 * 2u, wt_u32x4{r.w[0], r.w[1], r.w[2], r.w[3]});
  else if constexpr (PER == 4) wt_store8(win, d0 * 2u, wt_u32x2{r.w[0], r.w[1]});
  else if constexpr (PER == 2) wt_store4(win, d0 * 2u, r.w[0]);
  else wt_store2(win, d0 * 2u, (uint16_t)r.w[0]);
}

template <int PER, int NR>
__global__ void __launch_bounds__(256) qk_rope_kv_kernel(const RopeParams p) {
  __shared__ __attribute__((aligned(16))) float cos_t[256], sin_t[256];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t tok = blockIdx.x, h0 = (blockIdx.y * 4 + wave) * NR;
  const uint32_t n_heads = p.hq + 2 * p.hkv;
  const uint32_t hd = PER >= 2 ? PER * 64u : p.hd;   // (one element per lane: 64 or 32)
  // (the reference binds StepParams as a device buffer, qk_rope_kv.metal:30-38: read at execution time)
  const uint32_t kv_len = p.step_dev ? (uint32_t)__builtin_amdgcn_readfirstlane((int)p.step_dev[0]) : p.kv_len;
  const uint32_t kv_write_end = p.step_dev ? (uint32_t)__builtin_amdgcn_readfirstlane((int)p.step_dev[11]) : p.kv_write_end;
  const uint32_t pos = kv_len + tok;
  const bool kv_write = pos < kv_write_end;
  const int64_t slot = p.ring_mask ? (pos & p.ring_mask) : pos;

  // lane owns elements [PER*lane, PER*lane + PER); at hd < 64 only the first hd lanes own one
  const uint32_t d0 = lane * PER;
  const bool active = d0 < hd;
  const uint32_t half_rot = p.is_full ? hd / 8 : hd / 2;
  float freq = 0.f;
  if (threadIdx.x < half_rot) {
    const uint32_t e = threadIdx.x * (512u / hd);
    freq = p.is_full ? kInvFreq.proportional[e] : kInvFreq.split[e];
  }
  // Every row's elements and norm weights are asked for before anything is computed: behind one another they would be
  // as many trips to memory.  No branches around the loads: a row without a head of its own repeats the last one, an
  // idle lane the row's first element, a V row loads the key weights it does not use.
  RawRow<PER> xr[NR], wr[NR];
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const uint32_t h = min(h0 + n, n_heads - 1u);
    const bool is_q = h < p.hq, is_k = !is_q && h < p.hq + p.hkv;
    const uint32_t hh = is_q ? h : is_k ? h - p.hq : h - p.hq - p.hkv;
    const uint16_t* src = is_q ? p.q + ((size_t)tok * p.hq + hh) * hd
                               : ((is_k || p.v_from_k) ? p.k : p.v) + ((size_t)tok * p.hkv + hh) * hd;
    xr[n] = load_raw<PER>(src + (active ? d0 : 0u));
    wr[n] = load_raw<PER>((is_q ? p.qw : p.kw) + (active ? d0 : 0u));
  }
  // The angles depend on the position only: the workgroup's heads share one table of cos and sin,
  // one pair per thread, worked out while the rows are on their way (rotation, cpu.rs:31-65: pairs
  // (d, hd/2 + d) for d < rot/2; split-half: rot = hd, theta 1e4; proportional: rot = hd/4, theta 1e6,
  // everything else is left alone).
  if (threadIdx.x < hd / 2) {
    float sn = 0.f, cs = 1.f;
    if (threadIdx.x < half_rot) sincosf((float)pos * freq, &sn, &cs);
    cos_t[threadIdx.x] = cs;
    sin_t[threadIdx.x] = sn;
  }
  __syncthreads();
  // this lane's pairs: its element i belongs to pair pd + i, as the first member in the lower half of the lanes
  const uint32_t half_lanes = min(hd, 64u) / 2u;
  const uint32_t pd = (lane & (half_lanes - 1u)) * PER;
  const bool first = lane < half_lanes;
  const bool rotated = pd < half_rot;   // (half_rot is a multiple of PER: all of a lane's elements or none)
  float cs[PER], sn[PER];   // sn signed: the first member becomes x0 cos - x1 sin, the second x1 cos + x0 sin
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    cs[i] = cos_t[pd + i];
    sn[i] = first ? -sin_t[pd + i] : sin_t[pd + i];
  }
  const RowFormat cache_format = p.kv_dtype == DT_F16 ? ROW_F16 : ROW_BF16;
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const uint32_t h = h0 + n;
    if (h >= n_heads) return;   // the same for the whole wave; nothing below synchronises across waves
    const bool is_q = h < p.hq, is_k = !is_q && h < p.hq + p.hkv;
    const uint32_t hh = is_q ? h : is_k ? h - p.hq : h - p.hq - p.hkv;
    float x[PER];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      x[i] = active ? raw_elem(xr[n], i) : 0.f;
      ss += x[i] * x[i];
    }
    ss = wave_sum(ss);
    const float inv = inv_sqrt(ss * (1.0f / (float)hd) + kRmsEps);   // (hd is a power of two: the product is the quotient)
    if (p.dbg && lane == 0 && !(inv == inv && fabsf(inv) != INFINITY))
      dbg_report(p.dbg, DBG_ERR_NONFINITE, DBG_KERNEL_QK_ROPE_KV, (tok << 16) | h, tok);   // (qk_rope_kv.metal:77: tag = canvas row)

    float y[PER];
    if (!is_q && !is_k) {   // V: normalise without weight, write to the cache (cpu.rs:110-122)
      if (kv_write && active) {
#pragma unroll
        for (int i = 0; i < PER; ++i) y[i] = x[i] * inv;
        store_row<PER>((uint16_t*)p.vc + slot * p.v_tok_stride + (int64_t)hh * p.v_head_stride, d0, pack_row(y, cache_format));
      }
      continue;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) y[i] = x[i] * (inv * raw_elem(wr[n], i));   // x * (inv * w), the CPU twin's order (cpu.rs:71-74)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      float other;
      if (hd >= 64u) {
        const uint32_t u = __float_as_uint(y[i]);
        auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        other = __uint_as_float(first ? r[1] : r[0]);
      } else {
        other = __shfl_xor(y[i], 16, 64);
      }
      // (selected, not multiplied by cos 1 and sin 0: an infinite or NaN partner, or a zero's sign, must not cross to an
      // element that is left alone)
      y[i] = rotated ? y[i] * cs[i] + other * sn[i] : y[i];
    }
    if (!active) continue;
    if (is_k && kv_write)
      store_row<PER>((uint16_t*)p.kc + slot * p.k_tok_stride + (int64_t)hh * p.k_head_stride, d0, pack_row(y, cache_format));
    // Q always goes back in place; K only when V does not alias the raw k projection (cpu.rs:137-143)
    if (is_q || !p.v_from_k)
      store_row<PER>((is_q ? p.q + ((size_t)tok * p.hq + hh) * hd : p.k + ((size_t)tok * p.hkv + hh) * hd), d0,
                     pack_row(y, p.qk_trunc ? ROW_BF16_TRUNC : ROW_BF16));
  }
}

template <int PER, int NR>
void launch_rows(const RopeParams& p, hipStream_t s) {
  const uint32_t groups = (p.hq + 2 * p.hkv + 4 * NR - 1) / (4 * NR);
  hipLaunchKernelGGL((qk_rope_kv_kernel<PER, NR>), dim3(p.canvas, groups), dim3(256), 0, s, p);
}

template <int PER>
void launch_rope(const RopeParams& p, hipStream_t s) {
  // One row per wave while all waves are on the chip at once (32 on each of 256 compute units): the launch is then as
  // long as one wave's chain of dependent steps, which a second row only lengthens (256-row sliding layer, 8192 rows:
  // 3.6 -> 3.8 us).  With waves still to come what counts is bytes in flight, and a row of 512 bytes or less is too
  // little for a wave (sliding layer, 400 rows: 4.9 -> 4.6 us, 1024 rows: 9.3 -> 8.0); a row of 1 KiB is enough
  // (1024-row global layer: 7.8 us with one row, 8.2 with two).
  constexpr size_t kWavesOnChip = 8192;
  if (PER <= 4 && (size_t)p.canvas * (p.hq + 2 * p.hkv) > kWavesOnChip) launch_rows<PER, 2>(p, s);
  else launch_rows<PER, 1>(p, s);
}

}  // namespace
}  // namespace dg

extern "C" {

static int rope_launch(const dg_rope_desc* d, const dg_step_params* step_dev, void* q, void* k, const void* v, void* kv_base,
                       const void* q_norm_w, const void* k_norm_w, dg_debug_status* dbg, void* stream) {
  if (!d || !q || !k || !kv_base || !q_norm_w || !k_norm_w) return DG_ERR_NULL;
  if (((uintptr_t)step_dev % 4) != 0) return DG_ERR_LAYOUT;
  if (!d->v_from_k && !v) return DG_ERR_NULL;
  const uint32_t hd = d->head_dim;
  if (!(hd == 32 || hd == 64 || hd == 128 || hd == 256 || hd == 512)) return DG_ERR_SHAPE;
  if (d->canvas == 0 || d->n_q_heads == 0 || d->n_kv_heads == 0) return DG_ERR_SHAPE;
  if (d->kv_dtype != DG_F16 && d->kv_dtype != DG_BF16) return DG_ERR_DTYPE;
  if (d->kv_ring_mask != 0 && ((d->kv_ring_mask + 1) & d->kv_ring_mask) != 0) return DG_ERR_LAYOUT;
  if ((uint64_t)d->kv_len + d->canvas > 0xffffffffull) return DG_ERR_SHAPE;
  if (d->kv_region_bytes % 2 != 0) return DG_ERR_LAYOUT;
  if (d->k_tok_stride < (int64_t)hd || d->v_tok_stride < (int64_t)hd || d->k_head_stride < (int64_t)hd ||
      d->v_head_stride < (int64_t)hd)
    return DG_ERR_LAYOUT;
  dg::RopeParams p{};
  p.q = (uint16_t*)q;
  p.k = (uint16_t*)k;
  p.v = (const uint16_t*)v;
  char* region = (char*)kv_base + d->kv_region_bytes;
  p.kc = region;
  p.vc = region + d->v_base_off * 2;
  p.qw = (const uint16_t*)q_norm_w;
  p.kw = (const uint16_t*)k_norm_w;
  p.dbg = (uint32_t*)dbg;
  p.step_dev = (const uint32_t*)step_dev;
  p.k_tok_stride = d->k_tok_stride;
  p.k_head_stride = d->k_head_stride;
  p.v_tok_stride = d->v_tok_stride;
  p.v_head_stride = d->v_head_stride;
  p.canvas = d->canvas;
  p.hq = d->n_q_heads;
  p.hkv = d->n_kv_heads;
  p.hd = hd;
  p.kv_len = d->kv_len;
  p.kv_write_end = d->kv_write_end;
  p.ring_mask = d->kv_ring_mask;
  p.is_full = d->is_full ? 1u : 0u;
  p.v_from_k = d->v_from_k ? 1u : 0u;
  p.kv_dtype = d->kv_dtype == DG_F16 ? dg::DT_F16 : dg::DT_BF16;
  p.qk_trunc = (d->flags & DG_ROPE_F_QK_TRUNCATE) ? 1u : 0u;
  // vector accesses of `per` elements: rows and the cache region must be aligned to them
  const uint32_t per = hd >= 64 ? hd / 64 : 1;
  const uintptr_t align = 2 * per;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)p.kc | (uintptr_t)p.vc | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w |
       (d->v_from_k ? 0 : (uintptr_t)v)) % align != 0)
    return DG_ERR_LAYOUT;
  if ((d->k_tok_stride | d->k_head_stride | d->v_tok_stride | d->v_head_stride) % per != 0) return DG_ERR_LAYOUT;
  hipStream_t s = (hipStream_t)stream;
  switch (per) {
    case 8: dg::launch_rope<8>(p, s); break;
    case 4: dg::launch_rope<4>(p, s); break;
    case 2: dg::launch_rope<2>(p, s); break;
    default: dg::launch_rope<1>(p, s); break;
  }
  return hipGetLastError() == hipSuccess ? DG_OK : DG_ERR_LAUNCH;
}

int dg_qk_rope_kv(const dg_rope_desc* d, void* q, void* k, const void* v, void* kv_base, const void* q_norm_w,
                  const void* k_norm_w, dg_debug_status* dbg, void* stream) {
  return rope_launch(d, nullptr, q, k, v, kv_base, q_norm_w, k_norm_w, dbg, stream);
}

int dg_qk_rope_kv_dev(const dg_rope_desc* d, const dg_step_params* step_dev, void* q, void* k, const void* v, void* kv_base,
                      const void* q_norm_w, const void* k_norm_w, dg_debug_status* dbg, void* stream) {
  if (!step_dev) return DG_ERR_NULL;
  return rope_launch(d, step_dev, q, k, v, kv_base, q_norm_w, k_norm_w, dbg, stream);
}

// The reference's argument block -> descriptor; kv_len / kv_write_end from the host copy of P, or (P == null) left to
// the device copy.
static void rope_desc_from_reference(const dg_layer_offsets* L, const dg_step_params* P, const dg_attn_dims* dims,
                                     dg_rope_desc* out) {
  dg_rope_desc d{};
  d.canvas = dims->canvas;
  d.n_q_heads = dims->n_q_heads;
  d.n_kv_heads = L->n_kv_heads;
  d.head_dim = L->head_dim;
  d.kv_len = P ? P->kv_len : 0u;
  d.kv_write_end = P ? P->kv_write_end : 0xffffffffu;
  d.kv_ring_mask = L->kv_ring_mask;
  d.is_full = L->is_full;
  d.v_from_k = L->v_proj == 0 ? 1u : 0u;
  d.kv_dtype = DG_F16;
  d.flags = DG_ROPE_F_QK_TRUNCATE;   // arena_store truncates (common.metal:16-18)
  d.kv_region_bytes = L->kv_region;
  const int64_t row = (int64_t)L->n_kv_heads * L->head_dim;   // slot-major [slot][K: Hkv*d | V: Hkv*d]
  d.k_tok_stride = 2 * row;
  d.k_head_stride = L->head_dim;
  d.v_base_off = row;
  d.v_tok_stride = 2 * row;
  d.v_head_stride = L->head_dim;
  *out = d;
}

int dg_qk_rope_kv_dispatch(void* q, void* k, void* v, void* kvcache, const void* blob, const dg_layer_offsets* L,
                           const dg_step_params* P, const dg_attn_dims* dims, dg_debug_status* dbg, void* stream) {
  if (!L || !P || !dims || !blob) return DG_ERR_NULL;
  dg_rope_desc d;
  rope_desc_from_reference(L, P, dims, &d);
  return dg_qk_rope_kv(&d, q, k, v, kvcache, (const char*)blob + L->q_norm, (const char*)blob + L->k_norm, dbg, stream);
}

int dg_qk_rope_kv_dispatch_dev(void* q, void* k, void* v, void* kvcache, const void* blob, const dg_layer_offsets* L,
                               const dg_step_params* P_dev, const dg_attn_dims* dims, dg_debug_status* dbg, void* stream) {
  if (!L || !P_dev || !dims || !blob) return DG_ERR_NULL;
  dg_rope_desc d;
  rope_desc_from_reference(L, nullptr, dims, &d);
  return dg_qk_rope_kv_dev(&d, P_dev, q, k, v, kvcache, (const char*)blob + L->q_norm, (const char*)blob + L->k_norm, dbg,
                           stream);
}

}  // extern "C"
