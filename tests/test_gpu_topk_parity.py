"""GPU parity of top-k sparse attention (topk_scores_kernel + topk_select_kernel through the C ABI)
against the CPU oracle.  The reference's own matrix (attention_topk/mod.rs:463-534) first, then
selection exactness on inputs whose scores are exact in fp32, model-shaped rows with the
context-adaptive k, and the size-independent properties (k >= visible keys is dense attention,
k = 1 is the arg-max key's V row, run-to-run bit equality)."""
import ctypes as C

import numpy as np
import pytest

from diffgemma_amd import attention as A
from diffgemma_amd import attention_topk as T
from diffgemma_amd import capi, rounding as R, workloads as W
from helpers import assert_oracle, max_abs_diff, mean_abs_diff

pytestmark = pytest.mark.gpu


def topk_cpu(po, f, k, causal):
    """cpu::topk_causal / topk_denoise with round_kv_f16 = true (cpu.rs:28-38): Q -> bf16, KV -> f16,
    output -> bf16, all by the reference's truncating conversions."""
    q = R.bf16_bits_to_f32(R.f32_to_bf16_bits_trunc(f.q))
    kv = R.f16_bits_to_f32(R.f32_to_f16_bits_trunc(f.kvcache))
    d = po.make_desc(f.canvas, f.n_q_heads, f.n_kv(), f.head_dim(), f.kv_len, causal_rows=f.canvas if causal else 0)
    out = po.attention_topk_f32(d, T.fixed_k(k), q, kv)
    return po.round_array(out, po.ROUND_BF16_TRUNC).ravel()


# ------------------------------------------------------------------ the reference's tests
@pytest.mark.parametrize("causal,k,cos", [(True, 64, 0.9999), (False, 64, 0.9999), (True, 1, 0.999), (True, 128, 0.9999)])
def test_reference_full_grp8_fixture(gpu_ready, po, causal, k, cos):
    f = A.full_grp8_hd512_fixture()
    assert_oracle(T.gpu(f, causal, k), topk_cpu(po, f, k, causal), 2e-2, cos)


def test_reference_model_fixture_midsize(gpu_ready, po):
    """model_full_fixture (attention_gemm/mod.rs:364-432) at a prefix of many key tiles, k = 64."""
    f = A.model_full_fixture(1500, canvas=64)
    assert_oracle(T.gpu(f, True, 64), topk_cpu(po, f, 64, True), 2e-2, 0.9999)


def test_ragged_causal_tail(gpu_ready, po):
    """cpu.rs:315-323: canvas 256 behind 4 keys, k = 64 > the keys early rows see."""
    f = A.model_bench_fixture(512, 4, True)
    got = T.gpu(f, True, 64)
    assert np.isfinite(got).all()
    assert_oracle(got, topk_cpu(po, f, 64, True), 2e-2, 0.9999)


# ------------------------------------------------------------------ generic runner
def run_topk(po, canvas, hq, hkv, hd, kv_len, k_cfg, *, causal_rows=0, window=0, q=None, kv=None, seed=0, toks=None,
             kv_dtype=capi.DG_BF16, flags=0):
    """bf16 (or f16) storage, fp32 output: isolates selection and arithmetic from the output store."""
    rng = np.random.default_rng(seed)
    t_all = kv_len + canvas
    if q is None:
        q = rng.standard_normal((canvas, hq, hd)).astype(np.float32)
        kv = rng.standard_normal((t_all, 2, hkv, hd)).astype(np.float32)
        rms = lambda x: x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True) + 1e-6)
        q, kv = rms(q).astype(np.float32), rms(kv).astype(np.float32)
    from_bits = R.bf16_bits_to_f32 if kv_dtype == capi.DG_BF16 else R.f16_bits_to_f32
    got, qb, kb, _ = device_topk(canvas, hq, hkv, hd, kv_len, k_cfg, q, kv, causal_rows=causal_rows, window=window,
                                 kv_dtype=kv_dtype, flags=flags)
    od = po.make_desc(canvas, hq, hkv, hd, kv_len, causal_rows=causal_rows, window=window,
                      causal_sees_masked=int(bool(flags & capi.DG_ATTN_F_CAUSAL_SEES_MASKED)))
    ref = po.attention_topk_f32(od, k_cfg, R.bf16_bits_to_f32(qb).reshape(q.shape), from_bits(kb).reshape(kv.shape),
                                tok_list=toks)
    rows = np.arange(canvas) if toks is None else np.asarray(toks)
    return got[rows], ref[rows]


def device_topk(canvas, hq, hkv, hd, kv_len, k_cfg, q, kv, *, causal_rows=0, window=0, kv_dtype=capi.DG_BF16, flags=0):
    """(fp32 rows, the storage bits of q and kv, the workspace as the call left it) of one dg_attn_topk_forward."""
    import torch
    to_bits = R.f32_to_bf16_bits_rne if kv_dtype == capi.DG_BF16 else R.f32_to_f16_bits_rne
    qb, kb = R.f32_to_bf16_bits_rne(q), to_bits(kv)
    d = A.make_desc(canvas, hq, hkv, hd, kv_len, causal_rows=causal_rows, window=window, q_dtype=capi.DG_BF16,
                    kv_dtype=kv_dtype, out_dtype=capi.DG_F32, flags=flags)
    out = torch.zeros(canvas * hq * hd, dtype=torch.float32, device="cuda")
    ws = T.alloc_workspace(d, k_cfg)
    T.forward(d, k_cfg, A.to_device_bits(qb.reshape(-1)), A.to_device_bits(kb.reshape(-1)), out, ws)
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(canvas, hq, hd), qb, kb, ws


# ------------------------------------------------------------------ selection exactness
EXACT = [
    # canvas, hq, hkv, hd, kv_len, causal_rows, window, k
    (9, 4, 2, 32, 300, 0, 0, 16),
    (9, 4, 2, 64, 300, 9, 0, 16),
    (33, 8, 2, 128, 1000, 20, 0, 64),      # mixed rows
    (16, 16, 8, 256, 700, 16, 301, 40),    # causal + window
    (40, 16, 2, 512, 2100, 0, 0, 100),
    (5, 2, 1, 64, 9000, 0, 0, 700),        # threshold class larger than the candidate list
    (5, 2, 1, 64, 9000, 5, 0, 1024),
    (64, 16, 2, 512, 3, 64, 0, 64),        # ragged: early rows see fewer than k keys
    (3, 2, 2, 32, 5000, 0, 0, 1),
]


@pytest.mark.parametrize("case", EXACT)
def test_selection_is_exact_on_exact_scores(gpu_ready, po, case):
    """Q and K hold few-bit dyadic values: every dot product is exact in fp32 whatever the order of
    summation, so the kernel and the oracle see identical scores, full of ties; the kept sets and
    with them the outputs have to agree to fp32 summation error."""
    canvas, hq, hkv, hd, kvl, cr, win, k = case
    rng = np.random.default_rng(hash(case) & 0xFFFF)
    q = (rng.integers(-2, 3, (canvas, hq, hd)) / 4).astype(np.float32)
    kv = (rng.integers(-2, 3, (kvl + canvas, 2, hkv, hd)) / 4).astype(np.float32)
    kv[:, 1] = rng.standard_normal(kv[:, 1].shape).astype(np.float32)
    got, ref = run_topk(po, canvas, hq, hkv, hd, kvl, (k, 0, 0, 0), causal_rows=cr, window=win, q=q, kv=kv)
    assert np.isfinite(got).all()
    assert max_abs_diff(got, ref) < 2e-5


def test_all_scores_equal_keeps_the_first_k_positions(gpu_ready, po):
    """A zero query ties every key: the k lowest positions are kept (more ties than any list holds)."""
    canvas, hq, hkv, hd, kvl, k = 2, 2, 1, 64, 6000, 50
    q = np.zeros((canvas, hq, hd), np.float32)
    rng = np.random.default_rng(1)
    kv = rng.standard_normal((kvl + canvas, 2, hkv, hd)).astype(np.float32)
    got, ref = run_topk(po, canvas, hq, hkv, hd, kvl, (k, 0, 0, 0), q=q, kv=kv)
    want = R.bf16_bits_to_f32(R.f32_to_bf16_bits_rne(kv[:k, 1, 0])).reshape(k, hd).mean(axis=0)
    assert max_abs_diff(ref[0, 0], want) < 1e-5       # the oracle agrees with the closed form
    assert max_abs_diff(got, ref) < 1e-5


# ------------------------------------------------------------------ model-shaped inputs
@pytest.mark.parametrize("case", [
    # canvas, hq, hkv, hd, kv_len, causal_rows, k_cfg
    (64, 16, 2, 512, 4096, 0, T.adaptive_k()),        # denoise rows: k = 4160 / 128 -> 64 (k_min)
    (64, 16, 2, 512, 12000, 0, T.adaptive_k()),       # k = 94
    (64, 16, 2, 512, 12000, 64, T.adaptive_k()),      # causal rows: per-row k on the 256 grid
    (48, 16, 8, 256, 3000, 0, (200, 0, 0, 0)),
    (256, 8, 4, 128, 512, 128, (32, 0, 0, 0)),
])
def test_model_shaped_rows(gpu_ready, po, case):
    canvas, hq, hkv, hd, kvl, cr, k_cfg = case
    toks = np.unique(np.linspace(0, canvas - 1, 12).round().astype(np.uint32))
    got, ref = run_topk(po, canvas, hq, hkv, hd, kvl, k_cfg, causal_rows=cr, seed=hash(case[:6]) & 0xFFFF, toks=toks)
    assert np.isfinite(got).all()
    # the kernel's scores (MFMA summation order) and the oracle's (sequential) differ in the last
    # bits; keys whose scores are that close to the k-th carry the smallest kept weights
    assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3


def test_f16_cache_with_bf16_queries(gpu_ready, po):
    got, ref = run_topk(po, 32, 16, 2, 512, 2000, (64, 0, 0, 0), seed=4, kv_dtype=capi.DG_F16)
    assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3


def test_global_layer_at_32k_prefix_rows(gpu_ready, po):
    """The denoise shape of a global layer (canvas 256, 16 / 2 heads, hd 512, prefix 32768) with the
    production k rule (258 keys per row); the oracle runs a row sample."""
    import torch
    w = W.config("cfg3_global")
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc(causal_rows=0)
    d.out_dtype = capi.DG_F32
    k_cfg = T.adaptive_k()
    out = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.float32, device="cuda")
    T.forward(d, k_cfg, qd, kd, out, T.alloc_workspace(d, k_cfg))
    torch.cuda.synchronize()
    toks = np.array([0, 63, 64, 130, 255], dtype=np.uint32)
    od = po.make_desc(w.canvas, w.n_q_heads, w.n_kv_heads, w.head_dim, w.kv_len, layout=w.layout, t_cap=w.t_all)
    ref, idx, cnt = po.attention_topk_f32(od, k_cfg, q, kv, tok_list=toks, sel_cap=512)
    assert (cnt[toks] == 258).all()
    got = out.cpu().numpy().reshape(w.canvas, w.n_q_heads, w.head_dim)
    assert np.isfinite(got).all()
    assert max_abs_diff(got[toks], ref[toks]) <= 2e-2 and mean_abs_diff(got[toks], ref[toks]) <= 2e-3


def test_long_context_rows(gpu_ready, po):
    """131072-key prefix with 1% of the keys scaled x8 (config 4's inputs): k = 512 (the cap), score rows of
    525 KB, sixteen blocks of canvas rows."""
    import torch
    w = W.config("cfg4_long")
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc()
    d.out_dtype = capi.DG_F32
    k_cfg = T.adaptive_k()
    out = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.float32, device="cuda")
    T.forward(d, k_cfg, qd, kd, out, T.alloc_workspace(d, k_cfg))
    torch.cuda.synchronize()
    toks = np.array([0, 17, 128, 255], dtype=np.uint32)
    od = po.make_desc(w.canvas, w.n_q_heads, w.n_kv_heads, w.head_dim, w.kv_len, layout=w.layout, t_cap=w.t_all)
    ref, idx, cnt = po.attention_topk_f32(od, k_cfg, q, kv, tok_list=toks, sel_cap=512)
    assert (cnt[toks] == 512).all()
    got = out.cpu().numpy().reshape(w.canvas, w.n_q_heads, w.head_dim)
    assert np.isfinite(got).all()
    assert max_abs_diff(got[toks], ref[toks]) <= 2e-2 and mean_abs_diff(got[toks], ref[toks]) <= 2e-3


# ------------------------------------------------------------------ edge cases
EDGE = [
    # canvas, hq, hkv, hd, kv_len, causal_rows, window, k_cfg
    (1, 4, 2, 64, 0, 1, 0, (8, 0, 0, 0)),              # one row, one key
    (1, 16, 2, 512, 77, 0, 0, T.adaptive_k()),          # single denoise row, fewer keys than k_min
    (5, 2, 1, 32, 3, 0, 0, (1, 0, 0, 0)),               # less than one key tile in total
    (37, 12, 4, 64, 333, 20, 100, (17, 0, 0, 0)),       # ragged everything: group 3, mixed rows, window
    (256, 16, 8, 256, 0, 256, 0, T.adaptive_k()),       # prefill from an empty cache, per-row k
    (64, 16, 2, 512, 40000, 64, 0, (256, 128, 64, 512)),  # two blocks of canvas rows (score plane budget)
    (8, 8, 8, 128, 5000, 0, 0, (600, 0, 0, 0)),         # no GQA sharing
]


@pytest.mark.parametrize("case", EDGE)
def test_edge_cases(gpu_ready, po, case):
    canvas, hq, hkv, hd, kvl, cr, win, k_cfg = case
    toks = None if canvas <= 64 else np.unique(np.linspace(0, canvas - 1, 16).round().astype(np.uint32))
    got, ref = run_topk(po, canvas, hq, hkv, hd, kvl, k_cfg, causal_rows=cr, window=win, seed=hash(case[:7]) & 0xFFFF,
                        toks=toks)
    assert np.isfinite(got).all()
    assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3


# ------------------------------------------------------------------ thresholds instead of a score plane (head_dim 512, long rows)
FILTERED = [
    # canvas, hq, hkv, kv_len, causal_rows, k_cfg, what the keys look like
    (40, 16, 2, 2048, 0, T.adaptive_k(), "unit"),         # shortest prefix taken; 320 stacked rows: the second row tile is ragged
    (3, 6, 2, 2500, 2, (64, 0, 0, 0), "unit"),            # 9 stacked rows per KV head, group 3
    (17, 4, 1, 4077, 17, (512, 0, 0, 0), "unit"),         # odd key count, most keys kept, causal rows
    (8, 8, 8, 3001, 0, (1, 0, 0, 0), "unit"),             # no sharing, one key kept
    (6, 16, 2, 2100, 3, (100, 0, 0, 0), "ties"),          # exact scores full of ties: lists overflow or end inside a tie
    (6, 16, 2, 6000, 0, (100, 0, 0, 0), "few ties"),      # ties, but lists that fit: the tie-break inside the list
    (4, 4, 2, 3000, 0, (50, 0, 0, 0), "zero"),            # a zero query: every row is left to the general path
    (9, 16, 2, 5000, 0, (64, 0, 0, 0), "cluster"),        # the best keys are neighbours
    (9, 16, 2, 5000, 0, (64, 0, 0, 0), "half"),           # some rows left over, the others not
    (5, 16, 2, 36000, 5, T.adaptive_k(), "unit"),         # positions ranked in two windows
    (320, 16, 2, 40000, 320, T.adaptive_k(), "unit"),     # more rows than a pass takes
]


def check_thresholds_and_lists(po, case, kv_dtype=capi.DG_BF16, more_flags=0):
    canvas, hq, hkv, kvl, cr, k_cfg, keys = case
    rng = np.random.default_rng(sum(case[:5]))
    t_all, hd = kvl + canvas, 512
    rms = lambda x: (x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))).astype(np.float32)
    q, kv = rms(rng.standard_normal((canvas, hq, hd))), rms(rng.standard_normal((t_all, 2, hkv, hd)))
    exact = keys in ("ties", "few ties", "zero", "half")
    if exact:       # few-bit dyadic values in a few dimensions: scores exact in fp32 whatever the order of summation
        live = {"ties": 8, "half": 128}.get(keys, 256)
        q[:], kv[:, 0] = 0, 0
        q[..., :live] = rng.integers(-2, 3, (canvas, hq, live)) / 4
        kv[:, 0, :, :live] = rng.integers(-2, 3, (t_all, hkv, live)) / 4
        if keys == "zero":
            q[:] = 0
        if keys == "half":
            q[::2] = 0
    if keys == "cluster":
        kv[3000:3200, 0] *= 4
    toks = None if canvas <= 64 else np.array([0, 159, 160, 161, 319])
    run = lambda flag: run_topk(po, canvas, hq, hkv, hd, kvl, k_cfg, causal_rows=cr, q=q, kv=kv, flags=flag | more_flags, toks=toks,
                                kv_dtype=kv_dtype)
    got, ref = run(capi.DG_ATTN_F_TOPK_THRESHOLD)
    assert np.isfinite(got).all()
    if exact:       # same kept sets: outputs agree to fp32 summation error
        assert max_abs_diff(got, ref) < 2e-5
    else:
        assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3
        # both paths sum a score over d in the same order, so they keep the same keys: fp32 summation error again
        assert max_abs_diff(got, run(capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]) < 2e-5


@pytest.mark.parametrize("case", FILTERED)
def test_thresholds_and_lists(gpu_ready, po, case):
    check_thresholds_and_lists(po, case)


@pytest.mark.parametrize("case", [c for c in FILTERED if c[0] <= 64])
def test_thresholds_and_lists_over_an_f16_cache(gpu_ready, po, case):
    """The storage of the reference's own boundary: bf16 queries converted in the kernel, f16 K and V."""
    check_thresholds_and_lists(po, case, kv_dtype=capi.DG_F16)


@pytest.mark.parametrize("case", [
    (40, 16, 2, 2100, 25, T.adaptive_k(), "unit"),        # causal rows see the prefix, themselves and the masked canvas keys
    (33, 8, 2, 2069, 7, (200, 0, 0, 0), "unit"),          # the second range begins inside a key tile
    (6, 16, 2, 2100, 3, (100, 0, 0, 0), "ties"),
    (24, 4, 1, 5001, 23, (64, 0, 0, 0), "few ties"),      # a second range of one key
])
@pytest.mark.parametrize("kv_dtype", [capi.DG_BF16, capi.DG_F16])
def test_thresholds_and_lists_with_a_second_key_range(gpu_ready, po, case, kv_dtype):
    check_thresholds_and_lists(po, case, kv_dtype=kv_dtype, more_flags=capi.DG_ATTN_F_CAUSAL_SEES_MASKED)


def rows_left_over(ws, rows):
    """The marks the thresholds-and-lists path leaves at the workspace's start, one word per row and head: 0, or 1 where
    the general path redid it.  None where the words are no marks: the score plane begins there."""
    import torch
    left = ws.view(torch.int32)[:rows].cpu().numpy()
    return int(left.sum()) if ((left == 0) | (left == 1)).all() else None


@pytest.mark.parametrize("t_all,stride", [(8192 * 17, 17), (8192 * 17 + 1, 19), (8192 * 19, 19), (8192 * 19 + 1, 21), (8192 * 21, 21),
                                          (8192 * 21 + 1, None)])
def test_sample_strides_of_very_long_rows(gpu_ready, po, t_all, stride):
    """8192 sampled keys at most: every 17th, 19th or 21st key, and past that the score plane."""
    canvas, hq, hkv, hd, k_cfg = 3, 2, 1, 512, T.adaptive_k()
    rng = np.random.default_rng(t_all)
    rms = lambda x: x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))
    q = rms(rng.standard_normal((canvas, hq, hd), dtype=np.float32))
    kv = rms(rng.standard_normal((t_all, 2, hkv, hd), dtype=np.float32))
    args = (canvas, hq, hkv, hd, t_all - canvas, k_cfg, q, kv)
    got, qb, kb, ws = device_topk(*args, flags=capi.DG_ATTN_F_TOPK_THRESHOLD)
    assert rows_left_over(ws, canvas * hq) == (None if stride is None else 0)
    plane = device_topk(*args, flags=capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]
    assert np.isfinite(got).all() and max_abs_diff(got, plane) < 2e-5
    if stride in (None, 21):
        od = po.make_desc(canvas, hq, hkv, hd, t_all - canvas)
        ref = po.attention_topk_f32(od, k_cfg, R.bf16_bits_to_f32(qb).reshape(q.shape), R.bf16_bits_to_f32(kb).reshape(kv.shape))
        assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3


@pytest.mark.parametrize("canvas,kvl,causal", [
    (16, 2048, 0),         # one 128-row tile of stacked rows, full; 122 sampled keys in two splits, the last tile ragged
    (17, 2159, 17),        # a second one of 8 rows; the last sampled keys behind some rows' own
    (15, 2174, 15),        # ... and an odd number of tiles, so that one split has three
    (48, 17 * 544, 20),    # 17 full sampled tiles before the canvas, eight splits
    (130, 9001, 130),      # 1040 stacked rows: the last 128-row tile has 16
    (1024, 3000, 1024),    # few splits and keys kept: thresholds are uncertain, and the lists have to hold what that brings
])
@pytest.mark.parametrize("kv_dtype", [capi.DG_BF16, capi.DG_F16])
def test_thresholds_from_groups_of_sampled_keys(gpu_ready, canvas, kvl, causal, kv_dtype):
    """Random rows are never left over (thresholds neither too high nor so low that lists overflow), whatever number of sampled
    keys a group has; the same kept keys as through the score plane, fp32 summation error apart."""
    hq, hkv, hd, k_cfg = 16, 2, 512, T.adaptive_k()
    rng = np.random.default_rng(canvas + kvl)
    rms = lambda x: x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))
    q = rms(rng.standard_normal((canvas, hq, hd), dtype=np.float32))
    kv = rms(rng.standard_normal((kvl + canvas, 2, hkv, hd), dtype=np.float32))
    run = lambda flag: device_topk(canvas, hq, hkv, hd, kvl, k_cfg, q, kv, causal_rows=causal, kv_dtype=kv_dtype, flags=flag)
    got, _, _, ws = run(capi.DG_ATTN_F_TOPK_THRESHOLD)
    assert rows_left_over(ws, canvas * hq) == 0
    assert max_abs_diff(got, run(capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]) < 2e-5


@pytest.mark.parametrize("canvas,keys,k", [(c, t, k) for c, t in ((256, 2304), (128, 2200), (512, 2700), (256, 3300), (256, 5000))
                                           for k in (64, 128, 256, 384, 512)] + [(256, 170000, k) for k in (160, 258, 384)])
def test_random_rows_have_lists_that_hold_them(gpu_ready, canvas, keys, k):
    """Where two sampled keys of five lie above the threshold, several of them in one group; and where every 21st key alone is
    sampled.  By the binomial distribution of groups and lists 4e-6 of rows at most have a list too short or too long."""
    import torch
    hq, hkv, hd = 16, 2, 512
    g = torch.Generator(device="cuda")
    g.manual_seed(keys + k)
    q, kv = (torch.nn.functional.rms_norm(torch.randn(n, hd, device="cuda", generator=g), (hd,)).to(torch.bfloat16)
             for n in (canvas * hq, 2 * hkv * keys))
    runs = []
    for flag in (capi.DG_ATTN_F_TOPK_THRESHOLD, capi.DG_ATTN_F_TOPK_SCORE_PLANE):
        d = A.make_desc(canvas, hq, hkv, hd, keys - canvas, layout="head_major", t_cap=keys, out_dtype=capi.DG_F32, flags=flag)
        out, ws = torch.zeros(canvas, hq, hd, device="cuda"), T.alloc_workspace(d, (k, 0, 0, 0))
        T.forward(d, (k, 0, 0, 0), q, kv, out, ws)
        runs.append((out, ws))
    torch.cuda.synchronize()
    assert rows_left_over(runs[0][1], canvas * hq) == 0
    assert float((runs[0][0] - runs[1][0]).abs().max()) < 2e-5


def test_lists_hold_the_rows_of_a_prompt(gpu_ready):
    """1024 causal rows behind 32768 keys, 258 to 264 kept: the longest list has 1232 candidates of the 1280 a wave holds, two ranks
    past the one that a threshold is meant to have 1296."""
    import torch
    w = W.Workload("topk_prompt", 1024, 16, 2, 512, 32768, causal_rows=1024, seed=41)
    qd, kd = W.device_arrays(w, *W.generate(w))
    d = w.desc(flags=capi.DG_ATTN_F_TOPK_THRESHOLD)
    out, ws = torch.zeros(1024 * 16 * 512, dtype=torch.int16, device="cuda"), T.alloc_workspace(d, T.adaptive_k())
    T.forward(d, T.adaptive_k(), qd, kd, out, ws)
    torch.cuda.synchronize()
    assert rows_left_over(ws, 1024 * 16) == 0


GATHER_SLICES = [(64, 4), (65, 2), (128, 2), (129, 1)]      # canvas rows of 16 heads -> slices; test_split_map.py holds the rule to it


@pytest.mark.parametrize("canvas,slices", GATHER_SLICES)
@pytest.mark.parametrize("k", [1, 3, 4, 15, 16, 17, 33])
def test_gather_slices(gpu_ready, canvas, slices, k):
    """Every number of head_dim slices the gather deals out, at the edges of its groups of keys.  One element of every V row is an
    infinity: it stays in its own element, and stays an infinity there (0 times it, to fill a group of keys, would be NaN)."""
    hq, hkv, hd, kvl = 16, 2, 512, 2100
    rng = np.random.default_rng(canvas * 64 + k)
    rms = lambda x: x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))
    q = rms(rng.standard_normal((canvas, hq, hd), dtype=np.float32))
    kv = rms(rng.standard_normal((kvl + canvas, 2, hkv, hd), dtype=np.float32))
    kv[:, 1, :, 7 + 128 * (k % 4)] = np.inf
    run = lambda flag: device_topk(canvas, hq, hkv, hd, kvl, (k, 0, 0, 0), q, kv, flags=flag)
    got, _, _, ws = run(capi.DG_ATTN_F_TOPK_THRESHOLD)
    assert rows_left_over(ws, canvas * hq) == 0
    plane = run(capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]
    finite = np.delete(np.arange(hd), 7 + 128 * (k % 4))
    assert np.isfinite(got[..., finite]).all() and max_abs_diff(got[..., finite], plane[..., finite]) < 2e-5
    # (no weight underflows: a row's kept scores are at most 73 apart, e^-87 is the smallest normal number)
    assert np.isposinf(got[..., 7 + 128 * (k % 4)]).all()


@pytest.mark.parametrize("kv_dtype", [capi.DG_BF16, capi.DG_F16])
def test_nonfinite_scores_go_the_score_planes_way(gpu_ready, kv_dtype):
    """NaN scores sort below every other (never kept while enough others are visible), an infinite score is kept and
    makes its row NaN, -inf sorts low, a query row of NaN keeps the lowest positions: the same through both paths."""
    canvas, hq, hkv, hd, kvl = 12, 4, 1, 512, 3000
    rng = np.random.default_rng(5)
    rms = lambda x: (x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))).astype(np.float32)
    q, kv = rms(rng.standard_normal((canvas, hq, hd))), rms(rng.standard_normal((kvl + canvas, 2, hkv, hd)))
    kv[[0, 17, 31, 34, 1000, kvl + 3], 0] = np.nan              # sampled positions (multiples of 17) and others
    kv[2000:2040, 0] = np.nan
    kv[[51, 500], 0, :, 3] = np.inf                             # +inf or -inf, by the sign of the query's element 3
    q[:6, :, 3] = -np.abs(q[:6, :, 3])
    q[6:, :, 3] = np.abs(q[6:, :, 3])
    q[2, 1] = np.nan
    for k_cfg in (T.adaptive_k(), (1, 0, 0, 0), (512, 0, 0, 0)):
        args = (canvas, hq, hkv, hd, kvl, k_cfg, q, kv)
        with np.errstate(invalid="ignore"):
            got, _, _, ws = device_topk(*args, kv_dtype=kv_dtype, flags=capi.DG_ATTN_F_TOPK_THRESHOLD)
            plane = device_topk(*args, kv_dtype=kv_dtype, flags=capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]
        assert rows_left_over(ws, canvas * hq) == 1             # the NaN query's
        assert np.isfinite(np.delete(got[:6].reshape(24, hd), 2 * hq + 1, axis=0)).all()
        assert np.isnan(got[6:]).all() and np.isnan(got[2, 1]).all()
        assert np.array_equal(np.isnan(got), np.isnan(plane))
        assert max_abs_diff(got[~np.isnan(got)], plane[~np.isnan(got)]) < 2e-5


def test_dispatch_over_a_long_prefix_keeps_lists(gpu_ready, po):
    """The reference's argument block on rows long enough for thresholds: f16 slot-major cache, truncating store."""
    kvl, canvas, hq, hkv, hd = 2500, 160, 16, 2, 512
    rng = np.random.default_rng(77)
    rms = lambda x: (x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))).astype(np.float32)
    q = rms(rng.standard_normal((canvas, hq, hd), dtype=np.float32))
    kv = rms(rng.standard_normal((kvl + canvas, 2, hkv, hd), dtype=np.float32))
    f = A.Fixture(q.reshape(-1), kv.reshape(-1), A.LayerAttnParams(hd, hkv, True, 0), canvas, hq, kvl)
    for causal in (False, True):
        rig = A.AttnRig.from_fixture(f)
        T.run_dispatch(rig, causal, T.adaptive_k())
        got = rig.read_out_f32().reshape(canvas, hq, hd)
        (ws,) = rig._ws.values()
        assert rows_left_over(ws, canvas * hq) == 0
        toks = np.array([0, 1, 79, 127, 128, 159], dtype=np.uint32)
        d = po.make_desc(canvas, hq, hkv, hd, kvl, causal_rows=canvas if causal else 0)
        ref = po.attention_topk_f32(d, T.adaptive_k(), R.bf16_bits_to_f32(R.f32_to_bf16_bits_trunc(q)).reshape(q.shape),
                                    R.f16_bits_to_f32(R.f32_to_f16_bits_trunc(kv)).reshape(kv.shape), tok_list=toks)
        assert np.isfinite(got).all()
        # on top of the fp32 comparison's bounds the truncating store takes up to 2^-7 of a value, half of that on average
        err, mag = np.abs(got[toks] - ref[toks]), np.abs(ref[toks])
        assert np.all(err <= 2e-2 + mag * 2.0 ** -7) and err.mean() <= 2e-3 + mag.mean() * 2.0 ** -8


def test_random_rows_are_not_left_over(gpu_ready):
    """Five-sigma thresholds: on random rows the lists suffice, in every pass over the canvas rows (the workspace begins with
    a word per row and head that says whether the general path had to redo it)."""
    import torch
    w = W.Workload("left", 320, 16, 2, 512, 40000, causal_rows=320, seed=6)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc(flags=capi.DG_ATTN_F_TOPK_THRESHOLD)
    k_cfg = T.adaptive_k()
    ws = T.alloc_workspace(d, k_cfg)
    T.forward(d, k_cfg, qd, kd, torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.int16, device="cuda"), ws)
    torch.cuda.synchronize()
    left = ws.view(torch.int32)[:w.canvas * w.n_q_heads]
    assert int(((left != 0) & (left != 1)).sum()) == 0 and int(left.sum()) == 0      # (5120 rows, 4 in 10^6 of which the lists may not hold)


@pytest.mark.parametrize("canvas,kvl,causal,kv_dtype,lists", [
    (64, 18432 - 65, 0, capi.DG_BF16, False), (64, 18432 - 64, 0, capi.DG_BF16, True), (33, 18432 - 33, 33, capi.DG_F16, True),
    (32, 24576 - 33, 0, capi.DG_BF16, False), (65, 2047, 0, capi.DG_BF16, False), (65, 2048, 0, capi.DG_F16, True),
    (101, 2048, 101, capi.DG_BF16, True), (128, 8000, 60, capi.DG_BF16, True)])
def test_which_calls_keep_lists(gpu_ready, canvas, kvl, causal, kv_dtype, lists):
    """Where the thresholds-and-lists path begins without being asked for, and that it gives what the score plane gives there
    (the same kept sets: fp32 summation error)."""
    hq, hkv, hd = 16, 2, 512
    rng = np.random.default_rng(canvas + kvl)
    rms = lambda x: x / np.sqrt(np.mean(x * x, axis=-1, keepdims=True))
    q = rms(rng.standard_normal((canvas, hq, hd), dtype=np.float32))
    kv = rms(rng.standard_normal((kvl + canvas, 2, hkv, hd), dtype=np.float32))
    run = lambda flag: device_topk(canvas, hq, hkv, hd, kvl, T.adaptive_k(), q, kv, causal_rows=causal, kv_dtype=kv_dtype, flags=flag)
    got, _, _, ws = run(0)
    assert (rows_left_over(ws, canvas * hq) == 0) == lists
    assert max_abs_diff(got, run(capi.DG_ATTN_F_TOPK_SCORE_PLANE)[0]) < 2e-5


def test_workspace_of_the_score_plane_alone_is_enough(gpu_ready):
    """A caller with scratch for the score plane and no more gets the score plane's path, byte for byte."""
    import torch
    w = W.Workload("small_ws", 256, 16, 2, 512, 4000, seed=8)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    k_cfg = T.adaptive_k()
    outs = []
    plane = w.desc(flags=capi.DG_ATTN_F_TOPK_SCORE_PLANE)
    need = T.workspace_bytes(plane, k_cfg)
    assert need < T.workspace_bytes(w.desc(), k_cfg)
    for d in (plane, w.desc()):
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        outs.append(torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.int16, device="cuda"))
        T.forward(d, k_cfg, qd, kd, outs[-1], ws)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and bool((outs[0] != 0).any())


def test_thresholds_and_lists_replay_in_a_graph(gpu_ready):
    """Recorded once, replayed over other queries in the same buffers (one of them zero: rows left to the general path)."""
    import torch
    w = W.Workload("rep2", 64, 16, 2, 512, 5000, seed=32)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc(flags=capi.DG_ATTN_F_TOPK_THRESHOLD)
    k_cfg = T.adaptive_k()
    ws = T.alloc_workspace(d, k_cfg)
    out = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.int16, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        T.forward(d, k_cfg, qd, kd, out, ws)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        T.forward(d, k_cfg, qd, kd, out, ws)
    first = qd.clone()
    half = qd.numel() // 2
    for change in ("none", "half zero", "none", "shifted"):
        qd.copy_(first)
        if change == "half zero":
            qd.view(-1)[:half] = 0
        elif change == "shifted":
            qd.copy_(first.view(-1).roll(512 * 16).view(first.shape))
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        want = torch.zeros_like(out)
        T.forward(d, k_cfg, qd, kd, want, T.alloc_workspace(d, k_cfg))
        torch.cuda.synchronize()
        assert torch.equal(out, want) and bool((out != 0).any())


def test_ring_cache(gpu_ready, po):
    """Top-k over a wrapped ring (a sliding layer's storage): kept positions map to slots for the gather."""
    import torch
    canvas, hq, hkv, hd, kvl, window, ring, k = 32, 4, 2, 128, 3000, 1000, 2048, 40
    rng = np.random.default_rng(77)
    t_all = kvl + canvas
    q = rng.standard_normal((canvas, hq, hd)).astype(np.float32)
    lin = rng.standard_normal((t_all, 2, hkv, hd)).astype(np.float32)
    qb, lb = R.f32_to_bf16_bits_rne(q), R.f32_to_bf16_bits_rne(lin).reshape(lin.shape)
    ringbits = np.full((ring, 2, hkv, hd), 0x7FC0, dtype=np.uint16)          # NaN in every dead slot
    for pos in range(kvl - (window - 1), t_all):
        ringbits[pos & (ring - 1)] = lb[pos]
    d = A.make_desc(canvas, hq, hkv, hd, kvl, window=window, kv_ring_mask=ring - 1, out_dtype=capi.DG_F32)
    out = torch.zeros(canvas * hq * hd, dtype=torch.float32, device="cuda")
    cfg = (k, 0, 0, 0)
    T.forward(d, cfg, A.to_device_bits(qb.reshape(-1)), A.to_device_bits(ringbits.reshape(-1)), out, T.alloc_workspace(d, cfg))
    torch.cuda.synchronize()
    od = po.make_desc(canvas, hq, hkv, hd, kvl, window=window)
    ref = po.attention_topk_f32(od, cfg, R.bf16_bits_to_f32(qb).reshape(q.shape), R.bf16_bits_to_f32(lb).reshape(lin.shape))
    got = out.cpu().numpy().reshape(ref.shape)
    assert np.isfinite(got).all()
    assert max_abs_diff(got, ref) <= 2e-2 and mean_abs_diff(got, ref) <= 2e-3


# ------------------------------------------------------------------ properties
def test_k_at_least_the_visible_keys_is_dense_attention(gpu_ready):
    import torch
    w = W.Workload("dense", 64, 16, 2, 512, 900, causal_rows=32, seed=9)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc()
    d.out_dtype = capi.DG_F32
    dense = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.float32, device="cuda")
    A.forward(d, qd, kd, dense, None, A.alloc_workspace(d))
    k_cfg = (1024, 0, 0, 0)
    sparse = torch.zeros_like(dense)
    T.forward(d, k_cfg, qd, kd, sparse, T.alloc_workspace(d, k_cfg))
    torch.cuda.synchronize()
    a, b = dense.cpu().numpy(), sparse.cpu().numpy()
    assert max_abs_diff(a, b) <= 8e-3 and mean_abs_diff(a, b) <= 3e-4    # the dense kernel rounds P to bf16


def test_k1_is_the_value_row_of_the_best_key(gpu_ready, po):
    canvas, hq, hkv, hd, kvl = 16, 8, 2, 128, 777
    rng = np.random.default_rng(12)
    q = rng.standard_normal((canvas, hq, hd)).astype(np.float32)
    kv = rng.standard_normal((kvl + canvas, 2, hkv, hd)).astype(np.float32)
    got, ref = run_topk(po, canvas, hq, hkv, hd, kvl, (1, 0, 0, 0), q=q, kv=kv)
    vb = R.bf16_bits_to_f32(R.f32_to_bf16_bits_rne(kv[:, 1])).reshape(kvl + canvas, hkv, hd)
    for tok in range(canvas):
        for h in range(hq):
            assert any(np.array_equal(got[tok, h], vb[t, h // 4]) for t in range(kvl + canvas))
    assert max_abs_diff(got, ref) == 0.0      # N(0,1) scores at hd 128: no near-ties at the top


def test_runs_are_bit_identical_and_replay_in_a_graph(gpu_ready):
    import torch
    w = W.Workload("rep", 64, 16, 2, 512, 5000, seed=31)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc()
    k_cfg = T.adaptive_k()
    ws = T.alloc_workspace(d, k_cfg)
    outs = []
    for _ in range(3):
        out = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.int16, device="cuda")
        T.forward(d, k_cfg, qd, kd, out, ws)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    gout = torch.zeros_like(outs[0])
    with torch.cuda.stream(side):
        T.forward(d, k_cfg, qd, kd, gout, ws)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        T.forward(d, k_cfg, qd, kd, gout, ws)
    for _ in range(3):
        gout.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gout, outs[0])


def test_error_codes(gpu_ready):
    import torch
    d = A.make_desc(64, 16, 2, 512, 100)
    lib = capi.load()
    n = C.c_size_t(0)
    cfg = lambda *v: (C.c_uint32 * 4)(*v)
    assert lib.dg_attn_topk_workspace_bytes(C.byref(d), cfg(2000, 0, 0, 0), C.byref(n)) == capi.DG_ERR_SHAPE
    assert lib.dg_attn_topk_workspace_bytes(C.byref(d), cfg(256, 128, 64, 2048), C.byref(n)) == capi.DG_ERR_SHAPE
    assert lib.dg_attn_topk_workspace_bytes(C.byref(d), cfg(256, 128, 600, 512), C.byref(n)) == capi.DG_ERR_SHAPE
    d32 = A.make_desc(64, 16, 2, 512, 100, q_dtype=capi.DG_F32, kv_dtype=capi.DG_F32, out_dtype=capi.DG_F32)
    assert lib.dg_attn_topk_workspace_bytes(C.byref(d32), cfg(64, 0, 0, 0), C.byref(n)) == capi.DG_ERR_UNSUPPORTED
    assert lib.dg_attn_topk_workspace_bytes(C.byref(d), cfg(64, 0, 0, 0), C.byref(n)) == capi.DG_OK and n.value > 0
    buf = torch.zeros(1 << 20, dtype=torch.int16, device="cuda")
    small = torch.zeros(256, dtype=torch.uint8, device="cuda")
    rc = lib.dg_attn_topk_forward(C.byref(d), cfg(64, 0, 0, 0), buf.data_ptr(), buf.data_ptr(), buf.data_ptr(),
                                  small.data_ptr(), small.numel(), A.stream_handle())
    assert rc == capi.DG_ERR_WORKSPACE


def test_short_rows_give_the_same_bits_every_time(gpu_ready):
    """Rows that see few keys go straight into the candidate list; nothing of them may depend on which wave comes first."""
    canvas, hq, hkv, hd, kv_len = 300, 64, 8, 64, 2049
    rng = np.random.default_rng(6)
    q = rng.standard_normal((canvas, hq, hd)).astype(np.float32)
    kv = rng.standard_normal((kv_len + canvas, 2, hkv, hd)).astype(np.float32)
    outs = [device_topk(canvas, hq, hkv, hd, kv_len, T.adaptive_k(), q, kv, window=17)[0] for _ in range(16)]
    assert all(np.array_equal(o, outs[0]) for o in outs)
