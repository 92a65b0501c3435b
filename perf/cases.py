"""What a program that uses this package has it do, as cases that can be timed and compared.

A case is one unit of work at the package's boundary:

* ``layer``: one decoder layer's attention step, the way the step encoder issues it: the producer (per-head RMSNorm,
  RoPE, cache write of the canvas rows), then attention over the cached prefix and the canvas.  ``entry`` says through
  which of the two boundaries: ``dispatch`` is the reference's argument block (bf16 rows, f16 slot-major cache,
  truncating stores), ``forward`` the descriptor entries (bf16 head-major cache, log-sum-exp wanted).  ``full`` picks the
  layer type (global: 2 KV heads x 512, linear cache; sliding: 8 KV heads x 256, window 1024, ring cache), ``rows`` the
  canvas, ``causal_rows`` the mask (0 denoise, rows prefill, in between a partly committed canvas), ``topk`` the
  reference's sparse attention with its production rule instead of the dense one.
* ``iteration``: one denoise iteration's attention work, all 30 layers recorded once in a HIP graph and replayed.
* ``swap``: a conversation swap: the live cache of all layers gathered into a blob, another conversation's scattered.

Cached rows have unit RMS, as the producer leaves them.  ``q_gain`` is the query norm weight: at 1 the scores of a row
spread over sqrt(head_dim) (peaked rows), at 0.05 over about one (flat rows), and trained models lie in between.
Norm weights are constant so that a pass over rows that are already normalised leaves their distribution alone.
"""
import ctypes as C
import math

import torch

from diffgemma_amd import attention as A
from diffgemma_amd import attention_topk as T
from diffgemma_amd import capi, step_kv
from diffgemma_amd.schedule import DenoiseSchedule

HQ = step_kv.STEP_NQ_HEADS
WINDOW = step_kv.SLIDING_WINDOW
RING = step_kv.KV_RING_SLOTS


def _layer(name, full, entry, rows, prefix, causal_rows=0, topk=False, q_gain=1.0):
    c = {"kind": "layer", "full": full, "entry": entry, "rows": rows, "prefix": prefix, "causal_rows": causal_rows,
         "topk": topk, "q_gain": q_gain}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the first turn of a conversation: a short canvas behind a prompt of a few words; nothing but latency
        _layer("first_turn_sliding", False, "dispatch", 64, 22),
        # a chat a few messages in: a global layer whose keys are few
        _layer("short_chat_global", True, "forward", 256, 777, q_gain=0.25),
        # the layer a step runs 25 times of 30, on either storage
        _layer("denoise_sliding", False, "forward", 256, 4096),
        _layer("denoise_sliding_f16", False, "dispatch", 256, 33003, q_gain=0.25),
        # the global layer at the benchmark's depth, half of the canvas committed
        _layer("denoise_global_32k", True, "forward", 256, 32768, causal_rows=128),
        # the depth of the reference's own long-context figures, on its storage
        _layer("denoise_global_100k_f16", True, "dispatch", 256, 100256, q_gain=0.25),
        # a prompt's first super-chunk (triangular mask, empty cache) and one deep in a long document
        _layer("prefill_global_first", True, "forward", 1024, 0, causal_rows=1024),
        _layer("prefill_global_32k", True, "forward", 1024, 32768, causal_rows=1024, q_gain=0.25),
        # the last, ragged chunk of a prompt on a sliding layer
        _layer("prefill_sliding_tail", False, "forward", 901, 8192, causal_rows=901),
        # the global layer with the reference's sparse default
        _layer("topk_global_32k", True, "forward", 256, 32768, topk=True),
        {"name": "denoise_iteration_32k", "kind": "iteration", "prefix": 32768},
        {"name": "conversation_swap_8k", "kind": "swap", "prefix": 7777},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("layer", "topk", "iteration", "swap"), (12, 3, 2, 2))[0]
    if kind == "iteration":
        return {"kind": kind, "prefix": _log_int(rng, 1024, 32000)}
    if kind == "swap":
        return {"kind": kind, "prefix": _log_int(rng, 200, 20000)}
    entry = rng.choice(("dispatch", "forward"))
    q_gain = rng.choice((1.0, 0.25, 0.05))
    if kind == "topk":
        rows = rng.choice((64, 128, 256, 256))
        return _layer(None, True, entry, rows, _log_int(rng, 3000, 50000), topk=True, q_gain=q_gain)
    full = rng.random() < 0.6
    if rng.random() < 0.35:      # prompt: up to a super-chunk of rows, any count
        rows = _log_int(rng, 40, 1024)
        return _layer(None, full, entry, rows, rng.choice((0, _log_int(rng, 60, 36000))), causal_rows=rows, q_gain=q_gain)
    rows = rng.choice((64, 128, 256, 256, 256))
    committed = rng.randrange(1, rows) if entry == "forward" and rng.random() < 0.3 else 0
    return _layer(None, full, entry, rows, _log_int(rng, 16, 125000 if full else 60000), causal_rows=committed, q_gain=q_gain)


# ---- preparation ------------------------------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _unit_rows(g, rows, hd, dtype):
    """[rows, hd] of unit RMS in `dtype`, made in pieces (a long cache would not want its fp32 image beside it)."""
    x = torch.empty(rows, hd, dtype=dtype, device="cuda")
    for at in range(0, rows, 1 << 17):
        part = torch.randn(min(1 << 17, rows - at), hd, device="cuda", generator=g)
        x[at:at + (1 << 17)] = (part / part.pow(2).mean(-1, keepdim=True).sqrt()).to(dtype)
    return x


def _shape(case):
    """(head_dim, KV heads, cache slots, ring mask, window) of a layer."""
    t_all = case["prefix"] + case["rows"]
    if case["full"]:
        return 512, 2, t_all, 0, 0
    return 256, 8, RING, RING - 1, WINDOW


def _prepare_layer(case, seed):
    g = _generator(seed)
    hd, hkv, slots, ring_mask, window = _shape(case)
    rows, prefix, t_all = case["rows"], case["prefix"], case["prefix"] + case["rows"]
    dispatch = case["entry"] == "dispatch"
    kv_dtype = torch.float16 if dispatch else torch.bfloat16
    s = {"case": case, "lib": capi.load()}
    s["cache"] = _unit_rows(g, 2 * hkv * slots, hd, kv_dtype)
    s["q"] = torch.randn(rows, HQ, hd, device="cuda", generator=g).to(torch.bfloat16)
    s["k"] = torch.randn(rows, hkv, hd, device="cuda", generator=g).to(torch.bfloat16)
    s["v"] = torch.randn(rows, hkv, hd, device="cuda", generator=g).to(torch.bfloat16)
    s["norm_w"] = torch.ones(2, hd, dtype=torch.bfloat16, device="cuda")      # query weights, then key weights
    s["norm_w"][0] *= case["q_gain"]
    s["out"] = torch.zeros(rows, HQ, hd, dtype=torch.bfloat16, device="cuda")
    s["outputs"] = {"out": s["out"], "q": s["q"]}
    if not case["full"]:
        s["outputs"]["k"] = s["k"]       # (a global layer's V is the raw k projection, which stays)
    # the slots this pass writes: one run, or two where the ring wraps
    planes = s["cache"].view(slots, 2, hkv, hd) if dispatch else s["cache"].view(2, hkv, slots, hd)
    first = prefix & ring_mask if ring_mask else prefix
    for n, (a, b) in enumerate(((first, min(first + rows, slots)), (0, max(0, first + rows - slots)))):
        if b > a:
            s["outputs"]["cache%d" % n] = planes[a:b] if dispatch else planes[:, :, a:b]
    s["k_cfg"] = T.adaptive_k()
    if dispatch:
        L, P = capi.LayerOffsets(), A.step_params(prefix)
        L.q_norm, L.k_norm, L.v_proj = 0, hd * 2, 0 if case["full"] else 1
        L.head_dim, L.n_kv_heads, L.is_full, L.kv_ring_mask = hd, hkv, int(case["full"]), ring_mask
        dims = capi.AttnDims(rows, HQ, int(case["causal_rows"] > 0), window)
        s["L"], s["P"], s["dims"], s["cfg"] = L, P, dims, (C.c_uint32 * 4)(*s["k_cfg"])
        n = C.c_size_t(0)
        if case["topk"]:
            capi.check(s["lib"].dg_attention_topk_state_bytes(C.byref(L), C.byref(dims), prefix, s["cfg"], C.byref(n)))
        else:
            capi.check(s["lib"].dg_attention_state_bytes(C.byref(L), C.byref(dims), prefix, C.byref(n)))
        s["state"] = torch.empty(max(n.value, 256), dtype=torch.uint8, device="cuda")
        s["dbg"] = torch.zeros(4, dtype=torch.int32, device="cuda")
        s["outputs"]["dbg"] = s["dbg"]
        return s
    rd = capi.RopeDesc()
    rd.canvas, rd.n_q_heads, rd.n_kv_heads, rd.head_dim = rows, HQ, hkv, hd
    rd.kv_len, rd.kv_write_end, rd.kv_ring_mask = prefix, 0xFFFFFFFF, ring_mask
    rd.is_full, rd.v_from_k, rd.kv_dtype = int(case["full"]), int(case["full"]), capi.DG_BF16
    rd.k_tok_stride, rd.k_head_stride = hd, slots * hd
    rd.v_base_off, rd.v_tok_stride, rd.v_head_stride = hkv * slots * hd, hd, slots * hd
    s["rope"] = rd
    s["desc"] = A.make_desc(rows, HQ, hkv, hd, prefix, causal_rows=case["causal_rows"], window=window,
                            kv_ring_mask=ring_mask, layout="head_major", t_cap=slots,
                            flags=capi.DG_ATTN_F_F16_PARTIALS)      # V rows are RMS-normalised: far inside f16's range
    if case["topk"]:
        s["ws"] = T.alloc_workspace(s["desc"], s["k_cfg"])
    else:
        s["ws"] = A.alloc_workspace(s["desc"])
        s["lse"] = torch.zeros(rows, HQ, dtype=torch.float32, device="cuda")
        s["outputs"]["lse"] = s["lse"]
    return s


def _prepare_iteration(case, seed):
    sched = DenoiseSchedule(kv_len=case["prefix"], seed=seed).build()
    for lay in sched.layers:
        lay.q_norm_w.view(torch.bfloat16).fill_(1.0)
        lay.k_norm_w.view(torch.bfloat16).fill_(1.0)
    sched.regenerate(0)
    sched.run_eager()         # (code objects load outside the recording)
    torch.cuda.synchronize()
    sched.regenerate(0)
    sched.capture()
    outputs = [t for lay in sched.layers for t in (lay.out.view(torch.bfloat16), lay.lse)]
    return {"case": case, "sched": sched, "outputs": outputs}


def _prepare_swap(case, seed):
    g = _generator(seed)
    layers = step_kv.build_layout(case["prefix"] + step_kv.CANVAS)
    arr = step_kv.kv_layers(layers)
    cache = _unit_rows(g, step_kv.kv_cache_total_bytes(layers) // 512, 256, torch.float16)
    other = _unit_rows(g, step_kv.snapshot_bytes(arr, case["prefix"]) // 512, 256, torch.float16)
    return {"case": case, "arr": arr, "cache": cache, "other": other.view(torch.uint8).view(-1)}


def prepare(case, seed):
    return {"layer": _prepare_layer, "iteration": _prepare_iteration, "swap": _prepare_swap}[case["kind"]](case, seed)


# ---- one pass ---------------------------------------------------------------------------------------------------------

def _run_dispatch(s):
    """The layer through the reference's argument block, as its encoder would issue it."""
    lib, stream = s["lib"], A.stream_handle()
    L, P, dims, dbg = C.byref(s["L"]), C.byref(s["P"]), C.byref(s["dims"]), s["dbg"].data_ptr()
    q, cache, out, state = s["q"].data_ptr(), s["cache"].data_ptr(), s["out"].data_ptr(), s["state"]
    capi.check(lib.dg_qk_rope_kv_dispatch(q, s["k"].data_ptr(), s["v"].data_ptr(), cache, s["norm_w"].data_ptr(), L, P, dims,
                                          dbg, stream))
    if s["case"]["topk"]:
        capi.check(lib.dg_attention_topk_dispatch(q, cache, out, L, P, dims, s["cfg"], dbg, state.data_ptr(), state.numel(),
                                                  stream))
    else:
        capi.check(lib.dg_attention_dispatch(q, cache, out, L, P, dims, dbg, state.data_ptr(), state.numel(), stream))


def _run_forward(s):
    """The layer through the descriptor entries, as the 30-layer schedule issues it."""
    w = s["norm_w"]
    capi.check(s["lib"].dg_qk_rope_kv(C.byref(s["rope"]), s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                      s["cache"].data_ptr(), w.data_ptr(), w.data_ptr() + w.stride(0) * w.element_size(),
                                      None, A.stream_handle()))
    if s["case"]["topk"]:
        T.forward(s["desc"], s["k_cfg"], s["q"], s["cache"], s["out"], s["ws"])
    else:
        A.forward(s["desc"], s["q"], s["cache"], s["out"], s["lse"], s["ws"])


def run(s):
    kind = s["case"]["kind"]
    if kind == "iteration":
        s["sched"].replay()
        return s["outputs"]
    if kind == "swap":
        parked = step_kv.gather_kv_prefix(s["cache"], s["arr"], s["case"]["prefix"])
        step_kv.scatter_kv_prefix(s["cache"], s["arr"], s["case"]["prefix"], s["other"])
        s["other"] = parked
        return parked, s["cache"]
    (_run_dispatch if s["case"]["entry"] == "dispatch" else _run_forward)(s)
    return s["outputs"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _layer_work(case):
    hd, hkv, _, _, window = _shape(case)
    rows, prefix, causal = case["rows"], case["prefix"], case["causal_rows"]
    t_all = prefix + rows
    if case["entry"] == "dispatch" and causal:
        causal = rows
    lo_bidirectional = max(0, prefix - (window - 1)) if window else 0
    pairs, kept, first = 0, 0, t_all
    for r in range(rows):
        if r < causal:
            lo, hi = (max(0, prefix + r - (window - 1)) if window else 0), prefix + r + 1
        else:
            lo, hi = lo_bidirectional, t_all
        pairs += hi - lo
        kept += min(hi - lo, min(max((hi - lo) // 128, 64), 512))
        first = min(first, lo)
    row_bytes = 2 * hd
    kv_read = 2 * hkv * (t_all - first) * row_bytes
    canvas = rows * row_bytes * (HQ + (hkv if case["full"] else 2 * hkv))      # projections in
    canvas += rows * row_bytes * (HQ + 2 * hkv + (0 if case["full"] else hkv)) # rotated rows and cache rows out
    canvas += rows * row_bytes * HQ                                            # result out
    flops = 2.0 * hd * HQ * (pairs + (kept if case["topk"] else pairs))
    return {"bytes": float(kv_read + canvas), "flops": flops}


def work(case):
    if case["kind"] == "swap":
        layers = step_kv.build_layout(case["prefix"] + step_kv.CANVAS)
        blob = sum(min(case["prefix"], lay.slots) * 2 * lay.n_kv_heads * lay.head_dim * 2 for lay in layers)
        return {"bytes": 4.0 * blob, "flops": 0.0}          # out of the cache and back, each read and written
    if case["kind"] == "iteration":
        one = {full: _layer_work(_layer(None, full, "forward", step_kv.CANVAS, case["prefix"])) for full in (True, False)}
        n_full = len(step_kv.FULL_LAYERS)
        return {k: n_full * one[True][k] + (step_kv.N_LAYERS - n_full) * one[False][k] for k in ("bytes", "flops")}
    return _layer_work(case)


def tolerance(case):
    if case["kind"] == "swap":
        return "exact"
    return {"rel": 1e-2}       # bf16 rows and probabilities of 8 significant bits
