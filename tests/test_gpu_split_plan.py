"""The split kernel where its row tiles and split counts are awkward, against the CPU oracle."""
import dataclasses

import numpy as np
import pytest

from diffgemma_amd import attention as A
from diffgemma_amd import capi, workloads as W
from test_gpu_parity import check_tolerances, run_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("canvas,causal_rows,hd,hq,hkv,window", [
    (1, 0, 512, 16, 2, 0), (15, 15, 512, 16, 2, 0), (17, 17, 512, 16, 2, 0), (33, 20, 512, 16, 2, 0),
    (65, 65, 256, 16, 8, 100), (43, 21, 128, 9, 3, 0)])
def test_ragged_row_tiles(gpu_ready, po, canvas, causal_rows, hd, hq, hkv, window, splits):
    """A row tile (128 stacked rows) that the canvas does not fill: the rows past the last one are copies of it, with its
    bounds, and nothing of them may show."""
    w = W.Workload("ragged", canvas, hq, hkv, hd, 333, causal_rows=causal_rows, window=window, seed=canvas)
    check_tolerances(*run_workload(po, w, n_splits=splits, flags=capi.DG_ATTN_F_SPLIT_OVER_WORKGROUPS))


@pytest.mark.parametrize("canvas,kv_len,f16", [(64, 0, False), (64, 22, True), (64, 777, False), (128, 300, True), (256, 300, False),
                                               (40, 2000, False)])
def test_library_chosen_splits(gpu_ready, po, canvas, kv_len, f16):
    """head_dim 512 with the split count left to the library: from one tile a split to several, even and uneven."""
    w = dataclasses.replace(W.Workload("chosen", canvas, 16, 2, 512, kv_len, causal_rows=canvas // 3, seed=kv_len), kv_f16=f16)
    toks = np.unique(np.linspace(0, canvas - 1, 20).round().astype(np.uint32))
    check_tolerances(*run_workload(po, w, toks=toks))


def test_smaller_scratch_takes_fewer_splits(gpu_ready):
    """Scratch for splits of at least six key tiles is always enough (what a caller may have sized by an earlier library):
    the call takes that split count, the same bits as asking for it.  Less than that is refused."""
    import torch
    w = W.Workload("scratch", 64, 16, 2, 512, 777, seed=5)
    d, few = w.desc(), w.desc(n_splits=4)
    need, least = capi.workspace_bytes(d), capi.workspace_bytes(few)
    assert capi.resolved_splits(d) > 4 and need > least
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    outs = []
    for desc, size in ((few, least), (d, least), (d, need - 256), (d, need)):
        out = torch.zeros(w.canvas * w.n_q_heads * w.head_dim, dtype=torch.int16, device="cuda")
        A.forward(desc, qd, kd, out, None, torch.empty(size, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]) and not torch.equal(outs[0], outs[3])
    with pytest.raises(RuntimeError):
        A.forward(d, qd, kd, outs[0], None, torch.empty(least - 256, dtype=torch.uint8, device="cuda"))


# (canvas, prefix, causal rows, f16 cache, sees masked) of calls with a split map, and the order of its units (test_split_map.py holds it to
# the rules)
MAP_FORMS = [
    (1024, 0, 1024, False, False, "by row tile"), (1024, 300, 1024, True, False, "by row tile"), (901, 0, 901, False, False, "by row tile"),
    (700, 700, 700, True, False, "by row tile"), (1000, 5, 1000, False, True, "by row tile"), (800, 0, 500, False, False, "by row tile"),
    (700, 5060, 700, False, False, "by split"), (520, 4000, 520, True, False, "by split")]


def map_workload(canvas, kv_len, causal_rows, f16, sees_masked):
    return dataclasses.replace(W.Workload("map", canvas, 16, 2, 512, kv_len, causal_rows=causal_rows, sees_masked=sees_masked, seed=canvas), kv_f16=f16)


@pytest.mark.parametrize("canvas,kv_len,causal_rows,f16,sees_masked", [f[:5] for f in MAP_FORMS])
def test_split_counts_per_row_tile(gpu_ready, po, canvas, kv_len, causal_rows, f16, sees_masked):
    """Causal rows with a split map: row tiles of one split go straight to the output, the others are merged by counts of their own,
    with the units in either order.  Rows at the edges of row tiles against the oracle; the same bits on every run."""
    import torch
    w = map_workload(canvas, kv_len, causal_rows, f16, sees_masked)
    toks = np.unique(np.concatenate([np.arange(0, canvas, 61), np.arange(15, canvas, 160), np.arange(16, canvas, 160),
                                     [causal_rows - 1, min(causal_rows, canvas - 1), canvas - 1]])).astype(np.uint32)
    check_tolerances(*run_workload(po, w, toks=toks))
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d, first = w.desc(), None
    ws = A.alloc_workspace(d)
    for _ in range(3):
        out = torch.full((canvas * 16 * 512,), -1, dtype=torch.int16, device="cuda")
        A.forward(d, qd, kd, out, None, ws)
        torch.cuda.synchronize()
        first = out if first is None else first
        assert torch.equal(out, first)
        ws.fill_(255)      # NaN everywhere: nothing of an earlier call is read


def test_device_prefix_with_the_scratch_of_a_split_map(gpu_ready, po):
    """The entry point that reads the prefix on the device has one count for all row tiles and runs in the same scratch."""
    import torch
    w = W.Workload("map_dev", 1024, 16, 2, 512, 0, causal_rows=1024, seed=2)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc()
    outs = []
    for run in (lambda o: A.forward(d, qd, kd, o, None, A.alloc_workspace(d)),
                lambda o: A.forward_dev(d, A.device_step_params(0), qd, kd, o, None, A.alloc_workspace(d)),
                lambda o: A.forward(w.desc(n_splits=2), qd, kd, o, None, A.alloc_workspace(w.desc(n_splits=2)))):
        out = torch.zeros(w.canvas * 16 * 512, dtype=torch.int16, device="cuda")
        run(out)
        torch.cuda.synchronize()
        outs.append(out.view(torch.bfloat16).float())
    assert torch.equal(outs[1], outs[2])
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -7 * outs[1].abs().max()


@pytest.mark.parametrize("canvas,kv_len,f16", [(512, 0, False), (600, 200, True), (560, 90, False), (350, 300, False), (333, 333, True)])
def test_split_counts_of_short_shares(gpu_ready, po, canvas, kv_len, f16):
    """Prompts whose shares are a few key tiles against the oracle and against two equal splits."""
    import torch
    w = dataclasses.replace(W.Workload("short_map", canvas, 16, 2, 512, kv_len, causal_rows=canvas, seed=canvas), kv_f16=f16)
    check_tolerances(*run_workload(po, w, toks=np.unique(np.append(np.arange(0, canvas, 31), canvas - 1)).astype(np.uint32)))
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    outs = []
    for desc in (w.desc(n_splits=2), w.desc()):
        out = torch.zeros(canvas * 16 * 512, dtype=torch.int16, device="cuda")
        A.forward(desc, qd, kd, out, None, torch.empty(capi.workspace_bytes(desc), dtype=torch.uint8, device="cuda"))
        outs.append(out)
    torch.cuda.synchronize()
    x, y = (o.view(torch.bfloat16).float() for o in outs)
    # sums that differ by the rounding of partial rows, 2^-12 of them, can round to neighbouring bf16 values: one step, 2^-7 of the value at most
    assert float((x - y).abs().max()) <= 2.0 ** -7 * float(x.abs().max())


@pytest.mark.parametrize("canvas,alone", [(1024, 384), (901, 320), (700, 256)])
@pytest.mark.parametrize("f16", [False, True])
def test_rows_of_one_share_are_fp32_until_the_output(gpu_ready, canvas, alone, f16):
    """Behind no prefix the shares of a split map are 12, 10 and 8 key tiles long: row tiles that see no more (`alone` rows) have no
    16-bit partial rows, the bits of a call in one split."""
    import torch
    w = dataclasses.replace(W.Workload("alone", canvas, 16, 2, 512, 0, causal_rows=canvas, seed=canvas), kv_f16=f16)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    outs = []
    for desc in (w.desc(n_splits=1), w.desc()):
        out = torch.zeros(canvas, 16 * 512, dtype=torch.int16, device="cuda")
        A.forward(desc, qd, kd, out, None, torch.empty(max(capi.workspace_bytes(desc), 256), dtype=torch.uint8, device="cuda"))
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0][:alone], outs[1][:alone]) and not torch.equal(*outs)


@pytest.mark.parametrize("hd,hkv,splits", [(512, 2, 3), (256, 8, 2)])
def test_device_prefix_and_an_explicit_split_count(gpu_ready, hd, hkv, splits):
    """With n_splits given, the entry that reads the prefix on the device, planned for a longer one, gives the host entry's bits: causal
    rows that would have split counts of their own, and a range that would be one launch."""
    import torch
    kv_len, planned = 300, 700
    w = W.Workload("dev_splits", 256, 16, hkv, hd, planned, causal_rows=256, seed=7)
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    mk = lambda n: A.make_desc(w.canvas, 16, hkv, hd, n, causal_rows=256, layout="head_major", t_cap=w.t_all, n_splits=splits,
                               flags=capi.DG_ATTN_F_F16_PARTIALS)
    host, dev = mk(kv_len), mk(planned)
    assert capi.resolved_splits(host) == capi.resolved_splits(dev) == splits
    outs, lses = [], []
    for run in (lambda o, l: A.forward(host, qd, kd, o, l, A.alloc_workspace(host)),
                lambda o, l: A.forward_dev(dev, A.device_step_params(kv_len), qd, kd, o, l, A.alloc_workspace(dev))):
        out = torch.zeros(w.canvas * 16 * hd, dtype=torch.int16, device="cuda")
        lse = torch.zeros(w.canvas * 16, device="cuda")
        run(out, lse)
        torch.cuda.synchronize()
        outs.append(out)
        lses.append(lse)
    assert torch.equal(*outs) and torch.equal(*lses)


@pytest.mark.parametrize("canvas,kv_len,causal_rows,hkv,window,ring,f16", [
    (64, 4000, 0, 8, 1024, 2048, False), (33, 5000, 33, 8, 1024, 2048, True), (112, 3001, 40, 8, 1024, 0, False),
    (100, 830, 0, 8, 0, 0, True), (17, 1100, 17, 4, 1024, 2048, False)])
def test_short_range_shared_by_workgroups(gpu_ready, po, canvas, kv_len, causal_rows, hkv, window, ring, f16):
    """A few canvas rows over most of a window: several workgroups to a row tile of the one-launch kernel, their rows merged.
    Against the oracle (ring caches against the linear one, bit for bit); without scratch the call is one launch."""
    import torch
    w = dataclasses.replace(W.Workload("share", canvas, 16, hkv, 256, kv_len, causal_rows=causal_rows, window=window, seed=canvas), kv_f16=f16)
    d = w.desc()
    assert capi.resolved_splits(d) > 1 and capi.workspace_bytes(d) > 0
    check_tolerances(*run_workload(po, w))
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    dt = torch.int16
    shared, one, ringed = (torch.zeros(canvas * 16 * 256, dtype=dt, device="cuda") for _ in range(3))
    lse = torch.zeros(canvas * 16, device="cuda")
    ws = A.alloc_workspace(d)
    ws.fill_(255)
    A.forward(d, qd, kd, shared, lse, ws)
    A.forward(d, qd, kd, one, None, None)
    assert not torch.equal(shared, one)
    assert (shared.view(torch.bfloat16).float() - one.view(torch.bfloat16).float()).abs().max() <= 1.6e-2 * 2      # two bf16-P roundings, two stores
    if ring:
        planes = kd.view(dt).view(2, hkv, w.t_all, 256)
        rd = torch.zeros(2, hkv, ring, 256, dtype=dt, device="cuda")
        lo = max(0, w.t_all - ring)
        rd[:, :, torch.arange(lo, w.t_all, device="cuda") % ring] = planes[:, :, lo:]
        dr = A.make_desc(canvas, 16, hkv, 256, kv_len, causal_rows=causal_rows, window=window, kv_ring_mask=ring - 1, layout="head_major",
                         t_cap=ring, kv_dtype=d.kv_dtype, flags=d.flags)
        A.forward(dr, qd, rd, ringed, None, A.alloc_workspace(dr))
        assert torch.equal(ringed, shared)
    step = A.device_step_params(kv_len)
    A.forward_dev(d, step, qd, kd, one, None, ws)
    torch.cuda.synchronize()
    assert torch.equal(one, shared)
    # a device prefix far below the planned one: most workgroups of a row tile have no keys
    small = A.make_desc(canvas, 16, hkv, 256, 100, causal_rows=causal_rows, window=window, layout="head_major", t_cap=w.t_all, kv_dtype=d.kv_dtype,
                        flags=d.flags)
    A.forward_dev(d, A.device_step_params(100), qd, kd, one, None, ws)
    A.forward(small, qd, kd, shared, None, A.alloc_workspace(small))
    torch.cuda.synchronize()
    assert (shared.view(torch.bfloat16).float() - one.view(torch.bfloat16).float()).abs().max() <= 1.6e-2 * 2


@pytest.mark.parametrize("hd,hkv,f32_parts,out_f32", [(512, 2, False, False), (256, 8, False, False), (512, 2, True, False),
                                                      (512, 2, True, True), (256, 8, True, False), (64, 2, True, True)])
def test_merge_at_once_gives_the_bits_of_the_streamed_merge(gpu_ready, hd, hkv, f32_parts, out_f32):
    """Every instance of the merge that asks for all partial rows up front, on ragged rows, flat and peaked."""
    import torch
    canvas, kv_len = 37, 2000
    for n in (2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 16):
        for gain in (1.0, 0.05):
            w = W.Workload("merge", canvas, 16, hkv, hd, kv_len, causal_rows=5, seed=n)
            q, kv = W.generate(w)
            qd, kd = W.device_arrays(w, q, kv)
            qd = (qd.view(torch.bfloat16).float() * gain).to(torch.bfloat16)
            flag = capi.DG_ATTN_F_F32_PARTIALS if f32_parts else capi.DG_ATTN_F_F16_PARTIALS
            got = []
            for extra in (0, capi.DG_ATTN_F_STREAMED_MERGE):
                d = A.make_desc(canvas, 16, hkv, hd, kv_len, causal_rows=5, layout="head_major", t_cap=w.t_all, n_splits=n, flags=flag | extra |
                                capi.DG_ATTN_F_SPLIT_OVER_WORKGROUPS, out_dtype=capi.DG_F32 if out_f32 else capi.DG_BF16)
                out = torch.zeros(canvas, 16, hd, dtype=torch.float32 if out_f32 else torch.bfloat16, device="cuda")
                lse = torch.zeros(canvas, 16, device="cuda")
                A.forward(d, qd, kd, out, lse, A.alloc_workspace(d))
                torch.cuda.synchronize()
                got.append((out, lse))
            assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# (canvas, prefix, heads, KV heads, head_dim, causal rows), and the order of the units, how the rows are merged and the partial rows' type
# (test_split_map.py holds them to the rules)
ORDER_FORMS = [
    (1, 300, 16, 2, 512, 0, "by split, in turn, f32"), (16, 100, 16, 2, 512, 0, "by row tile, in runs, f32"),
    (32, 400, 16, 2, 512, 0, "by row tile, in runs, f16"), (40, 400, 16, 2, 512, 0, "by split, in turn, f16"),
    (64, 120, 16, 2, 512, 0, "by row tile, in runs, f32"), (49, 700, 16, 2, 512, 30, "by row tile, in runs, f16"),
    (64, 2496, 16, 2, 512, 0, "by row tile, in turn, f16"), (64, 2497, 16, 2, 512, 0, "by split, in turn, f16"),
    (72, 1528, 16, 2, 512, 30, "by row tile, in runs, f16"), (72, 1529, 16, 2, 512, 0, "by split, in turn, f16"),
    (200, 400, 16, 2, 512, 0, "by row tile, in runs, f16"), (250, 900, 16, 2, 512, 0, "by row tile, in runs, f16"),
    (37, 500, 8, 8, 512, 37, "by split, in runs, f16"), (65, 700, 9, 3, 512, 0, "by split, in turn, f16"),
    (140, 700, 9, 3, 512, 0, "by row tile, in runs, f16"), (64, 300, 16, 1, 512, 0, "by row tile, in runs, f16"),
    (37, 3500, 16, 16, 256, 0, "by split, in turn, f16"), (64, 2100, 16, 2, 256, 0, "by row tile, in runs, f16"),
    (64, 2100, 16, 2, 128, 0, "by split, in turn, f16"), (64, 4000, 16, 8, 256, 0, "shared, in runs, f32")]


def order_workload(canvas, kv_len, hq, hkv, hd, causal_rows):
    return W.Workload("order", canvas, hq, hkv, hd, kv_len, causal_rows=causal_rows, window=1024 if hkv == 8 and hd == 256 else 0, seed=canvas)


ORDER_FLAGS = capi.DG_ATTN_F_KV_CACHED      # (the order also depends on where the rows come from)


@pytest.mark.parametrize("canvas,kv_len,hq,hkv,hd,causal_rows", [f[:6] for f in ORDER_FORMS])
def test_units_by_row_tile_and_rows_merged_where_they_were_written(gpu_ready, po, canvas, kv_len, hq, hkv, hd, causal_rows):
    """Either order of the workgroups, with row tiles that are cut by an XCD's run and rows that do not fill one, against the oracle; and
    the merge that asks for all rows at once, its rows in turn or in runs, gives the bits of the one that looks at the weights first."""
    import torch
    w = order_workload(canvas, kv_len, hq, hkv, hd, causal_rows)
    d = w.desc(flags=ORDER_FLAGS)
    assert capi.resolved_splits(d) > 1
    check_tolerances(*run_workload(po, w, flags=ORDER_FLAGS, toks=np.unique(np.linspace(0, canvas - 1, 12).round().astype(np.uint32))))
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    got = []
    for flags in (d.flags, d.flags | capi.DG_ATTN_F_STREAMED_MERGE):
        d.flags = flags
        out = torch.zeros(canvas * hq * hd, dtype=torch.int16, device="cuda")
        lse = torch.zeros(canvas * hq, device="cuda")
        A.forward(d, qd, kd, out, lse, A.alloc_workspace(d))
        torch.cuda.synchronize()
        got.append((out, lse))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
