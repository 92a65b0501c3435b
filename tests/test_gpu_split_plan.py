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


@pytest.mark.parametrize("canvas,kv_len,causal_rows,f16,sees_masked", [
    (1024, 0, 1024, False, False), (1024, 300, 1024, True, False), (901, 0, 901, False, False), (700, 700, 700, True, False),
    (1000, 5, 1000, False, True), (800, 0, 500, False, False)])
def test_split_counts_per_row_tile(gpu_ready, po, canvas, kv_len, causal_rows, f16, sees_masked):
    """Causal rows behind a short prefix: row tiles of one split go straight to the output, the others are merged by counts of
    their own.  Rows at the edges of row tiles against the oracle; the same bits on every run."""
    import torch
    w = dataclasses.replace(W.Workload("map", canvas, 16, 2, 512, kv_len, causal_rows=causal_rows, sees_masked=sees_masked, seed=canvas),
                            kv_f16=f16)
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
