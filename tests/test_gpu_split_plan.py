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
