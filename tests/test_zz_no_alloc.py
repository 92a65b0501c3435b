"""dg_attn_forward_static, the entry point that allocates nothing: its split partial rows live in
device memory inside the library instead of a caller's workspace.  It has to give what
dg_attn_forward gives, bit for bit (same kernels), on calls that follow each other and share the
one scratch: a larger call first, a smaller one after it; calls that can do without scratch leave it alone."""
import ctypes as C

import numpy as np
import pytest

from diffgemma_amd import attention as A
from diffgemma_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


def both_ways(w, **desc_kw):
    import torch
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc(**desc_kw)
    assert capi.resolved_splits(d) > 1                      # the calls do use scratch
    assert 0 < capi.workspace_bytes(d) <= capi.load().dg_attn_static_scratch_bytes()
    n = w.canvas * w.n_q_heads
    out_a = torch.zeros(n * w.head_dim, dtype=torch.int16, device="cuda")
    out_b = torch.full((n * w.head_dim,), 0x7fc0, dtype=torch.int16, device="cuda")
    lse_a = torch.zeros(n, dtype=torch.float32, device="cuda")
    lse_b = torch.full((n,), float("nan"), dtype=torch.float32, device="cuda")
    A.forward(d, qd, kd, out_a, lse_a, A.alloc_workspace(d))
    capi.check(capi.load().dg_attn_forward_static(C.byref(d), qd.data_ptr(), kd.data_ptr(), out_b.data_ptr(),
                                                  lse_b.data_ptr(), A.stream_handle()))
    torch.cuda.synchronize()
    return out_a.cpu().numpy(), out_b.cpu().numpy(), lse_a.cpu().numpy(), lse_b.cpu().numpy()


def test_static_scratch_entry_equals_workspace_entry_on_two_calls_in_a_row(gpu_ready):
    big = W.scaled(W.config("cfg3_global"), 8192, "no_alloc_big")                                  # hd 512, 8 splits, f16 partial rows
    small = W.Workload("no_alloc_small", 64, 16, 8, 256, 1500, causal_rows=20, window=1024, seed=9)   # hd 256, fewer rows and splits
    for w, kw in ((big, {}), (small, {"n_splits": 3}), (small, {"n_splits": 2, "flags": capi.DG_ATTN_F_F32_PARTIALS})):
        out_a, out_b, lse_a, lse_b = both_ways(w, **kw)
        assert np.array_equal(out_a, out_b), w.name
        assert np.array_equal(lse_a.view(np.uint32), lse_b.view(np.uint32)), w.name
        assert np.isfinite(lse_a).all()


@pytest.mark.parametrize("w", [W.Workload("few_sliding", 64, 16, 8, 256, 4000, window=1024, seed=3), W.Workload("short_global", 64, 16, 2, 512, 250, seed=4)],
                         ids=lambda w: w.name)
def test_static_scratch_is_left_alone_by_calls_that_can_do_without(gpu_ready, w):
    """A few rows on a sliding layer, a short global range: dg_attn_forward splits their keys if it is given a workspace and runs
    without one, too.  The static entry takes the second form, so that such calls, on several streams, have no memory in common."""
    import torch
    q, kv = W.generate(w)
    qd, kd = W.device_arrays(w, q, kv)
    d = w.desc()
    assert capi.resolved_splits(d) > 1 and capi.workspace_bytes(d) > 0
    n = w.canvas * w.n_q_heads
    out = [torch.full((n * w.head_dim,), 0x7fc0, dtype=torch.int16, device="cuda") for _ in range(3)]
    lse = [torch.zeros(n, dtype=torch.float32, device="cuda") for _ in range(3)]
    A.forward(d, qd, kd, out[0], lse[0], A.alloc_workspace(d))
    A.forward(d, qd, kd, out[1], lse[1], None)
    capi.check(capi.load().dg_attn_forward_static(C.byref(d), qd.data_ptr(), kd.data_ptr(), out[2].data_ptr(), lse[2].data_ptr(),
                                                  A.stream_handle()))
    torch.cuda.synchronize()
    assert torch.equal(out[2], out[1]) and torch.equal(lse[2], lse[1])
    assert not torch.equal(out[2], out[0])                  # (the two forms round differently: it was not the first)


def test_static_scratch_entry_rejects_what_does_not_fit(gpu_ready):
    import torch
    lib = capi.load()
    d = W.config("cfg3_global").desc(flags=capi.DG_ATTN_F_F32_PARTIALS)       # 64.3 MiB of fp32 partial rows
    assert capi.workspace_bytes(d) > lib.dg_attn_static_scratch_bytes()
    dummy = torch.zeros(64, dtype=torch.int16, device="cuda")                 # never touched: the call enqueues nothing
    rc = lib.dg_attn_forward_static(C.byref(d), dummy.data_ptr(), dummy.data_ptr(), dummy.data_ptr(), None,
                                    A.stream_handle())
    assert rc == capi.DG_ERR_SCRATCH_LIMIT
    assert "scratch" in capi.strerror(rc)
    torch.cuda.synchronize()
    assert int(dummy.abs().sum()) == 0
