"""The split kernel where its row tiles and split counts are awkward, against the CPU oracle."""
import pytest

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
