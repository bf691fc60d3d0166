"""The watershed's pop indexes beyond what a record holds (runs of more than 2^24 pops; here the line is lowered to
just above the largest LDS frame): runs flooded from global memory on both sides of the line, beside small ones.
Whole numbers: equal to the oracle's cv::watershed, and decided by the decomposed flood."""
import numpy as np
import pytest

from tests._lib import o_cv_watershed
from tests.test_gpu_run_floods import STEPS, grid_of_runs

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("steps", ["low", "edges", "all"])
@pytest.mark.parametrize("box", [(60, 60), (80, 79), (84, 84), (120, 150)])
def test_indexes_beyond_a_record(box, steps, monkeypatch):
    from nscale_amd import gpu
    rng = np.random.default_rng(box[0])
    bgr, m = grid_of_runs(rng, 3, box, np.array(STEPS[steps], np.uint8))
    d, dm = torch.from_numpy(bgr).cuda(), torch.from_numpy(m).cuda()
    exp = o_cv_watershed(bgr, m)
    monkeypatch.setenv("NSC_WATERSHED", "fast")
    for cap in ("6401", "6800", "0"):
        monkeypatch.setenv("NSC_WS_POP_CAP", cap)
        print("pops", box, steps, cap, flush=True)
        got = gpu.cv_watershed(d, dm.clone()).cpu().numpy()
        assert np.array_equal(got, exp)
