"""The watershed's per-pixel passes on planes of a few pixels and around their groups of four: widths that
are no multiple of four, groups that wrap over a row's end, planes too small for a group's neighbours.
Whole numbers: equal to the oracle's cv::watershed."""
import numpy as np
import pytest

from tests._lib import o_cv_watershed

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(1, 1), (1, 5), (5, 1), (2, 2), (3, 3), (3, 4), (4, 3), (3, 5), (5, 5), (6, 7), (7, 6), (4, 9),
                                   (3, 257), (257, 3), (33, 34), (34, 35), (35, 33)])
def test_small_planes_match_the_oracle(shape):
    from nscale_amd import gpu
    for seed in range(6):
        rng = np.random.default_rng(seed)
        bgr = rng.integers(0, 4, shape + (3,)).astype(np.uint8) * 60
        bgr[rng.random(shape) < 0.4] = 0
        m = np.where(rng.random(shape) < 0.15, rng.integers(1, 4, shape), 0).astype(np.int32)
        m[rng.random(shape) < 0.05] = -1
        print("small planes", shape, seed, flush=True)
        flat = torch.zeros(bgr.size + 8, dtype=torch.uint8, device="cuda")
        d = flat[seed % 3:seed % 3 + bgr.size].view(bgr.shape)
        d.copy_(torch.from_numpy(bgr))
        got = gpu.cv_watershed(d, torch.from_numpy(m).cuda()).cpu().numpy()
        assert np.array_equal(got, o_cv_watershed(bgr, m))
