"""The watershed's run floods where their queues can go wrong: pushes of one pop at one level, levels on
both sides of each 64, runs that fill the image, single-pixel runs, leaves shared by several runs, and
run frames (box plus a 2-pixel margin) on both sides of the LDS sizes.  Whole numbers: equal to the
oracle's cv::watershed."""
import numpy as np
import pytest

from tests._lib import o_cv_watershed

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def grid_of_runs(rng, n, box, steps):
    """n runs of box pixels in a column, each around a seed, black (B) pixels between and inside them."""
    bh, bw = box
    h, w = n * (bh + 3) + 3, bw + 6
    bgr = np.zeros((h, w, 3), np.uint8)
    m = np.zeros((h, w), np.int32)
    for k in range(n):
        y = 3 + k * (bh + 3)
        bgr[y:y + bh, 3:3 + bw] = rng.choice(steps, size=(bh, bw, 3))
        bgr[y:y + bh, 3:3 + bw][rng.random((bh, bw)) < 0.08] = 0
        bgr[y, 3] = bgr[y + bh - 1, 2 + bw] = (9, 9, 9)  # the box's corners belong to the run's rows
        m[y + rng.integers(bh), 3 + rng.integers(bw)] = 2 * k + 1
        m[y + rng.integers(bh), 3 + rng.integers(bw)] = 2 * k + 2
    return bgr, m


STEPS = {"flat": [7], "two": [1, 255], "edges": [1, 64, 65, 66, 128, 129, 130, 192, 193, 194, 255],
         "low": [1, 2, 3, 4], "all": list(range(1, 256))}


@pytest.mark.parametrize("steps", sorted(STEPS))
@pytest.mark.parametrize("box", [(1, 1), (1, 40), (12, 28), (15, 23), (28, 28), (28, 29), (60, 28), (60, 29), (60, 60),
                                 (60, 61), (76, 76), (76, 77)])
def test_runs_match_the_oracle(box, steps):
    from nscale_amd import gpu
    rng = np.random.default_rng(box[0] * 1000 + box[1])
    bgr, m = grid_of_runs(rng, 4, box, np.array(STEPS[steps], np.uint8))
    print("runs", box, steps, flush=True)
    got = gpu.cv_watershed(torch.from_numpy(bgr).cuda(), torch.from_numpy(m).cuda()).cpu().numpy()
    assert np.array_equal(got, o_cv_watershed(bgr, m))
