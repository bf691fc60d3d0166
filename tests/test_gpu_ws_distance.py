"""The watershed's geodesic flood over black pixels: distances that span a region of windows within 16 bits and
beyond them (a diagonal serpentine whose far end comes back beside its start; its walls are single pixels, so
no component is large), and image sizes around one region.  Whole numbers: equal to the oracle's
cv::watershed."""
import collections

import numpy as np
import pytest

from tests._lib import o_cv_watershed

REGION = 124  # pixels of a region's side


def serpentine(n, seed):
    """Corridors along the anti-diagonals of an n x n square, joined at alternate ends, then back along the
    bottom and the left side.  Returns (bgr, markers)."""
    rng = np.random.default_rng(seed)
    h, w = n + 4, n + 5  # the square's top and right sides are the image's frame
    colour = rng.integers(30, 256, (h, w, 3)).astype(np.uint8)
    free = np.zeros((h, w), bool)
    y, x = np.mgrid[0:n, 0:n]
    inner = (x + y) % 3 != 0
    for s in range(3, 2 * n - 2, 3):  # one wall pixel of each diagonal opened, at alternate ends
        x0 = max(0, s - n + 1) if (s // 3) % 2 else min(n - 1, s)
        inner[s - x0, x0] = True
    free[1:1 + n, 4:4 + n] = inner
    free[2 + n, 2:4 + n] = True  # back along the bottom, from the last corner
    free[1 + n, 3 + n] = True
    free[4:3 + n, 2] = True      # and up the left side
    free[1 + n, 3] = True        # (the walls of the two sides apart)
    free[1, 3] = True            # black beside the seed
    bgr = np.where(free[..., None], 0, colour).astype(np.uint8)
    m = np.zeros((h, w), np.int32)
    bgr[1, 4] = 9
    m[1, 4] = 1
    return bgr, m


def spread(bgr, m):
    """Largest difference of path lengths inside the first region, from the seed."""
    free = (bgr == 0).all(2)
    d = np.full(free.shape, -1)
    y, x = np.argwhere(m > 0)[0]
    q = collections.deque([(y, x)])
    d[y, x] = 0
    while q:
        y, x = q.popleft()
        for v, u in ((y, x - 1), (y, x + 1), (y - 1, x), (y + 1, x)):
            if free[v, u] and d[v, u] < 0:
                d[v, u] = d[y, x] + 1
                q.append((v, u))
    return d[:REGION, :REGION].max()


def test_serpentine_spans():
    assert 0 < spread(*serpentine(60, 1)) < 0xFFFF - 4 * 64 * 64
    assert spread(*serpentine(290, 1)) > 0xFFFF - 4 * 64 * 64


@pytest.mark.gpu
@pytest.mark.parametrize("n", [12, 53, 60, 115, 116, 117, 180, 290])
def test_serpentine_matches_the_oracle(n):
    torch = pytest.importorskip("torch")
    from nscale_amd import gpu
    bgr, m = serpentine(n, n)
    print("serpentine", bgr.shape, flush=True)
    got = gpu.cv_watershed(torch.from_numpy(bgr).cuda(), torch.from_numpy(m).cuda()).cpu().numpy()
    print("decomposed, sequential calls, reason", gpu.watershed_stats(with_reason=True), flush=True)
    assert np.array_equal(got, o_cv_watershed(bgr, m))
