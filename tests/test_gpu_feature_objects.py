"""Object features where one object's statistics can go wrong: single pixels, lines, objects in the image's
corners and along its edges, constant and two-valued intensities, an object larger than a workgroup, boxes
that hold other labels.  Against the oracle with the feature tests' bounds (sums of the same terms in another
order: 1e-12 in 64 bits, 1e-5 in 32)."""
import numpy as np
import pytest

from tests.test_gpu_features import o_features

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def objects(h, w):
    lab = np.zeros((h, w), np.int32)
    parts = [(0, 0, 1, 1), (0, w - 1, 1, 1), (h - 1, 0, 1, 1), (h - 5, w - 7, 5, 7), (3, 0, 1, 9), (5, w - 1, 11, 1),
             (8, 4, 2, 2), (12, 4, 3, 40), (20, 10, 31, 47)]
    for k, (y, x, dh, dw) in enumerate(parts):
        lab[y:y + dh, x:x + dw] = k + 1
    yy, xx = np.mgrid[0:h, 0:w]
    ring = ((yy - 35) ** 2 + (xx - 100) ** 2 < 20 ** 2) & ((yy - 35) ** 2 + (xx - 100) ** 2 > 8 ** 2)
    lab[ring] = len(parts) + 1
    lab[32:38, 97:103] = len(parts) + 2  # inside the ring's box
    n = len(parts) + 2
    box = np.zeros((5, n), np.int32)
    for k in range(1, n + 1):
        ys, xs = np.nonzero(lab == k)
        box[:, k - 1] = (k, xs.min(), xs.max(), ys.min(), ys.max())
    return lab, box


@pytest.mark.parametrize("kind", ["noise", "constant", "two", "ramp"])
def test_single_objects(kind):
    from nscale_amd import gpu
    h, w = 70, 131
    rng = np.random.default_rng(3)
    gray = {"noise": rng.integers(0, 256, (h, w)), "constant": np.full((h, w), 200), "two": rng.integers(0, 2, (h, w)) * 255,
            "ramp": np.add.outer(np.arange(h), np.arange(w)) % 256}[kind].astype(np.uint8)
    lab, box = objects(h, w)
    print("feature objects", kind, flush=True)
    f = gpu.object_features(torch.from_numpy(lab).cuda(), torch.from_numpy(box).cuda(), torch.from_numpy(gray).cuda())
    exp = o_features(lab, box, gray)
    got = {k: v.cpu().numpy() for k, v in f.items()}
    assert np.array_equal(got["area"], exp["area"])
    for k in ("major_axis", "minor_axis", "eccentricity", "extent_ratio", "perimeter", "circularity"):
        assert np.allclose(got[k], exp[k], rtol=1e-12, atol=0, equal_nan=True), k
    for k in ("intensity", "gradient"):
        assert np.allclose(got[k], exp[k], rtol=1e-5, atol=1e-5, equal_nan=True), k
    assert np.array_equal(got["intensity"][:, 1:3], exp["intensity"][:, 1:3])
