"""The distance transform where columns' nearest zeros lie many 64-row segments away, above, below or both, beside
columns without any: planes with a few zeros only, at the edges of segments and of the column scan's steps.
Distances equal to the oracle's floats."""
import numpy as np
import pytest

from tests._lib import o_edt

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(64, 70), (65, 64), (128, 129), (640, 65), (1217, 64), (1300, 200), (200, 1300)])
def test_few_zeros(shape):
    from nscale_amd import gpu
    h, w = shape
    rng = np.random.default_rng(h + w)
    rows = sorted({r for r in (0, 63, 64, 127, 128, 575, 576, 639, 640, 1151, 1152, h - 1) if r < h})
    cases = [[(r, c)] for r in rows for c in (0, w - 1)]
    cases += [[(0, 1), (h - 1, w - 2)], [(r, (7 * r) % w) for r in rows],
              [(int(rng.integers(h)), int(rng.integers(w))) for _ in range(5)], [(h // 2, x) for x in range(w)]]
    for zeros in cases:
        img = np.full(shape, 255, np.uint8)
        for y, x in zeros:
            img[y, x] = 0
        print("far", shape, zeros[:3], flush=True)
        assert np.array_equal(gpu.dist_transform(torch.from_numpy(img).cuda()).cpu().numpy(), o_edt(img))
