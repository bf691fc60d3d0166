"""The chain's 19 x 19 disk: strips of 488 columns and 8 to 32 rows, at their edges, in planes narrower than a
lane, at odd addresses, for any constant outside; elements one pixel away from the disk.  Bytes: equal to
the oracle's."""
import numpy as np
import pytest

from tests._lib import DISK19, o_morph

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(1, 1), (1, 9), (20, 1), (3, 7), (8, 8), (19, 19), (7, 483), (9, 487), (17, 488), (33, 489), (16, 497), (40, 976), (8, 977),
          (65, 1500)]


@pytest.mark.parametrize("kind", ["erode", "dilate"])
@pytest.mark.parametrize("outside", [0, 255, 93])
def test_disk_matches_the_oracle(kind, outside):
    from nscale_amd import gpu
    disk = np.asarray(DISK19, np.uint8)
    for k, (h, w) in enumerate(SHAPES):
        rng = np.random.default_rng(k)
        for img in (rng.integers(0, 256, (h, w)), np.where(rng.random((h, w)) < 0.004, 255, 1),
                    np.where(rng.random((h, w)) < 0.004, 0, 254)):
            img = img.astype(np.uint8)
            print("disk", kind, outside, h, w, flush=True)
            flat = torch.full((h * w + 64,), 77, dtype=torch.uint8, device="cuda")
            d = flat[3:3 + h * w].view(h, w)
            d.copy_(torch.from_numpy(img))
            got = getattr(gpu, kind)(d, disk, outside).cpu().numpy()
            assert np.array_equal(got, o_morph(kind, img, disk, outside))


def test_other_elements_keep_their_kernel():
    from nscale_amd import gpu
    img = np.random.default_rng(1).integers(0, 256, (90, 500)).astype(np.uint8)
    for y, x in ((0, 9), (9, 9), (4, 1), (0, 0)):
        el = np.asarray(DISK19, np.uint8).reshape(19, 19).copy()
        el[y, x] ^= 1
        print("element", y, x, flush=True)
        assert np.array_equal(gpu.erode(torch.from_numpy(img).cuda(), el).cpu().numpy(), o_morph("erode", img, el, 255))


def test_long_strips_match_the_oracle():
    from nscale_amd import gpu
    img = np.random.default_rng(2).integers(0, 256, (3000, 12300)).astype(np.uint8)  # 26 strips of 32 rows
    got = gpu.dilate(torch.from_numpy(img).cuda(), np.asarray(DISK19, np.uint8)).cpu().numpy()
    assert np.array_equal(got, o_morph("dilate", img, np.asarray(DISK19, np.uint8), 0))
