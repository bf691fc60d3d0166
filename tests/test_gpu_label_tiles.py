"""Connected components by runs and the tiled distance transform where their tiles can go wrong: planes of
one row, column or pixel, partial 64-pixel words and tiles, components that cross many tile edges or touch
at corners only, several values side by side, and distances on both sides of a tile's halo.  Whole numbers
equal to the oracle's; distances equal to its floats."""
import numpy as np
import pytest

from tests._lib import o_bwareaopen2, o_bwselect, o_cc_label, o_edt, o_imfill, oracle, ptr

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(1, 1), (1, 200), (200, 1), (2, 63), (63, 64), (64, 65), (65, 63), (64, 64), (129, 128), (127, 130), (66, 321)]


def pictures(h, w, seed):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    yield "noise", (rng.random((h, w)) < 0.55).astype(np.uint8) * 255
    yield "checks", ((x + y) % 2).astype(np.uint8) * 255
    yield "full", np.full((h, w), 255, np.uint8)
    yield "comb", np.where((x % 2 == 0) | (y == h - 1), 255, 0).astype(np.uint8)
    yield "bars", np.where((y % 2 == 0) | (x == (0 if h % 4 else w - 1)), 255, 0).astype(np.uint8)
    yield "empty", np.zeros((h, w), np.uint8)


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("shape", SHAPES)
def test_binary_components(shape, conn):
    from nscale_amd import gpu
    h, w = shape
    for k, (name, img) in enumerate(pictures(h, w, h * w + conn)):
        print("components", shape, conn, name, flush=True)
        d = torch.from_numpy(img).cuda()
        lab = gpu.cc_label(d, conn)
        exp = o_cc_label(img, conn)
        assert np.array_equal(lab.cpu().numpy(), exp)
        n = gpu.cc_relabel(lab)
        e2 = exp.copy()
        assert n == oracle().orc_cc_relabel(w, h, ptr(e2), -1)
        assert np.array_equal(lab.cpu().numpy(), e2)
        lo, hi = 2, max(3, h * w // 2)
        got, m = gpu.bwareaopen2(d, lo, hi, conn)
        ref, me = o_bwareaopen2(img, lo, hi, conn)
        assert np.array_equal(got.cpu().numpy(), ref) and m == me
        seeds = (np.random.default_rng(k).random((h, w)) < 0.02).astype(np.uint8) * 255
        s = torch.from_numpy(seeds).cuda()
        assert np.array_equal(gpu.bwselect(d, s, conn).cpu().numpy(), o_bwselect(img, seeds, conn))
        assert np.array_equal(gpu.imfill(d, s, conn).cpu().numpy(), o_imfill(img, seeds, conn))


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("shape", SHAPES)
def test_components_of_several_values(shape, conn):
    from nscale_amd import gpu
    rng = np.random.default_rng(shape[0] + 7 * shape[1] + conn)
    coarse = rng.integers(0, 3, (shape[0] // 3 + 1, shape[1] // 3 + 1)).astype(np.uint8)
    for img in (rng.integers(0, 3, shape).astype(np.uint8), np.kron(coarse, np.ones((3, 3), np.uint8))[:shape[0], :shape[1]],
                rng.integers(254, 256, shape).astype(np.uint8)):
        img = np.ascontiguousarray(img)
        print("values", shape, conn, flush=True)
        for bg in (-1, 0, 255):
            got = gpu.cc_label(torch.from_numpy(img).cuda(), conn, bg).cpu().numpy()
            assert np.array_equal(got, o_cc_label(img, conn, bg))


@pytest.mark.parametrize("shape", SHAPES + [(31, 300), (300, 33), (100, 97)])
def test_distances(shape):
    from nscale_amd import gpu
    h, w = shape
    rng = np.random.default_rng(h + 1000 * w)
    y, x = np.mgrid[0:h, 0:w]
    disc = ((y - h // 2) ** 2 + (x - w // 2) ** 2 < 30 ** 2)
    for name, img in (("noise", rng.random(shape) < 0.7), ("sparse", rng.random(shape) < 0.999), ("disc", disc),
                      ("31", (x % 63 != 31)), ("32", (x % 65 != 32) | (y % 70 != 5)), ("33", (y % 67 != 33)),
                      ("corner", (x + y) > 0), ("none", np.zeros(shape, bool))):
        img = np.ascontiguousarray(img.astype(np.uint8) * 255)
        print("distances", shape, name, flush=True)
        if img.all():
            continue  # no zero pixel: not defined
        assert np.array_equal(gpu.dist_transform(torch.from_numpy(img).cuda()).cpu().numpy(), o_edt(img))
