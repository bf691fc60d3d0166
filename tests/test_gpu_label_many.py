"""Connected components where a tile holds as many components as it can, nearly all of them closed (they meet no other
tile) beside open ones along its edges: area opening of planes whose every pixel differs from its neighbours,
hole filling and binary reconstruction of checks and dots, plateaus of single pixels.  Whole numbers equal to the
oracle's."""
import numpy as np
import pytest

from tests._lib import o_bwareaopen2, o_cc_label, o_local_extrema, o_recon_binary, o_u8_unary

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(64, 64), (64, 65), (65, 64), (128, 128), (130, 191), (1, 129), (192, 3)]


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("shape", SHAPES)
def test_closed_and_open_components(shape, conn):
    from nscale_amd import gpu
    h, w = shape
    rng = np.random.default_rng(h + 31 * w + conn)
    y, x = np.mgrid[0:h, 0:w]
    dots = ((y % 2 == 1) & (x % 2 == 1)).astype(np.uint8) * 255
    edges = np.where((y % 64 == 63) | (x % 64 == 0), 255, dots).astype(np.uint8)  # open ones among closed ones
    four = (1 + (x % 2) + 2 * (y % 2)).astype(np.uint8)  # no two neighbours alike
    bits = rng.integers(1, 256, shape).astype(np.uint8)
    checks = ((x + y) % 2).astype(np.uint8) * 255
    for name, img in (("dots", dots), ("edges", edges), ("four", four), ("bits", bits), ("checks", checks)):
        print("many", shape, conn, name, flush=True)
        d = torch.from_numpy(img).cuda()
        assert np.array_equal(gpu.cc_label(d, conn).cpu().numpy(), o_cc_label(img, conn))
        for lo, hi in ((1, 2), (2, 1 << 30), (1, 1 << 30), (4, 5)):
            got, m = gpu.bwareaopen2(d, lo, hi, conn)
            ref, me = o_bwareaopen2(img, lo, hi, conn)
            assert np.array_equal(got.cpu().numpy(), ref) and m == me
        inv = np.where(img == 255, 0, 255).astype(np.uint8)
        for q in (img, inv):
            got = gpu.imfill_holes(torch.from_numpy(q).cuda(), conn).cpu().numpy()
            assert np.array_equal(got, o_u8_unary("orc_imfill_holes_u8", q, conn))
        seeds = (rng.random(shape) < 0.1).astype(np.uint8) * 255
        got = gpu.imreconstruct_binary(torch.from_numpy(seeds).cuda(), d, conn).cpu().numpy()
        assert np.array_equal(got, o_recon_binary(seeds, img, conn))
    f = rng.integers(0, 40, shape).astype(np.float32)
    t = torch.from_numpy(f).cuda()
    assert np.array_equal(gpu.local_maxima(t, conn).cpu().numpy(), o_local_extrema("maxima", f, conn))
    assert np.array_equal(gpu.local_minima(t, conn).cpu().numpy(), o_local_extrema("minima", f, conn))


@pytest.mark.parametrize("conn", [4, 8])
def test_many_tiles(conn):
    """More tiles than share their waves: the same with one wave a tile."""
    from nscale_amd import gpu
    rng = np.random.default_rng(conn)
    h, w = 1500, 1481
    y, x = np.mgrid[0:h, 0:w]
    for name, img in (("noise", (rng.random((h, w)) < 0.5).astype(np.uint8) * 255), ("checks", ((x + y) % 2).astype(np.uint8) * 255),
                      ("bits", rng.integers(1, 256, (h, w)).astype(np.uint8))):
        print("many tiles", conn, name, flush=True)
        d = torch.from_numpy(img).cuda()
        assert np.array_equal(gpu.cc_label(d, conn).cpu().numpy(), o_cc_label(img, conn))
        got, m = gpu.bwareaopen2(d, 2, 50, conn)
        ref, me = o_bwareaopen2(img, 2, 50, conn)
        assert np.array_equal(got.cpu().numpy(), ref) and m == me
        got = gpu.imfill_holes(d, conn).cpu().numpy()
        assert np.array_equal(got, o_u8_unary("orc_imfill_holes_u8", img, conn))
