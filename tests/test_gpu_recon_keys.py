"""Four-byte reconstruction windows over the whole range of their types: infinities, subnormals, both
zeros, the largest and lowest values, and NaN (a NaN marker's pixel stays NaN and feeds nobody, a NaN mask
bounds nothing).  Values equal to the oracle's."""
import numpy as np
import pytest

from tests._lib import o_recon

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

F = np.float32
VALUES = {"float": np.array([-np.inf, -3.4028235e38, -1.5, -1e-40, -0.0, 0.0, 1e-45, 1e-40, 2.0, 3.4028235e38, np.inf], F),
          "int": np.array([-2**31, -2**31 + 1, -70000, -1, 0, 1, 65536, 2**31 - 2, 2**31 - 1], np.int32)}
SHAPES = [(1, 1), (3, 70), (62, 63), (64, 125), (130, 66)]


def run(marker, mask, conn):
    from nscale_amd import gpu
    return gpu.imreconstruct(torch.from_numpy(marker).cuda(), torch.from_numpy(mask).cuda(), conn).cpu().numpy()


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("kind", ["float", "int"])
def test_extreme_values(kind, conn):
    for k, shape in enumerate(SHAPES):
        rng = np.random.default_rng(k)
        mask = rng.choice(VALUES[kind], shape)
        marker = np.where(rng.random(shape) < 0.3, rng.choice(VALUES[kind], shape), VALUES[kind][0])
        print("extremes", kind, shape, conn, flush=True)
        assert np.array_equal(run(marker, mask, conn), o_recon(marker, mask, conn))


@pytest.mark.parametrize("conn", [4, 8])
def test_nan(conn):
    for k, shape in enumerate(SHAPES):
        rng = np.random.default_rng(10 + k)
        mask = rng.integers(-40, 200, shape).astype(F)
        marker = (mask - rng.integers(0, 60, shape)).astype(F)
        bad_marker, bad_mask = rng.random(shape) < 0.04, rng.random(shape) < 0.04
        sign = np.where(rng.random(shape) < 0.5, F(np.nan), -F(np.nan))
        exp = o_recon(np.where(bad_marker, F(-np.inf), marker), np.where(bad_marker, F(-np.inf), np.where(bad_mask, F(np.inf), mask)),
                      conn)
        print("nan", shape, conn, flush=True)
        got = run(np.where(bad_marker, sign, marker).astype(F), np.where(bad_mask, sign, mask).astype(F), conn)
        assert np.isnan(got[bad_marker]).all()
        assert np.array_equal(got[~bad_marker], exp[~bad_marker])
