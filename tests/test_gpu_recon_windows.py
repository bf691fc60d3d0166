"""uint8 reconstruction windows where their packed lines can go wrong: planes of fewer than 4 pixels, widths
and heights around one and two 62-pixel tiles (partial tiles, the last ones' loads clamped into the plane),
planes at odd addresses, equal values, and the largest values.  Bytes: equal to the oracle's, and nothing
written outside the plane."""
import numpy as np
import pytest

from tests._lib import o_recon

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(1, 1), (1, 2), (3, 1), (1, 3), (2, 2), (1, 4), (3, 61), (61, 3), (62, 62), (63, 63), (64, 65), (66, 62), (5, 64),
          (64, 5), (123, 124), (124, 125), (125, 126), (126, 127), (65, 187), (311, 61)]


def plane(a, off, fill):
    """a's bytes at odd offset off of a larger buffer of fill bytes."""
    buf = torch.full((a.size + 256,), fill, dtype=torch.uint8, device="cuda")
    view = buf[off:off + a.size].view(a.shape)
    view.copy_(torch.from_numpy(a))
    return buf, view


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("off", [0, 1, 7, 129])
def test_windows_match_the_oracle(conn, off):
    from nscale_amd import gpu
    for k, (h, w) in enumerate(SHAPES):
        rng = np.random.default_rng(100 * k + conn)
        for kind in ("noise", "flat", "maze"):
            mask = {"noise": rng.integers(0, 256, (h, w)), "flat": np.full((h, w), 255),
                    "maze": np.where(rng.random((h, w)) < 0.65, 255, 3)}[kind].astype(np.uint8)
            marker = np.zeros_like(mask)
            marker[rng.integers(h), rng.integers(w)] = 255
            if kind == "noise":
                marker = np.maximum(marker, (mask.astype(int) - rng.integers(0, 90, (h, w))).clip(0, 255).astype(np.uint8))
            print("windows", h, w, kind, conn, off, flush=True)
            _, dm = plane(mask, off, 255)
            _, ds = plane(marker, 256 - 127, 255)
            buf, do = plane(np.zeros_like(mask), off, 171)
            gpu.call("nsc_imreconstruct_u8", gpu._ptr(ds), gpu._ptr(dm), gpu._ptr(do), w, h, conn, gpu._stream())
            torch.cuda.synchronize()
            assert np.array_equal(do.cpu().numpy(), o_recon(marker, mask, conn))
            rest = torch.cat([buf[:off], buf[off + mask.size:]])
            assert bool((rest == 171).all())
