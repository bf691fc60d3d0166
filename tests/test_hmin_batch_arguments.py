"""nsc_imhmin_f32_batched refuses a bad descriptor as an argument error, and before it uses any of the batch:
here in a batch whose first image is in place (the images of such a batch are copied before the passes).
No GPU is needed: the addresses are never read."""
import ctypes

import pytest

from nscale_amd._lib import ReconDesc, lib

NSC_ERR_ARG = -10
GOOD = dict(marker=None, mask=0x10000, out=0x10000, w=16, h=8, conn=8)


@pytest.mark.parametrize("bad", [dict(mask=None), dict(out=None), dict(w=0), dict(h=0), dict(w=-4, h=-4), dict(w=-4), dict(h=1 << 31),
                                 dict(conn=6)])
@pytest.mark.parametrize("at", [0, 1, 2])
def test_bad_descriptor_is_an_argument_error(bad, at):
    arr = (ReconDesc * 3)()
    for i in range(3):
        d = dict(GOOD, mask=0x10000 + 0x1000 * i, out=0x10000 + 0x1000 * i)
        if i == at:
            d.update(bad)
        arr[i] = ReconDesc(d["marker"], d["mask"], d["out"], d["w"], d["h"], d["conn"])
    L = lib()
    assert L.nsc_imhmin_f32_batched(arr, 3, ctypes.c_float(1.0), None) == NSC_ERR_ARG
    assert b"descriptor" in L.nsc_last_error()
