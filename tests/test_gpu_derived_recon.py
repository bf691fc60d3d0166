"""h-minima and local extrema read their mask and marker from the image itself: against the oracle at tile
edges (62-pixel windows), both signs, flat and signed-zero images, in place, and overlapping batches."""
import numpy as np
import pytest

from tests._lib import o_imhmin, o_local_extrema

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _image(h, w, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "levels":
        img = rng.integers(-6, 7, (h, w)).astype(np.float32)
    elif kind == "zeros":  # signed zeros and a few dips
        img = np.where(rng.random((h, w)) < 0.5, -0.0, 0.0).astype(np.float32)
        img[rng.random((h, w)) < 0.02] = -3.5
    else:  # a negated distance map with the background far below, as the chain makes it
        img = -np.minimum(rng.random((h, w)) * 9, 8).astype(np.float32)
        img[rng.random((h, w)) < 0.4] = -np.finfo(np.float32).max
    return img


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("kind", ["levels", "zeros", "far"])
@pytest.mark.parametrize("h,w", [(1, 1), (62, 63), (61, 125), (130, 64)])
def test_hmin_and_extrema(h, w, kind, conn):
    from nscale_amd import gpu
    img = _image(h, w, kind, h + w + conn)
    d = torch.from_numpy(img).cuda()
    print("derived", h, w, kind, conn, flush=True)
    hm = gpu.imhmin(d, 1.5, conn)
    mx, mn = gpu.local_maxima(d, conn), gpu.local_minima(d, conn)
    torch.cuda.synchronize()
    assert np.array_equal(hm.cpu().numpy(), o_imhmin(img, 1.5, conn))
    assert np.array_equal(mx.cpu().numpy(), o_local_extrema("maxima", img, conn))
    assert np.array_equal(mn.cpu().numpy(), o_local_extrema("minima", img, conn))


def test_in_place_and_overlapping_batches():
    import ctypes
    from nscale_amd._lib import ReconDesc, call
    from nscale_amd.gpu import _ptr, _stream
    imgs = [_image(h, w, "levels", k) for k, (h, w) in enumerate([(90, 200), (64, 64), (130, 70)])]
    exp = [o_imhmin(i, 1.0, c) for i, c in zip(imgs, (4, 8, 8))]
    one = torch.from_numpy(imgs[0]).cuda()
    call("nsc_imhmin_f32", _ptr(one), _ptr(one), 200, 90, ctypes.c_float(1.0), 4, _stream())
    torch.cuda.synchronize()
    assert np.array_equal(one.cpu().numpy(), exp[0])
    # outputs in place, and an output over another image's input
    ins = [torch.from_numpy(i).cuda() for i in imgs]
    outs = [ins[0], torch.empty_like(ins[1]), ins[2]]
    wide = torch.empty(imgs[1].size + 5, dtype=torch.float32, device="cuda")
    ins.append(wide[5:].view(64, 64).copy_(ins[1]))
    outs.append(wide[:-5].view(64, 64))  # starts 20 bytes before its own input
    arr = (ReconDesc * 4)()
    for k, (i, o, c) in enumerate(zip(ins, outs, (4, 8, 8, 8))):
        arr[k] = ReconDesc(None, _ptr(i), _ptr(o), i.shape[1], i.shape[0], c)
    call("nsc_imhmin_f32_batched", arr, 4, ctypes.c_float(1.0), _stream())
    torch.cuda.synchronize()
    for o, e in zip(outs, exp + [exp[1]]):
        assert np.array_equal(o.cpu().numpy(), e)
