"""The operators' scratch blocks (kept per thread between calls): results do not depend on which call
had a block before -- alternating sizes, calls interleaved over streams without synchronisation, several
threads, more streams than a thread keeps blocks for, and captured calls replayed between eager ones."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SIZES = [(70, 90), (1500, 1300), (257, 300), (900, 2000), (64, 64)]


def _mask(h, w, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.rand(h, w, device="cuda", generator=g) < 0.6).to(torch.uint8) * 255


def _ops(m):
    """Operators with one, two and several scratch buffers; the last ones read a count on the host."""
    from nscale_amd import gpu
    lab = gpu.bwlabel2(m, 8)
    n = gpu.cc_relabel(lab)
    return [gpu.dist_transform(m), gpu.imfill_holes(m, 4), gpu.bwselect(m, m, 8), gpu.bwareaopen2(m, 3, 50, 4)[0], lab,
            gpu.bounding_boxes(lab, n)[0], gpu.local_maxima(gpu.dist_transform(m), 8)]


def _same(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


def _reference(masks):
    ref = []
    for m in masks:
        ref.append(_ops(m))
        torch.cuda.synchronize()
    return ref


def test_alternating_sizes_and_many_streams():
    masks = [_mask(h, w, k) for k, (h, w) in enumerate(SIZES)]
    ref = _reference(masks)
    streams = [torch.cuda.Stream() for _ in range(7)]
    torch.cuda.synchronize()
    out = []
    for k in range(35):  # every stream meets every size; nothing waits in between
        s, i = streams[k % 7], (k * 3) % 5
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            print("call", k, SIZES[i], flush=True)
            out.append((i, _ops(masks[i])))
    torch.cuda.synchronize()
    for i, got in out:
        assert _same(got, ref[i]), SIZES[i]
    for k in range(80):  # past a window of calls that need far less than the block holds
        assert torch.equal(_ops(masks[0])[1], ref[0][1])
    assert _same(_ops(masks[1]), ref[1])


def test_threads():
    masks = [_mask(h, w, 10 + k) for k, (h, w) in enumerate(SIZES)]
    ref = _reference(masks)
    bad = []

    def work(t):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for k in range(6):
                i = (t + k) % len(masks)
                got = _ops(masks[i])
                s.synchronize()
                if not _same(got, ref[i]):
                    bad.append((t, k))

    torch.cuda.synchronize()
    print("threads", flush=True)
    ths = [threading.Thread(target=work, args=(t,)) for t in range(6)]
    for th in ths:
        th.start()
    for th in ths:
        th.join()
    assert not bad


@pytest.mark.parametrize("op", ["edt", "fill", "normalize"])
def test_captured_calls_replay_between_eager_ones(op):
    from nscale_amd import gpu
    m = _mask(700, 900, 5)
    bgr = torch.stack([m, m // 2, m // 3], 2).contiguous()
    fn = {"edt": lambda: gpu.dist_transform(m), "fill": lambda: gpu.imfill_holes(m, 4),
          "normalize": lambda: gpu.normalization(bgr, np.float32([-0.6, 0.02, 0.05]), np.float32([0.3, 0.05, 0.04]))}[op]
    ref = fn()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    print("capture", op, flush=True)
    with torch.cuda.graph(graph, stream=s):
        out = fn()
    other = _mask(700, 900, 6)
    for _ in range(3):
        out.zero_()
        graph.replay()
        _ops(other)  # eager calls that use the thread's blocks
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
