"""Operator calls on streams of their own while another stream is captured into a graph: the calls give their
results and the capture goes on, for calls from the capturing thread and from another one."""
import threading

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("thread", [False, True])
def test_capture_goes_on(mode, thread):
    from nscale_amd import gpu
    from nscale_amd._lib import call
    h, w = 700, 900
    g = torch.Generator(device="cuda").manual_seed(3)
    img = (torch.rand(h, w, device="cuda", generator=g) < 0.9).to(torch.uint8) * 255
    ref = gpu.dist_transform(img)
    outs = [torch.zeros_like(ref) for _ in range(8)]
    streams = [torch.cuda.Stream() for _ in range(3)]
    x = torch.ones(1000, device="cuda")
    torch.cuda.synchronize()

    def work(part):
        for k, o in enumerate(part):
            with torch.cuda.stream(streams[k % 2]):
                call("nsc_dist_transform_u8", gpu._ptr(img), gpu._ptr(o), w, h, gpu._stream())

    print("capture", mode, thread, flush=True)
    work(outs[:4])  # the thread's blocks have been used on these streams
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[2], capture_error_mode=mode):
        y = x * 2
        if thread:
            t = threading.Thread(target=work, args=(outs[4:],))
            t.start()
            t.join()
        else:
            work(outs[4:])
        y = y + 1
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert bool((y == 3).all())
    assert all(torch.equal(o, ref) for o in outs)
