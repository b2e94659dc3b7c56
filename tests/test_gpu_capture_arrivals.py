"""Arrival counters belong to a stream's eager calls: a captured dot or column
GEMV adds its partials in a second kernel, so that its graph, which may be replayed
on another stream, takes no part in the counters of the capture stream.  Replays
between eager calls of several sizes give the eager bits."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _hip():
    hip = ctypes.CDLL("libamdhip64.so")

    def ok(status):
        assert status == 0, status
    return hip, ok


@pytest.mark.parametrize("kind", ["dot", "gemv"])
def test_captured_calls_use_no_counters(dev, ompblas, kind):
    hip, ok = _hip()
    n = 600007
    x, y = torch.empty(n, device=dev), torch.empty(n, device=dev)
    ompblas.fill_uniform(x, 91, 0)
    ompblas.fill_uniform(y, 91, 1)
    # sizes of many workgroups or chunks, the captured one and two others
    sizes = (600007, 300007, 20001) if kind == "dot" else ((300, 2000), (100, 5000), (260, 1111))

    def call(size, out, s):
        if kind == "dot":
            return ompblas.sdot(size, x.data_ptr(), y.data_ptr(), out.data_ptr(), stream=s)
        m, k = size
        return ompblas.sgemv(m, k, 1.0, x.data_ptr(), 1, m, y.data_ptr(), 0.0, out.data_ptr(),
                             stream=s)

    length = [1 if kind == "dot" else size[0] for size in sizes]
    outs = [torch.full((k,), float("nan"), device=dev) for k in length]
    captured = torch.full((length[0],), float("nan"), device=dev)
    torch.cuda.synchronize()
    streams = []
    for _ in range(2):
        s = ctypes.c_void_p()
        ok(hip.hipStreamCreateWithFlags(ctypes.byref(s), 1))
        streams.append(s)
    mine, other = streams
    for size, out in zip(sizes, outs):
        ompblas.check(call(size, out, mine))
    torch.cuda.synchronize()
    want = [o.clone() for o in outs]
    graph, run, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    ok(hip.hipStreamBeginCapture(mine, 1))
    status = call(sizes[0], captured, mine)
    ok(hip.hipStreamEndCapture(mine, ctypes.byref(graph)))
    ompblas.check(status)
    ok(hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)))
    assert nodes.value == 2  # the partials, and their sum
    ok(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)))
    for _ in range(3):
        for size, out, w in zip(sizes, outs, want):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            ompblas.check(call(size, out, mine))
            torch.cuda.synchronize()
            assert torch.equal(out, w), size
        captured.fill_(float("nan"))
        torch.cuda.synchronize()
        ok(hip.hipGraphLaunch(run, other))
        torch.cuda.synchronize()
        assert torch.equal(captured, want[0])
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
    for s in streams:
        ok(hip.hipStreamDestroy(s))
