"""Partials added by the last workgroup to arrive: more streams than have
arrival counters (the rest take the second launch) give the same bits, call
after call, in any order of sizes (one workgroup, one level of counters, two
levels, and past the length from which a second launch is used)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = (300007, 4099, (1 << 24) + 5, 524289, 4095, 20001, 1 << 24, 524288)


def test_dot_on_more_streams_than_counters(dev, ompblas):
    lib = ompblas.lib()
    nmax = max(SIZES)
    x, y = torch.empty(nmax, device=dev), torch.empty(nmax, device=dev)
    ompblas.fill_uniform(x, 81, 0)
    ompblas.fill_uniform(y, 81, 1)
    want = torch.full((len(SIZES),), float("nan"), device=dev)
    torch.cuda.synchronize()
    for i, n in enumerate(SIZES):  # second launch: no counters
        ompblas.check(lib.omb_sdot_noalloc(n, x.data_ptr(), y.data_ptr(),
                                           want[i:].data_ptr(), None))
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so")
    streams = []
    for _ in range(70):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        streams.append(s)
    got = torch.full((len(streams), 2, len(SIZES)), float("nan"), device=dev)
    torch.cuda.synchronize()
    for k, s in enumerate(streams):
        for rep in range(2):
            for i, n in enumerate(SIZES):
                ompblas.check(lib.omb_sdot(n, x.data_ptr(), y.data_ptr(),
                                           got[k, rep, i:].data_ptr(), s))
    torch.cuda.synchronize()
    assert torch.equal(got, want.expand_as(got))
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
