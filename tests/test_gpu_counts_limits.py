"""mdmc_counts_read: the numbers of counts it takes, and work that outlasts the
host's 2 ms watch."""
from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch

    import framework_amd as fa

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.set_device(0)
    fa.setup()
    return torch, fa


def test_numbers_of_counts(env):
    torch, fa = env
    ctx = fa.Context()
    d = torch.arange(4 * 1024, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for n in (0, 1025, 1 << 30):
        out = np.full((4, 4), 9, np.uint32)
        rc = fa.lib().mdmc_counts_read(ctx._h, ctypes.c_void_p(d.data_ptr()), n, out.ctypes.data_as(ctypes.c_void_p),
                                       ctx._stream(None))
        assert rc == -1 and (out == 9).all(), n
    for n in (1, 1024, 3):
        assert np.array_equal(ctx._wait_counts(d, n, None).ravel(), np.arange(4 * n)), n
    ctx.close()


def test_work_that_outlasts_the_watch(env):
    torch, fa = env
    ctx = fa.Context()
    d = torch.zeros((2, 4), dtype=torch.int32, device="cuda")
    torch.cuda._sleep(1)  # (kernels load at their first use, which takes longer than the work)
    d.add_(0)
    ctx._wait_counts(d, 2, None)
    for rep in range(2):
        torch.cuda._sleep(40_000_000)  # 17 ms at 2.4 GHz
        d.add_(1)
        t = time.perf_counter()
        c = ctx._wait_counts(d, 2, None)
        assert time.perf_counter() - t > 2e-3  # the stream's own wait was taken
        assert (c == rep + 1).all()
    ctx.close()


def test_a_refused_read_leaves_the_context_free(env):
    """Refused under capture, it does not give the context to the graph."""
    torch, fa = env
    ctx = fa.Context()
    field = torch.rand(9, 8, 7, device="cuda")
    before = ctx.extract(field, 0.5)
    d = torch.zeros(4, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        d.fill_(1)
        with pytest.raises(fa.MDMCError, match="capture"):
            ctx._wait_counts(d, 1, None)
    after = ctx.extract(field, 0.5)
    assert torch.equal(before[1], after[1]) and before[2] == after[2]
    g.replay()
    assert (ctx._wait_counts(d, 1, None) == 1).all()
    ctx.close()
