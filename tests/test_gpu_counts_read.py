"""mdmc_counts_read: the counts behind everything the stream holds, whether they
arrive while the host watches or only after it has gone over to the stream's
own wait; on other streams; refused under capture."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import framework_amd as fa
import oracle


def test_null_arguments_and_sizes_are_rejected():
    raw = ctypes.CDLL(fa.mdmc.LIB_PATH)
    null = ctypes.c_void_p(None)
    assert raw.mdmc_counts_read(null, null, 1, null, null) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("queued", [0, 400])  # 400 extractions of 128^3 take over 2 ms
def test_counts_follow_the_queued_work(queued):
    import torch

    f = oracle.field_gyroid((128, 128, 128), 24.0, 3, 0.05)
    ref = oracle.run(f, 0.0, None, None)
    ctx = fa.Context()
    field = torch.from_numpy(f).cuda()
    v = torch.empty((len(ref["vertices"]), 3), device="cuda")
    q = torch.empty((len(ref["quads"]), 4), dtype=torch.int32, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    for s in (None, stream):
        counts = torch.full((3, 4), -1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for _ in range(queued):
            ctx.extract_into(field, 0.0, v, q, counts=counts[1], stream=s)
        ctx.extract_into(field, 0.0, v, q, counts=counts[2], stream=s)
        c = ctx._wait_counts(counts, 3, s)
        done = [ref["num_active"], len(ref["vertices"]), len(ref["quads"]), 0]
        assert c[2].tolist() == done
        assert c[1].tolist() == (done if queued else [0xFFFFFFFF] * 4) and c[0].tolist() == [0xFFFFFFFF] * 4
    ctx.close()


@pytest.mark.gpu
def test_refused_under_capture():
    import torch

    ctx = fa.Context()
    field = torch.zeros((8, 8, 8), device="cuda")
    ctx.extract(field, 0.5)
    ctx2 = fa.Context()
    counts = torch.zeros(4, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        counts.fill_(1)
        with pytest.raises(fa.MDMCError):
            ctx2._wait_counts(counts, 1, None)
    c = ctx._wait_counts(counts, 1, None)
    assert np.array_equal(c, np.zeros((1, 4), np.uint32))
    ctx.close()
