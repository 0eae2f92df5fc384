"""Emits and smoothing captured without the count they follow (GPU): each
replay starts from the coordinate tables that the replay before left, so what
is captured fills them itself.  Two boxes in one graph, in either order, and
smoothing of an eager emit's mesh beside an emit with another box."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = (70, 45, 38)
INDEX = ((0.0, 0.0, 0.0), tuple(float(d - 1) for d in DIMS))
OTHER = ((-5.0, -2.5, 1.0), (5.0, 7.5, 3.0))


@pytest.fixture(scope="module")
def env():
    import torch

    import framework_amd as fa

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.set_device(0)
    fa.setup()
    gen = fa.Context()
    field = gen.field_gyroid(DIMS, period=13.0, seed=3, noise_amp=0.1)
    torch.cuda.synchronize()
    yield torch, fa, gen, field
    gen.close()


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("boxes", [(INDEX, OTHER), (OTHER, INDEX), (INDEX, OTHER, INDEX)])
@pytest.mark.parametrize("before", ["count", "extract"])
def test_two_boxes_in_one_graph(env, boxes, before):
    torch, fa, gen, field = env
    ref = [gen.extract(field, 0.05, *b)[:2] for b in boxes]
    ctx = fa.Context()
    outs = [(torch.empty_like(v), torch.empty_like(q)) for v, q in ref]
    if before == "count":
        ctx.count(field, 0.05)
    else:
        ctx.extract_into(field, 0.05, *outs[0], xyz_min=boxes[0][0], xyz_max=boxes[0][1])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for (v, q), b in zip(outs, boxes):
            ctx.emit(field, v, q, *b)
    for rep in range(3):
        for v, q in outs:
            v.fill_(-1.0)
            q.fill_(-1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert int(ctx.counts_tensor()[3]) == 0
        for i, ((v, q), (rv, rq)) in enumerate(zip(outs, ref)):
            assert torch.equal(q, rq) and np.array_equal(_bits(v), _bits(rv)), (rep, i)
    del g
    ctx.close()


def test_smoothing_captured_after_an_eager_emit(env):
    torch, fa, gen, field = env
    v0, q0, _ = gen.extract(field, 0.05, *OTHER)
    smoothed = gen.extract(field, 0.05, *OTHER, num_smooth=2)[0]
    v1 = gen.extract(field, 0.05, *INDEX)[0]
    ctx = fa.Context()
    ctx.count(field, 0.05)
    v, q, w, r = torch.empty_like(v0), torch.empty_like(q0), torch.empty_like(v1), torch.empty_like(q0)
    ctx.emit(field, v, q, *OTHER)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.smooth(v, q, 2)
        ctx.emit(field, w, r, *INDEX)
    for rep in range(3):
        v.copy_(v0)
        w.fill_(-1.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(_bits(v), _bits(smoothed)) and np.array_equal(_bits(w), _bits(v1)), rep
        assert torch.equal(r, q0)
    del g
    ctx.close()
