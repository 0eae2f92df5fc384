"""A count prepares the coordinates of the index box; emits with that box and
with others, in any order, and negative zeros in the box, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(33, 30, 35), (2, 9, 5), (300, 21, 4)])
def test_emits_of_one_count_with_several_boxes(dims):
    import torch

    import framework_amd as fa

    X, Y, Z = dims
    f = np.random.default_rng(X).standard_normal((Z, Y, X)).astype(np.float32)
    field = torch.from_numpy(f).cuda()
    ctx = fa.Context()
    ctx.count(field, 0.1)
    index = ((0.0, 0.0, 0.0), tuple(float(max(d - 1, 1)) for d in dims))
    other = ((-5.0, -2.5, 1.0), (5.0, 7.5, 3.0))
    signed = ((-0.0, 0.0, -0.0), index[1])
    for box in (index, other, index, None, signed, None):
        ref = oracle.run(f, 0.1, *(box or (None, None)))
        v = torch.empty((len(ref["vertices"]), 3), device="cuda")
        q = torch.empty((len(ref["quads"]), 4), dtype=torch.int32, device="cuda")
        ctx.emit(field, v, q, *(box or (None, None)))
        torch.cuda.synchronize()
        assert ctx.read_counts()["status"] == 0
        assert np.array_equal(q.cpu().numpy(), ref["quads"])
        assert np.array_equal(v.cpu().numpy().view(np.uint32), ref["vertices"].view(np.uint32)), box
    ctx.close()
