"""Re-averaging walks each cell's crossed edges three at a time: cells with 3 to
12 crossed edges and 1 to 4 iso vertices, alone and mixed in a wave, against
the oracle, bitwise."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _field(kind, shape):
    rng = np.random.default_rng(5)
    if kind == "noise":  # every kind of cell in every wave
        return rng.standard_normal(shape).astype(np.float32)
    if kind == "plane":  # one iso vertex, 3 to 6 crossed edges
        z, y, x = np.meshgrid(*(np.arange(n, dtype=np.float32) for n in shape), indexing="ij")
        return (0.61 * x + 0.53 * y + 0.59 * z - 0.8 * shape[0]).astype(np.float32)
    f = np.where(rng.random(shape) < 0.02, 1.0, -1.0)  # "points": lone corners, a few ambiguous cells
    return (f * (0.5 + rng.random(shape))).astype(np.float32)


@pytest.mark.parametrize("kind", ["noise", "plane", "points"])
@pytest.mark.parametrize("shape", [(2, 2, 2), (3, 2, 259), (17, 18, 19), (9, 12, 301)])
def test_smoothing_matches_oracle(kind, shape):
    import torch

    import framework_amd as fa

    f = _field(kind, shape)
    ctx = fa.Context()
    for n in (1, 3):
        ref = oracle.run(f, 0.0, None, None, num_smooth=n)
        v, q, c = ctx.extract(torch.from_numpy(f).cuda(), 0.0, num_smooth=n)
        assert c["status"] == 0
        assert np.array_equal(q.cpu().numpy(), ref["quads"])
        assert np.array_equal(v.cpu().numpy().view(np.uint32), ref["vertices"].view(np.uint32))
    ctx.close()
