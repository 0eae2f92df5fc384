"""The scan by whole planes (small and medium volumes) and the look-back scan
at the edges of their ranges, against the oracle: one plane per workgroup, a
plane that just fits or just does not, one more sum than the plane scan takes."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.helpers import check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch

    import framework_amd as fa

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.set_device(0)
    fa.setup()
    c = fa.Context()
    yield c
    c.close()


# cell planes of 1, 2047, 2048 and 2049 segments (2048 is the most a workgroup
# takes), two x-tiles a row, and 32,760 / 32,770 / 33,000 sums (the plane scan takes 32,768)
@pytest.mark.parametrize("dims", [(5, 2, 2), (5, 2, 5000), (6, 2048, 9), (6, 2049, 9), (6, 2050, 9), (600, 1025, 4),
                                  (600, 1026, 4), (4, 71, 3277), (4, 71, 3278), (4, 71, 3301), (40, 33, 700)])
def test_plane_scan_edges(ctx, dims):
    import torch

    X, Y, Z = dims
    rng = np.random.default_rng(X + 10 * Y + 100 * Z)
    f = (rng.random((Z, Y, X)) < 0.03).astype(np.float32)  # isolated points: many empty rows between
    f[:, :, 0] = rng.standard_normal((Z, Y)) > 1.5
    check_against_oracle(ctx, torch.from_numpy(f).cuda(), 0.5)


# more segments than whole planes hold and more sums than the plane scan takes:
# the scan of tiles (2048 segments) from 96 tiles, with whole and ragged last ones, and the look-back below
@pytest.mark.parametrize("dims", [(5, 2050, 3), (5, 2050, 95), (5, 2049, 96), (5, 2049, 97), (5, 2050, 97), (600, 2049, 50),
                                  (4, 71, 3301), (3, 2100, 420), (20, 900, 300)])
def test_tile_scan_edges(ctx, dims):
    test_plane_scan_edges(ctx, dims)


def test_batch_active_counts(ctx):
    """Active cells of a volume: a search in the list of non-empty rows, 64 entries a round."""
    import torch

    import oracle

    rng = np.random.default_rng(7)
    shapes = [(2, 2, 2), (9, 70, 66), (2, 3, 2), (5, 65, 64), (4, 64, 65), (3, 2, 3), (6, 91, 90)]
    fields = [(rng.random(s) < 0.2).astype(np.float32) for s in shapes]
    fields[2][:] = 0.0  # no surface
    for n in (1, 3, len(shapes)):
        res = ctx.batch_extract([torch.from_numpy(f).cuda() for f in fields[:n]], [0.5] * n)
        for f, (_, _, c) in zip(fields, res):
            assert c["num_active"] == oracle.run(f, 0.5)["num_active"]
