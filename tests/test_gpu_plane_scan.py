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
