"""Row lengths at the edges of the classify's mappings, against the oracle:
16-byte row loads that end inside a row, narrow last x-tiles (64, 128, 256
points, and a full chunk with 64 or 128 more), rows of 2 and 3 points, and
lists of active cells that wrap (noise in every cell)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.helpers import assert_same_mesh, check_against_oracle

pytestmark = pytest.mark.gpu

WIDTHS = [2, 3, 4, 5, 7, 63, 64, 65, 66, 127, 128, 129, 130, 255, 256, 257, 258, 319, 320, 321, 322, 383, 384, 385,
          386, 511, 512, 513, 514, 575, 577, 640, 641, 769, 833, 897, 1025]


@pytest.fixture(scope="module")
def fa_mod():
    import torch

    import framework_amd as fa

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.set_device(0)
    fa.setup()
    return fa


def _field(X, Y, Z, seed):
    """Noise (every cell active, 2B/3B cells) in the first half of the rows, a
    few surface cells in the rest."""
    rng = np.random.default_rng(seed)
    f = rng.standard_normal((Z, Y, X)).astype(np.float32)
    f[:, Y // 2:, :] = 1.0
    f[:, Y // 2:, X // 3:X // 3 + 2] = rng.standard_normal((Z, Y - Y // 2, len(range(X)[X // 3:X // 3 + 2])))
    f[:, :, -1] = rng.standard_normal((Z, Y))
    return f


@pytest.mark.parametrize("X", WIDTHS)
def test_row_width(fa_mod, X):
    import torch

    ctx = fa_mod.Context()
    for Y, Z in ((8, 5), (17, 10)):
        check_against_oracle(ctx, torch.from_numpy(_field(X, Y, Z, X + Y)).cuda(), 0.1)
    ctx.close()


@pytest.mark.parametrize("widths", [[w for w in WIDTHS if w <= 256], WIDTHS, [2, 3, 500, 510, 300, 60, 200, 380]])
def test_batch_of_row_widths(fa_mod, widths):
    """256- and 512-cell x-tiles (the batch takes the one with fewer padded cells)."""
    import torch

    ctx = fa_mod.Context()
    host = [_field(X, 9, 6, 3 * X) for X in widths]
    res = ctx.batch_extract([torch.from_numpy(f).cuda() for f in host], [0.1] * len(host))
    for f, (v, q, c) in zip(host, res):
        ref = oracle.run(f, 0.1)
        assert (c["num_active"], c["num_vertices"], c["num_quads"]) == \
            (ref["num_active"], ref["num_vertices"], ref["num_quads"]), f.shape
        assert_same_mesh(v.cpu().numpy(), q.cpu().numpy(), ref)
    ctx.close()


def _tall_field(X, Y, Z):
    """Mostly empty: noise in a box in the middle and at the far corner."""
    rng = np.random.default_rng(X)
    f = np.ones((Z, Y, X), np.float32)
    for k, j in ((Z // 2, Y // 2), (Z - 9, Y - 9)):
        f[k:k + 10, j:j + 9, :] = rng.standard_normal(f[k:k + 10, j:j + 9, :].shape)
    return f


@pytest.mark.parametrize("shape", [(5, 645, 365), (64, 645, 362), (70, 645, 365), (128, 641, 367)])
def test_narrow_rows_many_tiles(fa_mod, shape):
    """Rows of one narrow x-tile in a grid of over 8192 tiles: tiles of 8 planes."""
    import torch

    ctx = fa_mod.Context()
    check_against_oracle(ctx, torch.from_numpy(_tall_field(*shape)).cuda(), 0.1)
    ctx.close()


@pytest.mark.parametrize("planes", [0, 2, 1, 4])
def test_batch_of_narrow_rows_many_tiles(fa_mod, planes):
    """Tall narrow tiles for every number of planes a full tile can have."""
    import torch

    ctx = fa_mod.Context()
    ctx.set_option(fa_mod.mdmc.OPT_BATCH_PLANES, planes)
    host = [_tall_field(*s) for s in ((60, 330, 365), (100, 331, 363), (300, 40, 39), (257, 9, 6), (3, 50, 40))]
    for f, (v, q, c) in zip(host, ctx.batch_extract([torch.from_numpy(f).cuda() for f in host], [0.1] * len(host))):
        assert_same_mesh(v.cpu().numpy(), q.cpu().numpy(), oracle.run(f, 0.1))
    ctx.close()
