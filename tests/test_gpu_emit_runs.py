"""Emits whose waves do not run over whole chunks in one go, against the
oracle: cells too far apart for one wave's 32-bit offsets, and outputs that end
inside a chunk."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.helpers import assert_same_mesh

pytestmark = pytest.mark.gpu


# Segments (cell rows of an x-tile) that share offsets: 2^31 / (4 cap) - 1 =
# 2,097,151 of the first volume's 2,247,001 (its records bind), and
# (2^31 / (4 * 513) - 4) / 2 = 523,264 of the second's 527,796 (its field does).
@pytest.mark.parametrize("dims,span", [((3, 1500, 1500), 2097151), ((513, 730, 725), 523264)])
def test_cells_of_one_chunk_far_apart(dims, span):
    import torch

    import framework_amd as fa

    X, Y, Z = dims
    f = np.ones((Z, Y, X), np.float32)
    for z, y in ((2, 5), (3, 3), (Z // 2, Y // 2), (Z - 4, 7), (Z - 2, Y - 3)):  # 8 cells each
        f[z, y, 1] = -1.0
    print("runs", dims, flush=True)
    ref = oracle.run(f, 0.25)
    assert ref["num_active"] == 40
    first, last = (int(ref["cell_index"][i]) // (X - 1) for i in (0, -1))  # (one x-tile a row)
    assert last - first > span
    ctx = fa.Context()
    v, q, c = ctx.extract(torch.from_numpy(f).cuda(), 0.25)
    assert (c["num_active"], c["status"]) == (40, 0)
    assert_same_mesh(v.cpu().numpy(), q.cpu().numpy(), ref)
    ctx.close()


@pytest.mark.parametrize("noise", [0.05, 1.5])  # one iso vertex a cell nearly everywhere; several in many cells
@pytest.mark.parametrize("skip", [0, 1, 2, 3])  # rows before the outputs: vertices at every alignment
def test_outputs_that_end_inside_a_chunk(noise, skip):
    """What fits is written whole cell by whole cell, the rest of the arrays and
    what lies around them is left as it was."""
    import torch

    import framework_amd as fa

    ctx = fa.Context()
    field = ctx.field_gyroid((60, 50, 40), period=12.0, seed=4, noise_amp=noise)
    v0, q0, c0 = ctx.extract(field, 0.0)
    V, Q = c0["num_vertices"], c0["num_quads"]
    begin = np.append(ctx.cells(c0["num_active"])["vertex_begin"], V)
    assert V > 5000 and Q > 2000
    for j, (vcap, qcap) in enumerate([(V // 2 + i, Q // 2 + i) for i in range(6)] + [(1, 1), (V - 1, Q - 1), (V, Q)]):
        verts = torch.full((V + 64, 3), -7.0, device="cuda")
        quads = torch.full((Q + 64, 4), -7, dtype=torch.int32, device="cuda")
        ctx.emit(field, verts[skip:skip + vcap], quads[skip:skip + qcap])
        torch.cuda.synchronize()
        assert ctx.read_counts()["status"] == (0 if j == 8 else 3)
        ctx.counts_tensor()[3] = 0
        nv = int(begin[np.searchsorted(begin, vcap, side="right") - 1])  # the last cell's end within vcap
        v, q = verts.cpu().numpy(), quads.cpu().numpy()
        assert (v[:skip] == -7).all() and (v[skip + nv:] == -7).all(), (vcap, nv)
        assert np.array_equal(v[skip:skip + nv].view(np.uint32), v0[:nv].cpu().numpy().view(np.uint32)), vcap
        nq = int((q[:, 0] != -7).sum())
        assert qcap - 3 < nq <= qcap and (q[:skip] == -7).all() and (q[skip + nq:] == -7).all(), (qcap, nq)
        assert np.array_equal(q[skip:skip + nq], q0[:nq].cpu().numpy()), qcap
    ctx.close()
