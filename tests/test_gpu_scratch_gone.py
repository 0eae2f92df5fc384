"""What a count or an emit left in a context's scratch is gone with it: later
steps are refused, and the context works again after a new count."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from tests.helpers import assert_same_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture()
def env():
    import torch

    import framework_amd as fa

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.set_device(0)
    fa.setup()
    ctx = fa.Context()
    f = np.random.default_rng(3).standard_normal((9, 11, 13)).astype(np.float32)
    field = torch.from_numpy(f).cuda()
    v, q, _ = ctx.extract(field, 0.1)
    yield torch, fa, ctx, f, field, v, q
    ctx.close()


def _usable_again(fa, ctx, f, field, v, q):
    for step in (lambda: ctx.emit(field, v, q), lambda: ctx.smooth(v, q, 1)):
        with pytest.raises(fa.MDMCError, match="without a preceding"):
            step()
    v1, q1, c = ctx.extract(field, 0.1, num_smooth=2)
    assert c["status"] == 0
    assert_same_mesh(v1.cpu().numpy(), q1.cpu().numpy(), oracle.run(f, 0.1, num_smooth=2))


def test_scratch_given_back(env):
    torch, fa, ctx, f, field, v, q = env
    lib = fa.lib()
    lib.mdmc_ctx_set_scratch.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64]
    assert lib.mdmc_ctx_set_scratch(ctx._h, None, 0) == 0
    _usable_again(fa, ctx, f, field, v, q)


def test_scratch_that_cannot_grow(env):
    """A count whose scratch (4 TB) no device holds gives the old one up."""
    torch, fa, ctx, f, field, v, q = env
    rc = fa.lib().mdmc_count_device(ctx._h, ctypes.c_void_p(field.data_ptr()), (ctypes.c_uint32 * 3)(2, 32768, 65535),
                                    ctypes.c_float(0.1), ctypes.c_void_p(ctx.counts_tensor().data_ptr()),
                                    ctx._stream(None))
    assert rc == -3  # no memory, before anything is launched
    _usable_again(fa, ctx, f, field, v, q)


def test_a_single_count_ends_a_batch(env):
    """Between a batch's count and its emit a count of one volume takes the
    scratch over: the batch's emit is refused."""
    torch, fa, ctx, f, field, v, q = env
    fields, isos = [field, field[:5].contiguous()], [0.1, 0.2]
    refs = [oracle.run(f, 0.1), oracle.run(f[:5], 0.2)]
    counts = ctx.batch_counts_tensor(2)
    outs = [(torch.empty((len(r["vertices"]), 3), device="cuda"),
             torch.empty((len(r["quads"]), 4), dtype=torch.int32, device="cuda")) for r in refs]
    ctx.batch_count(fields, isos, counts)
    ctx.count(field, 0.1)
    with pytest.raises(fa.MDMCError, match="without a matching batch count"):
        ctx.batch_emit(fields, isos, outs, counts)
    ctx.batch_count(fields, isos, counts)
    ctx.batch_emit(fields, isos, outs, counts)
    torch.cuda.synchronize()
    for (a, b), r in zip(outs, refs):
        assert_same_mesh(a.cpu().numpy(), b.cpu().numpy(), r)
