"""The three forms of the scan at the edges between them: the rule's choice on
the CPU, and each side of each edge against the oracle on the GPU."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

import oracle
from tests.helpers import assert_same_mesh

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a plane of 2048 segments and of one more; 32,768 sums and one row block's
# more; 95, 96, 4,096 and 4,097 tiles of 2048 segments
EDGES = [((5, 2049, 6), "planes"), ((5, 2050, 6), "lookback"), ((4, 57, 4097), "planes"), ((4, 57, 4098), "tiles"),
         ((5, 2081, 94), "lookback"), ((5, 2081, 95), "tiles"), ((5, 2897, 2897), "tiles"),
         ((5, 2898, 2897), "lookback")]


@pytest.fixture(scope="module")
def form_of(tmp_path_factory):
    exe = tmp_path_factory.mktemp("scan") / "scan_form_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "framework_amd", "csrc"),
                    os.path.join(ROOT, "tests", "golden", "scan_form_check.cpp"), "-o", str(exe)], check=True)
    return lambda dims: subprocess.run([str(exe), *map(str, dims)], capture_output=True, text=True,
                                       check=True).stdout.strip()


@pytest.mark.parametrize("dims,form", EDGES)
def test_rule(form_of, dims, form):
    assert form_of(dims) == form


@pytest.mark.gpu
@pytest.mark.parametrize("dims,form", EDGES)
def test_scan_at_the_edge(dims, form):
    import torch

    import framework_amd as fa

    X, Y, Z = dims
    rng = np.random.default_rng(X + 10 * Y + 100 * Z)
    f = np.ones((Z, Y, X), np.float32)
    n = max(64, X * Y * Z // 400)  # isolated points, and whole rows at both ends
    f[rng.integers(0, Z, n), rng.integers(0, Y, n), rng.integers(0, X, n)] = -1.0
    f[0, 0], f[-1, -1], f[Z // 2, Y // 2] = -0.5, -0.5, -0.5
    print("scan form", form, dims, flush=True)
    ref = oracle.run(f, 0.1)
    ctx = fa.Context()
    v, q, c = ctx.extract(torch.from_numpy(f).cuda(), 0.1)
    assert (c["num_active"], c["status"]) == (ref["num_active"], 0)
    assert_same_mesh(v.cpu().numpy(), q.cpu().numpy(), ref)
    ctx.close()
