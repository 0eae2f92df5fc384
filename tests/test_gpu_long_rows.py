"""Grids of few, very long rows: the scan has few threads, so the coordinate
tables are filled apart.  Both sides of the line, for every way to an emit."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

import oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# X x 2 x 2 points: one workgroup of 256 threads, 16,384 entries are its most
EDGES = [(16380, True), (16381, False), (500000, False)]


@pytest.mark.parametrize("X,fills", EDGES)
def test_rule(tmp_path, X, fills):
    src = tmp_path / "r.cpp"
    src.write_text('#include "mdmc_tilemap.h"\n#include <cstdio>\n'
                   f"int main() {{ std::printf(\"%d\", mdmc::scan_fills_coords({X} + 4, 256)); }}\n")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "framework_amd", "csrc"), str(src), "-o",
                    str(tmp_path / "r")], check=True)
    assert subprocess.run([str(tmp_path / "r")], capture_output=True, text=True).stdout == str(int(fills))


@pytest.mark.gpu
@pytest.mark.parametrize("X,fills", EDGES)
def test_long_rows(X, fills):
    import torch

    import framework_amd as fa

    rng = np.random.default_rng(X)
    f = np.ones((2, 2, X), np.float32)
    f[:, :, rng.integers(0, X, 500)] = -rng.random((2, 2, 500), dtype=np.float32) - 0.1
    f[:, :, -1] = -1.0
    field = torch.from_numpy(f).cuda()
    box = ((-5.0, -2.5, 1.0), (5.0, 7.5, 3.0))
    ctx = fa.Context()
    for b in (None, box):
        ref = oracle.run(f, 0.1, *(b or (None, None)))
        for way in ("extract_into", "extract", "emit", "emit again"):
            v = torch.empty((len(ref["vertices"]), 3), device="cuda")
            q = torch.empty((len(ref["quads"]), 4), dtype=torch.int32, device="cuda")
            if way == "extract":
                v, q, _ = ctx.extract(field, 0.1, *(b or (None, None)))
            elif way == "extract_into":
                ctx.extract_into(field, 0.1, v, q, *(b or (None, None)))
            else:
                ctx.emit(field, v, q, *(b or (None, None)))
            torch.cuda.synchronize()
            assert ctx.read_counts()["status"] == 0
            assert np.array_equal(v.cpu().numpy().view(np.uint32), ref["vertices"].view(np.uint32)), (b, way)
            assert np.array_equal(q.cpu().numpy(), ref["quads"]), (b, way)
    ctx.close()
