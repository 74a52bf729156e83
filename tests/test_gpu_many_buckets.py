"""Grids of very many tiles: the scan's block sums on either side of 16 blocks, from which
on a kernel scans them, and at the edges of that kernel's chunks (4096 blocks of 1024
buckets), against the CPU oracle at the suite's 1e-6 for FP32."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rick_amd import FP32, KAISERBESSEL, Plan

pytestmark = pytest.mark.gpu


# Planes of 4 x 4 cells are one tile each: 2, 3, 16, 17, 4096, 4097 and 8193 scan blocks.
@pytest.mark.parametrize("planes", [1025, 2049, 16 * 1024, 16 * 1024 + 1, 4096 * 1024, 4096 * 1024 + 1, 8192 * 1024 + 3])
def test_grids_of_many_tiles_match_oracle(planes):
    nx, n = 4, 30_000
    print(f"case many tiles planes={planes}", flush=True)
    plan = Plan(nx, nx, planes, kernel=KAISERBESSEL, support=7, precision=FP32, max_points=n,
                tile=(64, 64), rows_per_task=600)
    out = plan.new_grid()
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
        ww[:2000] = 1e-9                                    # split buckets at both ends
        ww[2000:4000] = 1.0 - 0.5 / planes
        vr, vi = (rng.normal(size=n).astype(np.float32) for _ in range(2))
        rows = [uu, vv, ww, vr, vi, np.ones(n, np.float32)]
        out.fill_(float("nan"))
        plan.grid(*[torch.from_numpy(a).to("cuda") for a in rows], 1, 1, out=out)
        stats = plan.grid_stats()
        plane = np.minimum(np.floor(ww * planes), planes - 1)
        assert stats["records"] == n and stats["split_buckets"] >= 2
        assert stats["nonempty_buckets"] == len(np.unique(plane))
        got = out.view(planes, 2 * nx * nx)
        assert bool(torch.isfinite(got).all())
        used = np.unique(plane).astype(np.int64)
        back = torch.from_numpy(used).to("cuda")
        assert int((got != 0).any(dim=1).sum()) <= used.size
        # The oracle grids the used planes alone: w moved to a stack of just those.
        stack = np.searchsorted(used, plane)
        ref = O.wstack(KAISERBESSEL, used.size, uu, vv, (stack + 0.5) / used.size, vr, vi, rows[5],
                       1, 1, 1.0 / nx, 1.0 / used.size, 7, nx, nx, threads=8)
        assert rel_l2(got[back].cpu().numpy().ravel(), ref) <= 1e-6
