"""Calls of far fewer rows than the plan was made for: their tasks are those of a plan of
their own size, and the grids match the CPU oracle (the suite's 1e-12 in FP64, 1e-6 for
an FP32 grid) before and after a call that fills the plan."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rick_amd import FP32, FP64, KAISERBESSEL, Plan

pytestmark = pytest.mark.gpu
NX, PLANES, CAPACITY = 256, 4, 2_700_000


def make_rows(n, seed):
    rng = np.random.default_rng(seed)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    k = int(n * 0.3)        # a hot tile, split over several tasks
    uu[:k], vv[:k], ww[:k] = (rng.uniform(0.5, 0.51, k) for _ in range(3))
    vr, vi = (rng.normal(size=n).astype(np.float32) for _ in range(2))
    return uu, vv, ww, vr, vi, rng.uniform(0.5, 1.5, n).astype(np.float32)


@pytest.mark.parametrize("support", [5, 7])     # record by record, by class
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_small_calls_on_a_large_plan(support, precision):
    kw = dict(kernel=KAISERBESSEL, support=support, precision=precision, tile=(64, 64))
    plan = Plan(NX, NX, PLANES, max_points=CAPACITY, **kw)
    for seed, n in enumerate((50_000, 1, CAPACITY, 50_001, 700, 400_000, CAPACITY - 1, 0, 20_000)):
        print(f"case support={support} precision={precision} n={n}", flush=True)
        rows = make_rows(n, seed)
        ins = [torch.from_numpy(a).to("cuda") for a in rows]
        out = plan.new_grid()
        out.fill_(float("nan"))
        got = plan.grid(*ins, 1, 1, out=out).cpu().numpy()
        stats = plan.grid_stats()
        ref = O.wstack(KAISERBESSEL, PLANES, *rows, 1, 1, 1.0 / NX, 1.0 / PLANES, support, NX, NX,
                       threads=8)
        assert np.isfinite(got).all()
        if n == 0:
            assert not got.any()
            continue
        assert rel_l2(got, ref) <= (1e-12 if precision == FP64 else 1e-6)
        own = Plan(NX, NX, PLANES, max_points=n, **kw)
        own.grid(*ins, 1, 1, out=out)
        assert own.grid_stats() == stats
