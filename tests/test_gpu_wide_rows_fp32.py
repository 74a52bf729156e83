"""FP32 records of rows of 12 values and more, all, few or none of a wave's rows inside the
grid, against the CPU oracle (the suite's 1e-6 for an FP32 grid)."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rick_amd import FP32, KAISERBESSEL, Plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,P", [(3, 4), (12, 1), (5, 4), (10, 2), (24, 1), (64, 1)])
@pytest.mark.parametrize("inside", [0, 16, 17, 64])
def test_fp32_wide_rows_match_oracle(F, P, inside):
    nx, planes, n = 256, 4, 4133
    print(f"case FP32 wide rows F={F} P={P} inside={inside}", flush=True)
    rng = np.random.default_rng(F * 100 + P + inside)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    for w0 in range(0, n, 64):
        out = rng.permutation(64)[inside:] + w0
        vv[out[out < n - 30]] += 1.5
    vr, vi = (rng.normal(size=n * F * P).astype(np.float32) for _ in range(2))
    vr[1::29] = np.nan
    wt = rng.uniform(0.5, 1.5, n * P).astype(np.float32)
    ref = O.wstack(KAISERBESSEL, planes, uu, vv, ww, vr, vi, wt, F, P, 1.0 / nx, 1.0 / planes, 7,
                   nx, nx, threads=8)
    plan = Plan(nx, nx, planes, kernel=KAISERBESSEL, support=7, precision=FP32, max_points=n)
    got = plan.grid(*[torch.from_numpy(a).to("cuda") for a in (uu, vv, ww, vr, vi, wt)], F,
                    P).cpu().numpy()
    assert np.isfinite(got).all()
    assert rel_l2(got, ref) <= 1e-6
