"""The drop-ins' host copies by several threads: arrays much shorter than a staging
piece next to longer ones, more pieces than are in flight, threads that start late.
Every call has to move every byte, so each is compared with the device path; the bar
is the suite's 1e-12 (only the order of the sums differs)."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
import rick_amd
from rick_amd import FP64, Plan, imaging

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,P", [(6250, 24, 4), (70001, 3, 1), (400000, 4, 2)])
def test_dropin_wstack_moves_whole_arrays(n, F, P):
    nx, planes = 128, 3
    print(f"case drop-in staging n={n} F={F} P={P}", flush=True)
    rng = np.random.default_rng(n)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    wt = rng.uniform(0.5, 1.5, n * P).astype(np.float32)
    plan = Plan(nx, nx, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=FP64, max_points=n)
    imaging.set_kernel(rick_amd.KAISERBESSEL)
    for call in range(12):      # other values each time: a part left behind shows
        vr, vi = (rng.normal(size=n * F * P).astype(np.float32) for _ in range(2))
        ins = [torch.from_numpy(a).to("cuda") for a in (uu, vv, ww, vr, vi, wt)]
        want = plan.grid(*ins, F, P).cpu().numpy()
        got = np.zeros(2 * planes * nx * nx)
        imaging.wstack(planes, n, F, P, uu, vv, ww, vr, vi, wt, 1.0 / nx, 1.0 / planes, 7, nx, nx,
                       got, num_threads=8)
        assert rel_l2(got, want) <= 1e-12
