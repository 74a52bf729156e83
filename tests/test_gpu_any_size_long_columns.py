"""Images of very long four-step columns, whose second factor has no launch of the fused
last column pass and phase (lines above 3072 points with a radix of 6 or 7), and one that
has, against the separate stages."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from rick_amd import FP64, KAISERBESSEL, Plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1", [3600, 3200])
def test_image_of_very_long_columns_matches_stages(n1):
    nx, ny, planes, n = 2, n1 * n1, 2, 2000
    print(f"case long columns {nx}x{ny}", flush=True)
    plan = Plan(nx, ny, planes, kernel=KAISERBESSEL, support=7, precision=FP64, max_points=n,
                dx=1.0 / ny, resolution=1e-8, wmin=-300.0, wmax=500.0)
    rng = np.random.default_rng(n1)
    ins = [torch.from_numpy(a).to("cuda") for a in (
        rng.uniform(0.0, nx / ny, n), rng.uniform(0.0, 1.0, n), rng.uniform(0.0, 0.99, n),
        rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32),
        np.ones(n, np.float32))]
    re, im, grid = plan.image(*ins)
    dense = plan.grid(*ins, out=grid)
    plan.fft(dense)
    wre, wim = plan.phase(dense)
    got, want = ((a.cpu().numpy() + 1j * b.cpu().numpy()) for a, b in ((re, im), (wre, wim)))
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    assert rel_l2(got, want) <= 1e-12
