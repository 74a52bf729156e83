"""The gridder's binning at the sizes where its launches change: blocks of 1,
4 or 16 rows per thread, one scan workgroup or two scan kernels, split buckets
spread over the scan's waves.  FP64 against the CPU oracle at the suite's
1e-12 (only the order of the sums differs)."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
import rick_amd
from rick_amd import FP64, Plan

pytestmark = pytest.mark.gpu


def make_rows(n, seed, hot):
    rng = np.random.default_rng(seed)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    k = int(n * hot)
    uu[:k], vv[:k], ww[:k] = (rng.uniform(0.5, 0.51, k) for _ in range(3))
    vr, vi = (rng.normal(size=n).astype(np.float32) for _ in range(2))
    return uu, vv, ww, vr, vi, rng.uniform(0.5, 1.5, n).astype(np.float32)


# Tiles are 64 x 64: 256^2 grids hold 16 buckets a plane, so 64 planes are the
# last grid of one scan workgroup (1024 buckets) and 65 the first of two.
@pytest.mark.parametrize("n,planes,rows_per_task", [
    (1, 4, 0), (1023, 64, 3), (1025, 65, 3), (524287, 64, 300), (524289, 65, 300),
    (2621439, 4, 4096), (2621443, 80, 4096)])
def test_binning_launch_edges_match_oracle(n, planes, rows_per_task):
    nx = 256
    print(f"case n={n} planes={planes} rows_per_task={rows_per_task}", flush=True)
    plan = Plan(nx, nx, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=FP64,
                max_points=n, tile=(64, 64), rows_per_task=rows_per_task)
    # Twice in a row with other rows, then fewer: the counters start clean each time.
    for seed, m in ((1, n), (2, n), (3, (n + 1) // 2)):
        rows = make_rows(m, seed, 0.3)
        ref = O.wstack(O.KAISERBESSEL, planes, *rows, 1, 1, 1.0 / nx, 1.0 / planes, 7, nx, nx,
                       threads=8)
        out = plan.new_grid()
        out.fill_(float("nan"))
        plan.grid(*[torch.from_numpy(a).to("cuda") for a in rows], 1, 1, out=out)
        got = out.cpu().numpy()
        assert np.isfinite(got).all()
        assert rel_l2(got, ref) <= 1e-12


# Rows of more than 16 values, or of 12, in 16-byte pieces shared by four lanes:
# the last piece missing on some lanes, weights that do and do not repeat with
# the piece, rows that end inside a wave, a misaligned array (scalar reads).
@pytest.mark.parametrize("F,P", [(3, 4), (5, 4), (8, 3), (12, 3), (64, 1), (17, 4), (10, 2)])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 4133])
def test_wide_rows_match_oracle(F, P, shift, n):
    nx, planes = 256, 4
    print(f"case wide rows F={F} P={P} shift={shift} n={n}", flush=True)
    rng = np.random.default_rng(F * 100 + P)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    vr, vi = (rng.normal(size=n * F * P).astype(np.float32) for _ in range(2))
    vr[1::29] = np.nan
    wt = rng.uniform(0.5, 1.5, n * P).astype(np.float32)
    ref = O.wstack(O.KAISERBESSEL, planes, uu, vv, ww, vr, vi, wt, F, P, 1.0 / nx, 1.0 / planes,
                   7, nx, nx, threads=8)
    plan = Plan(nx, nx, planes, kernel=rick_amd.KAISERBESSEL, support=7, max_points=n)

    def on_gpu(a):
        t = torch.zeros(a.size + shift, dtype=torch.float32, device="cuda")[shift:]
        return t.copy_(torch.from_numpy(a))
    got = plan.grid(*[torch.from_numpy(a).to("cuda") for a in (uu, vv, ww)], on_gpu(vr),
                    on_gpu(vi), torch.from_numpy(wt).to("cuda"), F, P).cpu().numpy()
    assert np.isfinite(got).all()
    assert rel_l2(got, ref) <= 1e-12


# Waves of which no row, few (to 16, ranked and read at once) or more lie in the grid.
@pytest.mark.parametrize("F,P", [(5, 4), (6, 4), (12, 3), (64, 1)])
@pytest.mark.parametrize("inside", [0, 1, 15, 16, 17, 40])
def test_wide_rows_mostly_outside_match_oracle(F, P, inside):
    nx, planes, n = 256, 4, 2500
    print(f"case wide rows F={F} P={P} inside={inside}", flush=True)
    rng = np.random.default_rng(F * 100 + P + inside)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    for w0 in range(0, n, 64):      # `inside` rows of every wave, and all of the last part's
        out = rng.permutation(64)[inside:] + w0
        vv[out[out < n - 30]] += 1.5
    vr, vi = (rng.normal(size=n * F * P).astype(np.float32) for _ in range(2))
    vr[1::29] = np.nan
    wt = rng.uniform(0.5, 1.5, n * P).astype(np.float32)
    ref = O.wstack(O.KAISERBESSEL, planes, uu, vv, ww, vr, vi, wt, F, P, 1.0 / nx, 1.0 / planes,
                   7, nx, nx, threads=8)
    plan = Plan(nx, nx, planes, kernel=rick_amd.KAISERBESSEL, support=7, max_points=n)
    got = plan.grid(*[torch.from_numpy(a).to("cuda") for a in (uu, vv, ww, vr, vi, wt)], F,
                    P).cpu().numpy()
    assert np.isfinite(got).all()
    assert rel_l2(got, ref) <= 1e-12
