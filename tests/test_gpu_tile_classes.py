"""The tile kernel's accumulation by footprint class, against the CPU oracle (the
suite's 1e-12 in FP64, 1e-6 for an FP32 grid): positions on and next to the
borders of the classes, at the grid's edges and below zero, every support and tile
that has classes, split buckets, non-finite data, and FP32 sums that do not depend
on the order of the rows."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rick_amd import FP32, FP64, GAUSS, KAISERBESSEL, Plan

pytestmark = pytest.mark.gpu
NX, NY, PLANES = 128, 100, 2


def positions(rng, n, cells):
    """Cell coordinates: uniform, on multiples of a tenth of a cell and one ulp
    beside them, at both edges."""
    p = rng.uniform(0.0, cells, n)
    k = n // 3
    p[:k] = np.floor(p[:k]) + rng.integers(0, 10, k) / 10.0
    p[:k // 3] = np.nextafter(p[:k // 3], 0.0)
    p[k // 3:2 * k // 3] = np.nextafter(p[k // 3:2 * k // 3], 1e9)
    p[k:k + 50] = rng.uniform(0.0, 3.0, 50)
    p[k + 50:k + 100] = cells - rng.uniform(0.0, 3.0, 50)
    return p


def make_rows(n, seed, below=0):
    rng = np.random.default_rng(seed)
    uu, vv = positions(rng, n, NX) / NX, positions(rng, n, NY) / NX
    if below:   # halo rows of a slab lie below its first row
        vv[-below:] = -rng.uniform(0.0, 3.0, below) / NX
    ww = rng.uniform(0.0, 1.0, n)
    vr, vi = (rng.normal(size=n).astype(np.float32) for _ in range(2))
    return [uu, vv, ww, vr, vi, rng.uniform(0.5, 1.5, n).astype(np.float32)]


def oracle(rows, kernel, support):
    return O.wstack(kernel, PLANES, *rows, 1, 1, 1.0 / NX, 1.0 / PLANES, support, NX, NY, threads=8)


def grid(plan, rows):
    out = plan.new_grid()
    out.fill_(float("nan"))
    plan.grid(*[torch.from_numpy(a).to("cuda") for a in rows], 1, 1, out=out)
    return out.cpu().numpy()


@pytest.mark.parametrize("tile", [(64, 64), (64, 32), (32, 32), (32, 64), (128, 32)])
@pytest.mark.parametrize("kernel,support", [(KAISERBESSEL, 7), (GAUSS, 7), (KAISERBESSEL, 9),
                                            (KAISERBESSEL, 11), (KAISERBESSEL, 5)])
@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("rows_per_task", [16384, 1500])
def test_dense_tiles_match_oracle(tile, kernel, support, precision, rows_per_task):
    n = 40000
    print(f"case classes tile={tile} kernel={kernel} support={support} precision={precision} "
          f"rows_per_task={rows_per_task}", flush=True)
    rows = make_rows(n, 7, below=400)
    plan = Plan(NX, NY, PLANES, kernel=kernel, support=support, precision=precision, max_points=n,
                tile=tile, rows_per_task=rows_per_task)
    ref = oracle(rows, kernel, support)
    for _ in range(2):
        got = grid(plan, rows)
        assert np.isfinite(got).all()
        assert rel_l2(got, ref) <= (1e-12 if precision == FP64 else 1e-6)


@pytest.mark.parametrize("rows_per_task", [16384, 5000, 1100])
def test_fp32_sums_do_not_depend_on_row_order(rows_per_task):
    # About 10,000 records a bucket: whole, in two parts and in nine or ten.
    n = 60000
    print(f"case order rows_per_task={rows_per_task}", flush=True)
    rows = make_rows(n, 11, below=100)
    plan = Plan(NX, NY, PLANES, kernel=KAISERBESSEL, support=7, precision=FP32, max_points=n,
                tile=(64, 64), rows_per_task=rows_per_task)
    first = grid(plan, rows)
    assert rel_l2(first, oracle(rows, KAISERBESSEL, 7)) <= 1e-6
    for seed in (1, 2):
        order = np.random.default_rng(seed).permutation(n)
        assert np.array_equal(grid(plan, [a[order] for a in rows]), first)


@pytest.mark.parametrize("precision", [FP64, FP32])
def test_non_finite_values_stay_in_their_footprints(precision):
    n = 30000
    print(f"case non-finite precision={precision}", flush=True)
    rows = make_rows(n, 13)
    rows[4][100] = np.nan            # imaginary parts propagate, as in the reference
    rows[4][200] = np.inf
    rows[3][300] = np.inf
    plan = Plan(NX, NY, PLANES, kernel=KAISERBESSEL, support=7, precision=precision, max_points=n,
                tile=(64, 64))
    ref, got = oracle(rows, KAISERBESSEL, 7), grid(plan, rows)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert rel_l2(got[ok], ref[ok]) <= (1e-12 if precision == FP64 else 1e-6)
