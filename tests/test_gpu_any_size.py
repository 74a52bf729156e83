"""Transforms of axes beside the power-of-two engine: every radix, the longest
and shortest one-pass lines, and the image chain on a sparse grid of such a
size against the separate stages on a dense one.

Bars: the suite's 1e-14 / 2e-6 relative L2 for a transform against numpy, and
1e-12 (FP64) / 1e-5 (FP32) for images."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
import rick_amd
from rick_amd import FP32, FP64, Plan

pytestmark = pytest.mark.gpu


def cube(plan, flat):
    c = flat.cpu().numpy().astype(np.float64).reshape(plan.planes, plan.ny, plan.nx, 2)
    return c[..., 0] + 1j * c[..., 1]


@pytest.mark.parametrize("nx,ny,planes", [
    (196, 81, 2), (240, 143, 1), (176, 156, 3), (4095, 12, 1), (3993, 14, 1), (4096, 100, 1),
    (3584, 18, 2), (130, 520, 2), (20, 3600, 1), (33, 257 * 2, 1), (17, 300, 1)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_lengths_of_every_radix_match_numpy(nx, ny, planes, precision):
    print(f"case fft {nx}x{ny}x{planes} precision={precision}", flush=True)
    plan = Plan(nx, ny, planes, precision=precision)
    rng = np.random.default_rng(nx + 7 * ny)
    src = torch.from_numpy(rng.normal(size=2 * planes * ny * nx)).to("cuda", plan.grid_dtype)
    want = np.fft.ifft2(cube(plan, src), axes=(1, 2))
    out = plan.fft(src, torch.empty_like(src))
    assert rel_l2(cube(plan, out), want) <= (1e-14 if precision == FP64 else 2e-6)
    plan.fft(src)   # in place
    assert rel_l2(cube(plan, src), want) <= (1e-14 if precision == FP64 else 2e-6)


# Rows in thin v-stripes that start and end inside tile rows, the whole grid
# width or a part of it; the grid starts as NaN, so a cell that the sparse
# chain reads without having written it shows.
@pytest.mark.parametrize("nx,ny,planes,tile", [
    (18, 300, 3, (32, 32)), (300, 200, 4, (64, 32)), (130, 600, 3, (64, 64)),
    (143, 169, 2, (0, 0)), (1000, 1500, 2, (128, 32)), (4095, 66, 2, (32, 64)),
    (12, 14, 1, (0, 0)), (100, 512, 2, (64, 64)),
    # power-of-two axes on both sides of the fused phase pass
    (1024, 512, 3, (64, 32)), (2048, 512, 3, (0, 0)), (32, 16, 5, (32, 32))])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_sparse_chain_matches_separate_stages(nx, ny, planes, tile, precision):
    print(f"case chain {nx}x{ny}x{planes} tile={tile} precision={precision}", flush=True)
    n = 20000
    plan = Plan(nx, ny, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=precision,
                max_points=n, tile=tile, resolution=1.0 / (4.0 * max(nx, ny)), wmin=-300.0,
                wmax=500.0)
    for call in range(2):
        rng = np.random.default_rng(11 + call)
        uu = rng.uniform(0.1 * call, 0.9, n)
        vv = (rng.choice([0.13, 0.47, 0.71], n) + rng.uniform(0.0, 0.04, n)) * ny / nx
        ww = rng.uniform(0.0, 0.6, n)             # the last planes stay empty
        ins = [torch.from_numpy(a).to("cuda") for a in (
            uu, vv, ww, rng.normal(size=n).astype(np.float32),
            rng.normal(size=n).astype(np.float32), np.ones(n, np.float32))]
        grid = plan.new_grid()
        grid.fill_(float("nan"))
        re, im, _ = plan.image(*ins, grid=grid)
        dense = plan.grid(*ins)
        plan.fft(dense)
        wre, wim = plan.phase(dense)
        got, want = ((a.cpu().numpy() + 1j * b.cpu().numpy()) for a, b in ((re, im), (wre, wim)))
        assert np.isfinite(want).all() and np.abs(want).max() > 0
        assert rel_l2(got, want) <= (1e-12 if precision == FP64 else 1e-5)


# The fused column/phase pass: lines with and without the prefetch (16 to 64 and 128
# to 512 points), strips wider than the grid, rows without a cell, one plane (no
# phase), two and an odd number of them.
@pytest.mark.parametrize("nx,ny", [
    (16, 1024), (64, 2048), (32, 4096), (16, 8192), (8192, 128), (4096, 256), (2048, 512)])
@pytest.mark.parametrize("planes", [1, 2, 5])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_phase_pass_of_every_line_length_matches_stages(nx, ny, planes, precision):
    print(f"case phase pass {nx}x{ny}x{planes} precision={precision}", flush=True)
    n = 5000
    plan = Plan(nx, ny, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=precision,
                max_points=n, resolution=1.0 / (4.0 * max(nx, ny)), wmin=-300.0, wmax=500.0)
    rng = np.random.default_rng(nx + ny + planes)
    uu = rng.uniform(0.0, 0.9, n)
    vv = (rng.choice([0.13, 0.71], n) + rng.uniform(0.0, 0.04, n)) * ny / nx
    ins = [torch.from_numpy(a).to("cuda") for a in (
        uu, vv, rng.uniform(0.0, 0.9, n), rng.normal(size=n).astype(np.float32),
        rng.normal(size=n).astype(np.float32), np.ones(n, np.float32))]
    grid = plan.new_grid()
    grid.fill_(float("nan"))
    re, im, _ = plan.image(*ins, grid=grid)
    dense = plan.grid(*ins)
    plan.fft(dense)
    wre, wim = plan.phase(dense)
    got, want = ((a.cpu().numpy() + 1j * b.cpu().numpy()) for a, b in ((re, im), (wre, wim)))
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    assert rel_l2(got, want) <= (1e-12 if precision == FP64 else 1e-5)


# Column transforms of one pass (up to 1024 rows in FP64, 2048 in FP32) and the
# first of two passes above: fewer strips than a round over the XCDs, and paired
# strips.
@pytest.mark.parametrize("nx,ny", [(16, 1024), (64, 2048), (512, 1024), (512, 2048), (256, 512)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_long_columns_match_numpy(nx, ny, precision):
    print(f"case columns {nx}x{ny} precision={precision}", flush=True)
    plan = Plan(nx, ny, 3, precision=precision)
    rng = np.random.default_rng(nx + ny)
    src = torch.from_numpy(rng.normal(size=6 * ny * nx)).to("cuda", plan.grid_dtype)
    want = np.fft.ifft2(cube(plan, src), axes=(1, 2))
    out = plan.fft(src, torch.empty_like(src))
    assert rel_l2(cube(plan, out), want) <= (1e-14 if precision == FP64 else 2e-6)
    plan.fft(src)
    assert rel_l2(cube(plan, src), want) <= (1e-14 if precision == FP64 else 2e-6)


# FP32 strips of 256 columns from 512 workgroups on (out of place here; in place, a
# plane at a time, stays below) and of 128 below or where rows lie over 2 MB apart.
@pytest.mark.parametrize("nx,ny,planes", [(1024, 4096, 2), (2048, 4096, 1), (512, 8192, 2)])
def test_wide_column_strips_match_numpy(nx, ny, planes):
    print(f"case wide columns {nx}x{ny}x{planes}", flush=True)
    plan = Plan(nx, ny, planes, precision=FP32)
    rng = np.random.default_rng(nx + ny)
    src = torch.from_numpy(rng.normal(size=2 * planes * ny * nx)).to("cuda", plan.grid_dtype)
    want = np.fft.ifft2(cube(plan, src), axes=(1, 2))
    out = plan.fft(src, torch.empty_like(src))
    assert rel_l2(cube(plan, out), want) <= 2e-6
    plan.fft(src)
    assert rel_l2(cube(plan, src), want) <= 2e-6


@pytest.mark.parametrize("planes", [7, 8])      # 448 and 512 workgroups of 256 columns
def test_wide_column_strips_on_a_sparse_grid(planes):
    print(f"case wide chain planes={planes}", flush=True)
    n, nx, ny = 20000, 1024, 1024
    plan = Plan(nx, ny, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=FP32,
                max_points=n, resolution=1.0 / (4.0 * nx), wmin=-300.0, wmax=500.0)
    rng = np.random.default_rng(planes)
    ins = [torch.from_numpy(a).to("cuda") for a in (
        rng.uniform(0.0, 0.9, n), rng.choice([0.13, 0.47], n) + rng.uniform(0.0, 0.04, n),
        rng.uniform(0.0, 0.9, n), rng.normal(size=n).astype(np.float32),
        rng.normal(size=n).astype(np.float32), np.ones(n, np.float32))]
    grid = plan.new_grid()
    grid.fill_(float("nan"))
    re, im, _ = plan.image(*ins, grid=grid)
    dense = plan.grid(*ins)
    plan.fft(dense)
    wre, wim = plan.phase(dense)
    got, want = ((a.cpu().numpy() + 1j * b.cpu().numpy()) for a, b in ((re, im), (wre, wim)))
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    assert rel_l2(got, want) <= 1e-5


# The last column pass of a four-step axis with and without the phase in it: rows at
# 1024 workgroups and below, strips that the width does not fill, a single radix, a
# factor of 11 (never in one).
@pytest.mark.parametrize("nx,ny,planes", [
    (1920, 2560, 3), (2000, 2000, 1), (1500, 1500, 2), (4095, 360, 3), (2100, 3300, 2),
    (3000, 1920, 2)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_any_size_phase_pass_matches_separate_stages(nx, ny, planes, precision):
    test_phase_pass_of_every_line_length_matches_stages(nx, ny, planes, precision)
