"""The drop-ins' staged copies in every direction over many pieces that do not divide the
arrays, pieces of both lengths in one process, and a pinned buffer that grows between a
call's upload and its download.  Each call gets new data; results are compared with the
device path (the same kernels: 1e-14; wstack() the suite's 1e-12)."""
import subprocess
import sys

import numpy as np
import pytest
import torch

from conftest import ROOT, rel_l2
import rick_amd
from rick_amd import FP64, Plan, imaging

pytestmark = pytest.mark.gpu


def test_fft_planes_and_phase_over_many_pieces():
    nx, ny, planes = 500, 510, 11      # 44.9 MB a grid: 11 pieces of 4 MB, the last one short
    plan = Plan(nx, ny, planes, precision=FP64, resolution=1e-4, wmin=-300.0, wmax=500.0)
    gridss = np.empty(2 * planes * ny * nx)
    for call in range(6):
        print(f"case drop-in fft and phase, call {call}", flush=True)
        grid = np.random.default_rng(call).normal(size=2 * planes * ny * nx)
        dev = torch.from_numpy(grid).to("cuda")
        plan.fft(dev)
        gridss.fill(np.nan)
        imaging.fft_planes(planes, nx, ny, grid, gridss)
        want = dev.cpu().numpy()
        assert rel_l2(gridss, want) <= 1e-14
        imaging.fft_planes(planes, nx, ny, grid, grid)          # in place
        assert rel_l2(grid, want) <= 1e-14
        wre, wim = (t.cpu().numpy() for t in plan.phase(dev))
        re, im = np.full(nx * ny, 2.0), np.full(nx * ny, -1.0)
        imaging.phase_correction(gridss, re, im, nx, ny, planes, nx, ny, 1e-4, -300.0, 500.0,
                                 num_threads=1 + 3 * call)
        assert rel_l2(re - 2.0, wre) <= 1e-12 and rel_l2(im + 1.0, wim) <= 1e-12


# Short inputs and a grid of 285 MB: the first call of the process uploads in pieces of 4 MB
# and downloads in pieces of 32 MB, for which the pinned buffer is made anew.
GROWING = """
import numpy as np, torch
import rick_amd
from rick_amd import FP64, Plan, imaging
imaging.set_kernel(rick_amd.KAISERBESSEL)
worst = 0.0
for call, (nx, planes, n, threads) in enumerate(((1024, 17, 300_000, 8), (128, 3, 70_001, 8),
                                                 (1024, 17, 300_000, 16), (128, 3, 5, 2))):
    rng = np.random.default_rng(call)
    uu, vv, ww = (rng.uniform(0.0, 1.0, n) for _ in range(3))
    vr, vi = (rng.normal(size=3 * n).astype(np.float32) for _ in range(2))
    wt = rng.uniform(0.5, 1.5, n).astype(np.float32)
    plan = Plan(nx, nx, planes, kernel=rick_amd.KAISERBESSEL, support=7, precision=FP64,
                max_points=n)
    ins = [torch.from_numpy(a).to("cuda") for a in (uu, vv, ww, vr, vi, wt)]
    want = plan.grid(*ins, 3, 1).cpu().numpy()
    got = np.ones(2 * planes * nx * nx)
    imaging.wstack(planes, n, 3, 1, uu, vv, ww, vr, vi, wt, 1.0 / nx, 1.0 / planes, 7, nx, nx, got,
                   num_threads=threads)
    worst = max(worst, float(np.linalg.norm(got - 1.0 - want) / np.linalg.norm(want)))
    print(f"call {call}: worst {worst:.3e}", flush=True)
assert worst <= 1e-12, worst
"""


def test_pinned_buffer_grows_between_upload_and_download():
    r = subprocess.run([sys.executable, "-c", GROWING], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
