"""Fused batches whose rows hold 12, 20, 24 or 64 values (16-byte pieces shared by four
lanes), of jobs that end inside a workgroup's rows, against each job's own plan: FP64
<= 1e-12, FP32 <= 1e-6 relative L2, as the batch tests."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from rick_amd import FP32, FP64, KAISERBESSEL, batch, plan_for, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chans,pols", [(3, 4), (5, 4), (12, 2), (64, 1)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_fused_batch_of_wide_rows_matches_plans(chans, pols, precision):
    print(f"case batch wide rows F={chans} P={pols} precision={precision}", flush=True)
    cfgs = [synth.ObsConfig(f"w{k}", "disk", 24, 1500.0, 45.0, times, -3.0, 3.0, 40.0 + k, 150e6,
                            150e6, chans, pols, 3, 256, planes, KAISERBESSEL, 7, seed=50 + k)
            for k, (times, planes) in enumerate(((61, 3), (1, 4), (97, 5)))]
    datasets = [synth.make_dataset(c, device="cuda:0") for c in cfgs]
    fused = batch.FusedBatch(datasets, precision)
    for _ in range(2):
        fused.run_eager()
        torch.cuda.synchronize()
        for ds, got in zip(datasets, fused.images()):
            re, im, _ = plan_for(ds, precision=precision).image(
                ds.uu, ds.vv, ds.ww, ds.vis_real, ds.vis_img, ds.weight, chans, pols)
            want = re.cpu().numpy() + 1j * im.cpu().numpy()
            assert np.isfinite(want).all() and np.abs(want).max() > 0
            assert rel_l2(got, want) <= (1e-12 if precision == FP64 else 1e-6)
