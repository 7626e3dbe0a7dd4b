"""Boxes whose z pencils have an odd number of complex points (nz / 2 odd):
the device noise draws four cells per Philox call, and there every other
pencil begins in the middle of a call."""
import numpy as np
import pytest
import torch

from oracle import box_oracle as bo
from oracle import philox

pytestmark = pytest.mark.gpu
TOL = 1e-5   # ||x32 - x64||_inf / ||x64||_inf, as for every box


@pytest.mark.parametrize("shape", [(8, 9, 18), (9, 15, 30), (12, 10, 90), (8, 25, 250), (8, 9, 750), (9, 9, 2250)])
def test_device_noise(cuda, shape):
    from saclaymocks_amd.box import BoxPlan
    print(f"[odd half] {shape}", flush=True)
    seed = 987654321
    n = int(np.prod(shape))
    w = philox.device_normals(seed, ((n + 3) // 4 * 4,))[:n].reshape(shape)
    plan = BoxPlan(*shape, cell=2.19)
    bk = plan.draw_boxk(seed=seed)
    want = np.fft.rfftn(w)
    assert np.abs(bk.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    box, sigma = plan.fft_and_store(bk)
    assert np.abs(box.cpu().numpy() - w).max() / np.abs(w).max() < TOL
    assert sigma == pytest.approx(float(np.std(w)), rel=1e-5)
    d, e, var, _ = plan.grf_box(seed=seed, aux="eta_zz")
    ref = bo.grf_box(w, 2.19, aux="eta_zz")
    for got, val in ((d, ref["delta"]), (e, ref["eta_zz"])):
        assert np.abs(got.cpu().numpy() - val).max() / np.abs(val).max() < TOL
    assert abs(var.item() / ref["var"] - 1) < 1e-5
