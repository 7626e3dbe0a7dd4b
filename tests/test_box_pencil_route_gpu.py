"""The R2C of 1280-point pencils with padded lines and without: small boxes
against the oracle for each variant, and a box large enough for the padded
variant 0, whose two variants must agree."""
import numpy as np
import pytest
import torch

from oracle import box_oracle as bo

pytestmark = pytest.mark.gpu
TOL = 1e-5   # ||x32 - x64||_inf / ||x64||_inf, as for every box


@pytest.mark.parametrize("variant", [0, 1])
def test_small_box(cuda, variant):
    from saclaymocks_amd.box import BoxPlan
    shape = (9, 18, 2560)
    print(f"[pencils] {shape} variant {variant}", flush=True)
    plan = BoxPlan(*shape, cell=2.19)
    plan.set_variant("z_r2c", variant)
    w = np.random.default_rng(5).standard_normal(shape).astype(np.float32)
    noise = torch.from_numpy(w).to(cuda)
    d, e, var, _ = plan.grf_box(noise=noise, aux="eta_zz")
    ref = bo.grf_box(w.astype(np.float64), 2.19, aux="eta_zz")
    for got, want in ((d, ref["delta"]), (e, ref["eta_zz"])):
        assert np.abs(got.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    bk = plan.draw_boxk(noise=noise)
    want = np.fft.rfftn(w.astype(np.float64))
    assert np.abs(bk.cpu().numpy() - want).max() / np.abs(want).max() < TOL


def test_large_box(cuda):
    from saclaymocks_amd.box import BoxPlan
    plan = BoxPlan(450, 450, 2560, cell=2.19)
    assert plan.get_variants()["z_r2c"] == 0
    print("[pencils] 450 x 450 x 2560", flush=True)
    ws = plan.alloc_workspace()
    a = plan.grf_box(seed=3, aux=None, workspace=ws)[0]
    plan.set_variant("z_r2c", 1)
    b = plan.grf_box(seed=3, aux=None, workspace=ws)[0]
    assert ((a - b).abs().max() / b.abs().max()).item() < TOL
