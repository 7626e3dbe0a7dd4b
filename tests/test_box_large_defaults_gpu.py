"""The variants that large boxes start with, on boxes small enough for the
oracle: the fused job and the drop-in steps, at every length that has one."""
import numpy as np
import pytest
import torch

from oracle import box_oracle as bo

pytestmark = pytest.mark.gpu
TOL = 1e-5   # ||x32 - x64||_inf / ||x64||_inf, as for every box


@pytest.mark.parametrize("n", [320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560])
@pytest.mark.parametrize("axis", ["x", "y"])
def test_variants(cuda, n, axis):
    from saclaymocks_amd.box import BoxPlan
    # two lines of 16 and one that ends inside a block of 16
    shape = (n, 18, 24) if axis == "x" else (18, n, 24)
    large = BoxPlan(*((n, 1280, 1280) if axis == "x" else (1280, n, 1280)), cell=2.19).get_variants()
    plan = BoxPlan(*shape, cell=2.19)
    kinds = ("x_spectral", "x_fwd", "x_inv") if axis == "x" else ("y_fwd", "y_inv")
    for k in kinds:
        plan.set_variant(k, large[k])
    print(f"[large defaults] {shape} { {k: large[k] for k in kinds} }", flush=True)
    assert any(large[k] for k in kinds) or n == 2560
    w = np.random.default_rng(n).standard_normal(shape).astype(np.float32)
    noise = torch.from_numpy(w).to(cuda)
    d, e, var, st = plan.grf_box(noise=noise, aux="eta_zz")
    ref = bo.grf_box(w.astype(np.float64), 2.19, aux="eta_zz")
    for got, want in ((d, ref["delta"]), (e, ref["eta_zz"])):
        assert np.abs(got.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    assert abs(var.item() / ref["var"] - 1) < 1e-5 and st.cpu().tolist() == [2, 2]
    bk = plan.draw_boxk(noise=noise)
    want = np.fft.rfftn(w.astype(np.float64))
    assert np.abs(bk.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    box, sigma = plan.fft_and_store(bk)
    assert np.abs(box.cpu().numpy() - w).max() / np.abs(w).max() < TOL
    assert sigma == pytest.approx(float(np.std(w.astype(np.float64))), rel=1e-5)
