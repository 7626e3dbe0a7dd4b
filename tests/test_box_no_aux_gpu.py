"""Boxes without an aux field against the oracle, with the spectral pass's own
default, with each variant set, and in the slab schedule (whose slabs share one
buffer of partial sums)."""
import numpy as np
import pytest
import torch

from oracle import box_oracle as bo

pytestmark = pytest.mark.gpu
TOL = 1e-5   # ||x32 - x64||_inf / ||x64||_inf, as for every box


@pytest.mark.parametrize("n", [512, 640, 1024, 2048])
def test_delta_alone(cuda, n):
    from saclaymocks_amd.box import BoxPlan
    shape = (n, 18, 40)
    w = np.random.default_rng(n).standard_normal(shape).astype(np.float32)
    noise = torch.from_numpy(w).to(cuda)
    ref = bo.grf_box(w.astype(np.float64), 2.19, aux="eta_zz")

    def check(plan, aux):
        d, e, var, st = plan.grf_box(noise=noise, aux=aux)
        assert np.abs(d.cpu().numpy() - ref["delta"]).max() / np.abs(ref["delta"]).max() < TOL
        if aux:
            assert np.abs(e.cpu().numpy() - ref["eta_zz"]).max() / np.abs(ref["eta_zz"]).max() < TOL
        assert abs(var.item() / ref["var"] - 1) < 1e-5
        assert st.cpu().tolist() == ([2, 2] if aux else [2, 0])

    for slabs in (0, 3):
        print(f"[no aux] {shape} slabs {slabs}", flush=True)
        plan = BoxPlan(*shape, cell=2.19)
        plan.set_schedule(slabs)
        check(plan, None)
        check(plan, "eta_zz")
        for v in plan.variants()["x_spectral"]:
            plan.set_variant("x_spectral", v)
            assert plan.get_variants()["x_spectral"] == v
            check(plan, None)
