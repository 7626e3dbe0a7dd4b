"""The pass variants a plan starts with: each exists for its length, and with
them the fused job and the drop-in steps agree with FP64 FFTs, at every line
length that has its own default; the null and NaN flags of the C2R pass, which
many blocks report through a few words, on boxes of one block and of
thousands."""
import numpy as np
import pytest
import torch

from oracle import box_oracle as bo

pytestmark = pytest.mark.gpu
TOL = 1e-5   # ||x32 - x64||_inf / ||x64||_inf, as for every variant


@pytest.mark.parametrize("n", [320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560])
@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_default_variants(cuda, n, axis):
    from saclaymocks_amd.box import BoxPlan
    # two lines of 16 and one that ends inside a block of 16
    shape = {"x": (n, 18, 24), "y": (18, n, 24), "z": (12, 18, 2 * n)}[axis]
    if axis == "z" and 2 * n > 4096:
        shape = (12, 18, n)
    print(f"[defaults] {shape}", flush=True)
    plan = BoxPlan(*shape, cell=2.19)
    valid = plan.variants()
    assert all(v in valid[k] for k, v in plan.get_variants().items())
    w = np.random.default_rng(n).standard_normal(shape).astype(np.float32)
    noise = torch.from_numpy(w).to(cuda)
    d, e, var, st = plan.grf_box(noise=noise, aux="eta_zz")
    ref = bo.grf_box(w.astype(np.float64), 2.19, aux="eta_zz")
    for got, want in ((d, ref["delta"]), (e, ref["eta_zz"])):
        assert np.abs(got.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    assert abs(var.item() / ref["var"] - 1) < 1e-5
    assert st.cpu().tolist() == [2, 2]
    bk = plan.draw_boxk(noise=noise)
    want = np.fft.rfftn(w.astype(np.float64))
    assert np.abs(bk.cpu().numpy() - want).max() / np.abs(want).max() < TOL
    box, sigma = plan.fft_and_store(bk)
    assert np.abs(box.cpu().numpy() - w).max() / np.abs(w).max() < TOL
    assert sigma == pytest.approx(float(np.std(w.astype(np.float64))), rel=1e-5)


@pytest.mark.parametrize("shape", [(16, 16, 32), (96, 256, 256)])
def test_status_flags(cuda, shape):
    from saclaymocks_amd.box import BoxPlan
    plan = BoxPlan(*shape, cell=2.19)
    noise = torch.zeros(shape, dtype=torch.float32, device=cuda)
    for aux, want in (("eta_zz", [0, 0]), (None, [0, 0])):
        assert plan.grf_box(noise=noise, aux=aux, check=False)[3].cpu().tolist() == want
    noise.normal_()
    assert plan.grf_box(noise=noise, aux=None)[3].cpu().tolist() == [2, 0]
    bk = plan.draw_boxk(noise=noise)
    bk.zero_()
    with pytest.raises(ValueError, match="null"):
        plan.fft_and_store(bk)
    # one NaN pencil, the last: the whole box after the x and y passes
    bk = plan.draw_boxk(noise=noise)
    bk[-1, -1, -1] = float("nan")
    for with_sigma in (True, False):
        with pytest.raises(ValueError, match="NaN"):
            plan.fft_and_store(bk.clone(), with_sigma=with_sigma)
