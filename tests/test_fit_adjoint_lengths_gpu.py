"""The gradient and the forward pass of paired forests at the ends of the
transform sizes' length classes, alone and in pairs, with pixels past the last
regrouped point, with and without saved modes, against the oracle."""
import numpy as np
import pytest

from oracle import fit_oracle as fto
from test_fit_gpu import _check_forward, _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("save_modes", [True, False])
@pytest.mark.parametrize("points", [(3, 64, 65, 511, 512), (513, 640, 1023, 1024, 700), (1025, 1536, 1537, 2047, 2048)])
def test_gradient_at_class_ends(cuda, m, save_modes, points):
    print(f"[fit lengths] m {m} save {save_modes} {points}", flush=True)
    # each length in two forests of one set and in one of another; m - 1 pixels left over
    lens = [n * m + (m - 1) for n in points for _ in range(2)] + [n * m for n in points] * 2
    lens = lens[:10] + lens[10:20]
    model, args, theta = _problem(cuda, seed=m, ns=2, per=10, m=m, lens=lens, save_modes=save_modes)
    th = theta * np.array([1.2, 0.9, 1.1] * 2)
    _check_forward(model, args, th)
    val, g = model.value_and_grad(th)
    want = fto.adjoint_grad(th, *args)
    # the bounds that the gradient's other tests have
    assert np.allclose(g, want, rtol=1e-7, atol=1e-9 * np.abs(want).max())
    assert abs(val / fto.chi2(th, *args) - 1) < 1e-10
