"""The fit's forward pass and gradient with as many pairs of more than 1024
points as one kernel of each kind takes and a few more, against the oracle."""
import numpy as np
import pytest

from oracle import fit_oracle as fto
from test_fit_gpu import _check_forward, _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("forests", [500, 530])
@pytest.mark.parametrize("save_modes", [True, False])
def test_gradient(cuda, m, forests, save_modes):
    print(f"[pair points] m {m} forests {forests} save {save_modes}", flush=True)
    # two forests of a length, m - 1 pixels left over
    lens = [(1025 + i // 2) * m + (m - 1) for i in range(forests)]
    model, args, theta = _problem(cuda, seed=m, ns=2, per=forests // 2, m=m, lens=lens, save_modes=save_modes)
    th = theta * np.array([1.2, 0.9, 1.1] * 2)
    _check_forward(model, args, th)
    val, g = model.value_and_grad(th)
    want = fto.adjoint_grad(th, *args)
    # the bounds that the gradient's other tests have
    assert np.allclose(g, want, rtol=1e-7, atol=1e-9 * np.abs(want).max())
    assert abs(val / fto.chi2(th, *args) - 1) < 1e-10
