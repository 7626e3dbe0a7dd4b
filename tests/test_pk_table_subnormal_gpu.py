"""Quotients P / vcell in the subnormal range of float32, where they can be the
exact middle of two numbers: rounded to even, as numpy's division does."""
import ctypes

import numpy as np
import pytest
import torch

from saclaymocks_amd import _lib, pk

pytestmark = pytest.mark.gpu


# below and above the size at which the blocks keep the spline in LDS
@pytest.mark.parametrize("shape", [(2, 3, 70), (64, 270, 260)])
@pytest.mark.parametrize("vcell", [6.0, 98.0, 196.0, 412.0])
def test_ties_round_to_even(cuda, vcell, shape):
    print(f"[pk subnormal] vcell {vcell} {shape}", flush=True)
    # P is constant between nodes: j 2^-149, j = 0 ... 3999, on unit intervals of k
    n = 4000
    x = np.arange(n + 1, dtype=np.float64)
    c = np.zeros((n, 4))
    c[:, 3] = np.arange(n) * 2.0 ** -149
    t = [torch.from_numpy(a).to(cuda) for a in (x, c, np.arange(n, dtype=np.int32))]
    sp = pk.SmkPkSpline()
    sp.x, sp.c, sp.guess = (a.data_ptr() for a in t)
    sp.n_int, sp.n_guess, sp.g_lo, sp.g_step = n, n, 0.0, 1.0
    # k = kz + 1/2: the modes of a row run through the intervals
    rng = np.random.default_rng(int(vcell))
    kz = (rng.integers(0, n, shape[2]) + 0.5).astype(np.float32)
    kz[:12] = np.array([147, 294, 309, 343, 588, 618, 686, 721, 735, 1127, 1133, 1323]) + np.float32(0.5)
    zero = [torch.zeros(m, device=cuda) for m in shape[:2]]
    out = torch.empty(shape, device=cuda)
    tz = torch.from_numpy(kz).to(cuda)
    _lib.check(_lib.lib().smk_pk_table(ctypes.byref(sp), _lib.ptr(zero[0]), _lib.ptr(zero[1]), _lib.ptr(tz), *shape,
                                       ctypes.c_float(vcell), _lib.ptr(out), _lib.stream_ptr()), "smk_pk_table")
    p = (np.floor(kz.astype(np.float64)) * 2.0 ** -149).astype(np.float32)
    want = np.sqrt(p / np.float32(vcell))
    assert np.array_equal(out.cpu().numpy(), np.broadcast_to(want, shape))
