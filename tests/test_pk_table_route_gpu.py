"""smk_pk_table at the edges of rows and groups of rows in each of its kernels,
the shapes taken from both sides of the lines between them."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 4001, 65), (2, 650001, 1), (3, 4099, 101), (1, 1, 1300001), (3, 19999, 41),
                                   (9, 5003, 37), (7, 4001, 161), (3, 80001, 41), (11, 30011, 29)])
def test_kernels_agree_with_numpy(cuda, shape):
    from saclaymocks_amd import _lib, pk
    nx, ny, nzh = shape
    print(f"[pk route] {shape}", flush=True)
    kn, pn = pk.p0_nodes(1.0)
    spl = pk.DeviceSpline(kn, pn, 2.0)
    rng = np.random.default_rng(nx + ny + nzh)
    kx, ky, kz = (rng.uniform(-1.3, 1.3, n).astype(np.float32) for n in shape)
    kx[0] = ky[0] = kz[0] = 0.0
    dx, dy, dz = (torch.from_numpy(a).to(cuda) for a in (kx, ky, kz))
    n = nx * ny * nzh
    out = torch.full((n + 8,), -1.0, dtype=torch.float32, device=cuda)
    vcell = float(np.float32(2.19 ** 3))
    _lib.check(_lib.lib().smk_pk_table(ctypes.byref(spl.struct), _lib.ptr(dx), _lib.ptr(dy), _lib.ptr(dz), nx, ny, nzh,
                                       ctypes.c_float(vcell), _lib.ptr(out), _lib.stream_ptr()), "smk_pk_table")
    got = out.cpu().numpy()
    assert np.all(got[n:] == -1.0)
    kk = (kx * kx)[:, None, None] + (ky * ky)[None, :, None] + (kz * kz)[None, None, :]
    p = np.maximum(spl.spline(np.sqrt(kk).astype(np.float64)), 0).astype(np.float32)
    want = np.sqrt(p / np.float32(vcell)).reshape(-1)
    # the spline's rounding may turn a float32 by one place, which the root halves
    assert np.all(np.abs(got[:n] - want) <= np.spacing(want))
    assert np.mean(got[:n] != want) < 0.01
