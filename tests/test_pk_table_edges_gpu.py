"""smk_pk_table at the edges of a thread's run of modes, a block and a row, on
tables that are not 16-byte aligned, and past the ends of the spline."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _want(spl, kx, ky, kz, vcell):
    """The float32 operations in numpy, the spline in FP64."""
    kk = (kx * kx)[:, None, None] + (ky * ky)[None, :, None] + (kz * kz)[None, None, :]
    assert kk.dtype == np.float32
    p = np.maximum(spl.spline(np.sqrt(kk).astype(np.float64)), 0).astype(np.float32)
    return np.sqrt(p / np.float32(vcell))


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 1), (7, 3, 2), (2, 9, 3), (5, 300, 4), (1, 2, 1023), (2, 3, 1025),
                                   (3, 1, 2050), (37, 11, 129)])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_table_edges(cuda, shape, shift):
    import ctypes
    from saclaymocks_amd import _lib, pk
    nx, ny, nzh = shape
    print(f"[pk edges] {shape} shift {shift}", flush=True)
    kn, pn = pk.p0_nodes(1.0)
    spl = pk.DeviceSpline(kn, pn, 2.0)      # the guess table ends within the axes' range
    rng = np.random.default_rng(nx + ny + nzh)
    kx, ky, kz = (rng.uniform(-2.0, 2.0, n).astype(np.float32) for n in (nx, ny, nzh))
    kx[0] = ky[0] = kz[0] = 0.0
    dx, dy, dz = (torch.from_numpy(a).to(cuda) for a in (kx, ky, kz))
    n = nx * ny * nzh
    buf = torch.full((n + 8,), -1.0, dtype=torch.float32, device=cuda)
    out = buf[shift:shift + n]
    vcell = float(np.float32(2.19 ** 3))
    _lib.check(_lib.lib().smk_pk_table(ctypes.byref(spl.struct), _lib.ptr(dx), _lib.ptr(dy), _lib.ptr(dz), nx, ny, nzh,
                                       ctypes.c_float(vcell), _lib.ptr(out), _lib.stream_ptr()), "smk_pk_table")
    got, all_ = out.cpu().numpy().reshape(shape), buf.cpu().numpy()
    assert np.all(all_[:shift] == -1.0) and np.all(all_[shift + n:] == -1.0)
    want = _want(spl, kx, ky, kz, vcell)
    # the spline's rounding may turn a float32 by one place, which the root halves
    assert np.all(np.abs(got - want) <= np.spacing(want)), np.abs(got - want).max()
    assert np.mean(got != want) < 0.01 or n < 1000


@pytest.mark.parametrize("nodes", [40, 1500, 9000])
@pytest.mark.parametrize("shape", [(3, 1001, 1411), (2, 2100000, 1), (4194400, 1, 1), (1400, 3, 1000)])
def test_large_tables(cuda, shape, nodes):
    """Tables large enough for the spline in LDS, with splines that fit there
    and that do not, axes past the guess table and past the nodes, and nodes
    dense enough for a bin to span several."""
    import ctypes
    from saclaymocks_amd import _lib, pk
    nx, ny, nzh = shape
    print(f"[pk large] {shape} {nodes} nodes", flush=True)
    kn = np.concatenate(([0.0], np.geomspace(1e-3, 1.9, nodes - 1)))
    spl = pk.DeviceSpline(kn, 1e3 * kn / (0.01 + kn ** 2), 1.7)
    rng = np.random.default_rng(nodes)
    kx, ky, kz = (rng.uniform(-1.2, 1.2, n).astype(np.float32) for n in (nx, ny, nzh))
    kx[0] = ky[0] = kz[0] = 0.0
    dx, dy, dz = (torch.from_numpy(a).to(cuda) for a in (kx, ky, kz))
    out = torch.full((nx * ny * nzh + 8,), -1.0, dtype=torch.float32, device=cuda)
    vcell = float(np.float32(2.19 ** 3))
    _lib.check(_lib.lib().smk_pk_table(ctypes.byref(spl.struct), _lib.ptr(dx), _lib.ptr(dy), _lib.ptr(dz), nx, ny, nzh,
                                       ctypes.c_float(vcell), _lib.ptr(out), _lib.stream_ptr()), "smk_pk_table")
    got = out.cpu().numpy()
    assert np.all(got[-8:] == -1.0)
    want = _want(spl, kx, ky, kz, vcell).reshape(-1)
    assert np.all(np.abs(got[:-8] - want) <= np.spacing(want))
    assert np.mean(got[:-8] != want) < 0.01
