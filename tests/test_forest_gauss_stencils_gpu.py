"""Every stencil of the Gaussian smoothing along radial lines, with eta and with
the velocities too, against the FP64 oracle; the largest takes nearly all of a
CU's LDS."""
import numpy as np
import pytest
import torch

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu

CELL, R0 = 2.0, 150.0
SHAPE = (24, 20, 28)
TOL = 2e-6   # float32 outputs of FP64 sums of O(1) fields


@pytest.mark.parametrize("dmax,nf", [(2, 10), (4, 7), (4, 10), (5, 10), (6, 10)])
@pytest.mark.parametrize("periodic", [True, False])
def test_stencils(cuda, dmax, nf, periodic):
    from saclaymocks_amd import forest
    print(f"[gauss stencils] dmax {dmax} fields {nf} periodic {periodic}", flush=True)
    rng = np.random.default_rng(10 * dmax + nf)
    n, dr, rmin = 16, 0.2, 125.0
    d = np.stack([rng.uniform(-0.15, 0.15, n), rng.uniform(-0.1, 0.1, n), np.ones(n)], 1)
    d /= np.linalg.norm(d, axis=1)[:, None]
    npix = rng.integers(100, 330, n).astype(np.int32)
    qr = rng.uniform(50, 400, n)
    q = d * qr[:, None]
    f = [rng.standard_normal(SHAPE).astype(np.float32) for _ in range(nf)]
    t = [torch.from_numpy(x).to(cuda) for x in f]
    b = forest.SkewerBatch(forest.GEOM_RADIAL, np.zeros(n, np.int32), npix, rmin, dr, q[:, 0], q[:, 1], q[:, 2], qr)
    box = forest.BoxView(t[0], t[1:7], cell=CELL, r0=R0, periodic=periodic, vel=t[7:] or None)
    out = forest.gather(b, box, interp="gauss343", want=("delta_l", "eta_par") + (("v_par",) if nf == 10 else ()),
                        dmax=dmax)
    R = np.concatenate([rmin + np.arange(k) * dr for k in npix])
    s = np.repeat(np.arange(n), npix)
    X, Y, Z = (R * q[s, a] / qr[s] for a in range(3))
    # a strict box's pixels whose stencil is inside have the periodic box's values, the others none
    vals, cell = fo.gauss343(f, X, Y, Z, [CELL * m for m in SHAPE], (CELL,) * 3, R0, dmax=dmax, periodic=True)
    good = np.ones(len(X), bool)
    if not periodic:
        for c, m in zip(cell, SHAPE):
            good &= (c >= dmax) & (c + dmax < m)
        assert good.any() and not good.all()
    want = [vals[0], fo.eta_par_radial(vals[1:7], X, Y, Z)]
    if nf == 10:
        want.append(fo.v_par_radial(vals[7:], X, Y, Z))
    for k, w in zip(("delta_l", "eta_par", "v_par"), want):
        got = out[k].cpu().numpy()
        assert np.all(np.isnan(got[~good])) and np.abs(got - w)[good].max() < TOL
