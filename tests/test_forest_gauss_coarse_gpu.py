"""The Gaussian smoothing along radial lines whose pixels lie a fraction of a
cell to several cells apart, so that a part of a line is anything from a whole
block's pixels to a few (each part begins with what fitted last), and on both
sides of the spacing where dmax 1 takes the general kernel: against the FP64
oracle."""
import numpy as np
import pytest
import torch

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu

CELL, R0 = 2.0, 150.0
SHAPE = (24, 20, 28)
TOL = 2e-6   # float32 outputs of FP64 sums of O(1) fields


@pytest.mark.parametrize("dmax", [1, 3])
@pytest.mark.parametrize("cells", [0.4, 1.0, 2.7, 2.8, 6.1])
def test_spacings(cuda, cells, dmax):
    from saclaymocks_amd import forest
    print(f"[gauss coarse] {cells} cells dmax {dmax}", flush=True)
    rng = np.random.default_rng(int(10 * cells) + dmax)
    n, dr, rmin = 24, cells * CELL, 90.0
    # along z, along x and in between: from one line to the next the parts' lengths differ
    d = np.concatenate([np.tile([0.05, 0.02, 1.0], (8, 1)), np.tile([1.0, 0.03, 0.01], (8, 1)), rng.uniform(-1, 1, (8, 3))])
    d = rng.permutation(d / np.linalg.norm(d, axis=1)[:, None])
    npix = rng.integers(45, 700, n).astype(np.int32)
    g0 = rng.integers(0, 50, n).astype(np.int32)
    qr = rng.uniform(50, 400, n)
    q = d * qr[:, None]
    f = [rng.standard_normal(SHAPE).astype(np.float32) for _ in range(7)]
    t = [torch.from_numpy(x).to(cuda) for x in f]
    b = forest.SkewerBatch(forest.GEOM_RADIAL, g0, npix, rmin, dr, q[:, 0], q[:, 1], q[:, 2], qr)
    out = forest.gather(b, forest.BoxView(t[0], t[1:], cell=CELL, r0=R0, periodic=True), interp="gauss343",
                        want=("delta_l", "eta_par"), cells=True, dmax=dmax)
    R = np.concatenate([rmin + (g + np.arange(k)) * dr for g, k in zip(g0, npix)])
    s = np.repeat(np.arange(n), npix)
    X, Y, Z = (R * q[s, a] / qr[s] for a in range(3))
    vals, cell = fo.gauss343(f, X, Y, Z, [CELL * m for m in SHAPE], (CELL,) * 3, R0, dmax=dmax, periodic=True)
    got = out["cells"].cpu().numpy()
    assert all(np.array_equal(got[:, a], cell[a]) for a in range(3))
    assert np.abs(out["delta_l"].cpu().numpy() - vals[0]).max() < TOL
    assert np.abs(out["eta_par"].cpu().numpy() - fo.eta_par_radial(vals[1:7], X, Y, Z)).max() < TOL
    assert out["status"].sum().item() == 0
