"""The Gaussian smoothing along very many very short radial lines, empty ones
among them, which the tubes take, against the same lines a few at a time, which
a thread per pixel takes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CELL, R0 = 2.0, 150.0
SHAPE = (24, 20, 28)
TOL = 2e-6   # float32 outputs of FP64 sums of O(1) fields


@pytest.mark.parametrize("dmax,nf", [(3, 7), (2, 10)])
def test_short_lines(cuda, dmax, nf):
    from saclaymocks_amd import forest
    print(f"[gauss short] dmax {dmax} fields {nf}", flush=True)
    rng = np.random.default_rng(dmax)
    n = 80000
    npix = rng.integers(0, 8, n).astype(np.int32)
    npix[0] = npix[-1] = 0
    assert npix.sum() >= 200000 and npix.sum() >= 2 * n
    d = np.stack([rng.uniform(-0.4, 0.4, n), rng.uniform(-0.4, 0.4, n), np.ones(n)], 1)
    d /= np.linalg.norm(d, axis=1)[:, None]
    qr = rng.uniform(50, 400, n)
    q = d * qr[:, None]
    g0 = rng.integers(0, 300, n).astype(np.int32)
    f = [torch.randn(SHAPE, device=cuda) for _ in range(nf)]
    box = forest.BoxView(f[0], f[1:7], cell=CELL, r0=R0, periodic=True, vel=f[7:] or None)
    want = ("delta_l", "eta_par") + (("v_par",) if nf == 10 else ())

    def run(lo, hi):
        b = forest.SkewerBatch(forest.GEOM_RADIAL, g0[lo:hi], npix[lo:hi], 100.0, 0.2, q[lo:hi, 0], q[lo:hi, 1],
                               q[lo:hi, 2], qr[lo:hi])
        return forest.gather(b, box, interp="gauss343", want=want, cells=True, dmax=dmax)

    got = run(0, n)
    parts = [run(lo, lo + 8000) for lo in range(0, n, 8000)]
    for k in want:
        ref = torch.cat([p[k] for p in parts])
        assert (got[k] - ref).abs().max().item() < TOL
    assert torch.equal(got["cells"], torch.cat([p["cells"] for p in parts]))
    assert got["status"].sum().item() == 0
