"""The Gaussian smoothing along lines of sight (one tube of cells per run of
pixels) against the FP64 oracle, for the lines whose tubes are not the usual
few cells along z: steep, backward and flat lines, pixels farther apart than
cells, positions outside a periodic box, skewers of a few pixels and empty
ones, and skewers that leave a strict box or a resident slab."""
import numpy as np
import pytest
import torch

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu

CELL, R0 = 2.0, 150.0
SHAPE = (24, 20, 28)
# float32 outputs of FP64 sums of O(1) fields
TOL = 2e-6


def _fields(n, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(SHAPE).astype(np.float32) for _ in range(n)]


def _lines(kind, rng):
    """(directions [n][3], pixels per skewer, rmin, dr)."""
    n = 40
    npix = rng.integers(1, 700, n)
    rmin, dr = 100.0, 0.2
    if kind == "steep":
        d = np.stack([rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.uniform(0.3, 1, n)], 1)
    elif kind == "backward":
        d = np.stack([rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n), -rng.uniform(0.5, 1, n)], 1)
    elif kind == "flat":
        d = np.stack([rng.uniform(-0.05, 0.05, n), rng.choice((-1.0, 1.0), n), np.zeros(n)], 1)
    elif kind == "coarse":
        d = np.stack([rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)], 1)
        dr = 7.3 * CELL
    else:
        d = np.stack([rng.uniform(-0.2, 0.2, n), rng.uniform(-0.2, 0.2, n), np.ones(n)], 1)
    if kind == "short":
        n = 900
        npix = rng.integers(0, 5, n)
        npix[0], npix[-1] = 0, 3
        d = np.resize(d, (n, 3))
    return d / np.linalg.norm(d, axis=1)[:, None], npix.astype(np.int32), rmin, dr


def _radial(kind, seed):
    rng = np.random.default_rng(seed)
    d, npix, rmin, dr = _lines(kind, rng)
    qr = rng.uniform(50, 400, len(npix))
    q = d * qr[:, None]
    g0 = rng.integers(0, 300, len(npix)).astype(np.int32)
    R = np.concatenate([rmin + (g + np.arange(k)) * dr for g, k in zip(g0, npix)])
    s = np.repeat(np.arange(len(npix)), npix)
    X, Y, Z = (R * q[s, a] / qr[s] for a in range(3))
    return q, qr, g0, npix, rmin, dr, X, Y, Z


@pytest.mark.parametrize("kind,dmax,nf", [("steep", 3, 7), ("steep", 6, 7), ("steep", 0, 1), ("backward", 3, 10),
                                          ("flat", 3, 7), ("flat", 1, 10), ("coarse", 3, 7), ("coarse", 4, 1),
                                          ("short", 3, 10), ("short", 2, 7), ("plain", 5, 7)])
def test_radial_lines_in_a_periodic_box(cuda, kind, dmax, nf):
    from saclaymocks_amd import forest
    print(f"[gauss radial] {kind} dmax {dmax} fields {nf}", flush=True)
    q, qr, g0, npix, rmin, dr, X, Y, Z = _radial(kind, 11)
    f = _fields(nf, 12)
    t = [torch.from_numpy(x).to(cuda) for x in f]
    box = forest.BoxView(t[0], t[1:7] if nf > 1 else None, cell=CELL, r0=R0, periodic=True, vel=t[7:] or None)
    b = forest.SkewerBatch(forest.GEOM_RADIAL, g0, npix, rmin, dr, q[:, 0], q[:, 1], q[:, 2], qr)
    want = ("delta_l",) + (("eta_par",) if nf > 1 else ()) + (("v_par",) if nf == 10 else ())
    out = forest.gather(b, box, interp="gauss343", want=want, cells=True, dmax=dmax)
    L, D = [CELL * n for n in SHAPE], (CELL,) * 3
    vals, cell = fo.gauss343(f, X, Y, Z, L, D, R0, dmax=dmax, periodic=True)
    got = out["cells"].cpu().numpy()
    assert all(np.array_equal(got[:, a], cell[a]) for a in range(3))
    assert np.abs(out["delta_l"].cpu().numpy() - vals[0]).max() < TOL
    if nf > 1:
        assert np.abs(out["eta_par"].cpu().numpy() - fo.eta_par_radial(vals[1:7], X, Y, Z)).max() < TOL
    if nf == 10:
        assert np.abs(out["v_par"].cpu().numpy() - fo.v_par_radial(vals[7:], X, Y, Z)).max() < TOL
    assert out["status"].sum().item() == 0


@pytest.mark.parametrize("eta", [False, True])
def test_plane_lines_outside_a_periodic_box_with_flux(cuda, eta):
    """x and y up to 1.5 box lengths outside (cells truncate towards zero),
    forests that start and end inside their pixels, the FGPA per skewer."""
    from saclaymocks_amd import forest
    print(f"[gauss plane] eta {eta}", flush=True)
    rng = np.random.default_rng(21)
    n = 60
    npix = rng.integers(1, 500, n).astype(np.int32)
    L, D = [CELL * s for s in SHAPE], (CELL,) * 3
    x, y = rng.uniform(-2 * L[0], 2 * L[0], n), rng.uniform(-2 * L[1], 2 * L[1], n)
    g0 = rng.integers(0, 100, n).astype(np.int32)
    imin, imax = (npix // 5).astype(np.int32), (npix - npix // 7).astype(np.int32)
    rmin, dr = R0 - L[2] / 2 - 9.3, 0.2
    f = _fields(2, 22)
    t = [torch.from_numpy(a).to(cuda) for a in f]
    box = forest.BoxView.plane(t[0], t[1] if eta else None, cell=CELL, r0=R0, periodic=True)
    b = forest.SkewerBatch(forest.GEOM_PLANE, g0, npix, rmin, dr, x, y, imin=imin, imax=imax,
                           pset=np.arange(n, dtype=np.int32))
    par = np.stack([rng.uniform(0.05, 0.2, n), rng.uniform(1, 2, n), rng.uniform(0.5, 1.5, n), np.full(n, 0.8)], 1)
    ds = rng.standard_normal(b.npix_total).astype(np.float32) * 0.3
    out = forest.gather(b, box, interp="gauss343", abcg=forest.fgpa_rows(*par.T), delta_s=torch.from_numpy(ds).to(cuda))
    s = np.repeat(np.arange(n), npix)
    i = np.concatenate([np.arange(k) for k in npix])
    Z = rmin + (g0[s] + i) * dr
    vals, _ = fo.gauss343(f, x[s], y[s], Z, L, D, R0, periodic=True)
    inside = (i >= imin[s]) & (i < imax[s])
    dl = np.where(inside, vals[0], -1e6)
    et = np.where(inside, vals[1], 0.0) if eta else np.zeros(len(s))
    assert np.abs(out["delta_l"].cpu().numpy() - dl).max() < TOL
    assert np.abs(out["eta_par"].cpu().numpy() - et).max() < TOL
    p = par.astype(np.float32).astype(np.float64)[s]
    flux = np.exp(-p[:, 0] * np.exp(p[:, 1] * p[:, 3] * (dl + ds + p[:, 2] * et)))
    assert np.abs(out["flux"].cpu().numpy() - flux).max() < 2e-6


def test_strict_box_and_slab_flags(cuda):
    """Of a strict box's x slab: the pixels whose stencil is inside agree with
    the whole periodic box, the others are NaN, and the status bits say why."""
    from saclaymocks_amd import forest
    q, qr, g0, npix, rmin, dr, X, Y, Z = _radial("plain", 31)
    f = _fields(7, 32)
    t = [torch.from_numpy(a).to(cuda) for a in f]
    b = forest.SkewerBatch(forest.GEOM_RADIAL, g0, npix, rmin, dr, q[:, 0], q[:, 1], q[:, 2], qr)
    whole = forest.gather(b, forest.BoxView(t[0], t[1:], cell=CELL, r0=R0, periodic=True), want=("delta_l", "eta_par"))
    a0, a1 = 5, 19
    slab = forest.BoxView(t[0][a0:a1].contiguous(), [x[a0:a1].contiguous() for x in t[1:]], cell=CELL, r0=R0,
                          periodic=False, x0=a0, nx=SHAPE[0])
    out = forest.gather(b, slab, want=("delta_l", "eta_par"))
    ix, iy, iz = fo.cell_index(X, Y, Z, [CELL * s for s in SHAPE], (CELL,) * 3, R0)
    off_box = np.zeros(len(ix), bool)
    for i, n in zip((ix, iy, iz), SHAPE):
        off_box |= (i < 3) | (i + 3 >= n)
    lo, hi = np.maximum(ix - 3, 0), np.minimum(ix + 3, SHAPE[0] - 1)
    off_slab = (hi >= lo) & ((lo < a0) | (hi >= a1))
    bad = off_box | off_slab
    assert bad.any() and not bad.all()
    for k in ("delta_l", "eta_par"):
        g = out[k].cpu().numpy()
        assert np.all(np.isnan(g[bad])) and np.array_equal(g[~bad], whole[k].cpu().numpy()[~bad])
    s = np.repeat(np.arange(b.n), npix)
    want = np.array([(1 if off_box[s == j].any() else 0) | (4 if off_slab[s == j].any() else 0) for j in range(b.n)])
    assert np.array_equal(out["status"].cpu().numpy(), want)
