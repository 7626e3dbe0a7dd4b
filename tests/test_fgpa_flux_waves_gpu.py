"""smk_fgpa_flux with two and eight waves to a skewer against one wave (which
other tests hold to the oracle): the same bits of F, at ragged and extreme
lengths."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _batch(npix, pset=None, imin=None, imax=None, ids=None):
    from saclaymocks_amd import forest
    n = len(npix)
    return forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(n, np.int32), np.asarray(npix, np.int32), 0.0, 0.2,
                              np.zeros(n), np.zeros(n), pset=pset, imin=imin, imax=imax, noise_id=ids)


# mean lengths on each side of the rule's 1400 pixels, counts on each side of 4096
@pytest.mark.parametrize("n,lo,hi", [(1, 1, 1), (3, 5000, 9000), (9, 1, 2900), (17, 1, 700), (700, 1399, 1401),
                                     (4097, 1, 90), (4100, 1400, 1403)])
@pytest.mark.parametrize("rows", ["pixel", "skewer"])
@pytest.mark.parametrize("with_eta", [True, False])
def test_flux_and_sums(cuda, n, lo, hi, rows, with_eta):
    from saclaymocks_amd import _lib
    print(f"[flux waves] {n} of {lo}..{hi} {rows} eta {with_eta}", flush=True)
    rng = np.random.default_rng(n + hi)
    npix = rng.integers(lo, hi + 1, n).astype(np.int32)
    imin = (npix * rng.uniform(0, 0.5, n)).astype(np.int32)
    imax = (imin + (npix - imin) * rng.uniform(0, 1, n)).astype(np.int32)
    n_row = int(npix.max()) if rows == "pixel" else 5
    pset = None if rows == "pixel" else rng.integers(0, n_row, n).astype(np.int32)
    tot = int(npix.sum())
    abcg = rng.uniform(0.3, 1.5, (n_row, 4))
    d, e = (rng.normal(0, 1, tot).astype(np.float32) for _ in range(2))

    def run(extra):
        # extra skewers of one pixel: 4096 or more in all take one wave each
        one = np.ones(extra, np.int32)
        b = _batch(np.concatenate((npix, one)), None if pset is None else np.concatenate((pset, 0 * one)),
                   np.concatenate((imin, 0 * one)), np.concatenate((imax, one)))
        td, te = (torch.from_numpy(np.concatenate((a, np.zeros(extra, np.float32)))).to(cuda) for a in (d, e))
        ta = torch.from_numpy(abcg).to(cuda)
        flux = torch.full((tot + extra + 1,), -1.0, dtype=torch.float64, device=cuda)
        fsum = torch.full((n + extra + 1,), -1.0, dtype=torch.float64, device=cuda)
        sk = b.struct()
        _lib.check(_lib.lib().smk_fgpa_flux(ctypes.byref(sk), _lib.ptr(td), _lib.ptr(te) if with_eta else None,
                                            _lib.ptr(ta), n_row, _lib.ptr(flux), _lib.ptr(fsum), _lib.stream_ptr()),
                   "smk_fgpa_flux")
        assert flux[-1].item() == -1.0 and fsum[-1].item() == -1.0
        return flux.cpu().numpy()[:tot], fsum.cpu().numpy()[:n]

    got, sums = run(0)
    extra = max(4096 - n, 0)
    while tot + extra >= 1400 * (n + extra):
        extra += 4096
    want, want_sums = run(extra)
    assert got.tobytes() == want.tobytes()
    s = np.repeat(np.arange(n), npix)
    i = np.arange(tot) - np.repeat(np.cumsum(npix) - npix, npix)
    inside = (i >= imin[s]) & (i < imax[s])
    # sums of positive FP64 terms in another order: up to 9000 of them, the
    # errors of whose partial sums grow as the number of terms per lane and step
    exact = np.bincount(s, weights=np.where(inside, got, 0.0), minlength=n)
    for q in (sums, want_sums):
        assert np.allclose(q, exact, rtol=1e-12, atol=0.0)
