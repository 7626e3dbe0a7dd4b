"""smk_fgpa_flux over the lines of its rule: a batch of few or long skewers,
which get two or eight waves each, against the same skewers among many short
ones, which get one: the same bits of F, the same sums."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lo,hi", [(50, 601, 1300), (1300, 700, 2600), (1537, 1400, 1800), (2500, 650, 900),
                                     (2200, 6000, 6100)])
@pytest.mark.parametrize("per_pixel", [True, False])
def test_batches_agree(cuda, n, lo, hi, per_pixel):
    from saclaymocks_amd import _lib, forest
    print(f"[flux route] {n} of {lo}..{hi} per pixel {per_pixel}", flush=True)
    rng = np.random.default_rng(n)
    npix = rng.integers(lo, hi + 1, n).astype(np.int32)
    n_row = hi if per_pixel else 5
    pset = rng.integers(0, 5, n).astype(np.int32)
    abcg = torch.from_numpy(rng.uniform(0.3, 1.5, (n_row, 4))).to(cuda)
    d, e = (torch.from_numpy(rng.normal(0, 1, int(npix.sum())).astype(np.float32)).to(cuda) for _ in range(2))

    def run(extra):
        zero = torch.zeros(extra, device=cuda)
        b = forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(n + extra, np.int32),
                               np.concatenate((npix, np.ones(extra, np.int32))), 0.0, 0.2, np.zeros(n + extra),
                               np.zeros(n + extra), pset=None if per_pixel else np.concatenate((pset, np.zeros(extra, np.int32))))
        td, te = torch.cat((d, zero)), torch.cat((e, zero))
        flux = torch.full((b.npix_total,), -1.0, dtype=torch.float64, device=cuda)
        fsum = torch.full((b.n,), -1.0, dtype=torch.float64, device=cuda)
        sk = b.struct()
        _lib.check(_lib.lib().smk_fgpa_flux(ctypes.byref(sk), _lib.ptr(td), _lib.ptr(te), _lib.ptr(abcg), n_row,
                                            _lib.ptr(flux), _lib.ptr(fsum), _lib.stream_ptr()), "smk_fgpa_flux")
        return flux[:len(d)], fsum[:n]

    flux, fsum = run(0)
    want, want_sum = run(100000)
    assert torch.equal(flux, want)
    # sums of up to 6100 positive FP64 terms in two orders
    assert torch.allclose(fsum, want_sum, rtol=1e-12, atol=0.0)
