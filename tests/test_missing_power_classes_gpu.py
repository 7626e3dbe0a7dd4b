"""The missing power of batches with empty length classes: only the classes
that have skewers are launched."""
import numpy as np
import pytest

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu


def _batch(npix, ids):
    from saclaymocks_amd import forest
    n = len(npix)
    return forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(n, np.int32), np.asarray(npix, np.int32), 0.0, 0.2,
                              np.zeros(n), np.zeros(n), noise_id=ids)


def test_missing_power_of_single_classes(cuda):
    """A skewer alone, with one class launched, has the bits that it has in a
    batch of every class (which other tests hold to the oracle), for lengths at
    the ends of the classes and for more skewers than a block's lines."""
    from saclaymocks_amd import forest
    npix = [8142, 1, 206, 207, 462, 463, 974, 975, 1998, 1999, 4046, 4047, 8142] + [100] * 20
    ids = np.arange(7, 7 + len(npix), dtype=np.uint64)
    filt, foff = forest.missing_power_filters(0.2, fo.p1d_missing_analytic)
    plan = forest.ForestPlan()
    b = _batch(npix, ids)
    together = b.split(forest.missing_power(plan, b, filt, foff, seed=99))
    for lo, hi in [(s, s + 1) for s in range(13)] + [(13, 33)]:
        print(f"[missing power alone] {npix[lo]} x {hi - lo}", flush=True)
        b = _batch(npix[lo:hi], ids[lo:hi])
        alone = b.split(forest.missing_power(plan, b, filt, foff, seed=99))
        for s in range(lo, hi):
            assert np.std(together[s]) > 0 or npix[s] == 1
            assert alone[s - lo].tobytes() == together[s].tobytes(), s
