"""The distribution of smk_forest_step's skewers over the blocks of the
instance for all length classes: whatever their number (fewer than the blocks,
one or two per block, more with a part in the queue), each is done, with the
bits that it has in a batch of few."""
import numpy as np
import pytest
import torch

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 513, 1025, 1537, 2049, 4001, 9000])
def test_each_skewer_once(cuda, n):
    from saclaymocks_amd import forest
    print(f"[step long queue] n {n}", flush=True)
    rng = np.random.default_rng(n)
    d, e = (torch.from_numpy(rng.normal(0, 1, (16, 16, 64)).astype(np.float32)).to(cuda) for _ in range(2))
    box = forest.BoxView.plane(d, e, cell=2.19, r0=3000.0, periodic=True)
    npix = rng.integers(1, 60, n).astype(np.int32)
    npix[::50] = 2100
    x, y = rng.uniform(-15, 15, n), rng.uniform(-15, 15, n)
    rows = forest.fgpa_rows(np.array([0.1, 0.2, 0.3]), 1.5, 1.0, 0.6)
    pset = rng.integers(0, 3, n).astype(np.int32)
    filt, foff = forest.missing_power_filters(0.2, fo.p1d_missing_analytic)
    plan = forest.ForestPlan()

    def run(lo, hi):
        b = forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(hi - lo, np.int32), npix[lo:hi], 3000.0, 0.2, x[lo:hi],
                               y[lo:hi], pset=pset[lo:hi], noise_id=np.arange(lo, hi, dtype=np.uint64))
        out = {"flux": torch.full((b.npix_total,), float("nan"), device=cuda),
               "status": torch.zeros(b.n, dtype=torch.int32, device=cuda)}
        return forest.step(plan, b, box, filt, foff, rows, seed=5, max_npix=2100, out=out, want=("flux",))["flux"]

    got = run(0, n)
    want = torch.cat([run(lo, min(lo + 200, n)) for lo in range(0, n, 200)])
    assert not torch.isnan(want).any()
    assert torch.equal(got, want)
