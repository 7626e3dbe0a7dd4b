"""The distribution of smk_forest_step's skewers over its blocks: whatever
their number (fewer than the blocks, a few per block, many with a part in the
queue), each is done, with the bits that it has in a batch of few."""
import numpy as np
import pytest
import torch

from oracle import forest_oracle as fo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2049, 4097, 20485, 30719, 40963, 61447])
def test_each_skewer_once(cuda, variant, n):
    from saclaymocks_amd import forest
    print(f"[step queue] variant {variant} n {n}", flush=True)
    rng = np.random.default_rng(n)
    nx, ny, nz = 16, 16, 64
    d, e = (torch.from_numpy(rng.normal(0, 1, (nx, ny, nz)).astype(np.float32)).to(cuda) for _ in range(2))
    box = forest.BoxView.plane(d, e, cell=2.19, r0=3000.0, periodic=True)
    npix = rng.integers(1, 40, n).astype(np.int32)
    npix[::97] = 300
    x, y = rng.uniform(-15, 15, n), rng.uniform(-15, 15, n)
    pset = rng.integers(0, 3, n).astype(np.int32)
    rows = forest.fgpa_rows(np.array([0.1, 0.2, 0.3]), 1.5, 1.0, 0.6)
    filt, foff = forest.missing_power_filters(0.2, fo.p1d_missing_analytic)
    plan = forest.ForestPlan()
    plan.set_step_variant(variant)

    def run(lo, hi):
        b = forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(hi - lo, np.int32), npix[lo:hi], 3000.0, 0.2, x[lo:hi],
                               y[lo:hi], pset=pset[lo:hi], noise_id=np.arange(lo, hi, dtype=np.uint64))
        out = {"flux": torch.full((b.npix_total,), float("nan"), device=cuda),
               "status": torch.zeros(b.n, dtype=torch.int32, device=cuda)}
        return forest.step(plan, b, box, filt, foff, rows, seed=5, max_npix=300, out=out, want=("flux",))["flux"]

    got = run(0, n)
    want = torch.cat([run(lo, min(lo + 1000, n)) for lo in range(0, n, 1000)])
    assert not torch.isnan(want).any()
    assert torch.equal(got, want)


@pytest.mark.parametrize("max_npix", [1, 206, 207, 462, 463, 974, 975, 1998])
def test_short_batches_have_the_general_instance_bits(cuda, max_npix):
    """Variant 0's instances for batches without the longer length classes
    against variant 1's, which has all of them: the same register tiles."""
    from saclaymocks_amd import forest
    print(f"[step short] {max_npix}", flush=True)
    rng = np.random.default_rng(max_npix)
    d, e = (torch.from_numpy(rng.normal(0, 1, (16, 16, 256)).astype(np.float32)).to(cuda) for _ in range(2))
    box = forest.BoxView.plane(d, e, cell=2.19, r0=3000.0, periodic=True)
    n = 300
    npix = rng.integers(1, max_npix + 1, n).astype(np.int32)
    npix[0] = max_npix
    b = forest.SkewerBatch(forest.GEOM_PLANE, np.zeros(n, np.int32), npix, 2800.0, 0.2, rng.uniform(-15, 15, n),
                           rng.uniform(-15, 15, n), pset=rng.integers(0, 3, n).astype(np.int32))
    rows = forest.fgpa_rows(np.array([0.1, 0.2, 0.3]), 1.5, 1.0, 0.6)
    filt, foff = forest.missing_power_filters(0.2, fo.p1d_missing_analytic)
    got = []
    for v in (0, 1):
        plan = forest.ForestPlan()
        plan.set_step_variant(v)
        got.append(forest.step(plan, b, box, filt, foff, rows, seed=5, want=("flux", "delta_s", "delta_l", "eta_par")))
    for k in ("flux", "delta_s", "delta_l", "eta_par", "status"):
        assert torch.equal(got[0][k], got[1][k]), k
