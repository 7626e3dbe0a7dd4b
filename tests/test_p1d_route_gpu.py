"""smk_p1d_rsd_rows with as many rows as the sum of fewer instructions takes:
ragged lengths, orders of k_perp that leave the spline segment at every point,
k_par out of its range, numbers and no numbers; and the same rows a few at a
time, which the general sum takes."""
import numpy as np
import pytest

from oracle import p1d_oracle as po

pytestmark = pytest.mark.gpu

BETA, DX, ZREF = 1.6, 2.19, 2.2
# FP64 on both sides, relative to the sum of the terms' magnitudes: the sums of
# a row's terms and their rounding (model 1: exponents up to 690)
TOL = 1e-12


@pytest.mark.parametrize("model,n", [(0, 1501), (0, 2050), (1, 351), (1, 514), (1, 1027), (2, 150), (2, 351), (2, 1031)])
@pytest.mark.parametrize("order", ["up", "shuffled"])
def test_many_rows(cuda, model, n, order):
    from saclaymocks_amd import p1d, pk, util
    print(f"[p1d route] model {model} n {n} {order}", flush=True)
    rng = np.random.default_rng(n)
    k_perp = np.concatenate(([0.0], np.sort(rng.uniform(1e-4, 25.0, n - 1))))
    if order == "shuffled":
        k_perp = rng.permutation(k_perp)
    k_par = np.concatenate(([0.0, 1e-20, 1e-3, np.pi / DX, np.pi / DX * (1 + 1e-13), np.nan], rng.uniform(0.01, 20.0, 2994)))
    k, p = pk.p0_nodes(1.0)
    g, par = util.fgrowth(ZREF), po.prats_params(ZREF)
    spl = pk.DeviceSpline(k, p, 30.0)
    run = lambda kp: p1d.rsd_rows(spl, kp, k_perp, BETA, model, params=par, growth=g, dx=DX)  # noqa: E731
    got = run(k_par)
    few = np.concatenate([run(k_par[i:i + 250]) for i in range(0, len(k_par), 250)])
    with np.errstate(all="ignore"):
        p3 = po.p3d_rsd(k_par, k_perp, po.spline_p(k, p), BETA, model, growth=g, params=par, dx=DX, kny=np.pi / DX)
    f = p3 * k_perp
    want = (0.5 * (f[:, 1:] + f[:, :-1]) * np.diff(k_perp)).sum(1) / (2 * np.pi)
    scale = 0.5 * ((np.abs(f[:, 1:]) + np.abs(f[:, :-1])) * np.abs(np.diff(k_perp))).sum(1) / (2 * np.pi)
    ok = np.arange(len(k_par)) != 5
    for v in (got, few):
        assert np.isnan(v[5]) and np.all(np.abs(v - want)[ok] <= TOL * scale[ok])
