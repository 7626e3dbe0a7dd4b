"""smk_p1d_rsd_rows where its short cuts end: rows of few points and of ragged
ends, orders of k_perp that leave the spline segment at every point, k_par and
k_perp of 0, out of the fast path's range and past the spline, rows within and
past the cut, and what is no number."""
import numpy as np
import pytest

from oracle import p1d_oracle as po

pytestmark = pytest.mark.gpu

BETA, DX, ZREF = 1.6, 2.19, 2.2
# FP64 on both sides; relative to the sum of the terms' magnitudes, which a
# shuffled order does not cancel
TOL = 1e-12


def _rows(k_par, k_perp, model):
    from saclaymocks_amd import p1d, pk, util
    k, p = pk.p0_nodes(1.0)
    g, par = util.fgrowth(ZREF), po.prats_params(ZREF)
    spl = pk.DeviceSpline(k, p, 30.0)
    got = p1d.rsd_rows(spl, k_par, k_perp, BETA, model, params=par, growth=g, dx=DX)
    with np.errstate(all="ignore"):
        p3 = po.p3d_rsd(k_par, k_perp, po.spline_p(k, p), BETA, model, growth=g, params=par, dx=DX, kny=np.pi / DX)
    return got, p3


@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("n", [2, 3, 65, 257, 258, 2050])
@pytest.mark.parametrize("order", ["up", "down", "shuffled"])
def test_rows_of_ragged_lengths_and_orders(cuda, model, n, order):
    print(f"[p1d edges] model {model} n {n} {order}", flush=True)
    rng = np.random.default_rng(n)
    k_perp = np.concatenate(([0.0], np.sort(rng.uniform(1e-4, 25.0, n - 1))))
    k_perp = {"up": k_perp, "down": k_perp[::-1].copy(), "shuffled": rng.permutation(k_perp)}[order]
    # 0, below and above the fast path's range, on both sides of the cut and of the segments' width
    k_par = np.concatenate(([0.0, 1e-20, 1e-3, np.pi / DX, np.pi / DX * (1 + 1e-13)], rng.uniform(0.01, 20.0, 36)))
    got, p3 = _rows(k_par, k_perp, model)
    f = p3 * k_perp
    seg = 0.5 * (f[:, 1:] + f[:, :-1]) * np.diff(k_perp)
    scale = 0.5 * ((np.abs(f[:, 1:]) + np.abs(f[:, :-1])) * np.abs(np.diff(k_perp))).sum(1) / (2 * np.pi)
    err = np.abs(got - seg.sum(1) / (2 * np.pi))
    assert np.all(err <= TOL * scale), (err / np.maximum(scale, 1e-300)).max()


@pytest.mark.parametrize("model", [0, 1, 2])
def test_rows_of_no_numbers(cuda, model):
    k_perp = np.linspace(0, 20, 700)
    k_par = np.array([0.5, np.nan, 3.0])
    got, _ = _rows(k_par, k_perp, model)
    assert list(np.isnan(got)) == [False, True, False]
    k_perp[350] = np.nan
    got, _ = _rows(k_par, k_perp, model)
    assert np.all(np.isnan(got))


def test_cut_rows_in_groups(cuda):
    """More rows than a block takes one of, in an order that mixes rows within
    and past the cut: each row as it is alone."""
    rng = np.random.default_rng(3)
    k_par = rng.permutation(np.linspace(0, 3, 2051 + 6200))
    k_perp = np.linspace(0, 4, 300)
    got, _ = _rows(k_par, k_perp, 2)
    for i in range(0, len(k_par), 997):
        assert got[i] == _rows(k_par[i:i + 1], k_perp, 2)[0][0]
