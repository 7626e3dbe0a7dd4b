"""The waves that a skewer of the FGPA flux gets, as measured on both sides of
the lines."""
import ctypes

import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    f = build(tmp_path_factory.mktemp("rule"),
              "int waves(int64_t n, int64_t pixels, int pp) { return flux_waves(n, pixels, pp); }").waves
    f.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return f


@pytest.mark.parametrize("per_pixel", [0, 1])
@pytest.mark.parametrize("n,mean,waves", [
    (600, 200, 1), (600, 700, 2), (600, 7500, 8), (1000, 1400, 8), (1500, 6500, 8), (1700, 4500, 8),
    (2000, 4500, 2), (2100, 3000, 8), (2500, 3000, 8), (2700, 3000, 2), (3000, 300, 1), (3000, 700, 2),
    (3000, 3000, 2), (3000, 9000, 8), (3100, 2000, 8), (3300, 4500, 8), (5000, 400, 1), (5000, 3000, 2),
    (6000, 1500, 1), (6300, 4500, 8), (10000, 1400, 1), (10000, 2000, 1), (20000, 900, 1), (20000, 1500, 1),
    (20000, 3000, 1), (50000, 2000, 1)])
def test_waves(rule, n, mean, waves, per_pixel):
    assert rule(n, n * mean, per_pixel) == waves


def test_parameters_per_pixel(rule):
    assert [rule(10000, 10000 * 6500, p) for p in (0, 1)] == [8, 1]
    assert [rule(2000, 2000 * 1000, p) for p in (0, 1)] == [1, 2]
    assert [rule(1500, 1500 * 1400, p) for p in (0, 1)] == [2, 8]
    assert [rule(4000, 4000 * 1400, p) for p in (0, 1)] == [1, 2]
    assert [rule(1100, 1100 * 1000, p) for p in (0, 1)] == [1, 2]
    assert rule(0, 0, 0) == 1
