"""Which kernel the smoothing along radial lines takes, as measured on both
sides of the lines."""
import ctypes

import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    f = build(tmp_path_factory.mktemp("rule"), "int radial(int dmax, int64_t n, int64_t pixels, double cells) "
              "{ return gather_radial(dmax, n, pixels, cells); }").radial
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_double]
    return f


@pytest.mark.parametrize("dmax,mean,cells,radial", [
    (3, 2400, 0.2 / 2.19, 1), (3, 2, 0.09, 1), (3, 1, 0.09, 0), (1, 50, 0.09, 1), (1, 20, 0.09, 0), (1, 600, 1.0, 1),
    (1, 600, 2.5, 1), (1, 600, 3.0, 0), (1, 600, 8.0, 0), (1, 600, -8.0, 0), (1, 600, float("nan"), 0), (2, 150, 8.0, 1),
    (3, 150, 8.0, 1), (6, 2400, 2.0, 1), (0, 2400, 0.09, 0)])
def test_faster_kernel(rule, dmax, mean, cells, radial):
    assert rule(dmax, 1000, 1000 * mean, cells) == radial
