"""Which kernel the smoothing along radial lines takes, as measured on both
sides of the lines."""
import ctypes

import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    f = build(tmp_path_factory.mktemp("rule"), "int radial(int dmax, int fields, int64_t n, int64_t pixels, double cells) "
              "{ return gather_radial(dmax, fields, n, pixels, cells); }").radial
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_double]
    return f


@pytest.mark.parametrize("dmax,mean,cells,radial", [
    (3, 2400, 0.2 / 2.19, 1), (3, 20, 0.09, 1), (3, 1, 0.09, 0), (1, 70, 0.09, 1), (1, 20, 0.09, 0), (1, 600, 1.0, 1),
    (1, 600, 2.5, 1), (1, 600, 3.0, 0), (1, 600, 8.0, 0), (1, 600, -8.0, 0), (1, 600, float("nan"), 0), (2, 150, 8.0, 1),
    (3, 150, 8.0, 1), (6, 2400, 2.0, 1), (0, 2400, 0.09, 0)])
def test_faster_kernel(rule, dmax, mean, cells, radial):
    assert rule(dmax, 7, 10000, 10000 * mean, cells) == radial


@pytest.mark.parametrize("dmax,fields,pixels,mean,radial", [
    (1, 7, 30000, 100, 0), (1, 7, 30000, 300, 1), (1, 7, 800000, 45, 0), (1, 7, 800000, 100, 1), (1, 10, 30000, 45, 0),
    (1, 10, 800000, 45, 1), (2, 7, 30000, 20, 0), (2, 7, 30000, 45, 1), (2, 7, 800000, 5, 0), (2, 10, 30000, 5, 0),
    (2, 10, 30000, 20, 1), (3, 7, 30000, 5, 0), (3, 7, 30000, 20, 1), (3, 7, 800000, 5, 1), (3, 10, 800000, 2, 1),
    (3, 7, 500, 500, 1)])
def test_batches_that_do_not_fill_the_card(rule, dmax, fields, pixels, mean, radial):
    assert rule(dmax, fields, pixels // mean, pixels, 0.09) == radial
