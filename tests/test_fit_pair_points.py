"""Points per thread of the fit's largest pair kernels: 8 while every pair has a
CU of its own, 16 from there on."""
import pytest

from route_rules import build


@pytest.mark.parametrize("pairs,points", [(1, 8), (200, 8), (256, 8), (257, 16), (10000, 16)])
def test_points(tmp_path, pairs, points):
    assert build(tmp_path, "int points(int pairs) { return fit_pair_points(pairs); }").points(pairs) == points
