"""The variant of the z passes that a plan starts with, and when the R2C of 1280
points pads its lines, as measured on both sides of the lines."""
import ctypes

import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    lib = build(tmp_path_factory.mktemp("rule"),
                "int pencil(int m, int c2r, int64_t n) { return box_pencil(m, c2r, n); }\n"
                "int padded(int v, int trans, int64_t n) { return box_r2c_padded(v, trans, n); }")
    lib.pencil.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    lib.padded.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    return lib


@pytest.mark.parametrize("side,r2c,pad", [(64, 1, 1), (200, 1, 1), (256, 1, 1), (320, 0, 0), (400, 0, 0), (512, 0, 1),
                                          (640, 0, 1)])
def test_1280_points(rules, side, r2c, pad):
    assert rules.pencil(1280, 0, side * side) == r2c
    assert rules.padded(r2c, 1, side * side) == pad
    assert rules.padded(r2c, 0, side * side) == 0
    assert rules.pencil(1280, 1, side * side) == 1


@pytest.mark.parametrize("m,r2c,c2r", [(320, 1, 1), (384, 1, 2), (768, 0, 2), (128, 0, 0), (512, 0, 0), (2560, 0, 0)])
def test_other_lengths(rules, m, r2c, c2r):
    for n in (100, 10 ** 6):
        assert (rules.pencil(m, 0, n), rules.pencil(m, 1, n)) == (r2c, c2r)
