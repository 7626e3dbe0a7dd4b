"""Which kernel a P(k) table takes: a thread per mode where the rows would leave
many lanes of a wave idle, as measured on both sides of the lines."""
import ctypes

import pytest

from route_rules import build

MODES, ROWS, LDS = 0, 1, 2


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    f = build(tmp_path_factory.mktemp("rule"), "int table(uint64_t modes, uint64_t nzh) { return pk_table(modes, nzh); }").table
    f.argtypes = [ctypes.c_uint64, ctypes.c_uint64]
    return f


# (modes in 2^20, modes per row, the faster kernel)
@pytest.mark.parametrize("m,nzh,want", [
    (1.0, 2, MODES), (60.0, 2, MODES), (1.0, 17, MODES), (60.0, 25, MODES), (2.0, 33, MODES), (3.0, 37, MODES),
    (3.0, 50, ROWS), (2.0, 64, ROWS), (2.0, 65, MODES), (2.0, 100, ROWS), (1.0, 65, MODES), (1.0, 257, ROWS),
    (4.3, 33, MODES), (6.0, 41, LDS), (8.0, 65, MODES), (6.0, 80, LDS), (12.0, 33, LDS), (24.0, 27, MODES),
    (60.0, 65, LDS), (75.0, 769, LDS), (4.3, 769, LDS), (3.9, 769, ROWS)])
def test_faster_kernel(rule, m, nzh, want):
    assert rule(int(m * 2 ** 20), nzh) == want
