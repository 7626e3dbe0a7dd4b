"""What smk_pk_table refuses before it looks at any buffer."""
import ctypes

import pytest

from saclaymocks_amd import _lib, pk


@pytest.mark.parametrize("shape,refused", [((8192, 8192, 8192), True), ((1 << 20, 1 << 19, 1), True),
                                           ((1, 1 << 20, (1 << 19) + 1), True), ((0, 8192, 8192), False)])
def test_tables_of_more_than_2_to_39_modes(shape, refused):
    sp = pk.SmkPkSpline()
    one = ctypes.c_void_p(256)   # never read
    sp.x = sp.c = sp.guess = 256
    sp.n_int, sp.n_guess, sp.g_lo, sp.g_step = 4, 4, 0.0, 1.0
    rc = _lib.lib().smk_pk_table(ctypes.byref(sp), one, one, one, *shape, ctypes.c_float(1.0), one, None)
    assert rc == (-1 if refused else 0), rc
    if refused:
        assert b"too large" in _lib.lib().smk_last_error()
