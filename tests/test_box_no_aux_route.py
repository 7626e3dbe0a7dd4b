"""The spectral pass's variant with an aux field and without, as measured: those
that keep a second register tile are not taken where it would stay empty."""
import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return build(tmp_path_factory.mktemp("rule"),
                 "int spectral(int n, int aux) { return box_strided(SMK_PASS_X_SPECTRAL, n, 512, 512, aux); }").spectral


@pytest.mark.parametrize("n,with_aux,without", [(512, 16, 0), (1024, 14, 0), (2048, 14, 0), (640, 10, 10), (1280, 12, 12),
                                                (2560, 1, 1), (768, 3, 3), (256, 0, 0), (900, 0, 0)])
def test_spectral(rule, n, with_aux, without):
    assert (rule(n, 1), rule(n, 0)) == (with_aux, without)
