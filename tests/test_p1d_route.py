"""Which kernel the rows of the missing 1D power take, as measured on both
sides of the lines."""
import pytest

from route_rules import build


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return build(tmp_path_factory.mktemp("rule"),
                 "int fast(int model, int n_par, int n_perp) { return p1d_fast(model, n_par, n_perp); }\n"
                 "int cut(int n_par, int n_perp) { return p1d_cut_rows(n_par, n_perp); }")


@pytest.mark.parametrize("model,n_par,n_perp,fast", [
    (1, 20000, 20000, 1), (1, 20000, 400, 1), (1, 20000, 200, 0), (1, 20000, 50, 0), (1, 900, 900, 1), (1, 1024, 600, 0),
    (1, 2000, 400, 0), (1, 2048, 900, 1), (1, 512, 20000, 0), (1, 1, 20000, 0), (1, 600, 2500, 1),
    (0, 20000, 20000, 1), (0, 20000, 600, 0), (0, 20000, 50, 0), (0, 2048, 2500, 1), (0, 768, 2500, 0),
    (0, 768, 10000, 1), (0, 200, 10000, 0), (0, 200, 20000, 1), (2, 20000, 20000, 0)])
def test_sum_of_fewer_instructions(rules, model, n_par, n_perp, fast):
    assert rules.fast(model, n_par, n_perp) == fast


@pytest.mark.parametrize("n_par,n_perp,rows", [(20000, 20000, 8), (8192, 300, 8), (8192, 50, 2), (4096, 100, 1),
                                               (1, 20000, 1), (300, 900, 0), (300, 5000, 1), (600, 600, 1)])
def test_rows_per_block_of_the_cut(rules, n_par, n_perp, rows):
    assert rules.cut(n_par, n_perp) == rows
