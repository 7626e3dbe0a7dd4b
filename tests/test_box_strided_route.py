"""The variants of the x and y passes that a plan starts with: the tuned ones from
the size on where they were measured to be the faster."""
import pytest

from route_rules import build

Y_FWD, X_SPECTRAL, Y_INV, X_FWD, X_INV = 1, 2, 3, 5, 6


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return build(tmp_path_factory.mktemp("rule"), "int variant(int kind, int nx, int ny, int nz) "
                 "{ return box_strided(kind, nx, ny, nz, true); }").variant


@pytest.mark.parametrize("kind,shape,want", [
    (Y_FWD, (250, 768, 300), 0), (Y_FWD, (400, 768, 400), 17), (Y_INV, (100, 768, 100), 0), (Y_INV, (200, 768, 200), 0),
    (Y_INV, (768, 768, 768), 18), (X_FWD, (768, 100, 100), 0), (X_FWD, (768, 256, 256), 17), (X_FWD, (640, 32, 32), 0),
    (X_FWD, (640, 400, 400), 17), (X_INV, (640, 100, 200), 17), (Y_FWD, (200, 512, 200), 0), (X_INV, (512, 160, 160), 0),
    (X_INV, (512, 512, 512), 17), (X_SPECTRAL, (384, 100, 100), 0), (X_SPECTRAL, (384, 512, 512), 17),
    (X_SPECTRAL, (768, 32, 32), 0), (X_SPECTRAL, (768, 128, 128), 3), (X_SPECTRAL, (1536, 16, 16), 0),
    (Y_INV, (200, 1536, 200), 0), (Y_INV, (512, 1536, 512), 6), (Y_INV, (64, 2048, 64), 0), (Y_INV, (256, 2048, 512), 3),
    (Y_FWD, (64, 1024, 64), 0), (Y_FWD, (400, 1024, 400), 3)])
def test_split_exchange(rule, kind, shape, want):
    assert rule(kind, *shape) == want


@pytest.mark.parametrize("kind,shape,want", [
    (Y_FWD, (16, 1280, 16), 6), (X_FWD, (1280, 16, 16), 6), (Y_INV, (16, 640, 16), 6), (X_SPECTRAL, (640, 16, 16), 10),
    (X_SPECTRAL, (512, 16, 16), 16), (X_SPECTRAL, (1024, 16, 16), 14), (X_SPECTRAL, (1280, 16, 16), 12),
    (X_SPECTRAL, (2560, 16, 16), 1), (X_SPECTRAL, (2560, 1280, 768), 1), (Y_FWD, (2560, 1280, 768), 6),
    (Y_FWD, (900, 900, 900), 0), (X_SPECTRAL, (256, 256, 256), 0), (Y_INV, (2560, 2560, 1536), 0)])
def test_at_any_size(rule, kind, shape, want):
    assert rule(kind, *shape) == want
