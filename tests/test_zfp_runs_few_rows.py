"""Packed fields with few rows to a plane, or short planes that are not whole 64-byte sectors, are stored row by row."""
import pytest

MIB = 1 << 20


@pytest.mark.parametrize("nx,ny,mb,want", [
    (28, 1, 150, 0), (4, 1, 20, 0), (3, 1, 100, 0), (15, 1, 20, 0), (35, 1, 20, 0), (16, 1, 100, 0),       # one row
    (100, 2, 150, 0), (28, 2, 20, 0), (14, 2, 100, 0), (35, 2, 20, 0), (3, 2, 100, 1), (7, 2, 20, 1), (8, 2, 100, 2), (16, 2, 20, 2),
    (4, 2, 20, 0), (4, 7, 100, 0), (8, 7, 100, 0), (12, 13, 100, 0), (28, 9, 20, 0), (36, 7, 20, 0),        # short planes
    (28, 10, 100, 2), (20, 13, 20, 2), (100, 3, 100, 2), (8, 6, 100, 2), (16, 3, 100, 2), (4, 4, 20, 2), (12, 4, 100, 2),
    (7, 3, 20, 1), (35, 3, 20, 2), (15, 5, 100, 1)])
def test_route(nx, ny, mb, want):
    from cswap_amd import _lib

    assert _lib.lib().cswap_test_zfp_decode_runs(nx, ny, mb * MIB // (4 * nx * ny), 0, 0, 0) == want
