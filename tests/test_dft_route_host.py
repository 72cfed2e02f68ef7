"""The Butterworth filter's DFT products fit the grid and LDS of the tiles they
are given: rows / 16 (or 32) at most 65,536, at most 8192 roots in LDS."""

import pytest

from tests.conftest import emu  # noqa: F401


@pytest.mark.parametrize("M,n,lds", [
    (1, 1, 1), (284, 272, 1), (8192, 8192, 1), (8193, 8193, 0), (5, 8193, 0),
    (1 << 20, 32, 1), ((1 << 20) + 1, 32, 0), (1 << 21, 1, 0), (1 << 21, 8192, 0)])
def test_tiles_fit_the_grid(emu, M, n, lds):  # noqa: F811
    assert emu.emu_dft_in_lds(M, n) == lds
    assert -(-M // (16 if lds else 32)) <= 65536
