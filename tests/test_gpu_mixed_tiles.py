"""Mixed-state scatters, one launch for all modes with the probe updated or
kept: wide tiles while a pixel meets few windows for the objects of all modes
together, the tiles of a single object otherwise.
Against the NumPy oracle with the bounds of the other mode launches (2e-5,
relative L2)."""

import pytest

from tests import test_gpu_mixed_batches as launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes,S,scan,px,batch,more", [
    (4, 64, (6, 6), 270, 20, {}),                       # 291,600 pixels, 1.1 windows: wide
    (4, 64, (6, 6), 270, None, dict(fix_probe=True)),   # 2.0 windows: wide
    (5, 32, (9, 9), 240, 64, dict(fix_probe=True)),     # 288,000 pixels, 1.1 windows: wide
    (4, 128, (13, 13), 270, None, dict(fix_probe=True)),  # 38 windows: a single object's
    (2, 128, (9, 9), 200, None, {}),                    # 80,000 pixels, 17 windows: a single object's
])
def test_mode_tiles_match_oracle(modes, S, scan, px, batch, more):
    launches.test_mode_launches_match_oracle(modes, S, scan, px, batch, more)
