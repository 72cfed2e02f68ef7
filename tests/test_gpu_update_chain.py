"""Object and probe steps after the scatter, and the end of an iteration, at
the sizes where their launches change: one and several 64-slot probe chunks
with a remainder, one or four probe pixels per lane (S * S / 64 * chunks up to
1024 work groups or beyond), the probe transform in one work group (32, 64 px)
or split over 16 (128 px), runs that end or continue after the recentring, and
a probe that is not recentred.  Against the NumPy oracle: float32 rounding of
the transforms is a few 1e-7 per step, so two iterations stay below 1e-5
(relative L2)."""

import numpy as np
import pytest
import scipy.ndimage

from oracle import OracleSingleslicePtychography
from tests.conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = {
    # S, scan, object, batch, reconstruct keywords
    "32px-one-slot-batches": (32, (2, 2), 64, 1, {}),
    "32px-chunk-remainder": (32, (9, 9), 96, 65, {}),
    "64px-full-batch": (64, (9, 9), 128, None, {}),
    "64px-no-recentring": (64, (8, 9), 131, 70, dict(fix_probe_com=False)),
    "64px-pure-phase-shrink": (64, (6, 6), 120, 18, dict(pure_phase_object=True, shrinkage_rad=0.01)),
    "128px-one-pixel-per-lane": (128, (16, 16), 208, 256, {}),
    "128px-four-pixels-per-lane": (128, (16, 17), 208, 257, {}),
    "128px-fixed-probe": (128, (5, 5), 160, 13, dict(fix_probe=True)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_updates_match_oracle(case):
    from py4dstem_amd import SingleslicePtychography
    from py4dstem_amd.synthetic import small_workload
    print(f"[gpu] update chain: {case}", flush=True)
    S, scan, px, batch, more = CASES[case]
    w = small_workload(seed=5, scan=scan, S=S, object_px=px)
    rng = np.random.default_rng(11)
    init = np.exp(0.4j * scipy.ndimage.gaussian_filter(rng.standard_normal((px, px)), 3)
                  / 0.05 * 0.05).astype(np.complex64) * np.float32(0.95)
    recon = dict(w["reconstruct"], num_iter=2, max_batch_size=batch, fix_probe=False, seed_random=4)
    recon.update(more)
    out = []
    for cls in (SingleslicePtychography, OracleSingleslicePtychography):
        p = cls(datacube=w["datacube"], **dict(w["init"], initial_object_guess=init.copy()))
        p.preprocess(**w["preprocess"])
        rc = dict(recon)
        if cls is OracleSingleslicePtychography:
            rc.pop("progress_bar", None)
        out.append(p.reconstruct(**rc))
    g, o = out
    errs = rel(np.array(g.error_iterations), np.array(o.error_iterations))
    print(f"[gpu] object {rel(g.object, o.object):.2e} probe {rel(g.probe, o.probe):.2e} "
          f"errors {errs:.2e}", flush=True)
    assert rel(g.object, o.object) < 1e-5
    assert rel(g.probe, o.probe) < 1e-5
    assert errs < 1e-5
