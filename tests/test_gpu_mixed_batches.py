"""The launches that mixed-state probe modes share after the far-field pass
(scatter and probe sums, overlaps and probe steps) at one, three and four
modes, one-slot and remainder batches, and with the probe kept.  Against the
NumPy oracle, without orthogonalisation (its phase is a gauge): float32
rounding is a few 1e-7 per step, so two iterations stay below 2e-5 (relative
L2)."""

import numpy as np
import pytest
import scipy.ndimage

from oracle import OracleMixedstatePtychography
from tests.conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("modes,S,scan,px,batch,more", [
    (1, 32, (3, 3), 65, 1, {}),
    (3, 32, (9, 9), 96, 65, {}),
    (4, 64, (8, 9), 131, 70, {}),
    (3, 64, (6, 6), 120, None, dict(fix_probe=True)),
])
def test_mode_launches_match_oracle(modes, S, scan, px, batch, more):
    from py4dstem_amd import MixedstatePtychography
    from py4dstem_amd.synthetic import small_workload
    print(f"[gpu] mixed launches: {modes} modes of {S} px, batch {batch}", flush=True)
    w = small_workload(seed=7, scan=scan, S=S, object_px=px)
    rng = np.random.default_rng(13)
    init = np.exp(0.4j * scipy.ndimage.gaussian_filter(rng.standard_normal((px, px)), 3)).astype(np.complex64)
    recon = dict(w["reconstruct"], num_iter=2, max_batch_size=batch, fix_probe=False, seed_random=4,
                 orthogonalize_probe=False)
    recon.update(more)
    out = []
    for cls in (MixedstatePtychography, OracleMixedstatePtychography):
        p = cls(datacube=w["datacube"], num_probes=modes, **dict(w["init"], initial_object_guess=init.copy()))
        np.random.seed(31)  # the modes' phase ramps
        p.preprocess(**w["preprocess"])
        p._probe *= np.float32(0.8) ** np.arange(modes, dtype=np.float32)[:, None, None]
        p._probe_initial = p._probe.copy()
        if hasattr(p, "_probe_dev"):
            del p._probe_dev
        out.append(p.reconstruct(**recon))
    g, o = out
    errs = rel(np.array(g.error_iterations), np.array(o.error_iterations))
    print(f"[gpu] object {rel(g.object, o.object):.2e} probe {rel(np.asarray(g.probe), o.probe):.2e} "
          f"errors {errs:.2e}", flush=True)
    assert rel(g.object, o.object) < 2e-5
    assert rel(np.asarray(g.probe), o.probe) < 2e-5
    assert errs < 2e-5
