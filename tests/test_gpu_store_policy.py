"""Frames of a launch on both sides of the size up to which they are kept in
the memory-side cache (224 MiB of shifted probes and updates): only where they
are stored differs, so one batch equals the same batch in stages below that
size, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("S,scan,px,stage", [(128, (30, 30), 200, 512), (64, (60, 62), 160, 1024)])
def test_streamed_equals_kept(S, scan, px, stage):
    from py4dstem_amd import SingleslicePtychography
    from py4dstem_amd.synthetic import small_workload
    n = scan[0] * scan[1]
    print(f"[gpu] {n} frames of {S} px, one launch and stages of {stage}", flush=True)
    assert n * S * S * 16 > 224 << 20 > stage * S * S * 16
    w = small_workload(seed=9, scan=scan, S=S, object_px=px)
    out = []
    for st in (0, stage):
        p = SingleslicePtychography(datacube=w["datacube"], **w["init"])
        p.preprocess(**w["preprocess"])
        p.set_stage(st)
        np.random.seed(2)  # one batch: its order comes from the global generator
        out.append(p.reconstruct(**dict(w["reconstruct"], num_iter=2, max_batch_size=None, fix_probe=False)))
    a, b = out
    assert np.isfinite(a.object).all()
    assert np.array_equal(a.object, b.object) and np.array_equal(a.probe, b.probe)
    assert a.error_iterations == b.error_iterations
