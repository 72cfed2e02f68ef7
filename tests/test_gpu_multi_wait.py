"""MultiPtychography.reconstruct's native call with use_graph returns after its
work is complete, and leaves the same results without."""

import numpy as np
import pytest

from tests.test_gpu_multi import _assert_same, _make

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_use_graph_waits_for_completion():
    from py4dstem_amd.multi import MultiPtychography
    from py4dstem_amd.synthetic import small_workload
    print("[gpu] batched run: completion on return", flush=True)
    w = small_workload(seed=30, scan=(16, 16), S=64, object_px=160)
    out = []
    for use_graph in (True, False):
        items = [_make(w), _make(w)]
        m = MultiPtychography(items)
        np.random.seed(3)
        runs = m._runs(6, [dict(max_batch_size=64, seed_random=i, reset=True) for i in range(2)])
        torch.cuda.synchronize()
        m.run_prepared(runs, 6, use_graph)
        if use_graph:
            assert torch.cuda.current_stream().query()
        torch.cuda.synchronize()
        for p, run in zip(items, runs):
            p._finish_run(run)
        out.append([(p.object, p.probe, p.error_iterations) for p in items])
    _assert_same(*out)
