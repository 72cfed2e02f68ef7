"""Batched runs choose the scatter's tile and the probe sums' pixels per lane
by all problems together, single runs by their own object and batch: results
stay bitwise those of the single runs on either side of both rules (25 windows
a pixel times the objects' share of 64 x 4096 pixels, squared below one; 1024
work groups at one pixel per lane), with short last stages and with fixed
probes between updated ones."""

import numpy as np
import pytest

from tests.test_gpu_multi import _assert_same, _make

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (frame, object, scan, batch, fixed probe) of each problem; stage
CASES = {
    # 54,500 pixels, 34 windows a pixel, 512 work groups
    "small-tiles-one-pixel": ([(128, 160, 7, 49, False), (128, 170, 8, 64, False)], 0),
    # 289,600 pixels, 8.9 windows a pixel, 576 work groups
    "wide-tiles-one-pixel": ([(128, 300, 6, 36, False), (128, 300, 7, 49, True),
                              (128, 300, 8, 64, False), (64, 140, 8, 30, False)], 0),
    # 178,601 pixels, 28 windows a pixel, 1,728 work groups
    "small-tiles-four-pixels": ([(128, 300, 9, 81, False), (128, 261, 11, 121, False),
                                 (64, 64, 12, 144, False), (128, 128, 9, 70, False)], 0),
    # 310,000 pixels, 17 windows a pixel, 1,152 work groups, stages of 128 with remainders
    "wide-tiles-four-pixels-staged": ([(128, 300, 9, 81, False), (128, 300, 12, 144, False),
                                       (64, 200, 12, 130, False), (128, 300, 9, 81, True)], 128),
}


@pytest.mark.parametrize("case", list(CASES))
def test_batched_tiles_equal_single_runs(case):
    from py4dstem_amd.multi import MultiPtychography
    from py4dstem_amd.synthetic import small_workload
    print(f"[gpu] batched tiles: {case}", flush=True)
    problems, stage = CASES[case]
    ws, kws = [], []
    for i, (S, px, n, batch, fix) in enumerate(problems):
        w = small_workload(seed=20 + i, scan=(n, n), S=S, object_px=px)
        guess = np.exp(0.3j * np.random.default_rng(i).random((px, px))).astype(np.complex64)
        w["init"] = dict(w["init"], initial_object_guess=guess)
        ws.append(w)
        kws.append(dict(max_batch_size=batch, fix_probe=fix, seed_random=i, step_size=0.5,
                        normalization_min=1, reset=True))
    single, items = [], [_make(w) for w in ws]
    for w, kw in zip(ws, kws):
        p = _make(w)
        p.set_stage(stage)
        p.reconstruct(num_iter=2, progress_bar=False, **kw)
        single.append((p.object.copy(), p.probe.copy(), list(p.error_iterations)))
    for p in items:
        p.set_stage(stage)
    MultiPtychography(items).reconstruct(2, kws)
    _assert_same([(p.object, p.probe, p.error_iterations) for p in items], single)
