"""The scatter's tile by windows per pixel: up to 64 x 4096 object pixels, 25
times the square of the object's share of these, batches on either side of the
rule.  Bit for bit against np.bincount (chi = 1 makes the float32 products
exact), every entry of the tile maxima written, and a batch whose last stage
takes the other tile than the first equal to the whole batch."""

import numpy as np
import pytest

from oracle import ptycho_oracle as po
from tests.test_gpu_pipeline import _run, _same

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# object, then the batches up to which a pixel meets few windows and beyond
@pytest.mark.parametrize("S,shape,batches", [
    (32, (130, 131), (1, 2)), (32, (257, 255), (99, 102)), (64, (300, 301), (65, 66)),
    (64, (509, 515), (1599, 1625)), (128, (401, 399), (90, 92)), (256, (300, 520), (21, 23))])
def test_few_and_many_windows(S, shape, batches):
    from py4dstem_amd import _lib, kernels as K
    from py4dstem_amd._lib import ptr, stream_handle
    share = shape[0] * shape[1] / (64 * 4096)
    few = [B * S * S <= 25 * share ** 2 * shape[0] * shape[1] for B in batches]
    assert few == [True, False]
    for B in batches:
        print(f"[gpu] scatter S={S} object {shape} B={B}", flush=True)
        rng = np.random.default_rng(S + B)
        pos = (rng.uniform(-0.5, 1.5, (B, 2)) * shape).astype(np.float32)
        order = rng.permutation(B).astype(np.int32)
        ps = (rng.standard_normal((B, S, S), np.float32)
              + 1j * rng.standard_normal((B, S, S), np.float32)).astype(np.complex64)
        psd, posd, ordd = (torch.from_numpy(a).cuda() for a in (ps, pos, order))
        chi = torch.ones_like(psd)
        grad = torch.empty(shape, dtype=torch.complex64, device="cuda")
        spsum = torch.empty(shape, dtype=torch.float32, device="cuda")
        tmax = torch.full((K.num_tiles(*shape),), float("nan"), device="cuda")
        _lib.call("pty_scatter_patches", ptr(psd), ptr(chi), ptr(posd), B, ptr(ordd), B, S,
                  *shape, ptr(grad), ptr(spsum), ptr(tmax), stream_handle())
        np.testing.assert_array_equal(grad.cpu().numpy(),
                                      po.scatter_bincount(np.conj(ps), pos[order], (S, S), shape))
        sq = (ps.real * ps.real + ps.imag * ps.imag).astype(np.float32)
        np.testing.assert_array_equal(spsum.cpu().numpy(),
                                      po.scatter_bincount(sq, pos[order], (S, S), shape))
        t = tmax.cpu().numpy()
        assert np.isfinite(t).all() and t.max() == spsum.max().item() and t.min() >= 0


@pytest.mark.parametrize("fix_probe", [False, True])
@pytest.mark.parametrize("pipeline", [False, True])
def test_stages_of_either_tile_equal_the_whole_batch(pipeline, fix_probe):
    from py4dstem_amd.synthetic import small_workload
    print(f"[gpu] stages of 128 and 16 slots, pipeline {pipeline}, fixed probe {fix_probe}", flush=True)
    w = small_workload(seed=17, scan=(12, 12), S=64, object_px=300)
    recon = dict(num_iter=2, max_batch_size=144, seed_random=3, fix_probe=fix_probe)
    _same(_run(w, 0, False, **recon), _run(w, 128, pipeline, **recon))
