"""Deterministic scatter: both tile shapes, both hit-list lengths and the
64-bit fallback, bit for bit against np.bincount in batch order (chi = 1 makes
every float32 product exact, so the float64 sums must match exactly)."""

import numpy as np
import pytest

from oracle import ptycho_oracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    from py4dstem_amd import _lib
    _lib.load()
    return torch.device("cuda", 0)


# 64-pixel tiles (4 x 16) up to 2^18 object pixels, 256-pixel tiles (8 x 32)
# beyond; edges that cut tiles, one full row of tiles, thin objects; batches
# below one chunk of hits and across the 1024-slot hit lists
@pytest.mark.parametrize("S,shape,B", [
    (32, (32, 32), 1), (32, (33, 47), 3), (32, (101, 83), 300), (32, (128, 128), 1025),
    (64, (65, 64), 17), (64, (71, 130), 1500), (128, (128, 131), 70),
    (64, (512, 512), 400), (64, (513, 512), 400), (32, (67, 4096), 700), (128, (601, 577), 90),
    (256, (258, 300), 9), (256, (700, 519), 12)])
def test_scatter_equals_bincount(dev, S, shape, B):
    from py4dstem_amd import kernels as K
    say(f"scatter S={S} object {shape} B={B}")
    rng = np.random.default_rng(S + shape[0] + B)
    # windows anywhere, also around both object edges
    pos = np.stack([rng.uniform(-S, shape[0] + S, B), rng.uniform(-S, shape[1] + S, B)],
                   1).astype(np.float32)
    order = rng.permutation(B).astype(np.int32)
    ps = (rng.standard_normal((B, S, S), np.float32)
          + 1j * rng.standard_normal((B, S, S), np.float32)).astype(np.complex64)
    psd = torch.from_numpy(ps).to(dev)
    grad, spsum, tmax = K.scatter(psd, torch.ones_like(psd), torch.from_numpy(pos).to(dev),
                                  torch.from_numpy(order).to(dev), shape)
    np.testing.assert_array_equal(grad.cpu().numpy(),
                                  po.scatter_bincount(np.conj(ps), pos[order], (S, S), shape))
    sq = (ps.real * ps.real + ps.imag * ps.imag).astype(np.float32)
    np.testing.assert_array_equal(spsum.cpu().numpy(),
                                  po.scatter_bincount(sq, pos[order], (S, S), shape))
    assert tmax.numel() == K.num_tiles(*shape)
    assert tmax.max().item() == spsum.max().item()


def test_scatter_outside_a_window_ignores_its_values(dev):
    """Pixels a window does not cover take nothing from it, also where the
    frame holds infinities and NaN."""
    from py4dstem_amd import kernels as K
    say("scatter of non-finite frames")
    S, shape = 32, (96, 96)
    ps = torch.ones((2, S, S), dtype=torch.complex64, device=dev)
    ps[1] = complex(float("inf"), float("nan"))
    pos = torch.tensor([[20.0, 20.0], [70.0, 70.0]], device=dev)
    order = torch.arange(2, dtype=torch.int32, device=dev)
    grad, spsum, _ = K.scatter(ps, torch.ones_like(ps), pos, order, shape)
    want = np.zeros(shape, np.float32)
    want[4:36, 4:36] = 1.0
    bad = np.zeros(shape, bool)
    bad[54:86, 54:86] = True
    np.testing.assert_array_equal(spsum.cpu().numpy()[~bad], want[~bad])
    np.testing.assert_array_equal(grad.cpu().numpy().real[~bad], want[~bad])
    assert not np.isfinite(spsum.cpu().numpy()[bad]).any()


@pytest.mark.parametrize("shape", [(300, 320), (640, 650)])
def test_scatter_beyond_the_buffer_range(dev, shape):
    """Frames of more than 2 GiB take the kernel with 64-bit offsets: frames
    of zeros add nothing, so the sums are those of the filled frames alone."""
    from py4dstem_amd import kernels as K
    say(f"scatter of 2.1 GiB of frames, object {shape}")
    S, B = 128, 16500
    rng = np.random.default_rng(7)
    pos = torch.from_numpy(np.stack([rng.uniform(0, shape[0], B), rng.uniform(0, shape[1], B)],
                                    1).astype(np.float32)).to(dev)
    ps = torch.zeros((B, S, S), dtype=torch.complex64, device=dev)
    chi = torch.zeros_like(ps)
    slots = torch.from_numpy(np.sort(rng.permutation(B)[:40])).to(dev)
    ps[slots] = torch.randn((40, S, S), dtype=torch.complex64, device=dev)
    chi[slots] = torch.randn((40, S, S), dtype=torch.complex64, device=dev)
    order = torch.from_numpy(rng.permutation(B).astype(np.int32)).to(dev)
    grad, spsum, tmax = K.scatter(ps, chi, pos, order, shape)
    few = K.scatter(ps[slots].contiguous(), chi[slots].contiguous(), pos,
                    order[slots].contiguous(), shape)
    assert torch.equal(grad, few[0]) and torch.equal(spsum, few[1])
    assert tmax.max().item() == spsum.max().item() and tmax.min().item() >= 0.0
