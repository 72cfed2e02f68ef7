"""Position correction of one batch over an object of more than 2^29 pixels
(4.3 GiB, beyond a 32-bit byte offset): the same windows of an object with
fewer columns give the same sums and positions, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ROWS, COLS = 24000, 256


@pytest.fixture(scope="module")
def objects():
    rng = np.random.default_rng(1)
    z = rng.standard_normal((ROWS, COLS)) + 1j * rng.standard_normal((ROWS, COLS))
    narrow = torch.from_numpy(z.astype(np.complex64)).cuda()
    wide = torch.zeros((ROWS, ROWS), dtype=torch.complex64, device="cuda")
    wide[:, :COLS] = narrow
    assert wide.numel() > 2 ** 29
    return narrow, wide


@pytest.mark.parametrize("S", [32, 64, 128])
def test_objects_beyond_32_bit_offsets(objects, S):
    from py4dstem_amd import kernels as K
    print(f"[gpu] position correction, {S} px frames, {ROWS}^2 object", flush=True)
    rng = np.random.default_rng(S)
    B = 6

    def z():
        a = rng.standard_normal((B, S, S)) + 1j * rng.standard_normal((B, S, S))
        return torch.from_numpy(a.astype(np.complex64)).cuda()

    ps, far = z(), z()
    amps = torch.from_numpy(rng.random((B, S, S), np.float32)).cuda()
    # the first, the last rows and what wraps between them; columns away from
    # either object's edge
    rows = [200.3, ROWS / 2 + 0.4, ROWS - 300.6, ROWS - 80.1, ROWS - 20.2, 3.7]
    pos = np.stack([rows, 100 + 50 * rng.random(B)], 1).astype(np.float32)
    order = torch.arange(B, dtype=torch.int32, device="cuda")
    out = []
    for obj in objects:
        p = torch.from_numpy(pos.copy()).cuda()
        sums = torch.zeros((B, 5), dtype=torch.float64, device="cuda")
        K.position_correction(K.position_params(p, p.clone(), 0.5), ps, far, obj, amps, order, sums)
        out.append((sums.cpu().numpy(), p.cpu().numpy()))
    assert np.isfinite(out[0][0]).all() and (out[0][0] != 0).all()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
