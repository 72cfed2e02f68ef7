"""Loss and gradients over an object of more than 2^28 pixels, which needs the
top bit of the 32-bit byte offset: those of the same windows in an object with
fewer columns, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_objects_up_to_the_byte_range():
    from py4dstem_amd.autograd import ptychographic_loss
    S, rows, cols, B = 64, 16500, 256, 5
    print(f"[gpu] loss, {rows}^2 object", flush=True)
    rng = np.random.default_rng(7)

    def z(*n):
        return torch.from_numpy((rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)).cuda()

    narrow, probe = z(rows, cols), z(S, S)
    wide = torch.zeros((rows, rows), dtype=torch.complex64, device="cuda")
    wide[:, :cols] = narrow
    assert 2 ** 28 < wide.numel() < 2 ** 29
    pos = np.stack([[40.2, rows / 2, rows - 200.3, rows - 40.4, rows - 3.1],
                    rng.uniform(60, 180, B)], 1).astype(np.float32)
    pos = torch.from_numpy(pos).cuda()
    amps = torch.from_numpy(rng.random((B, S, S), np.float32) * 50).cuda()
    out = []
    for obj in (narrow, wide):
        o, p = obj.requires_grad_(), probe.clone().requires_grad_()
        loss = ptychographic_loss(o, p, pos, amps)
        go, gp = torch.autograd.grad(loss, (o, p))
        out.append([t.detach().cpu().numpy() for t in (loss, go[:, :cols], gp)])
        assert not go[:, cols:].any()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
