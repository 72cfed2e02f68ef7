"""The probe step over objects with fewer rows or columns than the frame, down
to half of it, and one pixel to either side of the frame: a frame pixel's
object index is its offset from the rounded position modulo the object, also
where that wraps more than once.  Against NumPy in complex128.  The kernel
rounds the products to float32 and adds in float64, then forms the step in
float32: a few times 6e-8 in all, so 1e-6 (relative L2) bounds it."""

import numpy as np
import pytest

from tests.conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _reference(probe, chi, obj, pos, step, nmin):
    S = probe.shape[0]
    f = np.fft.fftfreq(S, 1 / S).astype(int)
    num, den = np.zeros((S, S), complex), np.zeros((S, S))
    for p, c in zip(np.rint(pos).astype(int), chi.astype(complex)):
        o = obj.astype(complex)[np.ix_((p[0] + f) % obj.shape[0], (p[1] + f) % obj.shape[1])]
        num += o.conj() * c
        den += np.abs(o) ** 2
    return probe + step * num / np.sqrt(1e-16 + ((1 - nmin) * den) ** 2 + (nmin * den.max()) ** 2)


@pytest.mark.parametrize("S,shape,B", [
    (32, (16, 33), 3), (32, (31, 32), 70), (64, (32, 32), 1), (64, (63, 65), 65),
    (128, (64, 127), 66), (128, (100, 96), 5), (128, (128, 129), 64), (256, (130, 255), 2)])
def test_probe_update_wraps_small_objects(S, shape, B):
    from py4dstem_amd import kernels as K
    print(f"[gpu] probe update S={S} object {shape}, {B} slots", flush=True)
    rng = np.random.default_rng(S + B)

    def z(*n):
        return (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)

    probe, chi, obj = z(S, S), z(B, S, S), z(*shape)
    pos = (rng.uniform(-0.5, 1.5, (B, 2)) * shape).astype(np.float32)
    dev = [torch.from_numpy(a).cuda() for a in
           (probe.copy(), chi, obj, pos, np.arange(B, dtype=np.int32))]
    got = K.probe_update(*dev, 0.5, 0.3).cpu().numpy()
    err = rel(got, _reference(probe, chi, obj, pos, 0.5, np.float64(np.float32(0.3))))
    print(f"[gpu] rel {err:.2e}", flush=True)
    assert err < 1e-6
