"""Gaussian smoothing of objects above 2^20 pixels: complex, pure phase, and a
potential inside a run whose step is zero.  Against scipy in float64 of the
same values below one: each axis rounds to float32 (6e-8), so results are
within 2e-7, the phase's angle and exponential another two ulps off: 5e-7."""

import numpy as np
import pytest
import scipy.ndimage

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(1025, 1024), (1031, 1200), (40, 30000)]


@pytest.mark.parametrize("shape", SHAPES)
def test_complex_and_phase(shape):
    from py4dstem_amd import kernels as K
    print(f"[gpu] gaussian of {shape}", flush=True)
    rng = np.random.default_rng(shape[0])
    z = (0.7 * np.exp(1j * rng.uniform(-1, 1, shape))).astype(np.complex64)
    got = K.object_gaussian(torch.from_numpy(z.copy()).cuda(), 1.3).cpu().numpy()
    ref = scipy.ndimage.gaussian_filter(z.astype(np.complex128), 1.3)
    assert np.abs(got - ref).max() <= 2e-7
    got = K.object_gaussian(torch.from_numpy(z.copy()).cuda(), 1.3, pure_phase_object=True).cpu().numpy()
    ref = np.exp(1j * scipy.ndimage.gaussian_filter(np.angle(z.astype(np.complex128)), 1.3))
    assert np.abs(got - ref).max() <= 5e-7


@pytest.mark.parametrize("shape", SHAPES)
def test_potential(shape):
    from ctypes import c_void_p

    from py4dstem_amd import kernels as K
    print(f"[gpu] gaussian of a potential of {shape}", flush=True)
    rng = np.random.default_rng(shape[1])
    v = rng.uniform(0, 1, shape).astype(np.float32)
    S, N = 32, 2
    obj = torch.from_numpy(v.copy()).cuda()
    probe = torch.ones((S, S), dtype=torch.complex64, device="cuda")
    pos = torch.tensor([[20.0, 20.0], [24.0, 29.0]], device="cuda")
    amps = torch.ones((N, S, S), device="cuda")
    w, r = K.gaussian_kernel1d(1.3)
    wd = torch.from_numpy(w).cuda()
    q = K.PtyGdParams()
    q.num_iter, q.max_batch, q.step_size, q.normalization_min, q.fix_probe = 1, N, 0.0, 1.0, 1
    q.gaussian_weights, q.gaussian_radius = c_void_p(wd.data_ptr()), r
    problem = K.make_problem(obj, probe, pos, amps, None, 1.0)
    ws = torch.empty(K.gd_workspace_bytes(problem, q), dtype=torch.uint8, device="cuda")
    orders = torch.arange(N, dtype=torch.int32, device="cuda")
    errors = torch.empty(1, dtype=torch.float64, device="cuda")
    K.gd_run(problem, q, orders, errors, ws)
    ref = scipy.ndimage.gaussian_filter(v.astype(np.float64), 1.3)
    assert np.abs(obj.cpu().numpy() - ref).max() <= 2e-7
