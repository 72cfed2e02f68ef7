"""256 px frames: positions per fused launch and the second stream are
performance settings, so object, probe and errors equal the whole batch's bit
for bit, and the errors are the ones that the batch entry point forms, which
has no room for the row groups' partial sums.  One slot's amplitudes carry
factors of twelve decades and outweigh the others' error beyond a float64's
last bit (its sum is about 1e15, ulp 0.1; the others' below 1e-14): it rounds, and
alone makes the iteration's error."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

S, SHAPE, N = 256, (300, 290), 128


def _run(data, stage, pipeline):
    from py4dstem_amd import kernels as K
    obj, probe, pos, amps = data
    obj, probe = obj.clone(), probe.clone()
    q = K.PtyGdParams()
    q.num_iter, q.max_batch, q.step_size, q.normalization_min = 2, N, 0.5, 1.0
    q.fix_probe_com, q.stage, q.pipeline = 1, stage, int(pipeline)
    problem = K.make_problem(obj, probe, pos, amps, None, 1.0 / N)
    ws = torch.empty(K.gd_workspace_bytes(problem, q), dtype=torch.uint8, device=obj.device)
    orders = torch.arange(N, dtype=torch.int32, device=obj.device).repeat(2)
    errors = torch.empty(2, dtype=torch.float64, device=obj.device)
    K.gd_run(problem, q, orders, errors, ws)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (obj, probe, errors)]


@pytest.mark.parametrize("slot", [0, 13, 63, 64, 90, 127])
def test_stages_and_errors(slot):
    from py4dstem_amd import kernels as K
    print(f"[gpu] 256 px, {N} slots, stages of 64, slot {slot}", flush=True)
    rng = np.random.default_rng(slot)
    amps = np.full((N, S, S), 1e-12, np.float32)
    amps[slot] = 10.0 ** rng.uniform(-6, 6, (S, S))
    z = rng.standard_normal((S, S)) + 1j * rng.standard_normal((S, S))
    data = [torch.from_numpy(a).cuda() for a in (
        np.exp(0.3j * rng.random(SHAPE)).astype(np.complex64), (1e-13 * z).astype(np.complex64),
        (rng.random((N, 2)) * SHAPE).astype(np.float32), amps)]
    whole = _run(data, 0, False)
    for pipeline in (False, True):
        for x, y in zip(whole, _run(data, 64, pipeline)):
            np.testing.assert_array_equal(x, y)
    order = torch.tensor([slot], dtype=torch.int32, device="cuda")
    _, _, err = K.forward_adjoint(K.probe_spectrum(data[1]), data[0], data[2], data[3], order)
    assert np.isfinite(whole[2]).all() and whole[2][0] == float(err[0])
