"""The scatter's phases on the host emulator, 64- and 256-pixel tiles beside the
kernel that serves frames of any size: hit lists around a chunk (16 and 4 hits)
and around a list's 1024 slots, waves without candidates, stages, and objects
whose last tile row and column are cut.  No LDS race, no access out of range,
every tile maximum written, all three bit for bit np.bincount in batch order."""

import numpy as np
import pytest

from oracle import ptycho_oracle as po
from tests.conftest import cptr, emu  # noqa: F401


def _case(S, shape, B, spread):
    rng = np.random.default_rng(B + shape[0])
    centre = np.array(shape) / 2
    pos = (centre + spread * rng.uniform(-1, 1, (B, 2)) * shape).astype(np.float32)
    order = rng.permutation(B).astype(np.int32)
    ps = (rng.standard_normal((B, S, S)) + 1j * rng.standard_normal((B, S, S))).astype(np.complex64)
    sq = (ps.real * ps.real + ps.imag * ps.imag).astype(np.float32)
    return pos, order, ps, (po.scatter_bincount(np.conj(ps), pos[order], (S, S), shape),
                            po.scatter_bincount(sq, pos[order], (S, S), shape))


def _outputs(emu, shape):  # noqa: F811
    return (np.zeros(shape, np.complex64), np.zeros(shape, np.float32),
            np.zeros(emu.emu_gather_num_tiles(*shape), np.float32))


@pytest.mark.parametrize("shape", [(32, 32), (35, 49)])
@pytest.mark.parametrize("B", [1, 3, 4, 5, 15, 16, 17, 255, 256, 257, 1023, 1024, 1025, 1044, 2049])
def test_list_lengths(emu, shape, B):  # noqa: F811
    S = 32
    # every window meets every tile of the smaller object
    pos, order, ps, (grad_ref, spsum_ref) = _case(S, shape, B, 0.0 if B % 2 else 0.3)
    grad, spsum, tmax = _outputs(emu, shape)
    emu.emu_reset()
    emu.emu_gather(S, cptr(ps), cptr(np.ones_like(ps)), cptr(pos), B, cptr(order), B, *shape,
                   cptr(grad), cptr(spsum), cptr(tmax))
    assert emu.emu_violations() == 0, emu.emu_first_violation()
    np.testing.assert_array_equal(grad, grad_ref)
    np.testing.assert_array_equal(spsum, spsum_ref)


@pytest.mark.parametrize("B,stage", [(70, 64), (9, 1), (1300, 1088)])
def test_stages(emu, B, stage):  # noqa: F811
    S, shape = 32, (37, 70)
    pos, order, ps, (grad_ref, spsum_ref) = _case(S, shape, B, 0.9)
    grad, spsum, tmax = _outputs(emu, shape)
    run = np.zeros(shape + (3,), np.float64)
    emu.emu_reset()
    emu.emu_gather_staged(S, cptr(ps), cptr(np.ones_like(ps)), cptr(pos), B, cptr(order), B, stage,
                          *shape, cptr(grad), cptr(spsum), cptr(tmax), cptr(run))
    assert emu.emu_violations() == 0, emu.emu_first_violation()
    np.testing.assert_array_equal(grad, grad_ref)
    np.testing.assert_array_equal(spsum, spsum_ref)
