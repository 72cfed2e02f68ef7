"""The loss and the forward model read the object through a 32-bit byte range:
from 2^29 pixels on they are refused before anything reaches the device."""

import ctypes

import pytest

from tests.test_abi_errors import FAKE, PTY_E_UNSUPPORTED, lib  # noqa: F401

F = ctypes.c_void_p(FAKE)


@pytest.mark.parametrize("shape", [(23171, 23171), (1 << 24, 32), (32, 1 << 24), (1 << 15, 1 << 16)])
def test_objects_beyond_the_byte_range_are_refused(lib, shape):  # noqa: F811
    Px, Py = shape
    L = lib.load()
    need = L.pty_loss_workspace_bytes(32, Px, Py, 10, 10)
    assert L.pty_loss_gradients(F, F, Px, Py, F, 10, F, F, 10, 10, 32, 1.0, F, F, F, F, need,
                                None) == PTY_E_UNSUPPORTED
    assert "2^29" in lib.last_error()
    assert L.pty_simulate_intensities(F, F, Px, Py, F, 10, 32, F, None) == PTY_E_UNSUPPORTED
    assert "2^29" in lib.last_error()
