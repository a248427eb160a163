"""Which grids a batch of uneven grids takes (checked before any HIP call;
no GPU): its row passes work on nz / 2 complex columns, so an odd nz is
refused, where it used to be stepped with wrong rows."""
import ctypes

import pytest

from pyaxisymflow_amd import _lib
from pyaxisymflow_amd.stepper import _Buffers, _Config


def refusal(*sizes):
    cfgs = (_Config * len(sizes))()
    for c, nz in zip(cfgs, sizes):
        c.nz, c.nr, c.kill_width = nz, 64, 3
        c.dx, c.nu, c.CFL = 1.0 / nz, 1e-3, 0.1
    bufs, handle = _Buffers(), ctypes.c_void_p()  # no buffers: the last refusal
    lib = _lib.load()
    st = lib.axs_rigid_batch_create(cfgs, len(sizes), ctypes.byref(bufs), ctypes.byref(handle))
    assert st == _lib.AXS_ERR_INVALID and not handle.value
    return lib.axs_last_error().decode()


@pytest.mark.parametrize("sizes", [(128, 129), (257, 128), (127, 129), (128, 96, 1023)])
def test_odd_nz_is_refused(sizes):
    assert "even nz" in refusal(*sizes)


@pytest.mark.parametrize("sizes", [(128, 96), (1024, 130), (129,), (129, 129)])
def test_others_are_not(sizes):
    assert "null buffer" in refusal(*sizes)
