"""What the tensor calls keep between calls belongs to the device and not to a
context: many live molecules hold no more of it than one (512 MB and the
slots), buffers and slots left by arrays of other sizes serve later calls, and
all of it goes back on request."""
import ctypes

import numpy as np
import pytest

from test_gpu_host_copies import _check, _context

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free_memory():
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_many_live_molecules():
    """Eight contexts with tensors of 134 MB and 268 MB of workspace each for
    the transformation.  Each context's own tables are allocated before the
    first reading (a few MB); 64 MB for the runtime's own."""
    n = 64
    live = [_context(n) for _ in range(8)]
    for c in live:
        c.schwarz()
        c.eri_list([[0, 0, 0, 0]])
    before = _free_memory()
    T, out = np.empty((n,) * 4), np.empty((n,) * 4)
    for c in live:
        c.eri_tensor(out=T)
        c.jk_tensor(T, np.eye(n))
        c.ao2mo(T, np.eye(n), out=out)
        assert np.array_equal(out, T)
    assert before - _free_memory() <= (512 + 64) * MB


def test_release():
    from mmd import _native
    c = _context(64)
    T = c.eri_tensor()
    held = _free_memory()
    _native.release_workspaces()
    assert _free_memory() - held >= 64 ** 4 * 8
    assert np.array_equal(c.eri_tensor(), T)
    with pytest.raises(ValueError):
        _native.release_workspaces(-1)


def test_other_sizes_in_turn():
    """Larger and smaller arrays than the buffers and slots kept: two slots
    (36), five (49), six and more (64)."""
    for n in (49, 36, 64, 41, 36):
        _check(n)
