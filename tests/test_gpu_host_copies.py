"""Copies of N^4 arrays between the device and ordinary host memory: below the
size that is staged (N = 35), just above it (36, a last slot that is not
full), whole slots only (64), pinned memory (not staged), and two contexts at
once.  A piece of the stored tensor in the wrong place breaks its symmetries,
which hold exactly; the transformation with C = 1 returns its input exactly.
J and K against numpy: sums of N^2 products, 1e-11 of the largest."""
import ctypes
import threading

import numpy as np
import pytest

from test_gpu_batch_step import _chain

pytestmark = pytest.mark.gpu


def _context(n):
    from mmd import _native
    from mmd.molecule import Molecule
    mol = Molecule(_chain(n), "sto-3g")
    ctx = _native.Context()
    ctx.set_basis_from_bfs(mol.bfs)
    return ctx


def _check(n):
    ctx = _context(n)
    T = ctx.eri_tensor(out=np.full((n,) * 4, np.nan))
    for perm in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(T, T.transpose(perm))
    rng = np.random.default_rng(n)
    idx = rng.integers(0, n, size=(20000, 4))
    ref = ctx.eri_list(idx)
    assert np.max(np.abs(T[tuple(idx.T)] - ref)) < 1e-12
    P, Q = rng.normal(size=(n, n)), rng.normal(size=(n, n))
    Jr, Ji, Kr, Ki = ctx.jk_tensor(T, P, Q)
    M = T.reshape(n * n, n * n)
    for J, K, D in ((Jr, Kr, P), (Ji, Ki, Q)):
        J0 = (M @ D.T.ravel()).reshape(n, n)
        K0 = np.stack([np.tensordot(T[p], D, axes=([0, 2], [0, 1])) for p in range(n)])
        assert np.max(np.abs(J - J0)) < 1e-11 * np.max(np.abs(J0))
        assert np.max(np.abs(K - K0)) < 1e-11 * np.max(np.abs(K0))
    out = np.full((n,) * 4, np.nan)
    ctx.ao2mo(T, np.eye(n), out=out)
    assert np.array_equal(out, T)


@pytest.mark.parametrize("n", [35, 36, 64])
def test_copies(n):
    _check(n)


def test_pinned_output():
    ctx = _context(36)
    T = ctx.eri_tensor()
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(T.nbytes), ctypes.c_uint(0)) == 0
    try:
        pinned = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), shape=T.shape)
        pinned[:] = np.nan
        ctx.eri_tensor(out=pinned)
        assert np.array_equal(pinned, T)
        assert all(np.array_equal(a, b) for a, b in zip(ctx.jk_tensor(pinned, T[0, 0], T[1, 1]),
                                                        ctx.jk_tensor(T, T[0, 0], T[1, 1])))
    finally:
        assert hip.hipHostFree(p) == 0


def test_two_contexts_at_once():
    errors = []

    def work(n):
        try:
            for _ in range(3):
                _check(n)
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in (36, 41)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
