"""Pair tables and work units where their steps change hands: up to 256 pairs
in one workgroup, more over many.  The symmetrised build on the tables against
the per-function kernels, which use none (the functions in reversed order form
no whole shells); both sum at most 1e6 FP64 terms: 1e-11 of max |G|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shells(n, seed):
    """n shells, the middle one a p shell, the others s, of one to three
    primitives, at random places."""
    from mmd.integrals.twoe import Basis
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        x = rng.uniform(0.0, 3.0 * n ** (1.0 / 3.0), 3)
        exps = np.sort(rng.uniform(0.2, 4.0, 1 + k % 3))[::-1]
        coefs = rng.uniform(0.2, 1.0, len(exps))
        for shell in [(1, 0, 0), (0, 1, 0), (0, 0, 1)] if k == n // 2 else [(0, 0, 0)]:
            out.append(Basis(x, shell, len(exps), exps, coefs.copy()))
    return out


def context(bfs):
    from mmd import _native
    ctx = _native.Context()
    ctx.set_basis_from_bfs(bfs)
    ctx.schwarz()
    return ctx


def check(bfs):
    N = len(bfs)
    rng = np.random.default_rng(N)
    D = rng.normal(size=(N, N))
    D = D + D.T
    G = context(bfs).fock_delta(D, tol=1e-12)[0]
    r = np.arange(N)[::-1]
    ref = context([bfs[i] for i in r]).fock_delta(D[np.ix_(r, r)], tol=1e-12, raw=True)[0][np.ix_(r, r)]
    assert np.max(np.abs(G - 0.5 * (ref + ref.T))) < 1e-11 * np.max(np.abs(G))


@pytest.mark.parametrize("n,pairs", [(1, 1), (2, 3), (22, 253), (23, 276)])
def test_one_workgroup_and_many(n, pairs):
    bfs = shells(n, n)
    assert n * (n + 1) // 2 == pairs and len(bfs) == n + 2
    check(bfs)


def test_small_after_large_and_back():
    """One context, tables of both kinds in turn in the same buffers."""
    from mmd import _native
    ctx = _native.Context()
    for n in (30, 4, 22, 30, 2):
        bfs = shells(n, 7 * n)
        N = len(bfs)
        D = np.random.default_rng(n).normal(size=(N, N))
        D = D + D.T
        ctx.set_basis_from_bfs(bfs)
        ctx.schwarz()
        G, ref = ctx.fock_delta(D, tol=1e-12)[0], context(bfs).fock_delta(D, tol=1e-12)[0]
        assert np.max(np.abs(G - ref)) < 1e-11 * np.max(np.abs(ref))
