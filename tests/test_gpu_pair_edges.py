"""Pair tables and work units where their steps change hands: up to 256 pairs
in one workgroup, more over many, and more than a block of the prefix sums
(1024 pairs), whose carries count from the second block on, and tables of more
than 64 MB, which are sized by what the device counted.  The symmetrised build on the tables against
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


def check_molecules(mols):
    """Several molecules in one basis: each block of the build as the molecule's own."""
    from mmd import _native
    nf = [len(b) for b in mols]
    f0 = np.concatenate([[0], np.cumsum(nf)])
    ctx = _native.Context()
    ctx.set_basis_from_bfs([b for m in mols for b in m])
    ctx.set_atoms(np.ones(len(mols)), np.arange(3.0 * len(mols)).reshape(-1, 3))
    ctx.set_molecules(nf, [1] * len(mols))
    ctx.schwarz()
    rng = np.random.default_rng(5)
    D = np.zeros((f0[-1], f0[-1]))
    for k, n in enumerate(nf):
        A = rng.normal(size=(n, n))
        D[f0[k]:f0[k + 1], f0[k]:f0[k + 1]] = A + A.T
    G = ctx.fock_delta(D, tol=1e-12)[0]
    for k, b in enumerate(mols):
        s = slice(f0[k], f0[k + 1])
        ref = context(b).fock_delta(D[s, s], tol=1e-12)[0]
        assert np.max(np.abs(G[s, s] - ref)) < 1e-11 * np.max(np.abs(ref))


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


@pytest.mark.parametrize("n,pairs", [(45, 1035), (64, 2080)])
def test_blocks_of_the_prefix_sums(n, pairs):
    assert n * (n + 1) // 2 == pairs and pairs > 1024
    check(shells(n, n))


def test_molecules_across_a_block():
    """Several molecules in one basis, the (ss) pairs of the second from 435 to
    1176."""
    ns = (30, 39, 2, 20)
    mols = [shells(n, n) for n in ns]
    ss = [n * (n - 1) // 2 for n in ns]   # all but the pairs with the p shell
    assert ss[0] < 1024 < ss[0] + ss[1]
    check_molecules(mols)


def test_large_tables():
    """Seventy molecules of 36 pairs of 144 primitive pairs."""
    from mmd.integrals.twoe import Basis

    def molecule(seed):
        rng = np.random.default_rng(seed)
        out = []
        for k in range(8):
            x, exps = rng.uniform(0.0, 5.0, 3), np.geomspace(900.0, 0.15, 12)
            for shell in [(1, 0, 0), (0, 1, 0), (0, 0, 1)] if k == 3 else [(0, 0, 0)]:
                out.append(Basis(x, shell, 12, exps, np.linspace(0.2, 1.0, 12)))
        return out
    mols = [molecule(1), molecule(2)] * 35
    assert len(mols) * 36 * 144 * 26 * 8 > 64 << 20
    check_molecules(mols)
