"""Pair tables and work units built on the device, at their edges: pairs whose
primitive pairs are all screened out (monomers 100 A apart), one shell only,
more pairs than one block of the prefix sums, molecules of unequal size in one
basis.  The symmetrised build on the tables against the per-function kernels,
which use none (the functions in reversed order form no whole shells); both
sum at most 1e6 FP64 terms: 1e-11 of max |G|."""
import numpy as np
import pytest

from geometries import water_cluster

pytestmark = pytest.mark.gpu

HELIUM = "0 1\nHe 0.0 0.0 0.0\n"
FAR = "0 1\nO 0 0 0\nH 0.76 0.59 0\nH -0.76 0.59 0\nO 100 0 0\nH 100.76 0.59 0\nH 99.24 0.59 0\n"


def _context(bfs):
    from mmd import _native
    ctx = _native.Context()
    ctx.set_basis_from_bfs(bfs)
    ctx.schwarz()
    return ctx


@pytest.mark.parametrize("geometry,basis", [(HELIUM, "sto-3g"), (FAR, "6-31g"),
                                            (water_cluster(6, 9.0, seed=1, perturb=True), "sto-3g")])
def test_build_on_tables(geometry, basis):
    from mmd.molecule import Molecule
    mol = Molecule(geometry, basis)
    N = mol.nbasis
    rng = np.random.default_rng(N)
    D = rng.normal(size=(N, N))
    D = D + D.T
    G, _, _ = _context(mol.bfs).fock_delta(D, tol=1e-12)
    r = np.arange(N)[::-1]
    if N == 1:   # one function is a whole shell in either order
        ref = _context(mol.bfs).fock_delta(D, tol=1e-12, raw=True)[0]
    else:
        ref = _context([mol.bfs[i] for i in r]).fock_delta(D[np.ix_(r, r)], tol=1e-12, raw=True)[0][np.ix_(r, r)]
    assert np.max(np.abs(G - 0.5 * (ref + ref.T))) < 1e-11 * np.max(np.abs(G))


def test_block_diagonal_basis():
    """Several molecules in one basis: each block as the molecule's own build."""
    from mmd import _native
    from mmd.molecule import Molecule
    mols = [Molecule(g, "6-31g") for g in (HELIUM, FAR, water_cluster(3, 6.0, seed=2, perturb=True), HELIUM)]
    n = [m.nbasis for m in mols]
    ctx = _native.Context()
    ctx.set_basis_from_bfs([b for m in mols for b in m.bfs])
    ctx.set_atoms([a.charge for m in mols for a in m.atoms], np.array([a.origin for m in mols for a in m.atoms]))
    ctx.set_molecules(n, [len(m.atoms) for m in mols])
    ctx.schwarz()
    rng = np.random.default_rng(3)
    D = np.zeros((sum(n), sum(n)))
    f0 = np.concatenate([[0], np.cumsum(n)])
    for k in range(len(mols)):
        A = rng.normal(size=(n[k], n[k]))
        D[f0[k]:f0[k + 1], f0[k]:f0[k + 1]] = A + A.T
    G, _, _ = ctx.fock_delta(D, tol=1e-12)
    for k, m in enumerate(mols):
        s = slice(f0[k], f0[k + 1])
        ref, _, _ = _context(m.bfs).fock_delta(D[s, s], tol=1e-12)
        assert np.max(np.abs(G[s, s] - ref)) < 1e-11 * np.max(np.abs(ref))
