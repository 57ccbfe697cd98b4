"""Shell-class kernels of the nuclear gradient against the per-function
kernels, which serve the bases whose functions do not form whole shells: the
same functions in reversed order (a p shell as z, y, x is no whole shell)
take that path.  P and W are random and not symmetric.  Both paths add up to
1e6 FP64 terms no larger than the result's scale: 1e-11 of max |g|."""
import numpy as np
import pytest

from geometries import water_cluster

pytestmark = pytest.mark.gpu


def _gradient(bfs, Z, xyz, P, W, atom, nuclei=None):
    from mmd import _native
    ctx = _native.Context()
    ctx.set_basis_from_bfs(bfs)
    ctx.set_atoms(Z, xyz)
    return ctx.rhf_gradient(P, W, atom, nuclei)


def _problem(n, basis):
    from mmd.forces import basis_atoms
    from mmd.molecule import Molecule
    mol = Molecule(water_cluster(n, 4.0 + n, seed=5, perturb=True), basis)
    rng = np.random.default_rng(n)
    P = rng.normal(size=(mol.nbasis, mol.nbasis))
    W = rng.normal(size=(mol.nbasis, mol.nbasis))
    Z = np.array([a.charge for a in mol.atoms], dtype=float)
    return mol, Z, np.array([a.origin for a in mol.atoms]), P, W, basis_atoms(mol)


# sto-3g: one tile of everything; 6-31g: ragged slices of the s and p classes;
# cc-pvdz: all 21 quartet classes; 6-31gs: the d classes with two d shells
@pytest.mark.parametrize("n,basis", [(1, "sto-3g"), (3, "6-31g"), (1, "cc-pvdz"), (2, "6-31gs")])
def test_shell_classes_vs_functions(n, basis):
    mol, Z, xyz, P, W, atom = _problem(n, basis)
    r = np.arange(mol.nbasis)[::-1]
    g = _gradient(mol.bfs, Z, xyz, P, W, atom)
    # the one-electron part reads the lower triangle, as the reversed order does of the upper
    Pr, Wr = P[np.ix_(r, r)].copy(), W[np.ix_(r, r)].copy()
    ref = _gradient([mol.bfs[i] for i in r], Z, xyz, Pr, Wr, atom[r])
    tri = np.tril(P - P.T, -1), np.tril(W - W.T, -1)
    one = _one_electron_difference(mol, Z, xyz, tri, atom)
    assert np.max(np.abs(g - ref - one)) < 1e-11 * np.max(np.abs(g))


def _one_electron_difference(mol, Z, xyz, tri, atom):
    """The one-electron part is linear in the lower triangles of P and W: the
    difference between reading the lower and the upper one, from the
    per-function kernels at P = t D, where the two-electron part is even in t."""
    r = np.arange(mol.nbasis)[::-1]
    bfs = [mol.bfs[i] for i in r]
    D, E = (a + a.T for a in tri)
    p = _gradient(bfs, Z, xyz, D[np.ix_(r, r)], E[np.ix_(r, r)], atom[r])
    m = _gradient(bfs, Z, xyz, -D[np.ix_(r, r)], -E[np.ix_(r, r)], atom[r])
    return 0.5 * (p - m)


def test_many_nuclei_and_repulsion():
    """More nuclei than a workgroup sums in LDS (257 with charges on three),
    functions on high atom numbers; the nuclear repulsion added on the device."""
    from mmd.forces import nuclear_repulsion_gradient
    mol, Z, xyz, P, W, atom = _problem(1, "6-31g")
    P, W = P + P.T, W + W.T
    nat = 257
    Zb, xb = np.zeros(nat), np.arange(3.0 * nat).reshape(nat, 3) + 10.0
    Zb[-3:], xb[-3:] = Z, xyz
    g = _gradient(mol.bfs, Zb, xb, P, W, atom + nat - 3, np.column_stack([Zb, xb]))
    ref = _gradient(mol.bfs, Z, xyz, P, W, atom) + nuclear_repulsion_gradient(mol.atoms)
    assert np.max(np.abs(g[-3:] - ref)) < 1e-11 * np.max(np.abs(ref))
    assert np.max(np.abs(g[:-3])) == 0.0


def test_shell_spread_over_atoms():
    """Functions of one shell on different atoms: the per-function kernels."""
    mol, Z, xyz, P, W, atom = _problem(1, "sto-3g")
    P, W = P + P.T, W + W.T
    a = atom.copy()
    a[3] = 1   # O 2p_y of the shell (x, y, z)
    r = np.arange(mol.nbasis)[::-1]
    g = _gradient(mol.bfs, Z, xyz, P, W, a)
    ref = _gradient([mol.bfs[i] for i in r], Z, xyz, P[np.ix_(r, r)], W[np.ix_(r, r)], a[r])
    assert np.max(np.abs(g - ref)) < 1e-11 * np.max(np.abs(g))
