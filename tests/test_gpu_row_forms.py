"""Ket slices of the row kernels' tables: slices of one, an odd number and all
primitive pairs of a ket, so that the last slice of a ket is short, for bases
of short (6-31G) and long (cc-pVDZ) contractions.  The symmetrised build
against the per-function kernels (functions in reversed order form no whole
shells); both sum at most 1e6 FP64 terms: 1e-11 of max |G|."""
import numpy as np
import pytest

from geometries import water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["sto-3g", "6-31g", "cc-pvdz"])
@pytest.mark.parametrize("kslice", [1, 2, 3, 16])
def test_ket_slices(basis, kslice):
    from mmd import _native
    from mmd.molecule import Molecule
    mol = Molecule(water_cluster(2, 5.0, seed=4, perturb=True), basis)
    N = mol.nbasis
    rng = np.random.default_rng(kslice)
    D = rng.normal(size=(N, N))
    D = D + D.T
    ctx = _native.Context()
    ctx.set_basis_from_bfs(mol.bfs)
    ctx.schwarz()
    ctx.set_ket_slices([kslice] * 21)
    G = ctx.fock_delta(D, tol=1e-12)[0]
    r = np.arange(N)[::-1]
    ref = _native.Context()
    ref.set_basis_from_bfs([mol.bfs[i] for i in r])
    ref.schwarz()
    R = ref.fock_delta(D[np.ix_(r, r)], tol=1e-12, raw=True)[0][np.ix_(r, r)]
    assert np.max(np.abs(G - 0.5 * (R + R.T))) < 1e-11 * np.max(np.abs(G))
