"""Integral-block kernels (stored tensor, formPT's unsymmetrised build) at the
edges of their classes, against the oracle: every quartet class (cc-pVDZ
water), ragged groups of lanes (6-31G, contractions of 1 to 36 primitive
pairs), the smallest basis.  Complex density differences that are not
Hermitian, with a screen that keeps nearly all and one that drops most
quartets.  Both sides sum at most 1e5 FP64 terms of the result's scale:
1e-11 of the largest element."""
import os

import numpy as np
import pytest

from geometries import HELIUM, water_cluster

pytestmark = pytest.mark.gpu

BASIS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcmurchie-davidson_amd",
                     "mmd", "basis")


def _pair(geometry, basis, oracle):
    from mmd.molecule import Molecule
    return Molecule(geometry, basis), oracle.OracleMolecule(geometry, os.path.join(BASIS, basis + ".gbs"))


CASES = [(HELIUM, "6-31g"), (water_cluster(1, 3.0, seed=2, perturb=True), "cc-pvdz"),
         (water_cluster(2, 5.0, seed=4, perturb=True), "6-31g")]


@pytest.mark.parametrize("geometry,basis", CASES)
def test_tensor(oracle, geometry, basis):
    mol, om = _pair(geometry, basis, oracle)
    T = mol.native.eri_tensor()
    ref = om.eri_tensor()
    assert np.max(np.abs(T - ref)) < 1e-11 * np.max(np.abs(ref))
    for perm in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):   # one producer per orbit: bitwise
        assert np.array_equal(T, T.transpose(perm))


@pytest.mark.parametrize("tol", [1e-12, 1e-2])
@pytest.mark.parametrize("geometry,basis", CASES)
def test_form_pt(oracle, geometry, basis, tol):
    from mmd.integrals.fock import formPT
    mol, om = _pair(geometry, basis, oracle)
    mol.build(direct=True)
    N = mol.nbasis
    rng = np.random.default_rng(N)
    P = rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))
    P *= 10.0 ** rng.uniform(-6, 0, size=(N, N))
    P_old = 0.1 * rng.normal(size=(N, N)) * (1 + 0j)
    G = formPT(P, P_old, mol.bfs, N, mol.screen, tol)
    ref, _ = om.form_pt(P, P_old, om.schwarz(), tol)
    assert np.max(np.abs(G - ref)) < 1e-11 * np.max(np.abs(ref))
    real = formPT(P.real.astype(complex), P_old, mol.bfs, N, mol.screen, tol)
    ref, _ = om.form_pt(P.real.astype(complex), P_old, om.schwarz(), tol)
    assert np.max(np.abs(real - ref)) < 1e-11 * np.max(np.abs(ref))


def test_form_pt_nan_is_kept(oracle):
    from mmd.integrals.fock import formPT
    mol, _ = _pair(CASES[0][0], "6-31g", oracle)
    mol.build(direct=True)
    P = np.full((mol.nbasis, mol.nbasis), np.nan, dtype=complex)
    assert np.isnan(formPT(P, np.zeros_like(P), mol.bfs, mol.nbasis, mol.screen, 1e-12)).all()
