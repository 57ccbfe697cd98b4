"""The per-molecule step of the batch engine at the sizes where its tiles,
rotations and leading dimensions change: 1 and 2 functions (one rotation or
none), odd and even n (the round-robin's dummy index, padded leading
dimensions), n around multiples of 16 (matrix-core tiles), 64 and 65 (a row
longer than a wavefront), 80 and 81 (the last in LDS) and 82 and 88 (the
matrices in global memory).

Chains of hydrogen atoms (with a helium atom where n is odd), one STO-3G
function each, give every n.  Step 0 of mmd/scf.py:41-61 needs no Fock
build: P = C_occ C_occ^T of the core Hamiltonian, against scipy's
generalised eigensolver in FP64.  Tolerance, from the reference: rounding of
relative size eps in n-term products of H and S^-1/2 turns the occupied space
by at most 4 eps n ||H|| cond(S) / gap.
"""
import numpy as np
import pytest
import scipy.linalg

import geometries  # noqa: F401  (puts the package on the path)

pytestmark = pytest.mark.gpu


def _chain(n):
    """n functions: H-H pairs 0.75 Angstrom wide, 1.35 apart, He first if n is odd."""
    odd = n % 2
    atoms, z = [], 0.0
    for k in range(n):
        atoms.append("%s 0.0 0.0 %.6f" % ("He" if odd and k == 0 else "H", z))
        z += 0.75 if k >= odd and (k - odd) % 2 == 0 else 1.35
    return "\n0 1\n" + "\n".join(atoms) + "\n"


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 32, 33, 52, 64, 65, 80, 81, 82, 88])
def test_core_density_of_hydrogen_chains(n):
    from mmd import _native
    from mmd.batch import _group_arrays
    if _native.device_count() < 1:
        pytest.fail("no HIP device: the GPU tests need an MI355X")
    sizes = [n, max(1, n - 1)]
    mols, (origin, lmn, nprim, exps, w) = _group_arrays([_chain(k) for k in sizes], "sto-3g")
    ctx = _native.Context(0)
    ctx.set_basis(origin, lmn, nprim, exps, w)
    ctx.set_atoms(np.concatenate([m[0] for m in mols]).astype(np.float64), np.concatenate([m[1] for m in mols]))
    ctx.set_molecules([m[5] for m in mols], [len(m[0]) for m in mols])
    res = ctx.batch_rhf([m[2] for m in mols], [m[3] for m in mols], maxiter=1, keep_density=True)
    o = 0
    for k, m in zip(sizes, mols):
        assert m[5] == k
        one = _native.Context(0)
        a, b = m[4], m[4] + m[5]
        q = np.concatenate([[0], np.cumsum(nprim)])
        one.set_basis(origin[a:b], lmn[a:b], nprim[a:b], exps[q[a]:q[b]], w[q[a]:q[b]])
        one.set_atoms(m[0].astype(np.float64), m[1])
        S, T, V = one.one_electron([0.0, 0.0, 0.0])[:3]
        e, C = scipy.linalg.eigh(T + V, S)
        gap = e[m[2]] - e[m[2] - 1] if m[2] < k else 1.0
        tol = 4 * np.finfo(float).eps * k * np.linalg.norm(T + V, 2) * np.linalg.cond(S) / gap
        ref = C[:, :m[2]] @ C[:, :m[2]].T
        P = res[3][o:o + k * k].reshape(k, k)
        o += k * k
        err = np.max(np.abs(P - ref))
        print("n=%d: max |P - P_ref| = %.2e (gap %.1e, tolerance %.1e)" % (k, err, gap, tol))
        assert tol < 1e-6
        assert err <= tol
