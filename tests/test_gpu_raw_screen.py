"""formPT's raw build keeps what does not compare as small: Schwarz values that
are negative or not numbers (their square root is none), in part of the
functions of a shell pair, and densities that are infinite or not numbers, also
where all primitive pairs of a distant shell pair are screened out.  Against
the per-function kernels (the functions in reversed order form no whole shells);
sums of at most 1e6 FP64 terms: 1e-11 of max |G|, and the same elements that are
not finite."""
import numpy as np
import pytest

from geometries import water_cluster

pytestmark = pytest.mark.gpu

FAR = "0 1\nO 0 0 0\nH 0.76 0.59 0\nH -0.76 0.59 0\nO 100 0 0\nH 100.76 0.59 0\nH 99.24 0.59 0\n"


def _both(geometry, basis, screen, dP, tol):
    """(G on the shell-class path, G on the per-function path); dP real or complex."""
    from mmd import _native
    from mmd.molecule import Molecule
    bfs = Molecule(geometry, basis).bfs
    N = len(bfs)
    out = []
    for order in (np.arange(N), np.arange(N)[::-1]):
        ctx = _native.Context()
        ctx.set_basis_from_bfs([bfs[i] for i in order])
        diag = ctx.schwarz()
        p = np.ix_(order, order)
        if screen is not None:
            ctx.set_schwarz(screen(diag[p])[p])
        D = dP(N)[p]
        re, im, _ = ctx.fock_delta(D.real, D.imag if np.iscomplexobj(D) else None, tol=tol, raw=True)
        back = np.argsort(order)
        b = np.ix_(back, back)
        out.append([re[b]] + ([] if im is None else [im[b]]))
    return out


def _density(N):
    D = np.random.default_rng(N).normal(size=(N, N))
    return D + D.T


def _sym_raw(G):
    # the canonical form of a quartet depends on the order of the functions
    return G + G.T


@pytest.mark.parametrize("value", [-1.0, np.nan, 0.0])
@pytest.mark.parametrize("share", [0.1, 1.0])
def test_schwarz_values(value, share):
    def screen(diag):
        N = len(diag)
        m = np.random.default_rng(7).random((N, N)) < share
        m = np.tril(m) | np.tril(m).T
        return np.where(m, value * np.abs(diag), diag)
    for basis in ("6-31g", "cc-pvdz"):
        (G,), (R,) = _both(water_cluster(1, 3.6, seed=4, perturb=True), basis, screen, _density, 1e-6)
        G, R = _sym_raw(G), _sym_raw(R)
        assert np.max(np.abs(G - R)) <= 1e-11 * np.max(np.abs(R))
        assert value == 0.0 or np.max(np.abs(R)) > 1e-3


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("imag", [False, True])
def test_density_values(value, imag):
    def dP(N):
        D = _density(N)
        E = _density(N)
        (E if imag else D)[0, N - 1] = (E if imag else D)[N - 1, 0] = value
        if not imag:
            return D
        Z = np.empty((N, N), dtype=complex)
        Z.real, Z.imag = D, E
        return Z
    for geometry, basis in ((FAR, "6-31g"), (water_cluster(1, 3.6, seed=4, perturb=True), "cc-pvdz")):
        for G, R in zip(*_both(geometry, basis, None, dP, 1e-12)):
            with np.errstate(invalid="ignore"):
                G, R = _sym_raw(G), _sym_raw(R)
            f = np.isfinite(R)
            assert np.array_equal(np.isfinite(G), f)
            assert not f.any() or np.max(np.abs(G[f] - R[f])) <= 1e-11 * np.max(np.abs(R[f]))
