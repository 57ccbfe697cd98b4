"""The primitive screen of the pair tables, decided once and read by the fill:
contractions of 8 and 9 (64 primitive pairs fill a word of keep bits, 72 and
81 reach into a second one), some of their primitive pairs screened out, and
distances at which one primitive pair's bound lies within a few roundings of
the threshold.  The symmetrised build on the tables against the per-function
kernels, which use none (the functions in reversed order form no whole
shells); both sum at most 1e6 FP64 terms: 1e-11 of max |G|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DROP = 1e-20


def _functions(R):
    """Shells s(8), s(9), p(3) at 0, R and 2R along a skew line, and s(1)."""
    from mmd.integrals.twoe import Basis
    u = np.array([0.6, 0.0, 0.8])
    out = []
    for x, l, exps in ((0.0, 0, np.geomspace(0.12, 9000.0, 8)), (R, 0, np.geomspace(0.09, 30000.0, 9)),
                       (2 * R, 1, np.array([0.3, 2.0, 11.0])), (0.0, 0, np.array([0.25]))):
        for shell in ([(0, 0, 0)] if l == 0 else [(1, 0, 0), (0, 1, 0), (0, 0, 1)]):
            out.append(Basis(x * u, shell, len(exps), exps, np.linspace(1.0, 0.3, len(exps))))
    return out


def _bounds(bfs):
    """Schwarz-type bound of every primitive pair, times the largest."""
    sh = [b for b in bfs if tuple(b.shell) in ((0, 0, 0), (1, 0, 0))]
    rows = []
    for i, a in enumerate(sh):
        for b in sh[:i + 1]:
            R2 = ((a.origin - b.origin) ** 2).sum()
            p = a.exps[:, None] + b.exps[None]
            K = (a.norm * a.coefs)[:, None] * (b.norm * b.coefs)[None] * np.exp(-a.exps[:, None] * b.exps[None] / p * R2)
            f = 4.0 * (1.0 + np.sqrt(R2) + 1.0 / np.sqrt(p))
            rows.append((np.sqrt(34.98683665524972497 / (p * p * np.sqrt(2 * p))) * abs(K) * f ** (a.shell.sum() + b.shell.sum())).ravel())
    return np.concatenate(rows) * max(r.max() for r in rows)


def _check(bfs):
    from mmd import _native
    N = len(bfs)
    rng = np.random.default_rng(N)
    D = rng.normal(size=(N, N))
    D = D + D.T
    r = np.arange(N)[::-1]
    G, ref = _native.Context(), _native.Context()
    G.set_basis_from_bfs(bfs)
    G.schwarz()
    G = G.fock_delta(D, tol=1e-14)[0]
    ref.set_basis_from_bfs([bfs[i] for i in r])
    ref.schwarz()
    ref = ref.fock_delta(D[np.ix_(r, r)], tol=1e-14, raw=True)[0][np.ix_(r, r)]
    assert np.max(np.abs(G - 0.5 * (ref + ref.T))) < 1e-11 * np.max(np.abs(G))


@pytest.mark.parametrize("R", [0.0, 0.7, 2.0, 7.0, 40.0])
def test_keep_words(R):
    kept = _bounds(_functions(R)) >= DROP
    assert kept.any() and (R < 1.0 or not kept.all())
    _check(_functions(R))


@pytest.mark.parametrize("rank", [40, 80, 120])
def test_pair_at_the_threshold(rank):
    """The rank-th smallest bound at the threshold, by bisection over R."""
    lo, hi = 0.1, 40.0
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        lo, hi = (lo, mid) if np.sort(_bounds(_functions(mid)))[rank] < DROP else (mid, hi)
    assert abs(np.sort(_bounds(_functions(lo)))[rank] / DROP - 1.0) < 1e-10
    for ulps in (-6, -3, -1, 0, 1, 3, 6):
        _check(_functions(lo * (1.0 + ulps * 2.3e-16)))
