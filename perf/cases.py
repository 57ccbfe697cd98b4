"""Performance cases: water clusters through the package's public entry points.

Each case is one call that a program of this package makes once per SCF
iteration, per geometry or per batch; the sizes are those of the tests and
of bench.py (clusters of 1 to 16 molecules, STO-3G to cc-pVDZ, batches of up
to 512 molecules).  Densities have the structure that an SCF meets: entries
of order one inside a monomer, decaying with the distance of the two centres,
scaled down to the size of a density difference where a case stands for a
later iteration.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mcmurchie-davidson_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from mmd.batch import run_batch_device               # noqa: E402
from mmd.integrals.fock import formPT                # noqa: E402
from mmd.integrals.twoe import doERIs                # noqa: E402
from mmd.molecule import Molecule                    # noqa: E402
from mmd.workloads import water_cluster              # noqa: E402

BASIS_DIR = os.path.join(PKG, "mmd", "basis")
BOHR = 0.52917721092
NBF = {"sto-3g": 7, "6-31g": 13, "6-31gs": 19, "cc-pvdz": 25}   # functions per water


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The symmetrised Fock build of a direct SCF, once per iteration: one
        # small molecule (launches and the read-back count), an odd-sized
        # cluster with d functions in the middle of its SCF, the cluster that
        # bench.py quotes Fock-build times on, and the largest one in use.
        {"name": "fock-1-631g", "kind": "fock", "n": 1, "basis": "6-31g", "scale": 1.0},
        {"name": "fock-3-631gs", "kind": "fock", "n": 3, "basis": "6-31gs", "scale": 1e-3},
        {"name": "fock-8-ccpvdz", "kind": "fock", "n": 8, "basis": "cc-pvdz", "scale": 1e-2},
        {"name": "fock-16-ccpvdz", "kind": "fock", "n": 16, "basis": "cc-pvdz", "scale": 1.0},
        # formPT with a complex density difference: the reference's own entry
        # point of the direct build, as a real-time propagation calls it.
        {"name": "formpt-2-631g", "kind": "formpt", "n": 2, "basis": "6-31g", "scale": 1.0},
        # The conventional path: the stored tensor (doERIs, once per
        # geometry), its J/K contraction with a complex density (every step
        # of a real-time propagation) and the four-index transformation (MP2).
        {"name": "doeris-4-631g", "kind": "doeris", "n": 4, "basis": "6-31g"},
        {"name": "jk-4-631g", "kind": "jk", "n": 4, "basis": "6-31g"},
        {"name": "ao2mo-3-631gs", "kind": "ao2mo", "n": 3, "basis": "6-31gs"},
        # Nuclear forces, once per geometry of an optimisation or trajectory:
        # one molecule in a basis with d functions, and bench.py's cluster.
        {"name": "forces-1-ccpvdz", "kind": "forces", "n": 1, "basis": "cc-pvdz"},
        {"name": "forces-4-631g", "kind": "forces", "n": 4, "basis": "6-31g"},
        # Whole batches from geometry strings to converged energies: an
        # ordinary odd-sized one that also wants the densities, and the
        # headline (512 clusters of 2 to 6, the learned start, four groups).
        {"name": "batch-45", "kind": "batch", "count": 45, "lo": 1, "hi": 5, "basis": "6-31g", "guess": "sad",
         "group": 64, "streams": 2, "density": True},
        {"name": "batch-512", "kind": "batch", "count": 512, "lo": 2, "hi": 6, "basis": "6-31g", "guess": "learned",
         "group": 128, "streams": 4, "density": False},
    ]


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["fock", "fock", "fock", "formpt", "doeris", "jk", "ao2mo", "forces", "forces", "batch", "batch"])
    if kind == "batch":
        basis = rng.choice(["sto-3g", "6-31g", "6-31g"])
        guess = rng.choice(["core", "sad", "learned"]) if basis == "6-31g" else rng.choice(["core", "sad"])
        lo = rng.randint(1, 4)
        hi = rng.randint(lo, 6)
        count = int(round(math.exp(rng.uniform(math.log(2), math.log(256)))))
        return {"kind": kind, "count": count, "lo": lo, "hi": hi, "basis": basis, "guess": guess,
                "group": rng.choice([32, 64, 100, 128]), "streams": rng.choice([1, 2, 3, 4]),
                "density": rng.random() < 0.5}
    basis = rng.choice(["sto-3g", "6-31g", "6-31gs", "cc-pvdz"])
    most = {"fock": 400, "formpt": 26, "doeris": 60, "jk": 60, "ao2mo": 60, "forces": 38}[kind]
    if kind == "forces" and basis in ("sto-3g", "6-31g"):
        most = 52
    top = max(1, min(16, most // NBF[basis]))
    n = int(round(math.exp(rng.uniform(0.0, math.log(top + 0.49)))))
    case = {"kind": kind, "n": n, "basis": basis, "geometry": rng.randint(1, 10 ** 6)}
    if kind in ("fock", "formpt"):
        case["scale"] = 10.0 ** rng.uniform(-6.0, 0.0)
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _geometry(case, seed):
    n = case["n"]
    return water_cluster(n, 3.6 * n ** (1.0 / 3.0), seed=1000003 * case.get("geometry", 0) + seed, perturb=True)


def _batch_geometries(case, seed):
    # the mix of sizes belongs to the case, the geometries to the seed
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    ns = rng.integers(case["lo"], case["hi"] + 1, case["count"])
    return [water_cluster(int(n), 2.0 + 1.4 * int(n), seed=100003 * seed + i, perturb=True) for i, n in enumerate(ns)]


def _centres(geometry, basis):
    """Coordinates (bohr) of every atom, and the atom of every basis function."""
    Z, X = _atoms(geometry)
    at = np.concatenate([np.full(sum(len(_CART[l]) for l, _, _ in _shells(basis, z)), a) for a, z in enumerate(Z)])
    return X, at


def _density(case, seed, tag=0):
    """A symmetric matrix with the decay of a density."""
    X, at = _centres(_geometry(case, seed), case["basis"])
    rng = np.random.default_rng([seed, 17, tag])
    R = np.linalg.norm(X[at][:, None] - X[at][None], axis=-1)
    W = rng.normal(size=R.shape)
    D = 0.25 * (W + W.T) * np.exp(-R / 1.5)
    D[np.diag_indices_from(D)] = rng.uniform(0.1, 1.0, len(D))
    return D


def _antisymmetric(case, seed):
    D = _density(case, seed, 1)
    return np.triu(D, 1) - np.triu(D, 1).T


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return {"case": case, "geometries": _batch_geometries(case, seed)}
    mol = Molecule(_geometry(case, seed), case["basis"])
    N = mol.nbasis
    state = {"case": case, "mol": mol}
    if kind in ("fock", "formpt"):
        mol.build(direct=True)
        state["P"] = case["scale"] * _density(case, seed)
        if kind == "formpt":
            state["P"] = state["P"] + 1j * case["scale"] * _antisymmetric(case, seed)
            state["P_old"] = np.zeros((N, N), dtype=complex)
    elif kind == "doeris":
        mol.native   # the basis on the device
        state["T"] = np.zeros((N, N, N, N))
    elif kind == "jk":
        mol.build(direct=False)
        mol.direct = False
        mol.P = _density(case, seed) + 1j * _antisymmetric(case, seed)
    elif kind == "ao2mo":
        mol.native
        state["T"] = mol.native.eri_tensor()
        state["C"] = _orbitals(N, seed)
        state["out"] = np.empty((N, N, N, N))
    elif kind == "forces":
        mol.native
        mol.P = _density(case, seed)
        mol.F = _density(case, seed, 2)
        mol.is_converged = True
    return state


def _orbitals(N, seed):
    return np.linalg.qr(np.random.default_rng([seed, 23]).normal(size=(N, N)))[0]


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "batch":
        res = run_batch_device(state["geometries"], case["basis"], group=case["group"], guess=case["guess"],
                               streams=case["streams"], class_streams=2, keep_density=case["density"])
        out = {"energy": np.array([r["energy"] for r in res])}
        if case["density"]:
            out["P"] = np.concatenate([r["P"].ravel() for r in res])
        return out
    mol = state["mol"]
    if kind == "fock":
        return mol.native.fock_delta(state["P"], tol=1e-12)[0]
    if kind == "formpt":
        return formPT(state["P"], state["P_old"], mol.bfs, mol.nbasis, mol.screen, 1e-12)
    if kind == "doeris":
        return np.asarray(doERIs(mol.nbasis, state["T"], mol.bfs))
    if kind == "jk":
        mol.buildFock()
        return {"J": mol.J, "K": mol.K, "F": mol.F}
    if kind == "ao2mo":
        return mol.native.ao2mo(state["T"], state["C"], out=state["out"])
    return mol.forces()


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _class_flops(la, lb, lc, ld):
    """Operations per primitive shell quartet: the two Hermite contractions,
    the R recursion and the Boys function."""
    H = lambda L: (L + 1) * (L + 2) * (L + 3) // 6                    # noqa: E731
    NR = lambda L: (L + 1) * (L + 2) * (L + 3) * (L + 4) // 24        # noqa: E731
    C = lambda a, b: (a + 1) * (a + 2) * (b + 1) * (b + 2) // 4       # noqa: E731
    return 2 * H(la + lb) * H(lc + ld) * C(lc, ld) + 2 * C(la, lb) * H(la + lb) * C(lc, ld) + 3 * NR(la + lb + lc + ld) + 40


def _quartet_flops(geometry, basis, dmax, tol, raise_l=0):
    """Operations over the primitive quartets whose contracted shell pairs
    pass the Schwarz bound q q' 4 dmax >= tol (s-type bounds)."""
    Z, X = _atoms(geometry)
    sh = [(l, X[a], e, w) for a, z in enumerate(Z) for l, e, w in _shells(basis, z)]
    pairs = {}
    for i, (la, A, ea, wa) in enumerate(sh):
        for lb, B, eb, wb in sh[:i + 1]:
            p = ea[:, None] + eb[None]
            K = np.abs(wa[:, None] * wb[None]) * np.exp(-ea[:, None] * eb[None] / p * ((A - B) ** 2).sum())
            s = np.sqrt(2 * np.pi ** 2.5 / (p * p * np.sqrt(2 * p))) * K * (0.5 / p) ** (0.5 * (la + lb))
            pairs.setdefault((max(la, lb), min(la, lb)), []).append((s.sum(), (s > 1e-14 * s.max() + 1e-18).sum()))
    arr = {k: np.array(sorted(v, key=lambda t: -t[0])) for k, v in pairs.items()}
    total = 0.0
    for k1, a in arr.items():
        for k2, b in arr.items():
            cum = np.concatenate([[0.0], np.cumsum(b[:, 1])])
            need = tol / (4 * dmax * np.maximum(a[:, 0], 1e-300))
            n = np.searchsorted(-b[:, 0], -need, side="right")
            total += 0.5 * float((a[:, 1] * cum[n]).sum()) * _class_flops(k1[0] + raise_l, k1[1], k2[0], k2[1])
    return total


def work(case):
    kind = case["kind"]
    if kind == "batch":
        sizes = range(case["lo"], case["hi"] + 1)
        per = case["count"] / len(sizes)
        fl = by = 0.0
        for n in sizes:
            N = n * NBF[case["basis"]]
            g = water_cluster(n, 2.0 + 1.4 * n, seed=1, perturb=True)
            # thirteen builds of shrinking density differences, and the
            # products and the eigensolver of each iteration
            fl += per * sum(_quartet_flops(g, case["basis"], 10.0 ** -k, 1e-12) for k in (0, 2, 4, 6)) / 4 * 13
            fl += per * 13 * 40.0 * N ** 3
            by += per * 8.0 * 3 * N * N
        return {"bytes": by, "flops": fl}
    N = case["n"] * NBF[case["basis"]]
    geometry = _geometry(case, 1)
    if kind == "fock":
        return {"bytes": 16.0 * N * N, "flops": _quartet_flops(geometry, case["basis"], case["scale"], 1e-12)}
    if kind == "formpt":
        return {"bytes": 32.0 * N * N, "flops": _quartet_flops(geometry, case["basis"], case["scale"], 1e-12)}
    if kind == "doeris":
        return {"bytes": 8.0 * N ** 4, "flops": _quartet_flops(geometry, case["basis"], 1.0, 0.0)}
    if kind == "jk":
        return {"bytes": 8.0 * N ** 4, "flops": 8.0 * N ** 4}
    if kind == "ao2mo":
        return {"bytes": 16.0 * N ** 4, "flops": 8.0 * N ** 5}
    return {"bytes": 24.0 * N * N, "flops": 3 * _quartet_flops(geometry, case["basis"], 1.0, 0.0, raise_l=1)}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain numpy and torch: Hermite Gaussian
# expansions of all function pairs as one matrix M, the Coulomb interaction of
# all primitive Hermite pairs as a second one, H, and (pq|rs) = M H M^T.
# ---------------------------------------------------------------------------
_CART = {l: [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)] for l in range(3)}
_BASIS = {}


def _atoms(geometry):
    rows = [r.split() for r in geometry.strip().split("\n")[1:]]
    return [{"H": 1, "O": 8}[r[0]] for r in rows], np.array([[float(v) for v in r[1:4]] for r in rows]) / BOHR


def _odd(n):
    return 1.0 if n < 2 else n * _odd(n - 2)


def _shells(basis, z):
    """(l, exponents, weights) of an element's shells, in file order; the
    weights are those of the first component (x^l), normalised."""
    key = (basis, z)
    if key not in _BASIS:
        sym, out = {1: "H", 8: "O"}[z], []
        with open(os.path.join(BASIS_DIR, basis + ".gbs")) as fh:
            blocks = [b.strip().split("\n") for b in fh.read().split("****")]
        rows = [r.split() for r in next(b for b in blocks if b[0].split()[0] == sym and b[0].split()[1] == "0")[1:]]
        i = 0
        while i < len(rows):
            name, n = rows[i][0], int(rows[i][1])
            tab = np.array([[float(v.replace("D", "E")) for v in r] for r in rows[i + 1:i + 1 + n]])
            for c, letter in enumerate(name):
                l = "SPD".index(letter)
                e, w = tab[:, 0], tab[:, 1 + c] * (2 * tab[:, 0] / np.pi) ** 0.75 * np.sqrt((4 * tab[:, 0]) ** l / _odd(2 * l - 1))
                s = e[:, None] + e[None]
                norm = (w[:, None] * w[None] * (np.pi / s) ** 1.5 * _odd(2 * l - 1) / (2 * s) ** l).sum()
                out.append((l, e, w / np.sqrt(norm)))
            i += 1 + n
        _BASIS[key] = out
    return _BASIS[key]


class _Boys(torch.autograd.Function):
    """F_0 .. F_n of x >= 0, stacked; dF_m/dx = -F_{m+1}."""

    @staticmethod
    def forward(ctx, x, n):
        top = n + 1
        small = x < 35.0
        xs = torch.where(small, x, torch.full_like(x, 35.0))
        e = torch.exp(-xs)
        term = torch.full_like(xs, 1.0 / (2 * top + 1))
        acc = term.clone()
        for k in range(1, 160):   # ascending series of F_top
            term = term * (2 * xs) / (2 * top + 2 * k + 1)
            acc += term
        F = [None] * (top + 1)
        F[top] = acc * e
        for m in range(top - 1, -1, -1):
            F[m] = (2 * xs * F[m + 1] + e) / (2 * m + 1)
        xb = torch.where(small, torch.full_like(x, 35.0), x)
        eb = torch.exp(-xb)
        f = 0.5 * torch.sqrt(math.pi / xb) * torch.erf(torch.sqrt(xb))
        for m in range(top + 1):
            F[m] = torch.where(small, F[m], f)
            f = ((2 * m + 1) * f - eb) / (2 * xb)
        F = torch.stack(F)
        ctx.save_for_backward(F)
        return F[:-1].clone()

    @staticmethod
    def backward(ctx, g):
        F, = ctx.saved_tensors
        return -(g * F[1:]).sum(0), None


def _r_table(L, X, Y, Z, seeds):
    """R_tuv, t + u + v <= L, from seeds[n] = (-2 alpha)^n F_n times a prefactor."""
    R = {(0, 0, 0, n): seeds[n] for n in range(L + 1)}
    for d in range(1, L + 1):
        for t in range(d, -1, -1):
            for u in range(d - t, -1, -1):
                h = [t, u, d - t - u]
                ax = next(k for k in range(3) if h[k])
                one = list(h)
                one[ax] -= 1
                two = list(one)
                two[ax] -= 1
                for n in range(L - d + 1):
                    v = (X, Y, Z)[ax] * R[(*one, n + 1)]
                    if two[ax] >= 0:
                        v = v + one[ax] * R[(*two, n + 1)]
                    R[(*h, n)] = v
    return R


def _e_table(LI, LJ, inv2p, PA, PB):
    """1-D Hermite coefficients E[i, j, t] without the Gaussian-product factor."""
    E = {(0, 0, 0): torch.ones_like(inv2p)}
    get = lambda i, j, t: E.get((i, j, t))   # noqa: E731

    def step(i, j, t, shift):
        v = torch.zeros_like(inv2p)
        for c, k, tt in ((inv2p, 1.0, t - 1), (shift, 1.0, t), (None, t + 1.0, t + 1)):
            e = get(i, j, tt)
            if e is not None:
                v = v + k * (e if c is None else c * e)
        return v
    for i in range(LI + 1):
        for j in range(LJ + 1):
            if i or j:
                for t in range(i + j + 1):
                    E[(i, j, t)] = step(i, j - 1, t, PB) if j else step(i - 1, j, t, PA)
    return E


class _System:
    """All function pairs p >= q of a molecule and their primitive expansions."""

    def __init__(self, geometry, basis, device, grad=False):
        Z, X = _atoms(geometry)
        self.Z = torch.tensor(Z, dtype=torch.float64, device=device)
        self.X = torch.tensor(X, dtype=torch.float64, device=device, requires_grad=grad)
        fn, prim = [], []                       # functions; primitive shells (atom, shell, l, exponent)
        ns = 0
        for a, z in enumerate(Z):
            for l, e, w in _shells(basis, z):
                ids = list(range(len(prim), len(prim) + len(e)))
                prim += [(a, ns, l, x) for x in e]
                for c in _CART[l]:
                    comp = math.sqrt(_odd(2 * l - 1) / (_odd(2 * c[0] - 1) * _odd(2 * c[1] - 1) * _odd(2 * c[2] - 1)))
                    fn.append((a, c, ids, w * comp))
                ns += 1
        self.fn, self.N = fn, len(fn)
        lmax = max(p[2] for p in prim)
        self.Lp = 2 * lmax
        self.herm = [(t, u, d - t - u) for d in range(self.Lp + 1) for t in range(d, -1, -1) for u in range(d - t, -1, -1)]
        sh = np.array([p[1] for p in prim])
        I, J = np.nonzero(sh[:, None] >= sh[None])
        self.index = np.full((len(prim), len(prim)), -1)
        self.index[I, J] = np.arange(len(I))
        t = lambda v: torch.tensor(np.asarray(v), dtype=torch.float64, device=device)   # noqa: E731
        at = torch.tensor([p[0] for p in prim], device=device)
        ex = t([p[3] for p in prim])
        self.b = ex[J]
        self.p = ex[I] + ex[J]
        A, B = self.X[at[I]], self.X[at[J]]
        self.P = (ex[I][:, None] * A + ex[J][:, None] * B) / self.p[:, None]
        self.K = torch.exp(-ex[I] * ex[J] / self.p * ((A - B) ** 2).sum(1))
        self.E = [_e_table(lmax, lmax + 2, 0.5 / self.p, (self.P - A)[:, x], (self.P - B)[:, x]) for x in range(3)]
        # M: function pairs x (primitive pairs x Hermite functions)
        nh = len(self.herm)
        rows, vals = [], []
        self.pairs = [(f, g) for f in range(self.N) for g in range(f + 1)]
        self.prims = []
        for r, (f, g) in enumerate(self.pairs):
            _, cf, pf, wf = fn[f]
            _, cg, pg, wg = fn[g]
            k = torch.tensor(self.index[np.ix_(pf, pg)].ravel(), device=device)
            w = t(np.outer(wf, wg).ravel()) * self.K[k]
            self.prims.append((k, w))
            for h, tuv in enumerate(self.herm):
                if all(tuv[x] <= cf[x] + cg[x] for x in range(3)):
                    v = w
                    for x in range(3):
                        v = v * self.E[x][(cf[x], cg[x], tuv[x])][k]
                    rows.append(r * len(I) * nh + k * nh + h)
                    vals.append(v)
        self.M = torch.zeros(len(self.pairs) * len(I) * nh, dtype=torch.float64, device=device).index_put(
            (torch.cat(rows),), torch.cat(vals)).view(len(self.pairs), -1)

    def coulomb(self, lo, hi, P):
        """Rows [lo, hi) of H: primitive Hermite pairs against all others."""
        L, nh = 2 * self.Lp, len(self.herm)
        p, q = self.p[lo:hi, None], self.p[None]
        D = P[lo:hi, None] - P[None]
        alpha = p * q / (p + q)
        F = _Boys.apply(alpha * (D * D).sum(-1), L)
        pref = 2 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
        R = _r_table(L, D[..., 0], D[..., 1], D[..., 2], [pref * (-2 * alpha) ** n * F[n] for n in range(L + 1)])
        H = torch.stack([torch.stack([R[(a[0] + b[0], a[1] + b[1], a[2] + b[2], 0)] * (-1.0) ** sum(b)
                                      for b in self.herm], -1) for a in self.herm], 1)   # (rows, nh, all, nh)
        return H.reshape((hi - lo) * nh, -1)

    def chunks(self):
        nh, n = len(self.herm), len(self.p)
        c = max(1, int(1.5e8 / (nh * nh * n)))
        return [(lo, min(n, lo + c)) for lo in range(0, n, c)]

    def eri(self):
        """(pair|pair) of all function pairs p >= q."""
        nh = len(self.herm)
        T = torch.zeros_like(self.M)
        for lo, hi in self.chunks():
            T += self.M[:, lo * nh:hi * nh] @ self.coulomb(lo, hi, self.P)
        return T @ self.M.T

    def unfold(self, V):
        """A tensor over pairs p >= q along the last axis, with both orders."""
        idx = np.zeros((self.N, self.N), dtype=np.int64)
        for r, (f, g) in enumerate(self.pairs):
            idx[f, g] = idx[g, f] = r
        return V[..., torch.tensor(idx, device=V.device)]

    def tensor(self):
        return self.unfold(self.unfold(self.eri()).permute(1, 2, 0))   # symmetric in bra and ket

    def gradient(self, P, W):
        """dE/dX of sum 2 P (T + V) - 2 W S + sum (2 P P - P P) (pq|rs) + V_NN at
        fixed P and W, by automatic differentiation."""
        dev, nh = self.X.device, len(self.herm)
        f, g = (torch.tensor(v, device=dev) for v in zip(*self.pairs))
        d = torch.where(f == g, 1.0, 2.0).to(torch.float64)
        gam = 2 * P[f, g][:, None] * P[f, g][None]
        gam = gam - 0.5 * (P[f][:, f] * P[g][:, g] + P[f][:, g] * P[g][:, f])
        gam = gam * d[:, None] * d[None]
        M, Pc = self.M.detach().requires_grad_(), self.P.detach().requires_grad_()
        for lo, hi in self.chunks():
            H = self.coulomb(lo, hi, Pc)
            ((M[:, lo * nh:hi * nh].T @ (gam @ M)) * H).sum().backward()
        # one-electron part
        zero = self.herm.index((0, 0, 0))
        cub = (math.pi / self.p) ** 1.5
        S = (self.M.view(len(self.pairs), -1, nh)[:, :, zero] * cub).sum(1)
        T = []
        for (k, w), (a, b) in zip(self.prims, self.pairs):
            i, j = self.fn[a][1], self.fn[b][1]
            e = lambda x, dj: self.E[x][(i[x], j[x] + dj, 0)][k] if j[x] + dj >= 0 else 0.0   # noqa: E731
            s = [e(x, 0) for x in range(3)]
            kin = [(2 * j[x] + 1) * self.b[k] * e(x, 0) - 2 * self.b[k] ** 2 * e(x, 2) - 0.5 * j[x] * (j[x] - 1) * e(x, -2)
                   for x in range(3)]
            T.append((w * cub[k] * (kin[0] * s[1] * s[2] + s[0] * kin[1] * s[2] + s[0] * s[1] * kin[2])).sum())
        r = 0.0
        for c in range(len(self.Z)):
            D = self.P - self.X[c]
            F = _Boys.apply(self.p * (D * D).sum(1), self.Lp)
            pref = -self.Z[c] * 2 * math.pi / self.p
            R = _r_table(self.Lp, D[:, 0], D[:, 1], D[:, 2], [pref * (-2 * self.p) ** n * F[n] for n in range(self.Lp + 1)])
            r = r + torch.stack([R[(*h, 0)] for h in self.herm], 1)
        V = self.M @ r.reshape(-1)
        one = (d * (2 * P[f, g] * (torch.stack(T) + V) - 2 * W[f, g] * S)).sum()
        i, j = torch.triu_indices(len(self.Z), len(self.Z), 1, device=dev)
        one = one + (self.Z[i] * self.Z[j] / (self.X[i] - self.X[j]).norm(dim=1)).sum()
        torch.autograd.backward([self.M, self.P, one], [M.grad, Pc.grad, None])
        return self.X.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch" or case["n"] * NBF[case["basis"]] > 60:
        return None
    dev = torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")
    S = _System(_geometry(case, seed), case["basis"], dev, grad=kind == "forces")
    N = S.N
    t = lambda v: torch.tensor(v, device=dev)   # noqa: E731
    if kind == "forces":
        P, F = _density(case, seed), _density(case, seed, 2)
        return -S.gradient(t(P), t(P @ F @ P)).cpu().numpy()
    T = S.tensor()
    if kind == "doeris":
        return T.cpu().numpy()
    if kind == "ao2mo":
        C = t(_orbitals(N, seed))
        for _ in range(4):   # the last index to the front, transformed
            T = (T.reshape(-1, N) @ C).reshape(N, N, N, N).permute(3, 0, 1, 2).contiguous()
        return T.cpu().numpy()
    if kind == "fock":
        D = t(case["scale"] * _density(case, seed))
        J = (T.reshape(N * N, -1) @ D.reshape(-1)).view(N, N)
        K = (T.permute(0, 2, 1, 3).reshape(N * N, -1) @ D.reshape(-1)).view(N, N)   # sum_rs (pr|qs) D_rs
        return (2 * J - K).cpu().numpy()
    if kind == "jk":
        parts = []
        for D in (_density(case, seed), _antisymmetric(case, seed)):
            D = t(D)
            parts.append(((T.reshape(N * N, -1) @ D.T.reshape(-1)).view(N, N).cpu().numpy(),
                          (T.permute(0, 2, 3, 1).reshape(N * N, -1) @ D.T.reshape(-1)).view(N, N).cpu().numpy()))
        # J_pq = sum (pq|rs) P_sr, K_pq = sum (ps|qr) P_sr; the core
        # Hamiltonian in F is left to the comparison with the start
        return {"J": parts[0][0] + 1j * parts[1][0], "K": parts[0][1] + 1j * parts[1][1], "F": None}
    # formPT: every canonical quartet once, with its degeneracy (no screening)
    P = case["scale"] * (_density(case, seed) + 1j * _antisymmetric(case, seed))
    V = T.cpu().numpy()
    G = np.zeros((N, N), dtype=complex)
    f, g = np.tril_indices(N)
    A, B = np.tril_indices(len(f))
    i, j, k, l = f[A], g[A], f[B], g[B]
    e = V[i, j, k, l] * np.where(i == j, 1, 2) * np.where(k == l, 1, 2) * np.where((i == k) & (j == l), 1, 2)
    for r, c, x, y, s in ((i, j, k, l, 1), (k, l, i, j, 1), (i, k, j, l, -0.25), (j, l, i, k, -0.25),
                          (i, l, j, k, -0.25), (k, j, i, l, -0.25)):
        np.add.at(G, (r, c), s * e * P[x, y])
    return G
