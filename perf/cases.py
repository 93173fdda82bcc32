"""Performance cases of the on-the-fly FCI / VQE operator library.

Each case is one call (or one solver step) that a user's program makes through binsim_amd: the
sigma build alone, blocks of vectors in the mixed-precision form, the VQE objective with and
without its gradient, the gradient over a whole generator pool, the Davidson inner loop's
subspace operations, and a complete Davidson solve.  Integrals are the seeded synthetic ones of
``binsim_amd.integrals`` (real, 8-fold symmetric, decaying with the orbital distance).

``exact`` evaluates the same quantities with plain torch in float64 from the definitions
(H = sum k_pq E_pq + 1/2 sum (pq|rs) E_pq E_rs; rotations exp(theta (T - T^dagger)) pair by
pair), on the GPU if there is one.
"""
from __future__ import annotations

import ctypes as C
import math
from itertools import combinations

import numpy as np
import torch

from binsim_amd import davidson as D
from binsim_amd import lib as L
from binsim_amd import otf
from binsim_amd.ansatz import ucc_spin_orbitals
from binsim_amd.integrals import chemist_integrals, one_body_layout, reference_layout


def listed():
    return [
        # one H x of a small active space: latency and launches
        dict(name="sigma_8o", kind="sigma", n=8, na=4, nb=4),
        # H x of the everyday active space (ground states, one sigma per Davidson iteration)
        dict(name="sigma_12o", kind="sigma", n=12, na=6, nb=6),
        # an open-shell state: unequal spins, odd row lengths
        dict(name="sigma_13o_5a7b", kind="sigma", n=13, na=5, nb=7),
        # the headline size: 165.6 million determinants
        dict(name="sigma_16o", kind="sigma", n=16, na=8, nb=8),
        # more orbitals, fewer electrons (73.4 million determinants)
        dict(name="sigma_18o_5a5b", kind="sigma", n=18, na=5, nb=5),
        # the mixed-precision Davidson's bulk: four correction vectors through one FP32 sigma
        dict(name="block_fp32_14o", kind="block", n=14, na=7, nb=7, nvec=4),
        # one objective call of a VQE optimisation: energy and all gradients
        dict(name="vqe_gradient_12o", kind="vqe_gradient", n=12, na=6, nb=6),
        dict(name="vqe_gradient_16o", kind="vqe_gradient", n=16, na=8, nb=8),
        # a line-search point: energy only, open shell
        dict(name="vqe_energy_14o_7a6b", kind="vqe_energy", n=14, na=7, nb=6),
        # ADAPT-style selection: the gradient of every generator of the pool on two vectors
        dict(name="pool_gradient_14o", kind="pool_gradient", n=14, na=7, nb=7),
        # one Davidson iteration's vector work on a subspace of 20 vectors
        dict(name="subspace_14o_m20", kind="subspace", n=14, na=7, nb=6, m=20),
        # a whole ground-state solve, FP32 bulk with FP64 refinement
        dict(name="davidson_12o", kind="davidson", n=12, na=6, nb=6),
    ]


# orbital range and largest determinant count of drawn cases, by kind
_RANGES = {
    "sigma": (6, 18, 1.2e8),
    "block": (6, 14, 1.3e7),
    "vqe_gradient": (6, 14, 1.3e7),
    "vqe_energy": (6, 15, 4.2e7),
    "pool_gradient": (6, 14, 1.3e7),
    "subspace": (8, 14, 1.3e7),
    "davidson": (6, 12, 9e5),
}


def draw(rng):
    kind = rng.choice(["sigma", "sigma", "sigma", "block", "vqe_gradient", "vqe_gradient", "vqe_energy",
                       "pool_gradient", "subspace", "davidson"])
    lo, hi, most = _RANGES[kind]
    while True:
        n = rng.randint(lo, hi)
        na, nb = (max(2, min(n - 2, n // 2 + rng.randint(-2, 2))) for _ in range(2))
        if n >= 17:  # few electrons: half filling does not fit the range
            na, nb = rng.randint(3, 5), rng.randint(3, 5)
        dim = math.comb(n, na) * math.comb(n, nb)
        if dim <= most and _flops_sigma(n, na, nb) <= 1.9e12 / (1 if n <= 16 else 2):
            break
    case = dict(kind=kind, n=n, na=na, nb=nb)
    if kind == "block":
        case["nvec"] = rng.randint(1, 8 if dim < 3e6 else 4)
    if kind == "subspace":
        case["m"] = rng.randint(1, 23)
    return case


# -----------------------------------------------------------------------------------------
# what a user's program holds before the call, and the call
# -----------------------------------------------------------------------------------------
def _unit_vectors(dim, count, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for _ in range(count):
        v = torch.rand(dim, dtype=torch.float64, device="cuda", generator=g).mul_(2.0).sub_(1.0)
        out.append(v.div_(torch.linalg.vector_norm(v)))
    return out


def _thetas(count, seed):
    return np.random.default_rng(seed).uniform(-0.1, 0.1, count)


def prepare(case, seed):
    n, na, nb, kind = case["n"], case["na"], case["nb"], case["kind"]
    s = {"kind": kind}
    if kind == "subspace":
        dim, m = math.comb(n, na) * math.comb(n, nb), case["m"]
        vs, av, coef = _subspace_inputs(dim, m, seed)
        s.update(dim=dim, m=m, V=vs, AV=av, coef=coef, e=-1.5, shift=1e-4,
                 diags=_unit_vectors(dim, 1, seed + 7)[0].mul_(math.sqrt(dim)), t=torch.empty_like(vs[0]),
                 Vp=D._pp(vs), AVp=D._pp(av), col=np.zeros(m))
        return s
    h, eri = chemist_integrals(n, seed)
    B = otf.HipBasisManager(otf.BasisManager(n, na, nb))
    ham = otf.HipOTF.from_integrals(n, one_body_layout(h), reference_layout(eri))
    pool = None
    if kind in ("vqe_gradient", "vqe_energy", "pool_gradient"):
        sos = ucc_spin_orbitals(n, na, nb)
        pool = otf.HipOTF.from_spin_orbitals(n, sos)
        s["thetas"], s["idxs"] = _thetas(len(sos), seed), np.arange(len(sos), dtype=np.int64)
    s["F"] = otf.HipOTF_Functions(B, ham=None if kind == "pool_gradient" else ham, pool=pool)
    if kind == "sigma":
        s["x"] = _unit_vectors(B.dim, 1, seed)[0]
        s["y"] = torch.empty_like(s["x"])
    elif kind == "block":
        s["x"] = _unit_vectors(B.dim, case["nvec"], seed)
        s["y"] = [torch.empty_like(v) for v in s["x"]]
    elif kind in ("vqe_gradient", "vqe_energy"):
        s["ref"] = torch.zeros(B.dim, dtype=torch.float64, device="cuda")
        s["ref"][0] = 1.0  # the Hartree-Fock determinant
        s["psi"], s["lam"] = torch.empty_like(s["ref"]), torch.empty_like(s["ref"])
    elif kind == "pool_gradient":
        s["l"], s["r"] = _unit_vectors(B.dim, 2, seed)
        s["theta_dev"] = torch.from_numpy(s["thetas"]).to("cuda")
        s["grads"] = torch.empty_like(s["theta_dev"])
    elif kind == "davidson":
        s["ham"], s["basis"] = ham, B
    return s


def run(s):
    kind = s["kind"]
    if kind == "sigma":
        s["F"].hvec(s["x"], s["y"])
        return s["y"]
    if kind == "block":
        s["F"].hvec_block(s["x"], s["y"], precision=1)
        return s["y"]
    if kind == "vqe_gradient":
        s["psi"].copy_(s["ref"])
        e, g, d2, n2 = s["F"].vqe_energy_grad(s["idxs"], s["thetas"], s["psi"], s["lam"])
        return {"energy": e, "gradient": g, "variance": d2, "norm2": n2, "psi": s["psi"]}
    if kind == "vqe_energy":
        s["psi"].copy_(s["ref"])
        e, d2, n2 = s["F"].vqe_energy(s["idxs"], s["thetas"], s["psi"], s["lam"])
        return {"energy": e, "variance": d2, "norm2": n2, "psi": s["psi"], "h_psi": s["lam"]}
    if kind == "pool_gradient":
        s["F"].batchgrad(s["l"], s["r"], s["grads"], s["theta_dev"])
        return s["grads"]
    if kind == "subspace":
        lib, dim, m, t = L.load(), s["dim"], s["m"], s["t"].data_ptr()
        c = s["coef"].ctypes.data_as(L._dp)
        r = lib.build_ritz_and_residual_f64(dim, m, c, s["e"], s["Vp"], s["AVp"], t)
        lib.apply_preconditioner_inplace_f64(dim, t, s["diags"].data_ptr(), s["e"], s["shift"])
        o = lib.mgs_orthogonalize_f64(dim, m, s["Vp"], t)
        lib.inplace_normalize_f64(dim, t)
        lib.compute_heff_col_f64(dim, m, s["Vp"], s["AV"][m - 1].data_ptr(), s["col"].ctypes.data_as(L._dp))
        return {"residual": r, "norm": o, "vector": s["t"], "column": s["col"]}
    e, _, _ = D.solve(s["basis"], s["ham"], nroots=1, mixed=True, tol=1e-8)
    return e


def _subspace_inputs(dim, m, seed):
    """m orthonormal vectors, m images, Ritz coefficients (host)."""
    vs = _unit_vectors(dim, m, seed)
    for i in range(m):  # orthonormalise
        for _ in range(2):
            for j in range(i):
                vs[i].sub_(vs[j] * torch.dot(vs[j], vs[i]))
        vs[i].div_(torch.linalg.vector_norm(vs[i]))
    av = _unit_vectors(dim, m, seed + 1)
    c = np.random.default_rng(seed + 2).normal(size=m)
    return vs, av, np.ascontiguousarray(c / np.linalg.norm(c))


# -----------------------------------------------------------------------------------------
# bytes and operations a pass cannot do without
# -----------------------------------------------------------------------------------------
def _flops_sigma(n, na, nb):
    sa, sb = na * (n - na), nb * (n - nb)
    da, db = (math.comb(k, 2) * math.comb(n - k, 2) for k in (na, nb))
    return 2.0 * math.comb(n, na) * math.comb(n, nb) * (1 + sa + sb + da + db + sa * sb)


def _rotation_pairs(n, na, nb):
    """Coupled determinant pairs summed over the UCC singles-doubles list."""
    def per_rank(k):
        return [math.comb(k, r) * math.comb(n - k, r) * (math.comb(n - 2 * r, k - r) if n >= 2 * r else 0)
                for r in range(3)]
    a, b = per_rank(na), per_rank(nb)
    return float(sum(a[i] * b[j] for i in range(3) for j in range(3 - i) if i + j > 0))


def work(case):
    n, na, nb, kind = case["n"], case["na"], case["nb"], case["kind"]
    dim = math.comb(n, na) * math.comb(n, nb)
    if kind == "sigma":
        return {"bytes": 16.0 * dim, "flops": _flops_sigma(n, na, nb)}
    if kind == "block":
        return {"bytes": 16.0 * dim * case["nvec"], "flops": _flops_sigma(n, na, nb) * case["nvec"]}
    if kind == "subspace":
        m = case["m"]
        return {"bytes": 8.0 * dim * (2 * m + 2), "flops": 2.0 * dim * 5 * m}
    pairs = _rotation_pairs(n, na, nb)
    if kind == "vqe_energy":
        return {"bytes": 24.0 * dim, "flops": 6.0 * pairs + _flops_sigma(n, na, nb)}
    if kind == "vqe_gradient":
        return {"bytes": 32.0 * dim, "flops": 26.0 * pairs + _flops_sigma(n, na, nb)}
    if kind == "pool_gradient":
        return {"bytes": 16.0 * dim, "flops": 8.0 * pairs}
    # a solve: at least the sigma builds of a few dozen iterations
    return {"bytes": 30 * 16.0 * dim, "flops": 30 * _flops_sigma(n, na, nb)}


# -----------------------------------------------------------------------------------------
# the same quantities in plain float64 torch
# -----------------------------------------------------------------------------------------
def _popcount(a):
    a = a.copy()
    c = np.zeros_like(a)
    while a.any():
        c += a & 1
        a >>= 1
    return c


class _Space:
    """Determinant strings of one spin in ascending order."""

    def __init__(self, n, k):
        self.n = n
        self.s = np.sort(np.array([sum(1 << p for p in c) for c in combinations(range(n), k)], dtype=np.int64))

    def singles(self, p, q):
        """(destination, source, sign) of a+_p a_q over the strings."""
        s = self.s
        j = np.nonzero(((s >> q) & 1 == 1) & ((p == q) | ((s >> p) & 1 == 0)))[0]
        src = s[j]
        par = _popcount(src & ((1 << q) - 1)) + _popcount((src ^ (1 << q)) & ((1 << p) - 1))
        dst = (src ^ (1 << q)) | (1 << p)
        return np.searchsorted(s, dst), j, 1.0 - 2.0 * (par & 1)


def _dev(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


class _Reference:
    def __init__(self, n, na, nb):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.n, self.A, self.B = n, _Space(n, na), _Space(n, nb)
        self.NA, self.NB = len(self.A.s), len(self.B.s)

    def gauge(self, x):
        """Signs between interleaved spin-orbitals (2p alpha, 2p+1 beta) and all alpha first."""
        m = np.zeros(self.NA, dtype=np.int64)
        for p in range(self.n):
            m ^= np.where((self.A.s >> p) & 1 == 1, (1 << p) - 1, 0)
        step = max(1, (1 << 26) // self.NB)
        for a0 in range(0, self.NA, step):
            par = _popcount(m[a0:a0 + step, None] & self.B.s[None, :]) & 1
            x[a0:a0 + step] *= _dev(1.0 - 2.0 * par, self.dev)
        return x

    def sigma(self, x, h, eri):
        n, n2, dev = self.n, self.n * self.n, self.dev
        X = self.gauge(x.reshape(self.NA, self.NB).clone())
        k = torch.from_numpy(np.ascontiguousarray(h - 0.5 * np.einsum("prrq->pq", eri)).reshape(-1)).to(dev)
        g = torch.from_numpy(0.5 * eri.reshape(n2, n2)).to(dev)
        ea = [[_dev(t, dev) for t in self.A.singles(p, q)] for p in range(n) for q in range(n)]
        eb = [[_dev(t, dev) for t in self.B.singles(p, q)] for p in range(n) for q in range(n)]
        out = torch.zeros_like(X)
        nc = int(max(1, min(self.NB, 4e9 // (n2 * self.NA * 8))))
        for c0 in range(0, self.NB, nc):
            c1 = min(self.NB, c0 + nc)
            d = torch.zeros((n2, self.NA, c1 - c0), dtype=torch.float64, device=dev)
            for i in range(n2):
                dst, src, sg = ea[i]
                d[i].index_add_(0, dst, X[src, c0:c1] * sg[:, None])
                dst, src, sg = eb[i]
                ok = (dst >= c0) & (dst < c1)
                d[i].index_add_(1, dst[ok] - c0, X[:, src[ok]] * sg[ok][None, :])
            flat = d.reshape(n2, -1)
            out[:, c0:c1] += (k[None, :] @ flat).reshape(self.NA, c1 - c0)
            gd = (g @ flat).reshape(n2, self.NA, c1 - c0)
            del d, flat
            for i in range(n2):
                dst, src, sg = ea[i]
                out[:, c0:c1].index_add_(0, dst, gd[i][src] * sg[:, None])
                dst, src, sg = eb[i]
                ok = (src >= c0) & (src < c1)
                out.index_add_(1, dst[ok], gd[i][:, src[ok] - c0] * sg[ok][None, :])
            del gd
        return self.gauge(out).reshape(-1)

    def pairs(self, so):
        """Row and column indices of the determinants T = a+.. a.. acts on, of their images, and
        T's sign (rows x columns, a product of one factor per spin)."""
        half = len(so) // 2
        out = []
        for spin, sp in ((0, self.A), (1, self.B)):
            cre = sum(1 << (p >> 1) for p in so[:half] if p & 1 == spin)
            ann = sum(1 << (p >> 1) for p in so[half:] if p & 1 == spin)
            u = np.nonzero(((sp.s & ann) == ann) & ((sp.s & cre) == 0))[0]
            s = sp.s[u].copy()
            par = np.zeros_like(s)
            for p in reversed(so):  # rightmost operator first
                q = p >> 1
                # orbitals of this spin that precede spin-orbital p
                m = (1 << q) - 1 if not (p & 1 == 1 and spin == 0) else (2 << q) - 1
                par += _popcount(s & m)
                if p & 1 == spin:
                    s ^= 1 << q
            out.append((_dev(u, self.dev), _dev(np.searchsorted(sp.s, s), self.dev),
                        _dev(1.0 - 2.0 * (par & 1), self.dev)))
        return out

    def rotate(self, x, pr, theta):
        (ua, wa, sa), (ub, wb, sb) = pr
        t = sa[:, None] * sb[None, :]
        xu, xw = x[ua[:, None], ub[None, :]], x[wa[:, None], wb[None, :]]
        c, s = math.cos(theta), math.sin(theta)
        x[ua[:, None], ub[None, :]] = c * xu - s * t * xw
        x[wa[:, None], wb[None, :]] = s * t * xu + c * xw

    def derivative(self, left, right, pr, theta):
        """<left| G e^{theta G} |right> restricted to the pairs' determinants."""
        (ua, wa, sa), (ub, wb, sb) = pr
        t = sa[:, None] * sb[None, :]
        lu, lw = left[ua[:, None], ub[None, :]], left[wa[:, None], wb[None, :]]
        ru, rw = right[ua[:, None], ub[None, :]], right[wa[:, None], wb[None, :]]
        c, s = math.cos(theta), math.sin(theta)
        return (lu * (-s * ru + c * t * rw) + lw * (-s * rw - c * t * ru)).sum()


def exact(case, seed):
    n, na, nb, kind = case["n"], case["na"], case["nb"], case["kind"]
    dim = math.comb(n, na) * math.comb(n, nb)
    if kind == "davidson" or (kind.startswith("vqe") and dim > 2e7) or (kind == "sigma" and dim > 2e8):
        return None
    if kind == "subspace":
        m = case["m"]
        vs, av, c = _subspace_inputs(dim, m, seed)
        t = torch.zeros_like(vs[0])
        for j in range(m):
            t += c[j] * (av[j] + 1.5 * vs[j])
        r = float(torch.linalg.vector_norm(t))
        d = _unit_vectors(dim, 1, seed + 7)[0].mul_(math.sqrt(dim)) + 1.5
        t /= torch.where(d.abs() < 1e-4, torch.copysign(torch.full_like(d, 1e-4), d), d)
        for j in range(m):
            t -= torch.dot(vs[j], t) * vs[j]
        o = float(torch.linalg.vector_norm(t))
        return {"residual": r, "norm": o, "vector": t / o,
                "column": np.array([float(torch.dot(v, av[m - 1])) for v in vs])}
    R = _Reference(n, na, nb)
    h, eri = chemist_integrals(n, seed)
    if kind == "sigma":
        return R.sigma(_unit_vectors(dim, 1, seed)[0], h, eri)
    if kind == "block":
        return [R.sigma(x, h, eri) for x in _unit_vectors(dim, case["nvec"], seed)]
    sos = ucc_spin_orbitals(n, na, nb)
    th = _thetas(len(sos), seed)
    pr = {}  # pair lists of a generator (at most one kept at a time for the large systems)

    def pairs(i):
        if i not in pr:
            if dim > 1e6:
                pr.clear()
            pr[i] = R.pairs(sos[i])
        return pr[i]

    if kind == "pool_gradient":
        l, r = (v.reshape(R.NA, R.NB) for v in _unit_vectors(dim, 2, seed))
        return torch.stack([R.derivative(l, r, pairs(i), th[i]) for i in range(len(sos))])
    psi = torch.zeros((R.NA, R.NB), dtype=torch.float64, device=R.dev)
    psi[0, 0] = 1.0
    for i in range(len(sos)):
        R.rotate(psi, pairs(i), th[i])
    lam = R.sigma(psi, h, eri).reshape(R.NA, R.NB)
    n2 = float((psi * psi).sum())
    e = float((psi * lam).sum()) / n2
    d2 = max(0.0, float((lam * lam).sum()) / n2 - e * e)
    if kind == "vqe_energy":
        return {"energy": e, "variance": d2, "norm2": n2, "psi": psi.reshape(-1), "h_psi": lam.reshape(-1)}
    g = [None] * len(sos)
    for i in reversed(range(len(sos))):
        R.rotate(psi, pairs(i), -th[i])
        g[i] = R.derivative(psi, lam, pairs(i), th[i]) * (2.0 / n2)
        R.rotate(lam, pairs(i), -th[i])
    return {"energy": e, "gradient": torch.stack(g), "variance": d2, "norm2": n2, "psi": psi.reshape(-1)}
