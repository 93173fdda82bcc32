"""Rotation runs on excitation levels (csrc/rot_levels.hpp) against one launch per generator
(sweep_mode 2), on pools and generator orders at the edges of the form: unequal spins, lists
longer than one word per thread, one-level runs, spectator orbitals outside the pool, shuffled and
repeated generators, triple excitations, and generalised pools that do not take it.

Tolerance: a sweep of m rotations in another summation order differs by at most a few m units of
rounding relative to the vector's norm (1); 1e-12 covers m up to 600 with a factor of 4.  A gradient
is a sum over the pairs of products bounded by the norms: 1e-12 as well."""
import numpy as np
import pytest

from binsim_amd import autotune as A
from binsim_amd import otf
from binsim_amd.ansatz import ucc_spin_orbitals
from tests.conftest import gpu_vec, host
from tests.helpers import integrals, seeded_vector

pytestmark = pytest.mark.gpu


def _generalised(n):
    return [[2 * p, 2 * q] for p in range(n) for q in range(n) if p > q] + \
           [[2 * p + 1, 2 * q + 1] for p in range(n) for q in range(n) if p > q] + \
           [[2 * 3, 2 * 2 + 1, 2 * 1, 2 * 0 + 1], [2 * 2, 2 * 4 + 1, 2 * 3, 2 * 1 + 1]]


def _window(n, na, nb, lo, hi):
    """UCC excitations among orbitals lo..hi only (the others are spectators)."""
    return [so for so in ucc_spin_orbitals(n, na, nb) if all(lo <= p // 2 < hi for p in so)]


def _triples(n, na):
    return [[2 * a, 2 * b, 2 * c + 1, 2 * i, 2 * j, 2 * k + 1] for a in range(na, n) for b in range(a + 1, n)
            for c in range(na, n) for i in range(na) for j in range(i + 1, na) for k in range(na)][:40]


CASES = [
    ("ucc", 6, 3, 3), ("ucc", 7, 3, 4), ("ucc", 8, 2, 5), ("ucc", 10, 5, 4), ("shuffled", 7, 3, 3),
    ("repeated", 6, 3, 2), ("window", 9, 4, 5), ("triples", 8, 4, 4), ("generalised", 6, 3, 3), ("ucc", 16, 1, 7),
    ("ucc", 16, 7, 1), ("ucc", 14, 2, 7),
]


@pytest.mark.parametrize("kind,n,na,nb", CASES)
def test_level_runs_match_single_launches(torch_cuda, kind, n, na, nb):
    print(f"level runs {kind} n={n} na={na} nb={nb}", flush=True)
    rng = np.random.default_rng(100 * n + 10 * na + nb)
    if kind == "generalised":
        sos = _generalised(n)
    elif kind == "window":
        sos = _window(n, na, nb, 1, n - 1)
    elif kind == "triples":
        sos = ucc_spin_orbitals(n, na, nb)[:60] + _triples(n, na)
    else:
        sos = ucc_spin_orbitals(n, na, nb)
    idx = np.arange(len(sos), dtype=np.int64)
    if kind == "shuffled":
        rng.shuffle(idx)
    elif kind == "repeated":
        idx = np.concatenate([idx, idx[::-1], idx[::2]])
    if len(idx) > 600:
        idx = np.sort(rng.choice(len(idx), 600, replace=False))
    th = rng.uniform(-0.4, 0.4, len(idx))
    _, _, h1, g2 = integrals(n)
    B = otf.HipBasisManager(otf.BasisManager(n, na, nb))
    F = otf.HipOTF_Functions(B, ham=otf.HipOTF.from_integrals(n, h1, g2), pool=otf.HipOTF.from_spin_orbitals(n, sos))
    x, y = seeded_vector(B.dim, n), seeded_vector(B.dim, n + 1)
    got = {}
    try:
        for mode in (2, 0, 4):
            A.set_config(0, {"sweep_mode": mode})
            psi, lam = gpu_vec(torch_cuda, x), torch_cuda.empty(B.dim, dtype=torch_cuda.float64, device="cuda")
            F.vqe_sweep(idx, th, psi, lam)
            fwd = host(psi).copy()
            psi = gpu_vec(torch_cuda, x)
            e, g, _, _ = F.vqe_energy_grad(idx, th, psi, lam)
            l, r = gpu_vec(torch_cuda, x), gpu_vec(torch_cuda, y)
            thd = gpu_vec(torch_cuda, rng.uniform(-0.4, 0.4, len(sos)) if mode == 2 else got[2][5])
            pg = torch_cuda.full((len(sos),), np.nan, dtype=torch_cuda.float64, device="cuda")
            F.batchgrad(l, r, pg, thd)
            got[mode] = (fwd, g, host(psi).copy(), host(pg).copy(), host(lam).copy(), host(thd).copy())
    finally:
        A.set_config(0, {})
    scale = (1.0, max(1.0, np.abs(got[2][1]).max()), 1.0, 1.0, max(1.0, np.linalg.norm(got[2][4])))
    for mode in (0, 4):
        for a, b, s in zip(got[mode], got[2], scale):
            assert np.max(np.abs(a - b)) < 1e-12 * s
    assert np.max(np.abs(got[4][2] - x)) < 1e-12  # the adjoint sweep undoes the forward one
