"""Which rotation runs go to excitation levels (csrc/rot.hip plan_sweep, csrc/rot_levels.hpp), against
one launch per generator (sweep_mode 2): pools on a window of the orbitals (blocks of a few elements,
many to a bin), run lengths on both sides of the rules, alpha singles in segments with and without a
plan, and runs cut where their gradient partials would pass the limit.

Tolerance: m rotations in another order of additions differ by a few m units of rounding relative to
the norm 1; 1e-12 covers m up to 1,000 with a factor of 4, 4e-12 the 2,352 of the longest case."""
import time

import numpy as np
import pytest

from binsim_amd import autotune as A
from binsim_amd import otf
from binsim_amd.ansatz import ucc_spin_orbitals
from tests.conftest import gpu_vec, host
from tests.helpers import integrals, seeded_vector

pytestmark = pytest.mark.gpu


def _functions(n, na, nb, sos):
    _, _, h1, g2 = integrals(n)
    B = otf.HipBasisManager(otf.BasisManager(n, na, nb))
    return B, otf.HipOTF_Functions(B, ham=otf.HipOTF.from_integrals(n, h1, g2),
                                   pool=otf.HipOTF.from_spin_orbitals(n, sos))


def _window(n, na, nb, lo, hi):
    return [so for so in ucc_spin_orbitals(n, na, nb) if all(lo <= p // 2 < hi for p in so)]


def _spins(so):
    """(alpha, beta) excitation ranks"""
    a = sum(p % 2 == 0 for p in so) // 2
    return a, len(so) // 2 - a


def _compare(torch, n, na, nb, sos, modes=(0, 4), tol=1e-12):
    idx = np.arange(len(sos), dtype=np.int64)
    th = np.random.default_rng(n + len(sos)).uniform(-0.4, 0.4, len(sos))
    B, F = _functions(n, na, nb, sos)
    x, y = seeded_vector(B.dim, n), seeded_vector(B.dim, n + 1)
    got = {}
    try:
        for mode in (2, *modes):
            A.set_config(0, {"sweep_mode": mode})
            psi, lam = gpu_vec(torch, x), torch.empty(B.dim, dtype=torch.float64, device="cuda")
            F.vqe_sweep(idx, th, psi, lam)
            fwd = host(psi).copy()
            psi = gpu_vec(torch, x)
            g = F.vqe_energy_grad(idx, th, psi, lam)[1]
            pg = torch.full((len(sos),), np.nan, dtype=torch.float64, device="cuda")
            F.batchgrad(gpu_vec(torch, x), gpu_vec(torch, y), pg, gpu_vec(torch, th))
            got[mode] = (fwd, g, host(psi).copy(), host(pg).copy())
    finally:
        A.set_config(0, {})
    scale = (1.0, max(1.0, np.abs(got[2][1]).max()), 1.0, 1.0)
    for mode in modes:
        for a, b, s in zip(got[mode], got[2], scale):
            assert np.max(np.abs(a - b)) < tol * s


@pytest.mark.parametrize("n,na,nb,lo,hi", [(10, 5, 5, 4, 6), (11, 5, 6, 3, 7), (12, 6, 6, 4, 8), (12, 5, 7, 2, 9),
                                           (13, 6, 3, 4, 8), (13, 3, 6, 1, 8)])
def test_pools_on_a_window_of_the_orbitals(torch_cuda, n, na, nb, lo, hi):
    print(f"window n={n} na={na} nb={nb} {lo}..{hi}", flush=True)
    sos = _window(n, na, nb, lo, hi)
    assert sos
    _compare(torch_cuda, n, na, nb, sos[:120] + sos[120:][-120:])


@pytest.mark.parametrize("m", [1, 2, 3, 7, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("n,na,nb", [(8, 4, 4), (9, 3, 4)])
def test_run_lengths_around_the_rules(torch_cuda, n, na, nb, m):
    """m beta excitations of one rank after each alpha single, with and without the alpha single
    itself, and m of one spin alone between others."""
    u = ucc_spin_orbitals(n, na, nb)
    sos = []
    for p in [so for so in u if _spins(so) == (1, 0)][:4]:
        mixed = [so for so in u if _spins(so) == (1, 1) and so[0] == p[0] and so[2] == p[1]]
        sos += [p] + mixed[:m] + [so for so in u if _spins(so) == (0, 2)][:m] + mixed[-m:]
        sos += [so for so in u if _spins(so) == (0, 1)][:m] + [so for so in u if _spins(so) == (2, 0)][:m]
    _compare(torch_cuda, n, na, nb, sos[:240])


def test_alpha_singles_of_a_generalised_pool(torch_cuda):
    """Alpha singles before mixed generators that have no level plan."""
    n = 7
    sos = []
    for p in range(1, 4):
        sos.append([2 * p, 0])
        sos += [[2 * p, 2 * r + 1, 0, 2 * t + 1] for r in range(n) for t in range(r)]
    sos += [[2 * p + 1, 2 * q + 1] for p in range(n) for q in range(p)]
    _compare(torch_cuda, n, 3, 3, sos)


def test_run_longer_than_its_gradient_partials_allow(torch_cuda):
    """8,008 rows in two bins: at most 2,095 generators to a launch."""
    doubles = [so for so in ucc_spin_orbitals(16, 6, 8) if _spins(so) == (0, 2)]
    assert len(doubles) == 784
    _compare(torch_cuda, 16, 6, 8, doubles * 3, modes=(4,), tol=4e-12)


@pytest.mark.parametrize("lo,hi", [(6, 8), (5, 9)])
def test_window_pools_take_no_longer_than_whole_rows(torch_cuda, lo, hi):
    """14 orbitals: with bins of the largest block alone the level runs took 14 to 26 times as long as
    the segments with staged rows (sweep_mode 3); a factor of 3 is far from both."""
    sos = _window(14, 7, 7, lo, hi)
    B, F = _functions(14, 7, 7, sos)
    x = gpu_vec(torch_cuda, seeded_vector(B.dim, 1))
    lam, idx, th = torch_cuda.empty_like(x), np.arange(len(sos), dtype=np.int64), np.full(len(sos), 0.01)
    took = {}
    try:
        for mode in (3, 0):
            A.set_config(0, {"sweep_mode": mode})
            runs = []
            for _ in range(6):
                torch_cuda.cuda.synchronize()
                t = time.perf_counter()
                F.vqe_sweep(idx, th, x, lam)
                torch_cuda.cuda.synchronize()
                runs.append(time.perf_counter() - t)
            took[mode] = min(runs)
    finally:
        A.set_config(0, {})
    assert took[0] < 3.0 * took[3]


def test_no_interleaved_copy_on_levels_alone(torch_cuda):
    """14 orbitals / 7 + 7: the adjoint sweep of a particle-hole pool has no pair segment, so the
    interleaved (l, r) copy (16 bytes per determinant) is not allocated.  Its other buffers (gradient
    partials of some 100 MB) are smaller than that copy."""
    sos = ucc_spin_orbitals(14, 7, 7)
    B, F = _functions(14, 7, 7, sos)
    x = gpu_vec(torch_cuda, seeded_vector(B.dim, 1))
    y, idx, th = torch_cuda.empty_like(x), np.arange(len(sos), dtype=np.int64), np.full(len(sos), 0.01)
    F.hvec(x, y)
    F.vqe_sweep(idx, th, x, y)
    torch_cuda.cuda.synchronize()
    before = torch_cuda.cuda.mem_get_info()[0]
    F.vqe_energy_grad(idx, th, x, y)
    torch_cuda.cuda.synchronize()
    assert before - torch_cuda.cuda.mem_get_info()[0] < 16 * B.dim
