"""The Davidson driver and its vector operations at the limits of what they take."""
import numpy as np
import pytest

from binsim_amd import davidson as D
from binsim_amd import lib as L
from tests.conftest import gpu_vec, host
from tests.helpers import seeded_vector
from tests.test_gpu_sigma import _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_guess_that_is_not_finite_is_an_error(torch_cuda, mixed, bad):
    """Not a converged solve with NaN energies."""
    B, H, F = _dev(6, 3, 3)
    x = seeded_vector(B.dim, 3)
    x[7] = bad
    with pytest.raises(L.HipOTFError):
        D.solve(B, H, nroots=1, mixed=mixed, guess=gpu_vec(torch_cuda, x))


@pytest.mark.parametrize("m", [64, 65, 130])
def test_subspace_matrix_beyond_64_vectors(torch_cuda, m):
    """Dot products of unit vectors of 500 elements: off by a few units of rounding, 1e-13."""
    N, lib = 500, L.load()
    V = np.stack([seeded_vector(N, 10 + j) for j in range(m)])
    Vd = [gpu_vec(torch_cuda, v) for v in V]
    t = seeded_vector(N, 5)
    td, col, heff = gpu_vec(torch_cuda, t), np.full(m, np.nan), np.zeros(m * m)
    lib.compute_heff_col_f64(N, m, D._pp(Vd), td.data_ptr(), col.ctypes.data_as(L._dp))
    assert np.max(np.abs(col - V @ t)) < 1e-13
    if m < 130:
        lib.rebuild_heff_f64(N, m, D._pp(Vd), D._pp(Vd), heff.ctypes.data_as(L._dp), m)
        assert np.max(np.abs(heff.reshape(m, m) - V @ V.T)) < 1e-13


@pytest.mark.parametrize("N", [5, 1030, 300001])
def test_gram_schmidt_against_a_subspace_that_holds_the_vector(torch_cuda, N):
    """Step by step as written: each projection sees the vector as the steps before left it.  Unit
    vectors, three steps of a few units of rounding: 1e-13."""
    a, b, t = (seeded_vector(N, 20 + j) for j in range(3))
    ad, bd, td = (gpu_vec(torch_cuda, v) for v in (a, b, t))
    want = t.copy()
    for v in (a, want, b):  # (want itself: the second vector of the subspace)
        want -= (v @ want) * v
    got = L.load().mgs_orthogonalize_f64(N, 3, D._pp([ad, td, bd]), td.data_ptr())
    assert np.max(np.abs(host(td) - want)) < 1e-13
    assert abs(got - np.linalg.norm(want)) < 1e-13


def test_tables_come_before_the_memory_check(torch_cuda):
    """18 orbitals / 6 + 6 with 64 subspace vectors: more than the card holds, refused before anything is
    computed.  The FP32 tables of the mixed solve (over 100 MB) are then there: their memory was not
    counted as free."""
    B, H, F = _dev(18, 6, 6)
    before = torch_cuda.cuda.mem_get_info()[0]
    with pytest.raises(L.HipOTFError, match="davidson: needs"):
        D.solve(B, H, nroots=1, mixed=True, maxspace=64)
    assert before - torch_cuda.cuda.mem_get_info()[0] > 100 << 20
