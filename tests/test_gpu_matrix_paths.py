"""The default (matrix-core) sigma kernels and the Davidson vector kernels at the edges of their
forms.

* FP64 sigma by default against the same sigma on the chunked alpha-beta kernel and the row SpMM of
  one string per wave (ab_kernel 3, rs_block 0): every orbital count's row tiles, the class split
  (16 orbitals / 8 beta, 17, 18), string counts that are no multiple of 8 or 16, odd row lengths, one
  beta string, and source lists in 1, 2 and 4 ranges.  Both add the same products in FP64 in another
  order: at most some thousand terms per element, so 1e-12 of the norm.
* FP32 block sigma in blocks of 4 strings against blocks of 8: the same sums in the same order, so
  the same bits.
* Gram-Schmidt, norms and subspace dot products against NumPy: a sum of N products is off by at most
  N / 2 units of rounding relative to the norms and, added in blocks, by far less: 1e-13."""
import numpy as np
import pytest

from binsim_amd import autotune as AT
from binsim_amd import lib as L
from tests.conftest import gpu_vec, host
from tests.helpers import rel_err, seeded_vector
from tests.test_gpu_davidson import _pp
from tests.test_gpu_sigma import _dev

pytestmark = pytest.mark.gpu

SIGMA = [(2, 1, 1), (4, 2, 1), (5, 3, 2), (7, 3, 4), (9, 4, 5), (10, 1, 9), (11, 5, 3), (13, 2, 6), (13, 6, 2),
         (14, 7, 1), (15, 2, 7), (15, 7, 2), (16, 6, 1), (16, 8, 1), (16, 1, 8), (16, 2, 7), (17, 2, 5), (17, 1, 6),
         (17, 5, 1), (18, 2, 5), (18, 5, 1), (18, 1, 4)]


@pytest.mark.parametrize("n,na,nb", SIGMA)
def test_default_sigma_matches_general_kernels(torch_cuda, n, na, nb):
    print(f"default sigma n={n} na={na} nb={nb}", flush=True)
    B, H, F = _dev(n, na, nb)
    x = gpu_vec(torch_cuda, seeded_vector(B.dim, 31 * n + na))
    y, ref = torch_cuda.empty_like(x), torch_cuda.empty_like(x)
    F.hvec(x, y)
    saved = AT.get_config(AT.FP64)
    try:
        AT.set_config(AT.FP64, dict(saved, ab_kernel=3, rs_block=0, rs_passes=1))
        F.hvec(x, ref)
    finally:
        AT.set_config(AT.FP64, saved)
    assert rel_err(host(y), host(ref)) < 1e-12


@pytest.mark.parametrize("n,na,nb,k", [(5, 2, 3, 1), (9, 4, 5, 3), (10, 5, 2, 4), (12, 6, 6, 2), (13, 6, 1, 5)])
def test_fp32_blocks_of_four_strings_keep_their_bits(torch_cuda, n, na, nb, k):
    B, H, F = _dev(n, na, nb)
    xs = [gpu_vec(torch_cuda, seeded_vector(B.dim, 40 + j)) for j in range(k)]
    ys, ref = [torch_cuda.empty_like(x) for x in xs], [torch_cuda.empty_like(x) for x in xs]
    F.hvec_block(xs, ys, precision=1)
    saved = AT.get_config(AT.FP32)
    try:
        AT.set_config(AT.FP32, dict(saved, rs_block=8, rs_passes=1))  # (one pass is the default's too)
        F.hvec_block(xs, ref, precision=1)
    finally:
        AT.set_config(AT.FP32, saved)
    assert all(torch_cuda.equal(y, r) for y, r in zip(ys, ref))


@pytest.mark.parametrize("N", [1, 63, 257, 4099, 524289, 1200007])
@pytest.mark.parametrize("m", [0, 1, 2, 23])
def test_subspace_kernels_at_odd_sizes(torch_cuda, N, m):
    rng = np.random.default_rng(N + m)
    m = min(m, N)
    V = np.linalg.qr(rng.standard_normal((N, m)))[0].T.copy() if m else np.empty((0, N))
    t = rng.standard_normal(N) + (3.0 * V.sum(0) if m else 0.0)
    Vd, td = [gpu_vec(torch_cuda, v) for v in V], gpu_vec(torch_cuda, t)
    pp = _pp(Vd)
    lib, scale = L.load(), np.linalg.norm(t)
    if m:
        col = np.empty(m)
        lib.compute_heff_col_f64(N, m, pp, td.data_ptr(), col.ctypes.data_as(L._dp))
        assert np.max(np.abs(col - V @ t)) < 1e-13 * scale
    want = t.copy()
    for v in V:
        want -= (v @ want) * v
    got = lib.mgs_orthogonalize_f64(N, m, pp, td.data_ptr())
    assert np.max(np.abs(host(td) - want)) < 1e-13 * scale
    assert abs(got - np.linalg.norm(want)) < 1e-13 * scale
    if m < N:
        assert abs(lib.inplace_normalize_f64(N, td.data_ptr()) - got) < 1e-13 * scale
        assert abs(np.linalg.norm(host(td)) - 1.0) < 1e-13
