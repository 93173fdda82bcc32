"""One infinity or NaN in the source of a sigma: with the row tables in blocks of 16 strings (from 2,048
strings of a spin, FP64) it reaches the determinants that one row at a time (rs_block 0) lets it reach
and no others, for that call only; (blocks of 8
reach the rest of their blocks, so the other spin here has as many strings or one)."""
import numpy as np
import pytest

from binsim_amd import autotune as AT
from tests.conftest import gpu_vec, host
from tests.helpers import rel_err, seeded_vector
from tests.test_gpu_sigma import _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,na,nb", [(14, 7, 7), (15, 5, 0), (15, 15, 5), (18, 4, 18)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_reach_of_an_element_that_is_not_finite(torch_cuda, n, na, nb, bad):
    print(f"not finite n={n} na={na} nb={nb} {bad}", flush=True)
    B, H, F = _dev(n, na, nb)
    x = seeded_vector(B.dim, n)
    xd = gpu_vec(torch_cuda, x)
    y, z, ref = (torch_cuda.empty_like(xd) for _ in range(3))
    F.hvec(xd, ref)
    xd[B.dim // 3 * 2 + 5] = bad
    F.hvec(xd, y)
    saved = AT.get_config(AT.FP64)
    try:
        AT.set_config(AT.FP64, dict(saved, rs_block=0, rs_passes=1))
        F.hvec(xd, z)
    finally:
        AT.set_config(AT.FP64, saved)
    y, z = host(y), host(z)
    ok = np.isfinite(z)
    assert 0 < ok.sum() < B.dim
    assert np.array_equal(np.isfinite(y), ok)
    assert rel_err(y[ok], z[ok]) < 1e-12
    xd = gpu_vec(torch_cuda, x)  # a finite source after it
    y = torch_cuda.empty_like(xd)
    F.hvec(xd, y)
    assert rel_err(host(y), host(ref)) < 1e-12
