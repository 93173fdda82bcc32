"""hipotf_hvec_noalloc after a preparation and a first call under other launch choices than its own
(tests/test_zz_no_alloc.py keeps them).  The same sums in another order: 1e-12 of the norm."""
import pytest

import binsim_amd.lib as L
from binsim_amd import autotune as AT
from binsim_amd import otf
from tests.conftest import gpu_vec, host
from tests.helpers import integrals, rel_err, seeded_vector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,na,nb", [(8, 4, 4), (12, 5, 6), (14, 7, 2)])
@pytest.mark.parametrize("before", [dict(ab_kernel=1), dict(deterministic=1), dict(rs_passes=2), {}])
@pytest.mark.parametrize("after", [dict(rs_passes=4), {}])
def test_first_call_under_other_choices(torch_cuda, n, na, nb, before, after):
    print(f"n={n} na={na} nb={nb} {before} {after}", flush=True)
    _check(torch_cuda, n, na, nb, before, after)


def _check(torch, n, na, nb, before, after):
    saved = AT.get_config(AT.FP64)
    _, _, h1, g2 = integrals(n)
    B = otf.HipBasisManager(otf.BasisManager(n, na, nb))
    x = gpu_vec(torch, seeded_vector(B.dim, n))
    y, ref = torch.full_like(x, float("nan")), torch.empty_like(x)
    try:
        AT.set_config(AT.FP64, dict(saved, **before))
        H = otf.HipOTF.from_integrals(n, h1, g2)
        F = otf.HipOTF_Functions(B, ham=H)  # hipotf_prepare
        F.hvec(x, ref)
        AT.set_config(AT.FP64, dict(saved, **after))
        assert L.load().hipotf_hvec_noalloc(B.ptr, H.ptr, x.data_ptr(), y.data_ptr()) == 0, L.last_error()
        torch.cuda.synchronize()
        F.hvec(x, ref)
    finally:
        AT.set_config(AT.FP64, saved)
    assert rel_err(host(y), host(ref)) < 1e-12
