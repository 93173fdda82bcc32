"""The row tables of the same-spin products as the device builds them (csrc/tables.hip): blocks of 4, 8
and 16 strings and the matrix-core tables, laid out at their largest and counted (13 orbitals and up),
one string, string counts around the 256 of a group of bits, against the rows of one string per wave
(rs_block 0).  Both precisions, source ranges in 1 and 4 passes.

Both add the same products in another order, some thousand terms per element: 1e-12 of the norm in FP64,
2e-5 in FP32 (24 bits, terms of both signs)."""
import pytest

from binsim_amd import autotune as AT
from tests.conftest import gpu_vec, host
from tests.helpers import rel_err, seeded_vector
from tests.test_gpu_sigma import _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,na,nb", [(4, 4, 1), (9, 4, 9), (10, 4, 5), (11, 4, 1), (13, 6, 1), (14, 7, 0), (16, 2, 8)])
@pytest.mark.parametrize("rb,passes", [(8, 0), (4, 1), (8, 4), (16, 1)])
def test_row_tables(torch_cuda, n, na, nb, rb, passes):
    print(f"tables n={n} na={na} nb={nb} rb={rb} passes={passes}", flush=True)
    saved = [AT.get_config(p) for p in (0, 1)]
    got = {}
    try:
        for form in ((0, 1), (rb, passes)):
            for p in (0, 1):
                AT.set_config(p, dict(saved[p], rs_block=form[0], rs_passes=form[1]))
            B, H, F = _dev(n, na, nb)  # (tables of the form that is chosen when they are built)
            x = gpu_vec(torch_cuda, seeded_vector(B.dim, 7 * n + na))
            for p in (0, 1):
                y = torch_cuda.empty_like(x)
                F.hvec_block([x], [y], precision=p)
                got[form, p] = host(y)
    finally:
        for p in (0, 1):
            AT.set_config(p, saved[p])
    assert rel_err(got[(rb, passes), 0], got[(0, 1), 0]) < 1e-12
    assert rel_err(got[(rb, passes), 1], got[(0, 1), 1]) < 2e-5
