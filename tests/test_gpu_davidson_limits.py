"""The Davidson driver and its vector operations at the limits of what they take."""
import numpy as np
import pytest

from binsim_amd import davidson as D
from tests.conftest import gpu_vec
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
    with pytest.raises(RuntimeError, match="finite|infinities"):
        D.solve(B, H, nroots=1, mixed=mixed, guess=gpu_vec(torch_cuda, x))
