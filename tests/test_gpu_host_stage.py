"""The Poisson solve's host transfers through pinned slots: fields of less than one slot, of a few slots with a
remainder, and large enough for the worker threads; the field that comes back is the one that the guess went in as."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [9, 64, 65, 95, 127, 128, 129])  # 64^3 doubles are one slot; 128^3 are 16 MiB
def test_a_guess_that_is_kept_comes_back_bit_for_bit(n, precision):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    rng = np.random.default_rng(n)
    s = lira.GpuSolver(n, 0.2, precision)
    rho = rng.standard_normal(n ** 3)
    guess = rng.standard_normal(n ** 3)
    for _ in range(2):  # with new pinned slots, and with the kept ones
        v, st = s.poisson(rho, v0=guess, tol=1e300)  # the guess satisfies the tolerance: no iteration changes it
        assert st.iterations == 0
        np.testing.assert_array_equal(v, guess)
    # rho arrived too: the residual of a zero guess against b is 1 exactly when b is what was sent, not zero
    v, st = s.poisson(rho, tol=1e300)
    assert st.iterations == 0 and st.residual == 1.0 and not v.any()
