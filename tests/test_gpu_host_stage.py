"""The Poisson solve's host transfers through pinned slots: fields of less than one slot, of a few slots with a
remainder, and large enough for the worker threads; the field that comes back is the one that the guess went in as, and
a solved field satisfies the equation of the density at every point, so each direction put its chunks in their place."""
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
    # some rho arrived too: the residual of a zero guess is 1 for every right-hand side but zero
    v, st = s.poisson(rho, tol=1e300)
    assert st.iterations == 0 and st.residual == 1.0 and not v.any()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [65, 127, 129])  # a little more than one slot; just below and above the worker threads' 16 MiB
def test_the_solved_field_satisfies_the_equation_of_the_density_that_was_sent(n, precision):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    rng = np.random.default_rng(n)
    h, tol = 0.2, 1e-9
    x = (np.arange(n) - (n - 1) / 2) * h
    g = np.exp(-x * x / (0.02 * (n * h) ** 2))
    # rough on every plane, row and point: no two chunks are alike
    rho = g[:, None, None] * g[:, None] * g * (1.0 + rng.uniform(0.0, 1.0, (n, n, n)))
    s = lira.GpuSolver(n, h, precision)
    v, st = s.poisson(rho.reshape(-1), tol=tol)
    f = v.reshape(n, n, n)
    c = [8.0 / 5.0, -1.0 / 5.0, 8.0 / 315.0, -1.0 / 560.0]
    i = slice(4, n - 4)
    lap = 3.0 * (-205.0 / 72.0) * f[i, i, i]
    for axis in range(3):
        for m, cm in enumerate(c, 1):
            for d in (-m, m):
                at = [i, i, i]
                at[axis] = slice(4 + d, n - 4 + d)
                lap += cm * f[tuple(at)]
    b = 4.0 * np.pi * rho[i, i, i]
    # The solver stops at tol times the norm of its right-hand side: 4 pi rho, and on the 24 n^2 points within four of a
    # face the potential outside, at most the faces' own, times the sum of |c_m| along each axis. MIXED rounds rho to f32.
    face = max(np.abs(f[j]).max() for j in ([0], [-1], (slice(None), 0), (slice(None), -1), (..., 0), (..., -1)))
    rhs = 4.0 * np.pi * np.linalg.norm(rho) + np.sqrt(24.0) * n * 3.0 * np.abs(c).sum() * face / h ** 2
    assert np.linalg.norm(lap / h ** 2 + b) <= tol * rhs + 2.0 ** -24 * np.linalg.norm(b)
    assert tol * rhs < 1e-5 * np.linalg.norm(b)  # small beside what a chunk out of its place would leave
    again, st = s.poisson(rho.reshape(-1), v0=v, tol=2.0 * tol)  # the solution as a guess: it needs no step
    assert st.iterations == 0
    np.testing.assert_array_equal(again, v)
