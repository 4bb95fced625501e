"""The fused coarse V-cycle (one workgroup from the 16^3 level down) against the same cycle in numpy, at every entry edge:
each class of tile, its remainders, and grids whose fine levels run outside it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRE, POST, COARSE, OMEGA = 2, 2, 12, 6.0 / 7.0  # V(2,2), twelve sweeps on the coarsest level (n <= 2)


def _cycle(n, h, d_low, d_high, b):
    """x = M b on an n^3 level: the 7-point operator with a missing neighbour (1 - 1/d) x0, damped Jacobi, full weighting
    about the odd points, trilinear interpolation."""
    edge = np.zeros(n)
    edge[0] += 1.0 - 1.0 / d_low
    edge[-1] += 1.0 - 1.0 / d_high
    diag = 6.0 - (edge[:, None, None] + edge[None, :, None] + edge[None, None, :])

    def around(x):
        p = np.pad(x, 1)
        return (p[:-2, 1:-1, 1:-1] + p[2:, 1:-1, 1:-1] + p[1:-1, :-2, 1:-1] + p[1:-1, 2:, 1:-1]
                + p[1:-1, 1:-1, :-2] + p[1:-1, 1:-1, 2:])

    def sweeps(x, count):
        for _ in range(count):
            x = x + OMEGA / diag * (h * h * b + around(x) - diag * x)
        return x

    x = np.zeros_like(b)
    if n <= 2:
        return sweeps(x, COARSE)
    x = sweeps(x, PRE)
    r = b + (around(x) - diag * x) / (h * h)
    nc = n // 2
    w = np.zeros((nc, n))  # one axis of the full weighting
    for i in range(nc):
        for d, v in ((-1, 0.25), (0, 0.5), (1, 0.25)):
            if 2 * i + 1 + d < n:
                w[i, 2 * i + 1 + d] = v
    bc = np.einsum("az,by,cx,zyx->abc", w, w, w, r, optimize=True)
    xc = _cycle(nc, 2.0 * h, (d_low + 1.0) / 2.0, (d_high + (n - 2 * nc)) / 2.0, bc)
    x = x + np.einsum("az,by,cx,abc->zyx", 2 * w, 2 * w, 2 * w, xc, optimize=True)
    return sweeps(x, POST)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 14, 15, 16, 17, 23, 24, 31, 32, 33])
def test_the_fused_cycle_matches_numpy(n, precision):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    h = 0.3
    rng = np.random.default_rng(n)
    r = rng.standard_normal(n ** 3).astype(np.float32).astype(np.float64)
    z = lira.GpuSolver(n, h, precision).mg_vcycle(r)
    want = _cycle(n, h, 1.0, 1.0, r.reshape(n, n, n)).reshape(-1)
    # about 40 sweeps and transfers, each a few roundings of values no larger than the result's maximum, damped from
    # level to level: 100 roundings
    bound = 100 * (2.0 ** -53 if precision == lira.FP64 else 2.0 ** -24)
    assert np.abs(z - want).max() <= bound * np.abs(want).max()


def _cycle_f32(n, h, d_low, d_high, b):
    """The same cycle with every operation rounded to f32 (the transfers once per point)."""
    f = np.float32
    edge = np.zeros(n)
    edge[0] += 1.0 - 1.0 / d_low
    edge[-1] += 1.0 - 1.0 / d_high
    diag = (6.0 - (edge[:, None, None] + edge[None, :, None] + edge[None, None, :])).astype(f)
    h2, factor = f(h * h), f(OMEGA) / diag

    def defect(x):  # the sum of the neighbours less diag x
        p = np.pad(x, 1)
        return (((((p[1:-1, 1:-1, :-2] + p[1:-1, 1:-1, 2:]) + p[1:-1, :-2, 1:-1]) + p[1:-1, 2:, 1:-1])
                 + p[:-2, 1:-1, 1:-1]) + p[2:, 1:-1, 1:-1]) - diag * x

    def sweeps(x, count):
        for _ in range(count):
            x = x + factor * (h2 * b + defect(x))
        return x

    x = np.zeros_like(b)
    if n <= 2:
        return sweeps(x, COARSE)
    x = sweeps(x, PRE)
    r = b + defect(x) / h2
    nc = n // 2
    w = np.zeros((nc, n))
    for i in range(nc):
        for d, v in ((-1, 0.25), (0, 0.5), (1, 0.25)):
            if 2 * i + 1 + d < n:
                w[i, 2 * i + 1 + d] = v
    bc = np.einsum("az,by,cx,zyx->abc", w, w, w, r, optimize=True).astype(f)
    xc = _cycle_f32(nc, 2.0 * h, (d_low + 1.0) / 2.0, (d_high + (n - 2 * nc)) / 2.0, bc)
    x = x + np.einsum("az,by,cx,abc->zyx", 2 * w, 2 * w, 2 * w, xc, optimize=True).astype(f)
    return sweeps(x, POST)


@pytest.mark.parametrize("n", [5, 6, 8, 11, 12, 13, 16])
def test_the_f32_cycle_is_as_accurate_as_its_operations(n):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    h, solver = 0.3, lira.GpuSolver(n, 0.3, lira.MIXED)
    ours = rounded = 0.0
    for seed in range(4):
        r = np.random.default_rng(10 * n + seed).standard_normal((n, n, n)).astype(np.float32)
        want = _cycle(n, h, 1.0, 1.0, r.astype(float))
        got = solver.mg_vcycle(r.astype(float).reshape(-1)).reshape(n, n, n)
        ours += np.log(np.linalg.norm(got - want))
        rounded += np.log(np.linalg.norm(_cycle_f32(n, h, 1.0, 1.0, r) - want))
    # the mean of the logarithms: the kernel's fused operations may only make its error smaller
    assert ours <= rounded
