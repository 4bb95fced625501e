"""The f32 H.X of orbital-like bands in an ionic potential: its error against 64 bits is no larger than that of the pair form
c_m [(f_m - f_0) + (f_{-m} - f_0)] with each operation rounded to f32."""
import numpy as np
import pytest

F = np.float32
C = [8 / 5, -1 / 5, 8 / 315, -1 / 560]


def _field(n, h, seed):
    """A band of a few Gaussians about two nuclei and the nuclei's softened potential."""
    rng = np.random.default_rng(seed)
    a = (np.arange(n) - (n - 1) / 2) * h
    x, v = np.zeros((n, n, n)), np.zeros((n, n, n))
    for _ in range(2):
        p = rng.uniform(-1.5, 1.5, 3)
        r2 = (a[:, None, None] - p[0]) ** 2 + (a[:, None] - p[1]) ** 2 + (a - p[2]) ** 2
        v -= rng.uniform(1, 6) / np.sqrt(r2 + h * h)
        x += rng.normal() * np.exp(-rng.uniform(0.15, 0.6) * r2) + rng.normal() * a * np.exp(-rng.uniform(0.15, 0.4) * r2)
    return x.astype(F), v.astype(F)


def _shift(x, axis, m):
    n, p = x.shape[0], np.pad(x, 4)
    at = [slice(4, 4 + n)] * 3
    at[axis] = slice(4 + m, 4 + m + n)
    return p[tuple(at)]


def _exact(x, v, h):
    x, v = x.astype(float), v.astype(float)
    lap = -205 / 24 * x
    for axis in range(3):
        for m, c in enumerate(C, 1):
            lap += c * (_shift(x, axis, m) + _shift(x, axis, -m))
    return -0.5 * lap / h ** 2 + v * x


def _pair_form(x, v, h):
    fma = lambda a, b, c: (a.astype(float) * b + c).astype(F)  # noqa: E731  (the product of two f32 is exact)
    axes = []
    for axis in (2, 1, 0):
        t = F(0) * x
        for m, c in enumerate(C, 1):
            t = fma((_shift(x, axis, m) - x) + (_shift(x, axis, -m) - x), F(c), t)
        axes.append(t)
    lap = ((axes[0] + axes[1]) + axes[2]) * F(1 / h ** 2)
    return fma(v, x, F(-0.5) * lap)


@pytest.mark.gpu
@pytest.mark.parametrize("n,h", [(33, 0.3), (40, 0.25), (63, 0.25), (72, 0.2), (95, 0.15), (96, 0.25)])
def test_the_error_is_no_larger_than_the_pair_forms(n, h):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    ours = pair = 0.0
    for seed in range(4):
        x, v = _field(n, h, 10 * n + seed)
        xd, vd = (torch.from_numpy(f.reshape(1, -1).copy()).cuda() for f in (x, v))
        out = torch.empty_like(xd)
        lira.hamiltonian(n, h, vd, xd, out, 1)
        want = _exact(x, v, h)
        size = np.linalg.norm(want)
        ours += np.log(np.linalg.norm(out.cpu().numpy().reshape(n, n, n) - want) / size)
        pair += np.log(np.linalg.norm(_pair_form(x, v, h) - want) / size)
    assert ours <= pair  # the mean over the fields, of the logarithm of the relative error


@pytest.mark.gpu
@pytest.mark.parametrize("h", [0.07, 0.12, 0.15, 0.2, 0.25, 0.3, 0.35])
def test_the_kinetic_energy_has_no_common_factor(h):
    # A smooth field's f32 -1/2 lap is that of 64 bits times 1 + d. Each point's rounding, 2^-24, averages out of d over some
    # 1100 points (by weight) to 1.8e-9, over three fields to 1e-9; the fields are 1e-6 of their peak at the faces.
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    n, d = 64, []
    a = (np.arange(n) - (n - 1) / 2) / n
    for seed in range(3):
        rng = np.random.default_rng(seed)
        p, w = rng.uniform(-0.05, 0.05, 3), rng.uniform(55, 75, 3)
        x = np.exp(-w[0] * (a[:, None, None] - p[0]) ** 2 - w[1] * (a[:, None] - p[1]) ** 2 - w[2] * (a - p[2]) ** 2).astype(F)
        want = _exact(x, np.zeros_like(x), h)
        out = torch.empty(1, n ** 3, dtype=torch.float32, device="cuda")
        lira.hamiltonian(n, h, torch.zeros(n ** 3, device="cuda"), torch.from_numpy(x.reshape(1, -1).copy()).cuda(), out, 1)
        got = out.cpu().numpy().reshape(n, n, n).astype(float)
        d.append((got * want).sum() / (want * want).sum() - 1.0)
    assert abs(np.mean(d)) < 3e-9
