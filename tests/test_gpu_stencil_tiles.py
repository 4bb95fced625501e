"""The stencil's tiles at their edges: grids one point below, at and above the tile widths and vector widths, chunk
remainders, one-plane grids, and fields at any element alignment, in every variant that takes the grid."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1), (2, 2), (3, 1), (5, 3), (31, 2), (32, 2), (33, 3), (63, 1), (64, 2), (65, 2), (95, 2), (96, 1), (97, 2),
         (127, 1), (128, 1), (129, 2), (177, 1), (191, 1), (192, 1), (193, 1)]


@pytest.fixture(scope="module")
def env():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    lira.lib()
    return torch, lira


def _shifted(torch, a, dtype, shift):
    """a on the device, its base `shift` elements past an allocation's start."""
    t = torch.empty(a.size + shift, dtype=dtype, device="cuda")
    t[shift:] = torch.tensor(a.reshape(-1), dtype=dtype)
    return t[shift:]


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("n,nb", GRIDS)
def test_tile_edges_match_the_oracle(env, n, nb, size):
    torch, lira = env
    dt = torch.float32 if size == 4 else torch.float64
    npdt = np.float32 if size == 4 else np.float64
    rng = np.random.default_rng(1000 * n + nb)
    h = 0.25
    x, r = (rng.standard_normal((nb, n ** 3)).astype(npdt).astype(np.float64) for _ in range(2))
    v = rng.uniform(-5, 0, n ** 3).astype(npdt).astype(np.float64)
    lam = rng.uniform(-1, 0, nb)
    hx = np.stack([O.hamiltonian(n, h, v, x[b]) for b in range(nb)])
    c0 = -205.0 / 72.0
    at_pi = c0 + 2.0 * (-8.0 / 5.0 - 1.0 / 5.0 - 8.0 / 315.0 - 1.0 / 560.0)
    omega, diag = 4.0 / (3.0 * at_pi / c0), -1.5 * c0 / (h * h)
    jac = np.stack([x[b] + omega / np.maximum(diag + v - lam[b], 0.1) * (r[b] - (hx[b] - lam[b] * x[b])) for b in range(nb)])
    lap = np.stack([-2.0 * (O.hamiltonian(n, h, np.zeros_like(v), x[b])) for b in range(nb)])
    # some 20 roundings of terms up to the largest result: 20 * 2^-24 in f32, the f64 bound of the kernel tests in f64
    bound = 1.2e-6 if size == 4 else 1e-12
    lamd = torch.tensor(lam, device="cuda")
    for shift in (0, 1, 3):
        xd, rd, vd = (_shifted(torch, a, dt, shift) for a in (x, r, v))
        guard = torch.full((nb * n ** 3 + 8,), 7.0, dtype=dt, device="cuda")
        out = guard[4:4 + nb * n ** 3]
        first = {}
        for var in [-1] + list(range(len(lira.stencil_variants()))):
            lira.lib().lira_set_stencil_variant(size, var)
            try:
                for mode, want in (("ham", hx), ("lap", lap), ("jac", jac)):
                    out.fill_(-3.0)
                    if mode == "ham":
                        lira.hamiltonian(n, h, vd, xd, out, nb)
                    elif mode == "lap":
                        lira.laplacian(n, h, xd, out, nb)
                    else:
                        lira.jacobi_sweep(n, h, vd, xd, rd, lamd, out, nb)
                    torch.cuda.synchronize()
                    got = out.cpu().numpy().reshape(nb, -1)
                    if mode not in first:
                        first[mode] = got
                        assert np.abs(got - want).max() <= bound * np.abs(want).max(), (mode, shift)
                    else:
                        assert np.array_equal(got, first[mode]), (mode, shift, var)
            finally:
                lira.lib().lira_set_stencil_variant(size, -1)
        g = guard.cpu().numpy()
        assert (g[:4] == 7.0).all() and (g[-4:] == 7.0).all()  # nothing outside the block is written
