"""The Gram's tiles at their edges: column counts about the 16-wide blocks and the tile limits, point counts below and just
above a wave's unit, bases at any element alignment, U beginning with S or not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 2), (2, 1), (3, 6), (15, 30), (16, 32), (17, 34), (16, 16), (24, 48), (31, 96), (33, 64), (32, 97),
          (48, 96), (49, 98), (40, 8), (65, 5), (90, 180), (50, 200)]


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 11, 21])
def test_tile_edges_match_numpy(n, size):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    dt, npdt = (torch.float32, np.float32) if size == 4 else (torch.float64, np.float64)
    N, h = n ** 3, 0.3
    rng = np.random.default_rng(n)
    for m, q in SHAPES:
        for own in (False, True):  # own: U begins with S
            if own and q < m:
                continue
            shift = (m + q) % 4
            cols = q if own else m + q
            a = rng.standard_normal((cols, N)).astype(npdt)
            d = torch.empty(cols * N + shift, dtype=dt, device="cuda")
            d[shift:] = torch.tensor(a.reshape(-1))
            s = d[shift:]
            u = s if own else s[m * N:]
            g = lira.gram(n, h, s, m, u, q)
            a = a.astype(np.float64)
            sa, ua = a[:m], (a if own else a[m:])
            want, scale = sa @ ua.T * h ** 3, np.abs(sa) @ np.abs(ua).T * h ** 3
            # sums of N exact products in f64, in any order: (N + 2) roundings of at most the sum of magnitudes
            assert (np.abs(g - want) <= (N + 2) * 2.0 ** -53 * scale).all(), (m, q, own)
            if own:
                assert np.array_equal(g[:, :m], g[:, :m].T), (m, q)  # S^T S is exactly symmetric
