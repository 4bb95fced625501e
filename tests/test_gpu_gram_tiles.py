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


@pytest.mark.parametrize("size,n,shapes", [
    # f32 columns a multiple of 8 MiB apart; 1 x 1 to 3 x 5 blocks, shared and not
    (4, 128, [(3, 6, True), (16, 33, True), (24, 48, True), (30, 60, True), (40, 80, True), (20, 30, False)]),
    # f64 grids of at least 6 Mi points, an odd edge: ragged chunks, columns at 8-byte alignment
    (8, 185, [(16, 64, True), (27, 54, True), (32, 64, True), (30, 60, False)]),
])
def test_the_loads_of_large_grids_match_a_library_product(size, n, shapes):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    dt, N, h = torch.float32 if size == 4 else torch.float64, n ** 3, 0.3
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randn(80 if size == 4 else 90, N, dtype=dt, device="cuda", generator=gen)
    for m, q, own in shapes:
        u = a[:q] if own else a[m:m + q]
        g = torch.from_numpy(lira.gram(n, h, a[:m], m, u, q))
        s64, u64 = a[:m].double(), u.double()
        want, scale = (s64 @ u64.T).cpu() * h ** 3, (s64.abs() @ u64.abs().T).cpu() * h ** 3
        # both are sums of N exact products in f64, each in its own order
        assert ((g - want).abs() <= 2 * (N + 2) * 2.0 ** -53 * scale).all(), (m, q, own)
        # and beyond that bound: a lane's points in another column's sum would cost sqrt(N) of N terms; rounding does not
        assert ((g - want).abs() <= 1e-12 * scale).all(), (m, q, own)
