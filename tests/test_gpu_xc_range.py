"""The LSDA kernel against 64-bit-mantissa arithmetic over its range: the vacuum cutoff to nuclear cusps, every spin
polarisation from none to full, counts around a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
L = np.longdouble


def _g(rs, a, a1, b1, b2, b3, b4):
    a, a1, b1, b2, b3, b4 = (L(np.float64(x)) for x in (a, a1, b1, b2, b3, b4))
    s = np.sqrt(rs)
    q0, q1 = -2 * a * (1 + a1 * rs), 2 * a * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs)
    q1p = a * (b1 / s + 2 * b2 + 3 * b3 * s + 4 * b4 * rs)
    ln = np.log1p(1 / q1)
    # and what a rounding of 1 + 1 / q1 is worth in both
    return q0 * ln, -2 * a * a1 * ln - q0 * q1p / (q1 * q1 + q1), -q0, 2 * a * a1


def _lsda(nu, nd):
    """(e, v_up, v_down) and the sums of the absolute values that e and the potentials are made of"""
    nu, nd = (np.maximum(x.astype(L), 0) for x in (nu, nd))
    n = nu + nd
    live = n >= 1e-20
    m = np.where(live, n, 1)
    pi = L("3.14159265358979323846264338327950288")
    cu, cd = np.cbrt(nu), np.cbrt(nd)
    ex = -L(3) / 4 * np.cbrt(6 / pi) * (nu * cu + nd * cd)
    rs, z = np.cbrt(3 / (4 * pi * m)), (nu - nd) / m
    g0, d0, qg0, qd0 = _g(rs, 0.031091, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
    g1, d1, qg1, qd1 = _g(rs, 0.015545, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
    ac, dac, qga, qda = _g(rs, 0.016887, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
    ac, dac = -ac, -dac
    den, fpp = np.cbrt(L(16)) - 2, L(np.float64(1.709921))
    op, om = np.cbrt(1 + z), np.cbrt(1 - z)
    f, fp = ((1 + z) * op + (1 - z) * om - 2) / den, L(4) / 3 * (op - om) / den
    ec = g0 + ac * f / fpp * (1 - z ** 4) + (g1 - g0) * f * z ** 4
    dr = d0 + dac * f / fpp * (1 - z ** 4) + (d1 - d0) * f * z ** 4
    dz = ac / fpp * (fp * (1 - z ** 4) - 4 * z ** 3 * f) + (g1 - g0) * (fp * z ** 4 + 4 * z ** 3 * f)
    vx = -np.cbrt(6 / pi)
    common = ec - rs / 3 * dr
    out = [np.where(live, x, 0) for x in (ex + m * ec, vx * cu + common - (z - 1) * dz, vx * cd + common - (z + 1) * dz)]
    # |f| <= 1 with 2 / (2^{4/3} - 2) ~ 4 units of rounding, |f'| <= 4/3 * 1.26 / 0.52 = 3.3; |1 -+ z| <= 2
    c = abs(g0) + 4 * abs(ac) + abs(g1) + qg0 + qg1 + qga
    # and a rounding of 1 +- z moves its cube root by that over 3 (1 +- z)^{2/3}
    root = sum(np.where(x > 0, np.maximum(x, L(1e-18)) ** (-L(2) / 3), 0) for x in (1 + z, 1 - z))
    scale_v = -vx * np.cbrt(m) + (16 + root) * c + rs * (abs(d0) + 4 * abs(dac) + abs(d1) + qd0 + qd1 + qda)
    return out, (abs(ex) + m * c, scale_v, scale_v)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n", [1, 5, 9, 17])
def test_the_lsda_kernel_over_its_range(n, dtype):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    N, rng = n ** 3, np.random.default_rng(n)
    total = 10.0 ** rng.uniform(-21, 6, N)
    share = rng.uniform(0, 1, N)
    kind = rng.integers(0, 6, N)
    share = np.select([kind == 0, kind == 1, kind == 2, kind == 3], [0.5, 0.0, 1.0, 0.5 + 1e-9 * share], share)
    nu, nd = (total * share).astype(dtype), (total * (1 - share)).astype(dtype)
    nd[kind == 4] = -1e-6  # a mixed density's negative tail counts as 0
    td = getattr(torch, dtype)
    a, b = (torch.from_numpy(x).cuda() for x in (nu, nd))
    outs = [torch.empty(N, dtype=td, device="cuda") for _ in range(3)]
    lira.xc_lsda(a, b, *outs)
    torch.cuda.synchronize()
    got = [o.cpu().numpy() for o in outs]
    want, scale = _lsda(nu, nd)
    # at most some twenty roundings of 2^-53 on the way, and one of the output type
    for g, w, s in zip(got, want, scale):
        assert (abs(g - w) <= 20 * 2.0 ** -53 * s + (2.0 ** -24 * abs(w) if dtype == "float32" else 0)).all()
    closed = (kind == 0) & (nu == nd)
    assert (got[1][closed] == got[2][closed]).all()  # equal spins have equal potentials, bit for bit
