"""The nonlocal operator's box sums and scatter at the edges of their chunks: boxes smaller than one block, one point to
either side of a block, many chunks, one to eight points per thread, clipped boxes, 1 to 9 rows, ragged band groups."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import oracle as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "atomic-sandbox_amd"))
import synthetic_tables as T  # noqa: E402

pytestmark = pytest.mark.gpu
H = 0.25


def _species(ls, reach):
    """One projector per l of ls, of radius reach * H (a nucleus on the grid has a box of 2 reach + 1 points a side)."""
    du, r = H / T.TABLE_POINTS_PER_H, reach * H
    projs = [T.Projector(l, 0.3 + 0.5 * l, r, T.uniform_table(du, r, 1.0, 0.4 * r)) for l in ls]
    return T.Species(8, 6.0, T.SIGMA_LR_OVER_H * H, du, T.uniform_table(du, 1.6, 4.0, 0.45), 1.6, None, 0.0, projs)


def _apply(lira, s, x, rows):
    """lira_nonlocal_apply with room for every row."""
    nb, out, c, got = x.shape[0], np.zeros_like(x), np.zeros((rows, x.shape[0])), C.c_int()
    assert lira.lib().lira_nonlocal_apply(s._h, x.reshape(-1), nb, out.reshape(-1), c.ctypes.data_as(C.c_void_p),
                                          c.size, C.byref(got)) == 0
    assert got.value == rows
    return out, c


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,ls,reach,ions,nb", [
    (17, (0,), 1, 1, 1),           # 27 points, one row
    (17, (0, 1), 3, 1, 5),         # 343 points: one block and a remainder
    (21, (0, 1, 2), 4, 2, 3),      # nine rows
    (33, (1, 2), 8, 1, 17),        # eight rows, a last group of one band
    (33, (0, 1), 7, 48, 4),        # three points per thread, several ions to a colour
    (25, (0, 1), 6, 200, 2),       # eight points per thread, many colours, clipped boxes
    (55, (0, 1, 2), 26, 1, 4),     # 149 k points in two points per thread: more chunks than a wave has lanes
])
def test_box_sums_and_scatter_match_the_oracle(n, ls, reach, ions, nb, precision):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    rng = np.random.default_rng(n + nb)
    edge = (n - 1) * H / 2
    # on grid points for one ion (the box is exactly 2 reach + 1 a side), anywhere in the box for several
    pos = [[H * (0 if n % 2 else 0.5)] * 3] if ions == 1 else (rng.uniform(-edge, edge, (ions, 3))).tolist()
    z = [8] * ions
    sp = _species(ls, reach)
    s = lira.GpuSolver(n, H, precision)
    s.set_ionic([sp])
    s.ionic_fields(pos, z, H)
    x = rng.standard_normal((nb, n ** 3)).astype(np.float32).astype(np.float64)
    out, c = _apply(lira, s, x, sum(2 * l + 1 for l in ls) * ions)
    nl = O.Nonlocal(n, H, pos, z, [sp])
    rows = sum(2 * l + 1 for l in ls)
    assert c.shape == (nl.rows, nb) == (rows * ions, nb)
    # |beta_lm| <= t(d) d^l sqrt((2 l + 1) / 4 pi). FP64: the tables and sums round differently (1e-12 of the sum of
    # absolute values). MIXED: beta and the output are rounded to 24 bits, the sums are not.
    axis = (np.arange(n) - (n - 1) / 2) * H
    eps = 1e-12 if precision == 0 else 2 * 2.0 ** -24
    total = np.zeros(nb)
    for i, p in enumerate(pos):
        d = np.sqrt((axis[:, None, None] - p[2]) ** 2 + (axis[None, :, None] - p[1]) ** 2 + (axis - p[0]) ** 2).ravel()
        r0 = i * rows
        for j, l in enumerate(ls):
            beta = T.bump_gaussian(d, 1.0, 0.4 * reach * H, reach * H) * d ** l * np.sqrt((2 * l + 1) / (4 * np.pi))
            size = np.abs(x) @ beta * H ** 3
            total += (2 * l + 1) * sp.projectors[j].e_kb * size * beta.max()
            for b in range(nb):
                want = nl.project(x[b])[r0:r0 + 2 * l + 1] if i % 50 == 0 else None
                if want is not None:
                    assert np.abs(c[r0:r0 + 2 * l + 1, b] - want).max() <= eps * size[b], (i, l, b)
            r0 += 2 * l + 1
    for b in range(nb):
        want = nl.apply_add(x[b], np.zeros(n ** 3))
        assert np.abs(out[b] - want).max() <= (2 + ions) * eps * total[b], b
