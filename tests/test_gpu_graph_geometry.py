"""A captured LOBPCG segment after the ions have moved: the nonlocal operator's launches depend on the boxes and on their
colouring, so a graph that was captured for one geometry must not be replayed for another."""
import os
import sys

import numpy as np
import pytest

import oracle as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "atomic-sandbox_amd"))
import synthetic_tables as T  # noqa: E402

pytestmark = pytest.mark.gpu
N, H, REACH = 25, 0.25, 5  # a nucleus on the grid has a box of 11 points a side


def _species():
    du, r = H / T.TABLE_POINTS_PER_H, REACH * H
    projs = [T.Projector(l, 0.3 + 0.5 * l, r, T.uniform_table(du, r, 1.0, 0.4 * r)) for l in (0, 1)]
    return T.Species(8, 6.0, T.SIGMA_LR_OVER_H * H, du, T.uniform_table(du, 1.6, 4.0, 0.45), 1.6, None, 0.0, projs)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("before,after", [
    # one ion, its box clipped to 216 points (one chunk), then 1331 points (six chunks)
    ([[12, 12, 12]], [[0, 0, 0]]),
    # two ions whose boxes are apart (one colour), then overlap (two): the same box sizes and rows
    ([[-6, 0, 0], [6, 0, 0]], [[-2, 0, 0], [2, 0, 0]]),
], ids=["box", "colours"])
def test_a_moved_geometry_is_not_replayed_from_the_old_graph(before, after, precision):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import lira
    k = 5
    z = [8] * len(after)
    guess = O.initial_orbitals(N, H, [[0.0, 0.0, 0.0]], k, 77)
    got = {}
    for graphs in (True, False):
        s = lira.GpuSolver(N, H, precision)
        s.set_graphs(graphs)
        s.set_ionic([_species()])
        out = []
        for pos, steps in ((after, (0, 0)), (before, (0, 0)), (after, (1, 0, 3))):
            v, _ = s.ionic_fields((H * np.array(pos, float)).tolist(), z, H)
            # A call of no steps measures its guess and leaves its graph; two of them leave the buffers in the arrangement
            # that they had, so the next call's first step meets the graphs of the geometry before.
            for n in steps:
                x, ev, st = s.lobpcg(v, guess, 1e-12, n, precond_lambda=-1.0)
                assert st.iterations == n
                out += [x, ev]
        got[graphs] = out
    for a, b in zip(got[True], got[False]):
        np.testing.assert_array_equal(a, b)
