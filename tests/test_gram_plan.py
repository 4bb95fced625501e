"""The Gram's work buffer over the shapes that one eigensolve puts through it: the plan's partial sums by compiling its header
(no GPU), and mixed eigensolves whose guess needs more of them than any later step."""
import os
import subprocess
import sys
import tempfile

import numpy as np
import pytest

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PLAN_TEST = r"""
#include "gram_plan.hpp"
#include <cstdio>
int main() {
    long bad = 0, inverted = 0;
    // sides from one point to the largest, k up to the 128 columns a block may have; q < 2 m: a display's projections
    for (int n : {1, 2, 3, 5, 11, 21, 25, 33, 48, 64, 95, 128, 160, 192, 256, 400})
        for (int esize : {4, 8})
            for (bool sym : {false, true})
                for (int m = 1; m <= 384; m++)
                    for (int q : {1, m / 2 + 1, m, 2 * m}) {
                        const long N = (long)n * n * n;
                        const size_t need = lira::gram_partials(m, q, N, esize, sym && q >= m);
                        if (need > lira::gram_partials_bound(m, q, N)) bad++;
                        // growing in both, so a buffer for (m, q) serves every product within it
                        if (lira::gram_partials_bound(m, q, N) > lira::gram_partials_bound(m + 1, q, N)) bad++;
                        if (lira::gram_partials_bound(m, q, N) > lira::gram_partials_bound(m, q + 1, N)) bad++;
                        if (q == 2 * m && m <= 128) {
                            if (need > lira::gram_partials_bound(3 * m, 6 * m, N)) bad++;
                            if (need > lira::gram_partials(3 * m, 6 * m, N, esize, sym)) inverted++;
                        }
                    }
    std::printf("%ld refused, %ld need more than three times their columns\n", bad, inverted);
    return bad != 0 || inverted == 0;
}
"""


def test_a_blocks_buffer_serves_every_product_within_it():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "plan.cpp"), os.path.join(d, "plan")
        with open(src, "w") as f:
            f.write(PLAN_TEST)
        subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "atomic-sandbox_amd", "csrc"), "-I",
                        os.path.join(ROOT, "include"), src, "-o", exe], check=True)
        subprocess.run([exe], check=True)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [81, 96])
def test_a_mixed_eigensolve_of_a_wide_block(k):
    # the lowest levels of the anisotropic oscillator; at these widths the guess's k x 2k Gram needs the most partials
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    sys.path.insert(0, os.path.join(ROOT, "atomic-sandbox_amd"))
    import lira
    n, h = 37, 0.3
    x, y, z = O.grid_points(n, h)
    w = (1.0, 1.13, 1.31)
    v = 0.5 * (w[0] ** 2 * x * x + w[1] ** 2 * y * y + w[2] ** 2 * z * z)
    levels = sorted(w[0] * (a + 0.5) + w[1] * (b + 0.5) + w[2] * (c + 0.5)
                    for a in range(12) for b in range(12) for c in range(12))[:k]
    guess = O.initial_orbitals(n, h, [[0.0, 0.0, 0.0]], k, 778)
    xs, ev, st = lira.GpuSolver(n, h, lira.MIXED).lobpcg(v, guess, 1e-4, 600, precond_lambda=1.5)
    assert st.max_residual < 1e-4
    assert np.abs(np.sort(ev) - np.array(levels)).max() < 3e-2
    assert np.abs(xs @ xs.T * h ** 3 - np.eye(k)).max() < 1e-5
