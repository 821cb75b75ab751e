"""The one-launch factorization and the block sweeps at the sizes where they
can go wrong: one block of four tile rows and one row more, a ragged last
block, one, two and a few tiles below the diagonal (no near and corner tasks,
only those, few others; links between blocks that miss columns), more than
four (no helper workgroup, a part of one, more than one).

The fused factor is bitwise the split one; the block sweeps, which start above
four tile rows, and the row sweeps solve the tangent to a normwise backward
error of FP64 round-off: 1e-13 is about 5 sqrt(neq) eps at the largest size
here."""
import numpy as np
import pytest

import cubens
from cubens import inputs
from helpers import model_file
from test_gpu_sweeps import _tangent_operator

pytestmark = pytest.mark.gpu


# (n, tile rows, tiles below the diagonal)
SHAPES = [(5, 3, 1), (6, 4, 1), (7, 6, 1), (9, 9, 2), (20, 40, 3), (31, 93, 4), (41, 162, 5), (75, 535, 8),
          (127, 1524, 13)]


@pytest.mark.parametrize("n,nt,w", SHAPES)
def test_factor_and_block_sweeps_at_the_edges(n, nt, w):
    path = model_file(f"blocks_{n}.txt", inputs.shell_panel(n=n, thick_sigma=0.1, imperfection=0.1).text)
    with cubens.GpuModel(path) as g:
        K = _tangent_operator(g)
        assert ((g.neq + 63) // 64, (g.info.bandwidth + 63) // 64) == (nt, w)
        b = np.random.default_rng(n).standard_normal(g.neq)
        det, piv = g.factor(cubens.options(factor_schedule=cubens.FACTOR_SPLIT))
        piv, xs = piv.copy(), g.solve(b)
        knorm = np.abs(K).sum(axis=1).max()
        for sweeps in (cubens.SWEEP_CHAIN, cubens.SWEEP_ROWS, cubens.SWEEP_LOOK2):
            d2, p2 = g.factor(cubens.options(sweep_schedule=sweeps))
            x = g.solve(b)
            assert d2 == det and np.array_equal(p2, piv)
            if sweeps == cubens.SWEEP_CHAIN:
                assert np.array_equal(x, xs)
            eta = np.abs(K @ x - b).max() / (knorm * np.abs(x).max() + np.abs(b).max())
            assert eta < 1e-13, (sweeps, eta)
