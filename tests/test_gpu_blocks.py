"""The one-launch factorization and the block sweeps at the sizes where they
can go wrong: one block of four tile rows and one row more, a ragged last
block, one, two and a few tiles below the diagonal (no near and corner tasks,
only those, few others; links between blocks that miss columns), more than
four (no helper workgroup, a part of one, more than one).

The fused factor is bitwise the split one; the block sweeps, which start above
four tile rows, and the row sweeps solve the tangent to a normwise backward
error of FP64 round-off: 1e-13 is 450 eps, while the errors of the 64-term
sums that a row takes part in one after another stay at a few eps."""
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


# five tile rows (one block and one row more); numberings that fill the band (w
# at or next to nt - 1, no or few columns of full height), in several blocks
def _five_rows():
    return inputs.truss_dome(n=11, load=-20.0, steps=20).text


def _full(n):
    return lambda: inputs.shell_panel(n=n, thick_sigma=0.1, imperfection=0.1, scramble=1).text


BANDS = {"dome11": (_five_rows, 5, 1), "full5": (_full(5), 3, 2), "full7": (_full(7), 6, 5),
         "full12": (_full(12), 15, 14), "full20": (_full(20), 40, 38), "full32": (_full(32), 99, 98)}


@pytest.mark.parametrize("case", sorted(BANDS))
def test_five_rows_and_full_bands(case):
    text, nt, w = BANDS[case]
    print(f"[blocks] {case}", flush=True)
    with cubens.GpuModel(model_file(f"blocks_{case}.txt", text())) as g:
        K = _tangent_operator(g)
        assert ((g.neq + 63) // 64, min((g.info.bandwidth + 63) // 64, nt - 1)) == (nt, w)
        b = np.random.default_rng(nt).standard_normal(g.neq)
        det, piv = g.factor(cubens.options(factor_schedule=cubens.FACTOR_SPLIT))
        piv = piv.copy()
        knorm = np.abs(K).sum(axis=1).max()
        xs = []
        for sweeps in (cubens.SWEEP_CHAIN, cubens.SWEEP_ROWS, cubens.SWEEP_LOOK2, cubens.SWEEP_LOOK3):
            d2, p2 = g.factor(cubens.options(sweep_schedule=sweeps))
            xs.append(g.solve(b))
            assert d2 == det and np.array_equal(p2, piv)
            eta = np.abs(K @ xs[-1] - b).max() / (knorm * np.abs(xs[-1]).max() + np.abs(b).max())
            assert eta < 1e-13, (sweeps, eta)
        assert np.array_equal(xs[2], xs[3])


# 2, 3, 5 and 13 tiles below the diagonal and a full band: near and corner
# tasks, block links that miss columns, helpers
@pytest.mark.parametrize("n,scramble", [(9, None), (20, None), (41, None), (127, None), (12, 1)])
def test_fp32_factor_schedules_and_sweeps(n, scramble):
    """FP32 band: fused and split factors bitwise equal, and every sweep
    schedule solves the tangent to the rounding of its FP32 matrices (five
    units of 2^-24; the sums are FP64)."""
    print(f"[blocks] FP32 n={n}", flush=True)
    text = inputs.shell_panel(n=n, thick_sigma=0.1, imperfection=0.1, scramble=scramble).text
    with cubens.GpuModel(model_file(f"blocks32_{n}.txt", text)) as g:
        K = _tangent_operator(g)
        g.tangent_fp32(cubens.GEN_BASE, cubens.GEN_BASE)
        b = np.random.default_rng(n).standard_normal(g.neq)
        opt = dict(judge=0, refine=0)
        det, piv = g.factor(cubens.options(cubens.SOLVER_BAND32, factor_schedule=cubens.FACTOR_SPLIT, **opt))
        piv, xs = piv.copy(), g.solve(b)
        knorm = np.abs(K).sum(axis=1).max()
        for sweeps in (cubens.SWEEP_CHAIN, cubens.SWEEP_ROWS, cubens.SWEEP_LOOK2):
            d2, p2 = g.factor(cubens.options(cubens.SOLVER_BAND32, sweep_schedule=sweeps, **opt))
            x = g.solve(b)
            assert d2 == det and np.array_equal(p2, piv)
            if sweeps == cubens.SWEEP_CHAIN:
                assert np.array_equal(x, xs)
            eta = np.abs(K @ x - b).max() / (knorm * np.abs(x).max() + np.abs(b).max())
            assert eta < 5 * 2.0**-24, (sweeps, eta)
