"""A call that ends with an error leaves the handle usable: a factorization
that the device code refuses can be repeated, and the next one works.  A solve
that has no factorization to solve with is such an error: on a handle that has
not factored, after other options have replaced the analysis, and as the
fallback of a Krylov solve without the FP64 judge."""
import numpy as np
import pytest

import cubens
from cubens import inputs
from helpers import model_file

pytestmark = pytest.mark.gpu


def test_refused_factorization_can_be_repeated():
    path = model_file("refused.txt", inputs.truss_dome(n=4, load=-20.0, steps=20).text)
    with cubens.GpuModel(path) as g, cubens.LearnedPrecond(1) as L:
        L.attach(g)
        g.tangent(cubens.GEN_BASE, cubens.GEN_BASE)
        for _ in range(3):
            print("[errors] refused factorization", flush=True)
            with pytest.raises(cubens.CubensError, match="6-slot joints"):
                g.factor(cubens.options(cubens.SOLVER_LEARNED_FGMRES, judge=0))
        _, piv = g.factor(cubens.options())
        assert np.isfinite(piv).all()
        assert np.isfinite(g.solve(g.load())).all()


@pytest.mark.parametrize("sweeps", [cubens.SWEEP_CHAIN, cubens.SWEEP_ROWS, cubens.SWEEP_LOOK2])
def test_solve_needs_a_factorization(sweeps):
    print(f"[unfactored] sweeps={sweeps}", flush=True)
    path = model_file("unfactored.txt", inputs.shell_panel(n=9).text)
    opt = cubens.options(sweep_schedule=sweeps)
    with cubens.GpuModel(path) as g:
        b = g.load()
        with pytest.raises(cubens.CubensError, match="no factorization"):
            g.solve(b)
        g.tangent(cubens.GEN_BASE, cubens.GEN_BASE)
        g.factor(opt)
        x = g.solve(b)
        assert np.isfinite(x).all() and np.abs(x).max() > 0
        # other options replace the analysis; its Krylov solve gives up after
        # two iterations and has no FP64 factor to fall back on
        g.factor(cubens.options(cubens.SOLVER_BJ_FGMRES, judge=0, maxit=2, sweep_schedule=sweeps))
        with pytest.raises(cubens.CubensError, match="tolerance"):
            g.solve(b)
        g.factor(opt)
        assert np.array_equal(g.solve(b), x)
