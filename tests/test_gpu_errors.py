"""A call that ends with an error leaves the handle usable: a factorization
that the device code refuses can be repeated, and the next one works."""
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
