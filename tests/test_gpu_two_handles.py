"""Two handles at work at once, each on a thread and a stream of its own: their
factorizations and solves wait for nothing of the other's and give the bits of a
handle alone.  Sizes with launches numbered by count (up to 1024 workgroups) and
by index, in every sweep schedule."""
import threading

import numpy as np
import pytest

import cubens
from cubens import inputs
from helpers import model_file

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sweeps", [cubens.SWEEP_CHAIN, cubens.SWEEP_ROWS, cubens.SWEEP_LOOK2])
def test_two_handles_give_the_results_of_each_alone(sweeps):
    opt = cubens.options(sweep_schedule=sweeps)
    models = [cubens.GpuModel(model_file(f"two_{n}.txt", inputs.shell_panel(n=n, thick_sigma=0.1, seed=n).text))
              for n in (40, 112)]
    try:
        alone, got, errors = [], [None, None], []
        for g in models:
            g.tangent(cubens.GEN_BASE, cubens.GEN_BASE)
            b = g.load()
            alone.append((g.factor(opt)[1], g.solve(b)))

        def work(i, reps):
            try:
                for _ in range(reps):
                    _, piv = models[i].factor(opt)
                    got[i] = (piv, models[i].solve(models[i].load()))
            except Exception as e:   # noqa: BLE001
                errors.append(e)

        print(f"[two handles] sweeps={sweeps}", flush=True)
        threads = [threading.Thread(target=work, args=a) for a in ((0, 40), (1, 6))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for a, g in zip(alone, got):
            assert np.array_equal(a[0], g[0]) and np.array_equal(a[1], g[1])
    finally:
        for g in models:
            g.close()
