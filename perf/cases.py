"""The work that users of this library have it do, as cases that can be timed.

A case is one call, or one short sequence of calls, of the public interface
(include/cubens.h through its Python mirror, cu-bens_amd/cubens).  The models
are those of the repository's generators (cubens.inputs): the truss dome, the
hinged shell panel whose 256 x 256 mesh is the headline benchmark, and the
space frames of the batch benchmark, at sizes from the smallest that the
tests run up to the benchmark's.

Kinds of case:
  dome        a whole Newton-Raphson analysis of a small truss: launches,
              copies and waits rather than arithmetic
  msal        the arc-length driver on the shell panel, from its first
              increment (a tangent, a factorization and about four solves
              per increment)
  factor      one factorization of a tangent that has just been assembled, with
              its pivots, as a program that keeps its own driver calls it
  solve       one back-substitution with a factor in hand (the modified Newton
              and arc-length loops do about a dozen per factorization)
  iteration   the routine-level binding: tangent, factorization, solve,
              geometry update and internal forces, each through its own call
              with host vectors
  fp32        the FP32 precision mode of the static drivers
  newmark     the nonlinear Newmark driver on one space frame
  batch       many space frames side by side, each on its own time steps
  learned     loss and gradient of the learned preconditioner's network
"""
import math
import os
import sys
import tempfile

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cu-bens_amd"))

import cubens  # noqa: E402
from cubens import inputs  # noqa: E402


def listed():
    return [
        # the 10 x 10 bay dome under Newton-Raphson (the smallest model of the
        # tests: 243 equations), five load steps
        {"name": "dome_nr", "kind": "dome", "n": 10, "steps": 5},
        # the smoke-test panel: 432 equations, everything is latency
        {"name": "panel8_msal", "kind": "msal", "n": 8, "steps": 4, "sweeps": 0},
        # the 64 x 64 panel with the library's default options
        {"name": "panel64_msal", "kind": "msal", "n": 64, "steps": 3, "sweeps": 0},
        # the headline benchmark's panel and sweep schedule, two increments
        {"name": "panel256_msal", "kind": "msal", "n": 256, "steps": 2, "sweeps": 2},
        # factorization and pivots of a large panel
        {"name": "panel200_factor", "kind": "factor", "n": 200},
        # back-substitution: a small panel and the benchmark's
        {"name": "panel24_solve", "kind": "solve", "n": 24, "sweeps": 0},
        {"name": "panel256_solve", "kind": "solve", "n": 256, "sweeps": 0},
        # one iteration of a driver that calls the routines one by one
        {"name": "panel97_iteration", "kind": "iteration", "n": 97},
        # FP32 tangent and factor with one refinement step per solve
        {"name": "panel64_fp32", "kind": "fp32", "n": 64},
        # a 400-member tower under Newmark
        {"name": "tower400_newmark", "kind": "newmark", "shape": "tower", "members": 400, "steps": 10},
        # 64 frames of 200 to 5000 members side by side, one graph per round
        {"name": "frames64_batch", "kind": "batch", "count": 64, "lo": 200, "hi": 5000, "steps": 4},
        # the network's training gradient on a 32 x 32 panel
        {"name": "panel32_learned", "kind": "learned", "n": 32, "vectors": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dome", "msal", "msal", "factor", "solve", "solve", "iteration", "fp32", "newmark", "batch",
                       "learned"])
    if kind == "dome":
        return {"kind": kind, "n": rng.randint(4, 14), "steps": rng.randint(1, 12)}
    if kind == "msal":
        n = _log_int(rng, 6, 230)
        return {"kind": kind, "n": n, "steps": rng.randint(1, 4) if n < 100 else rng.randint(1, 2),
                "sweeps": rng.choice([0, 0, 1, 2])}
    if kind == "factor":
        return {"kind": kind, "n": _log_int(rng, 5, 250)}
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 5, 256), "sweeps": rng.choice([0, 0, 1, 2])}
    if kind == "iteration":
        return {"kind": kind, "n": _log_int(rng, 6, 180)}
    if kind == "fp32":
        return {"kind": kind, "n": _log_int(rng, 8, 72)}
    if kind == "newmark":
        return {"kind": kind, "shape": rng.choice(["tower", "grid"]), "members": _log_int(rng, 60, 5000),
                "steps": rng.randint(2, 8)}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(5, 64), "lo": rng.choice([60, 200]), "hi": _log_int(rng, 400, 5000),
                "steps": rng.randint(2, 4)}
    return {"kind": kind, "n": _log_int(rng, 6, 48), "vectors": rng.randint(1, 7)}


# ---- models -----------------------------------------------------------------
def _panel(n, seed):
    """The benchmark's panel with thickness field and imperfection of this seed."""
    return inputs.shell_panel(n=n, thick_sigma=0.1, imperfection=0.1, seed=seed)


def _frame(members, shape, girder, seed, steps):
    """A tower, or a girder of the given cross-section, with a load history a little longer than the run."""
    return inputs.space_frame(members, kind=shape, slice_shape=girder, seed=seed, steps=steps + 2)


def _open(text, cls=cubens.GpuModel):
    with tempfile.TemporaryDirectory(prefix="cubens_cases_") as d:
        if isinstance(text, list):
            return cls([m.write(os.path.join(d, f"model{i}.txt")) for i, m in enumerate(text)])
        return cls(text.write(os.path.join(d, "model.txt")))


def _panel_neq(n):
    return 6 * (n + 1) * (n + 1) - 6 * (n + 1)


def _panel_band(n):
    return 6 * (n + 2)


def _rhs(g, rng):
    """A residual-like right-hand side: the load and small forces everywhere."""
    return g.load() + 0.1 * rng.standard_normal(g.neq)


def _call(rc):
    if rc != 0:
        raise cubens.CubensError(cubens.lib().cb_last_error().decode(errors="replace"))


# ---- preparation ------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = {"case": case}
    if kind == "dome":
        # a load that keeps the crown of every draw on its stable branch
        s["g"] = _open(inputs.truss_dome(n=case["n"], load=-20.0, seed=seed, steps=20))
        s["opt"] = cubens.options(max_steps=case["steps"])
    elif kind == "msal":
        s["g"] = _open(_panel(case["n"], seed))
        s["opt"] = cubens.options(max_steps=case["steps"], sweep_schedule=case["sweeps"])
    elif kind == "fp32":
        s["g"] = _open(_panel(case["n"], seed))
        # one increment: the arc of the next one would follow the iteration
        # count, which the rounding of an FP32 correction can change
        s["opt"] = cubens.options(cubens.SOLVER_BAND32, refine=1, judge=0, max_steps=1)
    elif kind in ("factor", "solve", "iteration"):
        g = s["g"] = _open(_panel(case["n"], seed))
        _call(cubens.lib().cb_tangent(g.h, cubens.GEN_BASE, cubens.GEN_BASE))
        s["opt"] = cubens.options(sweep_schedule=case.get("sweeps", 0))
        g.factor(s["opt"])              # the band and its workspaces are the handle's
        s["b"] = _rhs(g, rng)
        s["x0"] = g.get("x", g.nj * 3)
    elif kind == "newmark":
        s["g"] = _open(_frame(case["members"], case["shape"], (3, 3), seed, case["steps"]))
        s["opt"] = cubens.options(max_steps=case["steps"])
    elif kind == "batch":
        # sizes spread evenly over the range, towers and girders alternating;
        # the seed draws sections, spacings, loads and frequencies
        sizes = np.linspace(case["hi"], case["lo"], case["count"]).astype(int)
        models = [_frame(int(m), ("tower", "grid")[i % 2], (2 + i // 2 % 3, 2 + i // 6 % 3), seed + 7919 * (i + 1),
                         case["steps"]) for i, m in enumerate(sizes)]
        s["b"] = _open(models, cubens.GpuBatch)
    elif kind == "learned":
        g = s["g"] = _open(_panel(case["n"], seed))
        _call(cubens.lib().cb_tangent(g.h, cubens.GEN_BASE, cubens.GEN_BASE))
        g.factor(cubens.options())
        s["r"] = rng.standard_normal((case["vectors"], g.neq))
        s["u"] = np.stack([g.solve(r) for r in s["r"]])
        net = s["net"] = cubens.LearnedPrecond(int(seed) % (1 << 31))
        # a network some way into its training: the decoder of a new one is zero
        p = net.params()
        net.set_params(p + np.where(p == 0, 0.02, 0.0).astype(np.float32)
                       * rng.standard_normal(p.size).astype(np.float32))
    else:
        raise ValueError(kind)
    return s


# ---- one pass ----------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("dome", "msal", "newmark"):
        r = s["g"].run(s["opt"])
        return {"lpf": r["lpf"], "itecnt": r["itecnt"], "d": r["d"]}
    if kind == "fp32":
        r = s["g"].run(s["opt"])
        return {"lpf": r["lpf"], "d": r["d"]}
    if kind == "factor":
        det, piv = s["g"].factor(s["opt"])
        return {"det": det, "pivots": piv}
    if kind == "solve":
        return s["g"].solve(s["b"])
    if kind == "iteration":
        g = s["g"]
        _call(cubens.lib().cb_tangent(g.h, cubens.GEN_BASE, cubens.GEN_BASE))
        det, piv = g.factor(s["opt"])
        dd = g.solve(s["b"]) * 1e-2
        g.set("x_temp", s["x0"])
        g.update_geometry(dd, cubens.GEN_I)
        f = g.internal_force(dd, cubens.GEN_I)
        return {"pivots": piv, "dd": dd, "f": f}
    if kind == "batch":
        b = s["b"]
        b.run(max_steps=case["steps"], graph=True)
        paths = [b.path(i) for i in range(b.count)]
        return {"t": np.concatenate([p["lpf"] for p in paths]),
                "itecnt": np.concatenate([p["itecnt"] for p in paths]),
                "d": np.concatenate([p["d"].ravel() for p in paths])}
    if kind == "learned":
        loss, grad = s["net"].loss_grad(s["g"], s["r"], s["u"])
        return {"loss": loss, "grad": grad}
    raise ValueError(kind)


# ---- what a pass cannot do without --------------------------------------------
def _banded(neq, band, factors, solves, word=8):
    """LDL^T of a band: neq * band^2 flops and the factor written once per
    factorization; a solve reads the factor twice (forward and back)."""
    entries = neq * band
    return {"flops": factors * neq * float(band) ** 2 + solves * 4.0 * entries,
            "bytes": float(word) * entries * (factors + 2 * solves)}


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "dome":
        steps = case["steps"]       # about four iterations per load step
        return _banded(3 * (n - 1) ** 2, 3 * (n + 2), 4 * steps, 4 * steps)
    if kind == "msal":
        return _banded(_panel_neq(n), _panel_band(n), case["steps"], 4 * case["steps"])
    if kind == "fp32":              # each solve with its refinement step
        return _banded(_panel_neq(n), _panel_band(n), 1, 8, word=4)
    if kind == "factor":
        return _banded(_panel_neq(n), _panel_band(n), 1, 0)
    if kind == "solve":
        return _banded(_panel_neq(n), _panel_band(n), 0, 1)
    if kind == "iteration":
        w = _banded(_panel_neq(n), _panel_band(n), 1, 1)
        ne = 2 * n * n              # per element 8.6 and 3.4 kflop, 1612 and 900 bytes
        return {"flops": w["flops"] + 12000.0 * ne, "bytes": w["bytes"] + 2512.0 * ne}
    if kind == "newmark":           # about two iterations per time step
        neq, it = _frame_neq(case["members"], case["shape"]), 2 * case["steps"]
        return _banded(neq, 48, it, it)
    if kind == "batch":
        members = case["count"] * (case["lo"] + case["hi"]) / 2.0
        it = 2 * case["steps"]
        return _banded(_frame_neq(members, "tower"), 48, it, it)
    if kind == "learned":
        joints = (n + 1) ** 2
        edges = 3 * n * n + 2 * n   # edges of the triangulated grid
        # three passes (forward, and the two products of the backward one)
        # over an encoder, three layers and a decoder of 64 hidden units
        return {"flops": 3 * 2.0 * (joints + edges) * (48 * 64 + 3 * 3 * 64 * 64 + 64 * 36),
                "bytes": 8.0 * 36 * (joints + 2 * edges) + 16.0 * case["vectors"] * _panel_neq(n)}
    raise ValueError(kind)


def _frame_neq(members, shape):
    return 1.5 * members if shape == "tower" else 2.4 * members


def tolerance(case):
    kind = case["kind"]
    # four times what the sweep schedules, which sum in different orders, differ
    # by over these sizes: 1e-13 (8 x 8) to 1e-11 (150 x 150) of a path, 2e-15
    # of a solution, 1e-8 of an FP32 path (its state, not its factor, in other
    # orders) and 1.5e-5 with another refinement step
    if kind in ("dome", "msal", "newmark", "batch"):
        return {"rel": 1e-9, "max": 4e-8}
    if kind == "fp32":
        return {"rel": 1e-4, "max": 2e-3}
    if kind in ("factor", "solve"):
        return {"rel": 1e-11, "max": 1e-9}
    if kind == "iteration":
        return {"rel": 1e-9, "max": 4e-8}
    return {"rel": 2e-2, "max": 0.8}            # bf16 operands


def exact(case, seed):
    """Pivots and solutions of small panels from numpy's dense factorization of
    the assembled tangent, which is these cases' input."""
    kind, n = case["kind"], case.get("n", 0)
    if kind not in ("factor", "solve") or n > 28:
        return None
    s = prepare(case, seed)
    g = s["g"]
    jcode, _, _ = g.dofmaps()
    rowptr, colidx = g.pattern()
    vals = g.tangent()
    K = cubens.bsr_to_dense(vals, rowptr, colidx, g.info.bs, cubens.eq_of_slot(jcode, g.nj, g.info.bs), g.neq)
    if kind == "factor":
        d = np.diagonal(np.linalg.cholesky(K)) ** 2
        return {"det": None, "pivots": d}
    x = np.linalg.solve(K, s["b"])
    return x + np.linalg.solve(K, s["b"] - K @ x)
