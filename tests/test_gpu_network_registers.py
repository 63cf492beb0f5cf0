"""Batched networks whose rows fit the register-resident solver beside ones
that do not (a junction of more than four channels), at the sizes where the
rows per lane change, in both team sizes and precisions.

Each solution is held to the solver's own contract on the exported system:
the row-equilibrated residual is at most tol ||D b||, computed here in FP64
(slack 1e-13 for its own rounding: rows of at most 8 entries, values near the
inlet pressure)."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import network as NW

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 63, 64, 65, 127, 128, 129, 255, 256, 257, 383, 384, 385, 511, 512, 513, 1023, 1024, 1025, 1536, 1537,
         2047, 2048]


def build(hub_every):
    """One network per size: a ladder of width 2 (degree at most 4), and in
    every hub_every-th network a hub joined to six more nodes."""
    rng = np.random.default_rng(77)
    no, eo, ei, ej = [0], [0], [], []
    for s, n in enumerate(SIZES):
        e = [(k, k + 1) for k in range(n - 1)] + [(k, k + 2) for k in range(0, n - 2, 2)]
        if hub_every and s % hub_every == 0 and n > 20:
            e += [(1, 5 + 2 * q) for q in range(6)]
        ei += [a for a, _ in e]
        ej += [b for _, b in e]
        no.append(no[-1] + n)
        eo.append(eo[-1] + len(e))
    g = np.exp(rng.uniform(-1.0, 1.0, len(ei))) * 1e-12
    fixed = np.zeros(no[-1], np.uint8)
    value = np.zeros(no[-1])
    no = np.asarray(no)
    fixed[no[:-1]] = 1
    value[no[:-1]] = 1000.0
    fixed[no[1:] - 1] = 1
    return NW.NetworkBatch(no, np.asarray(eo), np.asarray(ei), np.asarray(ej), g, fixed, value)


@pytest.mark.parametrize("precision", [ca.Precision.FP64, ca.Precision.FP32_REFINED])
@pytest.mark.parametrize("wave_max", [0, 200, 512])
@pytest.mark.parametrize("hub_every", [0, 3, 1])
def test_register_and_memory_systems_meet_the_contract(hub_every, wave_max, precision):
    tol = 1e-10
    batch = build(hub_every)
    batch.schedule = {"wave_max_rows": wave_max, "blocks_per_cu": 2}
    x, reps = batch.solve(np.zeros(batch.n_rows),
                          ca.IterativeSolverConfig.new(tol).with_max_iterations(50000).with_precision(precision))
    rp, ci, v, b = batch.export()
    rows = np.repeat(np.arange(batch.n_rows), np.diff(rp))
    ax = np.bincount(rows, weights=v * x[ci], minlength=batch.n_rows)
    top = np.zeros(batch.n_rows)
    np.maximum.at(top, rows, np.abs(v))
    no = batch.node_offset
    for s in range(batch.n_sys):
        r = ((b - ax) / top)[no[s]:no[s + 1]]
        db = (b / top)[no[s]:no[s + 1]]
        assert reps[s].termination in (ca.Termination.Converged, ca.Termination.InitialResidual), (SIZES[s], reps[s])
        assert np.linalg.norm(r) <= (tol + 1e-13) * np.linalg.norm(db), SIZES[s]
        assert reps[s].precision == precision


def test_register_system_iteration_limit_and_warm_start():
    batch = build(0)
    cfg = ca.IterativeSolverConfig.new(1e-10).with_max_iterations(5)
    x, reps = batch.solve(np.zeros(batch.n_rows), cfg)
    assert reps[-1].termination == ca.Termination.MaxIterations and reps[-1].iterations == 5
    full = ca.IterativeSolverConfig.new(1e-10).with_max_iterations(50000)
    x, _ = batch.solve(x, full)
    _, again = batch.solve(x, full)
    assert all(r.termination == ca.Termination.InitialResidual and r.iterations == 0 for r in again)
