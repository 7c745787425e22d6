"""An adjoint sweep leaves the stepping state as the same number of plain
steps leaves it: with exact-root link fractions the recompute builds the link
tables of earlier steps again, of both parities, and the next step's table is
already there.  Against a twin that only steps, bit for bit: the current
table, the populations and loads of the steps that follow, and the objective
of a second sweep."""
import dataclasses

import numpy as np
import pytest

import birdflow_hip as bh
import cases
from birdflow_hip import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps,interval", [(6, 3), (5, 5), (7, 2)])
def test_steps_after_an_exact_root_sweep(steps, interval):
    print("case: exact roots,", steps, "steps, interval", interval, flush=True)
    p = cases.plate_params((96, 48, 48))
    seq = workloads.flapping_plate(2 * steps + 4, center=(24.0, 24.0, 24.0), span=20.0, chord=8.0, thickness=2.0,
                                   heave=4.0, period=60.0)
    config = dataclasses.replace(cases.solver_config(p), wall_rule=bh.WALL_INTERPOLATED_RAY)
    weights = np.random.default_rng(steps).normal(size=(steps, 6))
    with bh.BirdFlowSimulation(config) as swept, bh.BirdFlowSimulation(config) as plain:
        for sim in (swept, plain):
            sim.upload_mesh(seq.points, seq.times, seq.triangles, seq.parts, seq.half_thickness)
            sim.init_equilibrium()
        swept.adjoint_gradient(steps, weights, interval)
        plain.advance(steps)
        assert np.array_equal(swept.ray_links(), plain.ray_links())
        assert np.array_equal(swept.read_populations(), plain.read_populations())
        swept.advance(3)
        plain.advance(3)
        assert np.array_equal(swept.read_populations(), plain.read_populations())
        assert np.array_equal(swept.load_history(steps + 3), plain.load_history(steps + 3))
        objective, _, _ = swept.adjoint_gradient(steps, weights, interval)
        plain.advance(steps)
        assert objective == pytest.approx((weights * plain.load_history(steps)[:, :6]).sum(), rel=1e-12, abs=1e-12)
        assert np.array_equal(swept.read_populations(), plain.read_populations())
