"""bf_mesh_build between steps: it replaces the current step's geometry (the
next step's previous mask) by the mesh at another time, so the next step covers
and uncovers cells in tiles that the steps before it left wall-free.  Checked
against the FP32 oracle with the previous mask at that time and the current
mask at the step's own, populations bit for bit and loads (FP64 sums of the
same FP32 terms) to 1e-12; the last step's tile count in the profile is
untouched by the call."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases
from birdflow_hip import workloads

pytestmark = pytest.mark.gpu
SHAPE = (130, 22, 32)


@pytest.mark.parametrize("lead", [1, 2, 5])
def test_step_after_a_rebuild_at_another_time(lead):
    print("case: rebuild after", lead, "steps", flush=True)
    p = cases.plate_params(SHAPE)
    # heave 6 sin(2 pi t / 40): near +1..+5 while stepping, -6 at t = 30
    seq = workloads.flapping_plate(41, center=(62.0, 11.0, 16.0), span=10.0, chord=8.0, thickness=2.0, heave=6.0,
                                   pitch_deg=5.0, period=40.0)
    mask0, wall0 = cases.mesh_geometry_oracle(p, seq, 0.0)
    f, prev = bfref.init_equilibrium(p, mask0, wall0, np.float32), mask0
    ref = []
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        sim.upload_mesh(seq.points, seq.times, seq.triangles, seq.parts, seq.half_thickness)
        sim.init_equilibrium()
        sim.advance(lead)
        sim.build_mesh_geometry(30.0)
        built, _ = sim.read_geometry()
        sim.advance(3)
        got, loads = sim.read_populations(), sim.load_history(lead + 3)
    for s in range(1, lead + 4):
        mask, wall = cases.mesh_geometry_oracle(p, seq, float(s))
        f, load, _, _ = bfref.step(p, f, prev, mask, wall)
        ref.append(load)
        prev = mask
        if s == lead:
            prev, _ = cases.mesh_geometry_oracle(p, seq, 30.0)
            assert np.array_equal(built, prev) and not np.array_equal(prev, mask)
    ref = np.array(ref)
    assert np.abs(loads[:, :6] - ref[:, :6]).max() <= 1e-12 * np.abs(ref[:, :6]).max()
    assert np.array_equal(got, f)


def test_rebuild_keeps_the_last_steps_tile_count():
    p = cases.plate_params(SHAPE)
    seq = workloads.flapping_plate(41, center=(62.0, 11.0, 16.0), span=10.0, chord=8.0, thickness=2.0, heave=6.0,
                                   pitch_deg=5.0, period=40.0)
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        sim.upload_mesh(seq.points, seq.times, seq.triangles, seq.parts, seq.half_thickness)
        sim.init_equilibrium()
        sim.set_profiling(True, level=1)
        for _ in range(2):                # both parities of the list slot
            sim.advance(1)
            tiles = sim.read_profile()["general_tiles"]
            sim.build_mesh_geometry(30.0)
            assert tiles > 0 and sim.read_profile()["general_tiles"] == tiles
