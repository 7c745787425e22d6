"""Static geometry steps without rebuilding its wall-tile list and reduces
its loads in batches (bf_api.hip: step_static, at most 4 steps a batch): any
split of the steps into calls gives the same populations and load history bit
for bit, a previous mask of the caller's counts for the first step alone
(checked against the FP32 oracle), and a later geometry replaces the list."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases

pytestmark = pytest.mark.gpu
SHAPE = (70, 18, 12)


def setup(seed, differs):
    n = SHAPE[0] * SHAPE[1] * SHAPE[2]
    rng = np.random.default_rng(seed)
    p = bfref.make_params(SHAPE, omega_plus=1.5, omega_minus=1.2, collision=bfref.COLLISION_RR3, force_mode=6,
                          accumulate_loads=True, wall_rule=bfref.WALL_INTERPOLATED_SDF, body_position=(35.0, 9.0, 6.0))
    mask = np.zeros(SHAPE[::-1], np.uint8)
    mask[4:7, 6:10, 60:67] = 1            # across a tile edge
    prev = mask.copy()
    if differs:
        prev[4:7, 6:10, 60] = 0           # covered by the first step
        prev[4:7, 6:10, 67] = 1           # uncovered by it
    wall = rng.uniform(-0.02, 0.02, (n, 4)).astype(np.float32)
    wall[:, 3] = np.where(mask.ravel() != 0, -0.4, 0.7)
    f = (bfref.init_equilibrium(p, mask.ravel(), wall) * rng.uniform(0.98, 1.02, 19 * n)).astype(np.float32)
    return p, prev.ravel(), mask.ravel(), wall, f


def run(p, prev, mask, wall, f, calls):
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        sim.set_geometry(np.zeros_like(mask), wall)
        sim.advance(2)                    # an empty list first
        sim.set_geometry(mask, wall, mask_prev=prev)
        sim.write_populations(f)
        for k in calls:
            sim.advance(k)
        return sim.read_populations(), sim.load_history(sum(calls)), sim.read_loads()


@pytest.mark.parametrize("differs", [False, True])
@pytest.mark.parametrize("calls", [[1] * 9, [4, 5], [3, 1, 5]], ids=str)
def test_batches_match_one_call_and_the_oracle(calls, differs):
    print("case:", calls, differs, flush=True)
    p, prev, mask, wall, f = setup(3, differs)
    whole, loads, last = run(p, prev, mask, wall, f, [9])
    got, split, split_last = run(p, prev, mask, wall, f, calls)
    assert np.array_equal(got, whole) and np.array_equal(split, loads) and np.array_equal(split_last, last)
    assert np.array_equal(last, loads[-1])
    for s in range(9):
        f, ref, _, _ = bfref.step(p, f, prev, mask, wall)
        prev = mask
        assert np.abs(loads[s, :6] - ref[:6]).max() <= 1e-12 * np.abs(ref[:6]).max()
    assert np.array_equal(whole, f)
