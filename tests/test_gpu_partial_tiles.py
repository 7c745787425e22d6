"""Partial tiles (grids whose sides are not multiples of the 64 x 4 tile)
stream in the fast kernel: lanes beyond the grid load the last column / row
and store nothing.  Strict FP32 against the FP32 oracle, bit for bit, on sides
one below, at and one above the tile's, with populations rough enough that
the positivity limiters act, with and without an obstacle.  The limiter
counts of both kinds of tile must add up exactly (an integer and a maximum);
the force is an FP64 sum of the same FP32 terms in another order: 1e-12."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (63, 3, 2), (64, 4, 2), (65, 5, 3), (128, 9, 4), (130, 6, 5)]
FACES = {"periodic": ((0, 0),) * 3, "far": ((1, 1),) * 3, "channel": ((1, 2), (0, 0), (0, 0))}


@pytest.mark.parametrize("collision", [bfref.COLLISION_TRT, bfref.COLLISION_TRT_SYMMETRIC_LIMITER,
                                       bfref.COLLISION_RR3])
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_partial_tiles_match_the_oracle(shape, faces, collision):
    print("case:", shape, faces, collision, flush=True)
    n = shape[0] * shape[1] * shape[2]
    rng = np.random.default_rng(n + collision)
    p = bfref.make_params(shape, omega_plus=1.9, omega_minus=1.1, bc=FACES[faces], collision=collision, force_mode=6,
                          accumulate_loads=True, far_u=(0.05, 0.02, 0.0), sponge_strength=0.04 if faces == "far" else 0.0,
                          sponge_width=2.0, body_position=(1.0, 1.0, 1.0))
    w = np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12)
    f = (w[:, None] * (1.0 + 0.9 * rng.uniform(-1.0, 1.0, (19, n)))).astype(np.float32).ravel()
    mask = np.zeros(n, np.uint8)
    if shape[0] == 130:
        mask[70 + 130 * (2 + 6 * 2)] = 1       # one solid cell in the second tile column
    wall = np.zeros((n, 4), np.float32)
    steps = 3
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        sim.set_geometry(mask, wall)
        sim.write_populations(f)
        sim.advance(steps)
        got, loads = sim.read_populations(), sim.load_history(steps)
    for s in range(steps):
        f, ref, _, _ = bfref.step(p, f, mask, mask, wall)
        scale = max(np.abs(ref[:6]).max(), 1e-30)
        assert np.abs(loads[s, :6] - ref[:6]).max() <= 1e-12 * scale
        assert loads[s, 6] == ref[6] and loads[s, 7] == ref[7]
    if collision != bfref.COLLISION_TRT and n > 100:
        assert loads[0, 6] > 0
    assert np.array_equal(got, f)
