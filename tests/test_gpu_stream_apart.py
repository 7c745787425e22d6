"""The wall-free tiles in a launch of their own (fluid_stream) against the one
kernel for both kinds of tile (fluid_step): the cells' arithmetic is the same,
so populations, loads and the body are equal bit for bit.  BIRDFLOW_APART forces
either form at sizes where the rule would take the other, in a coupled flight
with its reduction and geometry beside the streaming, on whole and partial
tiles, for every storage."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases

pytestmark = pytest.mark.gpu
STORAGES = {"fp32": bh.STORAGE_FP32, "fp16": bh.STORAGE_FP16_OFFSET, "bf16": bh.STORAGE_BF16_OFFSET}
STEPS = 7


def flight(shape, storage, collision):
    p, cfg, geometry, _, sc = cases.compact_bird_case(free_flight=True, shape=shape)
    cfg.storage, cfg.collision = storage, collision
    sim = bh.BirdFlowSimulation(cfg)
    pose = list(cfg.body_position) + [0.0, 0.0, 0.0, 1.0] + [0.0] * 6
    sim.set_body(pose, bh.BodyParameters(mass=1e-4, inertia=(1e-8, 1e-8, 1e-8), gravity=(0.0, 0.0, -9.81)))
    sim.set_bird(geometry)
    return sim


CASES = {"flight": (flight, [(128, 48, 48), (61, 50, 48)])}


@pytest.mark.parametrize("storage", list(STORAGES))
@pytest.mark.parametrize("collision", [bfref.COLLISION_TRT, bfref.COLLISION_TRT_SYMMETRIC_LIMITER,
                                       bfref.COLLISION_REGULARIZED, bfref.COLLISION_RR3])
@pytest.mark.parametrize("case", list(CASES))
def test_one_launch_and_two_are_bit_identical(case, collision, storage, monkeypatch):
    make, shapes = CASES[case]
    for shape in shapes:
        print("case:", case, shape, collision, storage, flush=True)
        rough, out = None, []
        for apart in "01":
            monkeypatch.setenv("BIRDFLOW_APART", apart)
            with make(shape, STORAGES[storage], collision) as sim:
                sim.init_equilibrium()
                f = sim.read_populations()
                if rough is None:
                    rough = np.random.default_rng(4).uniform(0.8, 1.2, f.size).astype(np.float32)
                sim.write_populations(f * rough)
                sim.advance(3)
                sim.set_profiling(True, level=2)          # each kind of tile in a launch of its own
                sim.advance(1)
                sim.set_profiling(False)
                sim.advance(STEPS - 4)
                out.append((sim.read_population_storage(), sim.load_history(STEPS), sim.body_state()))
        for a, b in zip(*out):
            assert np.isfinite(a.astype(np.float64)).all() and np.array_equal(a, b)

