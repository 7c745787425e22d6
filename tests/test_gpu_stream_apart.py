"""The wall-free tiles in a launch of their own (fluid_stream) against the one
launch for both kinds of tile (fluid_step): the cells' arithmetic is the same,
so populations, loads and limiter counts are equal bit for bit.  BIRDFLOW_APART
forces either form at sizes where the rules would take the other; a moving
mesh, a static obstacle, a coupled flight with its reduction and geometry beside
the streaming, whole and partial tiles, every storage.  Without wall tiles the
form follows the kernel and the size: the one-cell kernel beyond a million
cells against the two-cell kernel."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases
from birdflow_hip import workloads

pytestmark = pytest.mark.gpu
STORAGES = {"fp32": bh.STORAGE_FP32, "fp16": bh.STORAGE_FP16_OFFSET, "bf16": bh.STORAGE_BF16_OFFSET}
STEPS = 7


def plate(shape, storage, collision):
    p = cases.plate_params(shape)
    p.collision = collision
    seq = workloads.flapping_plate(STEPS + 1, center=(shape[0] / 2 - 2.0, 11.0, 16.0), span=10.0, chord=8.0,
                                   thickness=2.0, heave=2.0, pitch_deg=5.0, period=120.0)
    sim = bh.BirdFlowSimulation(cases.solver_config(p, storage=storage))
    sim.upload_mesh(seq.points, seq.times, seq.triangles, seq.parts, seq.half_thickness)
    return sim


def obstacle(shape, storage, collision):
    p = cases.plate_params(shape)
    p.collision = collision
    mask = np.zeros(shape[::-1], np.uint8)
    mask[12:16, 8:14, 60:67] = 1
    sim = bh.BirdFlowSimulation(cases.solver_config(p, storage=storage))
    sim.set_geometry(mask.ravel(), np.tile(np.float32([0.01, 0.0, 0.0, 0.3]), (mask.size, 1)))
    return sim


def flight(shape, storage, collision):
    p, cfg, geometry, _, sc = cases.compact_bird_case(free_flight=True, shape=shape)
    cfg.storage, cfg.collision = storage, collision
    sim = bh.BirdFlowSimulation(cfg)
    pose = list(cfg.body_position) + [0.0, 0.0, 0.0, 1.0] + [0.0] * 6
    sim.set_body(pose, bh.BodyParameters(mass=1e-4, inertia=(1e-8, 1e-8, 1e-8), gravity=(0.0, 0.0, -9.81)))
    sim.set_bird(geometry)
    return sim


CASES = {"plate": (plate, [(128, 22, 32), (130, 22, 32)]), "obstacle": (obstacle, [(128, 22, 32), (130, 22, 32)]),
         "flight": (flight, [(128, 48, 48), (61, 50, 48)])}


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


@pytest.mark.parametrize("storage", ["fp16", "bf16"])
@pytest.mark.parametrize("planes", [81, 82])              # 995,328 and 1,007,616 cells
def test_a_box_without_wall_tiles(planes, storage, monkeypatch):
    shape = (128, 96, planes)
    print("case: box", shape, storage, flush=True)
    p = bfref.make_params(shape, omega_plus=1.6, omega_minus=1.1, collision=bfref.COLLISION_RR3)
    f = bfref.init_equilibrium(p, dtype=np.float32)
    f = f * np.random.default_rng(5).uniform(0.8, 1.2, f.size).astype(np.float32)
    out = []
    for pair in "01":
        monkeypatch.setenv("BIRDFLOW_PAIR_CELLS", pair)
        with bh.BirdFlowSimulation(cases.solver_config(p, storage=STORAGES[storage])) as sim:
            sim.write_populations(f)
            sim.advance(3)
            out.append(sim.read_population_storage())
    assert np.array_equal(*out)
