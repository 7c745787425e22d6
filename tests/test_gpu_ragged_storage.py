"""Partial tiles in the kernels that the FP32 strict test does not reach.

* The two-cell kernel on rows of whole tile pairs whose count is no multiple
  of four: the rows beyond the grid store nothing and count no limiter
  activation.  Against the one-cell kernel, bit for bit.
* The one-cell kernel with 16-bit storage and fused arithmetic on ragged
  grids, odd widths among them: each step against the FP64 oracle from the
  same stored populations.  Bound: the storage's half unit in the last place
  of the stored offset (2^-11, 2^-8 relative) and 1e-5 for the FP32 arithmetic
  (populations below 1, some hundred operations of 2^-24).
* The adjoint's wall-free kernel on a grid ragged along x and y, against FP64
  central differences of the oracle: 2e-4 relative, as on whole tiles."""
import os

import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases

pytestmark = pytest.mark.gpu

WEIGHTS = np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12)
STORAGES = {"fp16": (bh.STORAGE_FP16_OFFSET, 2.0 ** -11), "bf16": (bh.STORAGE_BF16_OFFSET, 2.0 ** -8)}
FACES = {"periodic": ((0, 0),) * 3, "far": ((1, 1),) * 3, "channel": ((1, 2), (0, 0), (0, 0))}


def case(shape, collision, faces, roughness):
    n = shape[0] * shape[1] * shape[2]
    rng = np.random.default_rng(n + collision)
    p = bfref.make_params(shape, omega_plus=1.9, omega_minus=1.1, bc=FACES[faces], collision=collision, force_mode=6,
                          accumulate_loads=True, far_u=(0.05, 0.02, 0.0), sponge_strength=0.04 if faces == "far" else 0.0,
                          sponge_width=2.0, body_position=(1.0, 1.0, 1.0))
    f = (WEIGHTS[:, None] * (1.0 + roughness * rng.uniform(-1.0, 1.0, (19, n)))).astype(np.float32).ravel()
    mask = np.zeros(shape[::-1], np.uint8)
    mask[shape[2] // 2, shape[1] - 1, shape[0] // 2] = 1          # in the last row of the grid
    return p, f, mask.ravel(), np.zeros((n, 4), np.float32)


@pytest.mark.parametrize("storage", list(STORAGES))
@pytest.mark.parametrize("collision", [bfref.COLLISION_TRT_SYMMETRIC_LIMITER, bfref.COLLISION_RR3])
@pytest.mark.parametrize("faces", ["periodic", "far"])
@pytest.mark.parametrize("rows", [1, 5, 6, 7])
def test_pair_kernel_on_a_row_count_off_four(rows, faces, collision, storage, monkeypatch):
    shape = (128, rows, 4)
    print("case:", shape, faces, collision, storage, flush=True)
    p, f, mask, wall = case(shape, collision, faces, 0.9)
    out = []
    for pair in "01":
        monkeypatch.setenv("BIRDFLOW_PAIR_CELLS", pair)
        with bh.BirdFlowSimulation(cases.solver_config(p, storage=STORAGES[storage][0])) as sim:
            sim.set_geometry(mask, wall)
            sim.write_populations(f)
            sim.advance(3)
            out.append((sim.read_population_storage(), sim.load_history(3)))
    assert out[0][1][0, 6] > 0                # the limiter acts
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1].view(np.uint64), out[1][1].view(np.uint64))


@pytest.mark.parametrize("storage", list(STORAGES))
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("shape", [(63, 3, 2), (65, 5, 3), (130, 6, 5), (203, 7, 3)],
                         ids=lambda s: "x".join(map(str, s)))
def test_one_cell_kernel_with_16_bit_storage(shape, faces, storage):
    print("case:", shape, faces, storage, flush=True)
    form, unit = STORAGES[storage]
    p, f, mask, wall = case(shape, bfref.COLLISION_RR3, faces, 0.3)
    w = np.repeat(WEIGHTS, f.size // 19)
    with bh.BirdFlowSimulation(cases.solver_config(p, storage=form)) as sim:
        sim.set_geometry(mask, wall)
        sim.write_populations(f)
        for _ in range(3):
            ref, _, _, _ = bfref.step(p, sim.read_populations().astype(np.float64), mask, mask, wall)
            sim.advance(1)
            got = sim.read_populations()
            assert (np.abs(got - ref) <= unit * np.abs(ref - w) + 1e-5).all()


def test_adjoint_on_a_ragged_grid():
    shape, steps = (70, 18, 14), 6
    print("case: adjoint dJ/df0", shape, flush=True)
    n = shape[0] * shape[1] * shape[2]
    rng = np.random.default_rng(8)
    p = bfref.make_params(shape, omega_plus=1.0 / 0.56, omega_minus=1.0 / 1.1, bc=((1, 1), (1, 1), (0, 0)),
                          collision=bfref.COLLISION_RR3, wall_rule=bfref.WALL_INTERPOLATED_SDF, force_mode=6,
                          accumulate_loads=True, sponge_strength=0.3, sponge_width=4.0, far_u=(0.05, 0.01, 0.0),
                          body_position=(35.0, 9.0, 7.0))
    solid = np.zeros(shape[::-1], np.uint8)
    solid[5:9, 10:15, 60:66] = 1              # 3 rows and 4 columns from the ragged edges
    wall = np.zeros((n, 4), np.float32)
    wall[:, :3] = rng.uniform(-0.04, 0.04, (n, 3))
    wall[:, 3] = rng.uniform(-1.0, 2.0, n)
    f0 = (bfref.init_equilibrium(p, dtype=np.float32).reshape(19, n)
          * rng.uniform(0.97, 1.03, (19, n)).astype(np.float32)).ravel()
    weights = rng.normal(size=(steps, 6))
    with bh.BirdFlowSimulation(cases.solver_config(p)) as sim:
        sim.set_geometry(solid.ravel(), wall)
        sim.write_populations(f0)
        sim.adjoint_gradient(steps, weights, checkpoint_interval=2)
        lam = sim.adjoint_sensitivity().astype(np.float64)

    def objective(f):
        total = 0.0
        for s in range(steps):
            f, loads, _, _ = bfref.step(p, f, solid.ravel(), solid.ravel(), wall)
            total += float(np.dot(weights[s], loads[:6]))
        return total

    edge = lam.reshape(19, shape[2], shape[1], shape[0])
    assert np.abs(edge[:, :, 16:, :]).sum() > 0.0 and np.abs(edge[:, :, :, 64:]).sum() > 0.0
    for _ in range(2):
        delta = rng.normal(size=19 * n) * f0
        h = 1e-6
        fd = (objective(f0 + h * delta) - objective(f0 - h * delta)) / (2 * h)
        assert abs(float(np.dot(lam, delta)) - fd) <= 2e-4 * abs(fd)
