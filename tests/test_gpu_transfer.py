"""Host copies through the pinned slots (bf_transfer.hip): populations written
and read back unchanged, and density read with velocity in one transfer, for
sizes on both sides of each choice it makes: one slot and one wait (below
4 MB), two threads, all threads with a ragged last block, several blocks per
thread.  Bytes are moved, so the comparison is exact; density and velocity
are the FP32 sums of the FP32 oracle."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 3, 2), (64, 27, 16), (53, 104, 10), (110, 73, 41), (128, 100, 71)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("storage", [bh.STORAGE_FP32, bh.STORAGE_FP16_OFFSET])
def test_round_trip(shape, storage):
    print("case:", shape, storage, flush=True)
    n = shape[0] * shape[1] * shape[2]
    rng = np.random.default_rng(n)
    cfg = bh.SolverConfig(shape=shape, omega_plus=1.2, omega_minus=1.1, storage=storage)
    with bh.BirdFlowSimulation(cfg) as sim:
        raw = (rng.uniform(0.02, 0.06, 19 * n).astype(np.float32) if storage == bh.STORAGE_FP32
               else rng.integers(0, 0x3000, 19 * n).astype(np.uint16))
        for _ in range(2):      # the second copy reuses the slots
            sim.write_population_storage(raw)
            assert np.array_equal(sim.read_population_storage(), raw)
            raw = raw[::-1].copy()
        f = sim.read_populations()
        sim.write_populations(f)
        assert np.array_equal(sim.read_populations(), f)
        rho, u = sim.copy_macroscopic_fields()
    ref_rho, ref_u = bfref.moments(bfref.make_params(shape, omega_plus=1.2, omega_minus=1.1), f)
    assert np.array_equal(rho, ref_rho) and np.array_equal(u, ref_u)
