"""The wing's link queue (wing_links: a tile's links collected in LDS, then
spread over the lanes): every fraction equals the oracle's bit for bit where
the queue can go wrong: tiles cut by the grid's edges, more links in a tile
than lanes (a thick coarse wing), a wing across a periodic face (sources
wrapped into another tile) and beside an outlet (clamped)."""
import numpy as np
import pytest

import bfref
import birdflow_hip as bh
import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,root,chord,face", [((64, 64, 32), (32.0, 32.0, 16.0), 8.0, 1),
                                                   ((70, 61, 33), (35.0, 30.0, 16.0), 8.0, 1),
                                                   ((130, 130, 40), (66.0, 64.0, 20.0), 18.0, 0),
                                                   ((66, 66, 33), (62.0, 32.0, 16.0), 8.0, 2)],
                         ids=["whole tiles", "ragged", "crowded tiles, periodic", "outlet"])
def test_link_table_matches_the_oracle(shape, root, chord, face):
    print("case:", shape, root, chord, face, flush=True)
    bc = ((face, face),) * 3
    p = bfref.make_params(shape, omega_plus=1.6, omega_minus=1.2, bc=bc, wall_rule=bfref.WALL_INTERPOLATED_LINKS,
                          force_mode=6, accumulate_loads=True, body_position=root)
    cfg = cases.solver_config(p, time_step=2.0, velocity_to_lattice=0.05)
    wing, ow = bh.FlappingWing.li_nabawy(chord, root, 200.0), bfref.li_nabawy_wing(chord, root, 200.0)
    with bh.BirdFlowSimulation(cfg) as sim:
        sim.set_flapping_wing(wing)
        prev = None
        for s in range(4):
            fr = bfref.wing_prepare(ow, np.float32(2.0 * s))
            mask, _ = bfref.wing_build(p, ow, fr, prev, 0.05)
            got, _ = sim.read_geometry()
            assert np.array_equal(got, mask) and mask.any()
            ref = np.asarray(bfref.wing_links(p, ow, fr, mask), np.float32)
            at = ref != 0                 # the links: a fraction is at least 1e-4
            assert at.sum() > 1000 and np.array_equal(sim.wing_links().ravel()[at], ref[at])
            prev = mask
            sim.advance(1)
