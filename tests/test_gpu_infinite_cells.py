"""Cells beyond the f16 range are stored as infinity: samples of them are infinite or
NaN, equal ones leave the heading alone.  The agents of a step over such cells equal the
oracle's, through tile windows and global memory alike, and so does what follows."""
import dataclasses

import numpy as np
import pytest

from parity_util import assert_bitwise, preset, run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge", [1.0, 0.5, 0.05])
def test_infinite_f16_cells(slm, orc, edge):
    s = dataclasses.replace(preset(slm, "Default"), pheromone_diffusion_rate=0.5)
    w, h, n = 320, 192, 60000
    rng = np.random.default_rng(6)
    t0 = rng.uniform(0, 1, (h, w)).astype(np.float32)
    t0[rng.random((h, w)) < edge] = 1e6
    a0 = np.stack([rng.uniform(0, w, n), rng.uniform(0, h, n), rng.uniform(0, 6.28, n),
                   rng.uniform(30, 50, n)], axis=1).astype(np.float32)
    a0[:4000, :2] = np.floor(a0[:4000, :2])  # weights of 0, with heading 0
    a0[:4000, 2] = 0.0
    later = []
    for tiled in (False, True):
        kw = dict(seed=3, params=s, storage="f16", resort_interval=1, graph_chunk=0,
                  tiled_sensing=tiled)
        ga, _, oa, ot = run_parity(slm, orc, w, h, n, 3, s, 1, agents0=a0, trail0=t0,
                                   **{k: v for k, v in kw.items() if k not in ("seed", "params")})
        assert np.isinf(ot).any()
        assert_bitwise(ga, oa, f"agents, tiled={tiled}")
        with slm.Simulation(w, h, n, **kw) as sim:
            sim.write_agents(a0)
            sim.write_trail(t0)
            sim.step(4)
            later.append((sim.read_agents(), sim.read_trail()))
    assert_bitwise(later[1][0], later[0][0], "agents, 4 steps")
    np.testing.assert_array_equal(later[1][1], later[0][1])
