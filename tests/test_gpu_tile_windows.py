"""The agent pass's tile windows: bit for bit the oracle's step, wherever the
windows are staged, clipped by the grid, too large, or left to global memory."""
import dataclasses

import numpy as np
import pytest

from parity_util import assert_bitwise, preset, run_parity

pytestmark = pytest.mark.gpu

# grids at the edges of 64-cell tiles and of rows of whole 16-byte chunks; windows
# that the grid clips on every side, on one, on none; reaches from 20 cells (staged)
# to 225 (whole-grid windows on small grids, none on larger ones)
FORCED = [
    dict(w=64, h=64, n=5000, storage="f32", name="Default", resort=1, cl=4),
    dict(w=65, h=63, n=4500, storage="bf16", name="Waves", resort=3, cl=3),
    dict(w=129, h=257, n=40000, storage="f16", name="Sponge", resort=4, cl=4),
    dict(w=384, h=320, n=130000, storage="f32", name="Firecracker Trees", resort=5, cl=3),
    dict(w=385, h=321, n=60000, storage="bf16", name="Default", resort=7, cl=4),
    dict(w=386, h=250, n=100000, storage="f16", name="Curls", resort=2, cl=2),
    dict(w=3, h=4000, n=9000, storage="f32", name="Default", resort=3, cl=4),
    dict(w=2050, h=5, n=9000, storage="bf16", name="Threads", resort=3, cl=4),
    dict(w=150, h=140, n=20000, storage="f32", name="Snake", resort=3, cl=4),
    dict(w=600, h=500, n=80000, storage="f32", name="Mesh", resort=3, cl=7),
]


@pytest.mark.parametrize("c", FORCED, ids=lambda c: f"{c['w']}x{c['h']}-{c['storage']}-{c['name'].replace(' ', '')}")
def test_forced_tile_windows_equal_the_oracle(slm, orc, c):
    ga, gt, oa, ot = run_parity(slm, orc, c["w"], c["h"], c["n"], 17, preset(slm, c["name"]), 9,
                                storage=c["storage"], resort_interval=c["resort"],
                                sort_cell_log2=c["cl"], graph_chunk=4, tiled_sensing=True)
    assert_bitwise(ga, oa, "agents")
    assert_bitwise(gt, ot, "trail")


@pytest.mark.parametrize("fields", [
    dict(agent_sensor_distance=-20.0), dict(agent_turn_speed=7.0), dict(agent_turn_speed=-0.3),
    dict(agent_sensor_angle=1500.0), dict(agent_speed_min=60.0, agent_speed_max=40.0),
    dict(agent_speed_min=-2000.0, agent_speed_max=2000.0), dict(agent_sensor_distance=5000.0),
    dict(pheromone_deposition_amount=0.25, agent_jitter=9.0)],
    ids=lambda f: "-".join(f"{k}{v}" for k, v in f.items()))
def test_tile_windows_outside_the_ordinary_range(slm, orc, fields):
    """Parameters and states that the windows' update hands to the general one,
    and angles, positions and speeds that a caller may write."""
    s = dataclasses.replace(preset(slm, "Default"), **fields)
    w, h, n = 200, 141, 30000
    rng = np.random.default_rng(23)
    a = np.stack([rng.uniform(0, w, n), rng.uniform(0, h, n), rng.uniform(-7, 7, n),
                  rng.uniform(20, 60, n)], axis=1).astype(np.float32)
    a[:64, 2] = 5000.0
    a[100:164, 2] = -2048.0
    a[200:204, :2] = [[0, 0], [w, h], [w, 0], [0, h]]
    a[300, 2] = -0.0
    ga, gt, oa, ot = run_parity(slm, orc, w, h, n, 3, s, 6, agents0=a, resort_interval=2,
                                graph_chunk=0, tiled_sensing=True,
                                trail0=rng.uniform(0, 1, (h, w)).astype(np.float32))
    assert_bitwise(ga, oa, "agents")
    assert_bitwise(gt, ot, "trail")


@pytest.mark.parametrize("w,h,storage,chunk", [(1600, 900, "f32", 4), (1601, 903, "bf16", 0)])
def test_windows_chosen_by_the_library_equal_the_oracle(slm, orc, w, h, storage, chunk):
    """2^21 agents: windows of the library's own accord, over preset changes under
    captured graphs (20-cell sensors, 225-cell ones, back) and a state written
    between two re-sorts."""
    n = 1 << 21
    presets = [preset(slm, p) for p in ("Default", "Snake", "Firecracker Trees")]
    with slm.Simulation(w, h, n, seed=4, params=presets[0], storage=storage, resort_interval=5,
                        graph_chunk=chunk) as sim:
        a, t = sim.read_agents(), sim.read_trail()
        for k, s in enumerate(presets):
            sim.set_params(s)
            sim.step(4)
            orc.step(a, t, s, 4, storage=storage)
            if k == 0:  # agents back in their first order, far from their tiles
                sim.write_agents(a)
                sim.step(1)
                orc.step(a, t, s, 1, storage=storage)
        assert_bitwise(sim.read_agents(), a, "agents")
        assert_bitwise(sim.read_trail(), t, "trail")


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
def test_tile_windows_with_f64_positions(slm, storage):
    """f64 positions: windows give what global memory gives."""
    s = preset(slm, "Firecracker Trees")
    got = []
    for tiled in (False, True):
        with slm.Simulation(391, 300, 120000, seed=8, params=s, storage=storage, resort_interval=4,
                            graph_chunk=0, tiled_sensing=tiled, f64_positions=True) as sim:
            sim.step(11)
            got.append((sim.snapshot()))
    assert got[0] == got[1]
