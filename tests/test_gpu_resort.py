"""The re-sort's workgroups of 1024 slots: bit for bit the oracle's steps, with a
re-sort every step, for agent counts around whole workgroups, agents in any order
(bins that meet in a workgroup's table) and crowds in distant bins that share an
entry of it, with f32 and f64 positions; and for pools of instances so small that a
workgroup holds many."""
import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key", [0, 3])
@pytest.mark.parametrize("w,h,n,cl,crowd", [
    (64, 64, 1, 4, False), (64, 64, 1023, 2, False), (300, 200, 1024, 3, False),
    (300, 200, 1025, 4, False), (2048, 2048, 5000, 2, False), (1000, 700, 30000, 3, False),
    (2048, 2048, 3000, 3, True), (64, 48, 9000, 6, True)])
def test_resorted_steps_equal_the_oracle(slm, orc, w, h, n, cl, crowd, key):
    rng = np.random.default_rng(n)
    a = np.stack([rng.uniform(0, w, n), rng.uniform(0, h, n), rng.uniform(0, 6.28, n),
                  rng.uniform(30, 50, n)], axis=1).astype(np.float32)
    if crowd:  # bins 32 and 64 apart have the same low bits of their Morton codes
        side = 32 << cl
        at = np.array([[0, 0], [side, 0], [0, side], [2 * side, 2 * side]]) % [w, h]
        a[:, :2] = at[np.arange(n) % 4] + rng.uniform(0, 3, (n, 2))
    print(f"[resort] {w}x{h} n={n} cl={cl} key={key}", flush=True)
    with slm.Simulation(w, h, n, seed=5, params=preset(slm, "Default"), resort_interval=1,
                        sort_cell_log2=cl) as sim:
        sim.set_tuning(sort_key=key)
        sim.write_agents(a)
        oa, ot = sim.read_agents(), sim.read_trail()
        sim.step(4)
        ga, gt = sim.read_agents(), sim.read_trail()
    orc.step(oa, ot, preset(slm, "Default"), 4)
    assert_bitwise(ga, oa, "agents")
    assert_bitwise(gt, ot, "trail")


@pytest.mark.parametrize("f64", [False, True])
def test_resorted_instances_equal_the_unsorted_run(slm, f64):
    rng = np.random.default_rng(4)
    specs = [slm.InstanceSpec(int(rng.integers(8, 90)), int(rng.integers(8, 90)),
                              int(rng.integers(0, 1500)), seed=k, params=preset(slm, "Waves"))
             for k in range(24)]
    out = []
    for resort in (0, 1):
        with slm.Batch(specs, resort_interval=resort, f64_positions=f64) as b:
            b.step(6)
            out.append([(b.read_agents(k), b.read_trail(k)) for k in range(len(specs))])
    for k, ((a0, t0), (a1, t1)) in enumerate(zip(*out)):
        assert_bitwise(a1, a0, f"agents {k}")
        assert_bitwise(t1, t0, f"trail {k}")
