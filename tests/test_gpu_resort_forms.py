"""Both forms of the re-sort, on either side of the agent count that parts them (3 * 2^20,
2^21 with f64 positions): agents in any order, crowds in bins that share a table entry,
and neighbouring instances whose agents wrap into each other's bins, equal the run that
is never re-sorted."""
import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f64", [(3 << 20, False), ((3 << 20) + 1, False), (1 << 21, True),
                                   ((1 << 21) + 1023, True)])
@pytest.mark.parametrize("key", [0, 3])
def test_crowds_and_strays(slm, n, f64, key):
    w, h, cl = 2048, 1536, 3
    rng = np.random.default_rng(n + key)
    a = np.stack([rng.uniform(0, w, n), rng.uniform(0, h, n), rng.uniform(0, 6.28, n),
                  rng.uniform(30, 50, n)], axis=1).astype(np.float32)
    side = 32 << cl  # bins this far apart have the same low bits
    at = np.array([[0, 0], [side, 0], [0, side], [2 * side, 2 * side], [3 * side, side]])
    crowd = n // 3
    a[:crowd, :2] = at[np.arange(crowd) % 5] + rng.uniform(0, 3, (crowd, 2))
    out = []
    for resort in (0, 1):
        print(f"[resort forms] n={n} f64={f64} key={key} resort={resort}", flush=True)
        with slm.Simulation(w, h, n, seed=5, params=preset(slm, "Default"), graph_chunk=0,
                            resort_interval=resort, sort_cell_log2=cl, f64_positions=f64) as sim:
            if resort:
                sim.set_tuning(sort_key=key)
            sim.write_agents(a)
            sim.step(3)
            out.append((sim.read_agents(), sim.read_trail()))
    assert_bitwise(out[1][0], out[0][0], "agents")
    assert_bitwise(out[1][1], out[0][1], "trail")


@pytest.mark.parametrize("count,agents,f64", [(40, 6001, False), (530, 6001, False),
                                              (360, 6001, True)])
def test_instances_of_many_bins(slm, count, agents, f64):
    specs = [slm.InstanceSpec(40, 300, agents, seed=k, params=preset(slm, "Waves"))
             for k in range(count)]
    some = (0, 1, count // 2, count - 1)
    out = []
    for resort in (0, 2):
        print(f"[resort forms] {count} instances f64={f64} resort={resort}", flush=True)
        with slm.Batch(specs, resort_interval=resort, f64_positions=f64, graph_chunk=0) as b:
            b.step(7)
            out.append([(b.read_agents(k), b.read_trail(k)) for k in some])
    for k, (a0, t0), (a1, t1) in zip(some, *out):
        assert_bitwise(a1, a0, f"agents {k}")
        assert_bitwise(t1, t0, f"trail {k}")
