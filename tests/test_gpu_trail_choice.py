"""The trail pass of pools that mix rows in column strips, by the library's choice and
because they are whole strips, with rows of one cell per lane: the same bits as with
strips everywhere, and as the oracle's."""
import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu

POOLS = [
    [(1001, 701), (9, 50001), (1000, 3), (701, 703)],
    [(33, 20001), (63, 20001), (128, 64)],
    [(101, 99)] * 120 + [(3, 7), (5, 4000), (64, 64)],
]


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("dims", POOLS, ids=lambda p: f"{len(p)}x{p[0][0]}x{p[0][1]}")
def test_mixed_pools(slm, orc, storage, dims):
    s = preset(slm, "Default")
    specs = [slm.InstanceSpec(w, h, 500, seed=k, params=s) for k, (w, h) in enumerate(dims)]
    rng = np.random.default_rng(len(dims))
    t0 = [rng.uniform(0, 1, (h, w)).astype(np.float32) for w, h in dims]
    out = []
    for rows in (0, 8):
        print(f"[trail choice] {len(dims)} instances {storage} rows={rows}", flush=True)
        with slm.Batch(specs, storage=storage, graph_chunk=0) as b:
            b.set_tuning(trail_rows=rows)
            for k, t in enumerate(t0):
                b.write_trail(k, t)
            a1, t1 = b.read_agents(1), b.read_trail(1)
            b.step(3)
            out.append([b.read_trail(k) for k in range(len(dims))])
            ga = b.read_agents(1)
    for k, (x, y) in enumerate(zip(*out)):
        assert_bitwise(x, y, f"trail {k}")
    orc.step(a1, t1, s, 3, storage=storage)
    assert_bitwise(ga, a1, "agents 1")
    assert_bitwise(out[0][1], t1, "trail 1")


def test_more_rows_than_one_launch_of_short_tiles(slm):
    """2^32 cells in rows of one strip: 4-row tiles would be 2^27 waves."""
    w, h, count = 8, 1 << 23, 64
    s = preset(slm, "Default")
    specs = [slm.InstanceSpec(w, h, 200, seed=k, params=s) for k in range(count)]
    with slm.Batch(specs, storage="bf16", graph_chunk=0) as b:
        b.step(2)
        got = {k: (b.read_agents(k), b.read_trail(k)) for k in (0, count - 1)}
    for k, (a, t) in got.items():
        print(f"[trail choice] instance {k} of {count}", flush=True)
        with slm.Simulation(w, h, 200, seed=k, params=s, storage="bf16") as sim:
            sim.step(2)
            assert_bitwise(a, sim.read_agents(), f"agents {k}")
            assert np.array_equal(t, sim.read_trail())
