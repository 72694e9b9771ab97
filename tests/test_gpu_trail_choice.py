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


# odd row lengths around whole strips, and whole waves of them, that a launch of many
# cells takes in strips (a row must have more than 34 cells in f32, 68 in 16 bits)
ODD = {"f32": [63, 65, 129, 255, 257, 259, 261, 511, 513, 1021], "16": [127, 129, 255, 511, 513, 517, 519, 521, 1025]}


@pytest.mark.parametrize("storage", ["f32", "bf16", "bf16sr", "f16"])
@pytest.mark.parametrize("rows,streaming", [(0, 0), (4, 3), (8, 0), (16, 3), (64, 1)])
def test_small_odd_grids_in_a_large_launch(slm, orc, storage, rows, streaming):
    s = preset(slm, "Default")
    kind = "bf16" if storage == "bf16sr" else storage
    widths = ODD["f32" if storage == "f32" else "16"]
    dims = [(w, (1, 2, 3, 5, 17, 67)[k % 6]) for k, w in enumerate(widths)]
    specs = [slm.InstanceSpec(w, h, 200, seed=k, params=s) for k, (w, h) in enumerate(dims)]
    specs.append(slm.InstanceSpec(8192, 4096, 0, seed=99, params=s))  # 33 million cells
    rng = np.random.default_rng(rows * 8 + streaming)
    print(f"[trail choice] odd grids {storage} rows={rows} streaming={streaming}", flush=True)
    with slm.Batch(specs, storage=kind, stochastic_rounding=storage == "bf16sr") as b:
        b.set_tuning(trail_rows=rows, streaming=streaming)
        state = []
        for k, (w, h) in enumerate(dims):
            b.write_trail(k, rng.uniform(0, 1, (h, w)).astype(np.float32))
            state.append((b.read_agents(k), b.read_trail(k)))
        b.step(3)
        for k, ((w, h), (a, t)) in enumerate(zip(dims, state)):
            orc.step(a, t, s, 3, storage=storage)
            assert_bitwise(b.read_trail(k), t, f"trail {w}x{h}")
            assert_bitwise(b.read_agents(k), a, f"agents {w}x{h}")


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
