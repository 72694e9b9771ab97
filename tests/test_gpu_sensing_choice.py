"""Which agent pass the library takes by itself, and that its results are the same."""
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu

# count x (width, height, agents): whole tiles with many agents sense through windows;
# small instances, slivers and few agents to a tile do not
POOLS = [
    ([(1600, 900, 1 << 21)], "f32", False, 1),
    ([(2048, 2048, 1 << 22)], "bf16", True, 1),
    ([(2048, 2048, 1 << 21)], "f32", True, 0),
    ([(1024, 1024, 1 << 20)], "f32", False, 0),
    ([(2900, 2900, 1 << 21)], "f32", False, 0),
    ([(512, 512, 1 << 18)] * 9, "f16", False, 1),
    ([(64, 64, 4096)] * 520 + [(200, 3, 50)], "f32", False, 1),
    ([(96, 96, 9216)] * 230, "f32", False, 0),
    ([(16, 16, 256)] * 8200, "f32", False, 0),
]


@pytest.mark.parametrize("dims,storage,f64,want", POOLS,
                         ids=lambda v: f"{len(v)}x{v[0][0]}x{v[0][1]}" if isinstance(v, list) else str(v))
def test_choice_by_agents_per_tile(slm, dims, storage, f64, want):
    specs = [slm.InstanceSpec(w, h, n, seed=k, params=preset(slm, "Default"))
             for k, (w, h, n) in enumerate(dims)]
    some = sorted({0, len(specs) // 2, len(specs) - 1})
    out = []
    for resort in (0, 10):
        with slm.Batch(specs, storage=storage, resort_interval=resort, graph_chunk=0,
                       f64_positions=f64) as b:
            print(f"[sensing] {len(specs)} x {dims[0]} resort={resort}", flush=True)
            assert b.sensing() == (want if resort else 0)
            b.step(3)
            assert b.sensing() == (want if resort else 0)
            out.append([(b.read_agents(k), b.read_trail(k)) for k in some])
    for k, (a0, t0), (a1, t1) in zip(some, *out):
        assert_bitwise(a1, a0, f"agents {k}")
        assert_bitwise(t1, t0, f"trail {k}")


def test_choice_follows_the_steps_that_windows_serve(slm):
    """Every second step re-sorted: the work list costs more than two steps win back."""
    with slm.Simulation(1600, 900, 1 << 21, seed=1, params=preset(slm, "Default"),
                        resort_interval=2) as sim:
        assert sim.sensing() == 0
        for interval in (5, 8):
            sim.set_tuning(resort_interval=interval)
            assert sim.sensing() == 1
        sim.set_params(preset(slm, "Snake"))  # sensors that no window covers
        assert sim.sensing() == 0


def test_replayed_chunks_lay_the_tiles_out(slm):
    """A captured chunk that re-sorts leaves a work list behind each time it runs, also
    after a snapshot was loaded; a chunk that starts between re-sorts uses it only where
    it is there."""
    kw = dict(seed=2, params=preset(slm, "Default"), resort_interval=20)
    with slm.Simulation(1600, 900, 1 << 21, graph_chunk=10, **kw) as sim, \
            slm.Simulation(1600, 900, 1 << 21, graph_chunk=0, **kw) as eager:
        start = sim.snapshot()
        sim.step(40)
        sim.load_snapshot(start)
        for steps in (10, 3):
            sim.step(steps)
            assert sim.sensing() == 1
        eager.step(13)
        middle = eager.snapshot()
        assert sim.snapshot() == middle
        sim.load_snapshot(middle)  # no list before the next re-sort, at step 20
        assert sim.sensing() == 0
        sim.step(10)  # one chunk, over the re-sort
        assert sim.sensing() == 1
        eager.step(10)
        assert sim.snapshot() == eager.snapshot()


def test_written_agents_sense_from_global_memory_until_the_next_resort(slm):
    """Agents written back stand in their first order, not in the work list's tiles."""
    kw = dict(seed=2, params=preset(slm, "Default"), resort_interval=20, graph_chunk=0)
    with slm.Simulation(1600, 900, 1 << 21, **kw) as sim:
        sim.step(3)
        a = sim.read_agents()
        assert sim.sensing() == 1
        sim.write_agents(a)
        assert sim.sensing() == 0
        sim.step(17)
        assert sim.sensing() == 1  # step 20 re-sorts
        sim.step(1)
        assert sim.sensing() == 1
    with slm.Batch([slm.InstanceSpec(512, 512, 1 << 18, seed=k, params=preset(slm, "Default"))
                    for k in range(9)], resort_interval=20, graph_chunk=0) as b:
        b.step(1)
        for k in range(5):  # windows serve the others while these are most agents
            assert b.sensing() == 1
            b.write_agents(k, b.read_agents(k))
        assert b.sensing() == 0


def test_parameters_moved_before_every_chunk(slm, orc):
    """Speeds that change how long the windows fit, set before every captured chunk of
    steps, and then left for some: the same bits as the unsorted run."""
    import dataclasses
    base = preset(slm, "Default")
    speeds = [base.agent_speed_max, 400.0, 90.0, 1500.0, 90.0, 90.0, 90.0, 5000.0, 60.0, 60.0]
    out = []
    for kw in (dict(), dict(resort_interval=12, graph_chunk=6)):
        with slm.Simulation(1600, 900, 1 << 21, seed=5, params=base, **kw) as sim:
            for k, v in enumerate(speeds):
                sim.set_params(dataclasses.replace(base, agent_speed_max=v, agent_speed_min=v / 2))
                sim.step(6 if k % 3 else 12)
            sim.step(2)
            out.append((sim.read_agents(), sim.read_trail()))
    assert_bitwise(out[1][0], out[0][0], "agents")
    assert_bitwise(out[1][1], out[0][1], "trail")


def test_parameters_are_set_without_waiting(slm):
    """slm_set_params returns while earlier steps still run, also where it changes how
    long the windows fit."""
    import dataclasses
    import time
    base = preset(slm, "Default")
    fast = dataclasses.replace(base, agent_speed_max=900.0)
    with slm.Simulation(4096, 4096, 1 << 24, seed=5, params=base, resort_interval=20,
                        graph_chunk=20) as sim:
        for s in (base, fast, base, fast):  # both captured
            sim.set_params(s)
            sim.step(80)
        sim.synchronize()
        t0 = time.perf_counter()
        sim.step(400)
        sim.set_params(base)
        returned = time.perf_counter() - t0
        sim.synchronize()
        total = time.perf_counter() - t0
    print(f"[set_params] returned after {returned * 1e3:.2f} of {total * 1e3:.2f} ms", flush=True)
    assert returned < 0.5 * total


def test_global_sensing_can_be_asked_for(slm):
    kw = dict(seed=4, params=preset(slm, "Default"), resort_interval=10)
    with slm.Simulation(1600, 900, 1 << 21, **kw) as sim, \
            slm.Simulation(1600, 900, 1 << 21, **kw) as ref:
        sim.set_tuning(tiled_sensing=4)
        assert sim.get_tuning().tiled_sensing == 4 and sim.sensing() == 0
        sim.step(13)
        assert sim.sensing() == 0
        sim.set_tuning(trail_rows=8)  # kept
        assert sim.get_tuning().tiled_sensing == 4 and sim.sensing() == 0
        sim.set_tuning(tiled_sensing=0)
        assert sim.sensing() == 0  # until a re-sort writes the list
        sim.step(7)
        assert sim.sensing() == 1
        ref.step(20)
        assert sim.snapshot() == ref.snapshot()
        chosen = sim.autotune(trial_steps=40)
        print(f"[global sensing] {chosen.as_dict()}", flush=True)
        sim.step(5)
        ref.step(5)
        assert sim.snapshot() == ref.snapshot()
