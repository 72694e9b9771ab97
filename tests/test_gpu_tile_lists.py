"""The tile work list of narrow grids: the Morton square that numbers the tiles is up to
2048 times as large as the grid, and the list and the launch are sized by the grid."""
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,n,tiled,f64", [
    (131072, 64, 1 << 21, False, False),  # windows of the library's own accord
    (64, 131072, 1 << 21, False, True),
    (131072, 64, 3000, True, False),      # fewer agents than tiles
    (65537, 3, 200000, True, False),
    (100, 90, 40, True, True),
    (100, 90, 0, True, False)])
def test_narrow_grids_equal_the_unsorted_run(slm, w, h, n, tiled, f64):
    out = []
    for kw in (dict(), dict(resort_interval=3, tiled_sensing=tiled)):
        print(f"[tile lists] {w}x{h} n={n} {kw}", flush=True)
        with slm.Simulation(w, h, n, seed=7, params=preset(slm, "Default"), graph_chunk=0,
                            f64_positions=f64, **kw) as sim:
            sim.step(5)
            out.append((sim.read_agents(), sim.read_trail()))
    assert_bitwise(out[1][0], out[0][0], "agents")
    assert_bitwise(out[1][1], out[0][1], "trail")
