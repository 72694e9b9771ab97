"""Render into narrow textures, whose rows share a wave, at the widths where a row takes
another number of lanes, and into one so tall that a workgroup draws several rounds for
the launch's sake; scale 1 and others, in every format: the oracle's bytes."""
import numpy as np
import pytest

from parity_util import assert_bitwise, display_point, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("w,h,textures", [
    (1, 700, [(1, 700), (1, 1048577), (2, 1400), (1, 3)]),
    (4, 333, [(4, 333), (5, 333), (3, 250), (8, 666), (9, 5000)]),
    (17, 2000, [(16, 2000), (17, 2000), (33, 4000), (8, 941), (32, 3000)]),
    (64, 300, [(64, 300), (65, 300), (63, 290), (128, 600), (129, 600), (7, 9)]),
    (260, 40, [(260, 40), (128, 128), (127, 20), (256, 40), (257, 41)]),
])
def test_narrow_textures(slm, orc, storage, w, h, textures):
    lut = np.random.default_rng(w).integers(0, 256, 768, dtype=np.uint8).tobytes()
    s = preset(slm, "Default")
    with slm.Simulation(w, h, 600, seed=3, params=s, storage=storage) as sim:
        sim.step(5)
        t = sim.read_trail()
        for tw, th in textures:
            print(f"[render narrow] {w}x{h} {storage} -> {tw}x{th}", flush=True)
            assert_bitwise(sim.render(lut, tw, th), orc.render(t, lut, tw, th),
                           f"{w}x{h} -> {tw}x{th}")
        a = sim.read_agents()
        shown = display_point(orc, a, t, s, storage)
        tw, th = textures[1]
        assert_bitwise(sim.step_render(1, lut, tw, th), orc.render(shown, lut, tw, th), "display")


def test_more_rows_than_a_launch_holds_groups(slm, orc):
    """4 rows to a round: 65535 groups of 4 rounds end at row 1048560."""
    w, h = 130, 1048577
    lut = bytes(range(256)) * 3
    with slm.Simulation(w, h, 100000, seed=3, params=preset(slm, "Default")) as sim:
        sim.step(2)
        t = sim.read_trail()
        print(f"[render narrow] {w}x{h}", flush=True)
        assert np.array_equal(sim.render(lut, w, h), orc.render(t, lut, w, h))
