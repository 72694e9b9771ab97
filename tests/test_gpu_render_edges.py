"""Render at the edges of its workgroups and lanes.

A lane draws four pixels of a row (neighbours when a pixel is a cell, else 64
apart), a workgroup 256 columns by 4 rows per round.  Widths around 4, 64 and 256,
textures one pixel wide or high, offsets that begin inside a lane's pixels, and a
texture so tall that a workgroup draws several rounds for the grid's sake: each
equals the oracle byte for byte.
"""
import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("w,h,textures", [
    (1, 1, [(1, 1), (5, 1), (1, 9)]),
    (3, 5, [(3, 5), (8, 5), (3, 262150)]),
    (255, 33, [(255, 33), (258, 33), (255, 40), (510, 66)]),
    (261, 70, [(261, 70), (268, 70), (261, 77), (130, 35), (65, 300)]),
    (1028, 1030, [(1028, 1030), (1031, 1030), (1028, 1033), (193, 1031)]),
])
def test_render_edges(slm, orc, storage, w, h, textures):
    lut = np.random.default_rng(w).integers(0, 256, 768, dtype=np.uint8).tobytes()
    with slm.Simulation(w, h, 400, seed=3, params=preset(slm, "Default"), storage=storage) as sim:
        sim.step(5)
        t = sim.read_trail()
        for tw, th in textures:
            print(f"[render edges] {w}x{h} {storage} -> {tw}x{th}", flush=True)
            assert_bitwise(sim.render(lut, tw, th), orc.render(t, lut, tw, th),
                           f"{w}x{h} -> {tw}x{th}")
