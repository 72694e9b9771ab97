"""The trail pass's column strips at every kind of row length.

A lane owns a 16-byte strip of columns; in a row that is no whole number of strips
the last one ends at the row's end and overlaps its neighbour.  Rows from one cell
(one cell per lane below a strip's width) over the edges of a strip and of a wave's
64 strips, with the shortest and with ragged tiles of rows, equal the oracle's step
bit for bit in every format, at the three forms of the diffuse mix.
"""
import dataclasses

import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu

# row lengths around V, 2V, 64V and 128V (V: 4 cells in f32, 8 in the 16-bit formats)
WIDTHS = {"f32": [1, 3, 4, 5, 7, 8, 9, 255, 256, 257, 259, 261, 513],
          "16": [1, 7, 8, 9, 15, 16, 17, 511, 512, 513, 519, 521, 1025]}


@pytest.mark.parametrize("storage", ["f32", "bf16", "bf16sr", "f16"])
@pytest.mark.parametrize("rows,streaming", [(0, 0), (4, 3), (8, 0), (16, 3), (64, 1)])
def test_strips_equal_the_oracle(slm, orc, storage, rows, streaming):
    rng = np.random.default_rng(rows * 8 + streaming)
    for k, w in enumerate(WIDTHS["f32" if storage == "f32" else "16"]):
        h = (1, 2, 3, 5, 17, 67)[k % 6]
        s = dataclasses.replace(preset(slm, "Default"),
                                pheromone_diffusion_rate=(1.0, 0.4, 0.0)[k % 3])
        print(f"[strips] {w}x{h} {storage} rows={rows} streaming={streaming}", flush=True)
        with slm.Simulation(w, h, 200, seed=k, params=s, stochastic_rounding=storage == "bf16sr",
                            storage="bf16" if storage == "bf16sr" else storage) as sim:
            sim.set_tuning(trail_rows=rows, streaming=streaming)
            sim.write_trail(rng.uniform(0, 1, (h, w)).astype(np.float32))
            a, t = sim.read_agents(), sim.read_trail()
            sim.step(3)
            ga, gt = sim.read_agents(), sim.read_trail()
        orc.step(a, t, s, 3, storage=storage)
        assert_bitwise(gt, t, f"trail {w}x{h}")
        assert_bitwise(ga, a, f"agents {w}x{h}")
