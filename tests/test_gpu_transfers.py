"""Copies to and from the host through the kept staging buffer: calls of rising and
falling sizes, below and above what is kept (16 MiB), return what was written; -0
cells are stored as +0 wherever they stand, and invalid entries are named by index."""
import numpy as np
import pytest

from parity_util import assert_bitwise, preset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_transfers_of_all_sizes(slm, storage):
    rng = np.random.default_rng(2)
    lut = bytes(range(256)) * 3
    with slm.Simulation(300, 257, 1 << 20, seed=1, params=preset(slm, "Default"),
                        storage=storage) as sim:
        for n in (10, 5000, (1 << 20) + 1, 3, 1 << 20, 700):
            sim.set_agent_count(n)
            a = np.stack([rng.uniform(0, 300, n), rng.uniform(0, 257, n), rng.uniform(0, 6, n),
                          rng.uniform(30, 50, n)], axis=1).astype(np.float32)
            sim.write_agents(a)
            t = rng.integers(0, 2, (257, 300)).astype(np.float32)
            signed = np.where(rng.random(t.shape) < 0.01, -0.0, 1.0).astype(np.float32) * t
            sim.write_trail(np.where(t == 0, signed, t))
            assert_bitwise(sim.read_agents(), a, f"agents {n}")
            assert_bitwise(sim.read_trail(), t, "trail")
            assert sim.render(lut, 2048, 2100).shape == (2100, 2048, 4)  # above 16 MiB
        t[256, 299] = np.nan
        with pytest.raises(slm.SlimeMoldError, match="trail cell 77099 "):
            sim.write_trail(t)
        a[699, 1] = -1.0
        with pytest.raises(slm.SlimeMoldError, match="agent 699:"):
            sim.write_agents(a)
