"""device_bytes counts the buffer that a handle keeps between copies to and from the
host, and only what is kept of it (16 MiB at most)."""
import pytest

from parity_util import preset

pytestmark = pytest.mark.gpu


def test_kept_staging_is_counted(slm):
    w, h, n = 500, 400, 3000
    lut = bytes(range(256)) * 3
    with slm.Simulation(w, h, n, seed=1, params=preset(slm, "Default"), storage="f16") as sim:
        bare = sim.info().device_bytes
        sim.read_agents()
        assert sim.info().device_bytes == bare + n * 16
        sim.read_trail()
        assert sim.info().device_bytes == bare + w * h * 4
        sim.read_agents()  # the larger one stays
        assert sim.info().device_bytes == bare + w * h * 4
        sim.render(lut, 2500, 2000)  # 20 MB: freed as the call ends
        assert sim.info().device_bytes == bare
