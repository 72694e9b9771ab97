"""The agent pass's short sin/cos form on every float of the range that turns reach."""
import numpy as np


def bits(x):
    return int(np.float32(x).view(np.uint32))


def test_small_form_on_every_float_of_a_turn(orc):
    assert orc.lib().orc_trig_small_mismatches(bits(1e-3), bits(7.0), 1) == 0
