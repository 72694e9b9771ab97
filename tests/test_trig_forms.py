"""The agent pass's short sin/cos forms equal the general one bit for bit."""
import numpy as np


def bits(x):
    return int(np.float32(x).view(np.uint32))


def test_small_form_equals_the_general_one(orc):
    # every float of the turn's range, a sample of the rest, and the last ones
    # below the limit
    assert orc.lib().orc_trig_small_mismatches(bits(0.0), bits(1e-3), 9973) == 0
    assert orc.lib().orc_trig_small_mismatches(bits(1e-3), bits(7.0), 11) == 0
    assert orc.lib().orc_trig_small_mismatches(bits(7.0), bits(4096.0), 101) == 0
    assert orc.lib().orc_trig_small_mismatches(bits(4096.0) - 5000, bits(4096.0), 1) == 0


def test_middle_form_equals_the_general_one(orc):
    top = bits(4294967296.0)
    assert orc.lib().orc_trig_mid_mismatches(bits(4096.0), top, 53) == 0
    for e in range(12, 32):  # both ends of every exponent
        lo, hi = bits(2.0 ** e), bits(2.0 ** (e + 1))
        assert orc.lib().orc_trig_mid_mismatches(lo, lo + 2000, 1) == 0
        assert orc.lib().orc_trig_mid_mismatches(hi - 2000, hi, 1) == 0
