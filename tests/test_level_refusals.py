"""Arguments of a level in one launch that are refused on the host, before any
device call (the CPU alone)."""
import ctypes

import pytest


def test_upper_flow_beyond_32_bit_offsets_is_refused():
    from flowfilter import _native as N
    from flowfilter import errors
    from flowfilter.autograd import _Level
    a = _Level(*[k * 4096 for k in range(1, 8)])  # image .. ymap, never read
    a.flow_out, a.bright_out, a.dflow_out = (k * 4096 for k in range(11, 14))
    for hu, wu in ((20000, 20000), (1, 2 ** 28), (2 ** 16, 2 ** 16), (2 ** 14, 2 ** 14)):
        with pytest.raises(errors.InvalidArgument, match="upper"):
            N.call("ff_ad_level_forward", ctypes.byref(a), 1, 1, 1, 8, 8, hu, wu, ctypes.c_float(1), 1,
                   ctypes.c_float(1), ctypes.c_float(1), None)
