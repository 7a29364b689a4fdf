"""The exact mode's square root (v_rsq_f32 and one residual correction) against
the correctly rounded one: every float from 2^-96 to the largest, and 0.  Below
2^-96, which no segment reaches, the two part: the comparison sees it."""
import ctypes as ct

import pytest

pytestmark = pytest.mark.gpu

FIRST = (127 - 96) << 23  # bits of 2^-96
LAST = 0x7F7FFFFF         # of the largest finite float


def _differ(first, count):
    from trace_amd import _capi
    n = ct.c_int64(-1)
    _capi.check(_capi.lib().trace_debug_sqrt_mismatches(0, first, count, ct.byref(n)))
    return n.value


def test_every_float_in_its_domain(gpu):
    print("square roots from 2^-96 on", flush=True)
    assert _differ(FIRST, LAST - FIRST + 1) == 0
    assert _differ(0, 1) == 0


def test_below_its_domain(gpu):
    n = 1 << 21
    assert _differ((127 - 98) << 23, n) == n  # from 2^-98 on: 31% too small


def test_range_is_checked(gpu):
    from trace_amd import TraceInvalid
    for first, count in ((0, 0), (LAST, 2), (0x7F800000, 1), (0xFFFFFFFF, 1)):
        with pytest.raises(TraceInvalid):
            _differ(first, count)
