"""Which kernel takes a large system: the rule is host arithmetic on the LDS
that a workgroup needs, asked of the library itself."""
import ctypes

import pytest

from uqcreator_amd import native

LDS = 160 * 1024


def _wide_takes(S, M, Q):
    f = getattr(native.lib(), "_ZN3uqk17newton_wide_takesEiiii")  # uqk::newton_wide_takes(int, int, int, int)
    f.restype = ctypes.c_bool
    return f(S, M, Q, LDS)


@pytest.mark.parametrize("S,M,Q,takes", [
    (3, 35, 125, True), (3, 35, 190, True),     # four and two wavefronts in LDS
    (3, 35, 205, False), (3, 35, 216, False),   # one, beside two resident workgroups
    (3, 35, 245, False),                        # none
    (4, 24, 216, True), (4, 24, 230, False),
    (4, 28, 256, True), (4, 31, 216, True),     # one, beside one resident workgroup
    (4, 21, 300, True),                         # one, and more points than the workgroup kernel takes
    (3, 37, 40, True), (3, 38, 40, False), (4, 31, 40, True), (4, 32, 40, False),  # 111 and 127 duals
])
def test_wide_kernel(S, M, Q, takes):
    assert _wide_takes(S, M, Q) == takes
