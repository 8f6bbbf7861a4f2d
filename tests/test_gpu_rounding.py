"""The kernels' short reciprocal, square root and quotient against the IEEE operations: every float, and 2^32 pairs for
the quotient, bit for bit."""
import ctypes as C

import pytest

from noor_amd._lib import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", [0, 1, 2, 3], ids=["reciprocal", "root", "reciprocal_root", "quotient"])
def test_short_forms_round_as_ieee(op):
    n = C.c_uint64(1)
    assert lib().noor_rounding_check(op, C.byref(n)) == 0
    assert n.value == 0


def test_comparison_counts():
    """The hardware's estimate alone is up to one ulp off."""
    n = C.c_uint64(0)
    assert lib().noor_rounding_check(4, C.byref(n)) == 0
    assert n.value > 1 << 24
    assert lib().noor_rounding_check(5, C.byref(n)) != 0
    assert lib().noor_rounding_check(0, None) != 0
