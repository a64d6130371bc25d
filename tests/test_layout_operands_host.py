"""``tace_layout_operands`` refuses tables that do not fit before any device work (CPU)."""

import ctypes

import pytest

from tace_amd import _native as N

GOOD = [1, 64, 48, 0, 2, 0, 1, 64, 4096, 20, 0, 8192, 28, 0] + [0] * 6   # three terms of [64, 48] in two segments
SIZE = 3 * 1024 * 2 * 3


@pytest.mark.parametrize("at,value,message", [
    (0, 3, "bad operand"), (0, -1, "bad operand"), (1, 0, "bad operand"), (2, -4, "bad operand"), (2, 1 << 24, "bad operand"),
    (3, 8, "bad operand"), (3, -16, "bad operand"), (4, 0, "bad operand"), (4, 5, "bad operand"), (5, 2, "bad operand"),
    (3, 16, "past out"), (8, 0, "bad segment"), (9, 0, "bad segment"), (12, 29, "operand's length"),
    (5, 1, "operand's length"), (4, 1, "operand's length")])
def test_bad_operands(at, value, message):
    row = list(GOOD)
    row[at] = value
    table = (ctypes.c_int64 * 40)(*GOOD, *row)   # behind a good one
    out = ctypes.create_string_buffer(64)
    rc = N.lib().tace_layout_operands(ctypes.addressof(table), 2, ctypes.addressof(out) // 16 * 16 + 16, SIZE, None)
    assert rc != 0 and message in N.lib().tace_last_error().decode()


def test_counts_and_pointers():
    table = (ctypes.c_int64 * 20)(*GOOD)
    call = lambda t, n, out: N.lib().tace_layout_operands(t, n, out, SIZE, None)
    assert call(None, 0, None) == 0
    for args in ((None, 1, 4096), (ctypes.addressof(table), 1, None), (ctypes.addressof(table), 1, 4104),
                 (ctypes.addressof(table), 65536, 4096), (ctypes.addressof(table), -1, 4096)):
        assert call(*args) != 0
