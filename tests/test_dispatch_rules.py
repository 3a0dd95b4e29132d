"""The library's choice between its kernels, asked of the host code: no GPU.  Where two kernels were timed against each other,
the shapes are some of those measured, with the times that decided (us)."""

import pytest

from tilelang_amd import _lib

UINT4, MXFP4, INT4, INT2 = range(4)
SCALE, ZEROS = 3, 5


def form(operands, M, N, K, group=0, mode=0, room=1):
    return _lib.load_library().dq_kwaves_form(operands, M, N, K, group, mode, room)


@pytest.mark.parametrize("operands", [MXFP4, INT4, INT2, UINT4])
def test_a_launch_that_fills_the_chip_is_counted_as_it_runs(operands):
    """Two passes of 32 rows over 8192 weight rows, 64 each, are 256 workgroups, one per CU.  Counted as more, they came after
    one pass of 64 rows, on half of the CUs."""
    assert form(operands, 64, 8192, 8192 if operands == MXFP4 else 4096 + 128, 128, SCALE) == 2
