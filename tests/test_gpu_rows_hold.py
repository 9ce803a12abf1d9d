"""By-row convolution with the weight in LDS (csrc/rows_hold.hip): long grids, whose waves go from unit to unit and phase to phase --
windows that fit, tiles that straddle lines and columns too deep for a window (gathers from the array), kernels of one, two and
three phases, the last tile's remainder, rows of every width -- against the sum over the book's own table in float64 (int8: exactly)."""
import pytest
from test_gpu_rows_split import _book, _check, _check_bad_rows

from sphconv_amd import _lib as L

pytestmark = pytest.mark.gpu

# (grid, share of the bins, kernel, stride)
GRIDS = {
    "subm": ((32, 1600, 32), 0.41, (3, 3, 3), (1, 1, 1)),
    "short lines": ((24000, 7, 8), 0.5, (3, 3, 3), (1, 1, 1)),
    "deep": ((4, 750, 333), 0.7, (3, 3, 3), (1, 1, 1)),
    "dense": ((40, 1300, 13), 0.97, (3, 3, 3), (1, 1, 1)),
    "9 offsets": ((32, 1600, 32), 0.4, (3, 3, 1), (1, 1, 1)),
    "8 offsets": ((33, 1501, 33), 0.4, (2, 2, 2), (1, 1, 1)),
    "25 offsets": ((32, 1600, 32), 0.4, (1, 5, 5), (1, 1, 1)),
    "strided": ((33, 1301, 31), 0.45, (3, 3, 3), (2, 2, 2)),
    "strided, full": ((47, 1021, 45), 0.9, (3, 3, 3), (2, 2, 2)),
}
LAYERS = [("f16", 16, 32), ("f16", 32, 32), ("bf16", 24, 24), ("bf16", 8, 32), ("f32", 16, 20), ("f32", 4, 32), ("i8", 64, 32), ("i8", 48, 32)]


@pytest.mark.parametrize("grid", list(GRIDS))
def test_long_grids_against_the_table_in_float64(grid):
    rows_in, rows, kv, buf = _book(*GRIDS[grid], seed=len(grid))
    assert buf.ntiles > (1024 if "strided" in grid else 5000)
    buf.native.middle_run = L.plane(32, 1)   # (that columns are shallow, which rows of 64 bytes have to say)
    for n, (dt, ic, oc) in enumerate(LAYERS):
        _check(rows_in, rows, kv, buf, dt, ic, oc, n, epilogue=n % 2 == 0)


@pytest.mark.parametrize("grid", ["subm", "deep"])
def test_rows_that_are_not_numbers(grid):
    """A row of infinities or NaN reaches the outputs that gather it and no other: not the empty slots that the window's row of
    zeros stands for, and not the next unit of a wave."""
    rows_in, rows, kv, buf = _book(*GRIDS[grid], seed=len(grid))
    buf.native.middle_run = L.plane(32, 1)
    for dt, ic, oc in (("f16", 32, 32), ("bf16", 24, 24), ("f32", 16, 20)):
        _check_bad_rows(rows_in, rows, kv, buf, dt, ic, oc)
