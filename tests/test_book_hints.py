"""What a book says of itself (``sph_book.middle_run``): the run of its middle offset, and of a book by row how many rows of
the gathered side lie between the first and the last column that a kernel's plane reaches."""
import pytest
import torch

from sphconv_amd import _lib as L
from sphconv_amd.rulebook import RuleBook, _geometry


def _book(shape, out, kernel, stride, dilation, rows, out_rows, subm):
    g = _geometry(2, shape, out, kernel, stride, [d * (k // 2) for k, d in zip(kernel, dilation)], dilation)
    z, oz = torch.zeros(rows, dtype=torch.int32), torch.zeros(out_rows, dtype=torch.int32)
    return RuleBook._of(g, z, torch.zeros(1), oz, torch.zeros(1), subm, None, None)


@pytest.mark.parametrize("kernel,dilation,plane", [([3, 3, 3], [1, 1, 1], 60), ([3, 3, 3], [1, 2, 1], 120), ([3, 5, 3], [1, 1, 1], 120),
                                                   ([3, 1, 3], [1, 1, 1], 1)])
def test_plane_of_a_submanifold_book(kernel, dilation, plane):
    book = _book([10, 20, 64], [10, 20, 64], kernel, [1, 1, 1], dilation, 12000, 12000, True)    # 30 rows to a column
    for transposed in (False, True):
        assert book._said(transposed, True) == L.RUN | L.plane(plane, 1)
        assert book._said(transposed, False) == L.RUN


def test_plane_of_a_strided_book():
    """The gathered side's columns: the inputs', two lines to a line of outputs, or the outputs' in the transposed book."""
    book = _book([10, 20, 64], [5, 10, 32], [3, 3, 3], [2, 2, 2], [1, 1, 1], 12000, 2900, False)
    assert book._said(False, True) == L.plane(60, 2)
    assert book._said(True, True) == L.plane(58, 1)
    assert book._said(False, False) == book._said(True, False) == 0


def test_plane_has_its_bits():
    assert L.plane(0, 1) == 1 << 8 | 1 << 20 and L.plane(10 ** 9, 1000) == 4095 << 8 | 127 << 20
    assert L.plane(4095, 127) & L.SAID == 0 and L.plane(4095, 127) < 2 ** 31
