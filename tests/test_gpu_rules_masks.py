"""The rule kernel by occupancy masks (csrc/rules_masks.h), which books kept by row only take on dense grids: every entry of the table against a look-up in a dense grid of row numbers."""
import ctypes as C

import pytest
import torch

from sphconv_amd import _lib as L
from sphconv_amd import rulebook
from sphconv_amd.rulebook import RuleBook
from test_gpu_rules_rows import _columns, _expected, _scene

pytestmark = pytest.mark.gpu


def _check(z_idx, z_ptr, col, shape, batch, kernel, stride, pad, cols="given"):
    if stride == (1, 1, 1):
        book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel), list(pad))
        ocol, oshape = col, shape
    else:
        oshape = [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)]
        book = RuleBook.build(z_idx, z_ptr, batch, list(shape), oshape, list(kernel), list(stride), list(pad))
        ocol = _columns(book.oz_ptr, book.out_rows)
    assert z_idx.numel() >= 4 * z_ptr.numel()
    buf = rulebook._Buffers(book.out_rows, book.kv, z_idx.device, True, False)
    buf.tile_nbr.fill_(-5)
    given = ocol.clone()
    if cols == "none":
        given = None
    elif cols == "one wrong":
        given[::777] += 1
    elif cols == "outside":
        given[5::333] = -7
        given[9::555] = 2 ** 31 - 1
    L.check(L.lib().sph_rules_build(L.ptr(z_idx), L.ptr(z_ptr), book.in_rows, L.ptr(book.oz_idx), L.ptr(book.oz_ptr), book.out_rows,
                                    C.byref(book.geom()), 0, C.byref(buf.struct()), L.ptr(given), L.stream()))
    k, row, own = _expected((book.oz_idx, ocol, oshape), (z_idx, col, shape), shape, kernel, stride, pad, False)
    want = torch.full((buf.ntiles, book.kv, L.TILE_ROWS), -1, dtype=torch.int32, device="cuda")
    want[own // L.TILE_ROWS, k, own % L.TILE_ROWS] = row.int()
    assert torch.equal(buf.tile_nbr, want)


@pytest.mark.parametrize("cols", ["given", "none", "one wrong", "outside"])
@pytest.mark.parametrize("kernel,per_column,depth,shuffle", [
    ((3, 3, 3), 6.1, 40, False), ((3, 3, 3), 17.0, 63, False), ((3, 3, 1), 9.0, 64, False), ((3, 3, 3), 4.3, 32, False),
    ((1, 3, 3), 7.0, 33, True), ((3, 1, 5), 8.0, 62, False), ((3, 3, 3), 9.0, 64, False)])
def test_submanifold(kernel, per_column, depth, shuffle, cols):
    batch, shape = 2, (29, int(50000 / per_column / 29) + 9, depth)
    z_idx, z_ptr, col = _scene(shape, batch, per_column, 3, shuffle)
    _check(z_idx, z_ptr, col, shape, batch, kernel, (1, 1, 1), [k // 2 for k in kernel], cols)


@pytest.mark.parametrize("cols", ["given", "none"])
@pytest.mark.parametrize("kernel,stride,pad", [((3, 3, 3), (2, 2, 2), (1, 1, 1)), ((3, 3, 3), (2, 2, 2), (0, 1, 0)),
                                               ((3, 3, 3), (1, 2, 3), (1, 1, 0)), ((2, 2, 2), (2, 2, 2), (0, 0, 0)),
                                               ((3, 2, 4), (2, 1, 2), (1, 0, 1))])
def test_strided(kernel, stride, pad, cols):
    batch, shape = 2, (62, 520, 40)
    z_idx, z_ptr, col = _scene(shape, batch, 8.0, 5)
    _check(z_idx, z_ptr, col, shape, batch, kernel, stride, pad, cols)


@pytest.mark.parametrize("size", [(1, 1), (3, 4), (9, 14), (12, 41)])
def test_small(size):
    """One column; less than a tile; a few tiles, the last of them not full."""
    z_idx, z_ptr, col = _scene((*size, 16), 1, 16, 8)
    if z_idx.numel() < 4 * z_ptr.numel():
        z_idx = torch.arange(16, dtype=torch.int32, device="cuda").repeat(size[0] * size[1])
        z_ptr = (torch.arange(size[0] * size[1], device="cuda").int() * 16 + 16).view(1, *size)
        col = torch.arange(size[0] * size[1], device="cuda").int().repeat_interleave(16)
    for cols in ("given", "none", "outside"):
        _check(z_idx, z_ptr, col, (*size, 16), 1, (3, 3, 3), (1, 1, 1), [1, 1, 1], cols)


def test_many_columns_in_a_tile():
    """Half of the grid holds one voxel a column (128 columns a tile), the other half is full."""
    shape, g = (40, 3000, 12), torch.Generator(device="cuda").manual_seed(1)
    occ = torch.zeros((shape[0], shape[1], shape[2]), dtype=torch.bool, device="cuda")
    occ[:20] = torch.rand((20, shape[1], shape[2]), generator=g, device="cuda") < 0.9
    occ[20:].scatter_(2, torch.randint(0, shape[2], (20, shape[1], 1), generator=g, device="cuda"), True)
    c, z = occ.view(-1, shape[2]).nonzero(as_tuple=True)
    z_ptr = occ.sum(2).view(-1).cumsum(0).int().view(1, shape[0], shape[1])
    _check(z.int(), z_ptr, c.int(), shape, 1, (3, 3, 3), (1, 1, 1), [1, 1, 1])


@pytest.mark.parametrize("cols", ["given", "outside"])
@pytest.mark.parametrize("kernel", [(3, 3, 3), (2, 2, 2), (5, 3, 2), (4, 5, 1), (1, 1, 4)])
@pytest.mark.parametrize("depth,low,high,share,block", [(16, 0.06, 0.6, 0.5, 256), (32, 0.02, 0.9, 0.3, 100), (40, 0.03, 0.5, 0.4, 7)])
def test_sparse_columns_beside_full_ones(depth, low, high, share, block, kernel, cols):
    """Tiles of up to 128 columns whose rows walk their fibers, of one entry to forty."""
    shape, g = (24, 1600, depth), torch.Generator(device="cuda").manual_seed(2)
    ncol = shape[0] * shape[1]
    dense = (torch.rand(ncol // block + 1, generator=g, device="cuda") < share).repeat_interleave(block)[:ncol, None]
    occ = torch.rand((ncol, depth), generator=g, device="cuda") < torch.where(dense, high, low)
    c, z = occ.nonzero(as_tuple=True)
    z_ptr = occ.sum(1).cumsum(0).int().view(1, shape[0], shape[1])
    _check(z.int().contiguous(), z_ptr, c.int().contiguous(), shape, 1, kernel, (1, 1, 1), [k // 2 for k in kernel], cols)


@pytest.mark.parametrize("rows,depth", [(510, 4), (2000, 4), (510, 6), (510, 8)])
def test_few_rows_to_a_column_of_the_outputs(rows, depth):
    """Outputs of a shallow full grid, two to four rows a column: the general kernel's up to 512 tiles where there are fewer than four."""
    shape = (2 * 32, 2 * rows, depth)
    ncol = shape[0] * shape[1]
    z_idx = torch.arange(depth, dtype=torch.int32, device="cuda").repeat(ncol)
    z_ptr = (torch.arange(ncol, device="cuda").int() * depth + depth).view(1, *shape[:2])
    col = torch.arange(ncol, device="cuda").int().repeat_interleave(depth)
    _check(z_idx, z_ptr, col, shape, 1, (3, 3, 3), (2, 2, 2), (1, 1, 1))
