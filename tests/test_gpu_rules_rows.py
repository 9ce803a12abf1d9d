"""The rule kernel with a thread per stationary row (csrc/rules_rows.h), which grids of more than 512 tiles take: every pair
against a look-up in a dense grid of row numbers, and the order of the groups."""
import ctypes as C

import numpy as np
import pytest
import torch

import gpu_helpers as G
from sphconv_amd import _lib as L
from sphconv_amd import rulebook
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _by_groups(monkeypatch):
    monkeypatch.setattr(rulebook, "BY_ROW_MIN_PAIRS", float("inf"))


def _scene(shape, batch, per_column, seed, shuffle=False):
    """z_idx, z_ptr and the column of every row; 0 to S2 voxels a column, `per_column` on average."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    S0, S1, S2 = shape
    occ = torch.rand((batch * S0 * S1, S2), generator=g, device="cuda") < torch.rand((batch * S0 * S1, 1), generator=g, device="cuda") * 2 * per_column / S2
    col, z = occ.nonzero(as_tuple=True)
    if shuffle:                                        # the order inside a column is the caller's
        order = torch.argsort(col * 4096 + torch.randint(0, 4096, col.shape, generator=g, device="cuda"), stable=True)
        col, z = col[order], z[order]
    z_ptr = occ.sum(1).cumsum(0).int().view(batch, S0, S1)
    return z.int().contiguous(), z_ptr.contiguous(), col.int().contiguous()


def _expected(q, p, shape_p, kernel, stride, pad, transposed):
    """(offset, gathered row, owner row) of all pairs, by offset and owner; q, p: (z_idx, column, shape) of the two sides."""
    (qz, qc, qs), (pz, pc, ps) = q, p
    per = ps[0] * ps[1]
    n_cells = (int(pc.max()) // per + 1) * per * ps[2] if pc.numel() else 0
    cells = torch.full((max(n_cells, 1),), -1, dtype=torch.long, device="cuda")
    cells.scatter_reduce_(0, pc.long() * ps[2] + pz.long(), torch.arange(pz.numel(), device="cuda"), "amax")
    b, c0, c1, z = qc.long() // (qs[0] * qs[1]), qc.long() // qs[1] % qs[0], qc.long() % qs[1], qz.long()
    out = []
    for k in range(kernel[0] * kernel[1] * kernel[2]):
        ks = (k // (kernel[1] * kernel[2]), k // kernel[2] % kernel[1], k % kernel[2])
        at, ok = [], torch.ones_like(z, dtype=torch.bool)
        for x, kd, s, pd, n in zip((c0, c1, z), ks, stride, pad, ps):
            if transposed:
                t = x + pd - kd
                ok &= (t >= 0) & (t % s == 0)
                y = torch.div(t, s, rounding_mode="floor")
            else:
                y = x * s - pd + kd
            ok &= (y >= 0) & (y < n)
            at.append(y.clamp(0, n - 1))
        cell = ((b * ps[0] + at[0]) * ps[1] + at[1]) * ps[2] + at[2]
        ok &= cell < cells.numel()
        row = torch.where(ok, cells[cell.clamp(max=cells.numel() - 1)], -1)
        own = (row >= 0).nonzero()[:, 0]
        out.append(torch.stack([torch.full_like(own, k), row[own], own]))
    return torch.cat(out, 1)


def _check(buf, want):
    nt, cap, kv = buf.ntiles, buf.cap, buf.kv
    koff, ngrp = buf.tile_koff[:nt].int(), buf.tile_ngrp[:nt]
    group = torch.arange(cap, device=koff.device)
    k = (group[None, :, None] >= koff[:, None, 1:]).sum(2)
    used = k < kv
    assert torch.equal(used.sum(1).int(), ngrp) and (koff[:, 0] == 0).all()
    assert torch.equal(buf.grp_k.view(-1, cap)[:nt][used], k[used].int())
    gat, own = buf.grp_gather.view(-1, cap, 16)[:nt], buf.grp_owner.view(-1, cap, 16)[:nt]
    live = (own >= 0) & used[:, :, None]
    assert torch.equal(live[used], (gat >= 0)[used])
    # groups are filled from the front, and only an offset's last one is not full
    assert (live[:, :, 1:] <= live[:, :, :-1]).all()
    full = live.all(2)
    same = (k[:, 1:] == k[:, :-1]) & used[:, 1:]
    assert full[:, :-1][same].all() and live[:, :, 0][used].all()
    tile = torch.arange(nt, device=own.device)[:, None, None].expand_as(own)
    assert torch.equal(own[live] // L.TILE_ROWS, tile[live].int())
    got = torch.stack([k[:, :, None].expand_as(own)[live].long(), gat[live].long(), own[live].long()])
    # in the book: tile by tile, offsets ascending, owners ascending
    order = torch.argsort((want[2] // L.TILE_ROWS) * 64 + want[0], stable=True)
    assert torch.equal(got, want[:, order])


def _columns(z_ptr, rows):
    return torch.searchsorted(z_ptr.view(-1).long(), torch.arange(rows, device="cuda"), right=True).int()


def _build(z_idx, z_ptr, oz_idx, oz_ptr, book, transposed, cols, run=0):
    buf = rulebook._Buffers(book.in_rows if transposed else book.out_rows, book.kv, z_idx.device)
    buf.struct().middle_run = run
    L.check(L.lib().sph_rules_build(L.ptr(z_idx), L.ptr(z_ptr), book.in_rows, L.ptr(oz_idx), L.ptr(oz_ptr), book.out_rows,
                                    C.byref(book.geom()), int(transposed), C.byref(buf.struct()), L.ptr(cols), L.stream()))
    return buf


SUBM = [((3, 3, 3), 1.5), ((3, 3, 3), 3.3), ((3, 3, 1), 1.5), ((1, 3, 3), 2.0), ((3, 1, 1), 1.5), ((3, 3, 3), 0.4)]


@pytest.mark.parametrize("columns", ["given", "none", "shifted", "random", "one wrong", "outside"])
@pytest.mark.parametrize("kernel,per_column", SUBM)
def test_submanifold(kernel, per_column, columns):
    batch, shape = 3, (31, int(27000 / per_column / 31) + 9, 40)
    z_idx, z_ptr, col = _scene(shape, batch, per_column, 3, shuffle=per_column == 2.0)
    book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel))
    assert book.fwd.ntiles > 512
    cols = col.clone()
    if columns == "none":
        cols = None
    elif columns == "shifted":
        cols = cols.roll(1)
    elif columns == "random":
        cols = torch.randint_like(cols, 0, batch * shape[0] * shape[1])
    elif columns == "one wrong":
        cols[::777] += 1
    elif columns == "outside":
        cols[5::333] = -7
        cols[9::555] = 2 ** 31 - 1
    want = _expected((z_idx, col, shape), (z_idx, col, shape), shape, kernel, (1, 1, 1), [k // 2 for k in kernel], False)
    _check(_build(z_idx, z_ptr, z_idx, z_ptr, book, False, cols), want)


@pytest.mark.parametrize("kernel,stride,pad", [((3, 3, 3), (2, 2, 2), (1, 1, 1)), ((3, 3, 3), (1, 2, 2), (1, 1, 1)),
                                               ((3, 3, 3), (3, 3, 2), (0, 1, 1)), ((2, 2, 1), (2, 2, 1), (0, 0, 0)),
                                               ((3, 2, 4), (2, 1, 2), (1, 0, 1)), ((2, 3, 3), (1, 1, 3), (0, 1, 1)),
                                               ((3, 3, 1), (2, 1, 1), (1, 1, 0))])
@pytest.mark.parametrize("hint", [True, False])
def test_strided(kernel, stride, pad, hint):
    batch, shape = 2, (62, 1500, 24)
    z_idx, z_ptr, col = _scene(shape, batch, 1.2, 5)
    oshape = [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)]
    book = RuleBook.build(z_idx, z_ptr, batch, list(shape), oshape, list(kernel), list(stride), list(pad))
    ocol = _columns(book.oz_ptr, book.out_rows)
    sides = (z_idx, col, shape), (book.oz_idx, ocol, oshape)
    assert book.in_rows > 1024 * L.TILE_ROWS and book.out_rows > 512 * L.TILE_ROWS
    _check(_build(z_idx, z_ptr, book.oz_idx, book.oz_ptr, book, False, ocol if hint else None),
           _expected(sides[1], sides[0], shape, kernel, stride, pad, False))
    _check(_build(z_idx, z_ptr, book.oz_idx, book.oz_ptr, book, True, col if hint else None),
           _expected(sides[0], sides[1], oshape, kernel, stride, pad, True))


@pytest.mark.parametrize("depth,per_column", [(24, 8.0), (32, 15.0), (12, 2.5)])
@pytest.mark.parametrize("hint", [True, False])
def test_transposed_long_columns(depth, per_column, hint):
    """Four to sixteen rows a column of the gathered side."""
    batch, shape, kernel, stride, pad = 2, (62, int(2300 / per_column), depth), (3, 3, 3), (2, 2, 2), (1, 1, 1)
    z_idx, z_ptr, col = _scene(shape, batch, per_column, 6)
    oshape = [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)]
    book = RuleBook.build(z_idx, z_ptr, batch, list(shape), oshape, list(kernel), list(stride), list(pad))
    assert 4 * book.oz_ptr.numel() <= book.out_rows <= 16 * book.oz_ptr.numel() and book.in_rows > 1024 * L.TILE_ROWS
    sides = (z_idx, col, shape), (book.oz_idx, _columns(book.oz_ptr, book.out_rows), oshape)
    _check(_build(z_idx, z_ptr, book.oz_idx, book.oz_ptr, book, True, col if hint else None),
           _expected(sides[0], sides[1], oshape, kernel, stride, pad, True))


@pytest.mark.parametrize("shape", [(2 ** 23 + 300, 1, 4), (1, 2 ** 23 + 300, 4)])
@pytest.mark.parametrize("transposed", [False, True])
def test_an_axis_of_more_columns_than_24_bit_products_take(shape, transposed):
    """Columns on either side of 2 ** 23 on one axis: a coordinate with that bit set is negative to a signed 24-bit product."""
    axis, rows = shape.index(max(shape)), 150000
    g = torch.Generator(device="cuda").manual_seed(9)
    span = 90000                                       # the last columns of the axis
    occ = torch.rand((span, shape[2]), generator=g, device="cuda") < 1.8 / shape[2]
    col, z = occ.nonzero(as_tuple=True)
    assert rows < col.numel()
    col, z = (col + shape[axis] - span).int(), z.int().contiguous()
    z_ptr = torch.bincount(col.long(), minlength=shape[axis]).cumsum(0).int().view(1, *shape[:2])
    kernel, pad = (3, 3, 3), (1, 1, 1)
    book = RuleBook.build_subm(z, z_ptr, 1, list(shape), list(kernel), lazy=True)
    assert book.out_rows > 1024 * L.TILE_ROWS
    side = z, col, shape
    _check(_build(z, z_ptr, z, z_ptr, book, transposed, col), _expected(side, side, shape, kernel, (1, 1, 1), pad, transposed))


@pytest.mark.parametrize("transposed", [False, True])
def test_arrays_of_a_caller_that_lie_anywhere(transposed):
    """A book whose arrays are aligned to their elements only: the same book as with arrays of the extension's."""
    batch, shape, kernel = 3, (31, 3800, 40), (3, 3, 3)
    z_idx, z_ptr, col = _scene(shape, batch, 0.4, 3)
    book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel), lazy=True)
    buf = _build(z_idx, z_ptr, z_idx, z_ptr, book, transposed, col)
    assert buf.ntiles > 1024
    fields = ("tile_ngrp", "tile_koff", "grp_k", "grp_gather", "grp_owner")
    for shift in (1, 2, 3):
        own, st = {}, L.Book()
        for name in fields:
            own[name] = torch.full((getattr(buf, name).numel() + 8,), -7, dtype=getattr(buf, name).dtype, device="cuda")
            setattr(st, name, own[name][shift:].data_ptr())
        st.rows, st.KV = buf.rows, buf.kv
        L.check(L.lib().sph_rules_build(L.ptr(z_idx), L.ptr(z_ptr), book.in_rows, L.ptr(z_idx), L.ptr(z_ptr), book.out_rows,
                                        C.byref(book.geom()), int(transposed), C.byref(st), L.ptr(col), L.stream()))
        used = torch.arange(buf.cap, device="cuda")[None] < buf.tile_ngrp[:buf.ntiles, None]
        for name in fields:
            want, got = getattr(buf, name).view(-1), own[name][shift:shift + getattr(buf, name).numel()]
            assert (own[name][:shift] == -7).all() and (own[name][shift + want.numel():] == -7).all()
            if name.startswith("grp_"):
                want, got = (x.view(buf.ntiles, buf.cap, -1)[used] for x in (want, got))
            assert torch.equal(got, want), name


LINES = [((k0, k1, 3), t) for k0 in (1, 2, 3) for k1 in (1, 2, 3) for t in (False, True)] + \
        [((3, 3, 1), True), ((3, 3, 2), False), ((1, 1, 32), False), ((2, 1, 13), True), ((3, 3, 3), False), ((2, 3, 5), False)]


@pytest.mark.parametrize("hint", [True, False])
@pytest.mark.parametrize("kernel,transposed", LINES)
def test_lines_and_columns(kernel, transposed, hint):
    """One to three lines of one to three columns, kernels of one offset to thirty-two, columns of up to eight entries."""
    batch, shape, pad = 2, (37, 1700, 40), [k // 2 for k in kernel]
    z_idx, z_ptr, col = _scene(shape, batch, 1.3, 7)
    book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel), lazy=True)
    assert book.out_rows > 1024 * L.TILE_ROWS and int(torch.diff(z_ptr.view(-1)).max()) > 6
    side = z_idx, col, shape
    _check(_build(z_idx, z_ptr, z_idx, z_ptr, book, transposed, col if hint else None),
           _expected(side, side, shape, kernel, (1, 1, 1), pad, transposed))


@pytest.mark.parametrize("shape,per_column,share", [((64, 1500, 40), 1.6, 1.0), ((64, 1250, 64), 3.7, 0.3), ((64, 4100, 512), 1.3, 0.1),
                                                    ((64, 1300, 512), 3.9, 0.3), ((64, 600, 512), 8.0, 0.5)])
@pytest.mark.parametrize("kernel,stride,transposed", [((3, 3, 3), (1, 1, 1), False), ((3, 3, 3), (2, 2, 2), False),
                                                      ((3, 3, 3), (2, 2, 2), True), ((1, 3, 3), (1, 2, 2), True)])
def test_uneven_columns(shape, per_column, share, kernel, stride, transposed):
    """Books of either side of every line on the entries of a column, with rows in a share of the columns only."""
    g = torch.Generator(device="cuda").manual_seed(8)
    ncol, pad = shape[0] * shape[1], [k // 2 for k in kernel]
    occ = torch.rand((ncol, shape[2]), generator=g, device="cuda") < per_column / share / shape[2]
    occ &= torch.rand((ncol, 1), generator=g, device="cuda") < share
    col, z = occ.nonzero(as_tuple=True)
    z_idx, col = z.int().contiguous(), col.int().contiguous()
    z_ptr = occ.sum(1).cumsum(0).int().view(1, *shape[:2]).contiguous()
    if stride == (1, 1, 1):
        book, oshape = RuleBook.build_subm(z_idx, z_ptr, 1, list(shape), list(kernel), lazy=True), shape
    else:
        oshape = [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)]
        book = RuleBook.build(z_idx, z_ptr, 1, list(shape), oshape, list(kernel), list(stride), pad, lazy=True)
    ocol = _columns(book.oz_ptr, book.out_rows)
    ins, outs = (z_idx, col, shape), (book.oz_idx, ocol, oshape)
    q, p = (ins, outs) if transposed else (outs, ins)
    _check(_build(z_idx, z_ptr, book.oz_idx, book.oz_ptr, book, transposed, q[1]),
           _expected(q, p, p[2], kernel, stride, pad, transposed))


@pytest.mark.parametrize("cols", ["given", "none", "one wrong"])
@pytest.mark.parametrize("tiles,per_column,share", [(560, 1.2, 1.0), (1279, 0.4, 0.2), (1290, 1.4, 0.5), (1000, 1.3, 0.05)])
def test_scans_in_flight(tiles, per_column, share, cols):
    """Rounds of two entries up to 1280 tiles, of four beyond; columns of up to forty entries."""
    shape = (64, int(tiles * 128 / per_column / 64), 48)
    g = torch.Generator(device="cuda").manual_seed(9)
    ncol = shape[0] * shape[1]
    occ = torch.rand((ncol, shape[2]), generator=g, device="cuda") < per_column / share / shape[2]
    occ &= torch.rand((ncol, 1), generator=g, device="cuda") < share
    col, z = occ.nonzero(as_tuple=True)
    z_idx, col = z.int().contiguous(), col.int().contiguous()
    z_ptr = occ.sum(1).cumsum(0).int().view(1, *shape[:2]).contiguous()
    book = RuleBook.build_subm(z_idx, z_ptr, 1, list(shape), [3, 3, 3], lazy=True)
    given = col.clone()
    if cols == "one wrong":
        given[::777] += 1
    side = z_idx, col, shape
    _check(_build(z_idx, z_ptr, z_idx, z_ptr, book, False, None if cols == "none" else given, L.RUN_IN_FLIGHT),
           _expected(side, side, shape, (3, 3, 3), (1, 1, 1), [1, 1, 1], False))
