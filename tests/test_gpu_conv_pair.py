"""fp32 layers of 64 channels two tiles at a time (csrc/conv.hip, conv_wave_pair_kernel): merged last groups, tiles too full to merge,
an odd number of tiles, rows and columns that end inside a step, empty tiles -- against the sum over the book's pairs in float64."""
import pytest
import torch
from test_gpu_wgrad import _scene

from sphconv_amd import _lib as L
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GRIDS = {  # (grid, batch, share of the bins, kernel, stride)
    "subm": ((64, 512, 32), 2, 0.07, (3, 3, 3), (1, 1, 1)),
    "sparse": ((200, 1200, 40), 1, 0.009, (3, 3, 3), (1, 1, 1)),
    "dense": ((16, 401, 16), 1, 0.9, (3, 3, 3), (1, 1, 1)),
    "odd tiles": ((16, 1323, 9), 1, 0.4450, (3, 3, 3), (1, 1, 1)),
    "strided": ((64, 512, 64), 1, 0.02, (3, 3, 3), (2, 2, 2)),
    "27 offsets, thin": ((32, 2048, 64), 1, 0.01, (3, 3, 3), (2, 1, 1)),
    "45 offsets": ((64, 512, 32), 2, 0.07, (5, 3, 3), (1, 1, 1)),
    "empty pairs of tiles": ((64, 128, 32), 1, 0.5, (3, 3, 3), (4, 1, 1)),   # transposed: every fourth plane reaches no output
}


@pytest.mark.parametrize("grid", list(GRIDS))
def test_against_the_pairs_in_float64(grid):
    shape, batch, keep, kernel, stride = GRIDS[grid]
    z_idx, z_ptr = _scene(shape, batch, keep, len(grid))
    while grid == "odd tiles" and -(-z_idx.numel() // L.TILE_ROWS) % 2 == 0:
        shape = (shape[0], shape[1] + 1, shape[2])
        z_idx, z_ptr = _scene(shape, batch, keep, len(grid))
    if stride == (1, 1, 1) and kernel[0] % 2:
        book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel))
        rows = z_idx.numel()
    else:
        out = [(s + 2 * (k // 2) - k) // t + 1 for s, k, t in zip(shape, kernel, stride)]
        book = RuleBook.build(z_idx, z_ptr, batch, list(shape), out, list(kernel), list(stride), [k // 2 for k in kernel])
        rows = book.oz_idx.numel()
    empty = grid == "empty pairs of tiles"
    rows_in, kv, buf = z_idx.numel(), book.kv, book.grouped(transposed=empty)
    buf.native.middle_run = L.THIN          # what a book has to say of itself to be taken two tiles at a time (a strided one on scattered voxels does)
    if empty:
        rows_in, rows = rows, rows_in
        ngrp = buf.tile_ngrp[:buf.ntiles // 2 * 2].view(-1, 2)
        assert bool((ngrp.sum(1) == 0).any()) and bool((ngrp.sum(1) > 0).any())
    assert buf.ntiles > 640 and kv >= 27
    if grid == "odd tiles":
        assert buf.ntiles % 2
    koff, cap = buf.tile_koff.long() & 0xffff, buf.cap
    gather, owner = (x.view(-1, cap * 16).long() for x in (buf.grp_gather, buf.grp_owner))
    at = torch.arange(cap, device=DEV)
    pairs = []
    for k in range(kv):
        mine = ((at >= koff[:, k, None]) & (at < koff[:, k + 1, None])).repeat_interleave(16, 1)
        pairs.append((gather[mine], owner[mine]))
    for n, (ic, oc, epilogue) in enumerate([(64, 64, False), (52, 60, True), (64, 36, True), (60, 64, False)]):
        g = torch.Generator(device=DEV).manual_seed(n)
        feat = torch.randn((rows_in, ic), generator=g, device=DEV)
        weight = torch.randn((kv, ic, oc), generator=g, device=DEV) * (2.0 / (4 * ic)) ** 0.5
        scale, shift = 0.5 + torch.rand(oc, generator=g, device=DEV), torch.randn(oc, generator=g, device=DEV)
        args = (scale, shift, True) if epilogue else (None, None, False)
        packed = ext._packed_weight(weight, False)
        got = ext._apply(feat, packed, ic, oc, buf, *args)
        want = torch.zeros((rows, oc), device=DEV, dtype=torch.float64)
        mag = torch.zeros_like(want)
        for k, (i, o) in enumerate(pairs):
            i, o = i[i >= 0], o[i >= 0]
            x, w = feat[i].double(), weight[k].double()
            want.index_add_(0, o, x @ w)
            mag.index_add_(0, o, x.abs() @ w.abs())
        if epilogue:
            want, mag = (want * scale.double() + shift.double()).clamp(min=0), mag * scale.double() + shift.double().abs()
        # fp32 sums of at most kv * ic products: each addition off by 2^-24 of a partial sum that the products' absolute sum
        # bounds, adding up as a walk (4 standard deviations), and the result's own rounding
        bound = 4 * (kv * ic + 16) ** 0.5 * 2.0 ** -24 * mag + 2.0 ** -24 * want.abs() + 1e-30
        assert bool(((got.double() - want).abs() <= bound).all()), (ic, oc)
        assert torch.equal(got, ext._apply(feat, packed, ic, oc, buf, *args))


def test_rows_that_are_not_numbers():
    """A row of infinities or NaN reaches the outputs that it is paired with and no other row of the merged groups."""
    shape, batch, keep, kernel, stride = GRIDS["27 offsets, thin"]
    z_idx, z_ptr = _scene(shape, batch, keep, 7)
    out = [(s + 2 * (k // 2) - k) // t + 1 for s, k, t in zip(shape, kernel, stride)]
    book = RuleBook.build(z_idx, z_ptr, batch, list(shape), out, list(kernel), list(stride), [k // 2 for k in kernel])
    buf = book.grouped()
    buf.native.middle_run = L.THIN
    assert buf.ntiles > 640
    cap = buf.cap
    used = (torch.arange(cap, device=DEV) < buf.tile_ngrp[:buf.ntiles, None]).repeat_interleave(16, 1)
    gather, owner = (x.view(-1, cap * 16).long()[:buf.ntiles][used] for x in (buf.grp_gather, buf.grp_owner))
    gather, owner = gather[owner >= 0], owner[owner >= 0]
    rows_in, rows = z_idx.numel(), book.oz_idx.numel()
    feat, weight = torch.randn((rows_in, 64), device=DEV), torch.randn((27, 64, 64), device=DEV)
    is_bad = torch.zeros(rows_in, dtype=torch.bool, device=DEV)
    is_bad[::97] = True
    feat[::97] = float("nan")
    feat[::194] = float("inf")
    got = ext._apply(feat, ext._packed_weight(weight, False), 64, 64, buf, None, None, False)
    hit = torch.zeros(rows, dtype=torch.bool, device=DEV)
    hit[owner[is_bad[gather]]] = True
    assert bool(hit.any()) and not bool(hit.all())
    assert not bool(torch.isfinite(got)[hit].any()) and bool(torch.isfinite(got)[~hit].all())


def test_which_books_are_thin():
    """Strided layers with up to 1.45 pairs to an output row say so in their forward book; denser ones, transposed books and
    submanifold ones say what they said."""
    said = {}
    for keep in (0.005, 0.5):
        z_idx, z_ptr = _scene((32, 64, 32), 1, keep, 5)
        book = RuleBook.build(z_idx, z_ptr, 1, [32, 64, 32], [16, 32, 16], [3, 3, 3], [2, 2, 2], [1, 1, 1])
        buf, back = book.grouped(), book.grouped(transposed=True)
        pairs = buf.num_pairs() / book.out_rows
        assert (pairs < 1.3) == (keep < 0.1)
        said[keep] = tuple(b.native.middle_run & L.SAID for b in (buf, back))
    assert said == {0.005: (L.THIN, 0), 0.5: (0, 0)}
    subm = RuleBook.build_subm(z_idx, z_ptr, 1, [32, 64, 32], [3, 3, 3])
    assert subm.grouped().native.middle_run & L.SAID == L.RUN
