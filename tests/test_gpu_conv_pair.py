"""fp32 layers of 64 channels two tiles at a time (csrc/conv.hip, conv_wave_pair_kernel): merged last groups, tiles too full to merge,
an odd number of tiles, rows and columns that end inside a step, empty tiles -- against the sum over the book's pairs in float64."""
import pytest
import torch
from test_gpu_wgrad import _scene

from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GRIDS = {  # (grid, batch, share of the bins, kernel, stride)
    "subm": ((64, 512, 32), 2, 0.07, (3, 3, 3), (1, 1, 1)),
    "sparse": ((200, 1000, 40), 1, 0.009, (3, 3, 3), (1, 1, 1)),
    "dense": ((16, 301, 16), 1, 0.9, (3, 3, 3), (1, 1, 1)),
    "odd tiles": ((16, 1024, 9), 1, 0.4450, (3, 3, 3), (1, 1, 1)),
    "strided": ((64, 512, 64), 1, 0.02, (3, 3, 3), (2, 2, 2)),
    "18 offsets": ((64, 512, 32), 2, 0.07, (2, 3, 3), (1, 1, 1)),
    "45 offsets": ((64, 512, 32), 2, 0.07, (5, 3, 3), (1, 1, 1)),
    "empty pairs of tiles": ((64, 128, 32), 1, 0.5, (3, 3, 3), (4, 1, 1)),   # transposed: every fourth plane reaches no output
}


@pytest.mark.parametrize("grid", list(GRIDS))
def test_against_the_pairs_in_float64(grid):
    shape, batch, keep, kernel, stride = GRIDS[grid]
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
    if empty:
        rows_in, rows = rows, rows_in
        ngrp = buf.tile_ngrp[:buf.ntiles // 2 * 2].view(-1, 2)
        assert bool((ngrp.sum(1) == 0).any()) and bool((ngrp.sum(1) > 0).any())
    assert buf.ntiles > 512 and rows_in <= rows
    if grid == "odd tiles":
        assert buf.ntiles % 2
    koff, cap = buf.tile_koff.long() & 0xffff, buf.cap
    gather, owner = (x.view(-1, cap * 16).long() for x in (buf.grp_gather, buf.grp_owner))
    at = torch.arange(cap, device=DEV)
    pairs = []
    for k in range(kv):
        mine = ((at >= koff[:, k, None]) & (at < koff[:, k + 1, None])).repeat_interleave(16, 1)
        pairs.append((gather[mine], owner[mine]))
    for n, (ic, oc, epilogue) in enumerate([(64, 64, False), (52, 60, True), (64, 36, True), (36, 64, False)]):
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
