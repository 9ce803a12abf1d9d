"""Weight gradient (csrc/wgrad.hip): its kernels where they can go wrong -- books of one tile and of several to a lane, chunks
left empty, shares of the centre offset that come to nothing, channels that end inside a block, several blocks, both lists'
orders, rows behind an array's end -- against the sum over the book's pairs in float64."""
import pytest
import torch

from sphconv_amd import _lib as L
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _scene(shape, batch, keep, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    occ = torch.rand((batch,) + shape, generator=g, device=DEV) < keep
    z_idx = occ.nonzero()[:, 3].int().contiguous()
    z_ptr = occ.sum(3).reshape(-1).cumsum(0).int().view(batch, shape[0], shape[1]).contiguous()
    return z_idx, z_ptr


# (grid, batch, share of the bins, kernel, stride)
GRIDS = {
    "1 tile": ((2, 9, 5), 1, 0.9, (3, 3, 3), (1, 1, 1)),
    "12 tiles": ((4, 40, 16), 1, 0.6, (3, 3, 3), (1, 1, 1)),
    "dense, 15 tiles": ((4, 117, 4), 1, 1.0, (3, 3, 3), (1, 1, 1)),
    "sparse": ((40, 300, 30), 1, 0.02, (3, 3, 3), (1, 1, 1)),
    "strided": ((33, 201, 15), 2, 0.3, (3, 3, 3), (2, 2, 2)),
    "strided, one offset": ((33, 201, 15), 1, 0.3, (1, 1, 1), (2, 2, 2)),
    "strided, 8 offsets": ((33, 201, 31), 2, 0.3, (2, 2, 2), (2, 2, 2)),
    "strided, long": ((64, 512, 64), 1, 0.1, (3, 3, 3), (2, 2, 2)),
    "8 offsets": ((4, 91, 16), 1, 0.5, (2, 2, 2), (1, 1, 1)),
    "1 offset": ((16, 301, 16), 1, 0.5, (1, 1, 1), (1, 1, 1)),
    "1100 tiles": ((16, 1101, 16), 1, 0.5, (3, 3, 3), (1, 1, 1)),
    "several tiles to a lane": ((64, 512, 20), 4, 0.5, (3, 3, 3), (1, 1, 1)),
}
LAYERS = [("f16", 64, 64), ("bf16", 24, 40), ("f16", 64, 128), ("bf16", 40, 72), ("f16", 32, 64), ("f16", 64, 16), ("bf16", 8, 48),
          ("f16", 32, 32), ("bf16", 16, 16), ("f32", 64, 64), ("f32", 4, 100), ("f32", 20, 36), ("f32", 32, 16), ("f32", 64, 12)]


@pytest.mark.parametrize("grid", list(GRIDS))
def test_against_the_pairs_in_float64(grid):
    shape, batch, keep, kernel, stride = GRIDS[grid]
    z_idx, z_ptr = _scene(shape, batch, keep, len(grid))
    if stride == (1, 1, 1) and kernel != (2, 2, 2):
        book = RuleBook.build_subm(z_idx, z_ptr, batch, list(shape), list(kernel))
        rows = z_idx.numel()
    else:
        out = [(s + 2 * (k // 2) - k) // t + 1 for s, k, t in zip(shape, kernel, stride)]
        book = RuleBook.build(z_idx, z_ptr, batch, list(shape), out, list(kernel), list(stride), [k // 2 for k in kernel])
        rows = book.oz_idx.numel()
    rows_in, kv = z_idx.numel(), book.kv
    buf = book.grouped()
    # pairs of every offset, from the groups' lists
    koff, cap = buf.tile_koff.long() & 0xffff, buf.cap
    lists = [x.view(-1, cap * 16).long() for x in (buf.grp_gather, buf.grp_owner)]
    at = torch.arange(cap, device=DEV)
    pairs = []
    for k in range(kv):
        mine = ((at >= koff[:, k, None]) & (at < koff[:, k + 1, None])).repeat_interleave(16, 1)
        i, o = lists[0][mine], lists[1][mine]
        pairs.append((i[i >= 0], o[i >= 0]))
    for dt, ic, oc in LAYERS:
        g = torch.Generator(device=DEV).manual_seed(ic + oc)
        feat = torch.randn((rows_in, ic), generator=g, device=DEV).to(DTYPES[dt])
        grad = torch.randn((rows, oc), generator=g, device=DEV).to(DTYPES[dt])
        got = [L.host().conv_wgrad(feat, grad, buf.native, False, True)]
        if rows_in and dt != "f16":
            got.append(L.host().conv_wgrad(feat, grad, book.grouped(True).native, True, True))
        x, y = feat.double(), grad.double()
        want = torch.stack([x[i].t() @ y[o] for i, o in pairs])
        mag = torch.stack([x[i].t().abs() @ y[o].abs() for i, o in pairs])
        # fp32 sums of n products in any order: each addition is off by 2^-24 of a partial sum that the products' absolute
        # sum bounds, and the errors of n of them add up as a walk (4 standard deviations)
        n = torch.tensor([i.numel() + 16 for i, _ in pairs], device=DEV, dtype=torch.float64).view(-1, 1, 1)
        for d in got:
            assert bool(((d.double() - want).abs() <= 4 * n.sqrt() * 2.0 ** -24 * mag + 1e-30).all()), (dt, ic, oc)
        again = L.host().conv_wgrad(feat, grad, buf.native, False, True)
        assert torch.equal(again, got[0]), (dt, ic, oc)
        # whether the middle offset is said to stand out decides how its groups are shared, not what comes out
        said = buf.native.middle_run
        buf.native.middle_run = 0 if said else L.RUN
        d = L.host().conv_wgrad(feat, grad, buf.native, False, True)
        buf.native.middle_run = said
        assert bool(((d.double() - want).abs() <= 4 * n.sqrt() * 2.0 ** -24 * mag + 1e-30).all()), (dt, ic, oc)


@pytest.mark.parametrize("dt,ic,oc", [("f32", 4, 4), ("f16", 24, 40)])
def test_rows_beyond_two_to_the_24(dt, ic, oc):
    """Gathered rows at the end of an array of more than 2^24 (their offsets are 32-bit products then): what the same book gives where
    they lie at the beginning, bit for bit, and not a number of the rows in front of them."""
    z_idx, z_ptr = _scene((8, 200, 16), 1, 0.5, 3)
    book = RuleBook.build_subm(z_idx, z_ptr, 1, [8, 200, 16], [3, 3, 3])
    rows, far = z_idx.numel(), 1 << 24
    g = torch.Generator(device=DEV).manual_seed(ic)
    feat = torch.randn((rows, ic), generator=g, device=DEV).to(DTYPES[dt])
    grad = torch.randn((rows, oc), generator=g, device=DEV).to(DTYPES[dt])
    for transposed in (False, True):
        buf = book.grouped(transposed)
        assert buf.ntiles > 4
        want = L.host().conv_wgrad(feat, grad, buf.native, transposed, True)
        small = grad if transposed else feat
        big = torch.full((far + rows, small.shape[1]), float("nan"), device=DEV, dtype=small.dtype)
        big[far:] = small
        kept = buf.grp_gather.clone()
        buf.grp_gather.copy_(torch.where(kept >= 0, kept + far, kept))
        got = L.host().conv_wgrad(*((feat, big) if transposed else (big, grad)), buf.native, transposed, True)
        buf.grp_gather.copy_(kept)
        assert torch.equal(got, want)
