"""The by-row convolution that gathers from an LDS window (csrc/conv.hip, conv_rows_win_kernel), on tables made by hand: phases of
nine offsets without a pair, with pairs in one wave's rows only, with windows of the most rows that fit and of one row more."""
import pytest
import torch

import gpu_helpers as G
from sphconv_amd import rulebook
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu


def _table(nt, kv, rows, gen):
    row = torch.arange(nt * 128, device="cuda").view(nt, 1, 128)
    rand = lambda lo, hi: torch.randint(lo, hi, (nt, kv, 128), generator=gen, device="cuda")
    nbr = (row + rand(-40, 41)).clamp(0, rows - 1)
    nbr[rand(0, 2) == 0] = -1
    kind = torch.arange(nt, device="cuda") % 8
    nbr[kind == 1] = -1
    nbr[kind == 2, :, :64] = -1
    nbr[kind == 3, :9] = -1
    nbr[kind == 4, 9:] = -1
    nbr[kind == 5] = rand(0, rows)[kind == 5]                    # far apart
    for tile in (kind >= 6).nonzero()[:, 0].tolist()[:40]:       # 254 to 257 rows
        base = min(tile * 128, rows - 300)
        nbr[tile] = -1
        nbr[tile, :, 5] = base
        nbr[tile, :, 77] = base + 252 + tile % 5
        nbr[tile, 1::2, 100:] = base + 3
    last = nt * 128 - rows
    if last:
        nbr[nt - 1, :, 128 - last:] = -1
    nbr[0, :, ::3] = -1                                          # lanes without a pair at the array's start
    return nbr.int()


@pytest.mark.parametrize("kernel", [[3, 3, 3], [3, 3, 1], [2, 2, 3], [1, 1, 2]])
@pytest.mark.parametrize("ic,oc,dtype", [(32, 32, torch.float16), (32, 64, torch.bfloat16), (24, 40, torch.float16), (8, 16, torch.float16),
                                         (16, 16, torch.bfloat16), (16, 64, torch.float32), (64, 64, torch.int8), (32, 16, torch.int8)])
def test_window(monkeypatch, kernel, ic, oc, dtype):
    _check(monkeypatch, kernel, ic, oc, dtype, 1030)


@pytest.mark.parametrize("kernel,ic,oc,dtype,tiles", [
    ([3, 3, 3], 32, 32, torch.float16, 1537), ([3, 3, 1], 24, 24, torch.bfloat16, 2048), ([3, 3, 3], 32, 32, torch.int8, 1600),
    ([2, 2, 3], 16, 32, torch.float32, 1700), ([3, 3, 3], 8, 24, torch.float32, 3585), ([3, 3, 2], 32, 24, torch.float16, 2049),
    ([3, 3, 3], 32, 64, torch.float16, 257), ([3, 3, 3], 64, 48, torch.int8, 256), ([3, 3, 1], 16, 64, torch.bfloat16, 769),
    ([3, 3, 1], 32, 64, torch.float16, 1024), ([3, 3, 2], 32, 48, torch.bfloat16, 300), ([3, 3, 5], 16, 64, torch.float32, 1281),
    ([3, 3, 3], 16, 64, torch.bfloat16, 1921), ([3, 3, 3], 16, 48, torch.float32, 1280), ([2, 2, 2], 32, 64, torch.float16, 1300)])
def test_either_side_of_the_lines(monkeypatch, kernel, ic, oc, dtype, tiles):
    """One wave per tile and two, 64 columns with the window and without, at the sizes where one takes over from the other."""
    _check(monkeypatch, kernel, ic, oc, dtype, tiles)


def _check(monkeypatch, kernel, ic, oc, dtype, tiles):
    monkeypatch.setattr(rulebook, "BY_ROW_MIN_PAIRS", 0.0)
    gen = torch.Generator(device="cuda").manual_seed(ic + oc)
    rows = (tiles - 1) * 128 + 57
    z_ptr = torch.arange(1, rows + 1, device="cuda").int().view(1, 1, rows)
    book = RuleBook.build_subm(torch.zeros(rows, dtype=torch.int32, device="cuda"), z_ptr, 1, [1, rows, 1], kernel,
                               padding=[k // 2 for k in kernel])
    buf = book.fwd
    assert buf.tile_nbr is not None and buf.ntiles == tiles
    buf.tile_nbr.copy_(_table(buf.ntiles, buf.kv, rows, gen))
    nbr = buf.tile_nbr.permute(0, 2, 1).reshape(-1, buf.kv)[:rows].long()
    if dtype == torch.int8:
        feat = torch.randint(-128, 128, (rows, ic), generator=gen, device="cuda", dtype=torch.int8)
        w = torch.randint(-128, 128, (buf.kv, ic, oc), generator=gen, device="cuda", dtype=torch.int8)
    else:
        feat = torch.randn((rows, ic), generator=gen, device="cuda").to(dtype)
        w = (torch.randn((buf.kv, ic, oc), generator=gen, device="cuda") / (ic * buf.kv) ** 0.5).to(dtype)
    want = torch.zeros((rows, oc), dtype=torch.float64, device="cuda")
    for k in range(buf.kv):
        has = (nbr[:, k] >= 0)[:, None]
        want += torch.where(has, feat[nbr[:, k].clamp(min=0)].double(), 0.0) @ w[k].double()
    if dtype == torch.int8:
        scale = torch.full((oc,), 2.0 ** -10, device="cuda")
        got = ext.rule_conv_int8(feat, w, scale, book, None, rows)
        assert torch.equal(got, (want * 2.0 ** -10).round().clamp(-128, 127).to(torch.int8))
        return
    got = ext.rule_conv(feat, w, book, None, rows).double()
    # one rounding to the type, and sums of up to 27 * 32 products of unit variance together in fp32
    tol = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}[dtype]
    assert ((got - want).abs() <= tol * want.abs() + 2e-5).all()
