"""By-row convolution with a row's offsets shared by the waves of a workgroup (csrc/rows_split.hip): every way through
its kernels at the sizes where it can go wrong -- a workgroup's last rows, tiles that straddle lines of the grid (a
window in two places), windows that find no room, rows shorter than their 64-byte steps, columns that end inside a
block -- against the sum over the book's own table in float64 (int8: exactly)."""
import ctypes as C

import numpy as np
import pytest
import torch

from sphconv_amd import _lib as L
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.rulebook import RuleBook, _Buffers

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}
# Rounding of the result (half an ulp: 2^-24, 2^-11, 2^-8) and of fp32 sums of at most 27 * 128 products in any order
# (each partial sum off by 2^-24 of a magnitude that the products' absolute sum bounds).
EPS = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def _scene(shape, keep, seed):
    """Occupied cells of a batch of one, compressed: (z_idx, z_ptr)."""
    g = np.random.default_rng(seed)
    occ = g.random(shape) < keep
    z = np.nonzero(occ)[2].astype(np.int32)
    ptr = np.cumsum(occ.sum(2).reshape(-1)).astype(np.int32).reshape(1, shape[0], shape[1])
    return torch.tensor(z, device=DEV), torch.tensor(ptr, device=DEV)


def _book(shape, keep, kernel, stride, seed):
    z_idx, z_ptr = _scene(shape, keep, seed)
    if stride == (1, 1, 1):
        book = RuleBook.build_subm(z_idx, z_ptr, 1, list(shape), list(kernel), lazy=True)
        oz_idx, oz_ptr = z_idx, z_ptr
    else:
        out = [(s + 2 * (k // 2) - k) // t + 1 for s, k, t in zip(shape, kernel, stride)]
        book = RuleBook.build(z_idx, z_ptr, 1, list(shape), out, list(kernel), list(stride), [k // 2 for k in kernel], lazy=True)
        oz_idx, oz_ptr = book.oz_idx, book.oz_ptr
    buf = _Buffers(oz_idx.numel(), book.kv, z_idx.device, True, False)
    L.check(L.lib().sph_rules_build(z_idx.data_ptr(), z_ptr.data_ptr(), z_idx.numel(), oz_idx.data_ptr(), oz_ptr.data_ptr(),
                                    oz_idx.numel(), C.byref(book.geom()), 0, C.byref(buf.struct()), None,
                                    torch.cuda.current_stream().cuda_stream))
    return z_idx.numel(), oz_idx.numel(), book.kv, buf


def _check(rows_in, rows, kv, buf, dt, ic, oc, seed, epilogue):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[dt]
    if dt == "i8":
        feat = torch.randint(-9, 10, (rows_in, ic), generator=g, device=DEV).to(dtype)
        weight = torch.randint(-9, 10, (kv, ic, oc), generator=g, device=DEV).to(dtype)
    else:
        feat = torch.randn((rows_in, ic), generator=g, device=DEV).to(dtype)
        weight = (torch.randn((kv, ic, oc), generator=g, device=DEV) * (2.0 / (kv * ic)) ** 0.5).to(dtype)
    scale = (0.5 + torch.rand(oc, generator=g, device=DEV)) * (2.0 ** -5 if dt == "i8" else 1.0)
    shift = torch.randn(oc, generator=g, device=DEV)
    if not epilogue and dt != "i8":
        scale = shift = None
    epi = L.Epilogue(L.ptr(scale), L.ptr(None if dt == "i8" else shift), int(epilogue))
    out = torch.full((rows, oc), 77, device=DEV).to(dtype)
    packed = ext._packed_weight(weight, False)
    L.check(L.lib().sph_conv_apply(L.dtype_code(dtype), feat.data_ptr(), rows_in, ic, packed.data_ptr(), oc, C.byref(buf.struct()),
                                   C.byref(epi), out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    table = buf.tile_nbr.permute(0, 2, 1).reshape(-1, kv)[:rows].long()            # [rows, KV]
    wide = torch.cat([feat.double(), torch.zeros((1, ic), device=DEV, dtype=torch.float64)])
    table = torch.where(table < 0, torch.full_like(table, rows_in), table)
    want = torch.zeros((rows, oc), device=DEV, dtype=torch.float64)
    mag = torch.zeros_like(want)
    for k in range(kv):
        x, w = wide[table[:, k]], weight[k].double()
        want += x @ w
        mag += x.abs() @ w.abs()
    if dt == "i8":
        v = torch.round(want.float() * scale).clamp(-128, 127)
        assert torch.equal(out.float(), v)
        return
    if epilogue:
        want, mag = (want * scale.double() + shift.double()).clamp(min=0), mag * scale.double() + shift.double().abs()
    n = kv * ic + 16
    bound = EPS[dt] * want.abs() + n ** 0.5 * 4 * 2.0 ** -24 * mag + (2.0 ** -24 if dt == "f16" else 1e-30)
    assert bool(((out.double() - want).abs() <= bound).all())


def _check_bad_rows(rows_in, rows, kv, buf, dt, ic, oc):
    table = buf.tile_nbr.permute(0, 2, 1).reshape(-1, kv)[:rows].long()
    dtype = DTYPES[dt]
    feat = torch.randn((rows_in, ic), device=DEV).to(dtype)
    bad = torch.arange(0, rows_in, 997, device=DEV)
    feat[bad] = float("nan")
    feat[bad[::2]] = float("inf")
    weight = torch.randn((kv, ic, oc), device=DEV).to(dtype)
    out = torch.empty((rows, oc), device=DEV, dtype=dtype)
    epi = L.Epilogue(None, None, 0)
    L.check(L.lib().sph_conv_apply(L.dtype_code(dtype), feat.data_ptr(), rows_in, ic, ext._packed_weight(weight, False).data_ptr(), oc,
                                   C.byref(buf.struct()), C.byref(epi), out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    is_bad = torch.zeros(rows_in + 1, dtype=torch.bool, device=DEV)
    is_bad[bad] = True
    hit = is_bad[torch.where(table < 0, torch.full_like(table, rows_in), table)].any(1)
    assert not bool(torch.isfinite(out)[hit].any()) and bool(torch.isfinite(out)[~hit].all()) and bool(hit.any()) and not bool(hit.all())


# grids by the tiles they come to: (grid, share of the bins, kernel, stride)
GRIDS = {
    "9 tiles": ((4, 40, 16), 0.45, (3, 3, 3), (1, 1, 1)),
    "40 tiles": ((8, 100, 16), 0.4, (3, 3, 3), (1, 1, 1)),
    "100 tiles": ((8, 200, 16), 0.5, (3, 3, 3), (1, 1, 1)),
    "short lines": ((400, 6, 8), 0.7, (3, 3, 3), (1, 1, 1)),            # a tile's rows lie on several lines
    "300 tiles": ((12, 400, 16), 0.5, (3, 3, 3), (1, 1, 1)),
    "1100 tiles": ((16, 1101, 16), 0.5, (3, 3, 3), (1, 1, 1)),
    "deep": ((3, 19, 333), 0.97, (3, 3, 3), (1, 1, 1)),                 # columns longer than a tile: windows of 600 rows
    "some windows": ((8, 100, 128), 0.6, (3, 3, 3), (1, 1, 1)),         # one or two of a tile's three find room
    "deep, 600 tiles": ((8, 70, 333), 0.45, (3, 3, 3), (1, 1, 1)),
    "strided, 1.6 to a row": ((24, 1801, 16), 0.2, (3, 3, 3), (2, 2, 2)),
    "strided, 3 to a row": ((24, 700, 16), 0.45, (3, 3, 3), (2, 2, 2)),
    "strided, 7 to a row": ((33, 601, 15), 0.9, (3, 3, 3), (2, 2, 2)),
    "45 offsets": ((8, 200, 16), 0.4, (5, 3, 3), (1, 1, 1)),
    "9 offsets": ((8, 200, 16), 0.5, (3, 3, 1), (1, 1, 1)),
    "8 offsets": ((4, 31, 16), 0.5, (2, 2, 2), (1, 1, 1)),
}
LAYERS = [("f16", 64, 64), ("bf16", 48, 40), ("f16", 32, 64), ("bf16", 24, 32), ("f16", 16, 16), ("f16", 64, 128), ("f32", 32, 32),
          ("f32", 16, 64), ("f32", 32, 64), ("f32", 4, 24), ("i8", 64, 64), ("i8", 128, 32), ("i8", 16, 48)]


@pytest.mark.parametrize("grid", list(GRIDS))
def test_against_the_table_in_float64(grid):
    rows_in, rows, kv, buf = _book(*GRIDS[grid], seed=len(grid))
    assert rows % 128 != 0 or grid == "deep"
    for i, (dt, ic, oc) in enumerate(LAYERS):
        _check(rows_in, rows, kv, buf, dt, ic, oc, 10 * i + len(grid), epilogue=i % 2 == 0)


@pytest.mark.parametrize("dt,ic,oc", [("f16", 64, 64), ("f16", 32, 32), ("f32", 32, 64), ("i8", 64, 64)])
def test_rows_in_two_places(dt, ic, oc):
    """Books whose tiles gather from the two ends of the feature array: a window in two pieces, and (from three places) none."""
    rows_in, rows, kv, buf = _book((12, 400, 16), 0.5, (3, 3, 3), (1, 1, 1), seed=3)
    table = buf.tile_nbr.clone()
    far = 3 * rows_in
    for places in (2, 3):
        g = torch.Generator(device=DEV).manual_seed(places)
        at = torch.randint(0, places, table.shape, generator=g, device=DEV, dtype=torch.int32)
        buf.tile_nbr.copy_(torch.where(table >= 0, table + at * far, table))
        _check(rows_in + far * (places - 1), rows, kv, buf, dt, ic, oc, places, epilogue=True)


@pytest.mark.parametrize("phases", [(0,), (1,), (2,), (0, 2), (1, 2)])
def test_phases_without_a_window(phases):
    """Some of a kernel's three phases gather rows too far apart for a window, the others do not."""
    rows_in, rows, kv, buf = _book((12, 400, 16), 0.5, (3, 3, 3), (1, 1, 1), seed=3)
    table = buf.tile_nbr.clone()
    g = torch.Generator(device=DEV).manual_seed(9)
    at = torch.randint(0, 3, table.shape, generator=g, device=DEV, dtype=torch.int32)
    for p in range(3):
        if p not in phases:
            at.view(-1, kv, L.TILE_ROWS)[:, 9 * p:9 * p + 9] = 0
    buf.tile_nbr.copy_(torch.where(table >= 0, table + at * 3 * rows_in, table))
    for n, (dt, ic, oc) in enumerate([("f16", 64, 64), ("f32", 32, 64), ("bf16", 24, 64), ("i8", 64, 32)]):
        _check(7 * rows_in, rows, kv, buf, dt, ic, oc, n, epilogue=n % 2 == 0)


def test_rows_that_are_not_numbers():
    """A row of infinities or NaN reaches the outputs that gather it and no other."""
    rows_in, rows, kv, buf = _book((12, 400, 16), 0.5, (3, 3, 3), (1, 1, 1), seed=5)
    table = buf.tile_nbr.permute(0, 2, 1).reshape(-1, kv)[:rows].long()
    for dt, ic, oc in (("f16", 64, 64), ("f32", 16, 32), ("bf16", 24, 64)):
        dtype = DTYPES[dt]
        feat = torch.randn((rows_in, ic), device=DEV).to(dtype)
        bad = torch.arange(0, rows_in, 997, device=DEV)
        feat[bad] = float("nan")
        weight = torch.randn((kv, ic, oc), device=DEV).to(dtype)
        out = torch.empty((rows, oc), device=DEV, dtype=dtype)
        epi = L.Epilogue(None, None, 0)
        L.check(L.lib().sph_conv_apply(L.dtype_code(dtype), feat.data_ptr(), rows_in, ic, ext._packed_weight(weight, False).data_ptr(), oc,
                                       C.byref(buf.struct()), C.byref(epi), out.data_ptr(), torch.cuda.current_stream().cuda_stream))
        is_bad = torch.zeros(rows_in + 1, dtype=torch.bool, device=DEV)
        is_bad[bad] = True
        hit = is_bad[torch.where(table < 0, torch.full_like(table, rows_in), table)].any(1)
        assert bool(torch.isnan(out).all(1)[hit].all()) and not bool(torch.isnan(out)[~hit].any())
