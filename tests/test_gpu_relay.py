"""The grouped convolution with its weight in registers (csrc/relay.hip), which large books take: against the sum over the
book's pairs in float64, on books just above the sizes it starts at, with a last tile that is not full."""
import ctypes as C

import numpy as np
import pytest
import torch

import gpu_helpers as G
from sphconv_amd import _lib as L
from sphconv_amd import rulebook
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.pipeline import ScanPipeline
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu
TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}


def _scene(rows, shape, per_column, seed):
    """z_idx, z_ptr of at least one scene's worth of `rows` voxels, `per_column` of them in an occupied column on average."""
    rng = np.random.default_rng(seed)
    S0, S1, S2 = shape
    counts = np.minimum(rng.poisson(per_column, S0 * S1), S2)
    bins = np.argsort(rng.random((S0 * S1, S2)), axis=1)
    keep = np.arange(S2)[None, :] < counts[:, None]
    cells = np.sort((np.arange(S0 * S1)[:, None] * S2 + bins)[keep])[:rows]
    assert cells.size == rows, "the grid holds %d voxels" % cells.size
    z_ptr = np.cumsum(np.bincount(cells // S2, minlength=S0 * S1)).astype(np.int32).reshape(1, S0, S1)
    return G.t((cells % S2).astype(np.int32)), G.t(z_ptr)


def _pairs(buf):
    """(offset, gathered row, owner row) of every pair of a book, on the GPU."""
    nt, cap, kv = buf.ntiles, buf.cap, buf.kv
    koff = buf.tile_koff[:nt].int()
    group = torch.arange(cap, device=koff.device)
    k = (group[None, :, None] >= koff[:, None, 1:]).sum(2)                    # offset of each group; kv behind the last
    gat, own = buf.grp_gather.view(-1, cap, L.GROUP)[:nt], buf.grp_owner.view(-1, cap, L.GROUP)[:nt]
    live = (own >= 0) & (k < kv)[:, :, None]
    return k[:, :, None].expand_as(own)[live].long(), gat[live].long(), own[live].long()


def _check(book, dtype, ic, oc, seed, hint=None, epilogue=False, inf=False):
    g = torch.Generator(device="cuda").manual_seed(seed)
    buf, n, m, kv = book.fwd, book.in_rows, book.out_rows, book.kv
    k, gat, own = _pairs(buf)
    int8 = dtype == torch.int8
    if int8:
        feat = torch.randint(-128, 128, (n, ic), generator=g, device="cuda", dtype=torch.int8)
        w = torch.randint(-128, 128, (kv, ic, oc), generator=g, device="cuda", dtype=torch.int8)
    else:
        feat = torch.randn((n, ic), generator=g, device="cuda").to(dtype)
        w = (torch.randn((kv, ic, oc), generator=g, device="cuda") / (kv * ic) ** 0.5).to(dtype)
    if inf:
        w[kv // 2, 0, 0] = float("inf")
        feat[n // 2, 0] = 0.0
    scale = torch.rand(oc, generator=g, device="cuda") + 0.5 if epilogue or int8 else None
    if int8:
        scale = scale / 3000.0
    shift = torch.randn(oc, generator=g, device="cuda") if epilogue else None
    want, size = torch.zeros((2, m, oc), device="cuda", dtype=torch.float64)
    for i in range(kv):
        at = k == i
        x, y = feat[gat[at]].double(), w[i].double()
        want.index_add_(0, own[at], x @ y)
        size.index_add_(0, own[at], x.abs() @ y.abs())
    packed = ext._packed_weight(w, False)
    st = buf.struct()
    was = st.middle_run
    if hint is not None:
        st.middle_run = hint
    epi = L.Epilogue(L.ptr(scale), L.ptr(shift), int(epilogue))
    outs = []
    for _ in range(2):
        out = torch.full((m + 1, oc), 3, device="cuda").to(dtype)          # a row behind the last that nobody may touch
        L.check(L.lib().sph_conv_apply(L.dtype_code(dtype), L.ptr(feat), n, ic, L.ptr(packed), oc, C.byref(st), C.byref(epi),
                                       L.ptr(out), L.stream()))
        outs.append(out)
    st.middle_run = was
    assert torch.equal(outs[0].view(torch.int8), outs[1].view(torch.int8)) and (outs[0][m] == 3).all()
    out = outs[0][:m]
    if int8:
        assert want.abs().max() < 2 ** 24                                  # integer sums below 2**24: exact in float32
        exact = torch.round(want.float() * scale).clamp(-128, 127)
        assert torch.equal(out.float(), exact)
        return
    if epilogue:
        want, size = torch.relu(want * scale + shift), size * scale + shift.abs()
    # fp32 sums of at most kv * ic products (of the few a row has), then one rounding to the storage type
    unit = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    bound = 1e-6 * size + unit * want.abs() + (2.0 ** -24 if dtype == torch.float16 else 0.0)
    if inf:
        fine = torch.isfinite(want)
        assert not fine.all() and torch.equal(torch.isfinite(out), fine)
        out, want, bound = out[fine], want[fine], bound[fine]
    assert ((out.double() - want).abs() <= bound).all(), float(((out.double() - want).abs() / bound).max())


@pytest.fixture(autouse=True)
def _by_groups(monkeypatch):
    monkeypatch.setattr(rulebook, "BY_ROW_MIN_PAIRS", float("inf"))


@pytest.mark.parametrize("dtype,ic,oc,tiles", [
    ("f16", 64, 64, 1025), ("bf16", 64, 64, 1032), ("f16", 32, 64, 1025), ("bf16", 24, 40, 1027), ("f16", 64, 32, 1025),
    ("bf16", 40, 24, 1025), ("f32", 16, 64, 1025), ("f32", 32, 32, 1026), ("f32", 32, 32, 1282), ("f32", 4, 16, 2049), ("f32", 4, 16, 3585), ("f16", 16, 16, 2049),
    ("f16", 16, 16, 3586),
    ("bf16", 64, 8, 2050), ("f16", 16, 32, 2049), ("i8", 64, 64, 1025), ("i8", 32, 16, 2049), ("i8", 32, 16, 3585), ("i8", 128, 48, 1025)])
@pytest.mark.parametrize("per_column", [0.9, 4.0])          # one group per offset and tile; two and more (several passes)
def test_submanifold(dtype, ic, oc, tiles, per_column):
    rows = tiles * L.TILE_ROWS - 77
    S1 = int(rows / per_column / 64 * 1.1) + 8
    z_idx, z_ptr = _scene(rows, (64, S1, 32), per_column, ic + oc)
    book = RuleBook.build_subm(z_idx, z_ptr, 1, [64, S1, 32], [3, 3, 3])
    _check(book, TYPES[dtype], ic, oc, 7, epilogue=dtype in ("bf16", "f32"))


@pytest.mark.parametrize("kernel,stride", [((3, 3, 3), (2, 2, 2)), ((2, 3, 3), (1, 2, 2)), ((5, 5, 1), (2, 2, 1)),
                                           ((2, 2, 3), (2, 1, 1)), ((5, 1, 2), (1, 1, 1))])
@pytest.mark.parametrize("dtype,ic,oc", [("f16", 32, 64), ("f32", 32, 32), ("bf16", 64, 64)])
def test_other_kernels(kernel, stride, dtype, ic, oc):
    """Kernel volumes of 10 to 27 offsets, which the gathering waves share unevenly, without the middle offset's run; and with
    a run claimed that is not there (its pairs are strewn over the tile's rows)."""
    z_idx, z_ptr = _scene(170000, (64, 1800, 32), 1.6, 11)
    book = RuleBook.build(z_idx, z_ptr, 1, [64, 1800, 32],
                          [(s + 2 * (k // 2) - k) // t + 1 for s, k, t in zip((64, 1800, 32), kernel, stride)],
                          list(kernel), list(stride), [k // 2 for k in kernel])
    assert book.fwd.ntiles > 1280
    _check(book, TYPES[dtype], ic, oc, 3)
    _check(book, TYPES[dtype], ic, oc, 3, hint=1)


@pytest.mark.parametrize("hint", [0, 1])
def test_a_weight_that_is_not_finite_reaches_its_pairs_only(hint):
    """An infinite weight at the middle offset: rows without that pair, padding slots and rows behind the last stay finite."""
    z_idx, z_ptr = _scene(140000, (64, 1600, 32), 1.6, 12)
    book = RuleBook.build(z_idx, z_ptr, 1, [64, 1600, 32], [64, 1600, 32], [3, 3, 3], [1, 1, 1], [1, 1, 1])
    _check(book, torch.float16, 32, 64, 5, hint=hint, inf=True)


@pytest.mark.parametrize("kernel,stride,pad", [((2, 3, 3), (1, 1, 1), (1, 1, 1)), ((3, 2, 3), (1, 1, 1), (1, 1, 1)),
                                               ((3, 3, 3), (1, 1, 1), (0, 0, 0)), ((3, 3, 3), (2, 2, 2), (1, 1, 1))])
@pytest.mark.parametrize("dtype,ic,oc", [("f32", 32, 32), ("f16", 64, 64), ("bf16", 16, 16), ("i8", 64, 64)])
def test_no_pair_at_the_middle_offset_of_the_first_tile(kernel, stride, pad, dtype, ic, oc):
    """A run claimed at a middle offset that pairs no row with itself (even kernels, padding other than K // 2, a stride),
    and of which the first tile holds nothing at all: its rows begin with zero, row 0 too."""
    rng = np.random.default_rng(23)
    shape, subm = (64, 4400, 32), stride == (1, 1, 1)
    occ = rng.random((64 * 4400, 32)) < 1.7 / 32
    odd = int(not subm)                                       # the middle offset's pairs lie an odd number of bins apart
    occ[:6400, 1 - odd::2] = False                            # (stride 2: at the even ones)
    col, z = np.nonzero(occ)
    z_ptr = G.t(np.cumsum(occ.sum(1)).astype(np.int32).reshape(1, 64, 4400))
    z_idx = G.t(z.astype(np.int32))
    if subm:
        book = RuleBook.build_subm(z_idx, z_ptr, 1, list(shape), list(kernel), list(pad))
    else:
        book = RuleBook.build(z_idx, z_ptr, 1, list(shape), [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)],
                              list(kernel), list(stride), list(pad))
    mid, koff = book.kv // 2, book.fwd.tile_koff[:book.fwd.ntiles].int()
    assert book.fwd.ntiles > 3584 and koff[0, mid] == koff[0, mid + 1] and (koff[:, mid] < koff[:, mid + 1]).any()
    for hint in (0, 1):
        _check(book, TYPES[dtype], ic, oc, 31, hint=hint)


@pytest.mark.parametrize("tiles", [1026, 1282])             # up to 1280 tiles scans in flight take the kernels of conv.hip
def test_scans_on_three_streams(tiles):
    """Scans in flight beside one another: each output is that of the call on its own."""
    rows = tiles * L.TILE_ROWS - 40
    S1 = int(rows / 64 / 1.5 * 1.1)
    g = torch.Generator(device="cuda").manual_seed(3)
    w = (torch.randn((27, 64, 64), generator=g, device="cuda") / 40).half()
    pipe = ScanPipeline(w, 1, [64, S1, 32], max_voxels=rows, streams=3)
    scans = []
    for seed in range(5):
        z_idx, z_ptr = _scene(rows - 900 * seed % 1300, (64, S1, 32), 1.5, seed)
        feat = torch.randn((z_idx.numel(), 64), generator=g, device="cuda").half()
        book = RuleBook.build_subm(z_idx, z_ptr, 1, [64, S1, 32], [3, 3, 3])
        scans.append((feat, z_idx, z_ptr, ext.rule_conv(feat, w, book, None, z_idx.numel())))
    torch.cuda.synchronize()
    for _ in range(3):
        held = []
        for feat, z_idx, z_ptr, want in scans:
            out, slot = pipe.submit(feat, z_idx, z_ptr)
            held.append((out, slot, want))
            if len(held) == 3:
                for out, slot, want in held:
                    pipe.wait(slot)
                    G.assert_same_conv(out, want)
                held = []
        for out, slot, want in held:
            pipe.wait(slot)
            G.assert_same_conv(out, want)


@pytest.mark.parametrize("dtype,ic,oc,tiles", [("f16", 64, 64, 1025), ("f32", 32, 32, 1281)])
def test_in_a_graph(dtype, ic, oc, tiles):
    """Captured once, replayed on new features with other work and synchronisations in between: the eager results."""
    rows = tiles * L.TILE_ROWS - 5
    S1 = int(rows / 64 / 1.5 * 1.1)
    z_idx, z_ptr = _scene(rows, (64, S1, 32), 1.5, 4)
    book = RuleBook.build_subm(z_idx, z_ptr, 1, [64, S1, 32], [3, 3, 3])
    g = torch.Generator(device="cuda").manual_seed(5)
    feat = torch.randn((rows, ic), generator=g, device="cuda").to(TYPES[dtype])
    w = (torch.randn((27, ic, oc), generator=g, device="cuda") / 40).to(TYPES[dtype])
    ext.rule_conv(feat, w, book, None, rows)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ext.rule_conv(feat, w, book, None, rows)
    for seed in range(4):
        feat.copy_(torch.randn((rows, ic), generator=g, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ext.rule_conv(feat, w, book, None, rows))
