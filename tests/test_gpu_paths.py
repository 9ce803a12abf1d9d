"""GPU tests of the paths that a size, a type or an alignment selects: each at the sizes where it can go wrong, against
the oracle or plain torch operations."""
import ctypes as C

import numpy as np
import pytest
import torch

import gpu_helpers as G
import helpers as H
import sphconv_amd as sphconv
from oracle import oracle as O
from sphconv_amd import _lib as L
from sphconv_amd import rulebook
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.datagen import merge_batch_torch
from sphconv_amd.rulebook import RuleBook, row_columns
from sphconv_amd.vfe import SimpleVoxel
from sphconv_amd.voxelize import points_to_voxel_v2

pytestmark = pytest.mark.gpu


def _cells(rng, n, B, shape):
    """n different cells of the grid in random order -> indices [n, 4]."""
    lin = rng.choice(B * shape[0] * shape[1] * shape[2], size=n, replace=False)
    return np.stack(np.unravel_index(lin, (B, *shape)), axis=1).astype(np.int32)


def _close(got, want, dtype):
    got = got.float().cpu().numpy()
    if dtype == torch.float32:
        np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)
    else:
        np.testing.assert_allclose(got, want, rtol=1e-2, atol=1e-3 * max(1.0, float(np.abs(want).max())))


@pytest.mark.parametrize("mirrored", [True, False])
@pytest.mark.parametrize("kv,ic,oc", [(27, 64, 64), (9, 24, 40), (1, 1, 3), (8, 128, 16), (27, 4, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_both_weight_copies_in_one_launch(dtype, kv, ic, oc, mirrored):
    """The copies for the forward pass and for dgrad, an fp32 weight rounded on the way, equal those of the rounded weight."""
    w = torch.randn((kv, ic, oc), generator=torch.Generator().manual_seed(kv * ic)).to(G.DEV)
    fwd, bwd = L.host().pack_weight_both(w, mirrored, L.dtype_code(dtype))
    assert torch.equal(fwd, ext._packed_weight(w.to(dtype), False))
    assert torch.equal(bwd, ext._packed_weight(w.to(dtype), True, mirrored))


@pytest.mark.parametrize("shape,n", [([3, 5, 64], 500), ([3, 5, 65], 500), ([8, 9, 300], 3000), ([256, 256, 130], 9000),
                                     ([257, 256, 500], 9000)])
@pytest.mark.parametrize("channels,dtype", [(1, torch.int8), (3, torch.float16), (5, torch.float32), (64, torch.float32),
                                            (68, torch.float32)])
def test_rows_moved_with_their_coordinates(shape, n, channels, dtype):
    """One word per column and several, one column and eight per thread of the scan (either side of 65 536 columns), rows
    of 1, 2, 4 and 16-byte granules moved by the placing kernel, and rows too long for it."""
    rng = np.random.default_rng(n + channels)
    idx = _cells(rng, n, 1, shape)
    feat = torch.tensor(rng.integers(-100, 100, (n, channels))).to(dtype)
    f, z_idx, z_ptr, perm, cols = ext._init_tensor(feat.to(G.DEV), G.t(idx), 1, shape)
    order = np.lexsort((idx[:, 3], idx[:, 2], idx[:, 1]))
    col = idx[:, 1].astype(np.int64) * shape[1] + idx[:, 2]
    assert torch.equal(f.cpu(), feat[torch.as_tensor(order)])
    assert np.array_equal(z_idx.cpu().numpy(), idx[order, 3]) and np.array_equal(cols.cpu().numpy(), col[order])
    assert np.array_equal(z_ptr.cpu().numpy().reshape(-1), np.cumsum(np.bincount(col, minlength=shape[0] * shape[1])))
    assert np.array_equal(perm.cpu().numpy()[order], np.arange(n))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.int8])
@pytest.mark.parametrize("B,shape,channels", [(2, [5, 6, 7], 3), (1, [4, 33, 2], 64), (3, [2, 2, 65], 17), (1, [1, 1, 1], 1)])
def test_dense_channels_first(B, shape, channels, dtype):
    rng = np.random.default_rng(channels)
    idx = _cells(rng, max(1, B * shape[0] * shape[1] * shape[2] // 5), B, shape)
    feat = torch.tensor(rng.integers(-100, 100, (idx.shape[0], channels))).to(dtype)
    x = sphconv.SparseConvTensor(feat.to(G.DEV), shape, B, indices=G.t(idx))
    want = torch.zeros((B, channels, *shape), dtype=dtype)
    i = torch.as_tensor(idx).long()
    want[i[:, 0], :, i[:, 1], i[:, 2], i[:, 3]] = feat
    got = x.dense()
    assert got.is_contiguous() and torch.equal(got.cpu(), want)


@pytest.mark.parametrize("sizes", [[1], [255, 0, 257], [7] * 64, [3] * 65])
def test_batch_coordinates_and_voxel_means(sizes):
    """One part, empty parts, as many parts as one launch takes and one more."""
    rng = np.random.default_rng(len(sizes))
    examples = [{"voxels": G.t(rng.standard_normal((m, 4)).astype(np.float32)),
                 "coordinates": G.t(rng.integers(0, 500, (m, 3)).astype(np.int32))} for m in sizes]
    got = merge_batch_torch(examples)
    want = torch.cat([torch.nn.functional.pad(e["coordinates"], (1, 0), value=b) for b, e in enumerate(examples)])
    assert torch.equal(got["coordinates"], want)
    assert torch.equal(got["voxels"], torch.cat([e["voxels"] for e in examples]))
    m = sum(sizes)
    voxels, num = torch.randn((m, 5, 6), device=G.DEV), torch.randint(1, 6, (m,), device=G.DEV, dtype=torch.int32)
    mean = SimpleVoxel(4)(voxels, num, None)
    torch.testing.assert_close(mean, voxels[:, :, :4].sum(1) / num.float()[:, None], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("n,ncells", [(511, 3), (512, 200), (513, 512), (1025, 1), (4096, 1500)])
def test_points_of_several_workgroups_meet_in_a_cell(n, ncells):
    rng = np.random.default_rng(n)
    pts = rng.normal(0, 1, (n, 4)).astype(np.float32)
    grid = [16, 16, 8]
    cells = rng.choice(rng.choice(16 * 16 * 8, size=ncells, replace=False), size=n)
    cells[rng.random(n) < 0.1] = -1
    coor = np.stack([cells // 256, cells // 16 % 16, cells % 16], 1)
    for max_points, max_voxels in ((2, 10 * n), (5, max(1, ncells // 2))):
        want = O.voxelize_cells(pts, pts, coor, cells >= 0, max_points, max_voxels, 0)
        res = points_to_voxel_v2(pts, None, [0] * 6, [6, -45, 87.5, 70.4, 45, 100], None, max_points, max_voxels,
                                 resolution_HWD=grid, coord_system="spherical", append_mode=0, cells=torch.tensor(cells))
        assert res["voxel_num"] == want["voxel_num"]
        for k in ("voxels", "coordinates", "num_points_per_voxel", "voxel_point_mask"):
            assert np.array_equal(res[k].cpu().numpy(), want[k]), k


@pytest.mark.parametrize("oc,tiles", [(64, 1), (64, 255), (64, 257), (64, 512), (64, 514), (32, 512), (32, 900), (16, 768), (16, 1100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_waves_that_share_a_tile(dtype, oc, tiles):
    """Four, two and one waves per tile, by the tiles that the chip's LDS holds: grouped kernel and one-launch kernel."""
    rng = np.random.default_rng(tiles + oc)
    n, shape, ic = tiles * L.TILE_ROWS - 5, [16, 40 * tiles, 8], 16
    case = G.build_case(_cells(rng, n, 1, shape), 1, shape, [3, 3, 3], [1, 1, 1], [1, 1, 1], True)
    book = case["book"]
    feat = torch.tensor(rng.standard_normal((n, ic)), dtype=torch.float32).to(dtype)
    w = torch.tensor(rng.standard_normal((27, ic, oc)) * 0.1, dtype=torch.float32).to(dtype)
    want = O.rule_conv(feat.float().numpy(), w.float().numpy(), case["oracle"][2], case["oracle"][3], n)
    grouped = ext.rule_conv(feat.to(G.DEV), w.to(G.DEV), book, None, n)
    _close(grouped, want, dtype)
    lazy = RuleBook.build_subm(book.z_idx, book.z_ptr, 1, shape, [3, 3, 3], row_cols=row_columns(book.z_ptr, n), lazy=True)
    lazy.keep = False
    fused = ext.rule_conv(feat.to(G.DEV), w.to(G.DEV), lazy, None, n)
    assert lazy.built == (tiles > RuleBook.FUSED_MAX_TILES)
    _close(fused, want, dtype)


@pytest.mark.parametrize("ic,oc,tiles", [(64, 64, 256), (64, 64, 257), (64, 32, 256), (64, 32, 257), (64, 16, 512), (64, 16, 513),
                                         (64, 16, 1025), (48, 32, 513)])
@pytest.mark.parametrize("subm", [True, False])
def test_long_rows_share_a_tile_or_have_helper_waves(ic, oc, tiles, subm):
    """Rows of 128 bytes: waves that share a tile up to 256 or 512 tiles, helper waves for the middle offset's run beyond,
    and sharing again where a book has no such run, the rows are shorter or the tiles so many that the helper waves do not
    pay."""
    rng = np.random.default_rng(tiles + oc)
    n, shape = tiles * L.TILE_ROWS - 5, [16, 40 * tiles, 8]
    case = G.build_case(_cells(rng, n, 1, shape), 1, shape, [3, 3, 3], [1, 1, 1], [1, 1, 1], True)
    book = case["book"]
    book.fwd.native.middle_run = int(subm)
    feat = torch.tensor(rng.standard_normal((n, ic)), dtype=torch.float32).half()
    w = torch.tensor(rng.standard_normal((27, ic, oc)) * 0.1, dtype=torch.float32).half()
    want = O.rule_conv(feat.float().numpy(), w.float().numpy(), case["oracle"][2], case["oracle"][3], n)
    _close(ext.rule_conv(feat.to(G.DEV), w.to(G.DEV), book, None, n), want, torch.float16)
    if subm:
        lazy = RuleBook.build_subm(book.z_idx, book.z_ptr, 1, shape, [3, 3, 3], row_cols=row_columns(book.z_ptr, n), lazy=True)
        lazy.keep = False
        fused = ext.rule_conv(feat.to(G.DEV), w.to(G.DEV), lazy, None, n)
        assert lazy.built == (tiles > RuleBook.FUSED_MAX_TILES)
        _close(fused, want, torch.float16)


def test_one_column_stride_too_wide_for_the_tile_kernel():
    """Output coordinates of a layer whose columns lie 64 input columns apart, 500 bins deep: the bin masks of a tile's
    input columns would not fit LDS."""
    rng = np.random.default_rng(8)
    shape, kernel, stride, padding = [3, 2000, 500], [3, 1, 3], [1, 64, 2], [1, 0, 1]
    case = G.build_case(_cells(rng, 30000, 2, shape), 2, shape, kernel, stride, padding, False)
    assert np.array_equal(case["book"].oz_idx.cpu().numpy(), case["oracle"][0])
    assert np.array_equal(case["book"].oz_ptr.cpu().numpy().ravel(), np.asarray(case["oracle"][1]).ravel())
    assert np.array_equal(G.book_triples(case["book"].fwd), G.oracle_triples(*case["oracle"][2:4]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,ic,oc", [(40, 16, 64), (3000, 24, 40), (9000, 64, 64), (9000, 128, 16), (500, 3, 5)])
def test_weight_gradient_from_the_transposed_book(dtype, n, ic, oc):
    """Both books of a strided layer hold the same pairs: the same gradient, and what backward() takes is the transposed
    one, where it has fewer rows."""
    rng = np.random.default_rng(n + ic)
    shape = [12, 60, 40]
    case = G.build_case(_cells(rng, n, 2, shape), 2, shape, [3, 3, 3], [2, 2, 2], [1, 1, 1], False)
    book = case["book"]
    f = torch.tensor(rng.standard_normal((n, ic)), dtype=torch.float32).to(dtype).to(G.DEV)
    d = torch.tensor(rng.standard_normal((book.out_rows, oc)), dtype=torch.float32).to(dtype).to(G.DEV)
    a = L.host().conv_wgrad(f, d, book.grouped(False).native, False, True)
    b = L.host().conv_wgrad(f, d, book.grouped(True).native, True, True)
    tri = torch.as_tensor(G.oracle_triples(*case["oracle"][2:4])).to(G.DEV)
    want = torch.zeros((27, ic, oc), dtype=torch.float64, device=G.DEV)
    for k in range(27):
        t = tri[tri[:, 0] == k]
        want[k] = f[t[:, 1]].double().T.contiguous() @ d[t[:, 2]].double()
    for got in (a, b):
        torch.testing.assert_close(got.double(), want, rtol=1e-5, atol=1e-5 * max(1.0, float(want.abs().max())))
    assert book.transposed_groups_built()
    assert torch.equal(ext.rule_conv_d_weight(f, d, book, None, torch.float32), b if n < book.out_rows else a)


@pytest.mark.parametrize("kernel,stride,cluster", [([3, 3, 3], [2, 2, 2], 1.0), ([2, 2, 2], [2, 2, 2], 1.0)])
def test_layers_behind_a_strided_one_count_its_clusters(monkeypatch, kernel, stride, cluster):
    """The rows that a strided layer makes of one input row lie together: the next layer's estimate of its pairs counts
    them, and whichever form the book takes the layer's result is the same."""
    rng = np.random.default_rng(1)
    shape, n = [16, 64, 32], 2000
    feat = torch.tensor(rng.standard_normal((n, 16)), dtype=torch.float32).to(G.DEV)
    idx = G.t(_cells(rng, n, 1, shape))
    down = sphconv.SparseConv3d(16, 32, kernel, stride=stride, padding=[k // 2 for k in kernel]).to(G.DEV).eval()
    conv = sphconv.SubMConv3d(32, 32, 3).to(G.DEV).eval()
    out = []
    for threshold in (rulebook.BY_ROW_MIN_PAIRS, 0.0, float("inf")):
        monkeypatch.setattr(rulebook, "BY_ROW_MIN_PAIRS", threshold)
        with torch.no_grad():
            x = down(sphconv.SparseConvTensor(feat, shape, 1, indices=idx))
            y = conv(x)
        assert conv.rule_book.cluster == x.cluster >= cluster
        g = conv.rule_book._geometry
        assert conv.rule_book._pairs_per_row(False) == pytest.approx(27 * x.feature.shape[0] / g.in_cells + x.cluster - 1)
        out.append(y.feature)
    assert x.cluster > 1.0 if kernel[0] > stride[0] else x.cluster == 1.0
    G.assert_same_conv(out[0], out[1])
    G.assert_same_conv(out[0], out[2])


def test_voxel_means_carry_tangents_and_transforms():
    """The mean of a voxel's points as one kernel stands for torch's operations: with a tangent, under vmap and with counts
    that lie on the host the result is still theirs."""
    import torch.autograd.forward_ad as fwAD
    voxels, num = torch.randn((50, 5, 6), device=G.DEV), torch.randint(1, 6, (50,), device=G.DEV, dtype=torch.int32)
    tangent, vfe = torch.randn_like(voxels), SimpleVoxel(4)
    want = lambda v: v[..., :4].sum(-2) / num.float()[:, None]
    with fwAD.dual_level():
        got = fwAD.unpack_dual(vfe(fwAD.make_dual(voxels, tangent), num, None))
    torch.testing.assert_close(got.primal, want(voxels), rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(got.tangent, want(tangent), rtol=1e-6, atol=1e-6)
    both = torch.stack([voxels, tangent])
    torch.testing.assert_close(torch.func.vmap(lambda v: vfe(v, num, None))(both), want(both), rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(vfe(voxels, num.cpu(), None), want(voxels), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("n", [30000, 400000])
def test_output_coordinates_hold_no_more_than_they_may(n):
    """Output coordinates written behind their count, into arrays of the most rows the layer can reach, and, where those
    would hold more than 16 MiB, after the wait into arrays of their size."""
    B, shape, out = 3, [64, 2048, 64], [32, 1024, 32]
    idx = _cells(np.random.default_rng(n), n, B, shape)
    order = np.lexsort(idx.T[::-1])
    idx = idx[order]
    counts = np.bincount((idx[:, 0] * shape[0] + idx[:, 1]) * shape[1] + idx[:, 2], minlength=B * shape[0] * shape[1])
    z_ptr = np.cumsum(counts).astype(np.int32).reshape(B, *shape[:2])
    book = RuleBook.build(G.t(idx[:, 3].copy()), G.t(z_ptr), B, shape, out, [3, 3, 3], [2, 2, 2], [1, 1, 1], lazy=True)
    reached = np.zeros((B, *out), dtype=bool)
    for k in np.ndindex(3, 3, 3):
        at = idx[:, 1:] + 1 - np.array(k)
        ok = (at % 2 == 0).all(1) & (at >= 0).all(1) & (at // 2 < np.array(out)).all(1)
        o = at[ok] // 2
        reached[idx[ok, 0], o[:, 0], o[:, 1], o[:, 2]] = True
    want = np.argwhere(reached)
    col = (want[:, 0] * out[0] + want[:, 1]) * out[1] + want[:, 2]
    assert np.array_equal(book.oz_idx.cpu().numpy(), want[:, 3])
    assert np.array_equal(book.out_row_cols.cpu().numpy(), col)
    assert np.array_equal(book.oz_ptr.cpu().numpy().ravel(), np.cumsum(np.bincount(col, minlength=B * out[0] * out[1])))
    for t in (book.oz_idx, book.out_row_cols):
        assert t.untyped_storage().nbytes() <= max(4 * book.out_rows + 512, 8 << 20)
    late = 8 * 8 * n > 16 << 20
    assert (book.oz_idx.untyped_storage().nbytes() <= 4 * book.out_rows + 512) == late


@pytest.mark.parametrize("plain_layer", [True, False])
@pytest.mark.parametrize("n", [3000, 150000])
def test_a_captured_layer_follows_its_weight(plain_layer, n):
    """A layer captured into a graph makes its own packed weight and affine map on each replay: it follows in-place updates,
    and what eager passes keep, use or drop in between does not matter to it (one launch per layer, and two)."""
    B, shape = 1, [32, 2048, 32]
    rng = np.random.default_rng(n)
    feat = torch.tensor(rng.standard_normal((n, 16)), dtype=torch.float32).half().to(G.DEV)
    x = sphconv.SparseConvTensor(feat, shape, B, indices=G.t(_cells(rng, n, B, shape)))
    conv = sphconv.SubMConv3d(16, 32, 3)
    net = (conv if plain_layer else sphconv.Sequential(conv, torch.nn.BatchNorm1d(32), torch.nn.ReLU())).to(G.DEV).half().eval()
    fresh = lambda: sphconv.SparseConvTensor(x.feature, shape, B, z_idx=x.z_idx, z_ptr=x.z_ptr, row_cols=x.row_cols)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad():
        with torch.cuda.stream(side):
            net(fresh())                                   # the stream now has kept copies
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = net(fresh()).feature
        for i in range(4):
            conv.weight.mul_(-1.5)                         # the kept copies are outdated
            if not plain_layer:
                net[1].running_mean.add_(0.25)
            with torch.cuda.stream(side):
                side.wait_stream(torch.cuda.default_stream())
                net(fresh())                               # ... and replaced
            want = net(fresh()).feature
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), i
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), i


@pytest.mark.parametrize("training,key", [(True, None), (False, None), (False, "k")])
@pytest.mark.parametrize("stride", [1, 2])
def test_a_layer_that_has_run_is_copied_and_saved(tmp_path, training, key, stride):
    import copy
    rng = np.random.default_rng(stride)
    feat = torch.tensor(rng.standard_normal((900, 16)), dtype=torch.float32).to(G.DEV)
    idx = G.t(_cells(rng, 900, 2, [12, 20, 16]))
    conv = (sphconv.SubMConv3d(16, 32, 3, indice_key=key) if stride == 1 else
            sphconv.SparseConv3d(16, 32, 3, stride=2, padding=1, indice_key=key)).to(G.DEV).train(training)
    make = lambda: sphconv.SparseConvTensor(feat, [12, 20, 16], 2, indices=idx)
    with torch.set_grad_enabled(training):
        want = conv(make()).feature
        twin = copy.deepcopy(conv)
        torch.save(conv, tmp_path / "conv.pt")
        saved = torch.load(tmp_path / "conv.pt", weights_only=False)
        for c in (twin, saved):
            assert torch.equal(c.rule_size, conv.rule_size)
            assert torch.equal(c(make()).feature, want)
    padded = RuleBook.from_padded(*conv.rule_book.padded((2, 2)), 900, want.shape[0])
    again = copy.deepcopy(padded)
    w = conv.weight.detach().view(27, 16, 32)
    assert torch.equal(ext.rule_conv(feat, w, again, None, want.shape[0]), ext.rule_conv(feat, w, padded, None, want.shape[0]))


def test_weight_gradient_of_fewer_rows_than_the_book_holds():
    """Features that end early: pairs beyond them count for nothing, whichever books exist; a gradient that does is refused."""
    rng = np.random.default_rng(4)
    case = G.build_case(_cells(rng, 300, 1, [12, 60, 40]), 1, [12, 60, 40], [3, 3, 3], [2, 2, 2], [1, 1, 1], False)
    book = case["book"]
    f, d = torch.randn((300, 16), device=G.DEV), torch.randn((book.out_rows, 24), device=G.DEV)
    book.transposed()
    assert book.in_rows < book.out_rows and book.transposed_groups_built()
    padded = torch.cat([f[:170], torch.zeros_like(f[170:])])
    torch.testing.assert_close(ext.rule_conv_d_weight(f[:170], d, book, None), ext.rule_conv_d_weight(padded, d, book, None),
                               rtol=1e-5, atol=1e-4)
    for transposed, a, b in ((True, f[:170], d), (False, f, d[:-1])):
        with pytest.raises(L.SphconvError, match="fewer rows"):
            L.host().conv_wgrad(a, b, book.grouped(transposed).native, transposed, False)
    with pytest.raises(L.SphconvError, match="output rows"):
        ext.rule_conv_d_weight(f, d[:-1], book, None)


def test_small_arrays_are_checked_before_the_launch():
    """What the kernels read beside the rows: one float per output channel of scale and shift, an index per row."""
    rng = np.random.default_rng(0)
    idx = G.t(_cells(rng, 200, 1, [6, 8, 10]))
    x = sphconv.SparseConvTensor(torch.randn((200, 16), device=G.DEV), [6, 8, 10], 1, indices=idx)
    book = RuleBook.build_subm(x.z_idx, x.z_ptr, 1, [6, 8, 10], [3, 3, 3])
    w = torch.randn((27, 16, 32), device=G.DEV)
    good = torch.rand(32, device=G.DEV)
    assert ext.rule_conv(x.feature, w, book, None, 200, scale=good, shift=good).shape == (200, 32)
    for bad in (good[:31].contiguous(), good.half(), good.double()):
        for kw in ({"scale": bad}, {"scale": good, "shift": bad}):
            with pytest.raises(L.SphconvError, match="one value per output channel"):
                ext.rule_conv(x.feature, w, book, None, 200, **kw)
    for z_idx, z_ptr in ((x.z_idx[:199], x.z_ptr), (x.z_idx.long(), x.z_ptr), (x.z_idx, x.z_ptr.long())):
        with pytest.raises(L.SphconvError, match="int32"):
            sphconv.SparseConvTensor(x.feature, [6, 8, 10], 1, z_idx=z_idx, z_ptr=z_ptr).dense()
    empty = SimpleVoxel(4)(torch.zeros((7, 0, 4), device=G.DEV), torch.ones(7, device=G.DEV, dtype=torch.int32), None)
    assert torch.equal(empty, torch.zeros((7, 4), device=G.DEV))
