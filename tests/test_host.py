"""CPU-only checks of the host side: the C-ABI library loads and exports every
symbol the public header declares, host arithmetic, and error paths that need no
GPU.  No kernel is launched here."""
import ctypes
import os
import re

import pytest
import torch

import sphconv_amd
from oracle import oracle as O
from sphconv_amd import _lib as L
from sphconv_amd import modules, utils

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    hdr = open(os.path.join(ROOT, "include", "sphconv_hip.h")).read()
    declared = set(re.findall(r"\b(sph_[a-z0-9_]+)\s*\(", hdr))
    declared -= {"sph_status", "sph_dtype"}
    assert declared, "no declarations found"
    assert os.path.exists(L.LIB_PATH), "libsphconv_hip.so is not built"
    lib = ctypes.CDLL(L.LIB_PATH)
    missing = [s for s in sorted(declared) if not hasattr(lib, s)]
    assert not missing, missing
    assert declared == set(L.EXPORTS), declared ^ set(L.EXPORTS)


def test_host_arithmetic_matches_oracle_closed_forms():
    lib = L.lib()
    assert lib.sph_abi_version() == L.ABI_VERSION
    assert lib.sph_book_tiles(0) == 0 and lib.sph_book_tiles(1) == 1 and lib.sph_book_tiles(129) == 2
    assert lib.sph_book_cap(27) == 27 * 8
    for B, shape, K, s, T, nnz in [(1, [64, 512, 32], [3, 3, 3], [1, 1, 1], [2, 2], 39256),
                                   (4, [64, 2048, 64], [3, 3, 3], [2, 2, 2], [2, 2], 630544),
                                   (8, [64, 512, 32], [3, 3, 3], [1, 1, 1], [4, 8], 314214),
                                   (2, [7, 9, 11], [2, 3, 1], [1, 2, 1], [3, 1], 50)]:
        out = utils.out_spatial(shape, K, s, [1, 1, 1])
        g = L.make_geom(B, shape, out, K, s, [1, 1, 1])
        assert lib.sph_tile_n_max(ctypes.byref(g), T[0], T[1], nnz) == O.tile_n_max(B, shape, K, s, T, nnz)
        assert lib.sph_num_tiles(ctypes.byref(g), T[0], T[1]) == -(-out[0] // T[0]) * -(-out[1] // T[1])
        assert out == O.out_spatial(shape, K, s, [1, 1, 1])


def test_argument_errors_without_gpu():
    lib = L.lib()
    g = L.make_geom(1, [4, 4, 4], [4, 4, 4], [7, 7, 7], [1, 1, 1], [3, 3, 3])     # KV = 343 > 128
    assert lib.sph_outcoords_blocks(ctypes.byref(g)) < 0
    assert b"geometry" in lib.sph_last_error()
    assert lib.sph_weight_packed_bytes(L.F16, 27, 64, 64) == 27 * 2 * 4 * 64 * 16
    assert lib.sph_weight_packed_bytes(L.F32, 27, 16, 16) == 27 * 1 * 1 * 64 * 16
    assert lib.sph_weight_packed_bytes(7, 27, 16, 16) == 0
    rc = lib.sph_conv_apply(L.F16, None, 0, 64, None, 64, None, None, None, None)
    assert rc == -1 and b"book" in lib.sph_last_error()
    with pytest.raises(L.SphconvError):
        L.check(rc)
    with pytest.raises(L.SphconvError):
        L.dtype_code(torch.float64)
    with pytest.raises(L.SphconvError):
        L.ptr(torch.zeros(4))            # not a GPU tensor


def test_module_construction_and_init():
    conv = sphconv_amd.SubMConv3d(16, 32, 3, padding=0, indice_key="k")
    assert tuple(conv.weight.shape) == (3, 3, 3, 16, 32) and conv.padding == (1, 1, 1) and conv.subm
    assert conv.bias is None and conv.rule_size is None
    # fan_in = oC * KV (reference utils/__init__.py:69-75): bound = sqrt(6/((1+5)*fan_in))
    bound = (6.0 / (6.0 * 32 * 27)) ** 0.5
    assert conv.weight.abs().max().item() <= bound
    c2 = sphconv_amd.SparseConv3d(4, 8, [3, 1, 3], stride=[2, 1, 2], padding=[1, 0, 1], bias=True)
    assert tuple(c2.weight.shape) == (3, 1, 3, 4, 8) and c2.bias.shape == (8,)
    assert "stride=(2, 1, 2)" in repr(c2)
    seq = sphconv_amd.SparseSequential(conv, torch.nn.ReLU(), c=c2)
    assert len(seq) == 3 and seq[0] is conv and seq[-1] is c2
    assert utils.out_spatial([64, 2048, 64], [3, 3, 3], [2, 2, 2], [1, 1, 1]) == [32, 1024, 32]
    assert utils._triple(3) == (3, 3, 3) and utils._triple([1, 2, 3]) == (1, 2, 3)
    sd = conv.state_dict()
    assert list(sd) == ["weight"]


def test_bench_refuses_more_than_one_gpu():
    """The path runs on one GPU; bench.py says so and exits before touching any device."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode == 2 and "ONE GPU" in r.stderr and r.stdout == ""


def test_training_channel_limit_is_reported_before_forward():
    """Forward takes up to 256 input channels, dgrad/wgrad up to 128: a module that wants gradients says so
    when it is called, not from inside backward()."""
    import torch
    import sphconv_amd
    from sphconv_amd.functional import ConvFunction
    feature = torch.zeros((4, 192), requires_grad=True)
    weight = torch.zeros((27, 192, 32), requires_grad=True)
    with pytest.raises(sphconv_amd.SphconvError, match="training takes 1..128 input channels"):
        ConvFunction.apply(feature, weight, None, None, [1, 1], 4)


def _launching_entry_points():
    """Entry points of the C ABI that take a stream."""
    hdr = open(os.path.join(ROOT, "include", "sphconv_hip.h")).read()
    names = re.findall(r"\b(sph_[a-z0-9_]+)\s*\([^;]*void \*stream\);", hdr)
    assert len(names) > 20
    return names


def test_the_host_extension_launches_on_its_tensors_device():
    """Every function of the host extension that launches has made its tensors' device current and takes the stream from
    there: a launch on the current device's stream is not ordered with what torch ran on the tensors' device."""
    src = open(os.path.join(ROOT, "sphconv_amd", "csrc", "host.cpp")).read()
    assert src.count("getCurrentHIPStream") == 1
    on_device = src[src.index("struct OnDevice"):]
    assert "DeviceGuard guard" in on_device[:on_device.index("};")] and "getCurrentHIPStream(t.device().index())" in on_device[:on_device.index("};")]
    launches = [m for m in re.finditer(r"\b(%s)\(" % "|".join(_launching_entry_points()), src)]
    assert len(launches) >= 13
    for m in launches:
        opening = list(re.finditer(r"\n( {4})?\{\n", src[:m.start()]))[-1]     # of the function that holds the launch
        head = src[max(src.rindex(end, 0, opening.start()) for end in ("}\n", ";\n")):opening.start()]
        assert "const OnDevice here(" in src[opening.end():m.start()] or "const OnDevice &here" in head, m.group(1)


def test_the_package_launches_on_its_tensors_device():
    """The same for the calls of the C ABI that Python makes itself."""
    import ast
    names = set(_launching_entry_points())
    seen = 0
    for file in sorted(os.listdir(os.path.join(ROOT, "sphconv_amd"))):
        if not file.endswith(".py"):
            continue
        tree = ast.parse(open(os.path.join(ROOT, "sphconv_amd", file)).read())
        guarded = [n for w in ast.walk(tree) if isinstance(w, ast.With) for n in ast.walk(w)
                   if any(isinstance(i.context_expr, ast.Call) and getattr(i.context_expr.func, "attr", "") == "on_device" for i in w.items)]
        for call in ast.walk(tree):
            if isinstance(call, ast.Call) and getattr(call.func, "attr", "") in names:
                seen += 1
                assert call in guarded, "%s:%d" % (file, call.lineno)
    assert seen >= 10


def test_stream_and_device_context_follow_the_tensors_device(monkeypatch):
    entered = []
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 1000 + index, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(L, "_current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "device", lambda d: entered.append(d) or L._IS_CURRENT)
    assert L.stream() == 1000 and L.stream(torch.device("cuda")) == 1000
    assert L.stream(torch.device("cuda", 1)) == 1001
    for d in (torch.device("cuda", 1), torch.device("cuda", 0), torch.device("cuda"), torch.device("cpu")):
        with L.on_device(d):
            pass
    assert entered == [torch.device("cuda", 1)]


def _affine_of(bn):
    x = torch.linspace(-2, 2, 5 * bn.num_features).view(5, bn.num_features)
    with torch.no_grad():
        want = bn(x)
        scale, shift = modules._bn_affine(bn, None)
    torch.testing.assert_close(x * scale + shift, want, rtol=1e-5, atol=1e-5)     # a few fp32 roundings


def test_batch_norm_whose_tensors_are_not_in_its_tables():
    """Pruned, replicated and weight-normed modules hold a weight or a mean as a plain attribute."""
    from torch.nn.utils import prune
    for name in ("weight", "bias", "running_mean", "running_var"):
        bn = torch.nn.BatchNorm1d(8).eval()
        with torch.no_grad():
            for t in (bn.weight, bn.bias, bn.running_mean, bn.running_var):
                t.uniform_(0.5, 2.0)
        _affine_of(bn)
        if name in bn._parameters:
            prune.random_unstructured(bn, name, 0.5)
        else:
            value = bn._buffers.pop(name)
            setattr(bn, name, value)
        for k in range(3):                      # its values change, at an address that may be an earlier one's
            with torch.no_grad():
                (bn._parameters.get(name + "_orig") if name + "_orig" in bn._parameters else getattr(bn, name)).mul_(1.5)
            _affine_of(bn)
        seq = sphconv_amd.Sequential(sphconv_amd.SubMConv3d(4, 8, 3), bn, torch.nn.ReLU()).eval()
        with torch.no_grad():
            n, found, relu = seq._fusable_tail(list(seq), 0)
        assert (n, found, relu) == ((0, None, False) if name + "_orig" in bn._parameters else (2, bn, True))


def test_modules_with_hooks_are_called_not_folded():
    """A hook sees every call of its module: such a module is not folded into the convolution before it."""
    seq = sphconv_amd.Sequential(sphconv_amd.SubMConv3d(4, 8, 3), torch.nn.BatchNorm1d(8), torch.nn.ReLU()).eval()
    conv, bn, act = list(seq)
    with torch.no_grad():
        assert seq._fusable_tail([conv, bn, act], 0) == (2, bn, True)
        h = act.register_forward_hook(lambda m, i, o: None)
        assert seq._fusable_tail([conv, bn, act], 0) == (1, bn, False)
        h.remove()
        h = bn.register_forward_pre_hook(lambda m, i: None)
        assert seq._fusable_tail([conv, bn, act], 0) == (0, None, False)
        h.remove()
        assert seq._fusable_tail([conv, bn, act], 0) == (2, bn, True)


def test_kept_affine_map_belongs_to_the_tensors_and_the_stream():
    """The affine map kept on a BatchNorm1d is not taken for another tensor that the allocator put at the same address, nor
    on a stream that is not ordered behind its computation; a copy of the module has its own."""
    import copy
    import numpy as np
    bn = torch.nn.BatchNorm1d(4).eval()
    memory = np.ones(4, dtype=np.float32)
    for value in (1.0, 2.0, 3.0):               # other values at one address, version 0 each time
        memory[:] = value
        bn.weight = torch.nn.Parameter(torch.from_numpy(memory))
        with torch.no_grad():
            torch.testing.assert_close(modules._bn_affine(bn, None)[0], torch.full((4,), value), rtol=1e-4, atol=0)
    with torch.no_grad():
        first = modules._bn_affine(bn, None)[0]
        assert modules._bn_affine(bn, None)[0] is first
        twin = copy.deepcopy(bn)
        twin.running_var.mul_(4.0)
        _affine_of(twin)
        assert modules._bn_affine(bn, None)[0] is first

        on7 = modules._bn_affine(bn, 7)[0]
        on8 = modules._bn_affine(bn, 8)[0]
        assert on8 is not on7 and modules._bn_affine(bn, 8)[0] is on8 and modules._bn_affine(bn, 7)[0] is on7


def test_a_count_started_ahead_outlives_the_tables_of_geometries(monkeypatch):
    """The tables of geometries start over after 4096 shapes: the layer whose count was started before is still that layer,
    and another layer's count is still refused."""
    from types import SimpleNamespace
    from sphconv_amd import rulebook

    def geometry(s0=16, stride=(2, 2, 2)):
        return rulebook.layer_geometry(2, s0, 40, 16, (3, 3, 3), stride, (1, 1, 1), (1, 1, 1), False)[0]

    z_idx, z_ptr = torch.zeros(5, dtype=torch.int32), torch.zeros((2, 16, 40), dtype=torch.int32)
    out = torch.zeros(7, dtype=torch.int32)
    monkeypatch.setattr(rulebook.L, "stream", lambda device=None: 3)

    def count(g):
        native = SimpleNamespace(stream=3, finish=lambda: (out, z_ptr, out))
        return SimpleNamespace(geometry=g, z_idx=z_idx, z_ptr=z_ptr, native=native)

    before = geometry()
    assert geometry() is before
    for s0 in range(17, 17 + 4096):
        geometry(s0)
    after = geometry()
    assert after is not before
    book = rulebook.RuleBook._strided(after, z_idx, z_ptr, count(before), None)
    assert book.out_rows == 7 and book.in_rows == 5
    for other in (geometry(18), geometry(16, (2, 2, 1))):
        with pytest.raises(L.SphconvError, match="another layer"):
            rulebook.RuleBook._strided(other, z_idx, z_ptr, count(before), None)


def test_what_is_more_than_values_does_not_go_past_torch(monkeypatch):
    """Tangents, transforms, traces and tensor subclasses go the way of torch's own operations."""
    import torch.autograd.forward_ad as fwAD
    from sphconv_amd import tensor as tensor_mod
    x = torch.randn(4, 3)
    assert utils.plain(x) and utils.plain(torch.nn.Parameter(x)) and utils.plain(torch.zeros(4, dtype=torch.int32))
    with fwAD.dual_level():
        assert utils.plain(x) and not utils.plain(fwAD.make_dual(x, x))
    seen = []
    look = lambda t: seen.append(utils.plain(t)) or t * 1
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.jit.trace(look, (x,), check_trace=False)
    assert seen == [False] * 3

    class Own(torch.Tensor):
        pass

    assert not utils.plain(x.as_subclass(Own))

    # a tensor made of rows with a tangent: refused by the autograd function, which has none, not dropped in silence
    zeros = torch.zeros(4, dtype=torch.int32)
    fake = lambda f, i, b, s: [f.detach().clone(), zeros, torch.zeros((1, 2, 2), dtype=torch.int32), zeros.clone(), zeros.clone()]
    monkeypatch.setattr(tensor_mod.ext, "_init_tensor", fake)
    indices = torch.zeros((4, 4), dtype=torch.int32)
    assert sphconv_amd.SparseConvTensor(x, [2, 2, 2], 1, indices=indices).feature.shape == (4, 3)
    with fwAD.dual_level(), pytest.raises(RuntimeError, match="jvp"):
        sphconv_amd.SparseConvTensor(fwAD.make_dual(x, x), [2, 2, 2], 1, indices=indices)


def test_threads_on_one_stream_have_scratch_books_of_their_own(monkeypatch):
    """A one-launch call that keeps no book writes its row count and kind into a scratch book before it launches: a call of
    another thread on the same stream must not get in between."""
    import threading
    from sphconv_amd import rulebook
    monkeypatch.setattr(rulebook.L, "stream", lambda device=None: 5)
    monkeypatch.setattr(rulebook.L, "capturing", lambda: False)
    cpu = torch.device("cpu")
    mine = rulebook._scratch_book(100, 27, cpu)
    assert rulebook._scratch_book(300, 27, cpu) is mine and mine.native.rows == 300
    theirs = []
    t = threading.Thread(target=lambda: theirs.append(rulebook._scratch_book(200, 27, cpu)))
    t.start()
    t.join()
    assert theirs[0].native.address != mine.native.address and theirs[0].struct().tile_ngrp != mine.struct().tile_ngrp
    assert mine.native.rows == 300 and theirs[0].native.rows == 200
    bigger = rulebook._scratch_book((1 << 17) + 1, 27, cpu)
    assert bigger is not mine and rulebook._scratch_book(10, 27, cpu) is bigger


def test_nothing_is_kept_or_reused_while_a_graph_is_captured(monkeypatch):
    """Under capture nothing is computed yet, memory is the graph's, and what it reads must not be given back later: packed
    weights, affine maps and scratch books are the graph's own."""
    from sphconv_amd import rulebook, sphconv_cuda as ext
    capturing = [False]
    monkeypatch.setattr(L, "capturing", lambda: capturing[0])
    monkeypatch.setattr(L, "stream", lambda device=None: 11)
    made = []

    class Host:
        def pack_weight(self, *a):
            made.append(torch.zeros(1))
            return made[-1]

    native = L.host()
    weight = torch.nn.Parameter(torch.zeros((27, 4, 8)))
    cpu = torch.device("cpu")
    with monkeypatch.context() as m, torch.no_grad():
        m.setattr(L, "host", lambda: Host())
        ext.invalidate_packed(weight)
        kept = ext._packed_weight(weight, False, cache=True)
        assert ext._kept_packed(weight) is kept and ext._packed_weight(weight, False, cache=True) is kept
        capturing[0] = True
        assert ext._kept_packed(weight) is None
        own = ext._packed_weight(weight, False, cache=True)
        assert own is not kept and ext._packed_weight(weight, False, cache=True) is not own
        capturing[0] = False
        assert ext._kept_packed(weight) is kept
        ext.invalidate_packed(weight)
    assert L.host() is native
    book = rulebook._scratch_book(50, 27, cpu)
    capturing[0] = True
    own = rulebook._scratch_book(50, 27, cpu)
    assert own is not book and own.native.address != book.native.address and rulebook._scratch_book(50, 27, cpu) is not own
    capturing[0] = False
    assert rulebook._scratch_book(50, 27, cpu) is book

    bn = torch.nn.BatchNorm1d(4).eval()
    rows = torch.zeros(3, 4)
    with torch.no_grad():
        first = modules._bn_affine(bn, 11)[0]
        on_gpu = type("OnGpu", (), {"is_cuda": True, "device": torch.device("cuda", 0)})
        assert modules._keeps_on(on_gpu) == 11 and modules._keeps_on(rows) is None
        capturing[0] = True
        assert modules._keeps_on(on_gpu) is False
        own = modules._bn_affine(bn, False)[0]
        assert own is not first and modules._bn_affine(bn, False)[0] is not own
        assert modules._bn_affine(bn, 11)[0] is first


def test_rule_books_can_be_copied_and_saved():
    """A module that has run holds its rule book, and is copied (for a moving average of its weights) and saved with it."""
    import copy
    import pickle
    z_idx, z_ptr = torch.zeros(5, dtype=torch.int32), torch.full((1, 4, 4), 5, dtype=torch.int32)
    book = sphconv_amd.RuleBook(z_idx, z_ptr, z_idx, z_ptr, 1, [4, 4, 8], [4, 4, 8], [3, 3, 3], [1, 1, 1], [1, 1, 1],
                                [1, 1, 1], True)
    conv = sphconv_amd.SubMConv3d(4, 8, 3)
    conv.__dict__["rule_book"] = book
    for twin in (copy.deepcopy(conv).rule_book, pickle.loads(pickle.dumps(book))):
        assert twin is not book and twin.z_idx is twin.oz_idx and torch.equal(twin.z_ptr, z_ptr) and not twin.built
        assert twin.kernel == [3, 3, 3] and twin.batch == 1 and twin.mirrored() and twin._geometry is book._geometry


@pytest.mark.parametrize("batch", [2, 2.0, torch.tensor(2), __import__("numpy").float32(2)])
def test_batch_sizes_and_shapes_of_any_number_type(monkeypatch, batch):
    """A batch size is often what a reduction over the coordinates returned."""
    from sphconv_amd import rulebook, sphconv_cuda as ext
    got = []

    class Host:
        def init_tensor(self, feature, indices, *size):
            got.append(size)
            return feature, None, None, None, None, 0, 0

    with monkeypatch.context() as m:
        m.setattr(L, "host", lambda: Host())
        ext.init_tensor(torch.zeros(3, 4), torch.zeros((3, 4), dtype=torch.int32), batch, [4.0, 5, 6])
    assert got == [(2, 4, 5, 6)] and all(type(v) is int for v in got[0])
    layer = lambda: rulebook.layer_geometry(batch, 4, 5, 6, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), True)[0]
    assert layer() is layer() is rulebook._geometry(2, [4, 5, 6], [4, 5, 6], (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1))
    assert layer().z_shape == (2, 4, 5)


def test_rows_of_another_width_do_not_reach_the_kernel(monkeypatch):
    """A module that keeps its packed weight knows its channels from the tensor's C; what is convolved are its rows, which
    somebody may have replaced."""
    from types import SimpleNamespace
    from sphconv_amd import sphconv_cuda as ext
    from sphconv_amd.rulebook import _Buffers
    z_idx, z_ptr = torch.zeros(3, dtype=torch.int32), torch.full((1, 2, 2), 3, dtype=torch.int32)
    conv = sphconv_amd.SubMConv3d(8, 16, 3).eval()
    book = sphconv_amd.RuleBook(z_idx, z_ptr, z_idx, z_ptr, 1, [2, 2, 4], [2, 2, 4], [3, 3, 3], [1, 1, 1], [1, 1, 1], [1, 1, 1], True)
    book.fwd = _Buffers(3, 27, torch.device("cpu"))
    monkeypatch.setattr(conv, "_rules", lambda *a, **k: (z_idx, z_ptr, book, None, [1, 1]))
    monkeypatch.setattr(ext, "_kept_packed", lambda *a: torch.zeros(4))
    x = sphconv_amd.SparseConvTensor(torch.zeros(3, 8), [2, 2, 4], 1, z_idx=z_idx, z_ptr=z_ptr)
    for rows, message in ((torch.zeros(3, 4), "mismatch"), (torch.zeros(3, 8, 1), "mismatch"), (torch.zeros(3, 8), "GPU tensor")):
        x.feature = rows
        with torch.no_grad(), pytest.raises(sphconv_amd.SphconvError, match=message):
            conv(x)


@pytest.mark.parametrize("call", ["init_tensor", "function"])
def test_coordinates_and_rows_are_checked_whoever_asks(call):
    """The autograd function of the public API is called by programs too: what the kernel reads is checked there as well."""
    from sphconv_amd import sphconv_cuda as ext
    from sphconv_amd.functional import InitTensorFunction
    make = ext.init_tensor if call == "init_tensor" else InitTensorFunction.apply
    rows, indices = torch.zeros(5, 3), torch.zeros((5, 4), dtype=torch.int32)
    for f, i in ((rows[:4], indices), (rows, indices.long()), (rows, indices[:, :3]), (rows, indices[0]), (rows[0], indices)):
        with pytest.raises(ValueError, match="must be"):
            make(f, i, 1, [2, 2, 2])
    with pytest.raises(sphconv_amd.SphconvError, match="GPU tensor"):
        make(rows, indices, 1, [2, 2, 2])


def test_weight_gradients_take_the_book_their_rows_fit(monkeypatch):
    """The gradient's kernel reads as many rows as its book is stationary on: fewer features than that keep to the forward
    book, which gathers them and checks each, and fewer gradient rows are refused."""
    from types import SimpleNamespace
    from sphconv_amd import sphconv_cuda as ext
    z_ptr = torch.full((1, 2, 2), 3, dtype=torch.int32)
    book = sphconv_amd.RuleBook(torch.zeros(3, dtype=torch.int32), z_ptr, torch.zeros(6, dtype=torch.int32), z_ptr, 1, [2, 2, 4],
                                [2, 2, 4], [3, 3, 3], [1, 1, 1], [1, 1, 1], [1, 1, 1], False)
    book.fwd, book._bwd = (SimpleNamespace(groups=True, native=side) for side in ("forward", "transposed"))
    monkeypatch.setattr(L, "host", lambda: SimpleNamespace(conv_wgrad=lambda f, d, native, transposed, f32: (native, transposed)))
    d_out = torch.zeros(6, 4)
    assert ext.rule_conv_d_weight(torch.zeros(3, 2), d_out, book, None) == ("transposed", True)
    assert ext.rule_conv_d_weight(torch.zeros(2, 2), d_out, book, None) == ("forward", False)
    with pytest.raises(sphconv_amd.SphconvError, match="output rows"):
        ext.rule_conv_d_weight(torch.zeros(3, 2), d_out[:5], book, None)


@pytest.mark.parametrize("momentum,affine", [(0.1, True), (0.1, False), (None, True)])
def test_kept_affine_map_follows_passes_in_training_mode(momentum, affine):
    """A training pass updates the running statistics without moving their version counters, also where no optimizer step
    follows (frozen or absent weights, statistics being gathered anew)."""
    bn = torch.nn.BatchNorm1d(4, momentum=momentum, affine=affine)
    for k in range(3):
        bn.train()
        bn(torch.randn(16, 4) * (k + 1) + 3)
        bn.eval()
        _affine_of(bn)
    bn.reset_running_stats()
    _affine_of(bn)
    bn.num_batches_tracked = None
    with torch.no_grad():
        _affine_of(bn)
        torch.nn.functional.batch_norm(torch.randn(16, 4), bn.running_mean, bn.running_var, training=True)
        _affine_of(bn)


def test_kept_packed_weight_is_dropped_when_the_program_trains(monkeypatch):
    """Optimizers and mixed-precision wrappers that write through ``weight.data`` leave no trace on the weight: a pass with
    gradients or in training mode, and a change of mode, drop the copy that evaluation keeps."""
    from types import SimpleNamespace
    from sphconv_amd import sphconv_cuda as ext
    z_idx, z_ptr = torch.zeros(3, dtype=torch.int32), torch.full((1, 2, 2), 3, dtype=torch.int32)
    conv = sphconv_amd.SubMConv3d(8, 16, 3).eval()
    book = sphconv_amd.RuleBook(z_idx, z_ptr, z_idx, z_ptr, 1, [2, 2, 4], [2, 2, 4], [3, 3, 3], [1, 1, 1], [1, 1, 1], [1, 1, 1], True)
    book.fwd = SimpleNamespace(groups=True, native=None)
    monkeypatch.setattr(conv, "_rules", lambda *a, **k: (z_idx, z_ptr, book, None, [1, 1]))
    x = sphconv_amd.SparseConvTensor(torch.zeros(3, 8), [2, 2, 4], 1, z_idx=z_idx, z_ptr=z_ptr)
    conv._layer(x)
    used, made = [], []
    host = SimpleNamespace(conv_apply=lambda f, packed, *a: used.append(packed) or torch.zeros(3, 16),
                           pack_weight=lambda w, *a: made.append(w.sum().item()) or made[-1])
    monkeypatch.setattr(L, "host", lambda: host)
    monkeypatch.setattr(L, "stream", lambda *a: 0)
    monkeypatch.setattr(L, "capturing", lambda: False)

    def evaluate():
        with torch.no_grad():
            conv(x)
        return used[-1]

    now = lambda: conv.weight.sum().item()
    assert evaluate() == now() and evaluate() == now() and len(made) == 1        # kept

    def step():
        conv.weight.data.add_(1.0)

    conv.train()
    step()
    conv.eval()
    assert evaluate() == now() and len(made) == 2
    conv.train()
    with torch.no_grad():
        conv(x)                                                                  # keeps nothing
    step()
    conv.training = False                                                        # without a call of eval()
    assert evaluate() == now()
    monkeypatch.setattr(sphconv_amd.conv.ConvFunction, "apply", lambda *a: torch.zeros(3, 16))
    conv(x)                                                                      # gradients in evaluation mode (fine-tuning)
    step()
    assert evaluate() == now()
    kept = len(made)
    assert evaluate() == now() and len(made) == kept
    step()
    conv.invalidate_packed()
    assert evaluate() == now()


def test_affine_map_is_dropped_where_the_module_runs_on_its_own(monkeypatch):
    bn = torch.nn.BatchNorm1d(4).eval()
    z_idx, z_ptr = torch.zeros(3, dtype=torch.int32), torch.full((1, 2, 2), 3, dtype=torch.int32)
    seq = sphconv_amd.Sequential(bn)
    with torch.no_grad():
        modules._bn_affine(bn, None)
    assert bn.__dict__["_sph_affines"]
    seq(sphconv_amd.SparseConvTensor(torch.zeros(3, 4), [2, 2, 4], 1, z_idx=z_idx, z_ptr=z_ptr))
    bn.weight.data.mul_(2.0)
    _affine_of(bn)
