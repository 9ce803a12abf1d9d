"""Output coordinates of a strided layer in two launches (csrc/outcoords.h) against the three of sph_outcoords_count and
sph_outcoords_fill, bit by bit: tiles that end inside a line, workgroups of several tiles, columns of one to eight words, sums over
one and many tiles, rows written ahead of the count and behind it, several counts in flight on streams and threads."""
import ctypes as C
import threading

import pytest
import torch

from sphconv_amd import _lib as L
from sphconv_amd.rulebook import RuleBook

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
CASES = [  # (batch, shape, kernel, stride, padding, share of the bins)
    (1, (1, 1, 1), (3, 3, 3), (2, 2, 2), (1, 1, 1), 1.0),
    (2, (9, 20, 12), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.2),
    (3, (47, 1021, 45), (3, 3, 3), (1, 2, 2), (1, 1, 1), 0.3),
    (1, (64, 2048, 64), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.5),
    (4, (64, 2048, 64), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.3),       # too many rows to write ahead of the count
    (8, (64, 512, 200), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.01),
    (1, (64, 300, 300), (3, 3, 3), (2, 2, 3), (0, 1, 1), 0.1),
    (2, (20, 333, 900), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.02),      # eight words a column
    (1, (20, 50, 1100), (3, 3, 3), (2, 2, 2), (1, 1, 1), 0.02),      # none kept: three launches
    (2, (600, 1500, 4), (3, 3, 3), (1, 1, 1), (1, 1, 1), 0.05),      # more tiles than two launches serve
    (2, (70, 129, 20), (5, 5, 5), (3, 2, 2), (2, 2, 2), 0.1),
    (1, (16, 600, 16), (2, 2, 2), (2, 2, 2), (0, 0, 0), 0.0),
]


def _scene(batch, shape, keep, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    occ = torch.rand((batch,) + shape, generator=g, device=DEV) < keep
    return occ.nonzero()[:, 3].int().contiguous(), occ.sum(3).reshape(-1).cumsum(0).int().view(batch, shape[0], shape[1]).contiguous()


def _out(shape, kernel, stride, padding):
    return [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, padding)]


def _three(z_idx, z_ptr, batch, shape, kernel, stride, padding):
    out = _out(shape, kernel, stride, padding)
    lib, g = L.lib(), L.make_geom(batch, list(shape), out, list(kernel), list(stride), list(padding), [1, 1, 1])
    n = lib.sph_outcoords_scratch_ints(C.byref(g))
    scratch = torch.empty(n + 2, dtype=torch.int32, device=DEV)
    oz_ptr = torch.empty((batch, out[0], out[1]), dtype=torch.int32, device=DEV)
    L.check(lib.sph_outcoords_count(L.ptr(z_idx), L.ptr(z_ptr), z_idx.numel(), C.byref(g), L.ptr(oz_ptr), L.ptr(scratch), None, L.stream()))
    m = int(oz_ptr.view(-1)[-1].item())
    oz_idx, cols = (torch.full((m,), -1, dtype=torch.int32, device=DEV) for _ in range(2))
    L.check(lib.sph_outcoords_fill(L.ptr(z_idx), L.ptr(z_ptr), z_idx.numel(), C.byref(g), L.ptr(scratch), L.ptr(oz_ptr), L.ptr(oz_idx), m,
                                   L.ptr(cols), L.stream()))
    return oz_idx, oz_ptr, cols


def _ahead(z_idx, z_ptr, batch, shape, kernel, stride, padding):
    return RuleBook.count_ahead(z_idx, z_ptr, batch, list(shape), _out(shape, kernel, stride, padding), list(kernel), list(stride), list(padding))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[1])))
def test_two_launches_equal_three(case):
    batch, shape, kernel, stride, padding, keep = case
    z_idx, z_ptr = _scene(batch, shape, keep, shape[1])
    want = _three(z_idx, z_ptr, batch, shape, kernel, stride, padding)
    for _ in range(3):                       # the cells a count adds to are zeros again for the next one
        got = _ahead(z_idx, z_ptr, batch, shape, kernel, stride, padding).native.finish()
        assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_counts_in_flight_on_streams_and_threads():
    args = (2, (33, 500, 40), (3, 3, 3), (2, 2, 2), (1, 1, 1))
    scenes = [_scene(args[0], args[1], 0.1 + 0.1 * i, i) for i in range(4)]
    want = [_three(*s, *args) for s in scenes]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    flying = [_ahead(*scenes[(i + j) % 4], *args) for j in range(3)]
                    for j, f in reversed(list(enumerate(flying))):
                        got = f.native.finish()
                        torch.cuda.current_stream().synchronize()
                        if not all(torch.equal(x, y) for x, y in zip(got, want[(i + j) % 4])):
                            bad.append((i, j))
        except Exception as e:              # noqa: BLE001 (reported by the assertion below)
            bad.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_counts_nobody_waits_for_give_their_cells_back():
    args = (1, (8, 40, 12), (3, 3, 3), (2, 2, 2), (1, 1, 1))
    scene = _scene(args[0], args[1], 0.3, 1)
    want = _three(*scene, *args)
    _ahead(*scene, *args).native.finish()    # the first page of cells is there
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for _ in range(130):                     # more than two pages
        left = _ahead(*scene, *args)
        torch.cuda.synchronize()
        del left
    assert torch.cuda.memory_allocated() == before
    got = _ahead(*scene, *args).native.finish()
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_counts_whose_arrays_find_no_memory_give_their_cells_back():
    """The count is on its way when the arrays of its rows (2 MB each) are asked for: a layer that raises there leaves nothing behind."""
    args = (1, (32, 1024, 128), (3, 3, 3), (2, 2, 2), (1, 1, 1))
    scene = _scene(args[0], args[1], 0.05, 3)
    want = _three(*scene, *args)
    _ahead(*scene, *args).native.finish()    # the first page of cells is there
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    raised, full = 0, []
    try:                                     # no new memory, and none left in what there is for more than the small arrays
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / torch.cuda.get_device_properties(0).total_memory)
        try:
            while True:
                full.append(torch.empty(2 << 20, dtype=torch.uint8, device=DEV))
        except torch.OutOfMemoryError:
            pass
        before = torch.cuda.memory_allocated()
        for _ in range(130):                 # more than two pages
            try:
                _ahead(*scene, *args)
            except torch.OutOfMemoryError:
                raised += 1
            torch.cuda.synchronize()
        after = torch.cuda.memory_allocated()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        del full
    assert raised == 130 and after == before
    got = _ahead(*scene, *args).native.finish()
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_the_default_stream_while_another_records():
    """The default stream cannot be recorded, and must not be asked: where a stream that waits for it is, the question is an error."""
    args = (1, (8, 40, 12), (3, 3, 3), (2, 2, 2), (1, 1, 1))
    scene = _scene(args[0], args[1], 0.3, 2)
    want = _three(*scene, *args)
    torch.cuda.synchronize()
    hip = C.CDLL("libamdhip64.so")
    other, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(other), 0) == 0        # a blocking one
    try:
        assert hip.hipStreamBeginCapture(other, 2) == 0
        try:
            flying = [_ahead(*scene, *args) for _ in range(70)]        # more than a page of cells
            all_got = [f.native.finish() for f in flying]
        finally:
            assert hip.hipStreamEndCapture(other, C.byref(graph)) == 0
    finally:
        if graph:
            hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(other)
    assert all(torch.equal(x, y) for got in all_got for x, y in zip(got, want))
