"""Rule book: this package's compact form of the reference's rule tensors.

The reference returns ``rules [NTile,KV,2,tile_n_max]`` padded with -1 plus
``rule_size [NTile,KV]`` (src/sphconv/rules.cu:364-369): hundreds of megabytes of
padding at LiDAR sizes.  A :class:`RuleBook` keeps the same pairs in the layout
the HIP kernels consume (see ``include/sphconv_hip.h``) and materialises the
padded tensors only when asked (:meth:`RuleBook.padded`).
"""
import ctypes as C
import threading
from typing import List, Optional, Sequence

import torch

from . import _lib as L
from .utils import out_spatial


class _Buffers:
    """Device arrays of one book (forward or transposed), carved out of ONE allocation by the host extension; the
    named tensors are views made on first access."""

    _FIELDS = ("tile_ngrp", "tile_koff", "grp_k", "grp_gather", "grp_owner", "tile_nbr")

    def __init__(self, rows: int, kv: int, device, by_row: bool = False, groups: bool = True):
        """``by_row`` also keeps the pairs by stationary row (``tile_nbr`` [NT,KV,128]), the form the
        convolution walks when neighbourhoods are dense; with it, ``groups=False`` leaves the groups out
        (forward-only use: the rule kernel then writes a fifth of the bytes)."""
        self.rows, self.kv = int(rows), int(kv)
        self.by_row = bool(by_row)
        self.groups = bool(groups) or not self.by_row
        if not isinstance(device, torch.device):
            device = torch.device(device)
        self.native = L.host().BookBuffers(self.rows, self.kv, device, self.by_row, self.groups)
        self._struct = None
        self._views = None

    def struct(self) -> L.Book:
        """The book as the C ABI takes it (the extension's own struct: what is set here, its calls see)."""
        if self._struct is None:
            self._struct = L.Book.from_address(self.native.address)
        return self._struct

    def __getattr__(self, name):
        if name in ("storage", "ntiles", "cap"):
            return getattr(self.native, name)
        # views of the single allocation, typed and shaped like the C arrays
        if name in _Buffers._FIELDS:
            if self._views is None:
                self._views = {}
            v = self._views.get(name)
            if v is None:
                first, size = self.native.range(_Buffers._FIELDS.index(name))
                raw = self.storage[first:first + size]
                v = raw.view(torch.int16 if name == "tile_koff" else torch.int32)
                if name == "tile_koff":
                    v = v.view(max(self.ntiles, 1), self.kv + 1)
                if name == "tile_nbr":
                    v = v.view(max(self.ntiles, 1), self.kv, L.TILE_ROWS) if self.by_row else None
                elif name.startswith("grp_") and not self.groups:
                    v = None
                self._views[name] = v
            return v
        raise AttributeError(name)

    def num_pairs(self) -> int:
        """Total pairs held (synchronises)."""
        if self.ntiles == 0:
            return 0
        if not self.groups:
            return int((self.tile_nbr[:self.ntiles] >= 0).sum().item())
        ng = self.tile_ngrp[:self.ntiles].long()
        own = self.grp_owner.view(self.ntiles, self.cap * L.GROUP)
        used = torch.arange(self.cap * L.GROUP, device=own.device)[None, :] < (ng * L.GROUP)[:, None]
        return int(((own >= 0) & used).sum().item())


# Pairs to a row up to which a strided layer's book is said to be thin (``SPH_THIN``).
THIN_PAIRS = 1.45


class _Geometry:
    """One convolution geometry: the C struct and what Python wants to know of it.  Made once per geometry and shared
    by every book that has it (a network meets a few dozen)."""

    __slots__ = ("native", "batch", "in_shape", "out_shape", "kernel", "stride", "padding", "dilation", "kv", "in_cells",
                 "out_cells", "steps", "odd_same", "z_shape", "cluster", "key", "thin", "plane")

    def __init__(self, batch, in_shape, out_shape, kernel, stride, padding, dilation):
        self.batch = batch
        # what two layers' geometries are compared by: the tables below start over now and then, and make another object
        self.key = (batch, *in_shape, *out_shape, *kernel, *stride, *padding, *dilation)
        self.in_shape, self.out_shape, self.kernel = list(in_shape), list(out_shape), list(kernel)
        self.stride, self.padding, self.dilation = list(stride), list(padding), list(dilation)
        self.kv = kernel[0] * kernel[1] * kernel[2]
        self.in_cells = max(batch * in_shape[0] * in_shape[1] * in_shape[2], 1)
        self.out_cells = max(batch * out_shape[0] * out_shape[1] * out_shape[2], 1)
        self.steps = stride[0] * stride[1] * stride[2]
        self.z_shape = (batch, in_shape[0], in_shape[1])
        # Outputs an input row makes, as an output row meets them (size-biased mean): an input reaches floor or ceil
        # of K / stride outputs on each axis, neighbours of one another -- 1 to 8, 4.6 as an output row sees it, for a
        # 3x3x3 kernel of stride 2.
        self.cluster = 1.0
        for k, s in zip(kernel, stride):
            reach = [len(range(r, k, s)) for r in range(s)]
            self.cluster *= sum(c * c for c in reach) / max(sum(reach), 1)
        # stationary rows from which a strided layer's book is thin, to an input row; rows that lie between a kernel plane's
        # first and last column, to a row of each side (``SPH_PLANE``)
        self.thin = self.kv / (THIN_PAIRS * self.steps)
        self.plane = tuple((kernel[1] - 1) * dilation[1] / max(batch * s[0] * s[1], 1) for s in (in_shape, out_shape))
        # odd kernel, stride 1, padding K//2: a submanifold book is then its own transpose, offsets mirrored
        self.odd_same = all(k % 2 == 1 for k in kernel) and self.steps == 1 and all(p == k // 2 for p, k in zip(padding, kernel))
        self.native = L.host().Geometry(batch, self.in_shape, self.out_shape, self.kernel, self.stride, self.padding,
                                        self.dilation)

    def __reduce__(self):
        return _geometry, (self.batch, self.in_shape, self.out_shape, self.kernel, self.stride, self.padding, self.dilation)


_GEOMETRIES = {}


def _geometry(batch, in_shape, out_shape, kernel, stride, padding, dilation) -> _Geometry:
    batch = int(batch)
    key = (batch, *in_shape, *out_shape, *kernel, *stride, *padding, *dilation)
    g = _GEOMETRIES.get(key)
    if g is None:
        if len(_GEOMETRIES) >= 4096:                     # a program with ever new shapes: start over
            _GEOMETRIES.clear()
        g = _Geometry(batch, *(tuple(int(v) for v in x) for x in (in_shape, out_shape, kernel, stride, padding, dilation)))
        _GEOMETRIES[key] = g
    return g

# A layer's geometry and output shape by what the layer and its input hold, so that a forward pass does not work them out
# again (shapes are a list comprehension with divisions, the geometry's key twenty numbers).
_LAYERS = {}


def layer_geometry(batch, D, W, H, kernel, stride, padding, dilation, subm):
    """-> (geometry, output shape) of a layer on a ``[batch, D, W, H]`` grid."""
    batch = int(batch)
    key = (batch, D, W, H, kernel, stride, padding, dilation, subm)
    hit = _LAYERS.get(key)
    if hit is None:
        shape = [D, W, H]
        out = shape if subm else out_spatial(shape, kernel, stride, padding, dilation)
        if len(_LAYERS) >= 4096:
            _LAYERS.clear()
        hit = _LAYERS[key] = (_geometry(batch, shape, out, kernel, (1, 1, 1) if subm else stride, padding, dilation), tuple(out))
    return hit


# Estimated pairs per stationary row from which a book also keeps its pairs by row (and the
# convolution walks that form).  float("inf") never does, 0 always.
BY_ROW_MIN_PAIRS = 10.0
# A book built for a forward pass that is known to go by rows, with no gradient being recorded, leaves
# its groups out (a fifth of the bytes the rule kernel writes), which moves the break-even down:
# measured on a 4x32x1024x32 grid, rules + convolution, by rows against by groups: 99/115 us at an
# estimate of 5.4 pairs per row, 113/149 at 6.75, 141/194 at 8.1 (32->32 fp16); 273/215, 347/314,
# 412/413 (64->64): one line between the two.  The threshold of such books is this fraction of the one
# above (where a book with groups and the table breaks even at 10.8: 298/297 and 653/670).
BY_ROW_FORWARD_ONLY = 0.65


class RuleBook:
    """Pairs of one convolution geometry on one sparse tensor."""

    def __init__(self, z_idx, z_ptr, oz_idx, oz_ptr, batch, in_shape, out_shape, kernel, stride,
                 padding, dilation, subm, row_cols=None, out_row_cols=None):
        self._take(_geometry(batch, in_shape, out_shape, kernel, stride, padding, dilation), z_idx, z_ptr, oz_idx, oz_ptr,
                   subm, row_cols, out_row_cols)

    @classmethod
    def _of(cls, geometry, z_idx, z_ptr, oz_idx, oz_ptr, subm, row_cols, out_row_cols) -> "RuleBook":
        rb = cls.__new__(cls)
        rb._take(geometry, z_idx, z_ptr, oz_idx, oz_ptr, subm, row_cols, out_row_cols)
        return rb

    def _take(self, geometry, z_idx, z_ptr, oz_idx, oz_ptr, subm, row_cols, out_row_cols):
        self._geometry = geometry
        self.z_idx, self.z_ptr = z_idx, z_ptr
        self.oz_idx, self.oz_ptr = oz_idx, oz_ptr
        # optional: the column of every input / output row (what init_tensor and the output-coordinate kernels know
        # when they write the rows); the rule kernel then need not search z_ptr for them
        self.row_cols, self.out_row_cols = row_cols, out_row_cols
        self.subm = bool(subm)
        self.kv = geometry.kv
        self.in_rows = z_idx.shape[0] if z_idx is not None else 0
        self.out_rows = oz_idx.shape[0] if oz_idx is not None else 0
        self._fwd: Optional[_Buffers] = None   # built on first use (see ``fwd``)
        self._bwd: Optional[_Buffers] = None
        self.keep = True                       # a fused rules + forward launch also writes the book (``fused_forward``)
        # (input channels, output channels, element size) of the forward pass a lazy book is made for, when no
        # gradient will be asked of it: lets a book that goes by rows leave its groups out (see ``_build``)
        self.forward_only: Optional[tuple] = None
        # rows that lie together in the gathered side's grid whatever its occupancy (``_Geometry.cluster`` of the layer
        # that made them; 1: nothing known)
        self.cluster = 1.0
        self._padded = None
        self._from_padded = None     # (rules, rule_size) when built from reference-format tensors

    # the geometry's numbers (None / 0 for a book made from padded tensors, which has none)
    batch = property(lambda self: self._geometry.batch if self._geometry is not None else 0)
    in_shape = property(lambda self: self._geometry.in_shape if self._geometry is not None else None)
    out_shape = property(lambda self: self._geometry.out_shape if self._geometry is not None else None)
    kernel = property(lambda self: self._geometry.kernel if self._geometry is not None else None)
    stride = property(lambda self: self._geometry.stride if self._geometry is not None else None)
    padding = property(lambda self: self._geometry.padding if self._geometry is not None else None)
    dilation = property(lambda self: self._geometry.dilation if self._geometry is not None else None)

    # -- construction -----------------------------------------------------
    @property
    def fwd(self) -> _Buffers:
        """The forward book (stationary on output rows); a book made with ``lazy=True`` is built here."""
        if self._fwd is None:
            self._fwd = self._convert(False) if self._from_padded is not None else self._build(False)
        return self._fwd

    @fwd.setter
    def fwd(self, buf):
        self._fwd = buf

    def __getstate__(self):
        """What a copy or a saved module takes along: the coordinates, not the pairs, which it makes again when it needs
        them."""
        return dict(self.__dict__, _fwd=None, _bwd=None)

    @property
    def built(self) -> bool:
        return self._fwd is not None

    def geom(self) -> L.Geom:
        return L.make_geom(self.batch, self.in_shape, self.out_shape, self.kernel, self.stride,
                           self.padding, self.dilation)

    def _pairs_per_row(self, transposed: bool) -> float:
        """Pairs a stationary row can expect: kernel volume x occupancy of the gathered side's grid
        (a stride thins the offsets that can pair with an input row), and the rest of a row's cluster where the
        gathered rows are the outputs of a strided layer: one scan's second encoder stage holds 4.1 pairs per row by
        its occupancy and about eight in fact (grouped 41 us per layer, by rows 22)."""
        g = self._geometry
        if transposed:
            return g.kv * self.out_rows / g.out_cells / g.steps
        return g.kv * self.in_rows / g.in_cells + self.cluster - 1.0

    def _said(self, transposed: bool, by_row: bool) -> int:
        """What the book says of its pairs (``sph_book.middle_run``): a submanifold layer pairs every row with itself at
        the middle offset; a strided layer's pairs are known (kernel volume / stride to an input row), and may be hardly more than
        its rows; and of a by-row book how far apart lies what a row gathers."""
        g = self._geometry
        if self.subm:
            said = L.RUN
        else:
            said = L.THIN if g.thin * self.in_rows <= (self.in_rows if transposed else self.out_rows) else 0
        if by_row:
            if transposed:
                said |= L.plane(self.out_rows * g.plane[1] + 0.999, 1)
            else:
                said |= L.plane(self.in_rows * g.plane[0] + 0.999, g.stride[0])
        return said

    def _rows_kernel_takes(self, weight, weight_transposed: bool) -> bool:
        """Whether ``sph_conv_apply`` can walk this layer by stationary row (rows of 16-byte multiples up
        to 128 bytes, 16-byte multiples out, a table that fits LDS): the conditions of the library."""
        kv, wa, wb = weight.shape
        kdim, ndim = (wb, wa) if weight_transposed else (wa, wb)
        return self._rows_kernel_takes_shape(kdim, ndim, weight.element_size())

    def _rows_kernel_takes_shape(self, kdim: int, ndim: int, es: int) -> bool:
        return (kdim * es) % 16 == 0 and kdim * es <= 128 and (ndim * es) % 16 == 0 and self.kv * L.TILE_ROWS * 4 <= 48 * 1024

    def _build(self, transposed: bool, weight=None, weight_transposed: bool = False, groups: Optional[bool] = None):
        """Launches the rule kernel.  With ``weight`` [KV,a,b] its fragment-ordered copy (what
        ``sph_weight_pack`` makes, for the contraction over ``a``, or over ``b`` when
        ``weight_transposed``) is produced by the same launch and returned with the buffers.
        ``groups`` None: a by-row book leaves its groups out when it is built for a forward pass that
        is known to go by rows and no gradient is being recorded (they are built on demand later:
        :meth:`grouped`)."""
        rows = self.in_rows if transposed else self.out_rows
        est = self._pairs_per_row(transposed)
        by_row = est >= BY_ROW_MIN_PAIRS
        if groups is None:
            forward_only = (weight is not None and not torch.is_grad_enabled() and weight.dim() == 3
                            and self._rows_kernel_takes(weight, weight_transposed))
            if weight is None and not transposed and self.forward_only is not None and not torch.is_grad_enabled():
                forward_only = self._rows_kernel_takes_shape(*self.forward_only)
            if forward_only:
                by_row = est >= BY_ROW_MIN_PAIRS * BY_ROW_FORWARD_ONLY
            groups = not (by_row and forward_only)
        buf = _Buffers(rows, self.kv, self.z_ptr.device, by_row, groups)
        buf.native.middle_run = self._said(transposed, by_row)
        hint = self.row_cols if transposed else self.out_row_cols
        where = (self.z_idx, self.z_ptr, self.oz_idx, self.oz_ptr, self._geometry.native, transposed, buf.native, hint)
        if weight is None:
            L.host().rules_build(*where)
            return buf
        w = weight.detach()
        if not w.is_contiguous():
            w = w.contiguous()
        if not w.is_cuda or w.dim() != 3:
            raise L.SphconvError("weight must be a GPU tensor [KV,iC,oC]")
        return buf, L.host().rules_build_pack(*where, w, int(bool(weight_transposed)), False, L.dtype_code(w.dtype))

    def _build_for_training(self, weight, dtype):
        """The forward book and, by the same launch, the layer's weight (its own type or fp32, rounded to ``dtype``)
        in fragment order for the forward pass and for dgrad; -> the two copies."""
        by_row = self._pairs_per_row(False) >= BY_ROW_MIN_PAIRS
        buf = _Buffers(self.out_rows, self.kv, self.z_ptr.device, by_row, True)
        buf.native.middle_run = self._said(False, by_row)
        both = L.host().rules_build_pack(self.z_idx, self.z_ptr, self.oz_idx, self.oz_ptr, self._geometry.native, False,
                                         buf.native, self.out_row_cols, weight, 2, self.mirrored(), L.dtype_code(dtype))
        self._fwd = buf
        return both

    @classmethod
    def build_subm(cls, z_idx, z_ptr, batch, shape, kernel, padding=None,
                   dilation=(1, 1, 1), weight=None, row_cols=None, lazy=False):
        """Submanifold rules (replaces get_rules_subm, rules.cu:326-390): stride 1,
        outputs are the inputs; ``padding`` defaults to K//2 (conv.py:210).
        With ``weight`` [KV,iC,oC] returns ``(book, packed_weight)``: the layer's weight is
        put in fragment order by the same kernel launch (pass it to ``rule_conv(..., packed=)``).
        ``row_cols`` (optional, int32 [NNZ]): the column of every row (``SparseConvTensor.row_cols``).
        ``lazy``: launch nothing yet; the pairs are generated by the first use -- by ``rule_conv`` in the same
        launch as the convolution where the library has that kernel (:meth:`fused_forward`)."""
        pad = [int(k) // 2 for k in kernel] if padding is None else padding
        geometry = _geometry(batch, shape, shape, kernel, (1, 1, 1), pad, dilation)
        rb = cls._subm(geometry, z_idx, z_ptr, row_cols)
        if lazy:
            return rb
        if weight is None:
            rb.fwd = rb._build(False)
            return rb
        rb.fwd, packed = rb._build(False, weight)
        return rb, packed

    @classmethod
    def count_ahead(cls, z_idx, z_ptr, batch, in_shape, out_shape, kernel, stride, padding, dilation=(1, 1, 1)):
        """First half of :meth:`build`, to be enqueued as soon as a strided layer's INPUT coordinates exist:
        the output rows per column are counted and scanned, the row count goes to pinned host memory, and the
        coordinates are written behind it.  Pass the returned object to ``build(..., ahead=)`` when the layer
        itself is reached: whatever the caller has enqueued in between (the convolutions of the layers before)
        keeps the GPU busy while the host reads the count, instead of the GPU waiting for the host."""
        return cls._count(_geometry(batch, in_shape, out_shape, kernel, stride, padding, dilation), z_idx, z_ptr)

    @classmethod
    def _subm(cls, geometry, z_idx, z_ptr, row_cols) -> "RuleBook":
        """A submanifold book, not built yet."""
        if not geometry.native.takes(z_idx, z_ptr):
            _check_index_tensors(z_idx, z_ptr, geometry.z_shape)          # says what is wrong
        return cls._of(geometry, z_idx, z_ptr, z_idx, z_ptr, True, row_cols, row_cols)

    @classmethod
    def _count(cls, geometry, z_idx, z_ptr) -> "_CountAhead":
        if not geometry.native.takes(z_idx, z_ptr):
            _check_index_tensors(z_idx, z_ptr, geometry.z_shape)          # says what is wrong
        if min(geometry.out_shape) <= 0:
            raise L.SphconvError("empty output grid %s" % geometry.out_shape)
        return _CountAhead(geometry, z_idx, z_ptr)

    @classmethod
    def _strided(cls, geometry, z_idx, z_ptr, ahead, row_cols) -> "RuleBook":
        """A strided layer's book: its output coordinates now, its pairs not built yet."""
        if ahead is None:
            ahead = cls._count(geometry, z_idx, z_ptr)
        elif ahead.geometry.key != geometry.key or ahead.z_idx.data_ptr() != z_idx.data_ptr() \
                or ahead.z_ptr.data_ptr() != z_ptr.data_ptr() or ahead.native.stream != L.stream(z_ptr.device):
            raise L.SphconvError("count_ahead() was called for another layer, tensor or stream")
        # the rows' columns are a by-product of the coordinates
        oz_idx, oz_ptr, out_cols = ahead.native.finish()
        return cls._of(geometry, z_idx, z_ptr, oz_idx, oz_ptr, False, row_cols, out_cols)

    @classmethod
    def build(cls, z_idx, z_ptr, batch, in_shape, out_shape, kernel, stride, padding,
              dilation=(1, 1, 1), weight=None, ahead=None, row_cols=None, lazy=False):
        """Strided rules (replaces get_rules, rules.cu:405-486): output coordinates
        (oz_ptr inclusive scan, oz_idx ascending per column) and pairs.  One wait for the
        output row count, as in the reference (rules.cu:461): the scan kernel writes it to pinned
        host memory and the host waits for that store alone -- behind it the kernel that writes the coordinates is
        enqueued already, so the GPU is not idle meanwhile.  ``ahead``: what :meth:`count_ahead` returned for the same
        arguments on the same stream."""
        geometry = _geometry(batch, in_shape, out_shape, kernel, stride, padding, dilation)
        rb = cls._strided(geometry, z_idx, z_ptr, ahead, row_cols)
        if lazy:                                     # output coordinates now, pairs with the first use
            return rb
        if weight is None:
            rb.fwd = rb._build(False)
            return rb
        rb.fwd, packed = rb._build(False, weight)    # (book, packed weight) as in build_subm
        return rb, packed

    @classmethod
    def from_padded(cls, rules, rule_size, in_rows: int, out_rows: int) -> "RuleBook":
        """Book from the reference's padded tensors (any tile size)."""
        if rules.dim() != 4 or rules.shape[2] != 2 or rule_size.dim() != 2 \
                or rule_size.shape[0] != rules.shape[0] or rule_size.shape[1] != rules.shape[1]:
            raise L.SphconvError("rules must be [NTile,KV,2,n] and rule_size [NTile,KV], got %s, %s"
                                 % (tuple(rules.shape), tuple(rule_size.shape)))
        if rules.dtype != torch.int32 or rule_size.dtype != torch.int32:
            raise L.SphconvError("rules and rule_size must be int32")
        rb = cls.__new__(cls)
        rb._geometry = None
        rb.z_idx = rb.z_ptr = rb.oz_idx = rb.oz_ptr = None
        rb.subm = False
        rb.kv = int(rules.shape[1])
        rb.in_rows, rb.out_rows = int(in_rows), int(out_rows)
        rb._bwd = None
        rb._fwd = None
        rb.keep = True
        rb.forward_only = None
        rb.row_cols = rb.out_row_cols = None
        rb.cluster = 1.0
        rb._padded = None
        rb._from_padded = (rules.contiguous(), rule_size.contiguous())
        rb.fwd = rb._convert(False)
        return rb

    def _convert(self, transposed: bool) -> _Buffers:
        rules, rule_size = self._from_padded
        rows = self.in_rows if transposed else self.out_rows
        buf = _Buffers(rows, self.kv, rules.device)
        nbr = torch.empty(max(rows, 1) * self.kv, dtype=torch.int32, device=rules.device)
        b = buf.struct()
        with L.on_device(rules.device):
            L.check(L.lib().sph_rules_from_padded(L.ptr(rules), L.ptr(rule_size), int(rules.shape[0]),
                                                  self.kv, int(rules.shape[3]), self.in_rows,
                                                  self.out_rows, int(transposed), L.ptr(nbr),
                                                  C.byref(b), L.stream()))
        return buf

    # Tiles up to which one launch for rules + forward beats two (three workgroups of four waves, or four of two,
    # per CU hold that many at once; beyond, the launch runs in rounds and the two kernels are as fast or faster:
    # measured on the 64 x 2048 x 64 grid, 64 -> 64 fp16: 746 tiles 21.8 against 26.1 us, 937 tiles 29.3 / 32.0,
    # 2457 tiles 68.6 / 66.9, 5957 tiles 140 / 142).
    FUSED_MAX_TILES = 1024

    def goes_in_one_launch(self, kdim: int, ndim: int, element_size: int) -> bool:
        """Whether this book's pairs are better made by the launch that convolves them (``fused_forward``)."""
        row_bytes, rows = kdim * element_size, self.out_rows
        return (self._fwd is None and self._from_padded is None and 0 < rows <= self.FUSED_MAX_TILES * L.TILE_ROWS
                and self.kv <= 32 and ndim <= 64 and row_bytes % 16 == 0 and row_bytes <= 128
                and self._pairs_per_row(False) < BY_ROW_MIN_PAIRS * BY_ROW_FORWARD_ONLY)

    def fused_forward(self, feature: torch.Tensor, packed: torch.Tensor, kdim: int, ndim: int, scale=None, shift=None,
                      relu: bool = False):
        """Pairs and forward convolution of this (not yet built) book in ONE launch (``sph_rules_conv``): replaces
        get_rules_subm / get_rules' pair half + rule_conv (rules.cu:326-486, rule_conv.cu:286-336) where the
        reference launches three kernels.  Returns the output rows, or None when this layer is better served by
        the two kernels (dense neighbourhoods that go by rows, more than FUSED_MAX_TILES tiles, shapes the
        library's fused kernel does not take).  With ``self.keep`` the book is written too and the object counts
        as built afterwards; without, only the output exists and a later use of the book generates it."""
        if not self.goes_in_one_launch(kdim, ndim, feature.element_size()):
            return None
        rows = self.out_rows
        dev = self.z_ptr.device
        # a book nobody keeps is the stream's own
        buf = _Buffers(rows, self.kv, dev) if self.keep else _scratch_book(rows, self.kv, dev)
        buf.native.middle_run = int(self.subm)
        out = L.host().rules_conv(self.z_idx, self.z_ptr, self.oz_idx, self.oz_ptr, self._geometry.native, buf.native,
                                  int(self.keep), self.out_row_cols, feature, packed, kdim, ndim, scale, shift, relu)
        if out is not None and self.keep:
            self._fwd = buf
        return out

    # -- views ------------------------------------------------------------
    def grouped(self, transposed: bool = False) -> _Buffers:
        """The forward (or transposed) book with its groups, which wgrad, the padded tensors and the
        grouped convolution kernels need; rebuilt once if it was made for a by-row forward pass only."""
        buf = self.transposed() if transposed else self.fwd
        if not buf.groups:
            buf = self._build(transposed, groups=True)
            if transposed:
                self._bwd = buf
            else:
                self._fwd = buf
        return buf

    def mirrored(self) -> bool:
        """True if the book is its own transpose up to mirroring the offsets (k <-> KV-1-k): submanifold,
        stride 1, odd kernel, padding K//2 -- then dgrad runs on the forward book with reversed weights."""
        return self.subm and self._geometry is not None and self.oz_idx is self.z_idx and self._geometry.odd_same

    def transposed(self) -> _Buffers:
        """Book stationary on input rows (what dgrad gathers through when the book is not mirrored)."""
        if self._bwd is None:
            self._bwd = self._convert(True) if self._from_padded is not None else self._build(True)
        return self._bwd

    def transposed_groups_built(self) -> bool:
        """True if the transposed book exists, with its groups."""
        return self._bwd is not None and self._bwd.groups

    def num_pairs(self) -> int:
        return self.fwd.num_pairs()

    def padded(self, tile_size: Sequence[int] = (2, 2)):
        """-> (rules [NTile,KV,2,tile_n_max], rule_size [NTile,KV]) in the reference's
        format, lists in ascending output row.  ``tile_n_max`` is the reference's
        heuristic (rules.cu:21-28) raised, if needed, to the longest list so that no
        pair is dropped (the reference drops them, rules.cu:301-308)."""
        if self._from_padded is not None:
            return self._from_padded
        key = (int(tile_size[0]), int(tile_size[1]))
        if self._padded is None:
            self._padded = {}
        if key not in self._padded:
            lib = L.lib()
            g, b = self.geom(), self.grouped().struct()
            dev = self.z_ptr.device
            ntile = lib.sph_num_tiles(C.byref(g), *key)
            nbr = torch.empty(max(self.out_rows, 1) * self.kv, dtype=torch.int32, device=dev)
            rule_size = torch.empty((ntile, self.kv), dtype=torch.int32, device=dev)
            with L.on_device(dev):
                L.check(lib.sph_rules_to_padded_count(C.byref(b), L.ptr(self.oz_ptr), C.byref(g), key[0],
                                                      key[1], L.ptr(nbr), L.ptr(rule_size), L.stream()))
            n_max = lib.sph_tile_n_max(C.byref(g), key[0], key[1], self.in_rows)
            longest = int(rule_size.max().item()) if rule_size.numel() else 0
            n_max = max(n_max, (longest + 15) & ~15, 16)
            rules = torch.empty((ntile, self.kv, 2, n_max), dtype=torch.int32, device=dev)
            with L.on_device(dev):
                L.check(lib.sph_rules_to_padded_fill(L.ptr(self.oz_ptr), C.byref(g), key[0], key[1],
                                                     L.ptr(nbr), self.out_rows, self.kv, n_max,
                                                     L.ptr(rules), L.stream()))
            self._padded[key] = (rules, rule_size)
        return self._padded[key]

    def tile_grid_shape(self, tile_size: Sequence[int] = (2, 2)) -> List[int]:
        """conv.py:32-38"""
        return [-(-self.out_shape[0] // int(tile_size[0])), -(-self.out_shape[1] // int(tile_size[1]))]


class _CountAhead:
    """Output-row counts of a strided layer on their way (RuleBook.count_ahead)."""

    __slots__ = ("geometry", "z_idx", "z_ptr", "native")

    def __init__(self, geometry, z_idx, z_ptr):
        self.geometry, self.z_idx, self.z_ptr = geometry, z_idx, z_ptr
        self.native = L.host().OutCoords(z_idx, z_ptr, geometry.native)


# Scratch books of one-launch calls that keep no book (the kernel still wants one for tiles with more groups than
# its LDS holds): one per thread, device, stream and kernel volume, grown on demand.  Calls on one stream run one after
# the other, so they can share its memory; calls on different streams get different ones.  Two threads may use one
# stream, and a call writes its row count and its kind into the book before it launches: each thread has its own.
_SCRATCH_BOOKS = threading.local()


def _scratch_book(rows: int, kv: int, device) -> "_Buffers":
    stream = L.stream(device)
    if stream and L.capturing():            # the graph's own, for as long as it needs it
        return _Buffers(rows, kv, device)
    books = getattr(_SCRATCH_BOOKS, "books", None)
    if books is None:
        books = _SCRATCH_BOOKS.books = {}
    key = (device.index, stream, kv)
    buf = books.get(key)
    if buf is None or buf.capacity < rows:
        if len(books) >= 64:
            books.clear()
        buf = _Buffers(max(rows, 1 << 17), kv, device)
        buf.capacity = buf.rows
        books[key] = buf
    buf.native.rows = rows
    return buf


def _row_cols_ptr(row_cols, rows: int):
    """Device pointer of a table of the rows' columns, or None when there is none (or it does not fit)."""
    if row_cols is None or not row_cols.is_cuda or row_cols.dtype != torch.int32 or not row_cols.is_contiguous() \
            or row_cols.dim() != 1 or row_cols.shape[0] != rows:
        return None
    return row_cols.data_ptr()


def row_columns(z_ptr: torch.Tensor, rows: int) -> torch.Tensor:
    """int32 [rows]: the column (index into the flattened ``z_ptr``) of every row."""
    out = torch.empty(int(rows), dtype=torch.int32, device=z_ptr.device)
    with L.on_device(z_ptr.device):
        L.check(L.lib().sph_row_columns(L.ptr(z_ptr), z_ptr.numel(), int(rows), L.ptr(out), L.stream()))
    return out


def _check_index_tensors(z_idx, z_ptr, want):
    """``want`` = (B, S0, S1)."""
    if z_idx.dtype != torch.int32 or z_ptr.dtype != torch.int32:
        raise L.SphconvError("z_idx and z_ptr must be int32")
    if z_idx.dim() != 1:
        raise L.SphconvError("z_idx must be [NNZ]")
    if z_ptr.shape != want:
        raise L.SphconvError("z_ptr must be [B,S0,S1] = %s, got %s" % (want, tuple(z_ptr.shape)))
    if not (z_idx.is_contiguous() and z_ptr.is_contiguous()):
        raise L.SphconvError("z_idx and z_ptr must be contiguous")
    if not (z_idx.is_cuda and z_ptr.is_cuda):
        raise L.SphconvError("z_idx and z_ptr must be GPU tensors")
