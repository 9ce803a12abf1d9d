"""Containers (reference: sphconv/modules.py:36-132)."""
import contextlib
import sys
from collections import OrderedDict

import torch
from torch import nn

from . import _lib as L


_NO_RANGE = contextlib.nullcontext()


class SphModule(nn.Module):
    """Marker base class: modules derived from it receive the SparseConvTensor
    itself inside :class:`Sequential`; any other module receives ``.feature``."""

    is_convolution = False


def is_sph_module(module) -> bool:
    return isinstance(module, SphModule)


def is_sparse_conv(module) -> bool:
    return isinstance(module, SphModule) and module.is_convolution


def _keeps_on(t: torch.Tensor):
    """The stream that what is kept now belongs to (None for tensors on the host), or False where nothing may be kept: a
    graph under capture computes everything itself."""
    if not t.is_cuda:
        return None
    stream = L.stream(t.device)
    return False if stream and L.capturing() else stream


def _bn_affine(bn: nn.BatchNorm1d, stream):
    """Evaluation-mode BatchNorm1d as y = x*scale + shift (fp32 [C]); computed once per state of the module's tensors and
    kept on the module, for the stream it was computed on (``_keeps_on``).  The state is the tensors themselves, which the entry holds (an
    address alone is handed out again once its tensor is gone), with their storage and version counter."""
    # (straight from the module's tables: asking the module four times takes longer than the key)
    p, b = bn._parameters, bn._buffers
    if stream is False:
        return _bn_affine_now(bn)
    try:
        mean, var, weight, bias = b["running_mean"], b["running_var"], p["weight"], p["bias"]
        # a pass in training mode changes the running statistics behind their version counters' back, and counts itself here
        passes = b["num_batches_tracked"]
    except KeyError:
        # a tensor that is not in its table is computed, or a replica's: another one on each pass, nothing to keep
        return _bn_affine_now(bn)
    if passes is None:
        return _bn_affine_now(bn)
    state = [bn.eps, passes._version, mean.data_ptr(), mean._version, mean.dtype, var.data_ptr(), var._version, var.dtype]
    if weight is not None:
        state += (weight.data_ptr(), weight._version, weight.dtype)
    if bias is not None:
        state += (bias.data_ptr(), bias._version, bias.dtype)
    kept = bn.__dict__.get("_sph_affines")
    if kept is None:
        kept = bn.__dict__["_sph_affines"] = {}
    hit = kept.get(stream)
    if hit is not None and hit[0] is mean and hit[1] is var and hit[2] is weight and hit[3] is bias and hit[4] is passes \
            and hit[5] == state:
        return hit[6], hit[7]
    scale, shift = _bn_affine_now(bn)
    if len(kept) >= 16:
        kept.clear()
    kept[stream] = (mean, var, weight, bias, passes, state, scale, shift)
    return scale, shift


def _bn_affine_now(bn: nn.BatchNorm1d):
    var = bn.running_var.float()
    scale = torch.rsqrt(var + bn.eps)
    if bn.weight is not None:
        scale = scale * bn.weight.float()
    shift = -bn.running_mean.float() * scale
    if bn.bias is not None:
        shift = shift + bn.bias.float()
    return scale.contiguous(), shift.contiguous()


class Sequential(SphModule):
    """Sequential container over sparse-conv and ordinary modules
    (modules.py:43-128).  Accepts positional modules, one OrderedDict, or keyword
    modules.

    With gradients disabled, a convolution followed by an evaluation-mode
    ``BatchNorm1d`` and/or a ``ReLU`` runs as one kernel: the affine map and the
    clamp are applied to the fp32 accumulators before the store (no reference
    counterpart: modules.py:124-125 runs them as separate passes over ``.feature``).
    ``fuse_eval = False`` switches this off."""

    fuse_eval = True
    # A strided convolution needs its output row count on the host before its rules can be generated.  The
    # container starts that count as soon as the layer's input coordinates exist -- at the container's input,
    # or behind the strided layer before it, submanifold layers in between change no coordinates -- so that
    # the host reads it while the convolutions in between keep the GPU busy (no reference counterpart:
    # rules.cu:461 waits where the layer runs).  False counts where the layer runs.
    count_ahead = True

    def __init__(self, *args, **kwargs):
        super().__init__()
        if len(args) == 1 and isinstance(args[0], OrderedDict):
            for key, module in args[0].items():
                self.add_module(key, module)
        else:
            for idx, module in enumerate(args):
                self.add_module(str(idx), module)
        for name, module in kwargs.items():
            if name in self._modules:
                raise ValueError("name exists.")
            self.add_module(name, module)

    def __getitem__(self, idx):
        if not (-len(self) <= idx < len(self)):
            raise IndexError("index {} is out of range".format(idx))
        if idx < 0:
            idx += len(self)
        return list(self._modules.values())[idx]

    def __len__(self):
        return len(self._modules)

    def add(self, module, name=None):
        if name is None:
            name = str(len(self._modules))
            if name in self._modules:
                raise KeyError("name exists")
        self.add_module(name, module)

    def _fusable_tail(self, mods, i):
        """(number of modules after mods[i] that fold into its store, BatchNorm1d or None, relu).  A module with hooks
        does not: a hook sees every call (pruning computes its weight in one)."""
        conv = mods[i]
        if not (self.fuse_eval and is_sparse_conv(conv)) or torch.is_grad_enabled():
            return 0, None, False
        weight = conv._parameters.get("weight")
        if (conv.weight if weight is None else weight).dtype not in (torch.float16, torch.bfloat16, torch.float32):
            return 0, None, False
        n, bn, relu = 0, None, False
        nxt = mods[i + 1] if i + 1 < len(mods) else None
        if (type(nxt) is nn.BatchNorm1d and not nxt.training
                and (nxt._buffers.get("running_mean") is not None or nxt.running_mean is not None)
                and nxt.num_features == conv.out_channels and not nxt._forward_pre_hooks and not nxt._forward_hooks):
            bn, n = nxt, 1
            nxt = mods[i + 2] if i + 2 < len(mods) else None
        if type(nxt) is nn.ReLU and not nxt._forward_pre_hooks and not nxt._forward_hooks:
            relu, n = True, n + 1
        return n, bn, relu

    def forward(self, input):
        from .tensor import SparseConvTensor
        mods = list(self._modules.items())
        only = [m for _, m in mods]
        conv = [is_sparse_conv(m) for m in only]
        profiling = torch.autograd._profiler_enabled()
        skip, keeps_on = 0, None
        ahead = {}      # index of a strided convolution -> its count on the way

        def start_count(first):
            """The next strided convolution at or behind module `first` that sees `input`'s coordinates."""
            if not (self.count_ahead and isinstance(input, SparseConvTensor)):
                return
            for j in range(first, len(only)):
                m = only[j]
                if conv[j] and not m.subm:
                    if hasattr(m, "count_ahead"):
                        h = m.count_ahead(input)
                        if h is not None:
                            ahead[j] = h
                    return
                if not conv[j] and is_sph_module(m):
                    return          # a module that may change the coordinates

        start_count(0)
        for i, (name, module) in enumerate(mods):
            if skip:
                skip -= 1
                continue
            if is_sph_module(module):
                assert isinstance(input, SparseConvTensor)
                # a range costs 5 us of host time per module: only for a profiler that is there to see it
                with (torch.autograd.profiler.record_function("sphconv:{}:{}".format(type(module).__name__, name))
                      if profiling else _NO_RANGE):
                    skip, bn, relu = self._fusable_tail(only, i)
                    kw = {"ahead": ahead.pop(i)} if i in ahead else {}
                    if skip:
                        scale = shift = None
                        if bn is not None:
                            if keeps_on is None:
                                keeps_on = _keeps_on(input.feature)
                            scale, shift = _bn_affine(bn, keeps_on)
                        input = module(input, epilogue=(scale, shift, relu), **kw)
                    else:
                        input = module(input, **kw)
                    if conv[i] and not module.subm:
                        start_count(i + 1)      # new coordinates: the next strided layer can start counting
            elif isinstance(input, SparseConvTensor):
                module.__dict__.pop("_sph_affines", None)       # run on its own, as while it is trained
                input.feature = module(input.feature)
            else:
                input = module(input)
        return input


SparseSequential = Sequential
