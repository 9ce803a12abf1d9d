"""What the framework is timed on: the work that a program built on it has it do, through its public entry points.

A case is a dict of plain values.  ``listed()`` names the ones that are always timed, ``draw(rng)`` makes further ones of
the same ranges, ``prepare`` builds what a program has in hand before the call, ``run`` is one pass, ``work`` the bytes
and operations a pass cannot do without, ``tolerance`` how far two correct implementations may lie apart.

Kinds of cases (``"kind"``):

layer     one convolution module on a tensor whose rules are not cached, without gradients (rules + forward): a layer of
          a network at inference, submanifold (stride 1) or strided.
train     the same module with gradients: forward, then the gradients of the features and of the weight.
int8      the rule book and the integer convolution with per-channel requantisation: a quantised layer.
stream    one scan of a stream of scans handed to ``ScanPipeline`` (rules + forward on its next stream).
encoder   voxels in the order a voxeliser leaves them -> sparse tensor -> the four-stage encoder with BatchNorm and ReLU in
          evaluation mode (12 convolutions, 8 rule books) -> dense tensor for the head behind it.
points    point clouds -> voxels, their means, merged into a batch -> sparse tensor: what stands in front of a network.
"""
import math

import torch

import sphconv_amd as sphconv
from sphconv_amd import sphconv_cuda as ext
from sphconv_amd.datagen import merge_batch_torch
from sphconv_amd.pipeline import ScanPipeline
from sphconv_amd.synth import encoder_stack
from sphconv_amd.vfe import SimpleVoxel
from sphconv_amd.voxelize import VoxelGeneratorV3

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1}
_STACK = (16, 32, 64, 64)          # the encoder's stage widths
_MARGIN = 18                       # columns of a row that a scene leaves free for its turns
_POINT_RANGE, _SPHERE_RANGE = [6, -40, -3, 70.4, 40, 1], [6, -45, 87.5, 70.4, 45, 100]


def _layer(name, kind, batch, grid, gen, p, ic, oc, dtype, kernel=(3, 3, 3), stride=(1, 1, 1)):
    """``grid``: rows x azimuth x depth bins.  ``gen``: "spread" = 1..3 bins anywhere in a column that is occupied with
    probability p, "surface" = 1..2 bins around a smooth range profile, as the surfaces a scan meets leave them."""
    c = {"kind": kind, "batch": batch, "s0": grid[0], "s1": grid[1], "s2": grid[2], "gen": gen, "p": p, "ic": ic, "oc": oc,
         "dtype": dtype, "k0": kernel[0], "k1": kernel[1], "k2": kernel[2], "t0": stride[0], "t1": stride[1], "t2": stride[2]}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a narrow crop of one scan (about 1.2 k voxels) in front of a first layer that takes the four point features:
        # the smallest call, all latency
        _layer("layer_crop_f32_4_16", "layer", 1, (16, 64, 32), "spread", 0.6, 4, 16, "f32"),
        # one scan of 39 k voxels through a narrow fp32 layer
        _layer("layer_scan_f32_16_16", "layer", 1, (64, 512, 32), "spread", 0.6, 16, 16, "f32"),
        # the benchmark's layer and scan size (about 120 k voxels), a stream of scans with its results left on their streams
        _layer("stream_scan_f16_64_64", "stream", 1, (64, 2048, 64), "surface", 0.629, 64, 64, "f16"),
        # eight such scans as one batch: the largest forward pass (760 k voxels)
        _layer("layer_scans8_bf16_64_64", "layer", 8, (64, 2048, 64), "surface", 0.5, 64, 64, "bf16"),
        # a downsampling layer on a batch of four scans: 630 k voxels in, 1.65 M out
        _layer("strided_scans4_f16_32_64", "layer", 4, (64, 2048, 64), "spread", 0.6, 32, 64, "f16", stride=(2, 2, 2)),
        # a quantised layer on a batch of eight
        _layer("int8_scans8_64_64", "int8", 8, (64, 512, 32), "spread", 0.6, 64, 64, "i8"),
        # a training step of a layer in mixed precision: fp16 features, fp32 master weight
        _layer("train_scans8_f16_64_64", "train", 8, (64, 512, 32), "spread", 0.6, 64, 64, "f16"),
        # the same in fp32 at a downsampling layer, on the fine spherical grid (512 depth bins)
        _layer("train_strided_scans8_f32_64_64", "train", 8, (64, 512, 512), "surface", 0.31, 64, 64, "f32", stride=(2, 2, 2)),
        # sizes that fit nothing: odd grid, 24 -> 40 channels, one axis left at full resolution
        _layer("train_ragged_bf16_24_40", "train", 3, (47, 1021, 45), "spread", 0.6, 24, 40, "bf16", stride=(1, 2, 2)),
        # a whole network pass for one scan (latency) and for a batch of four
        {"name": "encoder_scan_bf16", "kind": "encoder", "batch": 1, "s0": 64, "s1": 2048, "s2": 64, "gen": "surface",
         "p": 0.5, "dtype": "bf16"},
        {"name": "encoder_scans4_f16", "kind": "encoder", "batch": 4, "s0": 64, "s1": 2048, "s2": 64, "gen": "spread",
         "p": 0.6, "dtype": "f16"},
        # one sweep of 123 k points to the tensor a network takes
        {"name": "points_scan", "kind": "points", "batch": 1, "points": 122880, "max_points": 2, "max_voxels": 24000,
         "s0": 64, "s1": 512, "s2": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_CHANNELS = [(4, 16), (5, 16), (16, 16), (16, 32), (20, 36), (24, 40), (32, 32), (32, 64), (48, 48), (64, 64), (64, 128)]


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "train", "train", "train", "stream", "int8", "encoder", "points"])
    if kind == "points":
        return {"kind": kind, "batch": rng.randint(1, 3), "points": _log_int(rng, 5000, 150000), "max_points": rng.randint(1, 5),
                "max_voxels": rng.choice([12000, 20000, 24000, 30000]), "s0": rng.choice([32, 64]), "s1": 512, "s2": 512}
    gen = rng.choice(["spread", "surface"])
    p = round(rng.uniform(0.3, 0.7), 3)
    if kind == "encoder":
        return {"kind": kind, "batch": rng.randint(1, 3), "s0": rng.randint(32, 64), "s1": _log_int(rng, 256, 2048),
                "s2": rng.randint(32, 64), "gen": gen, "p": p, "dtype": rng.choice(["f16", "bf16"])}
    while True:
        grid = (_log_int(rng, 8, 64), _log_int(rng, 64, 2048), _log_int(rng, 16, 64) if rng.random() < 0.8 else 512)
        batch = 1 if kind == "stream" else rng.randint(1, 8)
        ic, oc = rng.choice(_CHANNELS)
        kernel, stride = (3, 3, 3), (1, 1, 1)
        if kind in ("layer", "train"):
            kernel = rng.choice([(3, 3, 3)] * 6 + [(3, 3, 1), (1, 3, 3), (3, 1, 1)])
            if rng.random() < 0.5:
                stride = rng.choice([(2, 2, 2), (2, 2, 2), (1, 2, 2), (2, 1, 1)])
        if kind == "stream":
            ic = oc = rng.choice([16, 32, 64])
        if kind == "int8":
            ic, oc = rng.choice([(16, 16), (32, 32), (32, 64), (64, 64)])
        dtype = "i8" if kind == "int8" else rng.choice(["f16", "bf16"] if kind == "stream" else ["f32", "f16", "bf16"])
        # voxels on the larger side, times channels: at most what the largest listed case of the kind holds
        rows = batch * grid[0] * grid[1] * p * 2 * (1 if stride == (1, 1, 1) else 2.6)
        most = {"layer": 760e3, "train": 200e3, "stream": 130e3, "int8": 310e3}[kind] * 64 * 64
        # dense grids hold more pairs per voxel than the listed ones
        if rows * ic * oc * (4 if dtype == "f32" else 1) <= most and batch * grid[0] * grid[1] * grid[2] <= 1.2e8 and rows >= 500:
            return _layer(None, kind, batch, grid, gen, p, ic, oc, dtype, kernel, stride)


# ---- inputs -------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _scene(case):
    """Flat cell numbers of the active voxels of a case's scene, ascending (int64), in all columns but the last _MARGIN of
    a row of the range image."""
    g = _generator(1)
    B, S0, S1, S2 = case["batch"], case["s0"], case["s1"], case["s2"]
    ncol = B * S0 * S1
    dev = "cuda"
    at = torch.arange(ncol, device=dev)
    col = (torch.rand(ncol, generator=g, device=dev) < case["p"]) & (at % S1 < S1 - _MARGIN)
    parts = []
    if case["gen"] == "spread":
        cnt = torch.randint(1, 4, (ncol,), generator=g, device=dev).clamp_(max=S2)
        b1 = torch.randint(0, S2, (ncol,), generator=g, device=dev)
        b2 = torch.randint(0, max(S2 - 1, 1), (ncol,), generator=g, device=dev)
        b2 = b2 + (b2 >= b1).long()
        lo, hi = torch.minimum(b1, b2), torch.maximum(b1, b2)
        b3 = torch.randint(0, max(S2 - 2, 1), (ncol,), generator=g, device=dev)
        b3 = b3 + (b3 >= lo).long()
        b3 = b3 + (b3 >= hi).long()
        bins = (b1, b2, b3)
    else:
        cnt = torch.randint(1, 3, (ncol,), generator=g, device=dev)
        scale = S2 / 64.0
        prof = (40.0 + 15.0 * torch.sin((at % S1).float() * (2.0 * math.pi / S1))) * scale
        bins = [torch.round(prof + 3.0 * scale * torch.randn(ncol, generator=g, device=dev)).clamp_(0, S2 - 1).long()
                for _ in range(2)]
    for j, b in enumerate(bins):
        use = col & (cnt > j)
        parts.append(at[use] * S2 + b[use])
    return torch.unique(torch.cat(parts))


def _cells(case, g):
    """The scene as one pass meets it: its samples in an order of ``g``'s, turned by an even number of columns.  (The sizes of
    outputs are then a property of the case; a stride of 2 splits the turned scene as it splits the scene itself.)"""
    cells = _scene(case)
    B, S2, per = case["batch"], case["s2"], case["s0"] * case["s1"] * case["s2"]
    order = torch.randperm(B, generator=g, device="cuda")
    turn = 2 * int(torch.randint(1, _MARGIN // 2, (1,), generator=g, device="cuda"))
    return torch.sort(order[cells // per] * per + cells % per + turn * S2)[0]


def _compressed(case, cells):
    B, S0, S1, S2 = case["batch"], case["s0"], case["s1"], case["s2"]
    counts = torch.bincount(cells // S2, minlength=B * S0 * S1)
    z_ptr = torch.cumsum(counts, 0).to(torch.int32).view(B, S0, S1).contiguous()
    return (cells % S2).to(torch.int32).contiguous(), z_ptr


def _coo(case, cells):
    S0, S1, S2 = case["s0"], case["s1"], case["s2"]
    return torch.stack([cells // (S0 * S1 * S2), cells // (S1 * S2) % S0, cells // S2 % S1, cells % S2], 1).to(torch.int32)


def _sweep(case, g, sample):
    """x, y, z, reflectance of one sweep of the front sector, as the beams deliver it: 64 beams, surfaces of a smooth range
    profile, some clutter.  ``g`` gives the direction at which the sensor begins its turn, and the reflectances."""
    m, fixed = case["points"], _generator(1 + sample)
    u = lambda: torch.rand(m, generator=fixed, device="cuda", dtype=torch.float64)
    beam = torch.floor(u() * 64)
    theta = torch.deg2rad(87.5 + (beam + 0.5 + 0.1 * (u() - 0.5)) * (15.9 / 64))
    azimuth = torch.sort(-45.0 + 90.0 * u())[0]
    phi = torch.deg2rad(azimuth)
    r = 30.0 + 18.0 * torch.sin(azimuth * 0.21) + 0.1 * beam
    r = r + 0.4 * torch.randn(m, generator=fixed, device="cuda", dtype=torch.float64)
    r = torch.where(u() < 0.2, 6.0 + 64.0 * u(), r).clamp(5.0, 72.0)
    xyz = [r * torch.sin(theta) * torch.cos(phi), r * torch.sin(theta) * torch.sin(phi), r * torch.cos(theta)]
    refl = torch.rand(m, generator=g, device="cuda", dtype=torch.float64)
    begin = int(torch.randint(0, m, (1,), generator=g, device="cuda"))
    return torch.roll(torch.stack(xyz + [refl], 1), begin, 0).float().contiguous()


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "points":
        shape = [case["s0"], case["s1"], case["s2"]]
        gen = VoxelGeneratorV3(None, _POINT_RANGE, _SPHERE_RANGE, case["max_points"], case["max_voxels"], shape[::-1],
                               coord_system="spherical")
        return {"kind": kind, "scans": [_sweep(case, g, i) for i in range(case["batch"])], "generator": gen, "vfe": SimpleVoxel(4),
                "shape": shape, "batch": case["batch"]}
    shape, batch, dtype = [case["s0"], case["s1"], case["s2"]], case["batch"], _DTYPES[case["dtype"]]
    cells = _cells(case, g)
    n = cells.numel()
    if kind == "encoder":
        net = encoder_stack(16, _STACK, seed=int(seed)).to("cuda").to(dtype)
        cells = cells[torch.randperm(n, generator=g, device="cuda")]       # the order in which points met the voxels
        return {"kind": kind, "net": net, "indices": _coo(case, cells), "shape": shape, "batch": batch,
                "feature": torch.randn((n, 16), generator=g, device="cuda").to(dtype)}
    z_idx, z_ptr = _compressed(case, cells)
    ic, oc, kernel = case["ic"], case["oc"], (case["k0"], case["k1"], case["k2"])
    stride = (case["t0"], case["t1"], case["t2"])
    kv = kernel[0] * kernel[1] * kernel[2]
    s = {"kind": kind, "z_idx": z_idx, "z_ptr": z_ptr, "shape": shape, "batch": batch}
    if kind == "int8":
        s["feature"] = torch.randint(-20, 20, (n, ic), generator=g, device="cuda", dtype=torch.int8)
        s["weight"] = torch.randint(-20, 20, (kv, ic, oc), generator=g, device="cuda", dtype=torch.int8)
        s["scale"] = 0.005 + 0.01 * torch.rand(oc, generator=g, device="cuda")
        s["kernel"] = list(kernel)
        return s
    s["feature"] = torch.randn((n, ic), generator=g, device="cuda").to(dtype)
    weight = torch.randn((kv, ic, oc), generator=g, device="cuda") * (2.0 / (kv * ic)) ** 0.5
    # the tensor comes from init_tensor or from a layer before: it knows its rows' columns
    s["row_cols"] = sphconv.SparseConvTensor(s["feature"], shape, batch, z_idx=z_idx, z_ptr=z_ptr).with_row_cols().row_cols
    if kind == "stream":
        s["pipeline"] = ScanPipeline(weight.to(dtype), batch, shape, kernel)
        return s
    pad = tuple(k // 2 for k in kernel)
    if stride == (1, 1, 1):
        conv = sphconv.SubMConv3d(ic, oc, kernel)
    else:
        conv = sphconv.SparseConv3d(ic, oc, kernel, stride=stride, padding=pad)
    conv = conv.to("cuda")
    with torch.no_grad():
        conv.weight.copy_(weight.view(conv.weight.shape))
    if kind == "layer":
        s["conv"] = conv.to(dtype).eval()
        return s
    s["conv"] = conv                                                       # fp32 master weight whatever the features are
    s["feature"].requires_grad_(True)
    if stride == (1, 1, 1):
        rows = n
    else:
        occ = torch.zeros(batch * shape[0] * shape[1] * shape[2], dtype=torch.bool, device="cuda")
        occ[cells] = True
        rows = int(_reach(occ.view(batch, *shape), kernel, stride, pad)[1].sum())
    s["d_out"] = torch.randn((rows, oc), generator=g, device="cuda").to(dtype)
    return s


# ---- one pass -----------------------------------------------------------------------------------

def run(state):
    s = state
    kind = s["kind"]
    if kind == "stream":
        # the scan's arrays are complete; its output stays on the pipeline's stream
        out, _slot = s["pipeline"].submit(s["feature"], s["z_idx"], s["z_ptr"], wait_inputs=False, row_cols=s["row_cols"])
        return out
    if kind == "int8":
        book = ext.get_rulebook_subm(s["z_idx"], s["z_ptr"], s["batch"], s["shape"], s["shape"], s["kernel"], [1, 1, 1],
                                     [k // 2 for k in s["kernel"]], [1, 1, 1])
        return ext.rule_conv_int8(s["feature"], s["weight"], s["scale"], book, None, s["feature"].shape[0])
    if kind == "points":
        examples = []
        for points in s["scans"]:
            res = s["generator"].generate(points)
            voxels = s["vfe"](res["voxels"], res["num_points_per_voxel"], res["coordinates"])
            examples.append({"voxels": voxels, "coordinates": res["coordinates"]})
        ex = merge_batch_torch(examples)
        x = sphconv.SparseConvTensor(ex["voxels"], s["shape"], s["batch"], indices=ex["coordinates"])
        return {"voxels": ex["voxels"], "coordinates": ex["coordinates"], "feature": x.feature, "z_idx": x.z_idx, "z_ptr": x.z_ptr}
    if kind == "encoder":
        with torch.no_grad():
            return s["net"](sphconv.SparseConvTensor(s["feature"], s["shape"], s["batch"], indices=s["indices"])).dense()
    x = sphconv.SparseConvTensor(s["feature"], s["shape"], s["batch"], z_idx=s["z_idx"], z_ptr=s["z_ptr"], row_cols=s["row_cols"])
    if kind == "layer":
        with torch.no_grad():
            y = s["conv"](x)
        return {"feature": y.feature, "z_idx": y.z_idx, "z_ptr": y.z_ptr}
    y = s["conv"](x)
    d_feature, d_weight = torch.autograd.grad(y.feature, (s["feature"], s["conv"].weight), s["d_out"])
    return {"feature": y.feature.detach(), "z_idx": y.z_idx, "z_ptr": y.z_ptr, "d_feature": d_feature, "d_weight": d_weight}


# ---- what a pass cannot do without --------------------------------------------------------------

def _reach(occ, kernel, stride, pad):
    """(pairs, occupancy of the output grid) of a convolution on the occupancy ``occ`` [B,S0,S1,S2]."""
    shape = occ.shape[1:]
    out = [(s + 2 * p - k) // t + 1 for s, k, t, p in zip(shape, kernel, stride, pad)]
    padded = torch.nn.functional.pad(occ, (pad[2], pad[2], pad[1], pad[1], pad[0], pad[0]))
    views = [padded[:, a:a + (out[0] - 1) * stride[0] + 1:stride[0], b:b + (out[1] - 1) * stride[1] + 1:stride[1],
                    c:c + (out[2] - 1) * stride[2] + 1:stride[2]]
             for a in range(kernel[0]) for b in range(kernel[1]) for c in range(kernel[2])]
    reached = torch.zeros_like(views[0])
    pairs = 0
    for v in views:
        reached |= v
        pairs += v.sum()
    return int(pairs), reached


def _subm_pairs(occ, kernel):
    pad = [k // 2 for k in kernel]
    shape = occ.shape[1:]
    padded = torch.nn.functional.pad(occ, (pad[2], pad[2], pad[1], pad[1], pad[0], pad[0]))
    return int(sum((occ & padded[:, a:a + shape[0], b:b + shape[1], c:c + shape[2]]).sum()
                   for a in range(kernel[0]) for b in range(kernel[1]) for c in range(kernel[2])))


def work(case):
    """Bytes: every array a pass is given and every one it hands on, once each (between the
    encoder's layers too: the rows do not fit the chip); pairs need not leave it.  Operations: two for each product."""
    kind = case["kind"]
    if kind == "points":
        m, cells = case["batch"] * case["points"], case["batch"] * case["s0"] * case["s1"]
        v = min(case["batch"] * case["max_voxels"], m)
        return {"bytes": 16 * m + v * (16 * case["max_points"] + 4 * case["max_points"] + 12 + 4 + 2 * 16 + 16 + 4) + 4 * cells, "flops": 0}
    cells = _scene(case)
    n, shape, e = cells.numel(), [case["s0"], case["s1"], case["s2"]], _BYTES[case["dtype"]]
    occ = torch.zeros(case["batch"] * shape[0] * shape[1] * shape[2], dtype=torch.bool, device="cuda")
    occ[cells] = True
    occ = occ.view(case["batch"], *shape)
    columns = case["batch"] * shape[0] * shape[1]
    if kind == "encoder":
        nbytes, flops, c_in = n * (16 + 16 * e), 0, 16
        for c in _STACK:
            pairs = _subm_pairs(occ, (3, 3, 3))
            cols = occ.shape[0] * occ.shape[1] * occ.shape[2]
            nbytes += 4 * cols + 4 * n + n * e * (c_in + 3 * c) + 27 * e * (c_in * c + c * c)
            flops += 2 * pairs * (c_in * c + c * c)
            pairs, occ = _reach(occ, (3, 3, 3), (2, 2, 2), (1, 1, 1))
            m = int(occ.sum())
            nbytes += n * e * c + m * e * c + 27 * e * c * c + 4 * m
            flops += 2 * pairs * c * c
            n, c_in = m, c
        nbytes += n * c_in * e + occ.numel() * c_in * e                    # the last rows in, the dense tensor out
        return {"bytes": nbytes, "flops": flops}
    ic, oc, kernel = case["ic"], case["oc"], (case["k0"], case["k1"], case["k2"])
    stride = (case["t0"], case["t1"], case["t2"])
    kv = kernel[0] * kernel[1] * kernel[2]
    index = 8 * n + 4 * columns                                            # z_idx, the rows' columns, z_ptr
    if stride == (1, 1, 1):
        pairs, m = _subm_pairs(occ, kernel), n
    else:
        pairs, out = _reach(occ, kernel, stride, [k // 2 for k in kernel])
        m = int(out.sum())
        index += 4 * m + 4 * out.shape[0] * out.shape[1] * out.shape[2]    # oz_idx, oz_ptr
    if kind != "train":
        return {"bytes": index + n * ic * e + m * oc * e + kv * ic * oc * e, "flops": 2 * pairs * ic * oc}
    # features and the gradient of the output in, output and the gradient of the features out; fp32 weight and its gradient
    return {"bytes": index + 2 * n * ic * e + 2 * m * oc * e + 8 * kv * ic * oc, "flops": 6 * pairs * ic * oc}


def tolerance(case):
    kind = case["kind"]
    if kind == "int8":
        return "exact"
    if kind == "points":
        # means of a few fp32 values; a point on the very edge of a bin may fall to either side
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    # one rounding of fp32 sums to the storage type; a dozen in a row for the encoder
    rel = {"f16": 1e-3, "bf16": 8e-3}[case["dtype"]]
    return {"rel": min(2.5 * rel, 0.02) if kind == "encoder" else rel, "max": 0.2 if kind == "encoder" else 20 * rel}
