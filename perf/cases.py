"""The calls whose time counts, over the sizes and types a program uses.

A case is a dict of plain values.  ``net`` is a chain of layers, one token per
layer, "kind c_in c_out kernel [stride padding] [key]":

    m  SubMConv3d           "m 16 32 3 a"
    d  SparseConv3d         "d 32 64 3 2 1 b"  (stride and padding after the kernel)
    u  SparseInverseConv3d  "u 64 32 3 b"      (undoes the d of the same key)

``op`` says what one pass is:

    kept   the chain on a tensor whose pairs are in hand: every layer of a
           stage after its first, every step of a sampler on one set of voxels
    frame  the chain on coordinates it has not seen, as every new scan is: a
           new SparseConvTensor, its pair builds and its convolutions
    dense  frame, then the dense volume a 2D head reads
    pairs  the pair lists and coordinates of the three builds themselves

``pre`` (kept) is a chain that runs before, in prepare: the strided layers
whose pairs the inverse layers of ``net`` undo.
"""
from __future__ import annotations

import functools
import math

import torch
import torch.nn as nn

import trispconv.pytorch as spconv
from trispconv_amd.pytorch.indices import (generate_inverse_indice_pairs,
                                           generate_strided_indice_pairs,
                                           generate_subm_indice_pairs)

DEV = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
LIDAR = "41x1600x1408"
# the VoxelNet-style encoder of the benchmark: 11 layers, four resolutions
ENCODER = ("m 4 16 3 a|d 16 32 3 2 1 b|m 32 32 3 c|m 32 32 3 c|d 32 64 3 2 1 e|m 64 64 3 f|"
           "m 64 64 3 f|d 64 64 3 2 1 g|m 64 64 3 h|m 64 64 3 h|d 64 128 3x1x1 2x1x1 0 i")


def _case(name, op, net, dtype, n, grid, batch=1, voxels="surface", bn=False, pre=""):
    c = {"op": op, "net": net, "dtype": dtype, "n": n, "grid": grid, "batch": batch,
         "voxels": voxels, "bn": bn, "pre": pre}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one layer of a small object, all launch latency
        _case("subm16_1k", "kept", "m 16 16 3 a", "f32", 1000, "64x64x64", voxels="uniform"),
        # per-voxel class scores of a segmentation network: 20 classes
        _case("scores20_120k", "kept", "m 96 20 1 a", "f16", 120_000, "192x192x192"),
        # the first layer of a colour point-cloud network: 3 channels, 5x5x5
        _case("stem5_80k", "frame", "m 3 32 5 a", "f16", 80_011, "160x160x160", bn=True),
        # the first stage of a LiDAR network on one scan: 5 values per point
        _case("lidar_first_60k", "frame", "m 5 16 3 a|m 16 16 3 a", "f16", 60_013, LIDAR,
              bn=True),
        # an ordinary layer inside a stage, in the default precision
        _case("subm64_f32_100k", "kept", "m 64 64 3 a", "f32", 100_000, "160x160x160"),
        # the benchmark's 128-channel layer, pairs in hand
        _case("subm128_500k", "kept", "m 128 128 3 a", "f16", 500_000, "256x256x256"),
        # a whole stage on a new scene of that size: build, order, two layers
        _case("stage128_500k", "frame", "m 128 128 3 a|m 128 128 3 a", "f16", 500_000,
              "256x256x256", bn=True),
        # a downsampling layer on a new LiDAR scan pair, in fp32
        _case("down64_2x200k", "frame", "d 64 64 3 2 1 a", "f32", 400_000, LIDAR, batch=2),
        # down and up again on clustered voxels
        _case("down_up_4x150k", "frame", "d 32 64 3 2 1 a|u 64 32 3 a", "bf16", 600_000,
              "512x512x64", batch=4, voxels="blob"),
        # a detector's whole 3D part on new scans, to its dense volume
        _case("encoder_4x60k", "dense", ENCODER, "f16", 240_000, LIDAR, batch=4, bn=True),
        # a decoder's wide upsampling block on one set of voxels, step after step
        _case("up768_30k", "kept", "u 768 192 3 a|m 192 192 3", "f16", 30_000, "64x64x64",
              pre="d 192 768 3 2 1 a"),
        # the pair lists themselves (submanifold, strided, inverse)
        _case("pairs_100k", "pairs", "", "f32", 100_003, "160x160x160"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cube(rng, n, voxels):
    """A grid of the density that scenes of n voxels have."""
    if voxels == "uniform":
        e = (n * rng.uniform(20, 120)) ** (1 / 3)
    else:
        e = math.sqrt(n / rng.uniform(3, 8))
    e = max(24, int(math.ceil(e)))
    return "%dx%dx%d" % (e, e + rng.randrange(5), e + rng.randrange(9))


def draw(rng):
    family = rng.choice(["layer", "layer", "layer", "stage", "stage", "first", "down", "down_up",
                         "encoder", "up", "pairs"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    bn = rng.random() < 0.5
    if family == "layer":
        n, voxels = _log(rng, 500, 250_000), rng.choice(["surface", "surface", "uniform"])
        c_in = rng.choice([4, 8, 16, 20, 32, 48, 64, 96, 128])
        c_out = rng.choice([3, 16, 20, 32, 40, 64, 96, 128])
        k = rng.choice([1, 3, 3, 3, 3, 5]) if c_in * c_out <= 1024 else rng.choice([1, 3, 3, 3])
        return _case("", "kept", "m %d %d %d a" % (c_in, c_out, k), dtype, n,
                     _cube(rng, n, voxels), voxels=voxels, bn=bn)
    if family == "stage":
        n, c = _log(rng, 2000, 250_000), rng.choice([16, 32, 48, 64, 96, 128])
        net = "|".join(["m %d %d 3 a" % (c, c)] * rng.choice([1, 2, 2, 3]))
        return _case("", "frame", net, dtype, n, _cube(rng, n, "surface"), bn=bn)
    if family == "first":
        c_in, c = rng.choice([1, 3, 4, 5, 6, 7, 9]), rng.choice([16, 24, 32])
        if rng.random() < 0.4:
            n = _log(rng, 2000, 120_000)
            return _case("", "frame", "m %d %d 5 a" % (c_in, c), dtype, n,
                         _cube(rng, n, "surface"), bn=bn)
        n = _log(rng, 5000, 200_000)
        return _case("", "frame", "m %d %d 3 a|m %d %d 3 a" % (c_in, c, c, c), dtype, n, LIDAR,
                     batch=rng.choice([1, 2]), bn=bn)
    if family == "down":
        n, c_in = _log(rng, 5000, 400_000), rng.choice([16, 32, 64])
        k = rng.choice(["3 2 1", "2 2 0", "3x1x1 2x1x1 0"])
        return _case("", "frame", "d %d %d %s a" % (c_in, rng.choice([c_in, 2 * c_in]), k), dtype,
                     n, LIDAR, batch=rng.choice([1, 2, 4]), bn=bn)
    if family == "down_up":
        n, c = _log(rng, 4000, 400_000), rng.choice([16, 32, 64])
        k = rng.choice(["3 2 1", "2 2 0"])
        return _case("", "frame", "d %d %d %s a|u %d %d %s a" % (c, 2 * c, k, 2 * c, c, k[0]),
                     dtype, n, "512x512x64", batch=rng.choice([1, 2, 4]), voxels="blob", bn=bn)
    if family == "encoder":
        b = rng.choice([1, 2, 4])
        return _case("", "dense", ENCODER, rng.choice(["f16", "bf16", "f32"]),
                     b * _log(rng, 8000, 60_000), LIDAR, batch=b, bn=True)
    if family == "up":
        n, c = _log(rng, 2000, 60_000), rng.choice([96, 192, 256])
        return _case("", "kept", "u %d %d 3 a|m %d %d 3" % (3 * c, c, c, c), dtype, n,
                     _cube(rng, n, "surface"), pre="d %d %d 3 2 1 a" % (c, 3 * c))
    n = _log(rng, 2000, 250_000)
    return _case("", "pairs", "", "f32", n, _cube(rng, n, "surface"))


# ---------------------------------------------------------------- inputs
def _shape(case):
    return tuple(int(v) for v in case["grid"].split("x"))


def _chain(text):
    """The layers of a chain: (kind, c_in, c_out, kernel, stride, padding, key)."""
    to3 = lambda t: (int(t),) * 3 if "x" not in t else tuple(int(v) for v in t.split("x"))  # noqa: E731
    got = []
    for token in filter(None, text.split("|")):
        t = token.split()
        kind, c_in, c_out, k = t[0], int(t[1]), int(t[2]), to3(t[3])
        s, p = (to3(t[4]), to3(t[5])) if kind == "d" else ((1, 1, 1), (0, 0, 0))
        rest = t[6:] if kind == "d" else t[4:]
        got.append((kind, c_in, c_out, k, s, p, rest[0] if rest else None))
    return got


def _patch(g, shape):
    """Cells of one random plane patch or cylinder, sampled at 0.45 cells."""
    D, H, W = shape
    thin, wide = D < 0.2 * min(H, W), min(H, W)
    r = torch.rand(16, generator=g, dtype=torch.float64)
    z = torch.randn(8, generator=g, dtype=torch.float64)
    centre = r[:3] * torch.tensor(shape, dtype=torch.float64)
    plane = float(r[3]) < 0.5
    if plane:  # thin grids: mostly near-horizontal ground, and walls
        axis = torch.stack([z[0] * 4.0, z[1], z[2]]) if thin else z[:3]
    else:      # thin grids: upright poles and trees
        axis = torch.stack([torch.ones((), dtype=torch.float64), z[0] * 0.1, z[1] * 0.1]) \
            if thin else z[:3]
    axis = axis / axis.norm()
    other = torch.zeros(3, dtype=torch.float64)
    other[0 if abs(float(axis[0])) < 0.9 else 1] = 1.0
    u = torch.linalg.cross(axis, other)
    u = u / u.norm()
    v = torch.linalg.cross(axis, u)
    c, axis, u, v = (t.to(DEV) for t in (centre, axis, u, v))
    ar = lambda a, b, s: torch.arange(a, b, s, dtype=torch.float64, device=DEV)  # noqa: E731
    if plane:
        e = float(0.15 + 0.35 * r[4]) * wide
        a = ar(-e / 2, e / 2, 0.45)
        p = c + a[:, None, None] * u + a[None, :, None] * v
    else:
        radius = 3.0 + 0.08 * wide * float(r[4])
        e = float(0.3 + 0.7 * r[5]) * (D if thin else 0.5 * wide)
        th, h = ar(0, 2 * math.pi, 0.45 / radius), ar(-e / 2, e / 2, 0.45)
        ring = radius * (th.cos()[:, None] * u + th.sin()[:, None] * v)
        p = c + ring[:, None, :] + h[None, :, None] * axis
    return p.reshape(-1, 3).floor().long()


def _blob(g, shape):
    centre = torch.rand(3, generator=g, dtype=torch.float64) * torch.tensor(shape, dtype=torch.float64)
    z = torch.randn(4096, 3, generator=g, dtype=torch.float64) * 8.0
    return (centre + z).round().long().to(DEV)


@functools.lru_cache(maxsize=8)
def _scene(shape, B, n, voxels):
    """(cells, room): B scenes' cells, n in all, as (b, z, y, x) in no order.
    Each axis keeps ``room`` cells free at its end, for the scene to move in."""
    D, H, W = shape
    room = [16 * (s // 64) for s in shape]
    size = torch.tensor([s - (r + 2 if r else 0) for s, r in zip(shape, room)], device=DEV)
    g = torch.Generator().manual_seed(((D * 4099 + H) * 4099 + W) * 31 + 7 * n + B)
    parts = []
    for b in range(B):
        want = n // B + (b < n % B)
        keys = torch.empty(0, dtype=torch.long, device=DEV)
        while len(keys) < want:
            batch = [keys]
            for _ in range(2 if voxels == "surface" else 16):
                if voxels == "uniform":
                    p = (torch.rand(max(want // 4, 64), 3, generator=g).to(DEV) * size).long()
                else:
                    p = _patch(g, shape) if voxels == "surface" else _blob(g, shape)
                p = p[((p >= 0) & (p < size)).all(1)]
                batch.append((p[:, 0] * H + p[:, 1]) * W + p[:, 2])
            every = torch.cat(batch)
            uniq, inv = torch.unique(every, return_inverse=True)
            first = torch.full((len(uniq),), len(every), dtype=torch.long, device=DEV)
            first.scatter_reduce_(0, inv, torch.arange(len(every), device=DEV), "amin")
            keys = every[first.sort().values]  # in the order in which they came
        parts.append(b * (D * H * W) + keys[:want])
    keys = torch.cat(parts)
    x, r = keys % W, keys // W
    y, r = r % H, r // H
    return torch.stack([r // D, r % D, y, x], 1).int(), room


def _voxels(case, seed):
    """(n, 4) int32 coordinates (b, z, y, x), none twice: the case's scenes, by
    the seed moved (by whole multiples of every stride, so that each seed has
    as many outputs as the others), dealt to the samples of the batch and put
    in random order."""
    cells, room = _scene(_shape(case), case["batch"], case["n"], case["voxels"])
    g = torch.Generator().manual_seed(seed)
    move = [16 * int(torch.randint(r // 16 + 1, (), generator=g)) for r in room]
    out = cells + torch.tensor([0] + move, dtype=torch.int32, device=DEV)
    out[:, 0] = torch.randperm(case["batch"], generator=g).int().to(DEV)[cells[:, 0].long()]
    return out[torch.randperm(len(out), generator=g).to(DEV)].contiguous()


def _rand(g, shape, bound, dtype):
    t = torch.rand(shape, generator=g, device=DEV, dtype=torch.float32)
    return ((2 * t - 1) * bound).to(dtype)


def _params(case, text, seed):
    """Weight (KRSC), bias and batch-norm statistics of each layer of a chain."""
    dtype = DTYPES[case["dtype"]]
    g = torch.Generator(DEV).manual_seed(seed + 1_000_003)
    got = []
    for _, c_in, c_out, k, _, _, _ in _chain(text):
        bound = math.sqrt(6.0 / (math.prod(k) * c_in))
        p = {"w": _rand(g, (c_out, *k, c_in), bound, dtype), "b": _rand(g, (c_out,), 0.1, dtype)}
        if case["bn"]:
            p["mean"], p["shift"] = _rand(g, (c_out,), 0.2, dtype), _rand(g, (c_out,), 0.2, dtype)
            p["var"] = _rand(g, (c_out,), 0.4, dtype) + 1
            p["scale"] = _rand(g, (c_out,), 0.4, dtype) + 1
        got.append(p)
    return got


def _features(case, rows, channels, seed):
    g = torch.Generator(DEV).manual_seed(seed + 2_000_003)
    t = torch.randn((rows, channels), generator=g, device=DEV, dtype=torch.float32)
    return t.to(DTYPES[case["dtype"]])


def _network(case, text, seed):
    mods = []
    for (kind, c_in, c_out, k, s, p, key), q in zip(_chain(text), _params(case, text, seed)):
        if kind == "m":
            conv = spconv.SubMConv3d(c_in, c_out, k, indice_key=key)
        elif kind == "d":
            conv = spconv.SparseConv3d(c_in, c_out, k, stride=s, padding=p, indice_key=key)
        else:
            conv = spconv.SparseInverseConv3d(c_in, c_out, k, indice_key=key)
        conv = conv.to(DEV).to(DTYPES[case["dtype"]])
        with torch.no_grad():
            conv.weight.copy_(q["w"])
            conv.bias.copy_(q["b"])
        mods.append(conv)
        if case["bn"]:
            norm = nn.BatchNorm1d(c_out, eps=1e-3).to(DEV).to(DTYPES[case["dtype"]])
            with torch.no_grad():
                norm.running_mean.copy_(q["mean"])
                norm.running_var.copy_(q["var"])
                norm.weight.copy_(q["scale"])
                norm.bias.copy_(q["shift"])
            mods += [norm, nn.ReLU()]
    return spconv.SparseSequential(*mods).eval().requires_grad_(False)


def _tensor(case, state):
    return spconv.SparseConvTensor(state["features"], state["indices"], list(_shape(case)),
                                   case["batch"])


def prepare(case, seed):
    state = {"case": case, "shape": _shape(case), "indices": _voxels(case, seed)}
    if case["op"] == "pairs":
        return state
    state["net"] = _network(case, case["net"], seed)
    first = _chain(case["pre"] or case["net"])[0]
    state["features"] = _features(case, case["n"], first[1], seed)
    if case["op"] == "kept":
        x = _tensor(case, state)
        if case["pre"]:
            x = _network(case, case["pre"], seed + 17)(x)
            x = x.replace_feature(_features(case, len(x.indices), x.features.shape[1], seed + 29))
        state["x"] = x
        for _ in range(2):  # the layers before it in the stage, the steps before this one
            state["net"](x)
    else:
        # the program's own earlier scan: weights are packed and laid out once
        state["net"](_tensor(case, state))
    return state


def run(state):
    case, shape = state["case"], state["shape"]
    if case["op"] == "kept":
        return state["net"](state["x"]).features
    if case["op"] == "pairs":
        idx, B = state["indices"], case["batch"]
        subm = generate_subm_indice_pairs(idx, shape, B, 3)
        down = generate_strided_indice_pairs(idx, shape, B, 2, 2, 0)
        up = generate_inverse_indice_pairs(down)
        return {"subm_in": torch.cat(subm.pairs_in), "subm_out": torch.cat(subm.pairs_out),
                "subm_num": subm.pair_num,
                "down_in": down.pairs_in, "down_out": down.pairs_out, "down_num": down.pair_num,
                "down_indices": down.out_indices,
                "up_in": up.pairs_in, "up_out": up.pairs_out, "up_indices": up.out_indices}
    y = state["net"](_tensor(case, state))
    if case["op"] == "dense":
        return y.dense()
    return {"features": y.features, "indices": y.indices}


# ------------------------------------------------- what it must give and do
def _key(idx, shape):
    i = idx.long()
    return ((i[:, 0] * shape[0] + i[:, 1]) * shape[1] + i[:, 2]) * shape[2] + i[:, 3]


def _offsets(k):
    return [(z, y, x) for z in range(k[0]) for y in range(k[1]) for x in range(k[2])]


def _subm(idx, shape, k):
    """Per slot (input rows, output rows), output rows ascending."""
    order = torch.argsort(_key(idx, shape))
    keys = _key(idx, shape)[order]
    size = torch.tensor(shape, device=idx.device)
    pairs = []
    for o in _offsets(k):
        at = idx.clone()
        at[:, 1:] += torch.tensor([a - b // 2 for a, b in zip(o, k)], device=idx.device, dtype=idx.dtype)
        inside = ((at[:, 1:] >= 0) & (at[:, 1:] < size)).all(1)
        want = _key(at, shape)
        pos = torch.searchsorted(keys, want).clamp(max=len(keys) - 1)
        rows = (inside & (keys[pos] == want)).nonzero()[:, 0]
        pairs.append((order[pos[rows]], rows))
    return pairs


def _down(idx, shape, k, s, p):
    """(per slot (input rows, output rows), output coordinates, output shape)."""
    out = tuple((n + 2 * b - a) // c + 1 for n, a, c, b in zip(shape, k, s, p))
    i = idx.long()
    size, step = torch.tensor(out, device=idx.device), torch.tensor(s, device=idx.device)
    found = []
    for o in _offsets(k):
        v = i[:, 1:] + torch.tensor([b - a for a, b in zip(o, p)], device=idx.device)
        q = torch.div(v, step, rounding_mode="floor")
        rows = ((v >= 0) & (v % step == 0) & (q < size)).all(1).nonzero()[:, 0]
        at = torch.cat([i[rows, :1], q[rows]], 1)
        found.append((rows, _key(at, out)))
    uniq = torch.unique(torch.cat([f[1] for f in found]))
    pairs = [(rows, torch.searchsorted(uniq, keys)) for rows, keys in found]
    x, r = uniq % out[2], uniq // out[2]
    y, r = r % out[1], r // out[1]
    return pairs, torch.stack([r // out[0], r % out[0], y, x], 1).int(), out


def _up(pairs, idx):
    """The inverse of such pairs: (per slot (input rows, output rows), coordinates)."""
    used = torch.unique(torch.cat([a for a, _ in pairs]))
    return [(b, torch.searchsorted(used, a)) for a, b in pairs], idx[used]


def _walk(case, text, idx, shape, down=None):
    """Each layer's (pairs, rows in, rows out), then the coordinates and shape
    after the chain and the strided layers' pairs by key."""
    steps, kept, down = [], {}, dict(down or {})
    for kind, _, _, k, s, p, key in _chain(text):
        rows = len(idx)
        if kind == "m":
            if key is None or key not in kept:
                kept[key] = _subm(idx, shape, k)
            steps.append((kept[key], rows, rows))
        elif kind == "d":
            pairs, out, out_shape = _down(idx, shape, k, s, p)
            down[key] = (pairs, idx, shape)
            steps.append((pairs, rows, len(out)))
            idx, shape = out, out_shape
        else:
            fwd, before, before_shape = down[key]
            pairs, out = _up(fwd, before)
            steps.append((pairs, rows, len(out)))
            idx, shape = out, before_shape
    return steps, idx, shape, down


@functools.lru_cache(maxsize=64)
def _work(items):
    case = dict(items)
    size = DTYPES[case["dtype"]].itemsize
    idx, shape, down = _voxels(case, 1), _shape(case), {}
    nbytes, flops = 0, 0
    if case["op"] == "pairs":
        subm = sum(len(a) for a, _ in _subm(idx, shape, (3, 3, 3)))
        pairs, out, _ = _down(idx, shape, (2, 2, 2), (2, 2, 2), (0, 0, 0))
        inverse, up = _up(pairs, idx)
        one = sum(len(a) for a, _ in pairs)
        # coordinates in; int64 pair lists and int32 coordinates out
        return {"bytes": 16 * (len(idx) + len(out) + len(up)) + 16 * (subm + 2 * one), "flops": 0}
    if case["pre"]:
        _, idx, shape, down = _walk(case, case["pre"], idx, shape)
    steps, idx, shape, _ = _walk(case, case["net"], idx, shape, down)
    for (kind, c_in, c_out, k, _, _, _), (pairs, rows_in, rows_out) in zip(_chain(case["net"]), steps):
        P = sum(len(a) for a, _ in pairs)
        flops += 2 * P * c_in * c_out
        nbytes += size * (rows_in * c_in + rows_out * c_out + math.prod(k) * c_in * c_out)
        if case["op"] == "kept":
            nbytes += 8 * P  # its pairs, in hand
    if case["op"] != "kept":
        nbytes += 16 * (case["n"] + len(idx))  # coordinates in and out
    if case["op"] == "dense":
        nbytes += size * case["batch"] * math.prod(shape) * _chain(case["net"])[-1][2]
    return {"bytes": nbytes, "flops": flops}


def work(case):
    return _work(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


def tolerance(case):
    if case["op"] == "pairs":
        return "exact"
    layers = len(_chain(case["net"]))
    # One rounding of the outputs (f16, bf16) or a sum of some thousand
    # products in another order (f32), about four times what is seen against
    # 64 bits (2.1e-4, 1.7e-3 and, at 27 x 64 channels, 5e-7); each further
    # layer reads the rounded outputs of the one before it.
    rel = {"f32": 4e-6, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]
    most = {"f32": 2e-5, "f16": 4e-3, "bf16": 3e-2}[case["dtype"]]
    return {"rel": rel * math.sqrt(layers), "max": most * math.sqrt(layers)}


def exact(case, seed):
    idx, shape, down = _voxels(case, seed), _shape(case), {}
    if case["op"] == "pairs":
        subm = _subm(idx, shape, (3, 3, 3))
        pairs, out, _ = _down(idx, shape, (2, 2, 2), (2, 2, 2), (0, 0, 0))
        inverse, up = _up(pairs, idx)
        num = lambda p: torch.tensor([len(a) for a, _ in p])  # noqa: E731
        return {"subm_in": torch.cat([a for a, _ in subm]), "subm_out": torch.cat([b for _, b in subm]),
                "subm_num": num(subm),
                "down_in": [a for a, _ in pairs], "down_out": [b for _, b in pairs],
                "down_num": num(pairs), "down_indices": out,
                "up_in": [a for a, _ in inverse], "up_out": [b for _, b in inverse],
                "up_indices": up}
    f = None
    if case["pre"]:
        _, idx, shape, down = _walk(case, case["pre"], idx, shape)
        f = _features(case, len(idx), _chain(case["pre"])[-1][2], seed + 29).double()
    if f is None:
        f = _features(case, case["n"], _chain(case["net"])[0][1], seed).double()
    steps, idx, shape, _ = _walk(case, case["net"], idx, shape, down)
    for (_, c_in, c_out, k, _, _, _), q, (pairs, _, rows) in zip(
            _chain(case["net"]), _params(case, case["net"], seed), steps):
        K = math.prod(k)
        w = q["w"].double()
        # (K, c_in, c_out); a 1x1x1 kernel's storage is read as (c_in, c_out)
        w = w.reshape(1, c_in, c_out) if K == 1 else w.reshape(c_out, K, c_in).permute(1, 2, 0)
        y = torch.zeros(rows, c_out, dtype=torch.float64, device=DEV)
        for j, (a, b) in enumerate(pairs):
            y.index_add_(0, b, f[a] @ w[j].contiguous())
        y += q["b"].double()
        if case["bn"]:
            y = (y - q["mean"].double()) / (q["var"].double() + 1e-3).sqrt() * q["scale"].double() \
                + q["shift"].double()
            y = y.clamp(min=0)
        f = y
    if case["op"] == "kept":
        return f
    if case["op"] == "dense":
        vol = torch.zeros(case["batch"], *shape, f.shape[1], dtype=torch.float64, device=DEV)
        vol.view(-1, f.shape[1])[_key(idx, shape)] = f
        return vol.permute(0, 4, 1, 2, 3).contiguous()
    return {"features": f, "indices": idx}
