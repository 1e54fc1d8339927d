"""Performance cases of the library: the calls that a program using it makes, from a few microseconds to a
few milliseconds each.

A case is a dict of plain values; ``kind`` names the call:

    layer    forward of one sparse convolution (inference) on a geometry that the program keeps
    step     forward and backward of one sparse convolution (features, weights, bias) on a kept geometry
    frame    a new voxel cloud per pass: submanifold geometry, submanifold layer, strided geometry, strided
             layer - inference, or with ``train`` forward and backward
    s8       int8 inference of one strided sparse convolution (scale, bias, saturating round)
    gemm     ``matmul2`` without indices: ``nt`` (x W^T), ``nn`` (dy W) or ``tn`` (dy^T x)
    scatter  ``matmul2`` ShuffleAC: C[c] = A[a] B + C0[c], one kernel offset of a gather-GEMM-scatter
    wgrad    ``matmul2`` ShuffleAB: dW = dY[a]^T X[b], the weight gradient of one kernel offset

Voxel clouds are Gaussian clusters (sigma 15 voxels) with 10 % uniform noise on a LiDAR-sized grid, as in
``cumm_amd.synth``; sizes are those of the benchmark, the tests and the smoke run.
"""
import functools
import math

import torch

from cumm_amd import pairs, torch_bridge, tuner
from cumm_amd import tensorview as tv
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.gemm.main import GemmMainUnitTest
from cumm_amd.tensorview.gemm import ConvOpType, ConvParams, GemmParams, ShuffleStrideType

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
TV_DTYPES = {"f16": tv.float16, "bf16": tv.bfloat16}
SIGMA = 15.0
MARGIN = 64                     # sites by which a seed may move a cloud along y and x
LIDAR = (41, 1600, 1408)        # z, y, x of the 120 k and 300 k voxel configurations
LARGE = (64, 2048, 2048)        # of the 1 M voxel configuration

# one per program: it keeps the descriptor it found for a kind of call
_TUNER = tuner.Tuner(steps=5, warmup=2)


# ---- cases

def _conv(name, kind, voxels, cin, cout, dtype, ksize=3, stride=1, **more):
    large = voxels > 500000
    return dict(name=name, kind=kind, voxels=voxels, clusters=_clusters(voxels), large_grid=large, cin=cin, cout=cout,
                dtype=dtype, ksize=ksize, stride=stride, **more)


def _clusters(voxels):
    return max(1, round(voxels / (5000 if voxels > 500000 else 2000)))


def listed():
    return [
        # the smallest call in use: one layer of a small cloud (the size of the smoke run), latency alone
        _conv("layer_f16_64_2k", "layer", 2000, 64, 64, "f16"),
        # a detector's inference on the next LiDAR sweep: everything from coordinates to features
        _conv("frame_infer_f16_64_128_120k", "frame", 119985, 64, 128, "f16", train=False),
        # a training iteration on a new, larger sweep
        _conv("frame_train_bf16_32_64_300k", "frame", 300001, 32, 64, "bf16", train=True),
        # the headline layer trained: 120 k voxels, 64 channels
        _conv("step_subm_f16_64_120k", "step", 119985, 64, 64, "f16"),
        # one layer of the wide bf16 stack, 1 M voxels (the largest)
        _conv("step_subm_bf16_128_1m", "step", 999645, 128, 128, "bf16"),
        # its down-sampling layer, on the 300 k voxel cloud
        _conv("step_down_bf16_128_256_300k", "step", 299905, 128, 256, "bf16", stride=2),
        # a large receptive field: 125 kernel offsets, several mask words per position
        _conv("step_5x5x5_f16_64_120k", "step", 119985, 64, 64, "f16", ksize=5),
        # quantised inference: stride 2, 64 -> 128 channels
        _conv("s8_down_64_128_300k", "s8", 299905, 64, 128, "s8", stride=2),
        # a large dense product of a linear layer's forward pass
        dict(name="gemm_nt_f16_4096", kind="gemm", m=4096, n=4096, k=4096, layout="nt", dtype="f16"),
        # its gradient for the input at an ordinary, ragged size
        dict(name="gemm_nn_bf16_2000x776x1160", kind="gemm", m=2000, n=776, k=1160, layout="nn", dtype="bf16"),
        # one kernel offset as gather-GEMM-scatter: 150 k pairs among 200 k rows
        dict(name="scatter_f16_64_64_150k", kind="scatter", rows=200000, pairs=150000, n=64, k=64, dtype="f16"),
        # and that offset's weight gradient
        dict(name="wgrad_f16_64_64_150k", kind="wgrad", rows=200000, pairs=150000, n=64, k=64, dtype="f16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, lo, hi, step=8):
    return max(step, step * int(round(_log(rng, lo, hi) / step)))


def draw(rng):
    kind = rng.choice(["layer", "frame", "step", "step", "step5", "s8", "gemm", "gemm", "scatter", "wgrad"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "layer":
        return _unnamed(_conv("", "layer", _log(rng, 1000, 300000), _channels(rng, 16, 128), _channels(rng, 16, 128), dtype,
                              stride=rng.choice([1, 2])))
    if kind == "frame":
        return _unnamed(_conv("", "frame", _log(rng, 2000, 300000), _channels(rng, 16, 64), _channels(rng, 16, 128), dtype,
                              train=rng.choice([False, True])))
    if kind == "step":
        stride = rng.choice([1, 2])
        voxels = _log(rng, 2000, 1000000 if stride == 1 else 300000)
        return _unnamed(_conv("", "step", voxels, _channels(rng, 16, 128), _channels(rng, 16, 128 if stride == 1 else 256),
                              dtype, stride=stride))
    if kind == "step5":
        return _unnamed(_conv("", "step", _log(rng, 2000, 120000), _channels(rng, 16, 64), _channels(rng, 16, 64), dtype,
                              ksize=5))
    if kind == "s8":
        return _unnamed(_conv("", "s8", _log(rng, 2000, 300000), _channels(rng, 16, 64, 16), _channels(rng, 16, 128, 16),
                              "s8", stride=rng.choice([1, 2])))
    if kind == "gemm":
        layout = rng.choice(["nt", "nn", "tn"])
        m, n, k = (_channels(rng, 64, 4096) for _ in range(3))
        if layout != "tn":        # the rows of a row-major operand may be any number
            m = max(1, m - rng.randrange(8))
        return dict(kind="gemm", m=m, n=n, k=k, layout=layout, dtype=dtype)
    rows = _log(rng, 2000, 200000)
    return dict(kind=kind, rows=rows, pairs=max(1, int(rows * rng.uniform(0.1, 1.0))), n=_channels(rng, 16, 128),
                k=_channels(rng, 16, 128), dtype=dtype)


def _unnamed(case):
    del case["name"]
    return case


# ---- inputs

def _grid(case):
    return LARGE if case["large_grid"] else LIDAR


@functools.lru_cache(None)
def _sites(voxels, clusters, large_grid):
    """``voxels`` unique sites (z, y, x) that keep 2 * MARGIN away from the far ends of y and x."""
    gen = _gen(1)
    dev = gen.device
    size = LARGE if large_grid else LIDAR
    size = (size[0], size[1] - 2 * MARGIN, size[2] - 2 * MARGIN)
    grid = torch.tensor(size, dtype=torch.float32, device=dev)
    weights = torch.tensor([size[1] * size[2], size[2], 1], dtype=torch.int64, device=dev)
    centers = torch.rand(clusters, 3, generator=gen, device=dev) * grid

    def keys(p):
        ok = ((p >= 0) & (p < grid)).all(1)
        return (p[ok].to(torch.int64) * weights).sum(1)

    sites = torch.empty(0, dtype=torch.int64, device=dev)
    want = voxels - voxels // 10
    for _ in range(20):
        m = int(1.6 * voxels) + 256
        cid = torch.randint(0, clusters, (m,), generator=gen, device=dev)
        p = torch.round(centers[cid] + SIGMA * torch.randn(m, 3, generator=gen, device=dev))
        sites = torch.unique(torch.cat([sites, keys(p)]))
        if sites.numel() >= want:
            break
    sites = sites[torch.randperm(sites.numel(), generator=gen, device=dev)[:want]]
    while sites.numel() < voxels:       # noise, topped up to the exact number
        noise = torch.floor(torch.rand(voxels - sites.numel(), 3, generator=gen, device=dev) * grid)
        sites = torch.unique(torch.cat([sites, keys(noise)]))
    return torch.stack([torch.div(sites, weights[0], rounding_mode="floor"),
                        torch.div(sites, weights[1], rounding_mode="floor") % size[1], sites % size[2]], 1)


def _cloud(case, gen):
    """[N, 4] int32 (batch, z, y, x), unique, in ascending order.  The seed mirrors the sites along y and
    x and moves them, by even numbers: a strided layer then has as many output sites for every seed."""
    p = _sites(case["voxels"], case["clusters"], case["large_grid"]).clone()
    grid = _grid(case)
    for d in (1, 2):
        mirror, shift = torch.randint(0, MARGIN, (2,), generator=gen, device=p.device)
        end = grid[d] - 2 * MARGIN
        p[:, d] = torch.where(mirror % 2 == 1, end - p[:, d], p[:, d]) + 2 * shift
    order = torch.argsort((p[:, 0] * grid[1] + p[:, 1]) * grid[2] + p[:, 2])
    coords = torch.zeros(p.shape[0], 4, dtype=torch.int32, device=p.device)
    coords[:, 1:] = p[order]
    return coords


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype)


def _geometry(case, coords, stride):
    k = (case["ksize"],) * 3
    pad = (case["ksize"] // 2,) * 3
    return torch_bridge.SparseConvGeometry(coords, _grid(case), k, None if stride == 1 else (stride,) * 3, pad)


def _weights(gen, cin, cout, kv, dtype):
    return _normal(gen, (cout, kv, cin), dtype, (2.0 / (3 * cin)) ** 0.5), _normal(gen, (cout,), dtype, 0.1)


def prepare(case, seed):
    gen = _gen(seed)
    return {"layer": _prepare_layer, "step": _prepare_layer, "frame": _prepare_frame, "s8": _prepare_s8, "gemm": _prepare_gemm,
            "scatter": _prepare_scatter, "wgrad": _prepare_wgrad}[case["kind"]](case, gen)


def _prepare_layer(case, gen):
    dtype, train = DTYPES[case["dtype"]], case["kind"] == "step"
    geometry = _geometry(case, _cloud(case, gen), case["stride"])
    w, b = _weights(gen, case["cin"], case["cout"], case["ksize"] ** 3, dtype)
    x = _normal(gen, (case["voxels"], case["cin"]), dtype)
    s = {"run": _run_step if train else _run_layer, "geometry": geometry}
    s["x"], s["w"], s["b"] = (t.requires_grad_(train) for t in (x, w, b))
    if train:
        s["grad"] = _normal(gen, (geometry.n_out, case["cout"]), dtype)
    return s


def _run_layer(s):
    return torch_bridge.sparse_conv(s["x"], s["w"], s["b"], s["geometry"], relu=True)


def _run_step(s):
    out = torch_bridge.sparse_conv(s["x"], s["w"], s["b"], s["geometry"], relu=True)
    return (out,) + torch.autograd.grad(out, (s["x"], s["w"], s["b"]), s["grad"])


def _prepare_frame(case, gen):
    dtype, train = DTYPES[case["dtype"]], case["train"]
    w1, b1 = _weights(gen, case["cin"], case["cin"], 27, dtype)
    w2, b2 = _weights(gen, case["cin"], case["cout"], 27, dtype)
    return {"run": _run_frame, "case": case, "coords": _cloud(case, gen), "x": _normal(gen, (case["voxels"], case["cin"]), dtype),
            "train": train, "weights": tuple(t.requires_grad_(train) for t in (w1, b1, w2, b2))}


def _run_frame(s):
    w1, b1, w2, b2 = s["weights"]
    subm = _geometry(s["case"], s["coords"], 1)
    down = _geometry(s["case"], s["coords"], 2)
    y = torch_bridge.sparse_conv(s["x"], w1, b1, subm, relu=True)
    out = torch_bridge.sparse_conv(y, w2, b2, down, relu=True)
    if not s["train"]:
        return out, down.out_coords
    # (the loss: half the sum of squares, whose gradient is the output itself)
    return (out.detach(), down.out_coords) + torch.autograd.grad(out, s["weights"], out.detach())


def _prepare_s8(case, gen):
    coords = torch_bridge.torch2tensor(_cloud(case, gen))
    bits = (1 << 27) - 1
    if case["stride"] == 1:
        table = pairs.subm_pairs_device(coords, _grid(case))
    else:
        table = pairs.sparse_conv_pairs_device(coords, _grid(case))
    mask, order = pairs.sort_by_mask_device(table.mask_fwd, bits, by_offset_count=True)
    n_out, cin, cout = int(table.indices_fwd.dim(1)), case["cin"], case["cout"]
    ints = functools.partial(torch.randint, -127, 128, generator=gen, device="cuda", dtype=torch.int8)
    scale = torch.rand(cout, generator=gen, device="cuda") * 0.009 + 0.001
    out = torch.zeros(n_out, cout, dtype=torch.int8, device="cuda")
    t = torch_bridge.torch2tensor
    p = ConvParams(3, ConvOpType.Forward)
    p.conv_algo_desp = [d for d in ConvMainUnitTest.get_all_conv_algo_desp() if d.dtype_a == tv.int8 and d.is_int8_inference][0]
    p.input, p.weight, p.output = t(ints((case["voxels"], cin))), t(ints((cout, 27, cin))), t(out)
    p.scale, p.bias = t(scale), t(torch.randn(cout, generator=gen, device="cuda"))
    p.mask, p.mask_argsort = mask, order
    p.indices, p.indices_by_position = pairs.pairs_by_position_device(table.indices_fwd, order), True
    _TUNER.tune_conv(p)
    return {"run": _run_s8, "params": p, "out": out}


def _run_s8(s):
    ConvMainUnitTest.implicit_gemm2(s["params"])
    return s["out"]


@functools.lru_cache(None)
def _gemm_desp(dtype, shuffle, trans_a, trans_b):
    for d in GemmMainUnitTest.get_all_algo_desp():
        if (d.dtype_a == dtype and d.dtype_c == dtype and d.shuffle_type == shuffle and d.trans_a == trans_a and
                d.trans_b == trans_b and not d.trans_c):
            return d
    raise KeyError((dtype, shuffle, trans_a, trans_b))


def _prepare_gemm(case, gen):
    m, n, k, dtype = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
    ta, tb = case["layout"][0] == "t", case["layout"][1] == "t"
    t = torch_bridge.torch2tensor
    out = torch.zeros(m, n, dtype=dtype, device="cuda")
    p = GemmParams()
    p.algo_desp = _gemm_desp(TV_DTYPES[case["dtype"]], ShuffleStrideType.NoShuffle, ta, tb).copy()
    p.a = t(_normal(gen, (k, m) if ta else (m, k), dtype))
    p.b = t(_normal(gen, (n, k) if tb else (k, n), dtype, 0.05))
    p.c = t(out)
    p.alpha, p.beta = 1.0, 0.0
    _TUNER.tune_gemm(p)
    return {"run": _run_gemm, "params": p, "out": out}


def _run_gemm(s):
    GemmMainUnitTest.matmul2(s["params"])
    return s["out"]


def _rows(gen, rows, pairs_):
    return torch.randperm(rows, generator=gen, device="cuda")[:pairs_].to(torch.int32)


def _prepare_scatter(case, gen):
    dtype, t = DTYPES[case["dtype"]], torch_bridge.torch2tensor
    out = torch.zeros(case["rows"], case["n"], dtype=dtype, device="cuda")
    p = GemmParams()
    p.algo_desp = _gemm_desp(TV_DTYPES[case["dtype"]], ShuffleStrideType.ShuffleAC, False, False).copy()
    p.a, p.b = t(_normal(gen, (case["rows"], case["k"]), dtype)), t(_normal(gen, (case["k"], case["n"]), dtype, 0.1))
    p.c = t(out)
    p.d = t(_normal(gen, (case["rows"], case["n"]), dtype))
    p.a_inds, p.c_inds = (t(_rows(gen, case["rows"], case["pairs"])) for _ in range(2))
    p.alpha, p.beta = 1.0, 1.0
    _TUNER.tune_gemm(p)
    return {"run": _run_gemm, "params": p, "out": out}


def _prepare_wgrad(case, gen):
    dtype, t = DTYPES[case["dtype"]], torch_bridge.torch2tensor
    out = torch.zeros(case["n"], case["k"], dtype=dtype, device="cuda")
    p = GemmParams()
    p.algo_desp = _gemm_desp(TV_DTYPES[case["dtype"]], ShuffleStrideType.ShuffleAB, True, False).copy()
    p.a, p.b = t(_normal(gen, (case["rows"], case["n"]), dtype)), t(_normal(gen, (case["rows"], case["k"]), dtype))
    p.c = t(out)
    p.a_inds, p.b_inds = (t(_rows(gen, case["rows"], case["pairs"])) for _ in range(2))
    p.alpha, p.beta = 1.0, 0.0
    _TUNER.tune_gemm(p)
    return {"run": _run_gemm, "params": p, "out": out}


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without

@functools.lru_cache(None)
def _counts(voxels, clusters, large_grid, ksize, stride):
    """(output sites, active pairs) of one such cloud."""
    case = dict(voxels=voxels, clusters=clusters, large_grid=large_grid)
    c = _cloud(case, _gen(1))[:, 1:].to(torch.int64)
    grid = torch.tensor(_grid(case), device=c.device)
    half = ksize // 2
    out_grid = grid if stride == 1 else (grid + 2 * half - ksize) // stride + 1
    n_pairs, sites = 0, []
    mine = (c[:, 0] * grid[1] + c[:, 1]) * grid[2] + c[:, 2]
    for dz in range(-half, half + 1):
        for dy in range(-half, half + 1):
            for dx in range(-half, half + 1):
                p = c + torch.tensor([dz, dy, dx], device=c.device)
                o = torch.div(p, stride, rounding_mode="floor")
                o = o[(p % stride == 0).all(1) & (p >= 0).all(1) & (o < out_grid).all(1)]
                o = (o[:, 0] * out_grid[1] + o[:, 1]) * out_grid[2] + o[:, 2]
                if stride == 1:
                    at = torch.searchsorted(mine, o).clamp_(max=mine.numel() - 1)
                    n_pairs += int((mine[at] == o).sum())
                else:
                    n_pairs += o.numel()
                    sites.append(o)
    return (voxels, n_pairs) if stride == 1 else (int(torch.unique(torch.cat(sites)).numel()), n_pairs)


def _of_layer(n_in, n_out, n_pairs, cin, cout, kv, eb, train, subm):
    """Rows in and out, weights, pair table, masks and order of a forward pass; with ``train`` also those of
    the two gradients: gradient rows in, input gradients out, weight and bias gradients out."""
    words = (kv + 31) // 32
    rows, w = n_in * cin * eb + n_out * cout * eb, kv * cin * cout * eb + cout * eb
    table = kv * n_out * 4 + n_out * 4 * (words + 1)
    passes = 1
    if train:
        table += 0 if subm else kv * n_in * 4 + n_in * 8
        rows, w, passes = 2 * rows, 2 * w, 3
    return rows + w + table, passes * 2.0 * n_pairs * cin * cout


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    if kind in ("scatter", "wgrad"):
        p, n, k = case["pairs"], case["n"], case["k"]
        rows = p * (k + 2 * n) if kind == "scatter" else p * (n + k)
        return {"bytes": 2 * (rows + n * k) + 8 * p, "flops": 2.0 * p * n * k}
    kv, n_in, cin, cout = case["ksize"] ** 3, case["voxels"], case["cin"], case["cout"]
    eb = 1 if case["dtype"] == "s8" else 2
    key = (n_in, case["clusters"], case["large_grid"], case["ksize"])
    if kind != "frame":
        n_out, n_pairs = _counts(*key, case["stride"])
        b, f = _of_layer(n_in, n_out, n_pairs, cin, cout, kv, eb, kind == "step", case["stride"] == 1)
        return {"bytes": b + (8 * cout if kind == "s8" else 0), "flops": f}
    (_, p1), (n_out, p2) = _counts(*key, 1), _counts(*key, 2)
    b1, f1 = _of_layer(n_in, n_in, p1, cin, cin, kv, eb, case["train"], True)
    b2, f2 = _of_layer(n_in, n_out, p2, cin, cout, kv, eb, case["train"], False)
    # preparation: coordinates in (twice) and out; forward and backward tables, masks and orders written
    prep = 32 * n_in + 16 * n_out + 4 * (2 * kv + 3) * n_in + 4 * (kv + 2) * n_out + 4 * (kv + 2) * n_in
    return {"bytes": b1 + b2 + prep, "flops": f1 + f2}


def tolerance(case):
    # Four times the distance of the outputs from the same calls computed in 64 bits on the same
    # inputs: results are rounded once from 32-bit sums, so that is the rounding of the type
    # (relative 2-norm 2.1e-4 for f16 and 1.7e-3 for bf16, 2.9e-4 and 2.4e-3 behind two layers).
    if case["dtype"] == "s8":
        return "exact"        # 32-bit integer sums, one fused scale-and-bias, round half to even
    rel = {"f16": 1e-3, "bf16": 8e-3}[case["dtype"]]
    # The largest single difference is ten roundings (measured: 5e-4 and 4e-3) - except behind the gate
    # of a ReLU, where a sum within its rounding of zero opens or closes the gate of one of the few
    # dozen products in an element of the input gradient (measured: 0.07).
    gated = case["kind"] == "step" or case["kind"] == "frame"
    return {"rel": rel, "max": 0.3 if gated else 10 * rel}
