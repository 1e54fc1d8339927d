"""torch <-> tv.Tensor views and the autograd functions over the sparse convolution, against the
same convolution written with torch indexing in fp32 (autograd gives the reference gradients)."""
import numpy as np
import pytest

import helpers as H
from cumm_amd import pairs
from cumm_amd import tensorview as tv

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _reference(feat32, w32, bias32, ind_f, relu):
    """out[o] = sum_k W[:, k, :] @ x[ind[k][o]] over the valid pairs, in fp32 on the CPU."""
    n_out = ind_f.shape[1]
    out = torch.zeros(n_out, w32.shape[0])
    for k in range(ind_f.shape[0]):
        o = np.nonzero(ind_f[k] >= 0)[0]
        if o.size:
            out = out.index_add(0, torch.as_tensor(o), feat32[torch.as_tensor(ind_f[k][o].astype(np.int64))] @ w32[:, k, :].T)
    if bias32 is not None:
        out = out + bias32
    return torch.relu(out) if relu else out


def test_views_share_memory_both_ways():
    from cumm_amd import torch_bridge as tb
    t = torch.arange(24, dtype=torch.float16, device="cuda").reshape(4, 6)
    v = tb.torch2tensor(t)
    assert v.shape == [4, 6] and v.dtype == tv.float16 and v.byte_pointer() == t.data_ptr()
    np.testing.assert_array_equal(H.host(v), t.cpu().numpy())
    back = tb.tensor2torch(v, clone=False)
    assert back.data_ptr() == t.data_ptr() and torch.equal(back, t)
    back[1, 2] = 100.0
    assert float(t[1, 2]) == 100.0
    assert tb.tensor2torch(v, clone=True).data_ptr() != t.data_ptr()
    # a strided view, bf16, and an unsigned tensor
    s = tb.torch2tensor(t[:, ::2])
    np.testing.assert_array_equal(H.host(s), t[:, ::2].cpu().numpy())
    b = torch.randn(5, 3, device="cuda").to(torch.bfloat16)
    assert torch.equal(tb.tensor2torch(tb.torch2tensor(b), clone=False), b)
    u = tv.zeros([7], tv.uint32, 0)
    with pytest.raises(ValueError):
        tb.tensor2torch(u)
    assert tb.tensor2torch(u, cast_uint_to_int=True).dtype == torch.int32


@pytest.mark.parametrize("strided", [False, True, "pad0"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_autograd_matches_torch_indexing(dtype, strided):
    from cumm_amd import torch_bridge as tb
    print("case torch bridge", dtype, strided, flush=True)
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    coords, grid = H.small_cloud(21, 2500)
    padding = (1, 1, 1)
    if strided == "pad0":
        # stride 2 without padding on even axes: the inputs on the last plane of an axis feed no
        # output site.  A whole plane of them fills several 128-row tiles whose mask is zero, which
        # the backward-input kernel skips: their gradient must still come back as zero.
        padding = (0, 0, 0)
        zz, yy = np.meshgrid(np.arange(grid[0]), np.arange(grid[1]), indexing="ij")
        plane = np.stack([np.zeros(zz.size, np.int64), zz.ravel(), yy.ravel(),
                          np.full(zz.size, grid[2] - 1)], axis=1).astype(np.int32)
        coords = np.unique(np.concatenate([coords, plane]), axis=0).astype(np.int32)
    c_in, k_out = 64, 96
    torch.manual_seed(3)
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, stride=(2, 2, 2) if strided else None,
                                padding=padding)
    host = pairs.sparse_conv_pairs(coords, grid, padding=padding) if strided else pairs.subm_pairs(coords, grid)
    if strided == "pad0":
        assert int((host.mask_bwd == 0).sum()) >= 3 * 128
    np.testing.assert_array_equal(H.host(geo.indices_fwd), host.indices_fwd)
    def rel(a, b):
        return float((a.float().cpu() - b).abs().max() / b.abs().max().clamp_min(1e-6))

    # the second pass runs on other tensors (the first pass's stay alive, so the addresses differ):
    # the bridge replays the argument blocks it validated in the first pass with the new pointers
    held = []
    for trip in range(2):
        feat = (torch.randn(coords.shape[0], c_in)).to(tdt)
        weight = (torch.randn(k_out, 27, c_in) * 0.05).to(tdt)
        bias = (torch.randn(k_out) * 0.1).to(tdt)
        gout = torch.randn(geo.n_out, k_out).to(tdt)

        f_d = feat.cuda().requires_grad_(True)
        w_d = weight.cuda().requires_grad_(True)
        b_d = bias.cuda().requires_grad_(True)
        out = tb.sparse_conv(f_d, w_d, b_d, geo, relu=True)
        g_d = gout.cuda()
        out.backward(g_d)
        held += [f_d, w_d, b_d, out, g_d]

        f_r = feat.float().requires_grad_(True)
        w_r = weight.float().requires_grad_(True)
        b_r = bias.float().requires_grad_(True)
        ref = _reference(f_r, w_r, b_r, host.indices_fwd, relu=True)
        # the ReLU gate of the reference must be the GPU's own (outputs within rounding of zero differ)
        gate = (out.detach().float().cpu() > 0).float()
        pre = _reference(f_r, w_r, b_r, host.indices_fwd, relu=False)
        (pre * gate * gout.float()).sum().backward()

        assert rel(out.detach(), ref.detach()) < 1e-2, trip
        assert rel(f_d.grad, f_r.grad) < 1e-2, trip
        assert rel(w_d.grad, w_r.grad) < 1e-2, trip
        assert rel(b_d.grad, b_r.grad) < 1e-2, trip
    assert len(geo._launches) == 3

    # other shapes on the same geometry do not meet the remembered calls
    with pytest.raises(ValueError):
        tb.sparse_conv(f_d[:-1], w_d, b_d, geo, relu=True)
    with pytest.raises(ValueError):
        tb.sparse_conv(f_d, w_d[:, :26], b_d, geo, relu=True)


@pytest.mark.parametrize("case", ["subm555", "strided335"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_autograd_with_kernel_volumes_above_32(dtype, case):
    """5 x 5 x 5 submanifold and strided 3 x 3 x 5 layers through the bridge: masks of several words
    made and sorted on the GPU, forward and backward-input on the dynamic_mask descriptors (one
    launch each), backward-weight offset by offset over the pair lists; outputs and all three
    gradients against the convolution written with torch indexing in fp32."""
    from cumm_amd import torch_bridge as tb
    print("case torch bridge large kernel", dtype, case, flush=True)
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    coords, grid = H.small_cloud(31, 1500, grid=(12, 30, 28))
    if case == "subm555":
        ksize, stride, padding = (5, 5, 5), None, (2, 2, 2)
        host = pairs.subm_pairs(coords, grid, ksize)
    else:
        ksize, stride, padding = (3, 3, 5), (2, 2, 2), (1, 1, 2)
        host = pairs.sparse_conv_pairs(coords, grid, ksize, stride, padding)
    kv = ksize[0] * ksize[1] * ksize[2]
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, ksize=ksize, stride=stride, padding=padding)
    assert geo.words == (kv + 31) // 32 and geo.kv == kv
    np.testing.assert_array_equal(H.host(geo.indices_fwd), host.indices_fwd)
    c_in, k_out = 64, 64
    torch.manual_seed(5)

    def rel(a, b):
        return float((a.float().cpu() - b).abs().max() / b.abs().max().clamp_min(1e-6))

    for trip in range(2):
        feat = torch.randn(coords.shape[0], c_in).to(tdt)
        weight = (torch.randn(k_out, kv, c_in) * 0.03).to(tdt)
        bias = (torch.randn(k_out) * 0.1).to(tdt)
        gout = torch.randn(geo.n_out, k_out).to(tdt)
        f_d, w_d, b_d = (t.cuda().requires_grad_(True) for t in (feat, weight, bias))
        out = tb.sparse_conv(f_d, w_d, b_d, geo, relu=True)
        out.backward(gout.cuda())
        f_r, w_r, b_r = (t.float().requires_grad_(True) for t in (feat, weight, bias))
        ref = _reference(f_r, w_r, b_r, host.indices_fwd, relu=True)
        gate = (out.detach().float().cpu() > 0).float()
        pre = _reference(f_r, w_r, b_r, host.indices_fwd, relu=False)
        (pre * gate * gout.float()).sum().backward()
        assert rel(out.detach(), ref.detach()) < 1e-2, trip
        assert rel(f_d.grad, f_r.grad) < 1e-2, trip
        assert rel(w_d.grad, w_r.grad) < 1e-2, trip
        assert rel(b_d.grad, b_r.grad) < 1e-2, trip


def test_module_stack_runs_and_trains_a_step():
    from cumm_amd import torch_bridge as tb
    coords, grid = H.small_cloud(22, 3000)
    c = torch.as_tensor(coords, device="cuda")
    geo = tb.SparseConvGeometry(c, grid)
    down = tb.SparseConvGeometry(c, grid, stride=(2, 2, 2))
    torch.manual_seed(1)
    l1 = tb.SparseConv3d(32, 64, relu=True)
    l2 = tb.SparseConv3d(64, 64, relu=True)
    l3 = tb.SparseConv3d(64, 128)
    x = torch.randn(coords.shape[0], 32, device="cuda").half()
    params = list(l1.parameters()) + list(l2.parameters()) + list(l3.parameters())
    y = l3(l2(l1(x, geo), geo) + l1(x, geo), down)          # a residual connection by torch
    assert y.shape == (down.n_out, 128) and torch.isfinite(y.float()).all()
    loss = y.float().pow(2).mean()
    loss.backward()
    assert all(p.grad is not None and torch.isfinite(p.grad.float()).all() for p in params)
    assert float(l1.weight.grad.float().abs().max()) > 0


def test_deterministic_switch_gives_the_same_weight_gradient_twice():
    """torch.use_deterministic_algorithms(True) selects the fixed-order backward-weight: two
    backward passes over the same tensors give the same bits (and the value stays within
    tolerance of the default variant's)."""
    from cumm_amd import torch_bridge as tb
    coords, grid = H.small_cloud(23, 3000)
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid)
    torch.manual_seed(2)
    layer = tb.SparseConv3d(64, 64, relu=True)
    x = torch.randn(coords.shape[0], 64, device="cuda").half()

    def weight_grad():
        layer.zero_grad(set_to_none=True)
        layer(x, geo).float().pow(2).mean().backward()
        return layer.weight.grad.clone()

    default = weight_grad()
    was = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True)
    try:
        first, second = weight_grad(), weight_grad()
    finally:
        torch.use_deterministic_algorithms(was)
    assert torch.equal(first, second)
    scale = float(default.float().abs().max())
    assert float((first.float() - default.float()).abs().max()) < 1e-2 * scale


@pytest.mark.parametrize("strided,shared", [(False, False), (False, True), (True, False)])
def test_a_call_validated_on_one_geometry_runs_on_another(monkeypatch, strided, shared):
    """Two clouds of different sizes in one power of two: the second one's forward and backward are the first
    one's validated calls with other addresses and row numbers - also when the first call's gradient was
    the layer's own input (``shared``)."""
    from cumm_amd import torch_bridge as tb
    print("case moved call", strided, shared, flush=True)
    channels = 40 + 8 * (2 * strided + shared)       # a kind of call that no other test has made
    stride = (2, 2, 2) if strided else None
    torch.manual_seed(11)
    weight = (torch.randn(channels, 27, channels) * 0.05).half()

    def rel(a, b):
        return float((a.float().cpu() - b).abs().max() / b.abs().max().clamp_min(1e-6))

    sizes = []
    for trip, n in enumerate((2300, 3100)):
        coords, grid = H.small_cloud(40 + trip, n)
        geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, stride=stride)
        host = pairs.sparse_conv_pairs(coords, grid) if strided else pairs.subm_pairs(coords, grid)
        sizes.append((geo.n_in, geo.n_out))
        feat = torch.randn(geo.n_in, channels).half()
        f_d, w_d = feat.cuda().requires_grad_(True), weight.cuda().requires_grad_(True)
        gout = torch.randn(geo.n_out, channels).half()
        g_d = gout.cuda()
        if shared and trip == 0:
            g_d, gout = f_d.detach(), feat
        if trip == 1:      # no prelude from here on
            monkeypatch.setattr(tb.ConvMainUnitTest, "implicit_gemm2", None)
        out = tb.sparse_conv(f_d, w_d, None, geo)
        out.backward(g_d)
        f_r, w_r = feat.float().requires_grad_(True), weight.float().requires_grad_(True)
        ref = _reference(f_r, w_r, None, host.indices_fwd, relu=False)
        (ref * gout.float()).sum().backward()
        assert rel(out.detach(), ref.detach()) < 1e-2, trip
        assert rel(f_d.grad, f_r.grad) < 1e-2, trip
        assert rel(w_d.grad, w_r.grad) < 1e-2, trip
    assert sizes[0] != sizes[1] and all(tb._size_class(a) == tb._size_class(b) for a, b in zip(*sizes))


@pytest.mark.parametrize("strided", [False, True])
def test_a_geometry_whose_tables_exceed_31_bits_of_bytes(strided):
    """More voxels than the launches take (a table of 2^31 bytes): the geometry has its tables, masks and order,
    a forward pass is refused.  A full box of voxels, so that every entry is known."""
    from cumm_amd import torch_bridge as tb
    print("case large tables", strided, flush=True)
    kv, shape = (27, (20, 1000, 1000)) if not strided else (25, (22, 1000, 1000))
    n = shape[0] * shape[1] * shape[2]
    assert 4 * kv * n >= 1 << 31
    row = torch.arange(n, dtype=torch.int32, device="cuda")
    zyx = [row // (shape[1] * shape[2]), row // shape[2] % shape[1], row % shape[2]]
    coords = torch.stack([torch.zeros_like(row)] + zyx, 1)
    ksize = (3, 3, 3) if not strided else (1, 5, 5)
    geo = tb.SparseConvGeometry(coords, shape, ksize, (1, 1, 1) if strided else None, tuple(k // 2 for k in ksize))
    del coords
    assert (geo.n_in, geo.n_out) == (n, n)
    t = lambda name: tb.tensor2torch(getattr(geo, name), clone=False, cast_uint_to_int=True)
    fwd, mask, order, pos, bwd, bwd_pos, bwd_order = (t(x) for x in ("indices_fwd", "mask_fwd", "order_fwd", "indices_fwd_pos",
                                                                     "indices_bwd", "indices_bwd_pos", "order_bwd"))
    bits = torch.zeros_like(row)
    for k in range(kv):
        at = (k // (ksize[1] * ksize[2]), k // ksize[2] % ksize[1], k % ksize[2])
        d = [a - s // 2 for a, s in zip(at, ksize)]
        inside = torch.ones(n, dtype=torch.bool, device="cuda")
        for c, e, s in zip(zyx, d, shape):
            inside &= (c + e >= 0) & (c + e < s)
        want = torch.where(inside, row + (d[0] * shape[1] + d[1]) * shape[2] + d[2], torch.full_like(row, -1))
        assert torch.equal(fwd[k], want) and torch.equal(bwd[kv - 1 - k], want), k
        assert torch.equal(pos[k], want[order.long()]) and torch.equal(bwd_pos[k], bwd[k][bwd_order.long()]), k
        bits |= torch.where(inside, 1 << k, 0).to(torch.int32)
    assert torch.equal(mask, bits[order.long()]) and torch.equal(torch.sort(order).values, row)
    with pytest.raises(RuntimeError):
        tb.sparse_conv(torch.zeros(n, 8, dtype=torch.float16, device="cuda"), torch.zeros(8, kv, 8, dtype=torch.float16, device="cuda"),
                       None, geo)


def test_a_geometry_shared_by_streams_and_threads():
    """Built on the default stream, used by two threads on streams of their own, each with its tensors, and on
    the default stream again; the threads' first passes make the validated calls at the same time."""
    import threading

    from cumm_amd import torch_bridge as tb
    print("case shared geometry", flush=True)
    coords, grid = H.small_cloud(51, 3000)
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, stride=(2, 2, 2))
    host = pairs.sparse_conv_pairs(coords, grid)
    c_in, k_out = 72, 88      # a kind of call that no other test has made
    gen = torch.Generator().manual_seed(4)
    jobs = []
    for _ in range(2):
        feat, weight = torch.randn(geo.n_in, c_in, generator=gen).half(), (torch.randn(k_out, 27, c_in, generator=gen) * 0.05).half()
        gout = torch.randn(geo.n_out, k_out, generator=gen).half()
        f_r, w_r = feat.float().requires_grad_(True), weight.float().requires_grad_(True)
        ref = _reference(f_r, w_r, None, host.indices_fwd, relu=False)
        (ref * gout.float()).sum().backward()
        jobs.append((feat.cuda(), weight.cuda(), gout.cuda(), (ref.detach(), f_r.grad, w_r.grad)))
    torch.cuda.synchronize()
    results, errors = [[], []], []

    def work(i, passes):
        try:
            feat, weight, gout, _ = jobs[i]
            for _ in range(passes):
                f_d, w_d = feat.clone().requires_grad_(True), weight.clone().requires_grad_(True)
                out = tb.sparse_conv(f_d, w_d, None, geo)
                out.backward(gout)
                results[i].append((out.detach(), f_d.grad, w_d.grad))
        except Exception as e:      # (a thread's exception is the test's)
            errors.append(e)

    def on_a_stream(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            work(i, 6)
        stream.synchronize()
    threads = [threading.Thread(target=on_a_stream, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    work(0, 1)
    torch.cuda.synchronize()
    assert errors == [] and [len(r) for r in results] == [7, 6]
    for got, (_, _, _, want) in zip(results, jobs):
        for passed in got:
            for a, b in zip(passed, want):
                assert float((a.float().cpu() - b).abs().max() / b.abs().max()) < 1e-2


@pytest.mark.parametrize("ksize,strided", [((3, 3, 3), False), ((3, 3, 3), True), ((5, 5, 5), False)])
def test_tables_by_position_are_whole_for_who_looks(ksize, strided):
    """The launches need entries only where a tile has the offset; the attribute is the whole table, and a layer that
    ran before gives the same bits after."""
    import torch
    from cumm_amd import pairs, torch_bridge as tb
    print("case whole tables", ksize, strided, flush=True)
    coords, grid = H.small_cloud(3, 3000, grid=(16, 60, 60))
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, ksize, (2, 2, 2) if strided else None, tuple(k // 2 for k in ksize))
    x = torch.randn(coords.shape[0], 64, device="cuda", dtype=torch.float16)
    w = torch.randn(64, geo.kv, 64, device="cuda", dtype=torch.float16) * 0.1
    before = tb.sparse_conv(x, w, None, geo)
    for side in ("fwd", "bwd"):
        table, order = H.host(getattr(geo, "indices_" + side)), H.host(getattr(geo, "order_" + side))
        np.testing.assert_array_equal(H.host(getattr(geo, "indices_%s_pos" % side)), pairs.pairs_by_position(table, order))
    assert torch.equal(before, tb.sparse_conv(x, w, None, geo))


def test_tables_by_position_read_on_another_stream_than_the_building_one():
    """The building stream is still busy when somebody on another one takes the tables, and is waited for only
    afterwards; and a geometry that a graph builds anew at every replay."""
    import torch
    from cumm_amd import pairs, torch_bridge as tb
    print("case whole tables, two streams", flush=True)
    coords, grid = H.small_cloud(3, 30000, grid=(16, 200, 200))
    coords = torch.as_tensor(coords, device="cuda")
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.randn(4096, 4096, device="cuda")

    def whole(geo, tables):
        for side, table in tables:
            by_row, order = H.host(getattr(geo, "indices_" + side)), H.host(getattr(geo, "order_" + side))
            np.testing.assert_array_equal(H.host(table), pairs.pairs_by_position(by_row, order))
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        for _ in range(10):
            busy @ busy
        geo = tb.SparseConvGeometry(coords, grid)
    with torch.cuda.stream(b):
        tables = [(side, getattr(geo, "indices_%s_pos" % side)) for side in ("fwd", "bwd")]
    b.wait_stream(a)
    torch.cuda.synchronize()
    whole(geo, tables)

    # (the same number of sites, elsewhere: runs of positions have other offsets)
    clouds = [coords] + [torch.as_tensor(H.small_cloud(s, 30000, grid=(16, 200, 200), sigma=30.0)[0], device="cuda") for s in (4, 5)]
    n = min(len(c) for c in clouds)
    clouds = [c[:n].contiguous() for c in clouds]
    now = clouds[0].clone()
    tb.SparseConvGeometry(now, grid)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        geo = tb.SparseConvGeometry(now, grid)
    for cloud in clouds:
        now.copy_(cloud)
        graph.replay()
        whole(geo, [(side, getattr(geo, "indices_%s_pos" % side)) for side in ("fwd", "bwd")])
