"""The torch bridge's native calls against its Python function: the same bits, the same refusals, and the parts of
autograd that a node of one's own has to keep (saved-tensor hooks, version checks, graphs kept and freed,
gradients nobody asked for, streams)."""
import pytest

import helpers as H

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _setup(ksize=3, strided=False, c=48, k=40, dtype=torch.float16, n=1500, seed=3):
    from cumm_amd import torch_bridge as tb
    coords, grid = H.small_cloud(seed, n)
    geo = tb.SparseConvGeometry(torch.as_tensor(coords, device="cuda"), grid, (ksize,) * 3, (2, 2, 2) if strided else None,
                                (ksize // 2,) * 3)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: (torch.randn(*s, generator=gen, device="cuda") * 0.2).to(dtype)
    return tb, geo, rnd(geo.n_in, c), rnd(k, ksize ** 3, c), rnd(k), rnd(geo.n_out, k)


def _grads(call, x, w, b, g, which=(True, True, True)):
    leaves = [t.detach().clone().requires_grad_(r) if t is not None else None for t, r in zip((x, w, b), which)]
    out = call(*leaves)
    asked = [t for t in leaves if t is not None and t.requires_grad]
    return (out.detach(),) + torch.autograd.grad(out, asked, g)


@pytest.mark.parametrize("ksize,strided,dtype", [(3, False, torch.float16), (3, True, torch.bfloat16), (5, False, torch.bfloat16)])
@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("k", [40, 72])      # (from 64 channels on the forward pass leaves its gate as bits)
def test_same_bits_as_the_python_function(ksize, strided, dtype, relu, with_bias, k):
    print("case native", ksize, strided, dtype, relu, with_bias, k, flush=True)
    tb, geo, x, w, b, g = _setup(ksize, strided, k=k, dtype=dtype)
    assert geo._native.tables() == {**geo._ptr, **{"reduced_%d" % w: a for w, a in geo._reduced_at.items()}}
    b = b if with_bias else None
    python = lambda *t: tb._SparseConvFunction.apply(*t, geo, relu)
    native = lambda *t: tb._native().forward(*t, geo, geo._native, relu)
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        want = _grads(python, x, w, b, g)
        got = _grads(native, x, w, b, g)
        assert len(got) == len(want) and all(torch.equal(a, c) for a, c in zip(got, want))
        # strided operands and gradients; gradients of some only
        wide = torch.empty(w.shape[0], w.shape[1], 2 * w.shape[2], dtype=w.dtype, device="cuda")[:, :, ::2].copy_(w)
        got = _grads(native, torch.stack([x, x], 1)[:, 0], wide, b, torch.stack([g, g], 2)[:, :, 1])
        assert all(torch.equal(a, c) for a, c in zip(got, want))
        for which in ((True, False, False), (False, True, False), (False, False, True)):
            if which[2] and not with_bias:
                continue
            got = _grads(native, x, w, b, g, which)
            assert torch.equal(got[1], want[1 + which.index(True)])
    finally:
        torch.use_deterministic_algorithms(False)
    with torch.no_grad():
        assert not tb.sparse_conv(x.requires_grad_(True), w, b, geo, relu).requires_grad


@pytest.fixture
def no_python():
    """A native backward pass that falls back to Python fails."""
    from cumm_amd import torch_bridge as tb

    def fell_back(*a):
        raise AssertionError("the backward pass went to Python")
    tb._native().set_backward(fell_back)
    yield
    tb._native().set_backward(tb._backward)


@pytest.mark.parametrize("ksize,strided,dtype", [(3, False, torch.float16), (3, True, torch.bfloat16), (5, False, torch.bfloat16)])
@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("k", [40, 64])
def test_a_known_backward_pass_stays_native(no_python, ksize, strided, dtype, relu, with_bias, deterministic, k):
    print("case stays native", ksize, strided, dtype, relu, with_bias, deterministic, k, flush=True)
    tb, geo, x, w, b, g = _setup(ksize, strided, k=k, dtype=dtype)
    b = b if with_bias else None
    torch.use_deterministic_algorithms(deterministic, warn_only=True)
    try:
        want = _grads(lambda *t: tb._SparseConvFunction.apply(*t, geo, relu), x, w, b, g)
        _, later, *_ = _setup(ksize, strided, k=k, dtype=dtype)      # (another geometry of the kind: only what was remembered serves it)
        got = _grads(lambda *t: tb._native().forward(*t, later, later._native, relu), x, w, b, g)
        # (the weight gradient's atomics: sums in any order, and one rounding to the type)
        for i, (a, c) in enumerate(zip(got, want)):
            if i == 2 and not deterministic:
                assert (a.float() - c.float()).norm() <= 2.0 ** -8 * c.float().norm()
            else:
                assert torch.equal(a, c)
    finally:
        torch.use_deterministic_algorithms(False)


def test_a_gradient_that_nobody_has(no_python):
    """The node is given no gradient at all: zeros."""
    class Nothing(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            ctx.set_materialize_grads(False)
            return t * 1

        @staticmethod
        def backward(ctx, grad):
            return None
    tb, geo, x, w, b, g = _setup()
    _grads(lambda *t: tb._SparseConvFunction.apply(*t, geo, True), x, w, b, g)
    leaves = [t.detach().clone().requires_grad_(True) for t in (x, w, b)]
    out = tb.sparse_conv(*leaves, geo, True)
    for got, leaf in zip(torch.autograd.grad(Nothing.apply(out), leaves, g), leaves):
        assert got.shape == leaf.shape and got.dtype == leaf.dtype and not got.any()


@pytest.mark.parametrize("k", [40, 64, 72])
def test_what_autograd_keeps(k):
    print("case what autograd keeps", k, flush=True)
    tb, geo, x, w, b, g = _setup(k=k)
    conv = lambda *t: tb.sparse_conv(*t, geo, True)
    want = _grads(conv, x, w, b, g)
    x, w, b = (t.detach().clone().requires_grad_(True) for t in (x, w, b))
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.data_ptr()) or t.cpu(), lambda t: t.cuda()):
        out = conv(x, w, b)
    assert out.grad_fn.name() == "_SparseConvFunctionBackward" and len(packed) == 3
    got = torch.autograd.grad(out, (x, w, b), g, retain_graph=True)
    assert all(torch.equal(a, c) for a, c in zip(got[::2], want[1::2]))
    again = torch.autograd.grad(out, (x, w, b), g)
    assert torch.equal(again[0], got[0])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, (x, w, b), g)
    for changed in (lambda o: o.add_(1), lambda o: w.data_ptr() and w.detach().add_(1)):
        out = conv(x, w, b)
        with torch.no_grad():
            changed(out)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(out, (x, w, b), g)
    # a graph that is kept, without hooks (the weights are others by now)
    want = _grads(conv, x, w, b, g)
    out = conv(x, w, b)
    for keep in (True, False):
        got = torch.autograd.grad(out, (x, w, b), g, retain_graph=keep)
        assert all(torch.equal(a, c) for a, c in zip(got[::2], want[1::2]))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, (x, w, b), g)
    # a gradient that nobody computed is zero
    out = conv(x, w, b)
    zero = torch.autograd.grad(out, (x, w, b), torch.zeros_like(out))
    assert all(not t.any() for t in zero)


@pytest.mark.parametrize("ksize,strided,k,dtype", [(3, False, 64, torch.float16), (3, True, 72, torch.bfloat16), (5, False, 128, torch.float16),
                                                   (3, False, 40, torch.float16)])
def test_a_bias_gradient_is_added_up_in_one_order(ksize, strided, k, dtype):
    """Gradients of which the large ones cancel, so that another order of the rows gives other bits: the Python
    function, a native pass with the gate's bits, one whose output went through saved-tensor hooks."""
    print("case one order of a bias gradient", ksize, strided, k, dtype, flush=True)
    tb, geo, x, w, b, g = _setup(ksize, strided, k=k, dtype=dtype, n=6000)
    python = lambda *t: tb._SparseConvFunction.apply(*t, geo, True)
    native = lambda *t: tb._native().forward(*t, geo, geo._native, True)
    y = python(x, w, b)
    turn = (y > 0).cumsum(0) % 4
    g = torch.where(turn == 1, 1000.0, torch.where(turn == 2, -1000.0, g.float())).to(dtype)
    want = _grads(python, x, w, b, g)[3]
    exact = torch.where(y > 0, g, 0).double().sum(0)
    assert ((want.double() - exact).abs() < 0.02 * exact.abs().max()).all()      # (2000 terms of 1000 in fp32, and one rounding)
    for _ in range(2):
        assert torch.equal(_grads(native, x, w, b, g)[3], want)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), lambda t: t):
        assert torch.equal(_grads(native, x, w, b, g)[3], want)


@pytest.mark.parametrize("k", [40, 64])
def test_a_node_used_by_two_threads_while_one_frees_it(k):
    """A backward pass that frees the graph, beside calls of the node from another thread: each call has the right
    gradients or the error of a freed graph."""
    import threading
    print("case two threads", k, flush=True)
    tb, geo, x, w, b, g = _setup(k=k)
    want = _grads(lambda *t: tb.sparse_conv(*t, geo, True), x, w, b, g)
    leaves = [t.detach().clone().requires_grad_(True) for t in (x, w, b)]
    torch.cuda.synchronize()
    for trip in range(20):
        out = tb.sparse_conv(*leaves, geo, True)
        start, calls, wrong = threading.Barrier(2), [0, 0], []

        def call(freeing):
            start.wait()
            for _ in range(1 if freeing else 8):
                try:
                    got = torch.autograd.grad(out, leaves, g) if freeing else out.grad_fn(g)
                    torch.cuda.synchronize()
                    calls[freeing] += 1
                    if not (torch.equal(got[0], want[1]) and torch.equal(got[2], want[3])):
                        wrong.append((trip, freeing))
                except RuntimeError as e:
                    if freeing or "second time" not in str(e):
                        wrong.append((trip, freeing, str(e)))
        threads = [threading.Thread(target=call, args=(f,)) for f in (True, False)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong and calls[1] == 1


def test_what_is_left_to_python():
    import torch.autograd.forward_ad as fwad
    tb, geo, x, w, b, g = _setup()
    tb.sparse_conv(x, w, b, geo)
    native = lambda *t: tb._native().forward(*t, geo, geo._native, False)
    assert native(x, w, b) is not None
    assert native(x[:-1], w, b) is None and native(x, w[:, :26], b) is None and native(x, w, b[:-1]) is None
    assert native(x.cpu(), w, b) is None and native(x.float(), w, b) is None and native(x, w.bfloat16(), b) is None
    assert native(x[:, :0], w[:, :, :0], b) is None
    with fwad.dual_level():
        dual = fwad.make_dual(x, torch.ones_like(x))
        assert native(dual, w, b) is None
        with pytest.raises(Exception):
            tb.sparse_conv(dual, w, b, geo)
    with pytest.raises(Exception):
        torch.func.vmap(lambda t: tb.sparse_conv(t, w, b, geo))(torch.stack([x, x]))
    with pytest.raises(ValueError):
        tb.sparse_conv(x[:-1], w, b, geo)
    with pytest.raises(ValueError):
        tb.sparse_conv(x, w.cpu(), b, geo)


@pytest.mark.parametrize("k", [40, 64])
def test_on_another_stream_and_after_the_geometry(k):
    print("case another stream", k, flush=True)
    tb, geo, x, w, b, g = _setup(k=k)
    conv = lambda *t: tb.sparse_conv(*t, geo, True)
    want = _grads(conv, x, w, b, g)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    x, w, b = (t.detach().clone().requires_grad_(True) for t in (x, w, b))
    with torch.cuda.stream(stream):
        out = conv(x, w, b)
        del geo
        got = torch.autograd.grad(out, (x, w, b), g)
    stream.synchronize()
    assert torch.equal(out.detach(), want[0]) and torch.equal(got[0], want[1]) and torch.equal(got[2], want[3])


@pytest.mark.parametrize("k", [40, 72])
def test_compiled_autograd(k):
    """A backward pass under torch's compiled autograd (its graph run as it is): the gradients of the ordinary one, also
    where the graph of one layer serves the next - another geometry of the same sizes."""
    from torch._dynamo import compiled_autograd
    for ksize, strided, relu, with_bias in ((3, False, True, True), (3, True, False, False), (5, False, True, False)):
        for seed in (3, 4):
            print("case compiled autograd", ksize, strided, relu, with_bias, seed, k, flush=True)
            tb, geo, x, w, b, g = _setup(ksize, strided, k=k, seed=seed)
            conv = lambda *t: tb.sparse_conv(*t, geo, relu)
            leaves = lambda: [t.detach().clone().requires_grad_(True) for t in ((x, w, b) if with_bias else (x, w))]
            of = lambda ts: tuple(ts) + (() if with_bias else (None,))
            torch.use_deterministic_algorithms(True, warn_only=True)
            try:
                one, two = leaves(), leaves()
                conv(*of(one)).backward(g)
                out = conv(*of(two))
                assert out.grad_fn.name() == "_SparseConvFunctionBackward"
                with compiled_autograd._enable(lambda graph: torch.compile(graph, backend="eager")):
                    out.backward(g)
                assert all(torch.equal(p.grad, q.grad) for p, q in zip(one, two))
            finally:
                torch.use_deterministic_algorithms(False)


@pytest.mark.parametrize("ksize,strided", [(3, False), (3, True), (5, False)])
@pytest.mark.parametrize("k", [40, 72])
def test_without_the_native_half(monkeypatch, ksize, strided, k):
    """On a machine without a host compiler the bridge's own functions make every call: the same tables and bits."""
    print("case without native", ksize, strided, k, flush=True)
    tb, geo, x, w, b, g = _setup(ksize, strided, k=k)
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        want = _grads(lambda *t: tb.sparse_conv(*t, geo, True), x, w, b, g)
        monkeypatch.setattr(tb, "_native_module", False)
        _, own, *_ = _setup(ksize, strided, k=k)
        assert own._native is None and own.out_shape == geo.out_shape and torch.equal(own.out_coords, geo.out_coords)
        for name in tb.SparseConvGeometry._TABLES:
            assert (H.host(getattr(own, name)) == H.host(getattr(geo, name))).all(), name
        got = _grads(lambda *t: tb.sparse_conv(*t, own, True), x, w, b, g)
        assert all(torch.equal(a, c) for a, c in zip(got, want))
    finally:
        torch.use_deterministic_algorithms(False)


def test_two_first_calls_at_once(monkeypatch):
    """Two threads' first calls of a kind - a forward pass and, while it is being remembered, a backward one: each
    pass of a later geometry is what it is."""
    import threading
    tb, geo, x, w, b, g = _setup(c=56, k=88)
    native, met = tb._native(), []
    remember = native.remember

    def both(*args):
        if not met:
            met.append(args)
            needed = (True, False, False)
            other = threading.Thread(target=tb._backward, args=(geo, x, w, None, g, needed, False, False, 64))
            other.start()
            other.join()
            met.append(None)
        return remember(*args)
    monkeypatch.setattr(native, "remember", both)
    tb._SparseConvFunction.apply(x, w, b, geo, False)
    assert len(met) == 2
    _, later, x, w, b, g = _setup(c=56, k=88)
    assert native.forward(x, w, b, later, later._native, False) is not None
    assert [key[0] for key in later._launches] == ["fwd"]


def test_one_order_where_reproducible_results_are_asked_for():
    """A scene's features alone and in a batch of 60 of it - few tiles, many tiles - under torch's switch: the same bits,
    natively and from Python; of the input gradient too."""
    tb, _, x, w, b, g = _setup(c=64, k=64)
    coords, grid = H.small_cloud(3, 1500)
    scene = torch.as_tensor(coords, device="cuda")
    batch = scene.repeat(60, 1)
    batch[:, 0] = torch.arange(60, device="cuda", dtype=torch.int32).repeat_interleave(len(scene))
    alone, many = (tb.SparseConvGeometry(c, grid, batch_size=n) for c, n in ((scene, 1), (batch.contiguous(), 60)))
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        for trip in range(2):      # (a first call, and one in native code)
            one = _grads(lambda *t: tb.sparse_conv(*t, alone, False), x, w, b, g)
            all_ = _grads(lambda *t: tb.sparse_conv(*t, many, False), x.repeat(60, 1), w, b, g.repeat(60, 1))
            for got, want in zip(all_[:2], one[:2]):
                assert all(torch.equal(part, want) for part in got.view(60, len(scene), -1)), trip
    finally:
        torch.use_deterministic_algorithms(False)
