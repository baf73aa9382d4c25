"""The calls that are made in C++ (difflogic_amd._host) against the Python functions they stand in for: the same kernels, so the
same bits, for every form of argument they take, and the same refusals for the others."""
import pytest
import torch

pytestmark = pytest.mark.gpu

F16, F32, F64 = torch.float16, torch.float32, torch.float64


@pytest.fixture(scope="module")
def dl():
    import difflogic_amd
    return difflogic_amd


def _python_only(monkeypatch, dl):
    for name in ("train_layer", "group_sum", "eval_layer", "net_forward", "eval_weights", "gate_ids_folded", "pack_rows", "count_rows",
                 "forward_logits", "backward_both", "backward_logits", "forward_group_sum"):
        monkeypatch.setattr(dl._host, name, lambda *a: None)


def _answered(monkeypatch, dl):
    """Counts the native calls that answered: {name: times}, train_layer along a schedule as "train_layer walked"."""
    counts = {}

    def counted(name, fn):
        def call(*args):
            out = fn(*args)
            if out is not None:
                key = name + (" walked" if name == "train_layer" and args[7] else "")
                counts[key] = counts.get(key, 0) + 1
            return out
        return call

    for name in ("train_layer", "group_sum", "eval_layer", "net_forward", "net_backward", "eval_weights", "gate_ids_folded", "pack_rows",
                 "count_rows", "forward_logits", "backward_both", "backward_logits", "forward_group_sum"):
        monkeypatch.setattr(dl._host, name, counted(name, getattr(dl._host, name)))
    return counts


def _views(x):
    """x [B, in] as it is, as the transposed view a layer returns, and as columns of a wider matrix."""
    wide = torch.zeros(x.shape[0], 2 * x.shape[1], dtype=x.dtype, device=x.device)
    wide[:, ::2] = x
    return x, x.t().contiguous().t(), wide[:, ::2]


@pytest.mark.parametrize("dtype,wdtype", [(F32, F32), (F16, F32), (F64, F32), (F16, F16), (F64, F64)])
@pytest.mark.parametrize("in_dim,out_dim,batch", [(20, 30, 1), (64, 50, 3), (300, 200, 100),
                                                  (4200, 20000, 33),       # a schedule, but too many inputs at several positions
                                                  (20000, 20000, 33),      # one-pass backward along the schedule
                                                  (33000, 33000, 30)])     # every kernel along it
def test_layer_and_group_sum(dl, monkeypatch, dtype, wdtype, in_dim, out_dim, batch):
    torch.manual_seed(batch)
    layer, total = dl.LogicLayer(in_dim, out_dim, grad_factor=1.5).train(), dl.GroupSum(10, 7.0)
    layer.weights = torch.nn.Parameter(layer.weights.detach().to(wdtype))
    x0 = torch.rand(batch, in_dim, device="cuda").to(dtype)
    gy, gs = torch.randn(batch, out_dim, device="cuda").to(dtype), torch.randn(batch, 10, device="cuda").to(dtype)

    def run():
        out, alone = [], []                               # alone: gradients of the weights in a task that asks for nothing else
        for view in range(3):
            for want_x, want_w in ((True, True), (True, False), (False, True), (False, False)):
                layer.weights.requires_grad_(want_w)
                layer.weights.grad = None
                x = x0.detach().clone().requires_grad_(want_x)
                y = layer(_views(x)[view])
                assert y.requires_grad == (want_x or want_w) and y.stride() == (1, batch)
                out.append(y.detach())
                if y.requires_grad:
                    torch.autograd.backward((y, total(y)), (gy, gs[:1].expand(batch, 10)), retain_graph=True)
                    out += [t.grad.clone() for t in (x, layer.weights) if t.grad is not None]
                    if want_x:
                        out += torch.autograd.grad(y, x, gy, retain_graph=True)
                    if want_w:
                        alone += torch.autograd.grad(y, layer.weights, gy, retain_graph=True)
        with torch.no_grad():
            out.append(layer(x0))
        layer.eval()
        out += [layer(v).detach() for v in _views(x0.clone().requires_grad_())] + [total(layer(x0))]
        layer.train()
        layer.weights.requires_grad_(True)
        return out, alone

    counts = _answered(monkeypatch, dl)
    native, alone = run()
    assert not native[-1].requires_grad
    assert counts["eval_layer"] == 4 and counts["group_sum"] > 0
    if in_dim < 4096:
        assert counts["train_layer"] == 13 and "train_layer walked" not in counts         # the four wants of three views, no_grad
    elif in_dim < out_dim:
        assert "train_layer" not in counts and "train_layer walked" not in counts and counts["backward_both"] > 0
    else:
        assert "train_layer" not in counts and counts["train_layer walked"] == 3          # where both gradients are wanted
    _python_only(monkeypatch, dl)
    want, want_alone = run()
    for u, v in zip(native, want, strict=True):
        assert u.dtype == v.dtype and u.shape == v.shape and torch.equal(u, v)
    for u, v in zip(alone, want_alone, strict=True):
        # (Python forms both gradients in one pass along a schedule, which adds the terms of short rows in another order: each
        # of the 16 sums has `batch` terms of at most |gy|, and the softmax multiplies by at most 1)
        eps = 2.0 ** -53 if dtype == F64 and wdtype == F64 else 2.0 ** -24
        bound = 4 * (batch + 2) * eps * gy.double().abs().sum(0)[:, None] + (2.0 ** -10 if wdtype == F16 else 0) * v.double().abs()
        assert u.dtype == v.dtype and u.shape == v.shape
        assert torch.equal(u, v) if in_dim < 20000 else bool(((u.double() - v.double()).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [F32, F16, F64])
@pytest.mark.parametrize("want_x,frozen", [(False, ()), (True, (1,)), (True, (0, 1, 2)), (False, (0,)), (False, (2,))])
def test_fused_net(dl, monkeypatch, dtype, want_x, frozen):
    torch.manual_seed(3)
    net = torch.nn.Sequential(dl.LogicLayer(60, 90, grad_factor=2.0), dl.LogicLayer(90, 120), dl.LogicLayer(120, 80), dl.GroupSum(4, 3.0))
    for i in frozen:
        net[i].weights.requires_grad_(False)
    fused = dl.fuse_for_training(net).train()
    x0, g = torch.rand(37, 60, device="cuda").to(dtype), torch.randn(37, 4, device="cuda").to(dtype)

    def run():
        fused.zero_grad(set_to_none=True)
        x = x0.clone().requires_grad_(want_x)
        y = fused(x)
        y.backward(g, retain_graph=True)
        first = [p.grad.clone() for p in fused.parameters() if p.grad is not None]
        y.backward(g)                                                 # a retained graph is walked again: gradients add up
        return [y.detach()] + ([x.grad] if want_x else []) + first + [p.grad for p in fused.parameters() if p.grad is not None]

    counts = _answered(monkeypatch, dl)
    native = run()
    assert counts["net_forward"] == 1 and counts["net_backward"] == 2
    _python_only(monkeypatch, dl)
    for u, v in zip(native, run(), strict=True):
        assert torch.equal(u, v)


def test_hooks_streams_and_freed_graphs(dl):
    torch.manual_seed(4)
    layer = dl.LogicLayer(300, 200).train()
    x = torch.rand(50, 300, device="cuda", requires_grad=True)
    layer(x).sum().backward()
    want = x.grad.clone(), layer.weights.grad.clone()
    x.grad = layer.weights.grad = None
    with torch.autograd.graph.save_on_cpu():
        y = layer(x)
    y.sum().backward()
    assert torch.equal(x.grad, want[0]) and torch.equal(layer.weights.grad, want[1])
    with pytest.raises(RuntimeError):
        y.sum().backward()                                            # the graph is freed
    y = layer(x)
    with torch.no_grad():
        x.add_(0)                                                     # (x itself is not what was saved: a transposed copy is)
    y.sum().backward()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    x.grad = layer.weights.grad = None
    with torch.cuda.stream(side):
        layer(x).sum().backward()
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(x.grad, want[0]) and torch.equal(layer.weights.grad, want[1])


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("change", ["dtype", "rows", "device"])
def test_saved_tensors_that_hooks_changed_are_refused(dl, fused, change):
    net = torch.nn.Sequential(dl.LogicLayer(30, 40), dl.LogicLayer(40, 50), dl.GroupSum(10)).train()
    net = dl.fuse_for_training(net) if fused else net
    x = torch.rand(5, 30, device="cuda", requires_grad=True)
    changes = {"dtype": lambda t: t.half(), "rows": lambda t: t[1:].contiguous(), "device": lambda t: t.cpu()}
    probabilities = lambda t: t.dim() == 2 and t.shape[1] == 16
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: changes[change](t) if probabilities(t) else t):
        y = net(x)
    with pytest.raises(RuntimeError):
        y.sum().backward()


def test_what_is_refused_stays_refused(dl):
    layer = dl.LogicLayer(30, 40).train()
    good = torch.rand(5, 30, device="cuda")
    for bad, error in ((torch.rand(5, 31, device="cuda"), AssertionError), (torch.rand(5, 30), AssertionError),
                       (torch.rand(30, device="cuda"), AssertionError), (good.int(), (RuntimeError, TypeError))):
        with pytest.raises(error):
            layer(bad).sum().backward()
    with pytest.raises(RuntimeError):
        torch.func.vmap(layer)(good[None])
    with pytest.raises(RuntimeError):
        torch.func.jvp(layer, (good,), (good,))
    with pytest.raises(AssertionError):
        dl.GroupSum(7)(layer(good))
    assert layer(torch.rand(0, 30, device="cuda")).shape == (0, 40)

    class Sub(torch.Tensor):
        pass

    assert torch.equal(layer(good.as_subclass(Sub)).as_subclass(torch.Tensor), layer(good))


@pytest.mark.parametrize("batch,bits", [(1, 8), (100, 32), (129, 64), (5000, 16)])
@pytest.mark.parametrize("top", [1000, 1200])
def test_packed_layers(dl, monkeypatch, batch, bits, top):
    torch.manual_seed(batch)
    net = torch.nn.Sequential(dl.LogicLayer(100, 1200), dl.LogicLayer(1200, top), dl.GroupSum(10)).eval()
    x = torch.rand(batch, 100, device="cuda") < 0.3
    counts = _answered(monkeypatch, dl)
    native = net(dl.PackBitsTensor(x, bit_count=bits))
    if top < 1200:                                    # a layer that narrows is deferred
        assert counts == {"pack_rows": 1, "eval_weights": 1, "gate_ids_folded": 1}
    elif batch <= 129:
        assert counts == {"pack_rows": 1, "eval_weights": 2, "count_rows": 1}
    else:
        assert counts["eval_weights"] + counts.get("gate_ids_folded", 0) == 2
    _python_only(monkeypatch, dl)
    assert torch.equal(native, net(dl.PackBitsTensor(x, bit_count=bits)))


@pytest.mark.parametrize("train", [True, False])
def test_compiled_modules(dl, train):
    """The compiler sees what it saw without the native calls: GroupSum on row-major scores is one graph, a net of the kernels
    runs with breaks around them."""
    torch.manual_seed(6)
    torch._dynamo.reset()
    total, x = dl.GroupSum(5, 3.0), torch.rand(7, 30, device="cuda")
    assert torch.equal(torch.compile(total, fullgraph=True, backend="eager")(x), total(x))
    net = torch.nn.Sequential(dl.LogicLayer(30, 40), dl.LogicLayer(40, 50), total).train(train)
    assert torch.equal(torch.compile(net, backend="eager")(x), net(x))


def test_group_sum_converts_tau_where_the_kernels_take_the_call(dl):
    """A tau per class broadcasts over scores that go to the torch formula, and the device is not waited for there."""
    x = torch.rand(7, 30, device="cuda")
    tau = torch.arange(1.0, 6.0, device="cuda")
    want = x.reshape(7, 5, 6).sum(-1)
    assert torch.equal(dl.GroupSum(5, tau)(x), want / tau)
    torch.cuda.set_sync_debug_mode("error")
    try:
        got = dl.GroupSum(5, tau[1])(x)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    assert torch.equal(got, want / tau[1])


def test_counts_of_rows_padded_by_more_than_31_bits(dl):
    """pad_len reaches the kernel whole: cut to 32 bits, the kernel would write far more samples than the result has."""
    words = (1 << 26) + 3
    b = torch.zeros(2, words, dtype=torch.int64, device="cuda")
    b[:, :4] = torch.randint(-2 ** 62, 2 ** 62, (2, 4), device="cuda")
    for samples in (70, 192, 200):
        got = dl.difflogic_cuda.groupbitsum(b, words * 64 - samples, 1)
        assert got.shape == (samples, 1)
        assert torch.equal(got, dl.difflogic_cuda.groupbitsum(b[:, :4].contiguous(), 256 - samples, 1))
