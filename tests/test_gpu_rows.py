"""Training kernels on rows that are not whole 16-byte vectors: the last vector of a row overlaps the one before
it, so what matters is that every element is written and that sums over the batch count it once.  Against fp64
arithmetic on the values as rounded to the activations' dtype, with the training path's tolerances."""
import pytest
import torch

from oracle import float_oracle as fo
from tests.helpers import within_budget

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.float32, torch.float64]
RTOL = {torch.float16: 4e-3, torch.float32: 1e-5, torch.float64: 1e-12}


@pytest.fixture(scope="module")
def ext():
    import difflogic_amd
    return difflogic_amd.difflogic_cuda


def _batches(dtype):
    """Row lengths around the edges: one vector and one element more, 32 / 64 / 128 / 256 vectors (the lane, register
    and segment limits of the kernels) less one element and more by one, and a last segment of one partial vector."""
    v = 16 // dtype.itemsize
    return [v + 1, 2 * v - 1, 32 * v - 1, 32 * v + 1, 64 * v + 1, 128 * v + 1, 256 * v - 1, 256 * v + 1]


CASES = [(d, n) for d in DTYPES for n in _batches(d)]


@pytest.mark.parametrize("dtype,batch", CASES)
def test_layer_kernels_on_rows_of_any_length(ext, monkeypatch, dtype, batch):
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)     # exercise the overflow rows on this wiring
    in_dim, out_dim, k = 30, 44, 4
    g = torch.Generator().manual_seed(batch)
    a = torch.randint(0, in_dim, (out_dim,), generator=g)
    b = torch.randint(0, in_dim, (out_dim,), generator=g)
    b[1] = a[1]
    x = torch.rand(in_dim, batch, generator=g).to(dtype)
    gy = torch.randn(out_dim, batch, generator=g).to(dtype)
    logits = torch.randn(out_dim, 16, generator=g).to(dtype)
    rtol = RTOL[dtype]

    def close(got, want64, ref32=None):
        assert got.dtype == dtype
        ok, report = within_budget(got, want64, ref32, rtol)
        assert ok, report

    l64 = logits.double().requires_grad_()
    x64 = x.double().t().contiguous().requires_grad_()
    y64 = fo.layer_forward_sequential(x64, a, b, torch.softmax(l64, -1))           # [B, out]
    (y64 * gy.double().t()).sum().backward()
    xd, ad, bd, ld, gd = x.cuda(), a.cuda(), b.cuda(), logits.cuda(), gy.cuda()
    sched = ext.schedule_for(ad, bd, in_dim)
    from difflogic_amd.functional import build_reverse_index
    start, idx = (t.cuda() for t in build_reverse_index(a, b, in_dim))
    for schedule in (None, sched):
        y, probs = ext.forward_logits(xd, ad, bd, ld, schedule)
        close(y, y64.t())
        close(ext.backward_logits(xd, ad, bd, gd, probs, schedule), l64.grad)
    close(ext.backward_x(xd, ad, bd, probs, gd, start, idx, 1.5), 1.5 * x64.grad.t())
    gl, gx = ext.backward_chained(xd, probs, gd, sched, 1.5, softmax_backward=True, any_rows=True)
    close(gl, l64.grad)
    close(gx, 1.5 * x64.grad.t())

    # the layer with the GroupSum after it, and the GroupSum alone
    sums = fo.group_sum(y64.detach().to(dtype).double(), k, 3.0)
    close(ext.forward_group_sum(xd, ad, bd, ld, k, 3.0)[0], sums)
    close(ext.group_sum_forward(y, k, 3.0), sums)
    gc = torch.randn(k, batch, generator=g).to(dtype)
    l64.grad = x64.grad = None
    yy = fo.layer_forward_sequential(x64, a, b, torch.softmax(l64, -1))
    (yy * gc.double().repeat_interleave(out_dim // k, 0).t()).sum().backward()
    for schedule in (None, sched):
        gl, gx = ext.backward_group_sum(xd, ad, bd, probs, gc.cuda(), start, idx, schedule, 1.0, True, True)
        close(gl, l64.grad)
        close(gx, x64.grad.t())
    back = ext.group_sum_backward(gc.t().contiguous().cuda(), out_dim, 1.0)
    assert torch.equal(back.cpu(), gc.repeat_interleave(out_dim // k, 0))


@pytest.mark.parametrize("dtype,batch", [c for c in CASES if c[1] * c[0].itemsize <= 2048 + 16])
def test_two_layers_at_once_on_rows_of_any_length(ext, monkeypatch, dtype, batch):
    """forward_logits_lower and backward_chained_lower against the two layers run one after the other."""
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    in0, in_dim, out_dim = 20, 30, 44
    g = torch.Generator().manual_seed(batch)
    draw = lambda hi, n: torch.randint(0, hi, (n,), generator=g).cuda()  # noqa: E731
    a0, b0, a, b = draw(in0, in_dim), draw(in0, in_dim), draw(in_dim, out_dim), draw(in_dim, out_dim)
    x0 = torch.rand(in0, batch, generator=g).to(dtype).cuda()
    l0 = torch.randn(in_dim, 16, generator=g).to(dtype).cuda()
    l1 = torch.randn(out_dim, 16, generator=g).to(dtype).cuda()
    gy = torch.randn(out_dim, batch, generator=g).to(dtype).cuda()
    sched = ext.schedule_for(a, b, in_dim)
    y1, p0 = ext.forward_logits(x0, a0, b0, l0)
    y2, p1 = ext.forward_logits(y1, a, b, l1)
    rtol = RTOL[dtype]
    ok = lambda got, want: within_budget(got, want, None, rtol)[0]  # noqa: E731
    if batch * dtype.itemsize <= 2048:
        got = ext.forward_logits_lower(x0, a0, b0, l0, l1, sched, any_rows=True)
        assert ok(got[0], y2) and ok(got[2], p1)
    gw, gx = ext.backward_chained(y1, p1, gy, sched, softmax_backward=True, any_rows=True)
    gw0 = ext.backward_logits(x0, a0, b0, gx, p0)
    for x in (y1, None) if dtype != torch.float16 else (y1,):        # None: the inner rows are recomputed
        both = ext.backward_chained_lower(x, p1, gy, sched, x0, a0, b0, p0, softmax_backward=True, any_rows=True)
        assert ok(both[0], gw) and ok(both[1], gw0)


@pytest.mark.parametrize("dtype,wdtype", [(d, d) for d in DTYPES] + [(torch.float16, torch.float32), (torch.float64, torch.float32)])
@pytest.mark.parametrize("in_dim,out_dim,batch", [(1, 1, 1), (30, 44, 3), (5, 9, 17), (33, 50, 128), (30, 44, 515), (64, 40, 2048),
                                                  (20, 24, 4100), (12, 16, 8196), (12, 16, 16392)])
def test_both_gradients_in_one_launch(ext, dtype, wdtype, in_dim, out_dim, batch):
    """backward_both is backward_x and backward_w / backward_logits, bit for bit; rows of every kind, one and several
    column tiles, the batch split over the workgroup's waves, a layer under a GroupSum."""
    from difflogic_amd.functional import build_reverse_index
    g = torch.Generator().manual_seed(batch + out_dim)
    a, b = (torch.randint(0, in_dim, (out_dim,), generator=g) for _ in range(2))
    start, idx = (t.cuda() for t in build_reverse_index(a, b, in_dim))
    a, b = a.cuda(), b.cuda()
    x = torch.rand(in_dim, batch, generator=g).to(dtype).cuda()
    gy = torch.randn(out_dim, batch, generator=g).to(dtype).cuda()
    p = torch.softmax(torch.randn(out_dim, 16, generator=g), -1).to(wdtype).cuda()
    gx = ext.backward_x(x, a, b, p, gy, start, idx, 1.5)
    gw, gx2 = ext.backward_both(x, a, b, p, gy, start, idx, 1.5, softmax_backward=True)
    assert torch.equal(gx2, gx) and torch.equal(gw, ext.backward_logits(x, a, b, gy, p))
    if wdtype == dtype:
        gw, gx2 = ext.backward_both(x, a, b, p, gy, start, idx, 1.5)
        assert torch.equal(gx2, gx) and torch.equal(gw, ext.backward_w(x, a, b, gy))
        k = 4 if out_dim % 4 == 0 else 1
        gc = torch.randn(k, batch, generator=g).to(dtype).cuda()
        gl, gx2 = ext.backward_group_sum(x, a, b, p, gc, start, idx, None, 1.5, True, True)
        assert torch.equal(gx2, ext.backward_group_sum(x, a, b, p, gc, start, idx, None, 1.5, True, False)[1])
        assert torch.equal(gl, ext.backward_group_sum(x, a, b, p, gc, start, idx, None, 1.5, False, True)[0])


def test_layers_walk_their_schedule_where_their_rows_are_long(ext, monkeypatch):
    """A layer too narrow for its schedule takes it on a batch whose rows are long enough; outputs and gradients are those
    of the other kernels.  A schedule that has not been built is not built under graph capture."""
    import difflogic_amd as dl
    torch.manual_seed(2)
    layer = dl.LogicLayer(5000, 6000, grad_factor=1.5)
    # (the forward kernel of 6000 neurons gains from 24 MB of rows on, batch 1000; up to then, 8.9 -> 11.5 us at 668, it loses)
    long, short = torch.rand(1024, 5000, device="cuda"), torch.rand(600, 5000, device="cuda")
    graph, fresh = torch.cuda.CUDAGraph(), dl.LogicLayer(5000, 6000).eval()
    layer(short), torch.cuda.synchronize()
    with torch.cuda.graph(graph), torch.no_grad():
        out = fresh(long)
    graph.replay()
    assert ext.built_schedule(*fresh.indices, 5000) is None
    with torch.no_grad():
        assert torch.equal(out, fresh(long)) and ext.built_schedule(*fresh.indices, 5000) is not None
    assert layer._train_schedule(short.t()) is None and layer._train_schedule(long.t()) is not None
    gy = torch.randn(1024, 6000, device="cuda")
    grads = []
    for least in (layer._CHAIN_MIN_BYTES, 1 << 60):
        monkeypatch.setattr(dl.LogicLayer, "_CHAIN_MIN_BYTES", least)
        x = long.clone().requires_grad_()
        layer.weights.grad = None
        y = layer(x)
        y.backward(gy)
        grads.append((y.detach(), layer.weights.grad, x.grad))
    (y0, w0, x0), (y1, w1, x1) = grads
    assert torch.equal(y0, y1) and torch.equal(w0, w1)
    assert within_budget(x0, x1, None, 1e-5)[0]


def test_both_gradients_of_more_rows_than_one_launch_takes(ext):
    """One workgroup per four input rows and the ones of grad_w after them are more than a launch takes along x."""
    in_dim, out_dim = (1 << 26) - 4, 16
    g = torch.Generator(device="cuda").manual_seed(0)
    a, b = (torch.randint(0, in_dim, (out_dim,), device="cuda", generator=g) for _ in range(2))
    a[0], b[1], a[2], b[3] = 0, in_dim - 1, in_dim - 1, 0
    inputs, idx = torch.cat([a, b]).sort()
    idx %= out_dim
    start = torch.searchsorted(inputs, torch.arange(in_dim + 1, device="cuda"))
    x = torch.rand(in_dim, 1, device="cuda", generator=g)
    gy = torch.randn(out_dim, 1, device="cuda", generator=g)
    p = torch.softmax(torch.randn(out_dim, 16, device="cuda", generator=g), -1)
    gw, gx = ext.backward_both(x, a, b, p, gy, start, idx, 1.5, softmax_backward=True)
    assert torch.equal(gw, ext.backward_logits(x, a, b, gy, p))
    assert torch.equal(gx, ext.backward_x(x, a, b, p, gy, start, idx, 1.5))
    assert torch.equal(gx.nonzero()[:, 0], inputs.unique())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [1, 3, 4, 5, 28, 29, 32, 33, 60, 61, 64, 65, 129, 1024])
def test_partial_class_sums(ext, dtype, splits):
    """The finishing pass of GroupSum around the four waves and the eight partial sums each takes at a time; sums that are
    exact in every type."""
    x = torch.randint(0, 8, (32 * splits, 65), generator=torch.Generator().manual_seed(splits)).double() / 8
    assert torch.equal(ext.group_sum_forward(x.to(dtype).cuda(), 1, 1.0).cpu().double()[:, 0], x.sum(0).to(dtype).double())


F16, F32, F64 = DTYPES


@pytest.mark.parametrize("in_dim,out_dim,batch,dtype,forward,weights", [
    (4200, 20000, 32, F32, False, False), (4200, 20000, 199, F32, False, False), (4200, 20000, 200, F32, True, False),
    (4200, 8400, 714, F32, False, False), (4200, 8400, 715, F32, True, False), (4200, 8400, 952, F32, True, False),
    (4200, 8400, 953, F32, True, True), (4200, 20000, 749, F16, False, False), (4200, 20000, 751, F16, True, False),
    (4200, 8400, 447, F64, True, False), (4200, 8400, 477, F64, True, True), (4200, 6300, 600, F64, False, False),
    (4200, 8400, 445, F64, False, False), (4200, 8400, 1025, F64, False, False), (4200, 33000, 4, F32, True, True),
    (4200, 33000, 9, F16, True, True)])
def test_kernels_of_narrower_layers_take_the_schedule_where_it_gains(ext, monkeypatch, in_dim, out_dim, batch, dtype, forward,
                                                                     weights):
    """Either side of the lines at which a layer below 32768 neurons walks its schedule, kernel by kernel; outputs and
    gradients are those of the kernels without it."""
    import difflogic_amd as dl
    torch.manual_seed(batch)
    layer = dl.LogicLayer(in_dim, out_dim).train()
    x, gy = torch.rand(batch, in_dim, device="cuda").to(dtype), torch.randn(batch, out_dim, device="cuda").to(dtype)
    walked, real_forward, real_weights = {}, ext.forward_logits, ext.backward_logits

    def spy_forward(x, a, b, logits, schedule=None):
        walked["forward"] = schedule is not None
        return real_forward(x, a, b, logits, schedule)

    def spy_weights(x, a, b, grad_y, probs, schedule=None):
        walked["weights"] = schedule is not None
        return real_weights(x, a, b, grad_y, probs, schedule)

    monkeypatch.setattr(ext, "forward_logits", spy_forward)
    monkeypatch.setattr(ext, "backward_logits", spy_weights)
    y = layer(x)
    y.backward(gy)
    assert walked == {"forward": forward, "weights": weights}
    xt, gt = x.t().contiguous(), gy.t().contiguous()
    want, probs = real_forward(xt, *layer.indices, layer.weights.detach())
    assert torch.equal(y.detach().t(), want) if dtype != F16 else within_budget(y.t(), want, None, RTOL[dtype])[0]
    want = real_weights(xt, *layer.indices, gt, probs)
    assert within_budget(layer.weights.grad, want, None, 1e-6)[0]


@pytest.mark.parametrize("in_dim,out_dim,calls", [(8000, 20000, ["both"]), (20000, 40000, ["x", "weights"]), (20000, 20000, [])])
def test_layers_that_widen(ext, monkeypatch, in_dim, out_dim, calls):
    """Where the one-pass backward does not apply, narrower layers form both gradients in one launch."""
    import difflogic_amd as dl
    torch.manual_seed(1)
    layer = dl.LogicLayer(in_dim, out_dim, grad_factor=1.5).train()
    x = torch.rand(24, in_dim, device="cuda").requires_grad_()
    gy = torch.randn(24, out_dim, device="cuda")
    seen = []
    for name, fn in (("x", "backward_x"), ("weights", "backward_logits"), ("both", "backward_both")):
        real = getattr(ext, fn)
        monkeypatch.setattr(ext, fn, lambda *a, real=real, name=name, **kw: seen.append(name) or real(*a, **kw))
    layer(x).backward(gy)
    assert seen == calls
    monkeypatch.setattr(dl.LogicLayer, "_train_schedule", lambda self, x=None: None)
    got = x.grad, layer.weights.grad
    x.grad = layer.weights.grad = None
    layer(x).backward(gy)
    assert within_budget(got[0], x.grad, None, 1e-5)[0] and within_budget(got[1], layer.weights.grad, None, 1e-6)[0]


def test_first_evaluation_builds_no_schedule(ext):
    """A narrower layer evaluated once takes the kernels without a schedule; from the second evaluation on it has one, where
    that gains.  Wider layers and training as ever."""
    import difflogic_amd as dl
    x, short = torch.rand(1024, 4200, device="cuda"), torch.rand(100, 4200, device="cuda")
    built = lambda layer: ext.built_schedule(*layer.indices, 4200) is not None  # noqa: E731
    layer = dl.LogicLayer(4200, 8400).eval()
    first = layer(x)
    assert not built(layer)
    assert torch.equal(layer(x), first) and built(layer)
    layer = dl.LogicLayer(4200, 20000).eval()
    layer(short), layer(short)
    assert not built(layer)
    layer.train()(short)
    assert built(layer)
    layer = dl.LogicLayer(4200, 33000).eval()
    layer(short)
    assert built(layer)


@pytest.mark.parametrize("dtype,batch", [c for c in CASES if c[0] != F16])
def test_elements_that_two_lanes_write(ext, monkeypatch, dtype, batch):
    """Outputs and input gradients on rows that end inside a vector are, bit for bit, those of the same call on the rows
    padded to whole vectors (half: tests of its rounding)."""
    from difflogic_amd.functional import build_reverse_index
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    in_dim, out_dim = 60, 88
    g = torch.Generator().manual_seed(batch)
    a, b = (torch.randint(0, in_dim, (out_dim,), generator=g) for _ in range(2))
    start, idx = (t.cuda() for t in build_reverse_index(a, b, in_dim))
    a, b = a.cuda(), b.cuda()
    sched = ext.schedule_for(a, b, in_dim)
    whole = -(-batch // 8) * 8
    x = torch.rand(in_dim, whole, generator=g).to(dtype).cuda()
    gy = torch.randn(out_dim, whole, generator=g).to(dtype).cuda()
    p = torch.softmax(torch.randn(out_dim, 16, generator=g), -1).to(dtype).cuda()
    xr, gr = x[:, :batch].contiguous(), gy[:, :batch].contiguous()
    for call in (lambda x, gy: ext.forward(x, a, b, p), lambda x, gy: ext.forward(x, a, b, p, sched),
                 lambda x, gy: ext.backward_x(x, a, b, p, gy, start, idx, 1.5),
                 lambda x, gy: ext.backward_chained(x, p, gy, sched, 1.5, any_rows=True)[1]):
        assert torch.equal(call(xr, gr), call(x, gy)[:, :batch])
