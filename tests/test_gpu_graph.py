"""A HIP-graph replay of the training step must reproduce the eager step on every replay,
with eager work and synchronisations between replays."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(dl, seed):
    torch.manual_seed(seed)
    mods, d = [torch.nn.Flatten()], 60
    for w in (400, 400, 300):
        mods.append(dl.LogicLayer(d, w, grad_factor=1.5))
        d = w
    return torch.nn.Sequential(*mods, dl.GroupSum(10, 10.0)).train()


def test_graphed_step_equals_eager_on_every_replay():
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    model = _model(dl, 0)
    loss_fn = torch.nn.CrossEntropyLoss()
    g = torch.Generator(device="cuda").manual_seed(0)
    xs = [(torch.rand(64, 60, device="cuda", generator=g) < 0.3).float() for _ in range(4)]
    ys = [torch.randint(0, 10, (64,), device="cuda", generator=g) for _ in range(4)]

    import copy
    eager = copy.deepcopy(model)                      # same logits and wiring, its own .grad tensors
    graphed = GraphedTrainStep(model, loss_fn, xs[0], ys[0])
    for rep in range(6):
        x, y = xs[rep % 4], ys[rep % 4]
        loss_g = graphed.step(x, y)
        torch.cuda.synchronize()
        # eager work between the replays
        eager.zero_grad(set_to_none=True)
        loss_e = loss_fn(eager(x), y)
        loss_e.backward()
        torch.cuda.synchronize()
        assert torch.equal(loss_g, loss_e.detach()), rep
        for pg, pe in zip(model.parameters(), eager.parameters()):
            assert pg.grad is not None and torch.equal(pg.grad, pe.grad), rep


@pytest.mark.parametrize("batch,features,feature_major", [(1, 60, False), (7, 1, False), (7, 60, True), (7, 60, False)])
def test_the_static_input_is_a_buffer_of_its_own(batch, features, feature_major):
    """Also where the example's transposed view is contiguous: one sample, one feature, a feature-major example."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    torch.manual_seed(2)
    model = torch.nn.Sequential(torch.nn.Flatten(), dl.LogicLayer(features, 40), dl.GroupSum(10, 10.0)).train()
    loss_fn = torch.nn.CrossEntropyLoss()
    example = torch.rand(features, batch, device="cuda").t() if feature_major else torch.rand(batch, features, device="cuda")
    y = torch.zeros(batch, dtype=torch.long, device="cuda")
    kept, other = example.clone(), torch.rand(batch, features, device="cuda")
    graphed = GraphedTrainStep(model, loss_fn, example, y)
    assert graphed.x.data_ptr() != example.data_ptr()
    for x in (other, kept, other):
        loss = graphed.step(x).clone()
        assert torch.equal(example, kept)
        assert torch.equal(loss, loss_fn(model(x), y).detach())
    example.fill_(0.5)                                # what the caller writes there later is not what is replayed
    assert torch.equal(graphed.step(), loss)


@pytest.mark.parametrize("who", ["subclass", "pre-hook of the model", "pre-hook of the layer", "hook of Flatten"])
def test_other_readers_of_the_static_input_see_its_strides(who):
    """A Sequential subclass with a forward of its own, and hooks, get the input laid out as the example is."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep

    class Halves(torch.nn.Sequential):
        def forward(self, x):
            return super().forward(x.view(-1, 30))        # (of a transposed view this would raise)

    torch.manual_seed(3)
    features = 30 if who == "subclass" else 60
    mods = [torch.nn.Flatten(), dl.LogicLayer(features, 40), dl.GroupSum(10, 10.0)]
    model = (Halves if who == "subclass" else torch.nn.Sequential)(*mods).train()
    seen = []
    if who == "pre-hook of the model":
        model.register_forward_pre_hook(lambda m, a: seen.append(a[0].view(-1)))
    elif who == "pre-hook of the layer":
        mods[1].register_forward_pre_hook(lambda m, a: seen.append(a[0].view(-1)))
    elif who == "hook of Flatten":
        mods[0].register_forward_hook(lambda m, a, y: seen.append(y.view(-1)))
    loss_fn = torch.nn.CrossEntropyLoss()
    x, other = torch.rand(8, 60, device="cuda"), torch.rand(8, 60, device="cuda")
    y = torch.zeros(16 if who == "subclass" else 8, dtype=torch.long, device="cuda")
    graphed = GraphedTrainStep(model, loss_fn, x, y)
    for inp in (other, x, other):
        assert torch.equal(graphed.step(inp), loss_fn(model(inp), y).detach())


def test_what_replays_read_is_no_memory_of_the_warm_up_stream():
    """Buffers kept beside the graph come from the stream that the graph is made and replayed on, so that freeing them waits for
    the replays; without warm-up steps the gradient of the loss is part of the graph."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    torch.manual_seed(4)
    model = torch.nn.Sequential(dl.LogicLayer(60, 40), dl.GroupSum(10, 10.0)).train()
    loss_fn = torch.nn.CrossEntropyLoss()
    x, y = torch.rand(8, 60, device="cuda"), torch.zeros(8, dtype=torch.long, device="cuda")
    for warmup in (2, 0):
        graphed = GraphedTrainStep(model, loss_fn, x, y, warmup=warmup)
        kept = [t for t in vars(graphed).values() if torch.is_tensor(t) and t is not graphed.loss]
        here = torch.cuda.current_stream().cuda_stream
        for t in kept:
            segment, = [s for s in torch.cuda.memory_snapshot() if s["address"] <= t.data_ptr() < s["address"] + s["total_size"]]
            assert segment["stream"] == here
        want = loss_fn(model(x), y)
        grads = torch.autograd.grad(want, list(model.parameters()))
        for _ in range(3):
            assert torch.equal(graphed.step(x), want.detach())
            assert all(torch.equal(p.grad, g) for p, g in zip(model.parameters(), grads))


def test_graphed_step_with_optimizer_tracks_eager_training():
    import copy

    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    model = _model(dl, 1)
    eager = copy.deepcopy(model)
    loss_fn = torch.nn.CrossEntropyLoss()
    g = torch.Generator(device="cuda").manual_seed(1)
    x = (torch.rand(32, 60, device="cuda", generator=g) < 0.3).float()
    y = torch.randint(0, 10, (32,), device="cuda", generator=g)
    opt_g = torch.optim.Adam(model.parameters(), lr=0.01, capturable=True)
    opt_e = torch.optim.Adam(eager.parameters(), lr=0.01, capturable=True)
    # the constructor's warm-up steps train the model too: keep the eager copy in step
    graphed = GraphedTrainStep(model, loss_fn, x, y, optimizer=opt_g, warmup=2)
    for _ in range(3):                                # 2 warm-ups + the captured (not executed) step is not run
        pass
    losses_g, losses_e = [], []
    for _ in range(2):
        opt_e.zero_grad(set_to_none=True)
        loss_fn(eager(x), y).backward()
        opt_e.step()
    for rep in range(5):
        losses_g.append(graphed.step().item())
        opt_e.zero_grad(set_to_none=True)
        le = loss_fn(eager(x), y)
        le.backward()
        opt_e.step()
        losses_e.append(le.item())
        torch.cuda.synchronize()
    assert losses_g == losses_e, (losses_g, losses_e)
    assert losses_g[-1] < losses_g[0]


def test_graphed_step_of_the_fused_model_equals_its_eager_step(monkeypatch):
    """fuse_for_training (first two layers with the inner activation recomputed, last layer with
    GroupSum) captured and replayed: every replay reproduces the eager step of the same fused
    model bit for bit, on changing inputs."""
    import copy

    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    monkeypatch.setattr(dl.LogicLayer, "_CHAIN_MIN_IN_DIM", 0)        # layers this narrow walk their schedules too
    monkeypatch.setattr(dl.LogicLayer, "_CHAIN_MIN_OUT_DIM", 0)
    monkeypatch.setattr(dl.difflogic_cuda, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    base = _model(dl, 2)
    model = dl.fuse_for_training(base).train()
    eager = dl.fuse_for_training(copy.deepcopy(base)).train()
    assert isinstance(model[1], dl.FusedLogicLayerPair) and isinstance(model[-2], dl.FusedLogicLayerGroupSum)
    loss_fn = torch.nn.CrossEntropyLoss()
    g = torch.Generator(device="cuda").manual_seed(0)
    xs = [(torch.rand(64, 60, device="cuda", generator=g) < 0.3).float() for _ in range(3)]
    ys = [torch.randint(0, 10, (64,), device="cuda", generator=g) for _ in range(3)]
    graphed = GraphedTrainStep(model, loss_fn, xs[0], ys[0])
    for rep in range(5):
        x, y = xs[rep % 3], ys[rep % 3]
        loss_g = graphed.step(x, y)
        torch.cuda.synchronize()
        eager.zero_grad(set_to_none=True)
        loss_e = loss_fn(eager(x), y)
        loss_e.backward()
        torch.cuda.synchronize()
        assert torch.equal(loss_g, loss_e.detach()), rep
        for pg, pe in zip(model.parameters(), eager.parameters()):
            assert pg.grad is not None and torch.equal(pg.grad, pe.grad), rep


@pytest.mark.parametrize("F,widths,k,B", [(64, [512, 512, 320], 10, 1000), (784, [12000, 12000, 12000], 10, 4096),
                                          (48, [96, 48], 4, 77), (784, [40000, 40000], 10, 1024)])
def test_graphed_packed_inference_equals_eager_on_every_replay(F, widths, k, B):
    """Packing, gate layers and count captured once (the narrow nets run resident in LDS, the wide ones
    stream) and replayed on new batches, with eager work and synchronisation between the replays; every
    replay equals the eager result and the bitwise oracle.  Gate weights changed in place are picked up."""
    import numpy as np
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedPackedInference
    from oracle import interp
    from tests.helpers import build_model, random_layers
    rng = np.random.default_rng(F + B)
    layers = random_layers(rng, F, widths)
    model = build_model(F, layers, k).eval()
    xs = [torch.as_tensor(rng.random((B, F)) < p).cuda() for p in (0.2, 0.5, 0.8, 0.35)]
    graphed = GraphedPackedInference(model, xs[0], bit_count=32)
    for i, x in enumerate(xs):
        got = graphed(x).clone()
        with torch.no_grad():
            eager = model(dl.PackBitsTensor(x, bit_count=32))
        torch.cuda.synchronize()
        assert torch.equal(got, eager), i
        if B <= 1024 or i == 0:
            assert np.array_equal(got.cpu().numpy(), interp.net_eval(x.cpu().numpy(), layers, k)), i
    # another gate table in the same storage: the graph reads the weights at replay time
    last = [m for m in model if isinstance(m, dl.LogicLayer)][-1]
    with torch.no_grad():
        last.weights.copy_(torch.randn_like(last.weights))
    got = graphed(xs[1]).clone()
    with torch.no_grad():
        eager = model(dl.PackBitsTensor(xs[1], bit_count=32))
    assert torch.equal(got, eager)


@pytest.mark.parametrize("fused", [False, True])
def test_captured_step_walks_the_schedules_of_the_warm_up(monkeypatch, fused):
    """A layer whose input needs no gradient never builds the plan of the one-pass backward; its captured step runs along
    the schedule all the same."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedTrainStep
    torch.manual_seed(0)
    model = torch.nn.Sequential(dl.LogicLayer(4200, 20000), dl.LogicLayer(20000, 20000), dl.GroupSum(10, 100.0))
    layers = [m for m in model if isinstance(m, dl.LogicLayer)]
    model = (dl.fuse_for_training(model) if fused else model).train()
    x, y = torch.rand(32, 4200, device="cuda"), torch.randint(0, 10, (32,), device="cuda")
    asked, real = [], dl.LogicLayer._train_schedule

    def spy(self, *args):
        schedule = real(self, *args)
        if torch.cuda.is_current_stream_capturing():
            asked.append((layers.index(self), schedule is not None))
        return schedule

    monkeypatch.setattr(dl.LogicLayer, "_train_schedule", spy)
    step = GraphedTrainStep(model, torch.nn.functional.cross_entropy, x, y)
    assert {i for i, _ in asked} == {0, 1} and all(ok for _, ok in asked)
    for _ in range(3):
        loss = step.step().item()
        grads = [p.grad.clone() for p in model.parameters()]
        model.zero_grad(set_to_none=False)
        eager = torch.nn.functional.cross_entropy(model(x), y)
        eager.backward()
        assert eager.item() == loss and all(torch.equal(p.grad, g) for p, g in zip(model.parameters(), grads))


def test_capture_without_the_backward_plan():
    """A schedule that only forward passes have used: its backward plan is not built under capture, the gradients come from
    the other kernels."""
    import difflogic_amd as dl
    torch.manual_seed(0)
    layer = dl.LogicLayer(4200, 20000).train()
    x = torch.rand(32, 4200, device="cuda").requires_grad_()
    with torch.no_grad():
        layer(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = dl.LogicLayer(4200, 4200).train()(x)                   # (the autograd thread starts outside the capture)
        torch.autograd.grad(other.sum(), x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gx, gw = torch.autograd.grad(layer(x).square().sum(), (x, layer.weights))
    schedule = dl.difflogic_cuda.built_schedule(*layer.indices, 4200)
    assert schedule._backward is None
    want_x, want_w = torch.autograd.grad(layer(x).square().sum(), (x, layer.weights))
    assert schedule._backward is not None
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(gx, want_x, rtol=1e-5, atol=1e-5) and torch.equal(gw, want_w)
