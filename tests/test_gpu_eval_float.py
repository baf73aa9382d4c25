"""The discretised net on float inputs: the argmax gate taken inside the forward kernels equals the kernels on a one-hot
matrix made in torch, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float64, torch.float64),
          (torch.float16, torch.float32), (torch.float64, torch.float32)]


def _weights(out_dim, dtype, g):
    w = torch.randn(out_dim, 16, generator=g).to(dtype)
    pick = lambda p: torch.rand(out_dim, generator=g) < p  # noqa: E731
    w[pick(0.2)] = 1.0                                     # ties: the first wins
    w[pick(0.1), 6] = float("nan")                         # a NaN counts as maximal, the first of several
    w[pick(0.1), 12] = float("nan")
    w[pick(0.1)] = -float("inf")
    w[pick(0.1), 9] = float("inf")
    return w.cuda()


@pytest.mark.parametrize("dtype,wdtype", DTYPES)
@pytest.mark.parametrize("out_dim,batch", [(1, 1), (3, 2), (17, 5), (64, 130), (50, 515), (40, 1000), (33, 1024), (24, 4099)])
def test_argmax_gates_in_the_forward_kernels(dtype, wdtype, out_dim, batch):
    from difflogic_amd import difflogic_cuda as ext
    g = torch.Generator().manual_seed(out_dim * 7 + batch)
    in_dim = 23
    a, b = (torch.randint(0, in_dim, (out_dim,), generator=g).cuda() for _ in range(2))
    x = torch.rand(in_dim, batch, generator=g).to(dtype).cuda()
    x[::3] = (x[::3] > 0.5).to(dtype)
    w = _weights(out_dim, wdtype, g)
    hot = torch.nn.functional.one_hot(w.argmax(-1), 16).to(dtype)
    for schedule in (None, ext.schedule_for(a, b, in_dim)):
        assert torch.equal(ext.forward(x, a, b, w, schedule, argmax=True), ext.forward(x, a, b, hot, schedule))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.float64])
def test_layer_in_eval_mode(dtype):
    """Through the module, with fp32 weights, weights of the inputs' dtype and weights that are not contiguous."""
    import difflogic_amd as dl
    torch.manual_seed(1)
    layer = dl.LogicLayer(20, 60).eval()
    x = torch.rand(70, 20, device="cuda").to(dtype)
    for w in (layer.weights.detach(), layer.weights.detach().to(dtype), layer.weights.detach().t().contiguous().t()):
        layer.weights = torch.nn.Parameter(w)
        hot = torch.nn.functional.one_hot(w.argmax(-1), 16).to(dtype)
        want = dl.difflogic_cuda.forward(x.t().contiguous(), *layer.indices, hot).t()
        got = layer(x)
        assert got.dtype == dtype and not got.requires_grad and torch.equal(got, want)
    assert tuple(layer(x[:0]).shape) == (0, 60)
