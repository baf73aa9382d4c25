"""Half activations: every output, input-gradient element and class score is the fp32 (fp64 for the last product) value of
its formula rounded to half ONCE, whatever its place in a vector, on rows that end inside a 16-byte vector (whose last
elements are written by two lanes) and on inputs whose gradient is summed from several positions of the schedule."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 1536


def _corners(p):
    """Corner sums in fp32, in the kernels' order of additions."""
    at = lambda i: ((p[:, i[0]] + p[:, i[1]]) + (p[:, i[2]] + p[:, i[3]])) + ((p[:, i[4]] + p[:, i[5]]) + (p[:, i[6]] + p[:, i[7]]))  # noqa: E731
    return (at((8, 9, 10, 11, 12, 13, 14, 15)), at((4, 5, 6, 7, 12, 13, 14, 15)), at((2, 3, 6, 7, 10, 11, 14, 15)),
            at((1, 3, 5, 7, 9, 11, 13, 15)))


def _fma32(x, y, z):
    return (x.astype(np.float64) * y + z).astype(np.float32)          # the product of a half and a float is exact in fp64


@pytest.fixture(scope="module")
def wiring():
    """Every input feeds two neurons: its gradient is a sum of two terms, the same in either order."""
    rng = np.random.default_rng(5)
    a = rng.permutation(N)
    b = np.roll(a, 1)[np.argsort(rng.random(N))]
    while (a == b).any():
        b = rng.permutation(N)
    return a, b


def _case(wiring, batch, wdtype):
    a, b = wiring
    g = torch.Generator().manual_seed(batch)
    x = torch.rand(N, batch, generator=g).half()
    gy = torch.randn(N, batch, generator=g).half()
    p = torch.softmax(torch.randn(N, 16, generator=g), -1).to(wdtype)
    p00, p01, p10, p11 = (c[:, None] for c in _corners(p.float().numpy()))
    av, bv, gv = x.numpy()[a].astype(np.float32), x.numpy()[b].astype(np.float32), gy.numpy().astype(np.float32)
    d0, d1 = p01 - p00, p11 - p10
    lo, hi = _fma32(bv, d0, p00), _fma32(bv, d1, p10)
    y = (av.astype(np.float64) * (hi - lo) + lo).astype(np.float16)
    dd, da = d1 - d0, p10 - p00
    acc = []
    for term in (lambda u, v, w: u * v + w, _fma32):     # in two roundings; fused (rows of whole vectors along the schedule)
        acc.append(np.zeros((N, batch), np.float32))
        acc[-1][a] = gv * term(bv, dd, da)
        acc[-1][b] += gv * term(av, dd, d0)
    return x, gy, p, y, *acc


def _same(got, want):
    got = got.cpu().numpy()
    assert got.dtype == np.float16 and got.shape == want.shape
    wrong = (got != want).sum()
    assert wrong == 0, (wrong, want.size)


@pytest.mark.parametrize("wdtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("batch", [9, 63, 255, 257, 500, 515, 1025, 2047, 2050])
def test_rows_that_end_inside_a_vector(monkeypatch, wiring, batch, wdtype):
    from difflogic_amd import difflogic_cuda as ext
    from difflogic_amd.functional import build_reverse_index
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    x, gy, p, y, acc, _ = _case(wiring, batch, wdtype)
    a, b = (torch.as_tensor(t).cuda() for t in wiring)
    start, idx = (t.cuda() for t in build_reverse_index(a.cpu(), b.cpu(), N))
    x, gy, p = x.cuda(), gy.cuda(), p.cuda()
    sched = ext.schedule_for(a, b, N)
    for schedule in (None, sched):
        _same(ext.forward(x, a, b, p, schedule), y)
    for scale in (1.0, 1.5):
        want = (acc.astype(np.float64) * scale).astype(np.float16)
        _same(ext.backward_x(x, a, b, p, gy, start, idx, scale), want)
        _same(ext.backward_both(x, a, b, p, gy, start, idx, scale)[1], want)
        _same(ext.backward_chained(x, p, gy, sched, scale, any_rows=True)[1], want)
    g = torch.randn(batch, 4, generator=torch.Generator().manual_seed(1)).half()
    want = (g.double().numpy().T * np.float64(np.float32(1 / 3.0))).astype(np.float16).repeat(8, 0)
    _same(ext.group_sum_backward(g.cuda(), 32, 3.0), want)


@pytest.mark.parametrize("batch", [64, 256, 512, 1024, 4096])
def test_sums_over_positions_on_whole_vectors(monkeypatch, wiring, batch):
    """(Scale 1: the product with another scale is rounded to fp32 first for some elements of a whole vector.)"""
    from difflogic_amd import difflogic_cuda as ext
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    x, gy, p, _, _, acc = _case(wiring, batch, torch.float32)
    a, b = (torch.as_tensor(t).cuda() for t in wiring)
    sched = ext.schedule_for(a, b, N)
    assert sched.backward_plan()[4] > 0
    _same(ext.backward_chained(x.cuda(), p.cuda(), gy.cuda(), sched)[1], acc.astype(np.float16))


@pytest.mark.parametrize("batch,per_class,tau", [(70001, 40, 1.7), (120000, 130, 0.9)])
def test_class_sums(batch, per_class, tau):
    """Values whose fp32 sums are exact (and have all 24 bits): a score is the sum times the reciprocal of tau in fp64,
    rounded once."""
    from difflogic_amd import difflogic_cuda as ext
    k = 4
    g = torch.Generator().manual_seed(batch)
    x = torch.zeros(k, per_class, batch, dtype=torch.float64)
    x[:, 0] = torch.randint(1024, 2048, (k, batch), generator=g).double()
    x[:, per_class // 2] = torch.randint(0, 1024, (k, batch), generator=g).double() / 8192
    want = (x.sum(1).numpy().T * (1.0 / tau)).astype(np.float16)
    _same(ext.group_sum_forward(x.view(k * per_class, batch).half().cuda(), k, tau), want)
