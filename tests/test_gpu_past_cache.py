"""Chained training kernels on matrices large enough that their rows are read, and weight gradients and probabilities written,
past the Infinity Cache (50 MB of input for the forward pass, 80 MB in half and double and for the one-pass backward, 280 MB of
input and output for the discretised forward, 240 MB for the weight gradient alone, 300 MB of GroupSum's input): against the kernels that take neurons one by one, which have no such choice.
Below, at and above a row's last full wave of vectors, whole and ragged rows, and inputs that hold infinities."""
import pytest
import torch

pytestmark = pytest.mark.gpu

RTOL = {torch.float16: 4e-3, torch.float32: 1e-5, torch.float64: 1e-12}


@pytest.fixture(scope="module")
def ext():
    import difflogic_amd
    return difflogic_amd.difflogic_cuda


def _same(u, v, dtype, rows=None):
    if dtype == torch.float16:        # a multiply-add and its conversion in one rounding or two: as the short rows' tests
        u, v = u.float(), v.float()
        return bool(((u - v).abs() <= 2.0 ** -10 * u.abs().clamp(min=2.0 ** -14) + 2e-3 * (rows is not None)).all())
    return torch.equal(u, v)


@pytest.mark.parametrize("dtype,width,batch", [(torch.float32, 26000, 500), (torch.float32, 26000, 512), (torch.float32, 42000, 511),
                                               (torch.float32, 40000, 1024), (torch.float32, 64000, 1000), (torch.float32, 170000, 128),
                                               (torch.float16, 42000, 1001), (torch.float16, 42000, 1024), (torch.float64, 42000, 256),
                                               (torch.float64, 42000, 255), (torch.float16, 40000, 1000), (torch.float16, 40000, 999),
                                               (torch.float64, 40000, 250), (torch.float64, 40000, 249)])
def test_rows_read_past_the_cache(ext, dtype, width, batch):
    from difflogic_amd.functional import get_random_connections
    torch.manual_seed(batch)
    a, b = get_random_connections(width, width, "cuda")
    start, idx = _reverse(a, b, width)
    x = torch.rand(width, batch, device="cuda").to(dtype)
    logits = torch.randn(width, 16, device="cuda").to(dtype)
    gy = torch.randn(width, batch, device="cuda").to(dtype)
    sched = ext.schedule_for(a, b, width)
    y0, p0 = ext.forward_logits(x, a, b, logits)
    y1, p1 = ext.forward_logits(x, a, b, logits, sched)
    assert _same(y0, y1, dtype) and _same(p0, p1, dtype)
    assert _same(ext.forward(x, a, b, logits, argmax=True), ext.forward(x, a, b, logits, sched, argmax=True), dtype)
    g0 = ext.backward_logits(x, a, b, gy, p0)
    assert _same(g0, ext.backward_logits(x, a, b, gy, p0, sched), dtype, batch)
    gw, gx = ext.backward_chained(x, p0, gy, sched, 1.5, softmax_backward=True, any_rows=True)
    if batch * dtype.itemsize > 32 * 16:
        assert _same(g0, gw, dtype, batch)
    else:                             # 8-byte vectors: another order of the same 128 terms, each sum to batch * 2^-24
        assert bool(((g0 - gw).abs() <= batch * 2.0 ** -24 * gy.abs().sum(1, keepdim=True)).all())
    want = ext.backward_x(x, a, b, p0, gy, start, idx, 1.5).double()
    scale = float(want.abs().max())
    assert bool(((gx.double() - want).abs() <= RTOL[dtype] * (scale + want.abs())).all())


def _reverse(a, b, width):
    from difflogic_amd.functional import build_reverse_index
    start, idx = build_reverse_index(a, b, width)
    return start.cuda(), idx.cuda()


@pytest.mark.parametrize("batch", [500, 501, 512])
def test_infinities_stay_in_their_rows(ext, batch):
    """Lanes past the end of a row take no part: a row's infinity reaches the neurons that read it, and no others."""
    from difflogic_amd.functional import get_random_connections
    width = 42000
    torch.manual_seed(batch)
    a, b = get_random_connections(width, width, "cuda")
    x = torch.rand(width, batch, device="cuda")
    hit = torch.tensor([0, 17, 30000], device="cuda")
    x[hit, batch - 1] = float("inf")
    logits, gy = torch.randn(width, 16, device="cuda"), torch.randn(width, batch, device="cuda")
    sched = ext.schedule_for(a, b, width)
    y0, p0 = ext.forward_logits(x, a, b, logits)
    y1, _ = ext.forward_logits(x, a, b, logits, sched)
    assert torch.equal(y0.nan_to_num(nan=7.0), y1.nan_to_num(nan=7.0))
    gw, _ = ext.backward_chained(x, p0, gy, sched, softmax_backward=True, any_rows=True)
    reads = torch.isin(a, hit) | torch.isin(b, hit)
    assert bool(gw[~reads].isfinite().all()) and int(reads.sum()) > 0
    assert torch.equal(gw[~reads], ext.backward_logits(x, a, b, gy, p0)[~reads])


@pytest.mark.parametrize("dtype,rows,batch", [(torch.float32, 73240, 1024), (torch.float32, 73250, 1024), (torch.float32, 75000, 1001),
                                              (torch.float16, 146480, 1024), (torch.float16, 150000, 1024), (torch.float16, 150000, 1001),
                                              (torch.float64, 36620, 1024), (torch.float64, 37500, 1001)])
def test_group_sum_past_the_cache(ext, dtype, rows, batch):
    """Eighths: the sums are exact in fp32 in any order, and rounded once to half."""
    torch.manual_seed(batch)
    x = torch.randint(0, 9, (rows, batch), device="cuda", dtype=torch.int8).to(dtype) / 8
    want = torch.stack([c.double().sum(0) for c in x.view(10, rows // 10, batch)], 1)
    assert torch.equal(ext.group_sum_forward(x, 10, 1.0), want.to(dtype))
