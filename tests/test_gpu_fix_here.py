"""One-pass backward: inputs at several schedule positions, or at none, finished by workgroups of the same launch (up to 64 of
them, and as many positions) against overflow rows and a launch of their own: the same sums in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import difflogic_amd
    return difflogic_amd.difflogic_cuda


def _wiring(in_dim, out_dim, used, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, used, (out_dim,), generator=g).cuda(), torch.randint(0, used, (out_dim,), generator=g).cuda()


# inputs at several positions: none but the trails' ends; a few; up to the limit; beyond it; and inputs that feed no neuron
WIRINGS = [(64, 64, 64), (20, 30, 12), (40, 44, 40), (150, 260, 150), (300, 40, 20), (60, 33, 60)]


@pytest.mark.parametrize("in_dim,out_dim,used", WIRINGS)
@pytest.mark.parametrize("dtype,batch", [(torch.float32, 36), (torch.float32, 129), (torch.float32, 512), (torch.float32, 1028),
                                         (torch.float32, 2052), (torch.float16, 40), (torch.float16, 500), (torch.float16, 1024),
                                         (torch.float64, 30), (torch.float64, 257), (torch.float64, 1025)])
def test_finished_in_the_launch_or_after_it(ext, monkeypatch, in_dim, out_dim, used, dtype, batch):
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    a, b = _wiring(in_dim, out_dim, used, in_dim)
    b[0] = a[0]
    torch.manual_seed(batch)
    x, gy = torch.rand(in_dim, batch, device="cuda").to(dtype), torch.randn(out_dim, batch, device="cuda").to(dtype)
    w = torch.softmax(torch.randn(out_dim, 16, device="cuda"), -1)
    w = w if batch % 2 else w.to(dtype)                              # fp32 probabilities beside half / double rows as well
    sched = ext.schedule_for(a, b, in_dim)
    here = ext.backward_chained(x, w, gy, sched, 1.5, softmax_backward=True, any_rows=True)
    monkeypatch.setattr(ext._lib, "DL_FIX_POSITIONS", 0)
    after = ext.backward_chained(x, w, gy, sched, 1.5, softmax_backward=True, any_rows=True)
    assert torch.equal(here[0], after[0])
    if dtype == torch.float16 and batch % 8 == 0:                    # whole vectors: the last rounding is the compiler's choice
        u, v = here[1].float(), after[1].float()
        assert bool(((u - v).abs() <= 2.0 ** -10 * v.abs() + 2.0 ** -24).all())
    else:
        assert torch.equal(here[1], after[1])


@pytest.mark.parametrize("in_dim,out_dim,used", WIRINGS)
@pytest.mark.parametrize("batch,recompute", [(36, False), (36, True), (260, False), (511, True), (512, False), (512, True)])
def test_layer_below_of_finished_inputs(ext, monkeypatch, in_dim, out_dim, used, batch, recompute):
    monkeypatch.setattr(ext, "BACKWARD_CHAIN_MAX_OVERFLOW", 1e9)
    a, b = _wiring(in_dim, out_dim, used, in_dim)
    la, lb = _wiring(20, in_dim, 20, out_dim)
    torch.manual_seed(batch)
    xl, gy = torch.rand(20, batch, device="cuda"), torch.randn(out_dim, batch, device="cuda")
    w, wl = (torch.softmax(torch.randn(n, 16, device="cuda"), -1) for n in (out_dim, in_dim))
    x = None if recompute else ext.forward(xl, la, lb, wl)
    sched = ext.schedule_for(a, b, in_dim)
    here = ext.backward_chained_lower(x, w, gy, sched, xl, la, lb, wl, 1.5, softmax_backward=True, any_rows=True)
    monkeypatch.setattr(ext._lib, "DL_FIX_POSITIONS", 0)
    after = ext.backward_chained_lower(x, w, gy, sched, xl, la, lb, wl, 1.5, softmax_backward=True, any_rows=True)
    assert torch.equal(here[0], after[0])
    # sums over the batch in another order on rows that take 8-byte vectors
    bound = batch * 2.0 ** -24 * float(after[1].abs().max()) * 4
    assert torch.equal(here[1], after[1]) or bool(((here[1] - after[1]).abs() <= bound).all())
