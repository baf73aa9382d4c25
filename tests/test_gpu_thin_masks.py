"""The thinned LDS net kernel's bookkeeping (masks, ranks, records, numbers of neurons left): widths around the words of the
masks, a thread's items and the widest layer, gate mixes that leave everything, little or nothing, class sizes from one up,
gate ids folded by the caller or not; against the same net evaluated whole."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import difflogic_amd
    return difflogic_amd.difflogic_cuda


@pytest.mark.parametrize("widths,k", [([31, 32, 33, 32], 32), ([1023, 1024, 1025, 1030], 10), ([64], 1), ([5120, 2049, 4100], 2),
                                      ([10240, 10240], 10240), ([9999, 4096, 2047, 640], 5)])
@pytest.mark.parametrize("gates", [range(16), (1, 7, 8, 14), (3, 5, 10, 12), (0, 15, 6), (0, 15)])
def test_thinned_equals_whole(ext, widths, k, gates):
    g = torch.Generator().manual_seed(sum(widths))
    pool = torch.tensor(list(gates), dtype=torch.uint8)
    dims, layers = [208] + widths, []
    for d, n in zip(dims, widths):
        layers.append((torch.randint(0, d, (n,), generator=g).cuda(), torch.randint(0, d, (n,), generator=g).cuda(),
                       pool[torch.randint(0, len(pool), (n,), generator=g)].cuda()))
    x = (torch.rand(300, 208, generator=g) < 0.3).cuda()
    packed = ext.tensor_packbits_batch_major_rows(x, 48)
    whole = ext.eval_net_lds(packed, layers, 84, k, scheduled=False)
    assert whole is not None
    folded = ext.fold_gate_constants(layers)
    for layers_, known in ((layers, False), (folded, True)):
        assert torch.equal(ext.eval_net_lds(packed, layers_, 84, k, thin=True, folded=known), whole)
        if max(widths[:-1], default=0) + 208 <= 10240:
            assert torch.equal(ext.eval_net_lds_bool(x, layers_, k, thin=True, folded=known), whole)
