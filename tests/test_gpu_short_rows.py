"""Packed inference on short rows: a layer straight from its weights, the pack kernel and the bit count for few words,
and PackBitsTensor choosing between layers evaluated at once and deferred ones.  Bit-exact against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import interp
from oracle import packed_oracle as po
from tests.helpers import build_model, random_layers

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import difflogic_amd
    return difflogic_amd.difflogic_cuda


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a)).cuda()


# vectors of 16 bytes per row around the lanes per neuron (4, 8, 16, 32, 64); neurons around a wave's 16 and a workgroup's
# 64, and enough of them that they are not shared out (512 workgroups)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("vectors,out_dim", [(1, 1), (1, 64), (3, 17), (4, 65), (5, 15), (8, 130), (9, 63), (16, 33), (17, 48),
                                             (32, 16), (32, 129), (33, 20), (64, 70), (65, 47), (128, 18), (200, 65),
                                             (33, 8192), (40, 16400), (20, 16385), (2, 33000)])
def test_layer_from_its_weights(ext, vectors, out_dim, dtype):
    rng = np.random.default_rng(vectors * 1009 + out_dim)
    in_dim = 37
    a, b = rng.integers(0, in_dim, out_dim), rng.integers(0, in_dim, out_dim)
    x = rng.integers(-2**62, 2**62, (in_dim, 2 * vectors), dtype=np.int64)
    w = torch.as_tensor(rng.standard_normal((out_dim, 16))).to(dtype)
    w[rng.random(out_dim) < 0.2, :] = 1.0                              # ties: the first wins
    w[rng.random(out_dim) < 0.1, 5] = float("nan")                     # a NaN counts as maximal, the first of several
    w[rng.random(out_dim) < 0.1, 14] = float("nan")
    w[rng.random(out_dim) < 0.1, :] = -float("inf")
    got = ext.eval_weights(_dev(x), _dev(a), _dev(b), w.cuda())
    assert np.array_equal(got.cpu().numpy(), po.eval_layer(x, a, b, w.argmax(-1).numpy().astype(np.uint8)))


# rows a thread counts around 8 and its 255; every width of a workgroup's columns; classes around the 8 XCDs; past the
# last word; rows and classes that the other kernel takes
@pytest.mark.parametrize("per_class,k,words,pad", [
    (1, 1, 2, 0), (1023, 1, 2, 5), (8193, 1, 2, 63), (261120, 1, 2, 0), (261121, 1, 2, 1), (300, 7, 6, 3), (130560, 2, 102, 9),
    (130561, 2, 102, 0), (129, 10, 22, 0), (65280, 3, 234, 0), (65281, 3, 234, 63), (500, 9, 80, 1), (33, 16, 126, 0),
    (1025, 17, 130, 7), (127, 20, 1152, 0), (40, 200, 18, 0), (40, 201, 18, 0),
    (200, 64, 130, 0), (200, 43, 300, 5), (200, 129, 16, 1), (201, 129, 16, 0), (5, 3, 1, 0), (77, 1, 2050, 64)])
def test_bit_count_of_short_rows(ext, per_class, k, words, pad):
    g = torch.Generator(device="cuda").manual_seed(per_class + k)
    x = torch.randint(-2**62, 2**62, (per_class * k, words), device="cuda", generator=g)
    if per_class > 1000:
        x[:per_class] = -1                                             # a class whose every row counts
    got = ext.groupbitsum(x, pad, k)
    bits = 0
    for c in range(k):                                                 # in torch, a word at a time: the sizes are the point
        rows = x[c * per_class:(c + 1) * per_class]
        bits = torch.stack([((rows >> s) & 1).sum(0) for s in range(64)], 1).reshape(-1)
        assert torch.equal(got[:, c].long(), bits[:words * 64 - pad]), c


# (the last four: more than one slice of the features per workgroup column, and one or two slices more than fit need)
@pytest.mark.parametrize("F,B", [(f, b) for f in (1, 15, 16, 17, 63, 65, 80, 784) for b in (1, 64, 65, 1000, 12288, 12289, 20000)]
                         + [(2368, 13000), (4096, 14000), (9216, 14000), (5008, 15001)])
def test_pack_into_rows(ext, F, B):
    rng = np.random.default_rng(F * 31 + B)
    raw = torch.as_tensor(rng.choice([0, 0, 1, 2, 255], (B, F)).astype(np.uint8))       # any non-zero byte counts
    x = raw.cuda().view(torch.bool)
    row_bytes = 16 * -(-B // 128)
    got = ext.tensor_packbits_batch_major_rows(x, row_bytes).cpu().numpy()
    bits = np.unpackbits(got.view(np.uint8), axis=1, bitorder="little")
    assert np.array_equal(bits[:, :B], (raw.numpy() != 0).T) and not bits[:, B:].any()


# either side of the bytes up to which the kernel for few words takes the batch: 16-byte, 4-byte and single loads in the other
@pytest.mark.parametrize("F,B", [(12288, 9358), (12288, 9359), (12304, 7721), (12304, 7722), (10004, 3998), (10004, 3999),
                                 (2001, 6746), (2001, 7990), (9217, 2495), (9217, 2496)])
def test_pack_many_features_into_rows(ext, F, B):
    x = torch.rand(B, F, device="cuda", generator=torch.Generator(device="cuda").manual_seed(F + B)) < 0.3
    words = -(-B // 64)
    got = ext.tensor_packbits_batch_major_rows(x, 16 * -(-B // 128))
    bit = torch.ones(64, dtype=torch.int64, device="cuda") << torch.arange(64, device="cuda")
    for w in range(words):
        piece = x[64 * w:64 * w + 64].long()
        assert torch.equal(got[:, w], (piece * bit[:piece.shape[0], None]).sum(0)), w
    assert not got[:, words:].any()


@pytest.mark.parametrize("widths,B,bits", [
    ([1000, 1200, 2000], 1, 8), ([4096, 2100, 4096], 100, 16), ([6000, 6000], 6144, 32), ([6000, 6000], 6145, 64),
    ([10250, 11000], 12288, 64), ([10250, 11000], 12289, 64), ([10250, 10900], 40960, 32), ([10250, 10900], 40961, 64), ([1000, 999, 1900, 1000], 300, 64), ([2000, 4000], 1000, 64)])
def test_layers_at_once_and_deferred_agree(monkeypatch, widths, B, bits):
    """Either side of every limit of the rules (layers at once; counted from stored rows), the counts are the oracle's whatever
    the route, and so are the words of deferred layers."""
    import difflogic_amd as dl
    from difflogic_amd import packbitstensor as pbt
    rng = np.random.default_rng(B + len(widths))
    F, k = 50, 5 if widths[-1] % 5 == 0 else 2
    layers = random_layers(rng, F, widths)
    x = rng.random((B, F)) < 0.4
    model = build_model(F, layers, k).eval()
    want = interp.net_eval(x, layers, k)
    xd = torch.as_tensor(x).cuda()
    for limit, stored in ((pbt._DIRECT_BYTES, pbt._STORED_BYTES), (0, pbt._STORED_BYTES), (0, 0)):
        monkeypatch.setattr(pbt, "_DIRECT_BYTES", limit)
        monkeypatch.setattr(pbt, "_STORED_BYTES", stored)
        with torch.no_grad():
            assert np.array_equal(model(dl.PackBitsTensor(xd, bit_count=bits)).cpu().numpy(), want)
            p = dl.PackBitsTensor(xd, bit_count=bits)
            for m in list(model)[:-1]:
                p = m(p)
            for _ in range(2):                                         # counting leaves the object as it is
                assert np.array_equal(p.group_sum(k).cpu().numpy(), want)
            words = p.t.cpu().numpy()
        if limit:
            at_once = words
    assert words.dtype == at_once.dtype and np.array_equal(words, at_once)


def test_words_written_between_layers_at_once():
    """`.t` read, written in place and rebound between layers that are evaluated at once; counting leaves the object as
    it is; a batch of no samples."""
    import difflogic_amd as dl
    rng = np.random.default_rng(3)
    F, B = 40, 200
    layers = random_layers(rng, F, [1000, 2000, 1000])
    model = build_model(F, layers, 10).eval()
    logic = [m for m in model if isinstance(m, dl.LogicLayer)]
    with torch.no_grad():
        p = logic[0](dl.PackBitsTensor(torch.as_tensor(rng.random((B, F)) < 0.5).cuda(), bit_count=64))
        assert not p._pending                                          # evaluated already
        fresh = torch.as_tensor(rng.integers(-2**62, 2**62, tuple(p.t.shape), dtype=np.int64)).cuda()
        p.t.copy_(fresh)
        p = logic[1](p)
        mid = po.eval_layer(fresh.cpu().numpy(), *layers[1])
        assert np.array_equal(p.t.cpu().numpy(), mid)
        p.t = _dev(~mid)
        p = logic[2](p)
        top = po.eval_layer(~mid, *layers[2])
        assert np.array_equal(p.group_sum(10).cpu().numpy(), po.groupbitsum(top, p.pad_len, 10))
        assert np.array_equal(p.group_sum(10).cpu().numpy(), po.groupbitsum(top, p.pad_len, 10))
        assert np.array_equal(p.t.cpu().numpy(), top)
        assert tuple(model(dl.PackBitsTensor(torch.zeros(0, F, dtype=torch.bool, device="cuda"))).shape) == (0, 10)


@pytest.mark.parametrize("width,B,at_once", [(6500, 4096, True), (6500, 4097, False), (4290, 6144, True), (4300, 6144, False)])
def test_replayed_net_that_fits_in_lds(monkeypatch, width, B, at_once):
    """Either side of the lines that hold for a replayed graph, in its warm-up calls too; every replay gives the oracle's
    counts.  Called eagerly all of them are evaluated at once."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedPackedInference
    rng = np.random.default_rng(B + width)
    layers = random_layers(rng, 50, [width, width])
    x, other = (rng.random((B, 50)) < 0.4 for _ in range(2))
    model = build_model(50, layers, 10).eval()
    calls, real = [], dl.PackBitsTensor.apply_weights
    monkeypatch.setattr(dl.PackBitsTensor, "apply_weights", lambda self, *a: calls.append(1) or real(self, *a))
    graph = GraphedPackedInference(model, torch.as_tensor(x).cuda())
    assert len(calls) == (6 if at_once else 0)                         # two warm-up calls and the captured one, two layers each
    for batch in (x, other, x):
        assert np.array_equal(graph(torch.as_tensor(batch).cuda()).cpu().numpy(), interp.net_eval(batch, layers, 10))
    calls.clear()
    with torch.no_grad():
        model(dl.PackBitsTensor(torch.as_tensor(x).cuda()))
    assert len(calls) == 2


@pytest.mark.parametrize("widths", [[12000], [6000, 12000], [6000, 6000, 6000, 12000]])
def test_counting_stored_rows(monkeypatch, widths):
    """Counting deferred layers from stored rows: the last layer's rows are given back, the object can be counted and read
    again, and words that are no whole vectors are copied into padded rows once, not to learn their length."""
    import difflogic_amd as dl
    from difflogic_amd import packbitstensor as pbt
    monkeypatch.setattr(pbt, "_DIRECT_BYTES", 0)
    monkeypatch.setattr(pbt, "lds_tail", lambda *a, **kw: 0)
    rng = np.random.default_rng(9)
    F, k, batch = 50, 10, 4064
    layers = random_layers(rng, F, widths)
    logic = [m for m in build_model(F, layers, k).eval() if isinstance(m, dl.LogicLayer)]
    words = rng.integers(-2**31, 2**31, (F, batch // 32), dtype=np.int32)            # 508 bytes: no whole 16-byte vectors
    x = np.unpackbits(words.view(np.uint8), axis=1, bitorder="little").T[:batch].astype(bool)
    want = interp.net_eval(x, layers, k)
    with torch.no_grad():
        p = dl.PackBitsTensor(torch.zeros(batch, F, dtype=torch.bool, device="cuda"), bit_count=32)
        p.t = _dev(words)
        for m in logic:
            p = m(p)
        copies, real = [], pbt.PackBitsTensor._adopt
        monkeypatch.setattr(pbt.PackBitsTensor, "_adopt", lambda self, v: copies.append(v.shape) or real(self, v))
        p._live_share(), torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        assert np.array_equal(p.group_sum(k).cpu().numpy(), want) and len(copies) == 1
        assert torch.cuda.memory_allocated() - before < 12000 * 512              # at most the rows of an earlier layer
        assert np.array_equal(p.group_sum(k).cpu().numpy(), want)
        want = words
        for a, b, op in layers:
            want = po.eval_layer(want, a, b, op)
        assert np.array_equal(p.t.cpu().numpy(), want)
        assert np.array_equal(p.group_sum(k).cpu().numpy(), po.groupbitsum(want, p.pad_len, k))


@pytest.mark.parametrize("widths,B,at_once", [([4000, 2000, 1000], 256, 1), ([4000, 2000, 1000], 257, 0), ([2000, 1000], 1024, 1),
                                              ([2000, 1000], 1025, 0), ([12000, 6000, 3000], 2000, 2)])
def test_replayed_net_that_narrows(monkeypatch, widths, B, at_once):
    """Layers before the narrow end are evaluated at once on short rows only, in the warm-up calls and the captured one."""
    import difflogic_amd as dl
    from difflogic_amd.graphs import GraphedPackedInference
    rng = np.random.default_rng(B)
    layers = random_layers(rng, 50, widths)
    x = rng.random((B, 50)) < 0.4
    model = build_model(50, layers, 10).eval()
    calls, real = [], dl.PackBitsTensor.apply_weights
    monkeypatch.setattr(dl.PackBitsTensor, "apply_weights", lambda self, *a: calls.append(1) or real(self, *a))
    graph = GraphedPackedInference(model, torch.as_tensor(x).cuda())
    assert len(calls) == 3 * at_once
    for _ in range(3):
        assert np.array_equal(graph(torch.as_tensor(x).cuda()).cpu().numpy(), interp.net_eval(x, layers, 10))
