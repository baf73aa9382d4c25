"""What this framework is used for, as cases that can be timed: bit-packed inference of discretised
logic-gate nets, training steps (forward, loss, backward, also with the optimizer and as a replayed HIP
graph), and the discretised net on float inputs as a training loop validates with it.

A case is a dict of plain values:

* ``kind``: ``infer`` (PackBitsTensor -> LogicLayers -> GroupSum counts), ``train`` (forward, cross entropy,
  backward), ``evaluate`` (eval mode on float inputs, no gradients);
* the net: ``features`` -> ``layers`` x ``width`` -> GroupSum(``k``, ``tau``), wired by ``connections``;
* ``batch``: samples per call;
* ``infer``: ``bits`` (word width), ``gates`` (which gate ids the net's argmax gives, see GATES), ``graph``
  (called through GraphedPackedInference);
* ``train`` / ``evaluate``: ``dtype`` of the inputs (the weights stay float32), ``form``: ``written`` (the
  nn.Sequential as written for the reference), ``fused`` (through fuse_for_training), ``graph`` (fuse_for_training
  with FusedAdam, replayed by GraphedTrainStep), ``grad_factor``.
"""
import math

import torch

import difflogic_amd as dl
from difflogic_amd.graphs import GraphedPackedInference, GraphedTrainStep

# gate ids the nets are made of: all 16 alike (a net with normally distributed logits), half of them the
# pass-through gates a, b, not a, not b (towards what trained nets look like), gates of two inputs only
GATES = {
    "uniform": tuple(range(16)),
    "pass_through": (3, 5, 10, 12) * 4 + tuple(range(16)),
    "two_input": (1, 2, 4, 6, 7, 8, 9, 11, 13, 14),
}
# half inputs: the loss is scaled by this and the batch, or its gradients underflow on the way down
LOSS_SCALE = 16384.0
DTYPES = {"float32": torch.float32, "float16": torch.float16, "float64": torch.float64}


def _infer(name, features, layers, width, batch, bits=64, gates="uniform", graph=False, k=10):
    case = {"kind": "infer", "features": features, "layers": layers, "width": width, "k": k, "tau": 30.0,
            "connections": "random", "batch": batch, "bits": bits, "gates": gates, "graph": graph}
    return dict(case, name=name) if name else case


def _float(name, kind, features, layers, width, batch, dtype="float32", form="written", connections="random",
           tau=30.0, grad_factor=1.0, k=10):
    case = {"kind": kind, "features": features, "layers": layers, "width": width, "k": k, "tau": tau,
            "connections": connections, "batch": batch, "dtype": dtype, "form": form, "grad_factor": grad_factor}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one batch of the size the reference's loaders hand out, a small net, its default word width
        _infer("infer_small_b100", 784, 6, 8000, 100, bits=32),
        # serving: the medium net behind a captured graph, a thousand requests at a time, nothing in the net to skip
        _infer("infer_serving_b1000", 784, 6, 64000, 1000, gates="two_input", graph=True),
        # accuracy over a whole test set of 10 000 in one call
        _infer("infer_testset_b10000", 784, 6, 64000, 10000, bits=32),
        # a CIFAR-sized net with three thresholds, trained-like gates, a batch that fills no word, line or tile evenly
        _infer("infer_cifar_b100003", 9216, 4, 128000, 100003, gates="pass_through"),
        # bulk scoring with the small net
        _infer("infer_small_b1m", 784, 6, 8000, 1 << 20),
        # bulk scoring with the medium net: the benchmark's own workload
        _infer("infer_bulk_b1m", 784, 6, 64000, 1 << 20),
        # a training step of the small net as written for the reference, at its batch size
        _float("train_small_b100", "train", 784, 4, 8000, 100, tau=10.0),
        # the same net trained as fast as the framework can: fused, Adam included, one graph replay per step
        _float("train_small_graph_b128", "train", 784, 4, 8000, 128, tau=10.0, form="graph"),
        # the medium net at a larger batch, unique wiring
        _float("train_medium_b512", "train", 784, 6, 64000, 512, form="fused", connections="unique"),
        # half inputs beside float32 weights, rows that end inside a vector
        _float("train_half_b500", "train", 784, 6, 64000, 500, dtype="float16", tau=1600.0),
        # a deep, wide CIFAR-sized net as written for the reference, gradients scaled up on their way down
        _float("train_deep_b1024", "train", 9216, 12, 128000, 1024, connections="random", tau=100.0, grad_factor=2.0),
        # validation between epochs: the discretised net on the float inputs of the training loader
        _float("evaluate_medium_b1000", "evaluate", 784, 6, 64000, 1000),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# gate-samples (training: neuron-samples) of the largest listed cases; a drawn case stays below a half of them
_MOST = {"infer": 6 * 64000 << 20, "train": 12 * 128000 * 1024, "evaluate": 12 * 128000 * 1024}


def draw(rng):
    kind = rng.choice(("infer", "infer", "train", "train", "evaluate"))
    k = rng.choice((2, 5, 10, 10, 10, 20))
    features = rng.choice((784, 784, 3072, 9216, _log_int(rng, 32, 4000)))
    layers = rng.randint(2, 6) if kind != "train" else rng.choice((2, 3, 4, 4, 5, 6, 8, 12))
    width = max(_log_int(rng, 1000, 256000 if kind == "infer" else 128000), features)
    width = -(-width // k) * k
    if kind == "infer":
        graph = rng.random() < 0.25
        batch = min(_log_int(rng, 1, 1 << 20), _MOST[kind] // (2 * layers * width), (1 << 31) // features)
        return _infer(None, features, layers, width, batch, bits=rng.choice((8, 16, 32, 32, 64, 64)),
                      gates=rng.choice(("uniform", "pass_through", "two_input")), graph=graph, k=k)
    batch = min(_log_int(rng, 32, 1024 if kind == "train" else 4096), _MOST[kind] // (2 * layers * width))
    dtype = rng.choice(("float32", "float32", "float32", "float16", "float64"))
    form = "written"
    if kind == "train":
        form = rng.choice(("written", "fused", "graph")) if dtype == "float32" else rng.choice(("written", "fused"))
    tau = rng.choice((10.0, 30.0, 100.0))
    if dtype == "float16" and kind == "train":        # scores of a few units, or they are too coarse for a softmax
        layers, tau = min(layers, 6), float(max(10, width // (4 * k)))
    # only so many pairs of distinct inputs exist
    unique = rng.random() < 0.5 and features * (features - 1) // 2 >= width
    return _float(None, kind, features, layers, width, batch, dtype=dtype, form=form, k=k,
                  connections="unique" if unique else "random", tau=tau, grad_factor=rng.choice((1.0, 1.0, 2.0)))


def _model(case, seed):
    torch.manual_seed(seed)
    mods, d = [torch.nn.Flatten()], case["features"]
    for _ in range(case["layers"]):
        mods.append(dl.LogicLayer(d, case["width"], grad_factor=case.get("grad_factor", 1.0),
                                  connections=case["connections"]))
        d = case["width"]
    return torch.nn.Sequential(*mods, dl.GroupSum(case["k"], case["tau"]))


def prepare(case, seed):
    model = _model(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    batch, features = case["batch"], case["features"]
    if case["kind"] == "infer":
        # binarised images: a fifth of the pixels set
        x = torch.empty(batch, features, dtype=torch.bool, device="cuda")
        for s in range(0, batch, 1 << 18):
            rows = x[s:s + (1 << 18)]
            torch.lt(torch.rand(rows.shape, device="cuda", generator=g), 0.2, out=rows)
        if case["gates"] != "uniform":
            pool = torch.tensor(GATES[case["gates"]], device="cuda")
            with torch.no_grad():
                for m in model:
                    if isinstance(m, dl.LogicLayer):
                        ids = pool[torch.randint(0, len(pool), (m.out_dim,), device="cuda", generator=g)]
                        m.weights.scatter_(1, ids[:, None], 8.0)
        model.eval()
        handle = GraphedPackedInference(model, x, bit_count=case["bits"]) if case["graph"] else None
        return {"case": case, "model": model, "x": x, "handle": handle}
    x = (torch.rand(batch, features, device="cuda", generator=g) < 0.2).to(DTYPES[case["dtype"]])
    y = torch.randint(0, case["k"], (batch,), device="cuda", generator=g)
    if case["kind"] == "evaluate":
        return {"case": case, "model": model.eval(), "x": x}
    model.train()
    handle = None
    if case["form"] != "written":
        model = dl.fuse_for_training(model)
    if case["form"] == "graph":
        optimizer = dl.FusedAdam(model.parameters(), lr=0.01)
        handle = GraphedTrainStep(model, torch.nn.functional.cross_entropy, x, y, optimizer)
    return {"case": case, "model": model, "x": x, "y": y, "handle": handle}


def run(state):
    case, model, x = state["case"], state["model"], state["x"]
    if case["kind"] == "infer":
        if state["handle"] is not None:
            return state["handle"](x)
        with torch.no_grad():
            return model(dl.PackBitsTensor(x, bit_count=case["bits"]))
    if case["kind"] == "evaluate":
        with torch.no_grad():
            return model(x)
    if state["handle"] is not None:
        loss = state["handle"].step(x, state["y"])
        return [loss] + [p.detach() for p in model.parameters()]
    model.zero_grad(set_to_none=True)
    out = model(x)
    if case["dtype"] == "float16":
        loss = torch.nn.functional.cross_entropy(out.float(), state["y"]) * (LOSS_SCALE * case["batch"])
    else:
        loss = torch.nn.functional.cross_entropy(out, state["y"])
    loss.backward()
    return [out.detach(), loss.detach()] + [p.grad for p in model.parameters()]


def work(case):
    """Inference: the bool input, the counts, and per neuron its 16 logits and its two int64 inputs; one logic
    operation per gate and 32 samples.  Training and evaluation: the input, the tables, and every activation
    between two layers (a randomly wired layer needs all of the one before) written once and read once by each
    pass that uses it, gradients between layers likewise; per neuron and sample three linear interpolations
    forwards, four corner sums and two derivatives backwards."""
    neurons, batch = case["layers"] * case["width"], case["batch"]
    if case["kind"] == "infer":
        return {"bytes": batch * case["features"] + 4 * batch * case["k"] + neurons * 80,
                "flops": neurons * math.ceil(batch / 32)}
    size = {"float32": 4, "float16": 2, "float64": 8}[case["dtype"]]
    hidden = (case["layers"] - 1) * case["width"] * batch * size
    ends = batch * case["features"] * size + 2 * batch * case["k"] * size
    if case["kind"] == "evaluate":
        return {"bytes": ends + 2 * hidden + neurons * 80, "flops": 6 * neurons * batch}
    tables = neurons * (64 + 16 + 64)
    if case["form"] == "graph":
        tables += neurons * 5 * 64                # weights written, both moments read and written
    return {"bytes": ends + 5 * hidden + tables, "flops": 22 * neurons * batch}


def tolerance(case):
    """Counts are whole numbers.  The float paths: about four times the largest difference seen between the case
    (and drawn ones) and the same step in float64.  Float32: gradients of deep nets with large class sums differ
    most.  Float16: scores near 2 are 2^-9 apart, and the gradients follow the softmax over them.  Float64: the
    weights and their softmax stay float32.  Adam divides a gradient by its own size, so a rounding error next to
    zero can turn one step of lr around."""
    if case["kind"] == "infer":
        return "exact"
    if case["kind"] == "evaluate":
        return {"rel": {"float32": 2.5e-7, "float16": 1e-3, "float64": 1e-12}[case["dtype"]]}
    if case["form"] == "graph":
        return {"rel": 1e-5, "max": 0.05}
    return {"float32": {"rel": 8e-5, "max": 8e-3}, "float16": {"rel": 0.02, "max": 0.7},
            "float64": {"rel": 4e-7, "max": 1.6e-5}}[case["dtype"]]
