"""HIP-graph replay of a whole training step, and of packed inference.

A logic-gate net's step is dozens of short kernels (per layer: softmax, forward, backward_x,
backward_w, softmax backward; each tens of microseconds at the reference's batch sizes), so an
eager step is bound by host launch overhead rather than by the GPU.  ``GraphedTrainStep``
captures forward + loss + backward (and optionally the optimizer step) once into a HIP graph on
static buffers and replays it per step.
"""
import torch


def _reads_feature_major(model, x):
    """Whether ``model`` is a Sequential whose first module that does anything to 2-D input is a 'cuda' logic layer, and nothing
    else sees its input: a subclass's own forward, or a hook, may want the strides of the example."""
    from .difflogic import FusedLogicLayerGroupSum, FusedLogicLayerPair, FusedSequential, LogicLayer
    if x.dim() != 2 or type(model) not in (torch.nn.Sequential, FusedSequential):
        return False
    first = next((m for m in model if type(m) is not torch.nn.Flatten), None)
    for m in (model, *model):
        if m._forward_pre_hooks or m._forward_hooks:
            return False
        if m is first:
            break
    if type(first) in (FusedLogicLayerGroupSum, FusedLogicLayerPair):
        first = first.layer if type(first) is FusedLogicLayerGroupSum else first.layer1
    return type(first) is LogicLayer and first.implementation == "cuda"


class GraphedTrainStep:
    """Captures ``loss = loss_fn(model(x), y); loss.backward()[; optimizer.step()]``.

    ``step(x, y)`` copies the batch into the static input buffers, replays the graph and returns
    the static loss tensor (valid until the next replay).  Parameter gradients are the
    ``.grad`` tensors of the parameters, rewritten by every replay.  Shapes and dtypes are fixed
    at construction; the static input ``x`` may be laid out feature-major (written with ``copy_``, not through a flat view).  With ``optimizer`` given it must be constructed with ``capturable=True``.
    """

    def __init__(self, model, loss_fn, example_x, example_y, optimizer=None, warmup=3):
        self.model, self.loss_fn, self.optimizer = model, loss_fn, optimizer
        # a model that starts with a logic layer reads its input feature-major: the static buffer is kept that way, so that the
        # copy into it is the transposition as well (784 -> 4 x 8000 at batch 128, with the gradient below: 91.6 -> 87.2 us a step);
        # a buffer of its own in either layout, also where the example is feature-major already
        if _reads_feature_major(model, example_x):
            self.x = example_x.detach().t().clone(memory_format=torch.contiguous_format).t()
        else:
            self.x = example_x.detach().clone()
        self.y = example_y.detach().clone()
        self._one, loss = None, None           # the loss's own gradient (made by backward() it would be a launch in every replay)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(warmup):
                loss = self._eager()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        if loss is not None and loss.dim() == 0:
            # on this stream, whose later work waits for the replays: memory of the warm-up's stream could be handed out
            # again beside the last of them
            self._one = torch.ones_like(loss, requires_grad=False)
        loss = None
        self.graph = torch.cuda.CUDAGraph()
        self._zero_grad()
        with torch.cuda.graph(self.graph):
            self.loss = self._eager(zero=False)

    def _zero_grad(self):
        if self.optimizer is not None:
            self.optimizer.zero_grad(set_to_none=True)
        else:
            self.model.zero_grad(set_to_none=True)

    def _eager(self, zero=True):
        if zero:
            self._zero_grad()
        loss = self.loss_fn(self.model(self.x), self.y)
        loss.backward(self._one)
        if self.optimizer is not None:
            self.optimizer.step()
        return loss

    def step(self, x=None, y=None):
        if x is not None:
            self.x.copy_(x, non_blocking=True)
        if y is not None:
            self.y.copy_(y, non_blocking=True)
        self.graph.replay()
        return self.loss


class GraphedPackedInference:
    """Captures ``model(PackBitsTensor(x, bit_count))`` -- packing, every gate layer, the count -- for a
    model in eval mode and a fixed input shape, and replays it per batch: one graph launch instead of
    a dozen kernel launches and their Python.  ``__call__(x)`` copies the bool batch ``[B, F]`` into
    the static input buffer, replays and returns the static ``[B, k]`` int32 counts (valid until the
    next call).  The gate ids are taken from the weights inside the graph, so weights updated in
    place between calls are seen; a model whose wiring tensors are replaced needs a new capture.
    """

    def __init__(self, model, example_x, bit_count=64, warmup=2):
        from .difflogic import LogicLayer
        from .packbitstensor import PackBitsTensor, replayed_rows
        assert not model.training, "packed inference runs the discretised net: call model.eval() first"
        assert example_x.dtype == torch.bool and example_x.dim() == 2 and example_x.is_cuda, (
            example_x.dtype, tuple(example_x.shape), example_x.device)
        self.model, self.bit_count = model, bit_count
        self.x = example_x.detach().clone()
        rows = replayed_rows([(m.in_dim, m.out_dim) for m in model.modules() if isinstance(m, LogicLayer)])

        def run():
            with torch.no_grad():
                packed = PackBitsTensor(self.x, bit_count=bit_count)
                packed._replayed = rows
                return model(packed)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(warmup):              # also builds and caches the wiring's schedules on the host
                run()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = run()

    def __call__(self, x=None):
        if x is not None:
            self.x.copy_(x, non_blocking=True)
        self.graph.replay()
        return self.out
