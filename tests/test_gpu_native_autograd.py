"""The layer's and the loss's autograd functions in native code against the Python ones, and what still takes the Python ones."""
import contextlib
import gc
import weakref

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


def _trainer(first=True):
    from eppgcn_amd import graphs, train
    g = graphs.uniform_graph(700, 2000, seed=3, device="cuda")
    tr = train.Trainer(g, dim=24, hidden=16, num_classes=22, backsize=4, labels="uniform")
    if first:
        tr.train_step(True)
    return tr


@pytest.fixture(scope="module")
def trained():
    return _trainer()


def _call(tr, X, layer=1):
    conv = tr.model.convs[layer]
    return conv(X, tr.inputInfo, tr.mask_props[layer], tr.back_props[layer], False, False)


def _python(tr, X, layer=1):
    from eppgcn_amd.gcn_conv import GNNAFunction
    conv = tr.model.convs[layer]
    return GNNAFunction.apply(X, conv.weights, tr.inputInfo, tr.mask_props[layer], tr.back_props[layer], False, False,
                              conv.relu_input)


def _is_native(out):
    # torch names the node of a native function with its C++ type, that of a Python one <class>Backward
    return "CppNode" in type(out.grad_fn).__name__ or "::" in out.grad_fn.name() or "<" in out.grad_fn.name()


def _input(tr, layer=1, seed=1):
    width = tr.model.convs[layer].weights.shape[0]
    return torch.randn(tr.dataset.num_nodes, width, generator=torch.Generator().manual_seed(seed)).cuda()


def _close(a, b):
    # the same kernels on the same data; sums whose order the atomics choose differ by a few roundings of 2^-24
    return float((a.double() - b.double()).norm()) <= 1e-6 * float(b.double().norm())


def _path_gradient(tr, shape):
    """An incoming gradient as the loss gives it: zero outside the training rows."""
    g = torch.randn(shape, generator=torch.Generator().manual_seed(9)).cuda()
    return g * tr.dataset.train_mask.view(-1, 1)


@pytest.mark.parametrize("unpruned", [False, True, 1], ids=["pruned", "unpruned", "truthy"])
@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("needs_dx", [False, True])
@pytest.mark.parametrize("grad", ["whole", "strided", "expanded"])
def test_layer_is_the_python_function(trained, unpruned, relu, needs_dx, grad, monkeypatch):
    tr = trained
    monkeypatch.setattr(tr.model.convs[1], "relu_input", relu)
    monkeypatch.setattr(tr.back_props[1], "unpruned", unpruned)
    got = []
    for run in (_call, _python):
        X = _input(tr).requires_grad_(needs_dx)
        out = run(tr, X)
        assert _is_native(out) == (run is _call)
        d = _path_gradient(tr, out.shape)
        if grad == "strided":
            d = d.t().contiguous().t()
        elif grad == "expanded":
            d = torch.ones((), device="cuda").expand(out.shape)
        wanted = [tr.model.convs[1].weights] + ([X] if needs_dx else [])
        got.append((out.detach(), *torch.autograd.grad(out, wanted, d)))
    assert all(_close(a, b) for a, b in zip(*got))


def test_layer_without_gradients_and_frozen_weights(trained):
    tr, X = trained, _input(trained)
    with torch.no_grad():
        out = _call(tr, X)
        assert not out.requires_grad and _close(out, _python(tr, X))
    with torch.inference_mode():
        assert _close(_call(tr, X), out)
    weights = tr.model.convs[1].weights
    weights.requires_grad_(False)
    try:
        assert not _call(tr, X).requires_grad
        X.requires_grad_(True)
        d = _path_gradient(tr, out.shape)
        assert _close(torch.autograd.grad(_call(tr, X), X, d)[0], torch.autograd.grad(_python(tr, X), X, d)[0])
    finally:
        weights.requires_grad_(True)


def test_graph_is_kept_freed_and_checked_as_in_python(trained):
    tr = trained
    X = _input(tr).requires_grad_()
    out = _call(tr, X)
    d = _path_gradient(tr, out.shape)
    first = torch.autograd.grad(out, X, d, retain_graph=True)[0]
    assert _close(torch.autograd.grad(out, X, d)[0], first)
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(d)
    Y = _input(tr)
    out = _call(tr, Y)
    Y.mul_(2.0)
    with pytest.raises(RuntimeError, match="inplace operation"):
        out.backward(d)
    seen = []
    X = _input(tr).requires_grad_()
    out = _call(tr, X)
    out.register_hook(lambda g: seen.append("out") or g * 2)
    out.grad_fn.register_hook(lambda *_: seen.append("node"))
    X.register_hook(lambda g: seen.append("in"))
    assert _close(torch.autograd.grad(out, X, d)[0], 2 * first) and seen == ["out", "node", "in"]


def test_records_are_read_in_the_pass_and_let_go(trained):
    import copy
    tr = trained
    X = _input(tr).requires_grad_()
    back = copy.copy(tr.back_props[1])
    del back.id
    conv = tr.model.convs[1]
    out = conv(X, tr.inputInfo, tr.mask_props[1], back, False, False)
    d = _path_gradient(tr, out.shape)
    with pytest.raises(AttributeError, match="id"):
        torch.autograd.grad(out, X, d, retain_graph=True)
    back.id = tr.back_props[1].id                       # filled in between the passes
    assert _close(torch.autograd.grad(out, X, d, retain_graph=True)[0], torch.autograd.grad(_python(tr, X), X, d)[0])
    back.partSize = "4"
    with pytest.raises(TypeError):
        torch.autograd.grad(out, X, d, retain_graph=True)
    info = copy.copy(tr.inputInfo)
    info.partSize = None
    with pytest.raises(TypeError):
        conv(X, info, tr.mask_props[1], back, False, False)
    gone = weakref.ref(back)
    del back, out
    gc.collect()
    assert gone() is None


@pytest.mark.parametrize("needs_dx", [False, True])
def test_grad_fn_shows_what_the_python_function_keeps(trained, needs_dx):
    """Records, launch hints and saved tensors are read from and set on a result's grad_fn as on the Python function's ctx."""
    import copy
    tr = trained
    X = _input(tr).requires_grad_(needs_dx)
    weights, back = tr.model.convs[1].weights, tr.back_props[1]
    outs = [run(tr, X) for run in (_call, _python)]      # a Python node's saved tensors go with its output
    nodes = [out.grad_fn for out in outs]
    ours, theirs = nodes
    assert vars(ours) == vars(theirs) and type(ours).__name__ == type(theirs).__name__
    for node in nodes:
        assert node.inputInfo is tr.inputInfo and node.backInfo is back and node.reluInput is tr.model.convs[1].relu_input
        assert (node.partSize, node.dimWorker, node.warpPerBlock) == (tr.inputInfo.partSize, tr.inputInfo.dimWorker,
                                                                      tr.inputInfo.warpPerBlock)
        assert type(node.saved_tensors) is tuple and [a is b for a, b in zip(node.saved_tensors, (X, weights))] == [True, True]
        assert node.needs_input_grad == (needs_dx, True) + (False,) * 6
        assert isinstance(node, torch.autograd.graph.Node)
        with pytest.raises(AttributeError):
            node.nothing
        with pytest.raises(AttributeError):
            del node.nothing
        with pytest.raises(AttributeError):
            node.saved_tensors = ()
    del node, nodes, ours, theirs, outs
    for run in (_call, _python):
        out = run(tr, X)
        out.grad_fn.note = 3
        gc.collect()
        assert out.grad_fn.note == 3                     # it is the node's, not the Python object's
        del out.grad_fn.note
        assert not hasattr(out.grad_fn, "note")
        other = copy.copy(back)
        del other.id
        out.grad_fn.backInfo = other                     # read when the backward pass runs
        d = _path_gradient(tr, out.shape)
        with pytest.raises(AttributeError, match="id"):
            torch.autograd.grad(out, weights, d, retain_graph=True)
        out.grad_fn.backInfo = back
        torch.autograd.grad(out, weights, d)
        assert out.grad_fn.backInfo is back
        with pytest.raises(RuntimeError, match="second time"):
            out.grad_fn.saved_tensors
        gone = weakref.ref(other)
        del other, out
        gc.collect()
        assert gone() is None


def test_grad_fn_of_the_loss_shows_what_the_python_function_keeps(trained):
    from eppgcn_amd import train
    tr = trained
    out = tr.model(tr.dataset.x, tr.inputInfo, tr.mask_props, tr.back_props, False, False).detach().requires_grad_()
    losses = tr._loss(out), train._TrainingLoss.apply(out, tr.train_idx, tr.row_labels)
    nodes = [loss.grad_fn for loss in losses]
    for node in nodes:
        assert node.num_rows == tr.train_idx.numel() and node.saved_tensors[0] is out
        assert torch.equal(node.saved_tensors[1], tr.row_labels) and node.needs_input_grad == (True, False, False)
        assert isinstance(node, torch.autograd.graph.Node)
    assert vars(nodes[0]) == vars(nodes[1]) and type(nodes[0]).__name__ == type(nodes[1]).__name__


def test_saved_tensor_hooks_and_checkpoint(trained):
    from torch.utils.checkpoint import checkpoint
    tr = trained
    X = _input(tr).requires_grad_()
    out = _python(tr, X)
    d = _path_gradient(tr, out.shape)
    want = torch.autograd.grad(out, X, d)[0]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = _call(tr, X)
    assert packed == [X.shape, tr.model.convs[1].weights.shape]
    assert _close(torch.autograd.grad(out, X, d)[0], want)
    with torch.autograd.graph.save_on_cpu():
        out = _call(tr, X)
    assert _close(torch.autograd.grad(out, X, d)[0], want)
    for reentrant in (False, True):
        out = checkpoint(lambda x: _call(tr, x) * 1.0, X, use_reentrant=reentrant)
        X.grad = None
        out.backward(d)
        assert _close(X.grad, want)
    with torch.autograd.set_detect_anomaly(True):
        out = _call(tr, X)
        assert _close(torch.autograd.grad(out, X, d)[0], want)


def test_compiled_autograd(trained):
    tr = trained
    compiled = pytest.importorskip("torch._dynamo.compiled_autograd")
    if not hasattr(compiled, "_enable"):
        pytest.skip("this torch enables compiled autograd in another way")
    got = []
    for context in (contextlib.nullcontext(), compiled._enable(torch.compile(backend="eager"))):
        tr.model.zero_grad()
        loss = tr._loss(tr.model(tr.dataset.x, tr.inputInfo, tr.mask_props, tr.back_props, False, False))
        with context:
            loss.backward()
        got.append([w.grad for w in tr.model.parameters()])
    assert all(_close(a, b) for a, b in zip(*got))


class _Count(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("how", ["dispatch_mode", "function_mode", "profiler", "forward_mode", "subclass", "patched_function",
                                 "patched_step", "patched_op", "first_iteration"])
def test_python_function_where_the_call_is_looked_into(trained, how, monkeypatch):
    from eppgcn_amd import gcn_conv, gnnadvisor
    tr = trained
    X = _input(tr)
    assert _is_native(_call(tr, X))
    context = contextlib.nullcontext()
    if how == "dispatch_mode":
        context = _Count()
    elif how == "function_mode":
        context = torch.overrides.BaseTorchFunctionMode()
    elif how == "profiler":
        context = torch.autograd.profiler.profile(use_device=None)
    elif how == "subclass":
        X = X.as_subclass(_Sub)
    elif how == "patched_function":
        monkeypatch.setattr(gcn_conv, "GNNAFunction", type("GNNAFunction", (gcn_conv.GNNAFunction,), {}))
    elif how == "patched_step":
        step = gcn_conv.GNNAFunction.backward
        monkeypatch.setattr(gcn_conv.GNNAFunction, "backward", staticmethod(lambda ctx, d: step(ctx, d)))
    elif how == "patched_op":
        op = gnnadvisor().forward
        monkeypatch.setattr(gnnadvisor(), "forward", lambda *a, **k: op(*a, **k))
    if how == "forward_mode":
        with torch.autograd.forward_ad.dual_level():
            with pytest.raises((RuntimeError, NotImplementedError)):
                _call(tr, torch.autograd.forward_ad.make_dual(X, torch.ones_like(X)))
        return
    with context:
        if how == "first_iteration":                     # it marks the path as well
            new = _trainer(first=False)
            out = new.model(new.dataset.x, new.inputInfo, new.mask_props, new.back_props, True, False)
        else:
            out = _call(tr, X)
    assert not _is_native(out)


@pytest.mark.parametrize("where", ["own", "torch"])
@pytest.mark.parametrize("what", ["layer", "loss"])
def test_a_replaced_apply_is_called_in_every_pass(trained, what, where, monkeypatch):
    from eppgcn_amd import gcn_conv, train
    tr, X = trained, _input(trained)
    logits = tr.model(tr.dataset.x, tr.inputInfo, tr.mask_props, tr.back_props, False, False).detach().requires_grad_()
    function = gcn_conv.GNNAFunction if what == "layer" else train._TrainingLoss
    run = (lambda: _call(tr, X)) if what == "layer" else (lambda: tr._loss(logits))
    torchs, calls = torch.autograd.Function.apply.__func__, []

    def counted(cls, *args):
        calls.append(cls)
        return torchs(cls, *args)

    monkeypatch.setattr(function if where == "own" else torch.autograd.Function, "apply", classmethod(counted))
    for k in range(2):
        assert not _is_native(run()) and calls == [function] * (k + 1)
    monkeypatch.undo()
    assert _is_native(run()) and len(calls) == 2


def test_function_transforms_refuse_as_before(trained):
    X = _input(trained)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: _call(trained, x))(X.unsqueeze(0))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: _call(trained, x).sum())(X)


def test_loss_is_the_python_function(trained):
    from eppgcn_amd import train
    tr = trained
    out = tr.model(tr.dataset.x, tr.inputInfo, tr.mask_props, tr.back_props, False, False).detach()
    got = []
    for run in (tr._loss, lambda x: train._TrainingLoss.apply(x, tr.train_idx, tr.row_labels)):
        x = out.clone().requires_grad_()
        loss = run(x)
        assert _is_native(loss) == (not got)
        (g,) = torch.autograd.grad(loss, x, create_graph=True)
        assert not g.requires_grad                       # nothing to differentiate: the incoming gradient is a constant
        scale = torch.tensor(0.5, device="cuda", requires_grad=True)
        (twice,) = torch.autograd.grad(run(x) * scale, x, create_graph=True)
        with pytest.raises(RuntimeError, match="once_differentiable"):
            twice.sum().backward()
        got.append((loss.detach(), g, twice.detach()))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    with torch.autograd.profiler.profile(use_device=None):
        assert not _is_native(tr._loss(out.clone().requires_grad_()))


def _weights(tr):
    return torch.cat([w.detach().flatten() for w in tr.model.parameters()])


def test_epochs_are_those_of_the_python_functions(monkeypatch):
    from eppgcn_amd import gnnadvisor
    ours, theirs = _trainer(), _trainer()
    for _ in range(4):
        ours.train_step(False)
    with monkeypatch.context() as m:
        for name in ("gcn_layer", "training_loss"):
            m.setattr(gnnadvisor(), name, lambda *_: None)
        m.setattr(theirs, "_zero_grad", theirs.optimizer.zero_grad)
        m.setattr(theirs, "_backward", lambda loss: loss.backward())
        for _ in range(4):
            theirs.train_step(False)
    # Adam's first steps are of size lr whatever a gradient's size: a rounding can turn a weight whose gradient is nearly zero
    assert float((_weights(ours) - _weights(theirs)).abs().mean()) <= 1e-5


def test_kept_unit_gradient(trained, monkeypatch):
    tr = _trainer()
    tr.train_step(False)
    kept = tr._unit_gradient[0]
    assert float(kept) == 1.0
    kept.mul_(3.0)                                       # seen by its version
    tr.train_step(False)
    assert tr._unit_gradient[0] is not kept and float(tr._unit_gradient[0]) == 1.0
    # whoever looks at the loss's gradient is handed one of autograd's own
    loss_of, handed = tr._loss, []

    def watched(out):
        loss = loss_of(out)
        loss.register_hook(lambda g: handed.append(g.data_ptr()))
        return loss

    monkeypatch.setattr(tr, "_loss", watched)
    tr.train_step(False)
    assert handed and handed[0] != tr._unit_gradient[0].data_ptr()


class _WritesIntoItsGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, d):
        d.data.mul_(3.0)
        return d


@pytest.mark.parametrize("how", ["function", "prehook", "hook", "tensor_hook"])
def test_each_epoch_starts_from_one(how, monkeypatch):
    """Whoever is handed the gradient that the backward pass starts from may write into it; no write is seen in another epoch."""
    tr = _trainer()
    tr.train_step(False)                                 # a gradient of one is kept now
    loss_of, starts = tr._loss, []

    def changed(out):
        loss = loss_of(out)
        if how == "function":
            loss = _WritesIntoItsGradient.apply(loss)
        elif how == "prehook":
            loss.grad_fn.register_prehook(lambda grads: grads[0].data.mul_(3.0) and None)
        elif how == "hook":
            loss.grad_fn.register_hook(lambda ins, outs: outs[0].data.mul_(3.0) and None)
        else:
            loss.register_hook(lambda grad: grad.data.mul_(3.0) and None)
        loss.grad_fn.register_prehook(lambda grads: starts.append(float(grads[0])))
        return loss

    monkeypatch.setattr(tr, "_loss", changed)
    for _ in range(3):
        tr.train_step(False)
    assert starts == [3.0 if how in ("prehook", "tensor_hook") else 1.0] * 3
    monkeypatch.undo()
    tr.train_step(False)
    assert float(tr._unit_gradient[0]) == 1.0


def test_unit_gradient_of_another_stream():
    tr = _trainer()
    tr.train_step(False)
    kept = tr._unit_gradient[0]
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        tr.train_step(False)
        assert tr._unit_gradient[0] is not kept          # its fill is ordered before the work of its own stream only
        there = tr._unit_gradient[0]
        tr.train_step(False)
        assert tr._unit_gradient[0] is there
    torch.cuda.current_stream().wait_stream(other)
    torch.cuda.synchronize()
    assert float(there) == 1.0


@pytest.mark.parametrize("how", ["plain", "instance", "subclass", "parameter"])
def test_gradients_are_dropped(how):
    tr = _trainer()
    called = []
    if how == "instance":
        zero = tr.optimizer.zero_grad
        tr.optimizer.zero_grad = lambda *a, **k: called.append(1) or zero(*a, **k)
    elif how == "subclass":
        class Mine(torch.optim.Adam):
            def zero_grad(self, set_to_none=True):
                called.append(1)
                super().zero_grad(set_to_none)
        tr.optimizer = Mine(tr.model.parameters())
    elif how == "parameter":
        class Weight(torch.nn.Parameter):
            pass
        tr.optimizer.param_groups[0]["params"].append(Weight(torch.zeros(3, device="cuda")))
    extra = torch.nn.Parameter(torch.ones(2, device="cuda"))     # a weight that no pass reaches: its gradient goes as well
    extra.grad = torch.ones(2, device="cuda")
    tr.optimizer.param_groups[0]["params"].append(extra)
    old = [w.grad for w in tr.model.parameters()]
    tr._zero_grad()
    assert extra.grad is None and all(w.grad is None for w in tr.model.parameters()) and all(g is not None for g in old)
    assert bool(called) == (how in ("instance", "subclass"))
