"""Adam in one launch against torch's own step: the same bits in weights and state, and torch's step for every other form."""
import copy

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pair(shapes, lr=0.01, **options):
    gen = torch.Generator().manual_seed(7)
    start = [torch.randn(s, generator=gen) for s in shapes]
    sides = []
    for _ in range(2):
        weights = [torch.nn.Parameter(w.clone().cuda()) for w in start]
        sides.append((weights, torch.optim.Adam(weights, lr=lr, **options)))
    return sides, gen


def _call(opt, weights):
    from eppgcn_amd import gnnadvisor
    group, states = opt.param_groups[0], [opt.state[w] for w in weights]
    return gnnadvisor().adam_step(list(weights), [w.grad for w in weights], [s["exp_avg"] for s in states],
                                  [s["exp_avg_sq"] for s in states], [s["step"] for s in states], group["lr"],
                                  *group["betas"], group["eps"])


def _same(one, other):
    for (a, oa), (b, ob) in [(x, y) for x, y in zip(one, other)]:
        assert torch.equal(a, b)
        for key in ("step", "exp_avg", "exp_avg_sq"):
            assert torch.equal(oa[key], ob[key]), key


def _states(side):
    weights, opt = side
    return [(w.detach(), opt.state[w]) for w in weights]


@pytest.mark.parametrize("shapes", [[(1,)], [(96, 16), (16, 22)], [(255,), (256,), (257,)], [(3, 5)] * 33, [(0, 4), (4, 4)],
                                    [(2048 * 256 + 1,)]], ids=["one", "model", "block", "two_launches", "empty", "strided"])
@pytest.mark.parametrize("options", [{}, {"betas": (0.6, 0.9), "eps": 1e-4}], ids=["default", "betas"])
def test_weights_and_state_have_the_bits_of_torch(shapes, options):
    # gradients from 1e-25 (squares below the normal range) to 1e6, zeros, and one NaN and infinity
    (ours, theirs), gen = _pair(shapes, **options)
    for step in range(6):
        for a, b in zip(ours[0], theirs[0]):
            g = torch.randn(a.shape, generator=gen) * 10.0 ** torch.randint(-25, 7, a.shape, generator=gen)
            g[torch.rand(a.shape, generator=gen) < 0.1] = 0.0
            a.grad, b.grad = g.cuda(), g.cuda()
        versions = [w._version for w in ours[0]]
        if step == 0:
            ours[1].step()
        else:
            assert _call(ours[1], ours[0])
        theirs[1].step()
        assert all(w._version > v for w, v in zip(ours[0], versions))
        _same(_states(ours), _states(theirs))
    if ours[0][0].numel() > 1:
        for w in (ours[0][0], theirs[0][0]):
            w.grad.view(-1)[0], w.grad.view(-1)[-1] = float("nan"), float("inf")
        assert _call(ours[1], ours[0])
        theirs[1].step()
        for a, b in zip(ours[0], theirs[0]):
            assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))


@pytest.mark.parametrize("spoil", ["double", "strided", "beta1", "gpu_step", "count"])
def test_other_forms_are_left_to_torch_unchanged(spoil):
    (ours, _), gen = _pair([(8, 6), (5,)], betas=(0.5, 0.9) if spoil == "beta1" else (0.9, 0.999))
    weights, opt = ours
    for w in weights:
        w.grad = torch.randn(w.shape, generator=gen).cuda()
    opt.step()
    if spoil == "double":
        opt.state[weights[0]]["exp_avg"] = opt.state[weights[0]]["exp_avg"].double()
    elif spoil == "strided":
        weights[0].grad = torch.randn(6, 8, generator=gen).cuda().t()
    elif spoil == "gpu_step":
        opt.state[weights[1]]["step"] = opt.state[weights[1]]["step"].cuda()
    elif spoil == "count":
        from eppgcn_amd import gnnadvisor
        assert not gnnadvisor().adam_step([], [], [], [], [], 0.01, 0.9, 0.999, 1e-8)
        return
    before = [(w.detach().clone(), {k: v.clone() for k, v in opt.state[w].items()}) for w in weights]
    assert not _call(opt, weights)
    _same(before, _states((weights, opt)))


def test_weights_that_share_a_step_counter():
    """The counter moves once for each of them before any of them reads it, as in torch's step."""
    sides, gen = _pair([(4, 3), (5,), (7,)])
    grads = [[torch.randn(w.shape, generator=gen) for w in sides[0][0]] for _ in range(3)]
    for step in range(3):
        for weights, opt in sides:
            for w, g in zip(weights, grads[step]):
                w.grad = g.cuda()
        if step == 0:
            for weights, opt in sides:
                opt.step()
                opt.state[weights[2]]["step"] = opt.state[weights[0]]["step"]
        else:
            assert _call(sides[0][1], sides[0][0])
            sides[1][1].step()
        _same(_states(sides[0]), _states(sides[1]))
    assert [float(sides[0][1].state[w]["step"]) for w in sides[0][0]] == [5.0, 3.0, 5.0]


@pytest.mark.parametrize("option", ["plain", "hook", "scheduler", "decay", "sgd", "no_grad", "class"])
def test_trainer_takes_the_step_its_optimizer_says(option, monkeypatch):
    from eppgcn_amd import graphs, train
    tr = train.Trainer(graphs.uniform_graph(300, 900, seed=1, device="cuda"), labels="uniform")
    calls = []
    if option == "decay":
        tr.optimizer = torch.optim.Adam(tr.model.parameters(), lr=0.01, weight_decay=0.1)
    elif option == "sgd":
        tr.optimizer = torch.optim.SGD(tr.model.parameters(), lr=0.01)
    elif option == "hook":
        tr.optimizer.register_step_post_hook(lambda *a: calls.append(a))
    elif option == "class":
        inner = torch.optim.Adam.step
        monkeypatch.setattr(torch.optim.Adam, "step", lambda self: calls.append(self) or inner(self))
    elif option == "scheduler":
        scheduler = torch.optim.lr_scheduler.ExponentialLR(tr.optimizer, 0.5)
    tr.train_step(True)
    if option == "scheduler":
        scheduler.step()
    weights = list(tr.model.parameters())
    if option == "no_grad":
        weights[0].requires_grad_(False)
    copies = [torch.nn.Parameter(w.detach().clone()) for w in weights]
    other = type(tr.optimizer)(copies, **{k: v for k, v in tr.optimizer.defaults.items()})
    other.load_state_dict(copy.deepcopy(tr.optimizer.state_dict()))
    tr.train_step(False)
    for w, c in zip(weights, copies):
        c.grad = None if w.grad is None else w.grad.clone()
    monkeypatch.undo()
    other.step()
    assert all(torch.equal(w, c) for w, c in zip(weights, copies))
    assert len(calls) == (2 if option in ("hook", "class") else 0)
    assert other.state_dict()["state"].keys() == tr.optimizer.state_dict()["state"].keys()
    for k, s in tr.optimizer.state_dict()["state"].items():
        assert all(torch.equal(s[n], other.state_dict()["state"][k][n]) for n in s if torch.is_tensor(s[n]))


def test_a_profile_has_the_range_of_the_optimizer():
    """Torch's step and the one in one launch are the same range of a profile, once per epoch."""
    from eppgcn_amd import graphs, train
    tr = train.Trainer(graphs.uniform_graph(300, 900, seed=1, device="cuda"))
    for epoch in range(3):                        # the first step is torch's
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
            tr.train_step(epoch == 0)
        assert [e.count for e in profile.key_averages() if e.key == "Optimizer.step#Adam.step"] == [1], epoch


@pytest.mark.parametrize("groups", [1, 2, 3])
def test_a_profile_has_one_range_of_dropped_gradients(groups):
    """Torch's zero_grad and the trainer's way round it are the same range of a profile, once whatever the groups."""
    from eppgcn_amd import graphs, train
    trainer = train.Trainer(graphs.uniform_graph(200, 400, seed=1, device="cuda"), dim=8, hidden=4, num_classes=3)
    for k in range(groups - 1):
        trainer.optimizer.add_param_group({"params": [torch.nn.Parameter(torch.ones(k + 2, device="cuda"))]})
    counts = []
    for drop in (trainer._zero_grad, trainer.optimizer.zero_grad):
        for group in trainer.optimizer.param_groups:
            for w in group["params"]:
                w.grad = torch.ones_like(w)
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
            drop()
        counts.append([e.count for e in profile.key_averages() if e.key == "Optimizer.zero_grad#Adam.zero_grad"])
        assert all(w.grad is None for group in trainer.optimizer.param_groups for w in group["params"])
    assert counts == [[1], [1]]
