"""The training loss and its gradient against torch in 64 bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from eppgcn_amd import gnnadvisor
    return gnnadvisor()


def _case(n, classes, share, seed, spread=3.0):
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(n, classes, generator=g) * spread
    mask = torch.rand(n, generator=g) < share
    y = torch.randint(0, classes, (n,), generator=g)
    labels = torch.where(mask, y, torch.full_like(y, -1)).int()
    return logits, mask, y, labels


@pytest.mark.parametrize("n,classes,share", [(1, 1, 1.1), (15, 3, 1.1), (16, 15, 0.5), (17, 16, 0.9), (1000, 17, 0.1),
                                             (4099, 22, 0.3), (70001, 47, 0.05), (333, 200, 0.6), (140000, 5, 1.1)])
def test_loss_and_gradient(ops, n, classes, share):
    logits, mask, y, labels = _case(n, classes, share, n + classes)
    rows = mask.nonzero().squeeze(1)
    x64 = logits.double().requires_grad_()
    want = torch.nn.functional.nll_loss(torch.log_softmax(x64, 1)[mask], y[mask])
    (want * 0.75).backward()
    x = logits.cuda()
    loss = ops.nll_forward(x, rows.cuda(), labels.cuda())
    # a row's loss is a difference of two numbers below 40, each rounded a few times at 2^-24 of its size
    assert loss.shape == () and abs(float(loss) - float(want)) <= 1e-5
    grad = ops.nll_backward(torch.tensor(0.75, device="cuda"), x, labels.cuda(), rows.numel()).cpu().double()
    scale = 0.75 / rows.numel()
    assert float((grad - x64.grad).abs().max()) <= 1e-5 * scale
    assert not grad[~mask].any()


def test_loss_of_no_rows_infinities_and_nan(ops):
    x = torch.randn(40, 7)
    none = torch.full((40,), -1, dtype=torch.int32)
    empty = torch.empty(0, dtype=torch.long)
    assert torch.isnan(ops.nll_forward(x.cuda(), empty.cuda(), none.cuda())).item()
    assert not ops.nll_backward(torch.ones((), device="cuda"), x.cuda(), none.cuda(), 0).any()
    x[3, 2], x[5, 1], x[9], x[11, 0] = float("-inf"), float("inf"), float("-inf"), float("nan")
    for row, label in ((3, 0), (3, 2), (5, 1), (5, 0), (9, 4), (11, 3)):
        labels = none.clone()
        labels[row] = label
        want = torch.nn.functional.nll_loss(torch.log_softmax(x.double(), 1)[row:row + 1], torch.tensor([label]))
        got = ops.nll_forward(x.cuda(), torch.tensor([row], device="cuda"), labels.cuda()).cpu().double()
        assert torch.allclose(got, want, rtol=1e-5, atol=1e-6, equal_nan=True), (row, label)


def test_trainer_refuses_labels_outside_the_classes():
    from eppgcn_amd import graphs, train
    g = graphs.uniform_graph(300, 600, seed=1, device="cuda")
    ds = train.GraphDataset(g, 8, 4, 2, train_ratio=0.5, labels="uniform")
    ds.y[ds.train_mask.nonzero()[0]] = 4
    with pytest.raises(ValueError, match="outside the 4 classes"):
        train.Trainer(g, hidden=8, dataset=ds).train_step(True)
