"""The reference driver's training loop around the aggregation path (EPPGCN/gcn_main.py:120-292)
as a library: a multi-layer GCN over the ``GNNAdvisor`` ops with the execution path prepared on
the first iteration, timed the way the reference times it; and the host-CPU comparison run (the
same model through ``torch.sparse.mm`` on the CPU)."""
from __future__ import annotations

import os
import time
from typing import List

import torch
import torch.nn.functional as F
import torch.optim.optimizer as torch_optimizer

from . import gnnadvisor, graphs
from .gcn_conv import GCNConv, _is_torchs, _parts
from .param import backInputProperty, inputProperty, maskInputProperty


class GraphDataset:
    """The fields of the reference's dataset object the path needs (EPPGCN/dataset.py:22-156):
    CSR, scale vector, features, labels, train mask and the per-run buffers the path mutates
    (neighbour masks = False, edge masks = -1, kept degrees = 0)."""

    def __init__(self, graph: graphs.Graph, dim=96, num_classes=22, num_layers=2, train_mask=None,
                 train_ratio=0.1, labels="ones", feature_seed=1, mask_seed=2, label_seed=4):
        dev = graph.column_index.device
        n, e = graph.num_nodes, graph.num_edges
        self.num_nodes, self.num_edges = n, e
        self.num_features, self.num_classes, self.num_layers = dim, num_classes, num_layers
        self.avg_degree = e / n
        self.avg_edgeSpan = -1
        self.row_pointers, self.column_index, self.degrees = graph.row_pointers, graph.column_index, graph.degrees
        self.x = graphs.normal32(feature_seed, (n, dim), dev)
        # the reference labels every vertex 1 (EPPGCN/dataset.py:133); "uniform" draws real classes
        self.y = (torch.ones(n, dtype=torch.long, device=dev) if labels == "ones"
                  else graphs.uniform_labels(label_seed, n, num_classes, dev))
        self.train_mask = (graphs.bernoulli_mask(n, train_ratio, mask_seed, dev) if train_mask is None
                           else train_mask.to(dev))
        self.ngh_masks = [torch.zeros(n, dtype=torch.bool, device=dev) for _ in range(num_layers - 1)]
        self.empty_mask = torch.zeros(0, dtype=torch.bool, device=dev)
        self.edge_masks = [torch.full((e,), -1, dtype=torch.int32, device=dev) for _ in range(num_layers)]
        self.node_degs = [torch.zeros(n, dtype=torch.int32, device=dev) for _ in range(num_layers)]


class _TrainingLoss(torch.autograd.Function):
    """Mean negative log-likelihood of log_softmax over the training rows in two kernels each way."""

    @staticmethod
    def forward(ctx, logits, rows, labels):
        ctx.save_for_backward(logits, labels)
        ctx.num_rows = rows.numel()
        return gnnadvisor().nll_forward(logits, rows, labels)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, d_loss):
        logits, labels = ctx.saved_tensors
        return gnnadvisor().nll_backward(d_loss.contiguous(), logits, labels, ctx.num_rows), None, None


_LOSS, _LOSS_PARTS = _TrainingLoss, _parts(_TrainingLoss) if _is_torchs(_TrainingLoss.apply) else None


class Net(torch.nn.Module):
    """The reference's model (EPPGCN/gcn_main.py:190-208): conv -> relu -> ... -> conv.  With
    ``fuse_relu`` (default) the activation between two layers is applied by the consuming layer
    while it loads its input instead of by a separate F.relu pass; the function computed is the
    same."""

    def __init__(self, dataset: GraphDataset, hidden: int, num_layers: int, weight_seed: int = None,
                 fuse_relu: bool = True):
        super().__init__()
        self.num_layers = num_layers
        self.fuse_relu = fuse_relu
        self.convs = torch.nn.ModuleList()
        for i in range(num_layers):
            fan_in = hidden if i != 0 else dataset.num_features
            fan_out = hidden if i < num_layers - 1 else dataset.num_classes
            conv = GCNConv(fan_in, fan_out, relu_input=fuse_relu and i != 0)
            if weight_seed is not None:
                with torch.no_grad():
                    conv.weights.copy_(graphs.uniform_weights(weight_seed + i, fan_in, fan_out))
            self.convs.append(conv)

    def forward(self, x, inputInfo, mask_props, back_props, isFirstIter, isBackModeNet):
        for i in range(self.num_layers):
            info = inputInfo.set_input() if i == 0 else inputInfo.set_hidden()
            x = self.convs[i](x, info, mask_props[i], back_props[i], isFirstIter, isBackModeNet)
            if i < self.num_layers - 1 and not self.fuse_relu:
                x = F.relu(x)
        return x


def _step_hooks(opt):
    """Where torch keeps the callables that run around an optimizer's step."""
    return ((opt, "_optimizer_step_pre_hooks"), (opt, "_optimizer_step_post_hooks"),
            (torch_optimizer, "_global_optimizer_pre_hooks"), (torch_optimizer, "_global_optimizer_post_hooks"))


class Trainer:
    """Wiring of EPPGCN/gcn_main.py: decider -> build_part -> mask/back records -> Net -> Adam."""

    def __init__(self, graph: graphs.Graph, dim=96, hidden=16, num_classes=22, num_layers=2, train_ratio=0.1,
                 train_mask=None, backsize_mode="constant", backsize=32, labels="ones", weight_seed=3, lr=0.01,
                 fuse_relu=True, dataset=None, part_size=32, dim_worker=32, warp_per_block=8, shared_mem=100,
                 manual_mode=False, verbose=False, prune=True):
        """``dataset``: a loaded ``eppgcn_amd.dataset.custom_dataset`` (or any object with the same
        attributes) to train on instead of synthetic features over ``graph``.  ``part_size`` ...
        ``manual_mode`` are the driver's forward launch flags (EPPGCN/gcn_main.py:34-40).  ``prune=False``: the
        backward of every layer runs the unpruned aggregation (the module's ``backward`` export) instead of the
        pruned one over the prepared path - the ablation next to which the pruned times are read."""
        self.prune = bool(prune)
        self.GNNA = gnnadvisor()
        self.backsize_mode, self.backsize = backsize_mode, backsize
        if dataset is not None:
            ds = dataset
            dim, num_classes, num_layers = ds.num_features, ds.num_classes, ds.num_layers
        else:
            ds = GraphDataset(graph, dim, num_classes, num_layers, train_mask, train_ratio, labels)
        self.dataset = ds
        self.num_layers = num_layers
        info = inputProperty(ds.row_pointers, ds.column_index, ds.degrees, part_size, dim_worker, warp_per_block,
                             shared_mem, hiddenDim=hidden, dataset_obj=ds, manual_mode=manual_mode, verbose=verbose)
        info.decider()
        if verbose:
            info.set_input().print_param()
            info.set_hidden().print_param()
        part_ptr, part2node = self.GNNA.build_part(info.partSize, ds.row_pointers)
        info.partPtr, info.part2Node = part_ptr.int(), part2node.int()
        self.inputInfo = info
        self.mask_props: List[maskInputProperty] = []
        self.back_props: List[backInputProperty] = []
        for i in range(num_layers):
            src = ds.ngh_masks[i - 1] if i != 0 else ds.train_mask
            dst = ds.ngh_masks[i] if i < num_layers - 1 else ds.empty_mask
            width = hidden if i < num_layers - 1 else num_classes
            self.mask_props.append(maskInputProperty(src, dst, ds.edge_masks[num_layers - 1 - i],
                                                     ds.node_degs[num_layers - 1 - i], num_layers, i + 1, width))
            self.back_props.append(backInputProperty(degrees=ds.degrees, dim=width, layer=i + 1))
            self.back_props[-1].unpruned = not self.prune
        self.model = Net(ds, hidden, num_layers, weight_seed, fuse_relu).to(ds.x.device)
        self.optimizer = torch.optim.Adam(self.model.parameters(), lr=lr)
        self.for_time = self.loss_time = self.back_time = self.build_time = 0.0
        self.losses: List[float] = []
        self.train_idx = self.train_y = None       # set by the first epoch, or by the caller
        self._unit_gradient = None                 # a one like the loss, and what it is valid for
        self.kept_edges = [None] * num_layers      # per conv layer, filled by build_back_part

    def build_back_part(self):
        """EPPGCN/gcn_main.py:151-168 ('net' mode, which needs an unpublished predictor, is not offered)."""
        ds = self.dataset
        for i in range(self.num_layers):
            ids, edge_list, info = self.GNNA.compact_back_edge(ds.edge_masks[i], self.inputInfo.column_index)
            valid_len = int(info[0].item())
            if self.backsize_mode == "map":
                part_size = self.GNNA.get_map_back_part_size(ds.node_degs[i], valid_len)
            elif self.backsize_mode == "wave64":
                part_size = self.GNNA.get_wave64_back_part_size(ds.node_degs[i], valid_len)
            else:
                part_size = max(1, self.backsize)
            part_pointer, num_parts = self.GNNA.split_back_part(ds.node_degs[i], ds.num_edges, part_size)
            self.back_props[i].fillProperty(ids, part_pointer, edge_list, part_size, int(num_parts[0].item()))
            self.kept_edges[i] = valid_len
            ds.edge_masks[i] = None      # the marking buffer is not needed after compaction

    # Training rows and their labels.  The loss kernels read them from row_labels (int32 class of every training row, -1 for
    # the other rows), made by _select_training_rows; rows or labels that the caller sets drop it.
    @property
    def train_idx(self):
        return self._train_idx

    @train_idx.setter
    def train_idx(self, rows):
        self._train_idx, self.row_labels = rows, None

    @property
    def train_y(self):
        return self._train_y

    @train_y.setter
    def train_y(self, labels):
        self._train_y, self.row_labels = labels, None

    def _select_training_rows(self, classes):
        """The training rows and their labels (`classes`: columns of the model's output), worked out once
        (EPPGCN/gcn_main.py:252-253 selects them with the boolean mask, a device-to-host round trip per epoch)."""
        ds = self.dataset
        self.train_idx = ds.train_mask.nonzero().squeeze(1)
        self.train_y = ds.y[self.train_idx]
        if self.train_y.numel():
            lo, hi = torch.stack(torch.aminmax(self.train_y)).tolist()
            if not 0 <= lo <= hi < classes:
                raise ValueError("a label of the training rows lies outside the %d classes" % classes)
        self.row_labels = torch.where(ds.train_mask.bool(), ds.y, -1).int()
        self._row_versions = (self.train_idx._version, self.train_y._version)

    def _loss(self, out):
        """Mean negative log-likelihood of the training rows (F.nll_loss of F.log_softmax, EPPGCN/gcn_main.py:252-253): in
        the library's kernels for what ``Net`` returns, in torch operations for a model of the caller's whose output is of
        another type, layout or row count, and for rows or labels that the caller has set or changed."""
        selected = self.row_labels is not None and self._row_versions == (self.train_idx._version, self.train_y._version)
        if (selected and out.dtype == torch.float32 and out.dim() == 2 and out.is_contiguous()
                and out.shape[0] == self.row_labels.numel()):
            ops = gnnadvisor()
            if (_TrainingLoss is _LOSS and _parts(_TrainingLoss) == _LOSS_PARTS
                    and getattr(ops, "native_functions", ())[3:] == (ops.nll_forward, ops.nll_backward)
                    and type(out) is torch.Tensor):
                loss = ops.training_loss(out, self.train_idx, self.row_labels)      # _TrainingLoss in native code
                if loss is not None:
                    return loss
            return _TrainingLoss.apply(out, self.train_idx, self.row_labels)
        logp = F.log_softmax(out.index_select(0, self.train_idx), dim=1)
        return -logp.gather(1, self.train_y.unsqueeze(1)).mean()

    def _zero_grad(self):
        """``optimizer.zero_grad()``, without torch's way round its own Adam (14 us, a fifteenth of a small graph's epoch)."""
        opt = self.optimizer
        if (type(opt) is not torch.optim.Adam or "zero_grad" in vars(opt) or not _is_torchs(torch.optim.Adam.zero_grad)
                or any(type(w) is not torch.nn.Parameter for group in opt.param_groups for w in group["params"])):
            return opt.zero_grad()
        self.GNNA.drop_gradients([w for group in opt.param_groups for w in group["params"]])

    def _backward(self, loss):
        """``loss.backward()`` with a gradient of one that is kept, where autograd would make one (a launch per epoch): for the
        library's own loss whose gradient nobody is handed - a function of another's may write to it unseen, through ``data`` -
        and outside a capture, whose graph may outlive the trainer."""
        if (type(loss) is not torch.Tensor or loss._backward_hooks or loss.retains_grad
                or not self.GNNA.gradient_stays_unseen(loss) or torch.cuda.is_current_stream_capturing()):
            return loss.backward()
        kept = self._unit_gradient
        stream = torch.cuda.current_stream(loss.device)      # a fill on another stream may not have run yet
        if kept is None or kept[1:] != (kept[0]._version, loss.device, stream):
            one = torch.ones_like(loss, requires_grad=False)
            kept = self._unit_gradient = one, one._version, loss.device, stream
        loss.backward(kept[0])

    def _adam_in_one_launch(self):
        """The optimizer's step in the library's kernel, with the rounding and the state of torch's own; False, with nothing
        changed, when it is torch's to take: another optimizer or form of Adam, options, hooks, a scheduler or a wrapper on its
        step or its class's, a first step (it makes the state), weights of another type or layout (``GNNA.adam_step`` looks at
        those)."""
        opt = self.optimizer
        if type(opt) is not torch.optim.Adam or "step" in vars(opt) or not _is_torchs(torch.optim.Adam.step):
            return False
        if any(getattr(owner, name, True) for owner, name in _step_hooks(opt)) or len(opt.param_groups) != 1:
            return False
        group = opt.param_groups[0]
        if (group["weight_decay"] or group["amsgrad"] or group["maximize"] or group["capturable"] or group["differentiable"]
                or group["fused"] or group["foreach"] is False or type(group["lr"]) is not float):
            return False
        weights, grads, averages, squares, steps = [], [], [], [], []
        for w in group["params"]:
            if w.grad is None:
                continue
            state = opt.state.get(w) or {}
            tensors = w.grad, state.get("exp_avg"), state.get("exp_avg_sq"), state.get("step")
            if type(w) is not torch.nn.Parameter or any(type(t) is not torch.Tensor for t in tensors):
                return False
            for column, t in zip((weights, grads, averages, squares, steps), (w, *tensors)):
                column.append(t)
        beta1, beta2 = group["betas"]
        if type(beta1) is not float or type(beta2) is not float:
            return False
        return self.GNNA.adam_step(weights, grads, averages, squares, steps, group["lr"], beta1, beta2, group["eps"])

    def train_step(self, is_first_iter: bool, record_loss: bool = False, phase_timers: bool = True):
        """One epoch.  ``phase_timers`` keeps the reference's three host synchronisations per epoch
        that split the time into forward / loss / backward (EPPGCN/gcn_main.py:242,254,260); without
        them the epoch is issued asynchronously and only the caller synchronises."""
        ds = self.dataset
        sync = torch.cuda.synchronize if phase_timers else (lambda: None)
        self.model.train()
        self._zero_grad()
        t = time.perf_counter()
        out = self.model(ds.x, self.inputInfo, self.mask_props, self.back_props, is_first_iter, False)
        sync()
        self.for_time += time.perf_counter() - t
        if is_first_iter:
            t = time.perf_counter()
            self.build_back_part()
            torch.cuda.synchronize()
            self.build_time += time.perf_counter() - t
        t = time.perf_counter()
        if self.train_idx is None:
            self._select_training_rows(out.shape[1])
        loss = self._loss(out)
        sync()
        self.loss_time += time.perf_counter() - t
        t = time.perf_counter()
        self._backward(loss)
        sync()
        self.back_time += time.perf_counter() - t
        if not self._adam_in_one_launch():
            self.optimizer.step()
        if record_loss:
            self.losses.append(float(loss.item()))
        return loss

    def run(self, epochs=100, warmup=10, record_loss=False, kernel_timing=False, phase_timers=True):
        """10 warm-up epochs (the first prepares the path), timers cleared, then `epochs` timed
        epochs between two synchronisations (EPPGCN/gcn_main.py:272-292)."""
        for i in range(warmup):
            self.GNNA.set_timing(i == 0)      # path marking runs once, here: keep its time for print_time
            self.train_step(i == 0, record_loss)
        self.for_time = self.loss_time = self.back_time = 0.0
        self.GNNA.clear_time()
        self.GNNA.set_timing(bool(kernel_timing))
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(epochs):
            self.train_step(False, record_loss, phase_timers)
        torch.cuda.synchronize()
        total = time.perf_counter() - t
        self.GNNA.set_timing(False)
        res = {"epochs": epochs, "warmup": warmup, "Time": round(total, 6), "for_time": round(self.for_time, 6),
               "loss_time": round(self.loss_time, 6), "back_time": round(self.back_time, 6),
               "build_time": round(self.build_time, 6),
               "backward_group_sizes": [b.partSize for b in self.back_props],
               "backward_groups": [b.numParts for b in self.back_props],
               "kept_edges": list(self.kept_edges), "pruned": self.prune}
        if kernel_timing:
            res["for_agg_time"] = round(self.GNNA.get_time_ms(0) / 1e3, 6)
            res["back_agg_time"] = round(self.GNNA.get_time_ms(1) / 1e3, 6)
            res["mask_time"] = round(self.GNNA.get_time_ms(2) / 1e3, 6)
            # l{k}_back_agg_time of the reference's report (EPPGCN_kernel.cu:96-106); the unpruned ablation has no
            # per-layer timers (its entry point has no layer argument)
            res["layer_back_agg_time"] = [round(self.GNNA.get_time_ms(101 + k) / 1e3, 6) for k in range(self.num_layers)]
        return res


    # ------------------------------------------------------------------ whole epoch as one HIP graph
    def capture_epoch(self):
        """Records one steady-state epoch (forward, loss, backward, Adam step) into a HIP graph
        and returns (graph, loss tensor the replays overwrite).  The path must be prepared
        (run at least one first-iteration step before).  The optimizer is rebuilt with
        capturable state; the layer ops allocate from the graph's private pool and the library
        itself records kernel nodes only."""
        ds = self.dataset
        if self.train_idx is None:
            raise RuntimeError("run a first-iteration train_step before capturing")
        state = self.optimizer.state_dict()
        self.optimizer = torch.optim.Adam(self.model.parameters(), lr=state["param_groups"][0]["lr"], capturable=True)
        if state["state"]:
            for entry in state["state"].values():
                if not torch.is_tensor(entry["step"]) or not entry["step"].is_cuda:
                    entry["step"] = torch.as_tensor(float(entry["step"]), dtype=torch.float32, device=ds.x.device)
            for group in state["param_groups"]:
                group["capturable"] = True
            self.optimizer.load_state_dict(state)

        def epoch():
            self.optimizer.zero_grad(set_to_none=True)
            out = self.model(ds.x, self.inputInfo, self.mask_props, self.back_props, False, False)
            loss = self._loss(out)
            loss.backward()
            self.optimizer.step()
            return loss

        self.GNNA.set_timing(False)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):            # warm-up on a side stream, as graph capture requires
            for _ in range(3):
                epoch()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            loss = epoch()
        return graph, loss

    def run_graphed(self, epochs=100):
        """`epochs` replays of the captured epoch between two synchronisations."""
        graph, loss = self.capture_epoch()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(epochs):
            graph.replay()
        torch.cuda.synchronize()
        return {"epochs": epochs, "Time": round(time.perf_counter() - t, 6), "last_loss": float(loss.item())}


def time_gpu_training(graph, wl=None, epochs=100, warmup=10, backsize_mode="constant", backsize=32):
    """100-epoch time of the 2-layer GCN (96 -> 16 -> 22) on the GPU; runs twice: once untimed
    per kernel (the headline `Time`), once with per-kernel events for the aggregation split."""
    train_mask = None if wl is None else wl.train_mask
    tr = Trainer(graph, train_mask=train_mask, backsize_mode=backsize_mode, backsize=backsize)
    res = tr.run(epochs, warmup)
    res["Time_without_phase_timers"] = tr.run(epochs, 0, phase_timers=False)["Time"]
    timed = tr.run(min(epochs, 20), 0, kernel_timing=True)
    res["agg_ms_per_epoch_in_training"] = round(
        (timed["for_agg_time"] + timed["back_agg_time"]) * 1e3 / timed["epochs"], 4)
    res["mask_time"] = timed["mask_time"]
    try:                                     # the same epoch replayed from one HIP graph
        res["Time_hip_graph"] = tr.run_graphed(epochs)["Time"]
    except Exception as exc:                 # capture support must never hide the eager figures
        res["Time_hip_graph"] = repr(exc)
    return res


def smoke_step(graph, wl=None):
    tr = Trainer(graph, train_mask=None if wl is None else wl.train_mask, backsize=8, labels="uniform")
    first = float(tr.train_step(True).item())
    for _ in range(5):
        last = float(tr.train_step(False).item())
    assert last == last and last < first, f"loss did not decrease: {first} -> {last}"


# ------------------------------------------------------------------ host-CPU comparison run
class _SymSparseMM(torch.autograd.Function):
    """A @ X through torch.sparse.mm; the backward uses A's symmetry (dX = A @ dY) so that no
    transposed copy of A is built per step.  Both products are timed."""

    @staticmethod
    def forward(ctx, a, x, clock):
        ctx.a, ctx.clock = a, clock
        t = time.perf_counter()
        y = torch.sparse.mm(a, x)
        clock[0] += time.perf_counter() - t
        return y

    @staticmethod
    def backward(ctx, dy):
        t = time.perf_counter()
        dx = torch.sparse.mm(ctx.a, dy.contiguous())
        ctx.clock[0] += time.perf_counter() - t
        return None, dx, None


def time_cpu_sparse_training(graph, train_mask, epochs=100, max_seconds=60.0, dim=96, hidden=16,
                             num_classes=22, lr=0.01, weight_seed=3):
    """The same 2-layer GCN through PyTorch CPU sparse aggregation on the host cores.  Runs at
    least 2 and at most `epochs` epochs within `max_seconds` after one warm-up epoch and
    extrapolates linearly to `epochs` (stated in the result)."""
    g = graph.to("cpu")
    n = g.num_nodes
    row = g.row_index()
    vals = g.degrees[row] * g.degrees[g.column_index.long()]
    a = torch.sparse_csr_tensor(g.row_pointers.long(), g.column_index.long(), vals, size=(n, n))
    x = graphs.normal32(1, (n, dim), "cpu")
    y = torch.ones(n, dtype=torch.long)
    mask = train_mask.cpu()
    w0 = graphs.uniform_weights(weight_seed, dim, hidden).requires_grad_()
    w1 = graphs.uniform_weights(weight_seed + 1, hidden, num_classes).requires_grad_()
    opt = torch.optim.Adam([w0, w1], lr=lr)
    clock = [0.0]

    def epoch():
        opt.zero_grad()
        h = F.relu(_SymSparseMM.apply(a, x @ w0, clock))
        out = _SymSparseMM.apply(a, h @ w1, clock)
        loss = F.nll_loss(F.log_softmax(out, dim=1)[mask], y[mask])
        loss.backward()
        opt.step()
        return float(loss.item())

    epoch()
    clock[0] = 0.0
    done = 0
    t0 = time.perf_counter()
    while done < epochs and (done < 2 or time.perf_counter() - t0 < max_seconds):
        epoch()
        done += 1
    dt = time.perf_counter() - t0
    return {"epochs_run": done, "seconds_run": round(dt, 3), "Time_extrapolated_to": epochs,
            "Time": round(dt / done * epochs, 3), "agg_ms_per_epoch": round(clock[0] / done * 1e3, 2),
            "threads": torch.get_num_threads(), "host_cpus": os.cpu_count(),
            "note": "torch.sparse.mm (CSR, fp32) forward and backward; linear extrapolation from epochs_run"}
