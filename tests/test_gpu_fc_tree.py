"""Three LogicLayers (the last two halving) and a GroupSum as one operation (difflogic/fc_tree.py): training against the float64
oracle at the edges of its lane layouts (1, 2 and 4 samples per lane, partly filled wavefronts, several passes over a
row), packed class counts against the modules one after the other."""
import pytest
import torch

import convlogic_amd as C
from convlogic_amd.convlogic.model import _forward
from convlogic_amd.difflogic import fc_tree
from oracle import convlogic_oracle as O
from tests.gpu_util import DEV, assert_grad_close, set_knobs

pytestmark = pytest.mark.gpu


def tail(in_dim, roots, k, seed):
    torch.manual_seed(seed)
    dims = [in_dim, 4 * roots, 2 * roots, roots]
    return [C.LogicLayer(a, b, implementation="cuda").to(DEV) for a, b in zip(dims, dims[1:])], C.GroupSum(k, tau=3.0)


@pytest.mark.parametrize("batch", [1, 4, 63, 64, 65, 68, 126, 128, 129, 132, 256, 258, 260, 513, 516])
@pytest.mark.parametrize("in_dim,roots,k", [(8, 2, 1), (40, 130, 10), (700, 663, 3)])
def test_training_against_the_oracle(batch, in_dim, roots, k):
    layers, gs = tail(in_dim, roots, k, batch + roots)
    plan = fc_tree.tree_plan(*layers)
    assert plan is not None and plan.roots == roots
    x = torch.rand(in_dim, batch, device=DEV).requires_grad_(True)
    go = torch.randn(batch, k, device=DEV)
    y = fc_tree.tree_train(layers, gs, x, plan)
    y.backward(go)
    h = xl = x.detach().double().cpu().t().contiguous().requires_grad_(True)
    ws = [m.weights.detach().double().cpu().requires_grad_(True) for m in layers]
    for m, w in zip(layers, ws):
        h = O.logic_fc_forward(h, m.indices_0.cpu(), m.indices_1.cpu(), torch.softmax(w, -1))
    want = O.group_sum(h, k, gs.tau)
    want.backward(go.double().cpu())
    # values: at most roots / k terms of one rounding error each, relative to a sum of as many values around 0.5
    assert (y.detach().double().cpu() - want.detach()).norm() <= 1e-6 * want.detach().norm()
    assert_grad_close(x.grad.t(), xl.grad, rel=1e-4, name="grad_x")
    for i, (m, w) in enumerate(zip(layers, ws)):
        assert_grad_close(m.weights.grad, w.grad, rel=1e-4, name=f"grad_logits {i}")
    grads = [x.grad.clone()] + [m.weights.grad.clone() for m in layers]
    for t in (x, *(m.weights for m in layers)):
        t.grad = None
    fc_tree.tree_train(layers, gs, x, plan).backward(go)
    assert all(torch.equal(a, b) for a, b in zip(grads, [x.grad] + [m.weights.grad for m in layers]))


# (words of 64 samples: lanes along roots below 32 of them, one block of columns, a partly filled second one; classes of fewer
# roots than a workgroup has lanes for, sliced classes, and more roots than a workgroup's counters hold)
@pytest.mark.parametrize("samples", [1, 64, 100, 1000, 2048, 2112, 20000])
@pytest.mark.parametrize("in_dim,roots,k", [(8, 3, 3), (100, 640, 10), (3000, 5000, 2), (64, 40000, 1)])
def test_packed_counts_equal_the_modules(samples, in_dim, roots, k):
    layers, gs = tail(in_dim, roots, k, samples + roots)
    for m in layers:
        m.eval()
    words = -(-samples // 64)
    bits = torch.randint(-2**63, 2**63 - 1, (in_dim, words), dtype=torch.int64, device=DEV)

    def packed():
        p = C.PackBitsTensor.__new__(C.PackBitsTensor)
        p.t, p.bit_count, p.pad_len, p.image = bits, 64, words * 64 - samples, False
        return p

    with torch.no_grad():
        want = torch.nn.Sequential(*layers, gs)(packed())
        got = fc_tree.tree_packed(layers, k, packed(), fc_tree.tree_plan(*layers))
    assert got.dtype == torch.int32 and torch.equal(got, want)


def test_wiring_that_makes_no_trees_and_rewired_layers():
    layers, gs = tail(40, 20, 2, 1)
    assert fc_tree.tree_plan(*layers) is not None
    with torch.no_grad():                                            # two operands on one neuron: no trees
        old = layers[1].indices_0[0].item()
        layers[1].indices_0[0] = layers[1].indices_1[5].item()
    assert fc_tree.tree_plan(*layers) is None
    with torch.no_grad():
        layers[1].indices_0[0] = old
        layers[0].indices_0.copy_(layers[0].indices_0.flip(0))       # another wiring of the first layer: another plan
    x = torch.rand(40, 16, device=DEV)
    y = fc_tree.tree_train(layers, gs, x, fc_tree.tree_plan(*layers))
    h = x.t()
    for m in layers:
        h = m(h)
    assert torch.allclose(y, gs(h), rtol=1e-5, atol=1e-5)
    assert fc_tree.tree_plan(layers[0], layers[2], layers[1]) is None   # not a chain of halving layers


def test_a_network_takes_its_tail_as_trees_and_equals_its_modules():
    torch.manual_seed(2)
    model = C.ConvLogicMnistModel(k_param=2, tau=6.5).to(DEV)
    x = torch.randint(0, 2, (32, 1, 28, 28), device=DEV).float()
    labels = torch.randint(0, 10, (32,), device=DEV)
    results = []
    for on in (True, False):
        model.tree_tail = on
        model.zero_grad()
        out = model(x)
        torch.nn.functional.cross_entropy(out, labels).backward()
        results.append([out.detach()] + [p.grad.clone() for p in model.parameters()])
        assert ("_Tree" in type(out.grad_fn).__name__) == on
    for i, (a, b) in enumerate(zip(*results)):
        assert_grad_close(a, b, rel=1e-4, name=f"result {i}")
    model.eval()
    bits = torch.randint(0, 2, (77, 1, 28, 28), device=DEV).bool()
    with torch.no_grad():
        counts = []
        for on in (True, False):
            model.tree_tail = on
            counts.append(model(C.PackBitsTensor(bits, 64)))
    assert torch.equal(*counts)


def test_logits_updated_between_forward_and_backward_leave_the_gradients_alone():
    layers, gs = tail(40, 20, 2, 3)
    x, go = torch.rand(40, 16, device=DEV).requires_grad_(True), torch.randn(16, 2, device=DEV)
    plan, results = fc_tree.tree_plan(*layers), []
    for update in (False, True):
        for t in (x, *(m.weights for m in layers)):
            t.grad = None
        y = fc_tree.tree_train(layers, gs, x, plan)
        if update:
            with torch.no_grad():
                for m in layers:
                    m.weights.add_(1.0).mul_(-2.0)
        y.backward(go)
        results.append([x.grad] + [m.weights.grad for m in layers])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("hook", ["register_forward_hook", "register_full_backward_hook", "register_full_backward_pre_hook", "forward"])
def test_modules_with_hooks_are_called_themselves(hook):
    torch.manual_seed(4)
    model, calls = C.ConvLogicMnistModel(k_param=1).to(DEV), []
    layer = model.network[-4]
    if hook == "forward":
        inner = layer.forward
        layer.forward = lambda x: (calls.append(1), inner(x))[1]
    else:
        getattr(layer, hook)(lambda *a: calls.append(1))
    model(torch.randint(0, 2, (4, 1, 28, 28), device=DEV).float()).sum().backward()
    assert calls == [1]
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: calls.append(type(m)))
    try:
        model(torch.randint(0, 2, (4, 1, 28, 28), device=DEV).float())
    finally:
        handle.remove()
    assert calls.count(C.LogicLayer) >= 2                              # the first two of the three (the last runs with the GroupSum)


@pytest.mark.parametrize("batch", [1, 63, 66, 128, 255, 256, 1001])
def test_evaluation_equals_the_modules(batch):
    layers, gs = tail(700, 663, 3, batch)
    net = torch.nn.Sequential(*layers, gs).eval()
    x = torch.randint(0, 2, (batch, 700), device=DEV).float()
    got = fc_tree.tree_eval(layers, gs, x.t().contiguous(), fc_tree.tree_plan(*layers))
    assert not got.requires_grad and torch.equal(got, net(x))          # class sums are whole numbers
    x = torch.rand(batch, 700, device=DEV)
    assert torch.allclose(fc_tree.tree_eval(layers, gs, x.t().contiguous(), fc_tree.tree_plan(*layers)), net(x), rtol=2e-6, atol=0)


def test_a_network_evaluates_its_tail_as_trees():
    torch.manual_seed(5)
    model = C.ConvLogicMnistModel(k_param=2).to(DEV).eval()
    x, results = torch.randint(0, 2, (33, 1, 28, 28), device=DEV).float(), []
    for on in (True, False):
        model.tree_tail = on
        results.append(model(x))
    assert torch.equal(*results) and not results[0].requires_grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_onehot_of_the_first_maximum(dtype):
    from convlogic_amd.hip import difflogic_hip
    logits = torch.randn(37, 7, 16, device=DEV, dtype=dtype)
    logits[0, 0] = 1.0                                                 # ties, NaN, infinities, zeros of both signs
    logits[0, 1, 5] = logits[0, 1, 9] = float("nan")
    logits[0, 2] = -float("inf")
    logits[0, 3, 7] = logits[0, 3, 11] = float("inf")
    logits[0, 4] = -0.0
    logits[0, 4, 6] = 0.0
    logits[0, 5] = -float("inf")
    logits[0, 5, 15] = float("nan")
    logits[0, 6] = torch.finfo(dtype).min
    got = difflogic_hip.gate_onehot(logits, dtype)
    assert got.dtype == dtype and torch.equal(got, torch.nn.functional.one_hot(logits.argmax(-1), 16).to(dtype))
    assert torch.equal(got.argmax(-1).to(torch.uint8), difflogic_hip.gate_argmax(logits))


# (the gate ids of more roots than one pass of a launch takes; 2^27 of them, 32 lanes each, were once refused)
@pytest.mark.parametrize("class_rows,k", [(1, 3), (129, 16257), (4096, 32768)])
def test_packed_counts_of_many_roots(class_rows, k):
    from convlogic_amd.hip import _lib
    roots = class_rows * k
    # every tree's leaves and middle gates are neuron 0 of their layer; the root's gate is "0" or, where logit 15 is above the others, "1"
    zero = torch.zeros(roots, 8, dtype=torch.int32, device=DEV)
    first = torch.zeros(1, 16, device=DEV)
    last = torch.zeros(roots, 16, device=DEV)
    last[:, 15] = torch.randn(roots, device=DEV)
    words = torch.randint(-2**63, 2**63 - 1, (5, 1), dtype=torch.int64, device=DEV)
    codes = torch.empty(roots, dtype=torch.int32, device=DEV)
    out = torch.empty(64, k, dtype=torch.int32, device=DEV)
    _lib.check(_lib.load().clg_fc_tree_packed(words.data_ptr(), zero.data_ptr(), zero.data_ptr(), first.data_ptr(), first.data_ptr(), last.data_ptr(),
                                              codes.data_ptr(), out.data_ptr(), 5, roots, k, 1, 64, _lib.stream_ptr(words)))
    want = (last[:, 15] > 0).view(k, class_rows).sum(1).int()
    assert torch.equal(out, want.expand(64, k))


@pytest.mark.parametrize("hard", [0, 1])
def test_ids_out_of_range_stay_inside_the_logits_and_the_probabilities(hard):
    from convlogic_amd.hip import _lib
    roots = 70
    logits = [torch.randn(n * roots, 16, device=DEV) for n in (4, 2, 1)]
    ids = torch.stack([torch.randint(0, (4 if q < 4 else 2) * roots, (roots,), dtype=torch.int32) for q in range(8)], 1)
    ids[3, 1], ids[5, 4], ids[9, 0], ids[11, 5] = 4 * roots, 2 * roots, -1, -2**31
    inside = torch.stack([ids[:, q].long().where((ids[:, q] >= 0) & (ids[:, q] < n * roots), torch.tensor(n * roots - 1))
                          for q, n in enumerate((4, 4, 4, 4, 2, 2))], 1).to(DEV)
    coef = torch.empty(roots, 7, 4, device=DEV)
    probs = torch.full((7 * roots + 64, 16), 7.0, device=DEV)             # (the rows behind the last one stay as they are)
    on_device = ids.to(DEV)
    _lib.check(_lib.load().clg_fc_tree_fold(*(l.data_ptr() for l in logits), on_device.data_ptr(), coef.data_ptr(), probs.data_ptr(), roots,
                                            hard, _lib.stream_ptr(coef)))
    tree = torch.cat([logits[0][inside[:, :4]], logits[1][inside[:, 4:]], logits[2][:, None]], 1).cpu().double()      # [roots, 7, 16]
    want = O.fold_coefficients(torch.nn.functional.one_hot(tree.argmax(-1), 16).double() if hard else torch.softmax(tree, -1))
    # a coefficient is a sum of at most 16 probabilities times 1 or 2, each a few roundings off
    assert (coef.cpu().double() - want).abs().max() <= 1e-5 and (probs[7 * roots:] == 7).all()


@pytest.mark.parametrize("at", [4, 5, 6])
def test_logits_of_another_size_are_refused(at):
    torch.manual_seed(6)
    model = C.ConvLogicMnistModel(k_param=2).to(DEV).eval()
    layer = model.network[at]
    layer.weights = torch.nn.Parameter(layer.weights.detach()[:-1].clone())
    with torch.no_grad(), pytest.raises(RuntimeError, match="shape|logits|neurons"):
        model(torch.zeros(8, 1, 28, 28, device=DEV))
    with torch.no_grad(), pytest.raises(RuntimeError, match="shape|logits|neurons"):
        model(C.PackBitsTensor(torch.zeros(8, 1, 28, 28, dtype=torch.bool, device=DEV), 64))


def assert_tail_equals_modules(model):
    """training, evaluation and packed counts with the trees and with the modules called themselves"""
    x = torch.randint(0, 2, (32, 1, 28, 28), device=DEV).float()
    results = []
    for on in (True, False):
        model.tree_tail = on
        model.train().zero_grad()
        out = model(x)
        assert ("_Tree" in type(out.grad_fn).__name__) == on
        out.square().sum().backward()
        grads = [p.grad.clone() for p in model.parameters()]
        with torch.no_grad():
            results.append([out.detach(), *grads, model.eval()(x), model(C.PackBitsTensor(x.bool(), 64))])
    # One element: a sum over 32 samples and up to 144 positions of products through seven layers, whose terms may be ten times the
    # mean element and cancel: 7 roundings of 6e-8 on each of them, sqrt(32 * 144) of a kind, 10 * 7 * 6e-8 * 68 = 3e-4 of the
    # mean.  (A wiring that did not arrive is off by the mean itself.)
    for i, (a, b) in enumerate(zip(*results)):
        assert_grad_close(a, b, rel=1e-4, rel_elem=3e-4, name=f"result {i}")


@pytest.mark.parametrize("route", ["data", "loaded on the cpu", "other layer"])
@pytest.mark.parametrize("at", [4, 5, 6])
def test_another_wiring_reaches_the_trees(route, at):
    torch.manual_seed(at)
    model = C.ConvLogicMnistModel(k_param=2).to(DEV)
    assert_tail_equals_modules(model)
    layer = model.network[at]
    if route == "data":
        layer.indices_0.data.copy_(layer.indices_0.flip(0))
        layer.invalidate()
    elif route == "other layer":
        model.network[at] = C.LogicLayer(layer.in_dim, layer.out_dim, implementation="cuda").to(DEV)
    else:
        state = C.ConvLogicMnistModel(k_param=2).state_dict()
        model.cpu().load_state_dict(state)
        model.to(DEV)
    assert_tail_equals_modules(model)


@pytest.mark.parametrize("in_dim,roots", [(1, 1), (2, 1), (8, 1), (3, 31), (40, 32), (64, 33), (700, 663), (2000, 250), (5, 5000)])
def test_the_tables_of_a_wiring(in_dim, roots):
    torch.manual_seed(in_dim + roots)
    layers = [C.LogicLayer(a, b, implementation="cuda").to(DEV) for a, b in ((in_dim, 4 * roots), (4 * roots, 2 * roots), (2 * roots, roots))]
    with torch.no_grad():                                              # some neurons read one feature twice, some features are not read
        layers[0].indices_1[::3] = layers[0].indices_0[::3]
        layers[0].indices_1[1::5] = in_dim // 2
    plan = fc_tree.tree_plan(*layers)
    a, b = ([getattr(m, name).cpu() for m in layers] for name in ("indices_0", "indices_1"))
    mid = torch.stack([a[2], b[2]], 1)
    leaf = torch.stack([a[1][mid], b[1][mid]], 2).flatten(1)
    operand = torch.stack([a[0], b[0]], 1)
    order = torch.argsort(operand.flatten(), stable=True)              # by feature, then by neuron, the first operand first
    place = torch.empty_like(order)
    place[order] = torch.arange(order.numel())
    slots = torch.arange(7 * roots).view(-1, 7)
    slot = torch.full((7 * roots,), -1)
    slot[leaf], slot[4 * roots + mid], slot[6 * roots:] = slots[:, :4], slots[:, 4:6], slots[:, 6]
    want = operand[leaf].flatten(1), place.view(-1, 2)[leaf].flatten(1), torch.cat([leaf, mid, torch.zeros_like(mid)], 1), slot
    for got, table in zip((plan.rows, plan.pos, plan.ids, plan.slot), want):
        assert torch.equal(got.cpu().long(), table.flatten())


class Head(torch.nn.Module):
    """a network that is nothing but its fully connected end"""

    def __init__(self, in_dim=40, roots=20, k=2):
        super().__init__()
        layers = [C.LogicLayer(a, b, implementation="cuda") for a, b in ((in_dim, 4 * roots), (4 * roots, 2 * roots), (2 * roots, roots))]
        self.network = torch.nn.Sequential(torch.nn.Flatten(), *layers, C.GroupSum(k, tau=3.0))

    def forward(self, x):
        return _forward(self, x)


def test_a_recorded_step_replays_the_loaded_wiring():
    torch.manual_seed(7)
    model, other = Head().to(DEV), Head().to(DEV)
    batches = [(torch.rand(32, 40, device=DEV), torch.randint(0, 2, (32,), device=DEV)) for _ in range(3)]
    loss_of = lambda x, y: torch.nn.functional.cross_entropy(model(x), y)
    step = C.GraphedStep(loss_of, batches[0], model.parameters())
    plan = fc_tree.tree_plan(*model.network[1:4])
    addresses = [t.data_ptr() for t in (plan.rows, plan.pos, plan.ids, plan.slot)]
    own, another = ({k: v.clone() for k, v in m.state_dict().items()} for m in (model, other))
    for state, between in ((own, True), (another, False), (own, False), (another, True)):
        model.load_state_dict(state)
        if between:                                                    # an eager pass on the loaded state before the replays
            with torch.no_grad():
                model.eval()(batches[0][0])
            model.train()
        other = [torch.randint(0, 2**31 - 1, (1 << 12,), dtype=torch.int32, device=DEV) for _ in range(32)]   # (takes freed memory)
        replayed = []
        for x, y in batches:
            loss = step(x, y)
            torch.cuda.synchronize()
            replayed.append([loss.clone()] + [p.grad.clone() for p in model.parameters()])
        for (x, y), got in zip(batches, replayed):
            grads = [p.grad for p in model.parameters()]
            for p in model.parameters():
                p.grad = None
            loss = loss_of(x, y)
            loss.backward()
            assert all(torch.equal(a, b) for a, b in zip(got, [loss.detach()] + [p.grad for p in model.parameters()]))
            for p, g in zip(model.parameters(), grads):
                p.grad = g                                              # the step's own
        assert fc_tree.tree_plan(*model.network[1:4]) is plan
    assert addresses == [t.data_ptr() for t in (plan.rows, plan.pos, plan.ids, plan.slot)]


def test_a_wiring_changed_between_forward_and_backward_is_refused():
    torch.manual_seed(8)
    model = C.ConvLogicMnistModel(k_param=2).to(DEV)
    for at in (4, 5, 6):
        out = model(torch.zeros(4, 1, 28, 28, device=DEV))
        with torch.no_grad():
            model.network[at].indices_0.copy_(model.network[at].indices_0.flip(0))
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            out.sum().backward()


def test_a_recording_without_the_tables_takes_the_modules():
    torch.manual_seed(9)
    model, x = Head().to(DEV).eval(), torch.randint(0, 2, (64, 40), device=DEV).float()
    with torch.no_grad():
        want = model.network(x)                                        # the modules have checked their wirings, no tables yet
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.network(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = model(x)
        for _ in range(3):
            x.copy_(torch.randint(0, 2, x.shape, device=DEV).float())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, model.network(x))
            assert torch.equal(got, model(x))


def test_a_wrapped_network_and_one_with_a_forward_of_its_own_are_called():
    class Doubled(torch.nn.Sequential):
        def forward(self, x):
            return 2 * super().forward(x)

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            return self.inner(x)

    torch.manual_seed(10)
    model, x = Head().to(DEV).eval(), torch.randint(0, 2, (64, 40), device=DEV).float()
    with torch.no_grad():
        want, network = model(x), model.network
        model.network = Doubled(*network)
        assert torch.equal(model(x), 2 * want)
        model.network = Wrapped(network)
        assert torch.equal(model(x), want)


@pytest.mark.parametrize("k,rows,samples,by_trees", [(600, 1, 64, False), (600, 1, 4096, False), (600, 1, 4097, True), (511, 1, 64, True),
                                                     (600, 16, 256, False), (600, 17, 64, True), (600, 16, 257, True)])
def test_many_small_classes_take_the_modules(k, rows, samples, by_trees, monkeypatch):
    from convlogic_amd.convlogic import model as M
    torch.manual_seed(12)
    model, bits = Head(k * rows, k * rows, k).to(DEV).eval(), torch.rand(samples, k * rows, device=DEV) < 0.5
    calls = []
    monkeypatch.setattr(M, "tree_packed", lambda *a: calls.append(1) or fc_tree.tree_packed(*a))
    with torch.no_grad():
        assert torch.equal(model(C.PackBitsTensor(bits, 64)), model.network(C.PackBitsTensor(bits, 64)))
    assert bool(calls) == by_trees


def test_more_classes_than_the_tree_kernels_take():
    # (the float class sums take no more either: they refuse, as for the modules)
    torch.manual_seed(11)
    model, bits = Head(140000, 70000, 70000).to(DEV).eval(), torch.rand(3, 140000, device=DEV) < 0.5
    with torch.no_grad():
        assert torch.equal(model(C.PackBitsTensor(bits, 64)), model.network(C.PackBitsTensor(bits, 64)))
        with pytest.raises(RuntimeError, match="k <= 65535"):
            model(bits.float())


@pytest.mark.parametrize("batch", [3, 66, 256])
@pytest.mark.parametrize("wanted", [(1, 0, 0, 0), (0, 1, 1, 1), (0, 0, 1, 0), (1, 1, 0, 1)])
def test_gradients_that_are_not_wanted_are_not_made(wanted, batch):
    layers, gs = tail(40, 130, 10, batch)
    x, go = torch.rand(40, batch, device=DEV), torch.randn(batch, 10, device=DEV)
    inputs = [x] + [m.weights for m in layers]
    results = []
    for some in ((1, 1, 1, 1), wanted):
        for t, want in zip(inputs, some):
            t.grad = None
            t.requires_grad_(bool(want))
        fc_tree.tree_train(layers, gs, x, fc_tree.tree_plan(*layers)).backward(go)
        results.append([t.grad for t in inputs])
    for all_of_them, some, want in zip(*results, wanted):
        assert torch.equal(all_of_them, some) if want else some is None


def test_a_frozen_end_allocates_no_gradients():
    layers, gs = tail(40, 1300, 10, 1)
    x, go = torch.rand(40, 256, device=DEV), torch.randn(256, 10, device=DEV)
    y = fc_tree.tree_train(layers, gs, x, fc_tree.tree_plan(*layers))
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y.backward(go)                                                     # x needs no gradient: no operand gradients [8 roots, batch]
    assert torch.cuda.max_memory_allocated() - before < 8 * 1300 * 256 * 4


@pytest.mark.parametrize("batch,pitch", [(3, 64), (100, 128), (60, 96), (200, 256), (257, 512), (300, 304)])
def test_what_a_row_holds_behind_the_batch_adds_nothing(batch, pitch):
    from convlogic_amd.hip import _lib
    lib, ptr = _lib.load(), lambda t: t.data_ptr()
    layers, _ = tail(40, 130, 10, batch)
    plan, (in_dim, roots, k) = fc_tree.tree_plan(*layers), (40, 130, 10)
    x, go = torch.rand(in_dim, pitch, device=DEV), torch.randn(batch, k, device=DEV)
    start = layers[0].given_x_indices_of_y_start
    results = []
    for behind in (0.0, float("nan"), float("inf")):
        x[:, batch:] = behind
        coef, probs, out = (torch.empty(*s, device=DEV) for s in ((roots, 28), (7 * roots, 16), (batch, k)))
        _lib.check(lib.clg_fc_tree_fold(*(ptr(m.weights) for m in layers), ptr(plan.ids), ptr(coef), ptr(probs), roots, 0, _lib.stream_ptr(x)))
        partial = torch.empty(lib.clg_fc_tree_partial_elems(roots, k, batch, pitch), device=DEV)
        _lib.check(lib.clg_fc_tree_forward(ptr(x), ptr(plan.rows), ptr(coef), ptr(partial), ptr(out), in_dim, roots, k, batch, pitch, 3.0, _lib.stream_ptr(x)))
        grads, gx = [torch.empty(n * roots, 16, device=DEV) for n in (4, 2, 1)], torch.empty(in_dim, pitch, device=DEV)
        rowgrad, sums = torch.empty(8 * roots, pitch, device=DEV), torch.empty(roots, 28, device=DEV)
        _lib.check(lib.clg_fc_tree_backward(ptr(x), ptr(plan.rows), ptr(plan.pos), ptr(plan.slot), ptr(coef), ptr(go), ptr(probs), *map(ptr, grads),
                                            ptr(rowgrad), ptr(sums), ptr(start), ptr(gx), in_dim, roots, k, batch, pitch, 3.0, _lib.stream_ptr(x)))
        results.append([out, *grads, gx[:, :batch].clone()])
    for other in results[1:]:
        for i, (a, b) in enumerate(zip(results[0], other)):
            assert torch.isfinite(a).all() and torch.equal(a, b), f"result {i}"


@pytest.mark.parametrize("batch", [1, 3, 64, 100])
@pytest.mark.parametrize("roots,k", [(4097, 1), (9000, 1), (40000, 1), (20000, 2)])
def test_one_or_two_large_classes(roots, k, batch):
    # more slices of a class than the 64 of larger launches: the sums against float64, the gradients against the modules
    model = Head(50, roots, k).to(DEV)
    x, go = torch.rand(batch, 50, device=DEV).requires_grad_(True), torch.randn(batch, k, device=DEV)
    results = []
    for on in (True, False):
        model.tree_tail = on
        model.train().zero_grad()
        x.grad = None
        out = model(x)
        out.backward(go)
        results.append([out.detach(), x.grad] + [p.grad for p in model.parameters()])
    h = x.detach().double()
    for m in list(model.network)[1:4]:
        a, b = h[:, m.indices_0], h[:, m.indices_1]
        c = O.fold_coefficients(torch.softmax(m.weights.detach().double(), -1).cpu()).to(DEV)
        h = c[:, 0] * a * b + c[:, 1] * a + c[:, 2] * b + c[:, 3]
    want = h.view(batch, k, -1).sum(-1) / 3.0
    # at most 512 + 40 additions in a row of values around 0.5, each a rounding of the sum so far: 0.5 * 552 * 6e-8 of it at worst
    assert ((results[0][0].double() - want).abs() <= 2e-5 * want).all()
    for i, (a, b) in enumerate(zip(*results)):
        assert_grad_close(a, b, rel=1e-4, name=f"result {i}")


def test_one_network_first_used_by_several_threads_and_streams():
    # every thread's first call meets a wiring that nobody has checked, tables that nobody has made, or those of another stream
    import threading
    torch.manual_seed(13)
    model = Head(300, 2000, 10).to(DEV).eval()
    x = [torch.randint(0, 2, (n, 300), device=DEV).float() for n in (64, 100, 257, 1000)]
    with torch.no_grad():
        want = [(model.network(t), model.network(C.PackBitsTensor(t.bool(), 64))) for t in x]
    for _ in range(5):
        for m in list(model.network)[1:4]:
            m.invalidate()
        got, start = [None] * len(x), threading.Barrier(len(x))

        def work(i):
            with torch.cuda.stream(torch.cuda.Stream()), torch.no_grad():
                start.wait()
                got[i] = model(x[i]), model(C.PackBitsTensor(x[i].bool(), 64))
                torch.cuda.current_stream().synchronize()

        torch.cuda.synchronize()
        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(x))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for (a, b), (c, d) in zip(got, want):
            assert torch.equal(a, c) and torch.equal(b, d)


# neurons in their own order and roots in theirs: a wavefront's 64, parts of one, layers that end inside one
@pytest.mark.parametrize("roots", [1, 9, 64, 130, 663])
@pytest.mark.parametrize("stream_mb", ["0", "100000"])
def test_folding_by_slots_gives_the_bits_of_folding_by_roots(roots, stream_mb, monkeypatch):
    from convlogic_amd.hip import _lib
    layers, _ = tail(max(2, roots), roots, 1, roots)
    plan, lib = fc_tree.tree_plan(*layers), _lib.load()
    logits = [torch.randn_like(m.weights) * 3 for m in layers]
    set_knobs(monkeypatch, CLG_STREAM_MB=stream_mb)
    got = []
    for table, call in ((plan.ids, lambda *a: lib.clg_fc_tree_fold(*a, roots, 0, None)), (plan.slot, lambda *a: lib.clg_fc_tree_fold_slots(*a, roots, None))):
        coef, probs = torch.full((roots, 28), 7.0, device=DEV), torch.full((7 * roots, 16), 7.0, device=DEV)
        torch.cuda.synchronize()
        assert call(*(w.data_ptr() for w in logits), table.data_ptr(), coef.data_ptr(), probs.data_ptr()) == 0
        torch.cuda.synchronize()
        got.append((coef, probs))
    monkeypatch.undo()
    _lib.reload_knobs()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
