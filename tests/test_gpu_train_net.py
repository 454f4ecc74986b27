"""A network's training step as one autograd node (convlogic/train_net.py) against its modules one after the other: outputs and gradients bit
for bit, for every set of wanted gradients; and what is left to the modules."""
import copy

import pytest
import torch

import convlogic_amd as C
from convlogic_amd.convlogic import train_net
from convlogic_amd.hip import _lib
from tests.gpu_util import DEV, set_knobs

pytestmark = pytest.mark.gpu


def network(topology, k, channels):
    torch.manual_seed(k)
    model = C.ConvLogicCifarModel(k_param=k, input_channels=channels) if topology == "cifar" else C.ConvLogicMnistModel(k_param=k, input_channels=channels)
    return model.to(DEV), 32 if topology == "cifar" else 28


@pytest.fixture
def at_once(monkeypatch):
    calls, train = [], train_net.train

    def spy(*a):
        out = train(*a)
        calls.append(out is not None)
        return out
    monkeypatch.setattr(train_net, "train", spy)
    return calls


def step(model, x, gy, tensors, by_modules):
    model.prefold = not by_modules                                    # (any other value than True calls the modules)
    y = model(x)
    wanted = [t for t in tensors if t.requires_grad]
    got = iter(torch.autograd.grad(y, wanted, gy))
    return y, [next(got) if t.requires_grad else None for t in tensors]


# batches below and from the 32 samples on from which the last CIFAR block writes feature-major; channels too many for the binary first block's
# lists to be short, the first block without its promise
@pytest.mark.parametrize("topology,k,channels,batch,binary", [("cifar", 8, 3, 5, True), ("cifar", 8, 9, 64, True), ("cifar", 16, 3, 33, False),
                                                              ("mnist", 8, 1, 70, True), ("mnist", 9, 2, 1, True), ("mnist", 10, 1, 31, False)])
def test_the_same_as_the_modules(at_once, topology, k, channels, batch, binary):
    model, side = network(topology, k, channels)
    model.network[0].binary_input = binary
    x = (torch.rand(batch, channels, side, side, device=DEV) < 0.5).float()
    params = list(model.parameters())
    gy = torch.randn(batch, 10, device=DEV)
    n = len(params)
    frozen_sets = [set(), set(range(n)), *({i} for i in range(n)), set(range(n - 3)), set(range(n - 3, n)), {0, 1}, {n - 2, n - 1}]
    for need_x in (False, True):
        for frozen in frozen_sets:
            if not need_x and len(frozen) == n:
                continue
            x.requires_grad_(need_x)
            for i, p in enumerate(params):
                p.requires_grad_(i not in frozen)
            at_once.clear()
            y, grads = step(model, x, gy, [x, *params], False)
            assert at_once == [True]
            y0, grads0 = step(model, x, gy, [x, *params], True)
            assert at_once == [True] and torch.equal(y, y0)
            for a, b in zip(grads, grads0, strict=True):
                assert (a is None) == (b is None) and (a is None or (torch.equal(a, b) and a.stride() == b.stride()))


def test_what_autograd_offers_around_the_node(at_once):
    model, side = network("mnist", 8, 1)
    x = (torch.rand(40, 1, side, side, device=DEV) < 0.5).float()
    params = list(model.parameters())
    want = torch.autograd.grad(model(x).sum(), params)
    moved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: moved.append(1) or t.cpu(), lambda t: t.to(DEV)):
        got = torch.autograd.grad(model(x).sum(), params)
    assert moved and all(torch.equal(a, b) for a, b in zip(got, want))
    again = torch.utils.checkpoint.checkpoint(model, x, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(again.sum(), params), want))
    y = model(x)
    assert all(torch.equal(a, b) for _ in range(2) for a, b in zip(torch.autograd.grad(y.sum(), params, retain_graph=True), want))
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
    y = model(x)
    with torch.no_grad():
        for p in params:
            p.data.mul_(2)                                            # an optimizer's update between the passes
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y.sum(), params), want))
    y = model(x)
    model.network[1].selection.add_(0)                                # the wiring written in between
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    with pytest.raises(RuntimeError):
        torch.func.vmap(model)(torch.zeros(2, 4, 1, side, side, device=DEV))
    assert all(at_once[:-1])


def test_what_the_modules_do_for_themselves_stays_theirs(at_once):
    model, side = network("mnist", 8, 1)
    x = (torch.rand(20, 1, side, side, device=DEV) < 0.5).float()
    want = model(x).detach()
    assert at_once == [True]
    seen = []
    for module in (model.network[0], model.network[2], model.network[3]):
        for register in (module.register_forward_hook, module.register_full_backward_hook):
            at_once.clear()
            handle = register(lambda *a: seen.append(1))
            y = model(x)
            y.sum().backward()
            assert torch.equal(y, want) and seen and True not in at_once
            handle.remove()
            seen.clear()

    def change(f):
        other = copy.deepcopy(model)
        f(other)
        at_once.clear()
        y = other(x)
        assert True not in at_once and torch.equal(y, want)
    change(lambda m: setattr(m, "prefold", "always"))
    change(lambda m: setattr(m.network[1], "grad_factor", 2.0))
    change(lambda m: setattr(m.network[1], "forward", m.network[1].forward))
    at_once.clear()
    assert torch.equal(model(x.expand(20, 1, side, side).flip(0).flip(0).transpose(2, 3).contiguous().transpose(2, 3)), want) and True not in at_once
    with pytest.raises(RuntimeError):
        model(x[:, :, 1:])
    large, side = network("mnist", 128, 1)                            # more logits than small networks have
    at_once.clear()
    large((torch.rand(2, 1, side, side, device=DEV) < 0.5).float())
    assert True not in at_once


def test_a_batch_that_the_trees_do_not_take_is_the_modules(at_once, monkeypatch):
    model, side = network("mnist", 8, 1)
    x = (torch.rand(20, 1, side, side, device=DEV) < 0.5).float()
    want = model(x)
    monkeypatch.setattr(train_net.fc_tree, "MAX_BATCH", 19)
    got = model(x)
    # (the modules' class sums add the rows of a class in another order)
    assert at_once == [True, False] and (got - want).abs().max() <= 1e-5 * want.abs().max()
    monkeypatch.setattr(train_net.fc_tree, "MAX_BATCH", 20)
    assert torch.equal(model(x), want) and at_once[-1]


def test_a_broken_promise_of_binary_inputs_is_reported():
    model, side = network("mnist", 8, 1)
    model(torch.rand(4, 1, side, side, device=DEV))
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="0 and 1"):
        model(torch.zeros(4, 1, side, side, device=DEV))


# one launch sets up to 16 blocks up and ends their weight gradients, another one more is set up layer by layer
@pytest.mark.parametrize("blocks,kernels", [(1, 3), (16, 5), (17, 5)])
def test_any_number_of_blocks(at_once, blocks, kernels):
    torch.manual_seed(blocks)
    model = C.ConvLogicMnistModel(k_param=8)
    channels = [2] + [kernels] * blocks
    model.network = torch.nn.Sequential(*(C.ConvLogicLayer(a, b, kernel=3, padding=2, complete=True, implementation="cuda") for a, b in zip(channels, channels[1:])),
                                        torch.nn.Flatten(), *(C.LogicLayer(a, b, implementation="cuda") for a, b in ((4 * kernels, 80), (80, 40), (40, 20))),
                                        C.GroupSum(10))
    model = model.to(DEV)
    x = torch.rand(37, 2, 2, 2, device=DEV).requires_grad_(True)     # (2 x 2 images stay 2 x 2)
    tensors, gy = [x, *model.parameters()], torch.randn(37, 10, device=DEV)
    y, grads = step(model, x, gy, tensors, False)
    y0, grads0 = step(model, x, gy, tensors, True)
    assert at_once == [True] and torch.equal(y, y0) and all(torch.equal(a, b) for a, b in zip(grads, grads0, strict=True))


# operand and tap gradients and the trees' logits past the caches or through them, rows of one to four samples per lane and ragged ones
@pytest.mark.parametrize("k,batch", [(8, 33), (8, 64), (8, 127), (4, 256), (4, 301)])
@pytest.mark.parametrize("by_modules", [False, True])
def test_gradients_past_the_caches(monkeypatch, k, batch, by_modules):
    model, side = network("cifar", k, 3)
    x, gy = (torch.rand(batch, 3, side, side, device=DEV) < 0.5).float(), torch.randn(batch, 10, device=DEV)
    got = []
    for megabytes in ("0", "100000"):
        set_knobs(monkeypatch, CLG_STREAM_MB=megabytes)
        got.append(step(model, x, gy, list(model.parameters()), by_modules)[1])
    monkeypatch.undo()
    _lib.reload_knobs()
    assert all(torch.equal(a, b) for a, b in zip(*got, strict=True))


# batches at which scratch is most of a step's memory: by one node no more of it than by the modules, whose scratch is one layer's at a time
@pytest.mark.parametrize("topology,k,channels,batch", [("cifar", 32, 9, 256), ("cifar", 16, 3, 512), ("mnist", 32, 1, 1000)])
def test_memory_of_a_step(at_once, topology, k, channels, batch):
    model, side = network(topology, k, channels)
    x = (torch.rand(batch, channels, side, side, device=DEV) < 0.5).float()
    peak = []
    for by_modules in (False, True):
        model.prefold = not by_modules
        for counted in (False, True):                                 # (plans are made in the first step)
            model.zero_grad()
            torch.cuda.empty_cache()
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            model(x).sum().backward()
        peak.append(torch.cuda.max_memory_allocated() - before)
    # what the node keeps longer than the modules: the saved activations of the layers behind (their gradients' scratch is larger), parts of the sums
    assert True in at_once and peak[0] <= 1.1 * peak[1], peak
