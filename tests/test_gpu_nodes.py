"""The C++ autograd nodes of the float32 training path against the Python functions that serve every other case (double precision,
traces): the same outputs and gradients bit for bit, for every set of wanted gradients and every layout that reaches them."""
import itertools

import pytest
import torch

import convlogic_amd as C
from convlogic_amd.hip import _lib
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


def both_routes(monkeypatch, make):
    """make() -> (output, gradients) of fresh state, by the nodes and by the Python functions"""
    results = []
    for by_python in (False, True):
        monkeypatch.setattr(_lib, "traced", lambda: by_python)
        torch.manual_seed(7)
        results.append(make())
    monkeypatch.undo()
    (out, grads), (ref, ref_grads) = results
    assert torch.equal(out, ref) and out.stride() == ref.stride() and out.requires_grad == ref.requires_grad
    for a, b in zip(grads, ref_grads, strict=True):
        assert (a is None) == (b is None) and (a is None or (torch.equal(a, b) and a.stride() == b.stride()))


def gradients(y, gy, tensors):
    wanted = [t for t in tensors if t.requires_grad]
    got = iter(torch.autograd.grad(y, wanted, gy)) if wanted else iter(())
    return [next(got) if t.requires_grad else None for t in tensors]


@pytest.mark.parametrize("batch", [1, 33, 256, 1030])                # (up to 1024 samples the two gradients come from one kernel)
@pytest.mark.parametrize("in_dim,out_dim", [(40, 60), (64, 32), (30, 15)])
@pytest.mark.parametrize("layout", ["samples", "features", "strided"])
def test_logic_layer(monkeypatch, batch, in_dim, out_dim, layout):
    for need_x, need_w, gy_kind in itertools.product((True, False), (True, False), ("dense", "transposed", "expanded")):
        def make():
            layer = C.LogicLayer(in_dim, out_dim, implementation="cuda").to(DEV)
            layer.weights.requires_grad_(need_w)
            x = torch.rand(batch, in_dim, device=DEV)
            x = {"samples": x, "features": x.t().contiguous().t(), "strided": torch.stack([x, x], 2)[:, :, 0]}[layout].requires_grad_(need_x)
            y = layer(x)
            gy = torch.randn(batch, out_dim, device=DEV)
            gy = {"dense": gy, "transposed": gy.t().contiguous().t(), "expanded": gy[:1].expand(batch, -1)}[gy_kind]
            return y, gradients(y, gy, [x, layer.weights])
        both_routes(monkeypatch, make)


@pytest.mark.parametrize("shape,c_out,kw", [((5, 3, 12, 12), 8, {}), ((33, 16, 4, 4), 40, {}), ((40, 64, 8, 8), 300, {}), ((3, 2, 15, 11), 6, dict(padding=0, kernel=2)),
                                            ((4, 3, 15, 16), 8, dict(stride=2)), ((6, 4, 28, 28), 8, dict(kernel=5, padding=0)), ((70, 200, 16, 16), 30, {})])
@pytest.mark.parametrize("kind", ["block", "feature_major", "binary"])
def test_blocks(monkeypatch, shape, c_out, kw, kind):
    for need_x, need_w, gy_kind in itertools.product((True, False), (True, False), ("dense", "feature_major", "channels_last")):
        def make():
            layer = C.ConvLogicLayer(shape[1], c_out, complete=True, implementation="cuda", **kw).to(DEV)
            layer.weights.requires_grad_(need_w)
            layer.feature_major_output, layer.binary_input = kind == "feature_major", kind == "binary"
            x = (torch.rand(shape, device=DEV) < 0.5).float() if kind == "binary" else torch.rand(shape, device=DEV)
            x.requires_grad_(need_x)
            y = layer(x)
            gy = torch.randn(y.shape, device=DEV)
            gy = {"dense": gy, "feature_major": gy.permute(1, 2, 3, 0).contiguous().permute(3, 0, 1, 2),
                  "channels_last": gy.contiguous(memory_format=torch.channels_last)}[gy_kind]
            return y, gradients(y, gy, [x, layer.weights])
        both_routes(monkeypatch, make)


@pytest.mark.parametrize("mode", [True, "always"])
@pytest.mark.parametrize("topology,batch", [("cifar", 3), ("cifar", 65), ("mnist", 100)])
def test_networks(monkeypatch, topology, batch, mode):
    def make():
        model = (C.ConvLogicCifarModel(k_param=8, input_channels=3) if topology == "cifar" else C.ConvLogicMnistModel(k_param=8)).to(DEV)
        model.prefold = mode
        x = (torch.rand(batch, 3 if topology == "cifar" else 1, *(2 * [32 if topology == "cifar" else 28]), device=DEV) < 0.5).float()
        y = model(x)
        return y, gradients(y, torch.randn_like(y), list(model.parameters()))
    both_routes(monkeypatch, make)


def test_what_autograd_offers_around_a_node():
    torch.manual_seed(3)
    layer = C.ConvLogicLayer(3, 8, complete=True, implementation="cuda").to(DEV)
    x = torch.rand(4, 3, 12, 12, device=DEV, requires_grad=True)
    want = torch.autograd.grad(layer(x).sum(), [x, layer.weights])
    moved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: moved.append(1) or t.cpu(), lambda t: t.to(DEV)):
        got = torch.autograd.grad(layer(x).sum(), [x, layer.weights])
    assert moved and all(torch.equal(a, b) for a, b in zip(got, want))
    again = torch.utils.checkpoint.checkpoint(layer, x, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(again.sum(), [x, layer.weights]), want))
    y = layer(x)
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
    with pytest.raises(RuntimeError):
        torch.func.vmap(layer)(torch.rand(2, 4, 3, 12, 12, device=DEV))
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
        layer(torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x)))
    with torch.no_grad():
        assert not layer(x).requires_grad
    y = layer(x)
    layer.weights.data.mul_(2)                                        # an optimizer's update between the passes
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y.sum(), [x, layer.weights]), want))


def test_a_trace_keeps_its_inputs():
    torch.manual_seed(4)
    layer = C.LogicLayer(40, 60, implementation="cuda").to(DEV)
    traced = torch.jit.trace(layer, (torch.rand(8, 40, device=DEV),), check_trace=False)
    x = torch.rand(8, 40, device=DEV)
    assert torch.equal(traced(x), layer(x))


def test_replaced_weights_of_another_shape_are_refused():
    layer = C.ConvLogicLayer(3, 8, complete=True, implementation="cuda").to(DEV)
    layer.weights = torch.nn.Parameter(torch.randn(4, 7, 16, device=DEV))
    with pytest.raises(RuntimeError, match="weights must have shape"):
        layer(torch.rand(2, 3, 8, 8, device=DEV))
