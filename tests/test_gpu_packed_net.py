"""A whole network on packed words in one call of the library against its modules called one after the other: class counts and the
words in front of the trees bit for bit, float evaluation of 0/1 images through the same kernels, and what is left to the modules."""
import copy

import pytest
import torch

import convlogic_amd as C
from convlogic_amd.convlogic import binarize, packed_net
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


def network(topology, k, channels):
    torch.manual_seed(k)
    model = (C.ConvLogicCifarModel(k_param=k, input_channels=channels, tau=6.5) if topology == "cifar"
             else C.ConvLogicMnistModel(k_param=k, input_channels=channels)).to(DEV).eval()
    with torch.no_grad():
        for p in model.parameters():
            p.add_(torch.randn_like(p), alpha=2.0)
    return model, 32 if topology == "cifar" else 28


def by_modules(model, x):
    with torch.no_grad():
        return model.network(x)


@pytest.fixture
def at_once(monkeypatch):
    calls = []
    evaluate = packed_net.evaluate
    monkeypatch.setattr(packed_net, "evaluate", lambda *a: calls.append(1) or evaluate(*a))
    return calls


# samples at the ends of words and of the 32 groups from which the last CIFAR block writes feature-major; classes in one slice and in several
@pytest.mark.parametrize("topology,k,channels,samples", [("cifar", 8, 3, 1), ("cifar", 8, 9, 64), ("cifar", 32, 9, 65), ("cifar", 16, 3, 1983),
                                                         ("cifar", 16, 3, 1985), ("cifar", 8, 1, 8200), ("mnist", 8, 1, 63), ("mnist", 24, 1, 1000),
                                                         ("mnist", 9, 2, 4097), ("cifar", 100, 6, 130), ("mnist", 300, 1, 70),
                                                         ("cifar", 64, 3, 1900), ("mnist", 300, 1, 500)])
def test_counts_and_sums_are_those_of_the_modules(at_once, topology, k, channels, samples):
    model, side = network(topology, k, channels)
    x = (torch.rand(samples, channels, side, side, device=DEV) < 0.5).float()
    packed, again = C.PackBitsTensor(x.bool(), 64), C.PackBitsTensor(x.bool(), 64)
    with torch.no_grad():
        got = model(packed)
    want = by_modules(model, again)
    head = by_modules(torch.nn.ModuleDict({"network": model.network[:-4]}), C.PackBitsTensor(x.bool(), 64))
    assert at_once and got.dtype == torch.int32 and torch.equal(got, want)
    assert not packed.image and torch.equal(packed.t, head.t) and packed.pad_len == again.pad_len
    at_once.clear()
    with torch.no_grad():
        sums = model(x)
    assert at_once
    # counts are whole numbers in either; the modules' division by tau may round once more
    assert sums.dtype == torch.float32 and torch.equal((sums * model.network[-1].tau).round().int(), want)
    assert torch.allclose(sums, by_modules(model, x), rtol=2e-7, atol=0)


def test_what_the_modules_do_for_themselves_stays_theirs(at_once):
    model, side = network("mnist", 8, 1)
    x = (torch.rand(200, 1, side, side, device=DEV) < 0.5).float()
    with torch.no_grad():
        want = model(x)
        assert at_once
        seen = []
        for module in (model.network[0], model.network[2], model.network[3]):
            at_once.clear()
            handle = module.register_forward_hook(lambda m, i, o: seen.append(type(o)))
            assert torch.equal(model(x), want) and seen and not at_once
            handle.remove()
        # the first block without its promise, weights of another type, a block in training (whose gates are mixed): sums by the modules
        for change, same in ((lambda m: setattr(m.network[0], "binary_input", False), True), (lambda m: m.network[1].double(), True),
                             (lambda m: m.network[1].train(), False)):
            other = copy.deepcopy(model)
            change(other)
            at_once.clear()
            got = other(x)
            # (the last layers may still run as trees, which divide by tau as a product: one more rounding)
            assert not at_once and torch.allclose(got, by_modules(other, x), rtol=1e-6, atol=0) and torch.equal(got, want) == same
        other = copy.deepcopy(model)
        other.network[2].return_indices = True
        with pytest.raises(AttributeError, match="'tuple' object has no attribute 'flatten'"):
            other(x)
        assert not at_once
        real = copy.deepcopy(model)
        real.network[0].binary_input = False
        half = x * 0.5
        assert torch.equal(real(half), real.network(half))
        with pytest.raises(RuntimeError, match="Expected x of shape"):
            model(x.expand(-1, 2, -1, -1))
        with pytest.raises(Exception):
            model(x[:, :, :27])


def test_a_value_that_is_not_binary_is_reported():
    model, side = network("mnist", 8, 1)
    x = (torch.rand(200, 1, side, side, device=DEV) < 0.5).float()
    for bad in (0.5, float("nan"), -1.0, 2.0):
        broken = x.clone()
        broken[199, 0, side - 1, side - 1] = bad
        with torch.no_grad():
            model(broken)
            with pytest.raises(RuntimeError, match="other than 0 and 1"):
                model.network[0].check_binary_input()
            assert torch.allclose(model(x), by_modules(model, x), rtol=2e-7, atol=0)


def test_forward_mode_is_refused_as_before():
    model, side = network("mnist", 8, 1)
    x = (torch.rand(200, 1, side, side, device=DEV) < 0.5).float()
    with torch.autograd.forward_ad.dual_level(), pytest.raises(Exception):
        model(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))


@pytest.mark.parametrize("n", [100, 300])
def test_recorded_evaluation_follows_weights_and_images(n):
    model, side = network("cifar", 32, 3)
    x = (torch.rand(n, 3, side, side, device=DEV) < 0.5).float()
    images = torch.rand(n, 3, side, side, device=DEV)
    thr = torch.tensor([0.5], device=DEV)
    with torch.no_grad():
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            model(x), model(binarize.pack_thresholds(images, thr))
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            sums, counts = model(x), model(binarize.pack_thresholds(images, thr))
        for _ in range(3):
            x.copy_((torch.rand_like(x) < 0.5).float())
            images.copy_(torch.rand_like(images))
            for p in model.parameters():
                p.copy_(torch.randn_like(p))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.allclose(sums, by_modules(model, x), rtol=2e-7, atol=0)
            assert torch.equal(counts, by_modules(model, binarize.pack_thresholds(images, thr)))


def test_bad_arguments_are_refused():
    from convlogic_amd.hip import _lib
    lib = _lib.load()
    table = (_lib.PackedBlock * 2)()
    for entry, (c_in, side, c_out) in zip(table, ((3, 16, 8), (9, 8, 16))):
        entry.geom = _lib.ConvGeom(2, c_in, side, side, c_out, 1, 1, 1, 1, 3, 3)
    assert lib.clg_net_packed_scratch_bytes(table, 2, 256, 20, 10, 100) == -1      # the second block takes 9 channels of 8
    table[1].geom.c_in = 8
    assert lib.clg_net_packed_scratch_bytes(table, 2, 255, 20, 10, 100) == -1
    assert lib.clg_net_packed_scratch_bytes(table, 2, 256, 20, 10, 100) > 0
    assert lib.clg_net_packed_scratch_bytes(table, 0, 256, 20, 10, 100) == -1
