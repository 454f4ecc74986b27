"""When the trees of three LogicLayers (difflogic/fc_tree.py) are derived again: after every way in which a wiring can change.
On the CPU, with a stand-in for the tables that notes the wiring it was made from."""
import copy
import pickle
import threading
import time

import pytest
import torch

import convlogic_amd as C
from convlogic_amd.difflogic import fc_tree


class Noted:
    device = torch.device("cpu")

    def __init__(self, *layers):
        self.build(*layers)

    def fits(self):
        return True

    def build(self, *layers):
        self.wiring = [t.clone() for m in layers for t in (m.indices_0, m.indices_1)]
        self.start, self.flat = layers[0].given_x_indices_of_y_start.clone(), layers[0].given_x_indices_of_y.clone()

    def of(self, layers):
        return all(torch.equal(t, w) for t, w in zip((t for m in layers for t in (m.indices_0, m.indices_1)), self.wiring))


@pytest.fixture
def layers(monkeypatch):
    monkeypatch.setattr(fc_tree, "TreePlan", Noted)
    return chain(0)


def chain(seed):
    torch.manual_seed(seed)
    return [C.LogicLayer(a, b, implementation="cuda") for a, b in ((24, 40), (40, 20), (20, 10))]


def swapped(layer):
    """another wiring of the layer in which every input is read as often as before"""
    return layer.indices_0.flip(0)


def test_the_plan_is_kept(layers):
    plan = fc_tree.tree_plan(*layers)
    assert plan.of(layers) and fc_tree.tree_plan(*layers) is plan
    for m in layers:                                                   # no move: the same buffers
        m.to("cpu").float().train()
    assert fc_tree.tree_plan(*layers) is plan


@pytest.mark.parametrize("at", [0, 1, 2])
def test_invalidate_after_a_write_through_data(layers, at):
    fc_tree.tree_plan(*layers)
    layers[at].indices_0.data.copy_(swapped(layers[at]))
    layers[at].invalidate()
    assert fc_tree.tree_plan(*layers).of(layers)


@pytest.mark.parametrize("at", [0, 1, 2])
def test_writes_in_place_and_other_buffers(layers, at):
    fc_tree.tree_plan(*layers)
    layers[at].indices_0.copy_(swapped(layers[at]))
    assert fc_tree.tree_plan(*layers).of(layers)
    layers[at].indices_0 = swapped(layers[at])
    assert fc_tree.tree_plan(*layers).of(layers)
    for _ in range(20):                                                # (the allocator hands the last buffer's address out again)
        new = swapped(layers[at])
        layers[at].indices_0 = torch.empty(0, dtype=torch.int64)
        del layers[at].indices_0
        layers[at].register_buffer("indices_0", new)
        assert fc_tree.tree_plan(*layers).of(layers)


@pytest.mark.parametrize("at", [0, 1, 2])
def test_a_key_that_is_the_same_after_a_move(layers, at, monkeypatch):
    # buffers that went to another device and came back have version 0 again and may have the old addresses
    fc_tree.tree_plan(*layers)
    old = [layers[at].indices_0, layers[at].indices_1]
    key = layers[at]._wiring_key()
    layers[at]._apply(lambda t: t.clone())
    for name, t in zip(("indices_0", "indices_1"), old):
        t.data.copy_(swapped(layers[at]) if name == "indices_0" else t)
        layers[at]._buffers[name] = t                                  # the old address, the old version, another wiring
    assert layers[at]._wiring_key()[:5] == key[:5]
    assert fc_tree.tree_plan(*layers).of(layers)


def test_other_layers_behind_the_first(layers):
    fc_tree.tree_plan(*layers)
    other = chain(1)
    key = layers[1]._wiring_key()
    other[1]._wiring_key = lambda: key                                 # as if the new layer's buffers had the old addresses
    other[1]._wiring_checked = key
    assert fc_tree.tree_plan(layers[0], other[1], layers[2]).of([layers[0], other[1], layers[2]])
    assert fc_tree.tree_plan(*layers).of(layers)
    assert fc_tree.tree_plan(layers[0], layers[1], other[2]).of([layers[0], layers[1], other[2]])


def test_a_loaded_wiring_and_copies(layers):
    plan = fc_tree.tree_plan(*layers)
    for copies in (copy.deepcopy(layers), pickle.loads(pickle.dumps(layers))):
        for m in copies:
            assert "_wiring_checked" not in m.__dict__
        assert fc_tree.tree_plan(*copies) is not plan and fc_tree.tree_plan(*copies).of(copies)
    for m, o in zip(layers, chain(1)):
        m.load_state_dict(o.state_dict())
        assert plan.of(layers)                                          # at once: a recorded step reads these tables
    assert fc_tree.tree_plan(*layers) is plan


@pytest.mark.parametrize("at", [0, 1, 2])
def test_a_loaded_wiring_that_is_refused_is_not_read(layers, at):
    # load_state_dict(assign=True) takes buffers of any type and stride: the tables are made from what a call accepts alone
    plan = fc_tree.tree_plan(*layers)
    before = copy.deepcopy(layers)
    for name in ("indices_0", "indices_1", "given_x_indices_of_y_start", "given_x_indices_of_y"):
        good = {k: v.clone() for k, v in layers[at].state_dict().items()}
        for bad in (good[name].int(), good[name].repeat_interleave(2)[::2], torch.full_like(good[name], 1 << 40)):
            if bad.dtype == torch.int64 and bad.is_contiguous() and name.startswith("given"):
                continue                                               # (these lists are made again from the wiring)
            layers[at].load_state_dict({**good, name: bad}, assign=True)
            assert plan.of(before)
            with pytest.raises(ValueError, match=name if name.startswith("given") else "indices"):
                fc_tree.tree_plan(*layers)
        layers[at].load_state_dict(good, assign=True)
        assert fc_tree.tree_plan(*layers) is plan and plan.of(before)


def test_the_reverse_lists_of_a_loaded_wiring(layers):
    # a state without the reverse lists: the tables are made with the lists of the loaded wiring
    plan = fc_tree.tree_plan(*layers)
    state = {k: v for k, v in chain(1)[0].state_dict().items() if not k.startswith("given")}
    layers[0].load_state_dict(state, strict=False)
    assert plan.of(layers) and torch.equal(plan.start, chain(1)[0].given_x_indices_of_y_start) and torch.equal(plan.flat, chain(1)[0].given_x_indices_of_y)


def test_the_tables_of_a_recorded_step_stay(layers):
    plan = fc_tree.tree_plan(*layers)
    other = chain(1)
    assert fc_tree.tree_plan(layers[0], other[1], layers[2]) is not plan    # a second network over the same first layer
    for m in layers:
        m.load_state_dict(m.state_dict())
    layers[1].indices_0.copy_(swapped(layers[1]))
    layers[2].invalidate()
    assert fc_tree.tree_plan(*layers) is plan and plan.of(layers)
    plan.fits = lambda: False                                          # a wiring that makes no trees: not used, not freed
    layers[0].invalidate()
    assert fc_tree.tree_plan(*layers) is None
    plan.fits = lambda: True
    layers[0].invalidate()
    assert fc_tree.tree_plan(*layers) is plan


def test_two_threads_check_a_wiring_once(layers):
    # a wiring that counts as new a second time would make the tables again under the kernels of the first thread
    layer, entered = layers[0], []
    check = layer._check_new_wiring

    def slowly():
        entered.append(1)
        time.sleep(0.2)
        return check()

    layer._check_new_wiring = slowly
    keys = []
    threads = [threading.Thread(target=lambda: keys.append(layer._check_wiring())) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(entered) == 1 and len(set(keys)) == 1 and layer._wiring_epoch == 1


def test_the_walk_plan_of_a_recorded_packed_layer_stays():
    from convlogic_amd.hip import difflogic_hip
    layer, other = chain(0)[0], chain(1)[0]
    address = layer._eval_plan().data_ptr()
    for change in (lambda: layer.load_state_dict(layer.state_dict()), lambda: layer.load_state_dict(other.state_dict()),
                   lambda: layer.indices_0.copy_(swapped(layer)), layer.invalidate):
        change()
        keep = [torch.full((40,), -1, dtype=torch.int32) for _ in range(64)]   # (takes freed memory)
        assert layer._eval_plan().data_ptr() == address
        assert torch.equal(layer._eval_plan(), difflogic_hip.eval_plan(layer.indices_0, layer.indices_1, layer.in_dim))
        del keep
