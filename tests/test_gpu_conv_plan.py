"""Per-layer plan of the fused block's backward pass (clg_convblock_plan / clg_convblock_backward_planned): the tables
that depend only on the selection are built once; a planned call gives the gradients of the unplanned entry points on
every kernel family (images in LDS, padded global copy, 4x4 one-sample-per-lane, any-shape gather), twice in a row,
with and without the coefficients folded by the forward launch."""
import copy
import ctypes
import pickle

import pytest
import torch

import convlogic_amd as C
from convlogic_amd.difflogic import fc_tree
from convlogic_amd.hip import _lib, convlogic_hip
from tests.gpu_util import DEV, assert_grad_close, block_oracle, set_knobs

pytestmark = pytest.mark.gpu

# (n, cin, cout, h, w, stride): LDS-tiled (few and many kernels), padded-copy kernels, 4x4 images, any-shape gather
SHAPES = [(24, 1, 32, 28, 28, 1), (6, 9, 40, 32, 32, 1), (40, 128, 64, 8, 8, 1), (70, 24, 48, 4, 4, 1), (5, 3, 6, 11, 15, 2),
          (3, 64, 32, 32, 32, 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", SHAPES)
def test_planned_backward_matches_unplanned(shape, dtype):
    n, cin, cout, h, w, stride = shape
    torch.manual_seed(n + cin)
    layer = C.ConvLogicLayer(cin, cout, stride=stride, padding=1, complete=True, implementation="cuda").to(DEV).to(dtype)
    x = torch.rand(n, cin, h, w, device=DEV, dtype=dtype)
    geo = (stride, stride, 1, 1)
    y, am, probs, folded = convlogic_hip.full_convlogic_forward_logits(x, layer.weights.detach(), layer.selection, *geo, 3, 3, want_folded=True)
    y0, am0, probs0 = convlogic_hip.full_convlogic_forward_logits(x, layer.weights.detach(), layer.selection, *geo, 3, 3)
    assert torch.equal(y, y0) and torch.equal(am, am0) and torch.equal(probs, probs0)
    # the folded coefficients are those of the probabilities: c_1 = sum of gates 8..15, c_a = p2+p3+p6+p7-p8-p9-p12-p13, ...
    p = probs.double()
    want_one = p[..., 8:].sum(-1)
    want_a = p[..., [2, 3, 6, 7]].sum(-1) - p[..., [8, 9, 12, 13]].sum(-1)
    assert (folded[..., 3].double() - want_one).abs().max().item() <= 1e-6
    assert (folded[..., 1].double() - want_a).abs().max().item() <= 1e-6
    gy = torch.randn_like(y)
    gx_ref, gl_ref = convlogic_hip.full_convlogic_backward_logits(gy, x, probs, am, layer.selection, *geo)
    _, gw_ref = convlogic_hip.full_convlogic_backward(gy, x, probs, am, layer.selection, *geo)
    plan, sig = convlogic_hip.make_backward_plan(x, cout, layer.selection, *geo, 3, 3)
    tol = 2e-5 if dtype == torch.float32 else 1e-12
    for rep in range(2):                                             # a plan is only read: the second call gives the same
        for fold in (folded, None):
            gx, gl = convlogic_hip.full_convlogic_backward_planned(gy, x, probs, fold, am, layer.selection, plan, sig, *geo)
            assert torch.equal(gx, gx_ref)                           # same kernels on the same tables
            assert (gl - gl_ref).abs().max().item() <= tol * gl_ref.abs().max().item()
        gx, gw = convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, layer.selection, plan, sig, *geo, wrt_logits=False)
        assert torch.equal(gx, gx_ref) and (gw - gw_ref).abs().max().item() <= tol * gw_ref.abs().max().item()
        none, gl = convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, layer.selection, plan, sig, *geo, need_grad_x=False)
        assert none is None and (gl - gl_ref).abs().max().item() <= tol * gl_ref.abs().max().item()
    if convlogic_hip.feature_major_supported(x, cout, *geo, 3, 3):     # the gradient of a feature-major output
        gy_fm = gy.permute(1, 2, 3, 0).contiguous()
        gx_fm, gl_fm = convlogic_hip.full_convlogic_backward_fm(gy_fm, x, probs, am, layer.selection, *geo)
        gx, gl = convlogic_hip.full_convlogic_backward_planned(gy_fm, x, probs, folded, am, layer.selection, plan, sig, *geo, feature_major=True)
        assert torch.equal(gx, gx_fm) and torch.equal(gl, gl_fm)
    else:
        with pytest.raises(RuntimeError, match="clg_convblock_fm_supported"):
            convlogic_hip.full_convlogic_backward_planned(gy.permute(1, 2, 3, 0).contiguous(), x, probs, folded, am, layer.selection, plan, sig,
                                                          *geo, feature_major=True, validate=False)


def test_plan_is_rejected_for_another_geometry_and_after_knob_changes(monkeypatch):
    layer = C.ConvLogicLayer(3, 8, padding=1, complete=True, implementation="cuda").to(DEV)
    x = torch.rand(4, 3, 16, 16, device=DEV)
    geo = (1, 1, 1, 1)
    y, am, probs, folded = convlogic_hip.full_convlogic_forward_logits(x, layer.weights.detach(), layer.selection, *geo, 3, 3, want_folded=True)
    plan, sig = convlogic_hip.make_backward_plan(x, 8, layer.selection, *geo, 3, 3)
    gy = torch.randn_like(y)
    convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, layer.selection, plan, sig, *geo)
    with pytest.raises(RuntimeError, match="plan was made for another"):
        convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, layer.selection, plan, sig + 1, *geo)
    x2 = torch.rand(6, 3, 16, 16, device=DEV)                        # another batch size: another plan
    y2, am2, probs2, folded2 = convlogic_hip.full_convlogic_forward_logits(x2, layer.weights.detach(), layer.selection, *geo, 3, 3,
                                                                        want_folded=True)
    big = torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    big[:plan.numel()] = plan
    with pytest.raises(RuntimeError, match="plan was made for another"):
        convlogic_hip.full_convlogic_backward_planned(torch.randn_like(y2), x2, probs2, folded2, am2, layer.selection, big, sig, *geo)
    set_knobs(monkeypatch, CLG_BWDX_DIRECT="1")                      # another kernel family: the old plan no longer fits
    with pytest.raises(RuntimeError, match="plan was made for another"):
        convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, layer.selection, big, sig, *geo)
    # the module keys its plans on the knob generation, so it simply builds a new one
    layer.train()
    xin = x.clone().requires_grad_(True)
    layer(xin).sum().backward()
    assert torch.isfinite(xin.grad).all()


@pytest.mark.parametrize("shape", [(16, 1, 32, 28, 28), (8, 9, 64, 32, 32), (40, 128, 64, 8, 8)])
def test_module_training_path_uses_the_plan_and_matches_the_oracle(shape):
    n, cin, cout, h, w = shape
    torch.manual_seed(cin)
    layer = C.ConvLogicLayer(cin, cout, padding=1, complete=True, implementation="cuda", return_indices=False).to(DEV)
    x = torch.randint(0, 2, (n, cin, h, w), device=DEV).float().requires_grad_(True)
    grads = []
    for step in range(2):
        layer.weights.grad = x.grad = None
        y = layer(x)
        gy = torch.randn(y.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))
        y.backward(gy)
        grads.append((y.detach().clone(), x.grad.clone(), layer.weights.grad.clone()))
    assert len(layer._plans) == 1
    for a, b in zip(*grads):
        assert torch.equal(a, b)                                     # same plan, same result
    _, am, _ = convlogic_hip.full_convlogic_forward_logits(x.detach(), layer.weights.detach(), layer.selection, 1, 1, 1, 1, 3, 3)
    idx = convlogic_hip.argmax_to_indices(am, w)
    routed, _, _, _, _, ll, xl, _ = block_oracle(x, layer.weights, layer.selection, (1, 1), (1, 1), (3, 3), idx)
    routed.backward(gy.cpu())
    assert (grads[0][0].cpu() - routed.detach()).abs().max().item() <= 1e-5
    assert_grad_close(grads[0][1], xl.grad, name="grad_x")
    assert_grad_close(grads[0][2], ll.grad, name="grad_logits")
    # another batch size gets a plan of its own; an in-place edit of the selection drops the old ones on the next call
    layer(x[:3].detach()).sum().backward()
    assert len(layer._plans) == 2


def crowded(sel, half=True):
    """the selection with channel 0 in place of the first channel of every second kernel (or of every kernel)"""
    ch, first = sel >> 16, (sel >> 16)[:, :1]
    there = (ch == first) & ((torch.arange(sel.shape[0], device=sel.device) % 2 == 0).view(-1, 1) | (not half))
    return (torch.where(there, torch.zeros_like(ch), ch) << 16) | (sel & 0xFFFF)


@pytest.mark.parametrize("shape", [(64, 16, 256, 8), (64, 32, 256, 28)])
def test_a_channel_that_many_kernels_read_keeps_the_kernels_of_long_lists(shape, monkeypatch):
    n, cin, cout, side = shape
    torch.manual_seed(n)
    layer = C.ConvLogicLayer(cin, cout, padding=1, complete=True, implementation="cuda").to(DEV)
    x, geo = torch.rand(n, cin, side, side, device=DEV), (1, 1, 1, 1)
    for sel, is_long in ((layer.selection, False), (crowded(layer.selection), True)):
        y, am, probs, folded = convlogic_hip.full_convlogic_forward_logits(x, layer.weights.detach(), sel, *geo, 3, 3, want_folded=True)
        gy = torch.randn_like(y)
        plans = [convlogic_hip.make_backward_plan(x, cout, sel, *geo, 3, 3, lists=how) for how in (-1, 0, 1)]
        assert [convlogic_hip.lists_of(sig) for _, sig in plans] == [is_long, 0, 1]
        # the kernels of long lists are those that the knob takes at this shape, bit for bit
        set_knobs(monkeypatch, CLG_BWDX_DIRECT="0")
        want = convlogic_hip.full_convlogic_backward_logits(gy, x, probs, am, sel, *geo)
        set_knobs(monkeypatch, CLG_BWDX_DIRECT=None)
        for plan, sig in plans:
            got = convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, sel, plan, sig, *geo)
            if convlogic_hip.lists_of(sig):
                assert torch.equal(got[0], want[0])
            for a, b in zip(got, want):
                assert_grad_close(a, b, rel=1e-4)
        padded = torch.empty(_lib.load().clg_convblock_padded_elems(0, ctypes.byref(convlogic_hip._geom(x, cout, *geo, 3, 3)), 1), device=DEV)
        if padded.numel():
            with pytest.raises(RuntimeError, match="short lists"):
                convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, sel, *plans[2], *geo, padded=padded)
    # a plan that is in use keeps its kernels when it is made again for another selection
    layer(x.requires_grad_(True)).sum().backward()
    with torch.no_grad():
        layer.selection.copy_(crowded(layer.selection))
    x.grad = None
    layer(x).backward(gy)
    (kept,) = layer._plans.values()
    assert convlogic_hip.lists_of(kept.plan[1]) == 0
    again = copy.deepcopy(layer)
    gx, x.grad = x.grad, None
    again(x).backward(gy)
    (kept,) = again._plans.values()
    assert convlogic_hip.lists_of(kept.plan[1]) == 1
    assert_grad_close(gx, x.grad, rel=1e-4)


def wide(sel, cin, part):
    """the selection with the taps of every `part`-th kernel in any channels"""
    ch = torch.randint(0, cin, sel.shape, device=sel.device, dtype=torch.int32)
    return torch.where((torch.arange(sel.shape[0], device=sel.device) % part == 0).view(-1, 1), (ch << 16) | (sel & 0xFFFF), sel)


# both gradients by planes unless some kernel's taps are in more than two channels: then by the kernels without planes, bit for bit (one with a padded
# copy from the forward call, one whose channels with many kernels take the kernels of long lists)
@pytest.mark.parametrize("shape", [(16, 32, 256, 6), (256, 32, 128, 16), (32, 16, 128, 20)])
def test_taps_in_many_channels_take_the_kernels_without_planes(shape, monkeypatch):
    n, cin, cout, side = shape
    torch.manual_seed(n)
    layer, lib = C.ConvLogicLayer(cin, cout, padding=1, complete=True, implementation="cuda").to(DEV), _lib.load()
    x, geo = torch.rand(n, cin, side, side, device=DEV), (1, 1, 1, 1)
    def gradients(sel, lists):
        plan, sig = convlogic_hip.make_backward_plan(x, cout, sel, *geo, 3, 3, lists=lists)
        geom = ctypes.byref(convlogic_hip._geom(x, cout, *geo, 3, 3))
        y, am, probs, folded, padded = convlogic_hip.full_convlogic_forward_logits(x, layer.weights.detach(), sel, *geo, 3, 3, want_folded=True, want_padded=True,
                                                                                   signature=sig)
        torch.manual_seed(1)
        gy = torch.randn_like(y)
        got = convlogic_hip.full_convlogic_backward_planned(gy, x, probs, folded, am, sel, plan, sig, *geo, padded=padded)
        return sig, lib.clg_convblock_backward_planned_scratch_bytes(0, geom, sig), None if padded is None else padded.numel(), got
    for sel, is_wide in ((layer.selection, 0), (wide(layer.selection, cin, cout), 2), (wide(layer.selection, cin, 1), 2), (wide(crowded(layer.selection, False), cin, 2), 2)):
        sig, scratch, padded, got = gradients(sel, -1)
        assert convlogic_hip.lists_of(sig) & 2 == is_wide
        for lists in (sig & 3, 0, 1, 2, 3):                           # (any choice is a right one)
            again = gradients(sel, lists)
            assert lists != sig & 3 or (again[:3] == (sig, scratch, padded) and all(torch.equal(a, b) for a, b in zip(got, again[3])))
            for a, b in zip(got, again[3]):
                assert_grad_close(a, b, rel=1e-4)
        if is_wide:
            set_knobs(monkeypatch, CLG_BWDX_PLANES="0")
            _, scratch0, padded0, want = gradients(sel, -1)
            set_knobs(monkeypatch, CLG_BWDX_PLANES=None)
            assert (scratch, padded) == (scratch0, padded0) and all(torch.equal(a, b) for a, b in zip(got, want))
    # a plan in use whose layer is given such a selection, and one without
    x.requires_grad_(True)
    for sel in (layer.selection.clone(), wide(layer.selection, cin, 1), layer.selection.clone()):
        with torch.no_grad():
            layer.selection.copy_(sel)
        y = layer(x)
        torch.manual_seed(1)
        got = torch.autograd.grad(y, [x, layer.weights], torch.randn_like(y))
        (kept,) = layer._plans.values()
        x.requires_grad_(False)
        sig, _, _, want = gradients(sel, -1)
        x.requires_grad_(True)
        assert kept.plan[1] == sig and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("cout", [256, 4100])                          # (whose selections are, and are not, looked at on the host)
def test_a_plan_is_made_again_in_its_place(cout):
    layer = C.ConvLogicLayer(600 if cout > 4096 else 32, cout, padding=1, complete=True, implementation="cuda").to(DEV)
    x = torch.rand(2, layer.in_channels, 6, 6, device=DEV)
    before, sig = layer._backward_plan(x, layer.selection)
    layer.selection.add_(0)                                           # (as a broadcast of the buffers does)
    layer._check_selection()
    after, again = layer._backward_plan(x, layer.selection)
    assert after.data_ptr() == before.data_ptr() and again == sig and len(layer._plans) == 1
    with torch.no_grad():
        layer.selection[7, 3] = layer.in_channels << 16               # a channel outside
    with pytest.raises(ValueError, match="outside"):
        layer(x)


@pytest.mark.parametrize("shape", [(256, 8, 32, 16), (300, 16, 128, 12)])
def test_a_first_block_takes_no_gradient_planes(shape):
    n, cin, cout, side = shape
    layer, x = C.ConvLogicLayer(cin, cout, padding=1, complete=True, implementation="cuda").to(DEV), torch.rand(n, cin, side, side, device=DEV)
    geom, (_, sig) = ctypes.byref(convlogic_hip._geom(x, cout, 1, 1, 1, 1, 3, 3)), layer._backward_plan(x, layer.selection)
    planes = 2 * cout * x[:, 0].numel() * 4
    assert _lib.load().clg_convblock_backward_planned_scratch_bytes(0, geom, sig) >= planes
    y = layer(x)
    gy = torch.randn_like(y)
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    (got,) = torch.autograd.grad(y, [layer.weights], gy)
    assert torch.cuda.max_memory_allocated() - before < planes // 2
    y = layer(x.requires_grad_(True))
    want = torch.autograd.grad(y, [x, layer.weights], gy)[1]
    # two orders of the same terms, each at most |grad_y|, that a gradient of a gate adds with coefficients of absolute sum <= 5, the softmax at most
    # doubling it; 12 roundings make a term, 16 additions a lane's sum, 73 join lanes, wavefronts and parts
    bound = 2 * 2 * 5 * (12 + 16 + 73) * 2.0**-24 * gy.abs().double().sum((0, 2, 3))
    assert ((got.double() - want.double()).abs().amax((1, 2)) <= bound).all()


def test_a_kept_plan_is_complete():
    # what a first call leaves for calls on other streams: the tables of a block's plan and of a network's trees
    torch.manual_seed(5)
    layer, x = C.ConvLogicLayer(8, 16, padding=1, complete=True, implementation="cuda").to(DEV), torch.rand(4, 8, 8, 8, device=DEV)
    chain = [C.LogicLayer(a, b, implementation="cuda").to(DEV) for a, b in ((40, 80), (80, 40), (40, 20))]
    busy = torch.randn(4096, 4096, device=DEV)
    torch.cuda.synchronize()
    for make in (lambda: layer._backward_plan(x, layer.selection), lambda: fc_tree.tree_plan(*chain)):
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            for _ in range(20):                                        # the stream is behind when the plan is asked for
                busy @ busy
            assert make() is not None and side.query()


def test_a_plan_made_in_a_recording_is_the_recordings_own():
    torch.manual_seed(6)
    layer = C.ConvLogicLayer(8, 16, padding=1, complete=True, implementation="cuda").to(DEV)
    static = torch.rand(4, 8, 8, 8, device=DEV)
    layer(static[:2]).sum().backward()                                 # (the selection is checked, no plan for four samples)

    def step():
        layer.weights.grad = None
        layer(static).square().sum().backward()
        return layer.weights.grad

    graph = torch.cuda.CUDAGraph()
    layer.weights.grad = None
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        layer(static).square().sum().backward()
    recorded = layer.weights.grad
    assert [key[0][0] for key in layer._plans] == [2]
    for _ in range(3):
        static.copy_(torch.rand_like(static))
        eager = step().clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, eager)


def test_a_recorded_step_replays_the_loaded_selection_and_its_plan_stays():
    torch.manual_seed(7)
    model, other = (C.ConvLogicMnistModel(k_param=2).to(DEV) for _ in range(2))
    batches = [(torch.randint(0, 2, (32, 1, 28, 28), device=DEV).float(), torch.randint(0, 10, (32,), device=DEV)) for _ in range(2)]
    loss_of = lambda x, y: torch.nn.functional.cross_entropy(model(x), y)
    step = C.GraphedStep(loss_of, batches[0], model.parameters())
    blocks = [m for m in model.network if isinstance(m, C.ConvLogicLayer) and m.__dict__.get("_plans")]
    recorded = [kept for m in blocks for kept in m._plans.values() if kept.recorded]
    assert len(recorded) == len(blocks) >= 2
    addresses = [kept.plan[0].data_ptr() for kept in recorded]
    own, another = ({k: v.clone() for k, v in m.state_dict().items()} for m in (model, other))
    for state, eager_first in ((own, True), (another, False), (own, False), (another, True)):
        model.load_state_dict(state)
        for n in range(1, 21) if eager_first else ():                  # more batch sizes than plans are kept
            model(batches[0][0][:n])
        taken = [torch.randint(0, 2**31 - 1, (1 << 12,), dtype=torch.int32, device=DEV) for _ in range(32)]   # (takes freed memory)
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
        del taken
    assert addresses == [kept.plan[0].data_ptr() for kept in recorded]
    assert all(any(kept is own for own in m._plans.values()) for m, kept in zip(blocks, recorded))
    assert all(len(m._plans) <= 17 for m in blocks)


def test_copies_and_pickles_carry_no_plans():
    layer = C.ConvLogicLayer(2, 4, complete=True, implementation="cuda")
    layer._plans = {"left by an earlier process": (None, 0)}
    for other in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer))):
        assert "_plans" not in other.__dict__ and torch.equal(other.weights, layer.weights)
    state = dict(layer.__dict__)                                       # as a pickle of an earlier version holds it
    other = C.ConvLogicLayer.__new__(C.ConvLogicLayer)
    other.__setstate__(state)
    assert "_plans" not in other.__dict__
    other.invalidate()


@pytest.mark.parametrize("route", ["moved", "dense copy"])
def test_another_selection_at_the_same_address_reaches_the_plan(route):
    torch.manual_seed(8)
    layer, other = (C.ConvLogicLayer(8, 16, padding=1, complete=True, implementation="cuda").to(DEV) for _ in range(2))
    other.weights.data.copy_(layer.weights)
    x = torch.rand(4, 8, 8, 8, device=DEV, requires_grad=True)
    if route == "dense copy":                                          # every call makes a contiguous copy of such a buffer
        layer.selection = layer.selection.t().contiguous().t()
    layer(x).sum().backward()
    if route == "moved":
        layer.cpu()
        layer.selection.copy_(other.selection)
        layer.to(DEV)
    else:
        layer.selection.copy_(other.selection)
    grads = []
    for m in (layer, other):
        x.grad = m.weights.grad = None
        m(x).square().sum().backward()
        grads.append((x.grad, m.weights.grad))
    assert all(torch.equal(a, b) for a, b in zip(*grads))
