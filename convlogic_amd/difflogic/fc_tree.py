"""A LogicLayer, two halving LogicLayers and a GroupSum -- the end of the reference's networks (src/convlogic/model.py:49-57,
102-107) -- as one operation.  Where every neuron of the first two layers is read exactly once, each neuron of the third is
the root of a tree of seven gates over eight input rows that no other root shares, so the three layers are evaluated, and
differentiated, without activations of their own (csrc/fc_tree.hip)."""
import threading
import weakref

import torch

from ..hip import _lib
from ..hip._lib import check, stream_ptr

MAX_BATCH = 1 << 20                                                   # samples of a call, within what the kernels' grids hold

# per first layer: the _Entry of every pair of layers that was seen behind it; kept outside the modules so that copies and pickles
# carry no derived buffers
_PLANS = weakref.WeakKeyDictionary()
_BUILDING = threading.Lock()


class TreePlan:
    """The trees of three layers' wiring: input rows, neuron ids and list positions of every root's eight operands, and the
    place of every neuron in its tree (int32 on the device; include/convlogic_amd.h).  The tables stay where they are for the
    plan's life: a recorded HIP graph reads them at these addresses."""

    def __init__(self, first, second, third):
        self.roots, self.device = third.out_dim, first._buffers["indices_0"].device
        tables = torch.empty((31 * self.roots,), dtype=torch.int32, device=self.device)
        self.rows, self.pos, self.ids, self.slot = tables.split([n * self.roots for n in (8, 8, 8, 7)])
        self.build(first, second, third)

    def build(self, first, second, third):
        wiring = wiring_of(first, second, third)
        wiring += [first._buffers[name] for name in ("given_x_indices_of_y_start", "given_x_indices_of_y")]
        check(_lib.load().clg_fc_tree_plan(*(t.data_ptr() for t in wiring), *(t.data_ptr() for t in (self.rows, self.pos, self.ids, self.slot)),
                                           first.in_dim, self.roots, stream_ptr(self.slot)))

    def fits(self):
        """True when every neuron of the first two layers is read exactly once, so that there are trees.  Waits for the tables."""
        return int(self.slot.min()) >= 0


class _Entry:
    def __init__(self, second, third):
        self.second, self.third = weakref.ref(second), weakref.ref(third)
        self.keys = self.plan = None
        self.fits = False

    def is_of(self, second, third):
        return self.second() is second and self.third() is third


def wiring_of(*layers):
    return [m._buffers[name] for m in layers for name in ("indices_0", "indices_1")]


def tree_plan(first, second, third):
    """The TreePlan of three LogicLayers, or None when their wiring does not make trees.  Made again, in the same tables, when
    a wiring buffer was modified in place, replaced or moved and when invalidate() was called on one of the layers.  (Made
    outside a recording only: making it waits for the device.)"""
    if 2 * second.out_dim != second.in_dim or 2 * third.out_dim != third.in_dim or second.in_dim != first.out_dim or third.in_dim != second.out_dim:
        return None
    keys = (first._check_wiring(), second._check_wiring(), third._check_wiring())
    for entry in _PLANS.get(first, ()):
        if entry.keys == keys and entry.is_of(second, third):
            break
    else:
        if first._buffers["indices_0"].is_cuda and torch.cuda.is_current_stream_capturing():
            return None
        with _BUILDING:
            entry = _make(first, second, third, keys)
    return entry.plan if entry.fits else None


def _make(first, second, third, keys):
    entries = _PLANS.setdefault(first, [])
    entry = next((e for e in entries if e.is_of(second, third)), None)
    if entry is None:
        entry = _Entry(second, third)
    elif entry.keys == keys:                                          # another thread made it meanwhile
        return entry
    entry.keys = None
    if entry.plan is None or entry.plan.device != first._buffers["indices_0"].device:
        entry.plan, had = TreePlan(first, second, third), False
    else:
        entry.plan.build(first, second, third)
        had = True
    entry.fits = entry.plan.fits()
    if not (entry.fits or had):
        entry.plan = None                                             # no trees, and nothing recorded with them
    entry.keys = keys
    _PLANS[first] = [e for e in entries if e.second() is not None and e.third() is not None and e is not entry] + [entry]
    return entry


def refresh(layer):
    """Makes the tables of the plans that `layer` belongs to again (a state was loaded into it): a step that was recorded with
    them replays the loaded wiring.  In the stream's order; the next tree_plan() looks at the result.  A wiring that the next
    call refuses (load_state_dict(assign=True) takes any type and stride) is not read: the tables stay as they were."""
    with _BUILDING:
        for first, entries in list(_PLANS.items()):
            for e in entries:
                second, third = e.second(), e.third()
                if e.plan is None or second is None or third is None or layer not in (first, second, third):
                    continue
                if all(t.device == e.plan.device for t in wiring_of(first, second, third)) and _checked(first, second, third):
                    e.plan.build(first, second, third)


def _checked(*layers):
    try:
        for m in layers:
            m._check_wiring()
    except ValueError:
        return False
    return True


class _TreeFunction(torch.autograd.Function):
    """x feature-major [features, B] -> class sums [B, k] / tau of the three layers; gradients of x and of the logits."""

    @staticmethod
    def forward(ctx, x, l0, l1, l2, start, wiring, plan, k, tau):
        lib, st = _lib.load(), stream_ptr(x)
        in_dim, batch = x.shape
        coef = torch.empty((plan.roots, 28), dtype=torch.float32, device=x.device)
        probs = torch.empty((7 * plan.roots, 16), dtype=torch.float32, device=x.device) if any(ctx.needs_input_grad[1:4]) else None
        check(lib.clg_fc_tree_fold(l0.data_ptr(), l1.data_ptr(), l2.data_ptr(), plan.ids.data_ptr(), coef.data_ptr(), _ptr(probs), plan.roots, 0, st))
        out = _tree_forward(lib, x, plan, coef, k, tau, st)
        # (probabilities, not logits, as in the modules: the logits may be updated between forward and backward; the wiring for
        # autograd's check that it was not)
        ctx.save_for_backward(x, start, coef, probs, *wiring)
        ctx.plan, ctx.k, ctx.tau = plan, k, tau
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x, start, coef, probs = ctx.saved_tensors[:4]
        plan, k = ctx.plan, ctx.k
        grad_out = _lib.check_input(grad_out.contiguous(), "grad_out", torch.float32, (x.shape[1], k))
        _lib.check_same_device(x, grad_out)
        (in_dim, batch), roots = x.shape, plan.roots
        need_x, need = ctx.needs_input_grad[0], ctx.needs_input_grad[1:4]
        gx = torch.empty_like(x) if need_x else None
        grads = [torch.empty((n * roots, 16), dtype=torch.float32, device=x.device) if needed else None for n, needed in zip((4, 2, 1), need)]
        rows = 8 * roots * batch if need_x else 0
        scratch = torch.empty((rows + 28 * roots,), dtype=torch.float32, device=x.device)       # rowgrad, then sums
        check(_lib.load().clg_fc_tree_backward(
            x.data_ptr(), plan.rows.data_ptr(), plan.pos.data_ptr(), plan.slot.data_ptr(), coef.data_ptr(), grad_out.data_ptr(), _ptr(probs),
            *(_ptr(g) for g in grads), scratch.data_ptr(), scratch.data_ptr() + 4 * rows, start.data_ptr(), _ptr(gx), in_dim, roots, k, batch,
            batch, float(ctx.tau), stream_ptr(x)))
        return gx, *grads, None, None, None, None, None


def _ptr(t):
    return None if t is None else t.data_ptr()


def _tree_forward(lib, x, plan, coef, k, tau, st):
    in_dim, batch = x.shape
    out = torch.empty((batch, k), dtype=torch.float32, device=x.device)
    partial = torch.empty((lib.clg_fc_tree_partial_elems(plan.roots, k, batch, batch),), dtype=torch.float32, device=x.device)
    check(lib.clg_fc_tree_forward(x.data_ptr(), plan.rows.data_ptr(), coef.data_ptr(), partial.data_ptr(), out.data_ptr(), in_dim,
                                  plan.roots, k, batch, batch, float(tau), st))
    return out


class _TreeEvalFunction(torch.autograd.Function):
    """The same class sums with the arg-max gates: evaluation, which has no gradient."""

    @staticmethod
    def forward(ctx, x, l0, l1, l2, plan, k, tau):
        lib, st = _lib.load(), stream_ptr(x)
        coef = torch.empty((plan.roots, 28), dtype=torch.float32, device=x.device)
        check(lib.clg_fc_tree_fold(l0.data_ptr(), l1.data_ptr(), l2.data_ptr(), plan.ids.data_ptr(), coef.data_ptr(), None, plan.roots, 1, st))
        return _tree_forward(lib, x, plan, coef, k, tau, st)


def tree_eval(layers, group_sum, x, plan):
    """group_sum(third(second(first(x)))) of layers in evaluation mode; x feature-major [features, B]."""
    with torch.no_grad():
        return _TreeEvalFunction.apply(x, *(layer.weights for layer in layers), plan, group_sum.k, group_sum.tau)


def tree_train(layers, group_sum, x, plan):
    """group_sum(third(second(first(x)))) in training; x feature-major [features, B]."""
    first, second, third = layers
    if not _lib.traced():
        return _lib.nodes().trees(x, first.weights, second.weights, third.weights, first._buffers["given_x_indices_of_y_start"], wiring_of(*layers),
                                  plan.rows, plan.pos, plan.ids, plan.slot, plan.roots, group_sum.k, float(group_sum.tau))
    return _TreeFunction.apply(x, first.weights, second.weights, third.weights, first._buffers["given_x_indices_of_y_start"],
                               wiring_of(*layers), plan, group_sum.k, group_sum.tau)


def tree_packed(layers, k, x, plan):
    """Class counts int32 [samples, k] of packed words x (a PackBitsTensor of 64 samples per word)."""
    words = x.t
    lib = _lib.load()
    samples = words.shape[1] * 64 - x.pad_len
    out = torch.empty((samples, k), dtype=torch.int32, device=words.device)
    codes = torch.empty((plan.roots,), dtype=torch.int32, device=words.device)
    l0, l1, l2 = (layer.weights.detach() for layer in layers)
    check(lib.clg_fc_tree_packed(words.data_ptr(), plan.rows.data_ptr(), plan.ids.data_ptr(), l0.data_ptr(), l1.data_ptr(), l2.data_ptr(),
                                 codes.data_ptr(), out.data_ptr(), words.shape[0], plan.roots, k, words.shape[1], samples, stream_ptr(words)))
    return out
