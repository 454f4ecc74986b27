"""A LogicLayer, two halving LogicLayers and a GroupSum -- the end of the reference's networks (src/convlogic/model.py:49-57,
102-107) -- as one operation.  Where every neuron of the first two layers is read exactly once, each neuron of the third is
the root of a tree of seven gates over eight input rows that no other root shares, so the three layers are evaluated, and
differentiated, without activations of their own (csrc/fc_tree.hip)."""
import weakref

import torch

from ..hip import _lib
from ..hip._lib import check, stream_ptr

# per first layer: (keys of the three wirings, weak references to the other two layers, plan); kept outside the modules so that
# copies and pickles carry no derived buffers
_PLANS = weakref.WeakKeyDictionary()


class TreePlan:
    """The trees of three layers' wiring: input rows, neuron ids and list positions of every root's eight operands, and the
    place of every neuron in its tree (int32 on the device; include/convlogic_amd.h).  `fits`: every neuron of the first two
    layers is read exactly once, so there are trees."""

    def __init__(self, first, second, third):
        roots = self.roots = third.out_dim
        tables = torch.empty((31 * roots,), dtype=torch.int32, device=first._buffers["indices_0"].device)
        self.rows, self.pos, self.ids, self.slot = tables.split([8 * roots, 8 * roots, 8 * roots, 7 * roots])
        wiring = [m._buffers[name] for m in (first, second, third) for name in ("indices_0", "indices_1")]
        wiring += [first._buffers[name] for name in ("given_x_indices_of_y_start", "given_x_indices_of_y")]
        check(_lib.load().clg_fc_tree_plan(*(t.data_ptr() for t in wiring), *(t.data_ptr() for t in (self.rows, self.pos, self.ids, self.slot)),
                                           first.in_dim, roots, stream_ptr(tables)))
        self.fits = int(self.slot.min()) >= 0


def tree_plan(first, second, third):
    """The TreePlan of three LogicLayers, or None when their wiring does not make trees.  Rebuilt when a wiring buffer was
    modified in place, replaced or moved, when invalidate() was called on one of the layers, and for other layers."""
    if 2 * second.out_dim != second.in_dim or 2 * third.out_dim != third.in_dim or second.in_dim != first.out_dim or third.in_dim != second.out_dim:
        return None
    keys = (first._check_wiring(), second._check_wiring(), third._check_wiring())
    cached = _PLANS.get(first)
    if cached is None or cached[0] != keys or cached[1]() is not second or cached[2]() is not third:
        plan = TreePlan(first, second, third)
        cached = _PLANS[first] = (keys, weakref.ref(second), weakref.ref(third), plan if plan.fits else None)
    return cached[3]


class _TreeFunction(torch.autograd.Function):
    """x feature-major [features, B] -> class sums [B, k] / tau of the three layers; gradients of x and of the logits."""

    @staticmethod
    def forward(ctx, x, l0, l1, l2, start, plan, k, tau):
        lib, st = _lib.load(), stream_ptr(x)
        in_dim, batch = x.shape
        coef = torch.empty((plan.roots, 28), dtype=torch.float32, device=x.device)
        probs = torch.empty((7 * plan.roots, 16), dtype=torch.float32, device=x.device)
        check(lib.clg_fc_tree_fold(l0.data_ptr(), l1.data_ptr(), l2.data_ptr(), plan.ids.data_ptr(), coef.data_ptr(), probs.data_ptr(),
                                   plan.roots, 0, st))
        out = _tree_forward(lib, x, plan, coef, k, tau, st)
        # (probabilities, not logits, as in the modules: the logits may be updated between forward and backward)
        ctx.save_for_backward(x, start, coef, probs)
        ctx.plan, ctx.k, ctx.tau = plan, k, tau
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x, start, coef, probs = ctx.saved_tensors
        plan, k = ctx.plan, ctx.k
        grad_out = _lib.check_input(grad_out.contiguous(), "grad_out", torch.float32, (x.shape[1], k))
        _lib.check_same_device(x, grad_out)
        in_dim, batch = x.shape
        gx = torch.empty_like(x)
        g0, g1, g2 = (torch.empty((n * plan.roots, 16), dtype=torch.float32, device=x.device) for n in (4, 2, 1))
        scratch = torch.empty((plan.roots * (8 * batch + 28),), dtype=torch.float32, device=x.device)   # rowgrad, then sums
        rowgrad, sums = scratch.data_ptr(), scratch.data_ptr() + plan.roots * 8 * batch * 4
        check(_lib.load().clg_fc_tree_backward(
            x.data_ptr(), plan.rows.data_ptr(), plan.pos.data_ptr(), plan.slot.data_ptr(), coef.data_ptr(), grad_out.data_ptr(),
            probs.data_ptr(), g0.data_ptr(), g1.data_ptr(), g2.data_ptr(), rowgrad, sums, start.data_ptr(),
            gx.data_ptr(), in_dim, plan.roots, k, batch, batch, float(ctx.tau), stream_ptr(x)))
        return gx, g0, g1, g2, None, None, None, None


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
    return _TreeFunction.apply(x, first.weights, second.weights, third.weights, first._buffers["given_x_indices_of_y_start"], plan,
                               group_sum.k, group_sum.tau)


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
