"""Network topologies of the reference's src/convlogic/model.py as plain nn.Modules: the caller side of
the logic-layer kernels.  Constructor arguments, layer order and the `network` attribute are the
reference's, so parameters are drawn in the same RNG order and state_dict keys (`network.<i>.weights`,
`network.<i>.selection`, `network.<i>.indices_0`, ...) match checkpoints written from there (the
Lightning wrapper of src/convlogic/model.py:111-200 prefixes them with `model.`)."""
import weakref

import torch
from torch import nn

from ..difflogic import GroupSum, LogicLayer
from ..difflogic.difflogic import _feature_major, logic_layer_group_sum
from ..difflogic import fc_tree
from ..difflogic.fc_tree import tree_eval, tree_packed, tree_plan, tree_train
from ..difflogic.packbitstensor import PackBitsTensor
from ..hip.convlogic_hip import bin_supported
from . import packed_net, train_net
from .convlogic_layer import ConvLogicLayer


# per network: (dtype, device), the layers that take a fold made ahead, and the bookkeeping of that launch (kept outside the
# module so that copies and pickles of a network carry no host pointers)
_FOLD_PLANS = weakref.WeakKeyDictionary()


_PREFOLD_MIN_ELEMS = 20 << 19                                     # 512 Ki rows of logits


def _prefold(owner, layers, x, mode=True):
    """Folds the logits of `layers` (a network's, in order) for a training step in ONE launch and leaves each layer its
    (probabilities, coefficients): softmax and fold are then no part of the layers' forward launches -- the LogicLayers run
    their plain streaming kernel, the deep blocks skip their set-up launch.  Same values as the per-layer folds (tested)."""
    from ..hip import difflogic_hip
    cache = _FOLD_PLANS.get(owner)
    if cache is not None and cache[0] != (x.dtype, x.device, len(layers)):
        cache = None
    if cache is not None:
        _, picked, plan = cache
        weights = [m._parameters["weights"] for m in picked]
        if plan is None:                                             # nothing to fold when the cache was made: look again
            cache = None
        elif not (plan.matches(weights) and all(m.prefold_candidate() is w for m, w in zip(picked, weights))):
            cache = None
    if cache is None:
        picked = [m for m in layers for w in [m.prefold_candidate()] if w is not None and w.dtype == x.dtype and w.device == x.device]
        picked = picked[:difflogic_hip.FOLD_MANY_MAX]
        weights = [m._parameters["weights"] for m in picked]
        plan = difflogic_hip.FoldPlan([w.detach() for w in weights]) if len(picked) >= 2 else None
        _FOLD_PLANS[owner] = ((x.dtype, x.device, len(layers)), picked, plan)
    if plan is None:
        return
    # An eager step of a small network whose modules are called is bound by the host, where the bookkeeping of this launch costs more than
    # the layers' own allocations save (+15 us per step): by default only networks whose step the GPU bounds fold ahead.  "always" is for smaller
    # ones that are replayed from a HIP graph and cannot run as one node (train_net.py), which by default sets all layers up in one launch and is
    # the faster way: replayed step of the k = 32 CIFAR network with 256 images 267 us as one node, 291 with "always", 292 without; MNIST, 100
    # images, 140, 163 and 161.
    if mode != "always" and plan.total < _PREFOLD_MIN_ELEMS:
        return
    for m, (probs, folded) in zip(picked, difflogic_hip.fold_many([w.detach() for w in weights], plan)):
        m.set_prefold(probs, folded)


def _called_for_itself(module):
    """True when a call of the module does more than its class's forward: hooks of either pass, a replaced forward."""
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or "forward" in module.__dict__)


def _tree_tail(net):
    """The last four modules of a network -- three LogicLayers and a GroupSum -- when nothing but a call of the modules
    themselves stands against evaluating them as one operation (difflogic/fc_tree.py), else None."""
    if type(net) is not nn.Sequential or len(net._modules) < 4 or _called_for_itself(net) or torch.nn.modules.module._has_any_global_hook():
        return None                                                   # (a wrapped network, or one with a forward of its own, is called)
    *layers, gs = list(net._modules.values())[-4:]
    if type(gs) is not GroupSum or _called_for_itself(gs):
        return None
    device = None
    for m in layers:
        if type(m) is not LogicLayer or m.implementation != "cuda" or m.grad_factor != 1.0 or _called_for_itself(m):
            return None
        w = m._parameters["weights"]
        device = device or w.device
        if not (w.is_cuda and w.dtype == torch.float32 and w.shape == (m.out_dim, 16) and w.is_contiguous() and w.device == device):
            return None
    if layers[-1].out_dim % gs.k != 0 or gs.tau == 0:
        return None
    if gs.k > 65535 or layers[0].in_dim >= 1 << 31 or layers[-1].out_dim >= 1 << 28:   # (what the tree kernels' indices hold)
        return None
    return layers, gs


def _forward(owner, x):
    """The network on x.  Three things happen that a plain nn.Sequential call would not do: the three LogicLayers and the
    GroupSum at its end are evaluated as one operation where their wiring allows (`tree_tail`, default on; training steps,
    evaluation and packed inference), in training of a small network the blocks in front of them as well (unless `prefold` is set); else the
    logits of the other layers are folded in one launch where that pays (`prefold`), and a last LogicLayer and GroupSum that do not run as trees run as one autograd node (`fused_tail`, default on), whose
    backward needs no GroupSum launch."""
    net = owner.network
    tail = _tree_tail(net) if owner.__dict__.get("tree_tail", True) else None
    if isinstance(x, PackBitsTensor):
        trees = tail is not None and not any(m.training for m in (owner, *tail[0])) and x.is_cuda and x.bit_count == 64
        plan = tree_plan(*tail[0]) if trees else None
        if plan is None:
            return net(x)
        counts = _counts_at_once(net, tail, plan, x)
        if counts is not None:
            return counts
        h = _head_of(net, x)
        if (type(h) is not PackBitsTensor or h.image or h.t.shape[0] != tail[0][0].in_dim or not h.t.is_contiguous()
                or h.t.device != tail[0][0]._parameters["weights"].device or _many_small_classes(plan.roots, tail[1].k, h.t.shape[1])):
            return _rest(net, h)
        return tree_packed(tail[0], tail[1].k, h, plan)
    if not (isinstance(x, torch.Tensor) and x.is_cuda):
        return net(x)
    trees = tail is not None and x.dtype == torch.float32 and x.dim() > 0 and x.shape[0] > 0
    if not (owner.training and torch.is_grad_enabled()):
        if not trees or any(m.training for m in tail[0]) or (plan := tree_plan(*tail[0])) is None:
            return net(x)
        out = _sums_at_once(net, tail, plan, x)
        if out is not None:
            return out
        h = _head_of(net, x)
        if _trees_take(h, tail[0][0]):
            return tree_eval(tail[0], tail[1], _feature_major(h.detach()), plan)
        return _rest(net, h)
    plan = tree_plan(*tail[0]) if trees and all(m.training for m in tail[0]) else None
    mode = owner.__dict__.get("prefold", True)                       # True: where it pays, "always", False
    if plan is not None and mode is True:
        out = train_net.train(net, tail, plan, x, _called_for_itself)
        if out is not None:
            return out
    if mode:
        layers = [m for m in net if isinstance(m, (ConvLogicLayer, LogicLayer))]
        _prefold(owner, layers if plan is None else layers[:-3], x, mode)
    if plan is not None:
        h = _head_of(net, x)
        if _trees_take(h, tail[0][0]):
            return tree_train(tail[0], tail[1], _feature_major(h), plan)
        return _rest(net, h)
    n = len(net)
    if (owner.__dict__.get("fused_tail", True) and n >= 2 and isinstance(net[n - 2], LogicLayer) and isinstance(net[n - 1], GroupSum)
            and not (net._forward_hooks or net._forward_pre_hooks)):
        h = x
        for i, m in enumerate(net):
            if i == n - 2:
                break
            h = m(h)
        return logic_layer_group_sum(net[n - 2], net[n - 1], h)
    return net(x)


def _counts_at_once(net, tail, plan, x):
    """Class counts of packed images with every module of the network in one call (packed_net), or None where the modules have to be
    called.  x holds the words in front of the trees afterwards, as after the modules."""
    t, (layers, gs) = x.t, tail
    if not (type(x) is PackBitsTensor and x.image and t.dim() == 4 and t.dtype == torch.int64 and t.is_contiguous() and t.shape[0] > 0
            and 0 <= x.pad_len < 64):
        return None
    blocks = packed_net.blocks_of(net, _called_for_itself)
    if blocks is None or t.device != blocks[0]._parameters["weights"].device or t.device != layers[0]._parameters["weights"].device:
        return None
    geoms = packed_net.geometries(blocks, *t.shape, layers[0].in_dim)
    if geoms is None or _many_small_classes(plan.roots, gs.k, t.shape[0]):
        return None
    x.t, counts = packed_net.evaluate(blocks, geoms, t, layers, plan, gs.k, t.shape[0] * 64 - x.pad_len)
    x.image = False
    return counts


def _sums_at_once(net, tail, plan, x):
    """Class sums of 0/1 images (the first block's binary_input, verified by the kernels) on packed bits, or None.  The activations become
    bits, which is exact: each is 0 or 1, and a class sum is a whole number.  Against the float kernels, replayed from a recorded graph
    (called eagerly): 206 -> 49 us (199 -> 61) for 1000 images of the k = 32 CIFAR network, 714 -> 74 (697 -> 70) at k = 128; one image
    of networks from MNIST k = 8 to CIFAR k = 256 38 to 92 -> 30 to 64 (120 to 156 -> 53 to 67)."""
    layers, gs = tail
    if x.dim() != 4 or x.shape[0] > 65535 * 64 or gs.k >= 512:
        return None
    blocks = packed_net.blocks_of(net, _called_for_itself)
    if blocks is None or not blocks[0].__dict__.get("binary_input") or not (
            x.device == blocks[0]._parameters["weights"].device == layers[0]._parameters["weights"].device):
        return None
    n, c, h, w = x.shape
    first = blocks[0]
    geoms = packed_net.geometries(blocks, -(-n // 64), c, h, w, layers[0].in_dim)
    if geoms is None or not bin_supported(x, first.out_channels, *first.stride, *first.padding, *first.kernel):
        return None
    return packed_net.evaluate_images(blocks, geoms, x.contiguous(), layers, gs, plan)


def _many_small_classes(roots, k, words):
    """True for packed words on which the modules are the faster ones: the trees' workgroups each add up the counts of a class,
    which costs as much for one root as for hundreds (1000 classes of one root, 256 samples: 22 us, 13 by the modules; of
    16 roots: 34 and 37; of one root, 20 000 samples: 149 and 288)."""
    rows = roots // k
    return k >= 512 and rows <= 16 and rows * words * 64 <= 4096


def _trees_take(h, first):
    """True for what the modules themselves would accept (they raise for anything else), up to the kernels' grid"""
    return (h.dim() == 2 and h.shape[1] == first.in_dim and h.dtype == torch.float32 and h.device == first._parameters["weights"].device
            and h.shape[0] <= fc_tree.MAX_BATCH)


def _head_of(net, h):
    """all but the last four modules of a network"""
    for m in list(net._modules.values())[:-4]:
        h = m(h)
    return h


def _rest(net, h):
    """the last four"""
    for m in list(net._modules.values())[-4:]:
        h = m(h)
    return h


def _block(c_in, c_out, implementation, **kw):
    return ConvLogicLayer(in_channels=c_in, out_channels=c_out, residual_init=True, complete=True,
                          implementation=implementation, **kw)


def _head(dims, tau, implementation):
    fc = [LogicLayer(a, b, grad_factor=1, residual_init=True, implementation=implementation) for a, b in zip(dims, dims[1:])]
    return [nn.Flatten(), *fc, GroupSum(k=10, tau=tau)]


class ConvLogicCifarModel(nn.Module):
    """Four 3x3 / padding 1 blocks of k, 4k, 16k, 32k kernels (each halves the image), then three
    LogicLayers of 10, 5 and 2.5 times the flattened width (doubled from k = 1024) and a 10-class
    GroupSum (src/convlogic/model.py:11-60)."""

    def __init__(self, k_param=32, input_channels=3, input_size=32, tau=20, implementation="cuda"):
        super().__init__()
        self.input_size = input_size
        self.k_param = k_param
        self.extra_layers = 2 if k_param >= 1024 else 1
        widths = [input_channels] + [m * k_param for m in (1, 4, 16, 32)]
        blocks = [_block(a, b, implementation, padding=1, groups=1) for a, b in zip(widths, widths[1:])]
        side = input_size // 2 ** len(blocks)
        flat = widths[-1] * side * side
        m = self.extra_layers
        dims = [flat, m * flat * 10, m * flat * 5, m * (flat * 10) // 4]
        # the last block feeds nn.Flatten and a LogicLayer, which reads feature-major memory: when the block's kernels
        # can write that layout (4x4 images on the GPU) its output is the [N, C, 2, 2] view of a [C, 2, 2, N] tensor
        blocks[-1].feature_major_output = implementation == "cuda"
        # the network's input is the thresholded image (src/convlogic/data.py:46-50): every element is 0 or 1
        blocks[0].binary_input = implementation == "cuda"
        self.network = nn.Sequential(*blocks, *_head(dims, tau, implementation))

    def forward(self, x):
        return _forward(self, x)


class ConvLogicMnistModel(nn.Module):
    """A 5x5 / padding 0 block of k kernels (28 -> 24 -> 12), two 3x3 / padding 1 blocks of 3k and 9k
    kernels (-> 6 -> 3), then LogicLayers 81k -> 1280k -> 640k -> 320k and a 10-class GroupSum
    (src/convlogic/model.py:63-108)."""

    def __init__(self, input_channels=1, input_size=28, k_param=32, tau=6.5, implementation="cuda"):
        super().__init__()
        k = k_param
        blocks = [_block(input_channels, k, implementation, kernel=5, padding=0),
                  _block(k, 3 * k, implementation, kernel=3, padding=1),
                  _block(3 * k, 9 * k, implementation, kernel=3, padding=1)]
        blocks[0].binary_input = implementation == "cuda"          # binarised digits, as in the CIFAR topology
        self.network = nn.Sequential(*blocks, *_head([81 * k, 1280 * k, 640 * k, 320 * k], tau, implementation))

    def forward(self, x):
        return _forward(self, x)
