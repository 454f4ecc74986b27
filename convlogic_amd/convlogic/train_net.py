"""A training step of a whole small network -- complete blocks, nn.Flatten, three LogicLayers as trees, GroupSum -- as one autograd node
(csrc/nodes.cpp): the kernels of the modules one after the other without the host's work between them, the set-up of all layers in one launch and
the sums that end their weight gradients in another (csrc/net_step.hip)."""
import ctypes
import types

import torch
from torch import nn

from ..difflogic import fc_tree
from ..difflogic.fc_tree import wiring_of
from ..hip import _lib
from ..hip._lib import ConvGeom
from .convlogic_layer import ConvLogicLayer

# Elements of all logits.  A larger network's step is bound by the GPU, and its gradients are handed on layer by layer, while the rest of
# the backward pass runs.
MAX_LOGITS = 4 << 20


def blocks_of(net, called_for_itself, device):
    """The blocks of a network whose modules before the last four are ConvLogicLayers in training and a Flatten, with nothing but a call of the
    modules themselves against evaluating them together, else None."""
    *blocks, flatten = list(net._modules.values())[:-4] or [None]
    if type(flatten) is not nn.Flatten or flatten.start_dim != 1 or flatten.end_dim != -1 or called_for_itself(flatten) or not blocks:
        return None
    for m in blocks:
        if (type(m) is not ConvLogicLayer or m.implementation != "cuda" or not (m.complete and m.training) or m.return_intermediate or m.return_indices
                or m.grad_factor != 1.0 or called_for_itself(m)):
            return None
        w, sel = m._parameters.get("weights"), m._buffers["selection"]
        if w is None or not (w.is_cuda and w.dtype == torch.float32 and w.is_contiguous() and w.shape == (m.out_channels, 7, 16) and sel.is_contiguous()
                             and sel.device == w.device == device):
            return None
    return blocks


def train(net, tail, plan, x, called_for_itself):
    """Class sums / tau of a training step, or None where the modules have to be called."""
    layers, group_sum = tail
    if type(x) is not torch.Tensor or x.dim() != 4 or x.shape[0] > fc_tree.MAX_BATCH or not x.is_contiguous() or _lib.traced() or layers[0]._parameters["weights"].device != x.device:
        return None
    blocks = blocks_of(net, called_for_itself, x.device)
    if blocks is None or 16 * 7 * (plan.roots + sum(m.out_channels for m in blocks)) > MAX_LOGITS:
        return None
    n, c, h, w = x.shape
    shapes = []
    for m in blocks:
        (sh, sw), (ph, pw), (kh, kw) = m.stride, m.padding, m.kernel
        if c != m.in_channels or h + 2 * ph < kh or w + 2 * pw < kw:
            return None
        shapes.append((n, c, h, w))
        c, h, w = m.out_channels, ((h + 2 * ph - kh) // sh + 1) // 2, ((w + 2 * pw - kw) // sw + 1) // 2
    last = blocks[-1]
    if not 0 < c * h * w == layers[0].in_dim or any(m.__dict__.get("feature_major_output") and m is not last for m in blocks):
        return None
    lib, args = _lib.load(), []
    for m, shape in zip(blocks, shapes):
        geo, sel, flag = (*m.stride, *m.padding, *m.kernel), m._buffers["selection"], 0
        if m.__dict__.get("binary_input"):
            if m is not blocks[0]:
                return None
            if lib.clg_convblock_bin_supported(_lib.CLG_F32, ctypes.byref(ConvGeom(*shape, m.out_channels, *geo))):
                flag = m.binary_flag_checked().device_ptr
        m._check_selection()
        made = (sel, 0) if flag else m._backward_plan(types.SimpleNamespace(shape=shape, dtype=x.dtype, device=x.device), sel)
        args.append((sel, geo, *made, m.__dict__.get("feature_major_output", False), flag))
    return _lib.nodes().network(x, [m._parameters["weights"] for m in (*blocks, *layers)], args, layers[0]._buffers["given_x_indices_of_y_start"],
                                wiring_of(*layers), plan.rows, plan.pos, plan.ids, plan.slot, plan.roots, group_sum.k, float(group_sum.tau))
