"""Evaluation of a whole network -- complete blocks, nn.Flatten, three LogicLayers as trees, GroupSum -- on packed bits in one call
of the library: what the modules do one after the other, without the host's work between their launches.  A network on
0/1 float images in evaluation is the same bits: every activation is 0 or 1 and a class sum a whole number."""
import ctypes

import torch
from torch import nn

from ..hip import _lib, convlogic_hip
from ..hip._lib import ConvGeom, PackedBlock, check, stream_ptr
from .convlogic_layer import ConvLogicLayer

MAX_BLOCKS = 16


def blocks_of(net, called_for_itself):
    """The blocks of a network whose modules before the last four are ConvLogicLayers and a Flatten that can be evaluated together,
    else None."""
    *blocks, flatten = list(net._modules.values())[:-4] or [None]
    if (type(flatten) is not nn.Flatten or flatten.start_dim != 1 or flatten.end_dim != -1 or called_for_itself(flatten)
            or not 0 < len(blocks) <= MAX_BLOCKS):
        return None
    for m in blocks:
        if (type(m) is not ConvLogicLayer or m.implementation != "cuda" or not m.complete or m.training or m.return_intermediate or m.return_indices
                or called_for_itself(m) or m.out_channels > 65535):
            return None
        w, sel = m._parameters["weights"], m._buffers["selection"]
        if not (w.is_cuda and w.dtype == torch.float32 and w.is_contiguous() and w.shape == (m.out_channels, 7, 16) and sel.is_contiguous()
                and sel.device == w.device == blocks[0]._parameters["weights"].device):
            return None
    return blocks


def geometries(blocks, n, c, h, w, features):
    """The ConvGeom of every block for n groups of images [c, h, w], or None for what a block or the trees would refuse."""
    out = []
    for m in blocks:
        (sh, sw), (ph, pw), (kh, kw) = m.stride, m.padding, m.kernel
        if c != m.in_channels or h + 2 * ph < kh or w + 2 * pw < kw:
            return None
        out.append(ConvGeom(n, c, h, w, m.out_channels, sh, sw, ph, pw, kh, kw))
        ho, wo = (h + 2 * ph - kh) // sh + 1, (w + 2 * pw - kw) // sw + 1
        if ho % 2 or wo % 2:
            return None
        c, h, w = m.out_channels, ho // 2, wo // 2
    return out if c * h * w == features else None


def evaluate(blocks, geoms, words, layers, plan, k, samples, tau=None):
    """-> (words between blocks and trees [features, groups], class counts int32 [samples, k], or with tau their quotients by it)."""
    lib, dev = _lib.load(), words.device
    n = len(blocks)
    table = (PackedBlock * n)()
    for entry, m, g in zip(table, blocks, geoms):
        m._check_selection()
        entry.geom, entry.logits, entry.selection = g, m._parameters["weights"].data_ptr(), m._buffers["selection"].data_ptr()
    in_dim = layers[0].in_dim
    scratch = convlogic_hip._scratch(lib.clg_net_packed_scratch_bytes(table, n, in_dim, plan.roots, k, samples), dev)
    features = torch.empty((in_dim, words.shape[0]), dtype=torch.int64, device=dev)
    out = torch.empty((samples, k), dtype=torch.int32 if tau is None else torch.float32, device=dev)
    counts, sums = (out.data_ptr(), None) if tau is None else (None, out.data_ptr())
    check(lib.clg_net_packed(table, n, words.data_ptr(), plan.rows.data_ptr(), plan.ids.data_ptr(),
                             *(m._parameters["weights"].data_ptr() for m in layers), features.data_ptr(), counts, sums,
                             1.0 if tau is None else float(tau), in_dim, plan.roots, k, samples, scratch.data_ptr(), stream_ptr(words)))
    return features, out


class _EvalFunction(torch.autograd.Function):
    """0/1 float images -> class sums / tau; evaluation, which has no gradient."""

    @staticmethod
    def forward(ctx, x, flag, blocks, geoms, layers, plan, k, tau, *logits):
        n, c, h, w = x.shape
        words = torch.empty((geoms[0].n, c, h, w), dtype=torch.int64, device=x.device)
        check(_lib.load().clg_pack_binary_images(x.data_ptr(), words.data_ptr(), n, c, h * w, flag.device_ptr, stream_ptr(x)))
        return evaluate(blocks, geoms, words, layers, plan, k, n, tau)[1]


def evaluate_images(blocks, geoms, x, layers, group_sum, plan):
    flag = blocks[0].binary_flag_checked()
    with torch.no_grad():
        return _EvalFunction.apply(x, flag, blocks, geoms, layers, plan, group_sum.k, group_sum.tau,
                                   *(m._parameters["weights"] for m in (*blocks, *layers)))
