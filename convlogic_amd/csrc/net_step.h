// What the layers of a network leave to launches that serve all of them (net_step.hip).
#pragma once

#include <string.h>

#include "clg_common.h"

// clg_late_sums: which sums (and gradients) a backward call has left, and the argument of the function that takes them: CoefSums<float>
// (conv_common.h), BinSums (conv_binary.h), TreeSums (fc_tree.h).
enum { kLateNone = 0, kLateCoef = 1, kLateBin = 2, kLateTree = 3 };
template <typename T>
static inline clg_late_sums clg_late(int kind, int blocks, const T &arg)
{
    clg_late_sums l = {};
    static_assert(sizeof(T) <= sizeof(l.field), "the argument fits");
    l.kind = kind;
    l.blocks = blocks;
    memcpy(l.field, &arg, sizeof(T));
    return l;
}
