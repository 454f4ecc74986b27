// Folding the logits of trees (fc_tree.hip) and the gradients of the logits, as what a workgroup of 256 threads does: launches of their own, or part
// of one for all layers of a network (net_step.hip).
#pragma once

#include "conv_common.h"
#include "conv_pair.h"

namespace {

// ---- coefficients ---------------------------------------------------------------------------------------------------
// ids [roots][8]: the neurons of a tree, 0..3 of the first layer, 4..5 of the second; the root is neuron j of the third.
// coef [roots][7][4]: fold16 of the softmax (training) or of the arg-max gate (evaluation) of their logits, in tree order, so
// that a root's 28 coefficients are one run of 112 bytes.
struct TreeLogits {
    const float *l[3];
};
// (A bad id names a wrong neuron; it never leaves the logits or the probabilities, which are written at the same place.)
__device__ __forceinline__ int64_t tree_neuron(const int32_t *__restrict__ ids, int j, int q, int roots)
{
    return q < 6 ? min((uint32_t)ids[(int64_t)j * 8 + q], (q < 4 ? 4u : 2u) * (uint32_t)roots - 1u) : (uint32_t)j;
}
// probs (or null): the probabilities, neurons of the first layer first.  The backward pass reads these: logits that an
// optimizer updates between the two passes must not reach it.
// A lane per gate does the arithmetic, four lanes per gate move its 64 bytes: the 16-byte pieces of a row go through LDS, so that an
// access of a wavefront is 16 rows in place of 64 pieces of 64 rows (131072 features, 655360 roots: 211 -> 188 us, 94080 roots 38 -> 28; what is left
// are 0.66 GB of rows, read and written in tree order).
constexpr int kFoldPitch = 20;                                       // floats of a row in LDS: 16-byte pieces, lanes spread over the banks
struct TreeFold {
    TreeLogits lg;
    const int32_t *ids;
    float *coef, *probs;
    int roots, hard;
};
__device__ __forceinline__ void tree_fold(const TreeFold &f, int64_t block)
{
    const TreeLogits &lg = f.lg;
    const int32_t *__restrict__ ids = f.ids;
    float *__restrict__ coef = f.coef, *__restrict__ probs = f.probs;
    const int roots = f.roots, hard = f.hard;
    __shared__ __align__(16) float rows[256 / kWave][kWave * kFoldPitch];
    const int lane = threadIdx.x & (kWave - 1);
    float *mine = rows[threadIdx.x >> 6];
    const int64_t gates = (int64_t)roots * 7, e0 = block * 256 + (threadIdx.x & ~(kWave - 1)), e = e0 + lane;
    if (e0 >= gates) return;                                          // (a whole wavefront; none meets another one)
    const int64_t ec = e < gates ? e : gates - 1;
    const int j = (int)(ec / 7), q = (int)(ec - (int64_t)j * 7);
    const int layer = q < 4 ? 0 : (q < 6 ? 1 : 2);
    const int neuron = (int)tree_neuron(ids, j, q, roots);
    const int place = neuron + roots * (layer == 0 ? 0 : (layer == 1 ? 4 : 6));   // of the neuron among all (below 2^31: roots < 2^28)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int from = 16 * i + (lane >> 2), l = __shfl(layer, from, kWave), n = __shfl(neuron, from, kWave);
        const float *w = l == 0 ? lg.l[0] : (l == 1 ? lg.l[1] : lg.l[2]);
        const f32x4u v = reinterpret_cast<const f32x4u *>(w + (int64_t)n * 16)[lane & 3];
        // (logits at any 4-byte boundary)
        *reinterpret_cast<float4 *>(mine + from * kFoldPitch + 4 * (lane & 3)) = make_float4(v.x, v.y, v.z, v.w);
    }
    wave_fence();                                                     // (lanes read what others wrote)
    float w[16], p[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(mine + lane * kFoldPitch + 4 * i);
        w[4 * i] = v.x, w[4 * i + 1] = v.y, w[4 * i + 2] = v.z, w[4 * i + 3] = v.w;
    }
    if (hard) {
        float best = w[0];
        int at = 0;
#pragma unroll
        for (int i = 1; i < 16; ++i)
            if (w[i] > best || (w[i] != w[i] && best == best)) best = w[i], at = i;
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = i == at ? 1.f : 0.f;
    } else {
        softmax16(w, p);
    }
    const Coef<float> c = fold16(p);
    if (e < gates) reinterpret_cast<float4 *>(coef)[e] = make_float4(c.ab, c.a, c.b, c.one);
    if (probs == nullptr) return;
    wave_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4 *>(mine + lane * kFoldPitch + 4 * i) = make_float4(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]);
    wave_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int from = 16 * i + (lane >> 2), at = __shfl(place, from, kWave);
        const float4 v = *reinterpret_cast<const float4 *>(mine + from * kFoldPitch + 4 * (lane & 3));
        if (e0 + from < gates) reinterpret_cast<float4 *>(probs + (int64_t)at * 16)[lane & 3] = v;
    }
}

// The same for training, neuron by neuron in the order of the layers: logits and probabilities in whole lines, the 16 bytes of coefficients at the
// neuron's slot (root * 7 + gate).  In tree order both are pieces of 64 bytes, half a line each (655360 roots: 193 us, here 169, the coefficients' pieces are what is left).
struct TreeFoldSlots {
    TreeLogits lg;
    const int32_t *slot;
    float *coef, *probs;
    int64_t end[3];       // neurons of the first one, two, three layers
};
template <bool STREAM>
__device__ __forceinline__ void tree_fold_slots(const TreeFoldSlots &f, int64_t block)
{
    __shared__ __align__(16) float rows[256 / kWave][kWave * kFoldPitch];
    const int lane = threadIdx.x & (kWave - 1);
    float *mine = rows[threadIdx.x >> 6];
    const int64_t e0 = block * 256 + (threadIdx.x & ~(kWave - 1)), e = e0 + lane, all = f.end[2];
    if (e0 >= all) return;                                            // (a whole wavefront; none meets another one)
    const uint32_t slot = e < all ? (uint32_t)f.slot[e] : 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int from = 16 * i + (lane >> 2);
        const int64_t n = min(e0 + from, all - 1);
        const int layer = n < f.end[0] ? 0 : (n < f.end[1] ? 1 : 2);
        const f32x4u v = reinterpret_cast<const f32x4u *>(f.lg.l[layer] + (n - (layer ? f.end[layer - 1] : 0)) * 16)[lane & 3];
        *reinterpret_cast<float4 *>(mine + from * kFoldPitch + 4 * (lane & 3)) = make_float4(v.x, v.y, v.z, v.w);
    }
    wave_fence();                                                     // (lanes read what others wrote)
    float w[16], p[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(mine + lane * kFoldPitch + 4 * i);
        w[4 * i] = v.x, w[4 * i + 1] = v.y, w[4 * i + 2] = v.z, w[4 * i + 3] = v.w;
    }
    softmax16(w, p);
    const Coef<float> c = fold16(p);
    if (e < all && slot < (uint64_t)all) reinterpret_cast<float4 *>(f.coef)[slot] = make_float4(c.ab, c.a, c.b, c.one);
    if (f.probs == nullptr) return;
    wave_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4 *>(mine + lane * kFoldPitch + 4 * i) = make_float4(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]);
    wave_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int from = 16 * i + (lane >> 2);
        const float4 v = *reinterpret_cast<const float4 *>(mine + from * kFoldPitch + 4 * (lane & 3));
        if (e0 + from < all) store_vec<STREAM>(reinterpret_cast<f32x4u *>(f.probs + (e0 + from) * 16) + (lane & 3), f32x4u{v.x, v.y, v.z, v.w});
    }
}

// ---- gradients of the logits --------------------------------------------------------------------------------------------
// Gradients of the logits, four lanes per neuron of the three layers in order, four gates each: whole lines of probabilities and gradients.  slot:
// where the neuron's four sums are (root * 7 + gate of the tree).  A layer whose gradient is not wanted has a null pointer.
// (A thread per neuron left 64 bytes between the accesses of two lanes: 655360 roots 170 -> 162 us, 10240 5.4 -> 4.9; nontemporal with it, 261.)
struct TreeGrads {
    float *g[3];
    int64_t end[3];       // neurons of the first one, two, three layers
};
struct TreeSums {
    TreeGrads gr;
    const float *probs, *sums;
    const int32_t *slot;
    int64_t slots;
};
template <bool STREAM>
__device__ __forceinline__ void tree_logit_grad(const TreeSums &t, int64_t block)
{
    const TreeGrads &gr = t.gr;
    const float *__restrict__ probs = t.probs, *__restrict__ sums = t.sums;
    const int32_t *__restrict__ slot = t.slot;
    const int64_t slots = t.slots, e = (block * 256 + threadIdx.x) >> 2;
    const int part = threadIdx.x & 3;
    if (e >= gr.end[2]) return;                                       // (four lanes together)
    const int layer = e < gr.end[0] ? 0 : (e < gr.end[1] ? 1 : 2);
    const int64_t n = e - (layer ? gr.end[layer - 1] : 0);
    if (gr.g[layer] == nullptr) return;
    const f32x4u p = load_vec<STREAM>(reinterpret_cast<const f32x4u *>(probs + e * 16) + part);
    const float4 s = reinterpret_cast<const float4 *>(sums)[min((uint64_t)(uint32_t)slot[e], (uint64_t)slots - 1)];
    float gi[4], dot = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) gi[i] = coef_transpose_row<float>(4 * part + i, s.x, s.y, s.z, s.w);
    // the sum over the 16 gates in their order: every lane goes on from what the lanes of the gates before have
    auto go_on = [&](float d) {
#pragma unroll
        for (int i = 0; i < 4; ++i) d = fma_t(p[i], gi[i], d);
        return d;
    };
    dot = dpp_zero<0x00, 0xF>(go_on(dot));
    dot = dpp_zero<0x55, 0xF>(go_on(dot));
    dot = dpp_zero<0xAA, 0xF>(go_on(dot));
    dot = dpp_zero<0xFF, 0xF>(go_on(dot));
    store_vec<STREAM>(reinterpret_cast<f32x4u *>(gr.g[layer] + n * 16) + part,
                      f32x4u{p[0] * (gi[0] - dot), p[1] * (gi[1] - dot), p[2] * (gi[2] - dot), p[3] * (gi[3] - dot)});
}

}  // namespace

int clg_check_tree(const char *name, int64_t in_dim, int64_t roots, int64_t k);
