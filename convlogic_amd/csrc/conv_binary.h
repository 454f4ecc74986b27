// The first and the last launch of the block on 0/1 inputs (conv_binary.hip), as what a workgroup of 256 threads does: a launch of their own, or part
// of one for all layers of a network (net_step.hip).
#pragma once

#include "conv_tile.h"

// blocks [0, C): kernel c -- softmax / fold, the 256-entry table, the derivative tables, tap descriptors
// blocks [C, C + list_blocks): per input channel, the kernels that read it (increasing order) with their tap masks
// blocks from pack0 on: the image as bit rows, and the check that it is binary
struct PrepArgs {
    const float *x, *w;
    const int32_t *sel;
    uint32_t *bits;
    float *lut, *probs, *folded, *ftab;
    int32_t *tapinfo, *xtap, *count, *hits;
    int32_t *bad;            // set to 1 when some x is neither 0 nor 1 (may be host memory the device can write)
    int w_logits, list_blocks, pack0, RP, prs;
    FastDiv d_h, d_cinh;
};

namespace {

constexpr int kFtab = 160;          // per kernel: F1[2][16], F2[8][16]

// ---- set-up launch ------------------------------------------------------------------------------------------------
// block of `blocks`
__device__ __forceinline__ void bin_prepare(const PrepArgs &a, const Geom &g, int block, int blocks)
{
    const int tid = threadIdx.x, lane = tid & 63;
    if (block < g.c) {
        __shared__ float cf[28];
        const int c = block;
        if (tid < 7) {
            const int64_t q = (int64_t)c * 7 + tid;
            float pr[16];
            if (a.w_logits) {
                softmax16(a.w + q * 16, pr);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) pr[i] = a.w[q * 16 + i];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) a.probs[q * 16 + i] = pr[i];
            const Coef<float> k = fold16(pr);
            cf[4 * tid] = k.ab, cf[4 * tid + 1] = k.a, cf[4 * tid + 2] = k.b, cf[4 * tid + 3] = k.one;
            a.folded[q * 4] = k.ab, a.folded[q * 4 + 1] = k.a, a.folded[q * 4 + 2] = k.b, a.folded[q * 4 + 3] = k.one;
        }
        if (tid >= 64 && tid < 72) {
            const int t = tid - 64;
            const Tap tp = unpack_tap(a.sel[(int64_t)c * 8 + t], tap_limit(g));   // (forced into the layer's ranges)
            const int sh = tp.rx - g.pw;                              // tap word = row word >> sh (<< -sh)
            a.tapinfo[c * 8 + t] = ((tp.ch * a.RP + tp.ry) << 16) | ((sh < 0 ? -sh : 0) << 8) | (sh > 0 ? sh : 0);
            a.xtap[c * 8 + t] = tp.ry * a.prs + tp.rx;                 // offset of the tap in a gradient plane
        }
        __syncthreads();
        Tree<float> tr;
#pragma unroll
        for (int q = 0; q < 7; ++q) tr.g[q] = Coef<float>{cf[4 * q], cf[4 * q + 1], cf[4 * q + 2], cf[4 * q + 3]};
        float tap[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) tap[i] = (float)((tid >> i) & 1);
        const TreeVals<float> tv = eval_tree(tr, tap);
        a.lut[(int64_t)c * 256 + tid] = tv.root;
        if (tid < kFtab) {
            // F1[q][nib of the OTHER side] = d root / d mid_q; F2[i][own nibble] = d mid / d leaf * d leaf / d tap_i
            float v;
            const int nib = tid & 15;
            float nb[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) nb[i] = (float)((nib >> i) & 1);
            auto coef = [&](int q) { return Coef<float>{cf[4 * q], cf[4 * q + 1], cf[4 * q + 2], cf[4 * q + 3]}; };   // (run-time gate index)
            if (tid < 32) {
                const int q = tid >> 4;                              // F1[q] is indexed by the nibble of side 1 - q
                const int o = 1 - q;
                const float l0 = gate(coef(2 * o), nb[0], nb[1]), l1 = gate(coef(2 * o + 1), nb[2], nb[3]);
                const float mo = gate(coef(4 + o), l0, l1);
                v = q == 0 ? gate_da(tr.g[6], mo) : gate_db(tr.g[6], mo);
            } else {
                const int i = (tid - 32) >> 4;                       // tap 0..7
                const int p = i >> 1, q = p >> 1, pl = p & 1, s = i & 1;   // leaf, side, leaf inside the side, operand
                const float pa = pl ? nb[0] : nb[2], pb = pl ? nb[1] : nb[3];            // taps of the partner leaf
                const float oa = pl ? nb[2] : nb[0], ob = pl ? nb[3] : nb[1];            // taps of the own leaf
                const float partner = gate(coef(2 * q + (1 - pl)), pa, pb);
                const float dm = pl == 0 ? gate_da(coef(4 + q), partner) : gate_db(coef(4 + q), partner);
                const float dl = s == 0 ? gate_da(coef(p), ob) : gate_db(coef(p), oa);
                v = dm * dl;
            }
            a.ftab[(int64_t)c * kFtab + tid] = v;
        }
        return;
    }
    if (block < g.c + a.list_blocks) {
        // one wavefront per input channel: lanes test 64 kernels at a time, matches are appended in order
        const int ch = uniform((block - g.c) * 4 + (tid >> 6));
        if (ch >= g.cin) return;
        int n = 0;
        for (int c0 = 0; c0 < g.c; c0 += kWave) {
            const int c = c0 + lane;
            int mask = 0;
            if (c < g.c) {
#pragma unroll
                for (int t = 0; t < 8; ++t) mask |= (tap_channel(a.sel[c * 8 + t], g.cin) == ch) << t;
            }
            const uint64_t vote = __ballot(mask != 0);
            if (mask) {
                const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(vote >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)vote, 0));
                a.hits[(int64_t)ch * g.c + n + before] = c | (mask << 16);
            }
            n += __popcll(vote);
        }
        if (lane == 0) {
            a.count[2 * ch] = n;
            a.count[2 * ch + 1] = ch * g.c;
        }
        return;
    }
    // bit rows: a wavefront packs two image rows per step (lane = row of the pair * 32 + column)
    const int64_t rows = (int64_t)g.n * g.cin * g.h;
    const int r = lane >> 5, col = lane & 31;
    const int64_t wave0 = (int64_t)(block - a.pack0) * 4 + (tid >> 6), nwaves = (int64_t)(blocks - a.pack0) * 4;
    bool bad = false;
    for (int64_t pair0 = wave0; pair0 * 2 < rows; pair0 += 4 * nwaves) {   // four loads in flight
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t row = (pair0 + u * nwaves) * 2 + r;
            v[u] = row < rows && col < g.w ? a.x[row * g.w + col] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t row = (pair0 + u * nwaves) * 2 + r;
            bad = bad || (v[u] != 0.f && v[u] != 1.f);
            const uint64_t m = __ballot(v[u] != 0.f);
            if (col == 0 && row < rows) {
                const uint32_t plane = fdiv((uint32_t)row, a.d_h), iy = (uint32_t)row - plane * (uint32_t)g.h;
                uint32_t *dst = a.bits + (int64_t)plane * a.RP;
                dst[iy + g.ph] = (uint32_t)(r ? m >> 32 : m);
                if (iy == 0)
                    for (int k = 0; k < g.ph; ++k) dst[k] = 0;
                if (iy == (uint32_t)g.h - 1)
                    for (int k = 0; k < g.ph; ++k) dst[g.ph + g.h + k] = 0;
            }
        }
    }
    if (bad) *a.bad = 1;
}

// ---- weight gradient from the histograms ----------------------------------------------------------------------------
// A workgroup of 256 threads per kernel: thread t weights the derivative of the tree at tap byte t with the histogram; the 28 coefficient
// sums are added over t in a fixed order, then the transform to the 16 gates (and the softmax backward for logits).
struct BinSums {
    const float *hpart, *folded, *probs;                             // probs (or null): the gradient is that of the logits
    float *gw;
    int parts;
};
__device__ __forceinline__ void bin_sums(const BinSums &s, int c)
{
    const float *__restrict__ hpart = s.hpart, *__restrict__ folded = s.folded, *__restrict__ probs = s.probs;
    float *__restrict__ gw = s.gw;
    const int parts = s.parts;
    __shared__ float sums[28];
    const int t = threadIdx.x;
    float H = 0.f;
    const float *hp = hpart + (int64_t)c * parts * 256 + t;
    int k = 0;
    for (; k + 8 <= parts; k += 8) {                                  // eight loads in flight, added in the order of one by one
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = hp[(k + u) * 256];
#pragma unroll
        for (int u = 0; u < 8; ++u) H += v[u];
    }
    for (; k < parts; ++k) H += hp[k * 256];
    Tree<float> tr;
    const float *fc = folded + (int64_t)c * 28;
#pragma unroll
    for (int q = 0; q < 7; ++q) tr.g[q] = Coef<float>{fc[4 * q], fc[4 * q + 1], fc[4 * q + 2], fc[4 * q + 3]};
    float tap[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) tap[i] = (float)((t >> i) & 1);
    const TreeVals<float> tv = eval_tree(tr, tap);
    float acc[28];
    auto put = [&](int q, float g, float a, float b) {
        const float ga = g * a;
        acc[4 * q] = ga * b, acc[4 * q + 1] = ga, acc[4 * q + 2] = g * b, acc[4 * q + 3] = g;
    };
    put(6, H, tv.mid[0], tv.mid[1]);
    const float g_m0 = H * gate_da(tr.g[6], tv.mid[1]), g_m1 = H * gate_db(tr.g[6], tv.mid[0]);
    put(4, g_m0, tv.leaf[0], tv.leaf[1]);
    put(5, g_m1, tv.leaf[2], tv.leaf[3]);
    const float g_l0 = g_m0 * gate_da(tr.g[4], tv.leaf[1]), g_l1 = g_m0 * gate_db(tr.g[4], tv.leaf[0]);
    const float g_l2 = g_m1 * gate_da(tr.g[5], tv.leaf[3]), g_l3 = g_m1 * gate_db(tr.g[5], tv.leaf[2]);
    put(0, g_l0, tap[0], tap[1]);
    put(1, g_l1, tap[2], tap[3]);
    put(2, g_l2, tap[4], tap[5]);
    put(3, g_l3, tap[6], tap[7]);
    block_sum_store<float, 28, 256>(acc, sums);
    __syncthreads();
    if (t < 112) {
        const int q = t >> 4, i = t & 15;
        float gi = coef_transpose_row<float>(i, sums[4 * q], sums[4 * q + 1], sums[4 * q + 2], sums[4 * q + 3]);
        if (probs != nullptr) gi = softmax16_backward(gi, probs[(int64_t)c * 112 + t]);
        gw[(int64_t)c * 112 + t] = gi;
    }
}

}  // namespace

// What the set-up of a forward call is given, with the call's checks; `blocks` of 256 threads
int clg_bin_prepare_args(const char *name, int dtype, const clg_conv_geom *gg, const void *x, const void *w, const int32_t *selection, void *ctx, bool w_logits,
                         int32_t *not_binary, Geom *g, PrepArgs *a, int *blocks);
