// Weight gradient of the fused float32 conv-logic block from planes that a wavefront stages for itself (conv_pair.h; the forward pass in
// conv_pair.hip has the layout): the tree is recomputed at the arg-max position of a window, lane = pooled cell.
//
// The kernel with lanes along a padded copy of x asks the vector cache for eight addresses per lane and cell, 16 clocks each of the
// one that four SIMDs share: 128 of the 270 clocks it takes per 64 cells.  Here they come as two 16-byte loads of a
// lane.  102 vector instructions per 64 cells bound it from there ([128,4096,8,8] -> 16384: 253 -> 172 us, 81 of them those;
// [128,1024,16,16] -> 4096: 191 -> 162; [256,128,8,8] -> 512: 16.9 -> 13).
// Both gradients (PLANES): the same visit gives the tap gradients, which are added to gradient planes of the wavefront in LDS -- 16 more accesses per
// 64 cells, about three lanes to a bank as the arg-max positions fall -- and go out as the kernel's share of its two channels; a
// second kernel sums the shares of a channel.  Every kernel is evaluated once, where an owner per (sample, channel) evaluates it for
// each of its channels with taps gathered from a padded copy of x, which nobody needs here.  [256,32,16,16] -> 128: 33 + 13 us
// -> 24 (LDS: 490 clocks per 64 cells and CU) + 14 (67 MB from the last-level cache); its bounds stand at backward_planes_wanted.
// With an owner's planes the input gradient was built the same way (own planes resident, the other channel's staged per kernel, gradient planes in LDS) and
// taken back: [128,4096,8,8] -> 16384 620 to 640 us for both gradients against 597 with the kernel that gathers; a chain of scalar loads, staging
// and read-add-write rounds per kernel of a list bounds both.
#include <algorithm>

#include "conv_ops.h"
#include "conv_pair.h"

namespace {

// A pooled cell of a group of samples: where its window begins in LDS, its place in grad_y (in elements, from the group's first sample).
struct PairCell {
    int at;
    uint32_t out, s, py, px;
    bool live;
};
__device__ __forceinline__ PairCell pair_cell(const Geom &g, const PairPlan &p, int row_step, uint32_t u, int cells, int I, int wp)
{
    PairCell r;
    r.live = (int)u < cells;
    const uint32_t uu = r.live ? u : 0;
    r.s = fdiv(uu, p.d_cells);
    const uint32_t cell = uu - r.s * (uint32_t)I;
    r.py = fdiv(cell, p.d_wp), r.px = cell - r.py * (uint32_t)wp;
    r.at = (int)(r.s * p.sample + 2 * r.py * row_step + 2 * r.px);
    r.out = r.s * (uint32_t)(g.c * I) + cell;
    return r;
}

// The 28 sums of a workgroup: those of its wavefronts meet in LDS.
__device__ __forceinline__ void pair_block_sums(const float (&v)[28], float *__restrict__ meet, float *__restrict__ dst, int lane, int wave)
{
    int at;
    const float mine = wave_sums28(v, lane, at);
    __syncthreads();                                                 // (the planes are done with)
    if (at >= 0) meet[wave * 28 + at] = mine;
    __syncthreads();
    if (threadIdx.x < 28) {
        float s = meet[threadIdx.x];
#pragma unroll
        for (int w = 1; w < kPairWaves; ++w) s += meet[w * 28 + threadIdx.x];
        dst[threadIdx.x] = s;
    }
}

// A wavefront owns a kernel and every 4 nb-th group of samples; the planes, grad_y and arg-max codes of the next
// group are in flight while the current one is evaluated, and the 28 sums (7 gates x (ab, a, b, 1)) stay in registers over all of
// them.  partial [c][nb][28], added in order by reduce_coef_partials.
// PLANES: the tap gradients as well, added to gradient planes beside the staged ones and written to planes [c][2][n][h w]: those of a kernel's
// first and second channel, for plane_sums_kernel.  (Of a kernel with taps in more than two channels nothing is written.)
template <int NL, int RS, bool ROWS, bool ONE, bool PLANES, bool STREAM>
__global__ __launch_bounds__(kPairWaves *kWave) void convblock_backward_w_pair_kernel(const float *__restrict__ gy, const float *__restrict__ x,
                                                                                    const float *__restrict__ folded, const int32_t *__restrict__ sel,
                                                                                    const uint8_t *__restrict__ argmax, float *__restrict__ partial,
                                                                                    float *__restrict__ planes, Geom g, PairPlan p, int nb)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    float *mine = reinterpret_cast<float *>(smem) + wave * p.wave_elems, *grads = mine + kPairWaves * p.wave_elems;
    for (int i = lane * 4; i < p.wave_elems; i += kWave * 4) *reinterpret_cast<u32x4 *>(mine + i) = (u32x4)0u;
    // workgroups that read the same samples (one part, every kernel) follow each other on one XCD and share its L2
    const unsigned logical = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int bx = uniform((int)(logical / (unsigned)g.c)), c = uniform((int)logical) - bx * g.c;
    const int wp = g.wo >> 1, I = (g.ho >> 1) * wp, cells = p.G * I, blocks = ONE ? 1 : (cells + kWave - 1) / kWave;
    const int row_step = RS ? RS : p.rs;
    const float *fc = folded + (int64_t)c * 28;
    Tree<float> tr;
#pragma unroll
    for (int q = 0; q < 7; ++q) tr.g[q] = Coef<float>{fc[4 * q], fc[4 * q + 1], fc[4 * q + 2], fc[4 * q + 3]};
    int ch0, ch1, off[8];
    bool wide = false;                                               // (taps in more than two channels, by a caller-made selection)
    {
        Tap tp[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) tp[t] = unpack_tap(sel[c * 8 + t], tap_limit(g));
        ch0 = ch1 = tp[0].ch;
#pragma unroll
        for (int t = 7; t >= 1; --t) ch1 = tp[t].ch != ch0 ? tp[t].ch : ch1;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            wide |= tp[t].ch != ch0 && tp[t].ch != ch1;
            off[t] = uniform((tp[t].ch != ch0 ? p.plane : 0) + tp[t].ry * row_step + tp[t].rx + p.lead - p.pw);
        }
    }
    const uint32_t plane_bytes = (uint32_t)(g.h * g.w) * 4u, o0 = (uint32_t)ch0 * plane_bytes, d = (uint32_t)ch1 * plane_bytes - o0;
    PairPieces<float, NL, ROWS, false> in;
    in.place(g, p, row_step, p.G, lane);
    // where a lane's pieces of the gradient planes go, from the group's first sample of the kernel's first channel
    int out_at[PLANES ? NL : 1], out_sample[PLANES ? NL : 1];
    if constexpr (PLANES) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t v = lane + i * kWave, pl = fdiv(v, p.d_pieces), e = (v - pl * p.pieces) * 4;
            out_sample[i] = (int)(pl >> 1);
            out_at[i] = (int)(((pl & 1) * (uint32_t)g.n + (pl >> 1)) * (uint32_t)(g.h * g.w) + e);
        }
    }
    const PairCell first = pair_cell(g, p, row_step, lane, cells, I, wp);
    float acc[28];
#pragma unroll
    for (int k = 0; k < 28; ++k) acc[k] = 0.f;
    // the last group is moved back so that it is full; what it shares with the one before does not count again
    const int step = kPairWaves * nb, sample = g.cin * g.h * g.w;
    auto start_of = [&](int q) { return min(q * p.G, g.n - p.G); };
    auto fetch = [&](int q) { in.fetch(x + (int64_t)start_of(q) * sample, o0, d); };
    int code = 0;
    float gout = 0.f;
    auto load_cell = [&](int q, const PairCell &cell) {
        const int64_t row = ((int64_t)start_of(q) * g.c + c) * I;
        code = argmax[row + cell.out];
        gout = gy[row + cell.out];
    };
    int q = bx * kPairWaves + wave;
    if (q < p.groups) {
        fetch(q);
        load_cell(q, first);
    }
    for (; q < p.groups; q += step) {
        wave_fence();
        in.store(mine);
        if constexpr (PLANES)
            for (int i = lane * 4; i < p.wave_elems; i += kWave * 4) *reinterpret_cast<u32x4 *>(grads + i) = (u32x4)0u;
        wave_fence();
        const int qn = q + step, n0 = start_of(q);
        if (qn < p.groups) fetch(qn);
        for (int b = 0; b < blocks; ++b) {
            const PairCell cell = ONE ? first : pair_cell(g, p, row_step, b * kWave + lane, cells, I, wp);
            const int code_now = code;
            const float gq = gout;
            if (b + 1 < blocks) load_cell(q, pair_cell(g, p, row_step, (b + 1) * kWave + lane, cells, I, wp));
            else if (qn < p.groups) load_cell(qn, first);
            if (!(cell.live && n0 + (int)cell.s >= q * p.G)) continue;
            float tap[8];
            if (!wide) {
                const float *at = mine + cell.at + (code_now >> 1) * row_step + (code_now & 1);
#pragma unroll
                for (int t = 0; t < 8; ++t) tap[t] = at[off[t]];
            } else {
                const float *xn = x + (int64_t)(n0 + (int)cell.s) * sample;
#pragma unroll
                for (int t = 0; t < 8; ++t) 
                    tap[t] = read_tap(xn, g, unpack_tap(sel[c * 8 + t], tap_limit(g)), (int)(2 * cell.py) + (code_now >> 1), (int)(2 * cell.px) + (code_now & 1));
            }
            const TreeVals<float> tv = eval_tree(tr, tap);
            auto add = [&](int k, float gk, float a, float b2) {
                const float ga = gk * a;
                acc[4 * k] = fma_t(ga, b2, acc[4 * k]);
                acc[4 * k + 1] += ga;
                acc[4 * k + 2] = fma_t(gk, b2, acc[4 * k + 2]);
                acc[4 * k + 3] += gk;
            };
            add(6, gq, tv.mid[0], tv.mid[1]);
            const float gm[2] = {gq * gate_da(tr.g[6], tv.mid[1]), gq * gate_db(tr.g[6], tv.mid[0])};
            float gl[4];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const float la = tv.leaf[2 * m], lb = tv.leaf[2 * m + 1];
                add(4 + m, gm[m], la, lb);
                gl[2 * m] = gm[m] * gate_da(tr.g[4 + m], lb);
                gl[2 * m + 1] = gm[m] * gate_db(tr.g[4 + m], la);
                add(2 * m, gl[2 * m], tap[4 * m], tap[4 * m + 1]);
                add(2 * m + 1, gl[2 * m + 1], tap[4 * m + 2], tap[4 * m + 3]);
            }
            if constexpr (PLANES) {
                if (wide) continue;
                // for one tap the targets of all lanes are distinct elements; taps are applied one after the other
                float *at = grads + cell.at + (code_now >> 1) * row_step + (code_now & 1);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const Coef<float> &k = tr.g[t >> 1];
                    at[off[t]] += gl[t >> 1] * (t & 1 ? gate_db(k, tap[t ^ 1]) : gate_da(k, tap[t ^ 1]));
                    wave_fence();
                }
            }
        }
        if constexpr (PLANES) {
            wave_fence();
            float *dst = planes + (int64_t)(2 * c) * g.n * (g.h * g.w) + (int64_t)n0 * (g.h * g.w);
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                u32x4 v;
                if constexpr (ROWS) {
                    v = *reinterpret_cast<const u32x4 *>(grads + in.to[i][0]);
                } else {
                    float part[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) part[j] = grads[in.to[i][j]];
                    __builtin_memcpy(&v, part, 16);
                }
                if (!wide && out_sample[i] < p.G && n0 + out_sample[i] >= q * p.G) store_vec<STREAM>(reinterpret_cast<u32x4 *>(dst + out_at[i]), v);
            }
        }
    }
    pair_block_sums(acc, reinterpret_cast<float *>(smem), partial + ((int64_t)c * nb + bx) * 28, lane, wave);
}

// gx = the sum of a channel's gradient planes, in the order of the kernels: four consecutive elements per thread, `parts` workgroups per channel.
// A kernel that wrote none (its list entry says so) is evaluated here, element by element: slow (taps_are_wide in conv_block.hip), and so only
// in plans that were made, or are read, by a recording.
template <bool STREAM>
__global__ __launch_bounds__(256) void plane_sums_kernel(const float *__restrict__ planes, const int32_t *__restrict__ count, const int32_t *__restrict__ hits,
                                                       const float *__restrict__ gy, const float *__restrict__ x, const float *__restrict__ folded,
                                                       const int32_t *__restrict__ sel, const uint8_t *__restrict__ argmax, float *__restrict__ gx, Geom g,
                                                       unsigned parts, FastDiv d_parts, FastDiv d_hw, FastDiv d_w)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    const unsigned b = xcd_contiguous_block(blockIdx.x, gridDim.x), ch = fdiv(b, d_parts), part = b - ch * parts;
    const uint32_t hw = (uint32_t)(g.h * g.w), plane = (uint32_t)g.n * hw, e = (part * 256 + threadIdx.x) * 4;
    if (e >= plane) return;
    const uint32_t n = fdiv(e, d_hw), in = e - n * hw;
    const int nhits = count[2 * ch];
    const int32_t *hit = hits + count[2 * ch + 1];
    const float *from = planes + e;
    f32x4 sum = 0.f;
    auto piece = [&](int ent) {
        return load_vec<STREAM>(reinterpret_cast<const f32x4 *>(from + (int64_t)(2 * (ent & 0xFFFF) + ((ent >> 16) & 1 ? 0 : 1)) * plane));
    };
    int k = 0;
    while (k < nhits) {
        int ent[8];
        const int some = min(8, nhits - k);
        bool wide = false;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            ent[i] = hit[k + min(i, some - 1)];
            wide |= (ent[i] & kHitWide) != 0;
        }
        if (!wide && some == 8) {
            f32x4 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = piece(ent[i]);
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += v[i];
            k += 8;
            continue;
        }
        if (!wide) {
            for (int i = 0; i < some; ++i) sum += piece(hit[k + i]);
            k += some;
            continue;
        }
        const int one = hit[k++];
        if ((one & kHitWide) == 0) {
            sum += piece(one);
            continue;
        }
        const int c = one & 0xFFFF;
        const float *fc = folded + (int64_t)c * 28, *xn = x + (int64_t)n * g.cin * hw;
        Tree<float> tr;
#pragma unroll
        for (int q = 0; q < 7; ++q) tr.g[q] = Coef<float>{fc[4 * q], fc[4 * q + 1], fc[4 * q + 2], fc[4 * q + 3]};
        const int wp = g.wo >> 1, I = (g.ho >> 1) * wp;
#pragma unroll 1
        for (int u = 0; u < 4; ++u) {
            const uint32_t iy = fdiv(in + u, d_w), ix = in + u - iy * (uint32_t)g.w;
            float add = 0.f;
#pragma unroll 1
            for (int t = 0; t < 8; ++t) {
                if (!((one >> (16 + t)) & 1)) continue;
                const Tap tp = unpack_tap(sel[c * 8 + t], tap_limit(g));
                const int oy = (int)iy + g.ph - tp.ry, ox = (int)ix + g.pw - tp.rx;
                if (oy < 0 || ox < 0 || oy >= g.ho || ox >= g.wo) continue;
                const int64_t cell = ((int64_t)n * g.c + c) * I + (oy >> 1) * wp + (ox >> 1);
                if (argmax[cell] != ((oy & 1) * 2 + (ox & 1))) continue;
                float tap[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) tap[q] = read_tap(xn, g, unpack_tap(sel[c * 8 + q], tap_limit(g)), oy, ox);
                const TreeVals<float> v = eval_tree(tr, tap);
                const float gm[2] = {gy[cell] * gate_da(tr.g[6], v.mid[1]), gy[cell] * gate_db(tr.g[6], v.mid[0])};
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int l = q >> 1, m = l >> 1;
                    const float gl = gm[m] * (l & 1 ? gate_db(tr.g[4 + m], v.leaf[l ^ 1]) : gate_da(tr.g[4 + m], v.leaf[l ^ 1]));
                    const float d = gl * (q & 1 ? gate_db(tr.g[l], tap[q ^ 1]) : gate_da(tr.g[l], tap[q ^ 1]));
                    add += q == t ? d : 0.f;
                }
            }
            sum[u] += add;
        }
    }
    *reinterpret_cast<f32x4_any *>(gx + ((int64_t)n * g.cin + ch) * hw + in) = sum;
}

}  // namespace

template <int NL, int RS, bool ROWS, bool ONE, bool PLANES, bool STREAM>
static int launch_pair_w(const Geom &g, const PairPlan &p, int nb, const float *gy, const float *x, const float *folded, const int32_t *sel,
                         const uint8_t *argmax, float *partial, float *planes, hipStream_t st, const char *name)
{
    const size_t lds = (size_t)(PLANES ? 2 : 1) * kPairWaves * p.wave_elems * 4;
    if (int e = allow_lds(convblock_backward_w_pair_kernel<NL, RS, ROWS, ONE, PLANES, STREAM>, lds, name)) return e;
    hipLaunchKernelGGL((convblock_backward_w_pair_kernel<NL, RS, ROWS, ONE, PLANES, STREAM>), dim3((unsigned)(g.c * nb)), dim3(kPairWaves *kWave), lds, st, gy, x,
                       folded, sel, argmax, partial, planes, g, p, nb);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}
template <int NL, bool PLANES, bool STREAM>
static int launch_pair_w_nl(const Geom &g, const PairPlan &p, int nb, const float *gy, const float *x, const float *folded, const int32_t *sel,
                            const uint8_t *argmax, float *partial, float *planes, hipStream_t st, const char *name)
{
    const bool one = p.G * (g.ho / 2) * (g.wo / 2) <= kWave;
    auto *launch = launch_pair_w<NL, 0, true, false, PLANES, STREAM>;
    if (g.w % 4 != 0) launch = one ? launch_pair_w<NL, 0, false, true, PLANES, STREAM> : launch_pair_w<NL, 0, false, false, PLANES, STREAM>;
    else if (one)
        launch = p.rs == 20 ? launch_pair_w<NL, 20, true, true, PLANES, STREAM>
                            : (p.rs == 12 ? launch_pair_w<NL, 12, true, true, PLANES, STREAM> : launch_pair_w<NL, 0, true, true, PLANES, STREAM>);
    return launch(g, p, nb, gy, x, folded, sel, argmax, partial, planes, st, name);
}

// Workgroups per kernel.  A lane adds one term per block of cells it visits to the same sum, so there are as many as keep that chain no longer
// than in the kernel of the padded copy, which gives a thread 8 terms, 16 from 65536 cells of a kernel on, in at most 64 parts (one
// part for each of 4096 kernels had 32 terms and an error 1.2 times as large at [128,1024,16,16] -> 4096, 157 us where four
// take 162; 1.5 times at [1000,40,8,8] -> 2000).  A group's blocks of cells stay together, so a lane takes whole groups.  More workgroups up to
// 1024 in all ([256,32,16,16] -> 128, both gradients: 52.7 us without this kernel, 46.9 with 8 per kernel, 50.8 with
// 16, 63 with 2), as long as a wavefront has four blocks of cells for its 28 reductions.
constexpr int kMaxParts = 64;                                        // (what the scratch holds)
struct Chain {
    int64_t blocks, limit;                                           // blocks of 64 cells of a group; terms of the other kernel
};
static Chain chain_of(const Geom &g, const PairPlan &p)
{
    const int64_t I = (int64_t)(g.ho / 2) * (g.wo / 2), cells = I * g.n, terms = cells >= 65536 ? 16 : 8;
    const int64_t parts = std::min<int64_t>(kMaxParts, clg_ceil_div(cells, 256 * terms));
    return {clg_ceil_div(p.G * I, kWave), clg_ceil_div(cells, 256 * parts)};
}
int clg_pair_grad_w_parts(const Geom &g, const PairPlan &p)
{
    const Chain ch = chain_of(g, p);
    const int64_t groups = std::max<int64_t>(1, ch.limit / ch.blocks);      // of a wavefront
    const int64_t fill = std::min<int64_t>(clg_ceil_div(1024, g.c), p.groups * ch.blocks / (4 * kPairWaves));
    return (int)std::max<int64_t>(1, std::min<int64_t>(kMaxParts, std::max(fill, clg_ceil_div(p.groups, groups * kPairWaves))));
}
// With the planes a CU holds four workgroups, or what LDS has room for, and a launch of a little more than all CUs hold takes twice as long ([200,48,16,16] ->
// 192 in 7 parts: 1344 workgroups, 45 us; step of the k = 48
// CIFAR network 362 -> 356 us with 10).  Of the numbers of parts from the shortest chain's on, the one with the fewest
// rounds of the launch times groups of a wavefront, and as long as two for what a workgroup does before and after.
static int planes_parts(const Geom &g, const PairPlan &p)
{
    const Chain ch = chain_of(g, p);
    const int64_t groups = std::max<int64_t>(1, ch.limit / ch.blocks), least = std::min<int64_t>(kMaxParts, clg_ceil_div(p.groups, groups * kPairWaves));
    const int64_t slots = 256 * std::max<int64_t>(1, std::min<int64_t>(4, kLdsLimit / (2ll * kPairWaves * p.wave_elems * 4)));
    int64_t best = least, cost = INT64_MAX;
    for (int64_t nb = least; nb <= std::min<int64_t>(kMaxParts, std::max(least, clg_ceil_div(p.groups, (int64_t)kPairWaves))); ++nb) {
        const int64_t now = clg_ceil_div(g.c * nb, slots) * (clg_ceil_div(p.groups, nb * kPairWaves) * ch.blocks + 2);
        if (now < cost) best = nb, cost = now;
    }
    return (int)best;
}
// Lanes that idle in every block of cells can make the chain longer than the other kernel's even with the most parts.
bool clg_pair_grad_w_wanted(const Geom &g, const PairPlan &p)
{
    const Chain ch = chain_of(g, p);
    return clg_ceil_div(p.groups, (int64_t)clg_pair_grad_w_parts(g, p) * kPairWaves) * ch.blocks <= std::max(ch.limit, ch.blocks);
}

int clg_pair_grad_w(const Geom &g, const PairPlan &p, int nb, const float *gy, const float *x, const float *folded, const int32_t *sel,
                    const uint8_t *argmax, float *partial, hipStream_t st, const char *name)
{
    if (p.loads <= 2) return launch_pair_w_nl<2, false, false>(g, p, nb, gy, x, folded, sel, argmax, partial, nullptr, st, name);
    if (p.loads <= 4) return launch_pair_w_nl<4, false, false>(g, p, nb, gy, x, folded, sel, argmax, partial, nullptr, st, name);
    return launch_pair_w_nl<8, false, false>(g, p, nb, gy, x, folded, sel, argmax, partial, nullptr, st, name);
}

bool clg_pair_planes_fit(const Geom &g, const PairPlan &p)
{
    return p.loads <= 4 && 2ll * kPairWaves * p.wave_elems * 4 <= 64 * 1024 && 2ll * g.n * g.h * g.w < (1ll << 30) && (int64_t)g.c * g.n < (1ll << 40) &&
           clg_ceil_div((int64_t)g.n * g.h * g.w, 1024) * g.cin < (1ll << 24);
}
size_t clg_pair_planes_bytes(const Geom &g) { return (size_t)2 * g.c * g.n * g.h * g.w * 4; }

int clg_pair_grads(const Geom &g, const PairPlan &p, int *parts_of_sums, const float *gy, const float *x, const float *folded, const int32_t *sel, const uint8_t *argmax,
                   const int32_t *count, const int32_t *hits, float *planes, float *partial, float *gx, hipStream_t st, const char *name)
{
    const int nb = *parts_of_sums = planes_parts(g, p);
    // Past the caches where the planes, x and its gradient together are more than the last-level cache keeps between the two kernels: forward and backward, us
    // through the caches and past them, [275,144,20,20] -> 144, 121 MB of planes and 2 x 63, 139 and 131, [268,233,10,10] -> 932, 191 and 2 x 25, 198 and 189,
    // [126,381,14,14] -> 1143, 215 and 2 x 38, 236 and 210; [297,706,8,8] -> 706, 102 and 2 x 54, 104 and 111, [209,31,20,20] -> 248, 158 and 2 x 10, 142 and 147.
    const bool stream = clg_past_caches((int64_t)clg_pair_planes_bytes(g) + (int64_t)g.n * g.cin * g.h * g.w * 8, 215);
    auto *launch = p.loads <= 2 ? (stream ? launch_pair_w_nl<2, true, true> : launch_pair_w_nl<2, true, false>)
                                : (stream ? launch_pair_w_nl<4, true, true> : launch_pair_w_nl<4, true, false>);
    if (int e = launch(g, p, nb, gy, x, folded, sel, argmax, partial, planes, st, name)) return e;
    const unsigned parts = (unsigned)clg_ceil_div((int64_t)g.n * g.h * g.w, 1024);
    hipLaunchKernelGGL((stream ? plane_sums_kernel<true> : plane_sums_kernel<false>), dim3(parts * (unsigned)g.cin), dim3(256), 0, st, (const float *)planes,
                       count, hits, gy, x, folded, sel, argmax, gx, g, parts, make_fastdiv(parts), make_fastdiv((uint32_t)(g.h * g.w)),
                       make_fastdiv((uint32_t)g.w));
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}
