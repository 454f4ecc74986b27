// Fused conv-logic block, forward, a wavefront at a time: a kernel's taps lie in at most two input planes, so a wavefront copies the two
// planes of its kernel for the samples of 64 pooled cells into LDS of its own and evaluates the kernel there, lane = pooled
// cell, the four positions of the window in registers.  No image of all channels (which does not fit LDS from some hundred
// channels on), no padded copy of x, no barriers.  Element policies of conv_ops.h: float gates with a max pool and its arg-max code, or
// bitwise gates on 64 samples per word with an OR pool.
//
// The planes arrive as 16-byte pieces, requested while the kernel before is evaluated, and go to LDS with halos that are zeroed once: a row
// is `lead` zeros (16 bytes of them, at least the padding), the w pixels and the zeros behind, even columns and odd ones apart; the
// bottom halo of a plane is the top of the next.  An image of more than 64 cells is staged in bands of whole rows of cells with halo rows of
// their own.  A tap is two offsets added to the lane's position, of a window's first and
// second column; the second row is an immediate offset of the same read.
//
// Bound by LDS and the vector ALU together: per kernel and 64 cells 97 vector instructions of float gates and 16 two-value reads
// ([128,4096,8,8] -> 16384: 240 us, the vector instructions alone 111; the kernel before read its taps from a padded copy, 355 us), 56 + 30 of
// words ([1024,128,8,8] -> 512: 66 us).  With even and odd columns in one row the lanes of a read were two elements apart and met in
// the banks two to four times: 265 and 84 us.  Which shapes come here: pair_is_faster in conv_forward.hip.
#include <algorithm>

#include "conv_ops.h"
#include "conv_pair.h"

int clg_convblock_check(const clg_conv_geom *gg, Geom *g, int dtype, const char *name);

namespace {

// What a launch needs besides x and the selection, in one launch: table, folded coefficients (float gates; the softmax of logits
// first), the zero-padded copy of x that the backward pass reads.
template <typename Ops, typename P, typename T, bool STREAM>
__global__ __launch_bounds__(256) void pair_prepare_kernel(const P *__restrict__ w, const int32_t *__restrict__ sel, T *__restrict__ folded,
                                                         int32_t *__restrict__ table, PairPlan p, Geom g, PadJob<T> pad,
                                                         int pad_block0, int from_logits, T *__restrict__ probs_out)
{
    if ((int)blockIdx.x >= pad_block0) {
        pad_image_elems<STREAM>(pad, blockIdx.x - pad_block0);
        return;
    }
    const int C = g.c;
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if constexpr (!Ops::kOrPool) {
        if (folded != nullptr && q < (int64_t)C * 7) {
            fold_gate<P, T>(w, q, from_logits, probs_out, folded);
        }
    }
    if (q == 0) *reinterpret_cast<Geom *>(table + (int64_t)C * kPairTable) = g;
    if (q < C) {
        pair_table_row(table, sel, q, pair_offsets(p), g);
        if constexpr (Ops::kOrPool) table[q * kPairTable + 2] = (int32_t)tree_code(w + q * 7);
    }
}

template <typename Ops>
__device__ __forceinline__ typename Ops::Params pair_params(const void *__restrict__ folded, const int32_t *__restrict__ row, int c)
{
    if constexpr (Ops::kOrPool) {
        return Ops::unpack((uint32_t)row[2]);
    } else {
        typename Ops::Params pr = Ops::load_global(folded, c);
        pin_addends(pr.tr);
        return pr;
    }
}

// NL: 16-byte pieces per lane.  RS: the row stride where it is known at compile time (else 0).  ROWS: no piece crosses a row.  ONE: the
// cells of a group of samples are at most 64; else, with ROWS, a group is a band of a sample (the launch checks that the plan has bands
// then, and only then), and without, 64 cells after the other.  What a lane needs per kernel is worked out once, and the geometry's
// fields are read again where a kernel's taps are in more than two channels: with them in scalar registers all along the loop spilled
// some.
template <typename Ops, int NL, int RS, bool ROWS, bool ONE>
__global__ __launch_bounds__(kPairWaves *kWave) void convblock_forward_pair_kernel(const typename Ops::Elem *__restrict__ x, const void *__restrict__ folded,
                                                                                 const int32_t *__restrict__ table, const int32_t *__restrict__ sel,
                                                                                 typename Ops::Elem *__restrict__ y, uint8_t *__restrict__ argmax,
                                                                                 Geom g, PairPlan p)
{
    using T = typename Ops::Elem;
    constexpr int PER = 16 / (int)sizeof(T);
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    T *mine = reinterpret_cast<T *>(smem) + wave * p.wave_elems;
    for (int i = lane * PER; i < p.wave_elems; i += kWave * PER) *reinterpret_cast<u32x4 *>(mine + i) = (u32x4)0u;
    // the kernel tiles of a group of samples follow each other on one XCD: its L2 holds their planes
    const unsigned logical = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int grp = uniform((int)fdiv(logical, p.d_tiles)), tile = uniform((int)logical) - grp * p.tiles;
    constexpr bool BAND = ROWS && !ONE;
    const int n0 = BAND ? uniform((int)fdiv(grp, p.d_bands)) : grp * p.G, g_here = BAND ? 1 : min(p.G, g.n - n0);
    const int r0 = BAND ? (grp - n0 * p.bands) * p.band_rows : 0;     // a band's first row of cells
    const int hw = g.h * g.w, wp = g.wo >> 1, I = (g.ho >> 1) * wp;
    const int row_step = RS ? RS : p.rs;
    // the row strides that have an instantiation come with their offset of the odd columns
    const int odd = RS ? (RS / 2 + 1) & ~1 : p.odd;
    PairPieces<T, NL, ROWS, true> in;
    if constexpr (BAND) in.place_band(g, p, row_step, 2 * r0 - g.ph, lane);
    else in.place(g, p, row_step, g_here, lane);
    // cell of this lane: where its window begins in LDS, where its value goes
    struct Cell {
        int at;
        uint32_t out, code, s, py, px;
        bool live;
    };
    auto cell_of = [&](uint32_t u) {
        Cell r;
        r.live = (int)u < (BAND ? min(p.band_rows, (g.ho >> 1) - r0) * wp : g_here * I);
        const uint32_t uu = r.live ? u : 0;
        r.s = BAND ? 0 : fdiv(uu, p.d_cells);
        uint32_t cell = uu - r.s * (uint32_t)I;
        r.py = fdiv(cell, p.d_wp), r.px = cell - r.py * (uint32_t)wp;
        r.at = (int)(r.s * p.sample + 2 * r.py * row_step + r.px);
        if (BAND) {
            r.py += r0;
            cell += r0 * wp;
        }
        r.out = r.s * (uint32_t)p.out_sample + cell * (uint32_t)p.out_cell;
        r.code = r.s * (uint32_t)(g.c * I) + cell;                    // (arg-max codes stay sample by sample)
        return r;
    };
    const T *xg = x + (int64_t)n0 * g.cin * hw;
    T *yg = y + (int64_t)n0 * p.out_sample;
    uint8_t *ag = argmax + (int64_t)n0 * g.c * I;
    const int kernel_cells = I * p.out_cell;
    const int blocks = ONE || BAND ? 1 : (g_here * I + kWave - 1) / kWave;
    const uint32_t plane_bytes = (uint32_t)hw * (uint32_t)sizeof(T);
    auto fetch = [&](int c) {
        const int32_t *row = table + c * kPairTable;
        const uint32_t o0 = (uint32_t)row[0] * plane_bytes;
        in.fetch(xg, o0, (uint32_t)max(row[1], 0) * plane_bytes - o0);
    };
    const int c_end = min(g.c, (tile + 1) * p.ct);
    int c = tile * p.ct + wave;
    if (c >= c_end) return;
    fetch(c);
    const Cell first = cell_of(lane);
    for (;;) {
        const int32_t *row = table + c * kPairTable;
        wave_fence();
        in.store(mine, odd);
        wave_fence();
        const typename Ops::Params pr = pair_params<Ops>(folded, row, c);
        int off[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) off[t] = row[4 + t];
        const bool wide = row[1] < 0;
        const int cn = c + kPairWaves;
        if (cn < c_end) fetch(cn);                                    // in flight while this kernel is evaluated
        for (int b = 0; b < blocks; ++b) {
            const Cell cell = ONE || BAND ? first : cell_of(b * kWave + lane);
            T r[4];
            if (!wide) {
                const T *at = mine + cell.at;
                Ops::root4(pr, [&](int t, T (&v)[4]) {
                    const T *q = at + (off[t] & 0xFFFF), *q1 = at + ((uint32_t)off[t] >> 16);
                    v[0] = q[0];
                    v[1] = q1[0];
                    v[2] = q[row_step];
                    v[3] = q1[row_step];
                }, r);
            } else {
                // taps in more than two channels (caller-made selection): from global memory, a position at a time
                const Geom &full = *reinterpret_cast<const Geom *>(table + g.c * kPairTable);
                const T *xn = xg + (int64_t)cell.s * full.cin * full.h * full.w;
#pragma unroll 1
                for (int k = 0; k < 4; ++k) {
                    T v[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        v[t] = read_tap(xn, full, unpack_tap(sel[c * 8 + t], tap_limit(full)), (int)(2 * cell.py) + (k >> 1), (int)(2 * cell.px) + (k & 1));
                    const T rk = Ops::root(pr, v);
                    r[0] = k == 0 ? rk : r[0], r[1] = k == 1 ? rk : r[1], r[2] = k == 2 ? rk : r[2], r[3] = k == 3 ? rk : r[3];
                }
            }
            int code;
            const T best = Ops::pool4(pr, r, code);
            if (cell.live) {
                reinterpret_cast<T *>(reinterpret_cast<char *>(yg + (int64_t)c * kernel_cells) + (size_t)(cell.out * (uint32_t)sizeof(T)))[0] = best;
                if constexpr (!Ops::kOrPool) (ag + (int64_t)c * I)[cell.code] = (uint8_t)code;
            }
        }
        if (cn >= c_end) return;
        c = cn;
    }
}

template <typename Ops, int NL, int RS, bool ROWS, bool ONE>
int launch_pair_one(const Geom &g, const PairPlan &p, const void *x, const void *folded, const int32_t *table, const int32_t *sel, void *y, uint8_t *argmax,
                hipStream_t st, const char *name)
{
    using T = typename Ops::Elem;
    CLG_REQUIRE((p.bands > 0) == (ROWS && !ONE), "%s: a plan of %d bands for another kernel", name, p.bands);
    const size_t lds = (size_t)kPairWaves * p.wave_elems * sizeof(T);
    if (int e = allow_lds(convblock_forward_pair_kernel<Ops, NL, RS, ROWS, ONE>, lds, name)) return e;
    hipLaunchKernelGGL((convblock_forward_pair_kernel<Ops, NL, RS, ROWS, ONE>), dim3((unsigned)(p.tiles * p.groups)), dim3(kPairWaves * kWave), lds, st,
                       (const T *)x, folded, table, sel, (T *)y, argmax, g, p);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}
template <typename Ops, int NL, int RS, bool ROWS>
int launch_pair(const Geom &g, const PairPlan &p, const void *x, const void *folded, const int32_t *table, const int32_t *sel, void *y, uint8_t *argmax,
                hipStream_t st, const char *name)
{
    if (p.G * (g.ho / 2) * (g.wo / 2) <= kWave) return launch_pair_one<Ops, NL, RS, ROWS, true>(g, p, x, folded, table, sel, y, argmax, st, name);
    return launch_pair_one<Ops, NL, RS, ROWS, false>(g, p, x, folded, table, sel, y, argmax, st, name);
}
template <typename Ops, int NL>
int launch_pair_nl(const Geom &g, const PairPlan &p, const void *x, const void *folded, const int32_t *table, const int32_t *sel, void *y,
                   uint8_t *argmax, hipStream_t st, const char *name)
{
    constexpr int PER = 16 / (int)sizeof(typename Ops::Elem);
    if (g.w % PER != 0) return launch_pair<Ops, NL, 0, false>(g, p, x, folded, table, sel, y, argmax, st, name);
    constexpr int kWide = PER == 4 ? 28 : 20, kNarrow = PER == 4 ? 18 : 14;    // 3 x 3 kernels on rows of 16 and of 8
    if (PER == 2 && p.rs == 9 && !p.bands) return launch_pair_one<Ops, NL, PER == 2 ? 9 : 0, true, true>(g, p, x, folded, table, sel, y, argmax, st, name);   // of 4
    if (p.rs == 40 && p.bands) return launch_pair_one<Ops, NL, 40, true, false>(g, p, x, folded, table, sel, y, argmax, st, name);   // of 28 and 32
    if (p.rs == kWide) return launch_pair<Ops, NL, kWide, true>(g, p, x, folded, table, sel, y, argmax, st, name);
    if (p.rs == kNarrow) return launch_pair<Ops, NL, kNarrow, true>(g, p, x, folded, table, sel, y, argmax, st, name);
    return launch_pair<Ops, NL, 0, true>(g, p, x, folded, table, sel, y, argmax, st, name);
}

}  // namespace

// Split rows: a window's two columns are read by instructions of their own, so that the lanes of one (cells of a row) read consecutive
// elements; with both in one row they were two apart and met in the 64 banks of LDS at least twice.  Row and sample strides put
// the rows and samples of a wavefront next to each other modulo the banks where their numbers are powers of two (an access of
// floats takes 64 lanes, of words 32): conflicts of a read 2 -> 1 for floats on 16 x 16 and 8 x 8, 4 and 3 -> 1 for words.
static bool split_rows(const Geom &g, int elem, PairPlan *p)
{
    const int hp = g.ho / 2, wp = g.wo / 2, half = (p->lead + g.w + g.pw + 1) / 2, step = elem == 4 ? 2 : 1, banks = elem == 4 ? 64 : 32;
    int wp2 = 1, hp2 = 1;
    while (wp2 < wp) wp2 *= 2;
    while (hp2 < hp) hp2 *= 2;
    const bool align = wp2 >= 2 * step;                               // (floats are stored in pairs: even strides)
    for (p->rs = (2 * half + step - 1) / step * step; ; p->rs += step) {
        p->odd = (p->rs / 2 + 1) & ~1;
        if (p->odd >= half && p->odd + half <= p->rs && (!align || p->rs % wp2 == wp2 / 2)) break;
    }
    p->plane = (p->bands ? 2 * p->band_rows + g.kh - 1 : g.h + g.ph) * p->rs;   // (a band has its halo rows itself)
    p->sample = 2 * p->plane;
    const int tile = wp2 * hp2;
    if (p->G > 1 && tile < banks && tile % step == 0)
        while (p->sample % (2 * tile) != tile) p->sample += step;
    return p->plane + p->sample < (1 << 15);                          // (offsets of 16 bits)
}

bool clg_plan_pair(const Geom &g, int elem, PairPlan *p, bool split)
{
    const int per = 16 / elem;
    *p = PairPlan{};
    if (!split && elem != 4) return false;                           // (the weight gradient, which words do not have)
    if (g.sh != 1 || g.sw != 1 || !taps_inside(g) || g.ho % 2 || g.wo % 2 || g.pw > per || (g.h * g.w) % per) return false;
    const int I = (g.ho / 2) * (g.wo / 2);
    p->lead = per;
    p->pw = g.pw;
    p->G = std::max(1, std::min(kWave / I, g.n));
    p->pieces = (uint32_t)(g.h * g.w / per);
    // an image of more than 64 cells whose rows are whole pieces goes in bands of whole rows of cells, or not at all
    if (split && I > kWave && g.w % per == 0) {
        if (g.wo / 2 > kWave) return false;
        const int rows = kWave / (g.wo / 2), hp = g.ho / 2;
        p->bands = (int)clg_ceil_div(hp, rows);
        p->band_rows = (int)clg_ceil_div(hp, p->bands);
        p->pieces = (uint32_t)((2 * p->band_rows + g.kh - 1) * (g.w / per));
    }
    p->loads = (int)clg_ceil_div((int64_t)2 * p->G * p->pieces, kWave);
    if (p->loads > 8 || (elem == 8 && p->loads > 6)) return false;
    if (split) {
        if (!split_rows(g, elem, p)) return false;
    } else {
        p->rs = g.w + per;
        p->plane = (g.h + g.ph) * p->rs;
        // samples 16 floats apart modulo the 64 banks, so that the rows of neighbouring samples do not meet there
        p->sample = (int)clg_ceil_div(2 * p->plane, per) * per;
        if (p->G > 1)
            while (p->sample % 64 != 16) p->sample += per;
    }
    p->wave_elems = (int)(clg_ceil_div((int64_t)p->G * p->sample + g.ph * p->rs + per + g.kw, per) * per + per + (p->odd + per) / per * per);   // (the end takes what lanes without a piece write)
    if ((int64_t)kPairWaves * p->wave_elems * elem > 64 * 1024) return false;
    if (p->bands && (int64_t)g.n * p->bands >= (1ll << 31)) return false;
    p->groups = p->bands ? g.n * p->bands : (int)clg_ceil_div(g.n, p->G);
    // 32-bit offsets inside a group of samples and in the table
    if ((int64_t)p->G * g.cin * g.h * g.w * elem >= (1ll << 32) || (int64_t)p->G * g.c * I * elem >= (1ll << 32) || g.c > 65535) return false;
    p->out_sample = g.y_fm ? 1 : g.c * I;
    p->out_cell = g.y_fm ? g.n : 1;
    if (g.y_fm && (int64_t)I * g.n * elem >= (1ll << 31)) return false;
    // kernels per workgroup: many, for the planes of a sample to be found in L2, as long as there are 8192 wavefronts
    int64_t ct = 64;
    while (ct > 4 * kPairWaves && (int64_t)p->groups * clg_ceil_div(g.c, ct) < 2048) ct /= 2;
    while (ct > kPairWaves && (int64_t)p->groups * clg_ceil_div(g.c, ct) < 512) ct /= 2;
    p->ct = (int)ct;
    p->tiles = (int)clg_ceil_div(g.c, ct);
    if (split && (int64_t)p->tiles * p->groups >= (1ll << 24)) return false;   // (workgroups of 256: fewer than 2^32 threads)
    p->d_tiles = make_fastdiv((uint32_t)p->tiles);
    p->d_bands = make_fastdiv((uint32_t)std::max(1, p->bands));
    p->d_pieces = make_fastdiv(p->pieces);
    p->d_w = make_fastdiv((uint32_t)g.w);
    p->d_wp = make_fastdiv((uint32_t)(g.wo / 2));
    p->d_cells = make_fastdiv((uint32_t)I);
    p->folded_bytes = elem == 4 ? ((size_t)g.c * 28 * 4 + 255) & ~(size_t)255 : 0;
    p->total_bytes = p->folded_bytes + (size_t)g.c * kPairTable * 4 + sizeof(Geom);
    return true;
}

// float: w = probabilities or, with from_logits, logits; folded_in: coefficients that are made already, folded_out: where they go
// (null: scratch).  padded_out: where the zero-padded copy of x goes (strides rs, chs), or null.
int clg_forward_pair_f32(const Geom &g, const PairPlan &p, const float *x, const float *w, const int32_t *sel, float *y, uint8_t *argmax, void *scratch,
                         bool from_logits, float *probs_out, const float *folded_in, float *padded_out, int pad_rs, int pad_chs, int pad_sample,
                         hipStream_t st, const char *name, float *folded_out, bool prepared)
{
    unsigned char *base = reinterpret_cast<unsigned char *>(scratch);
    float *folded = folded_out ? folded_out : reinterpret_cast<float *>(base);
    int32_t *table = clg_pair_table(p, scratch);
    if (!prepared || padded_out) {                                    // (prepared: coefficients and table are there)
        const PadJob<float> job = padded_out ? make_pad_job(x, padded_out, g, pad_rs, pad_chs, pad_sample) : no_pad_job<float>();
        const unsigned prep = (unsigned)clg_ceil_div((int64_t)g.c * (folded_in ? 1 : 7), 256);
        // (a large copy goes past the caches: it is read in the backward pass; [128,1024,16,16] and [128,4096,8,8], 160 and 215 MB, copy and forward
        // 241 -> 225 and 229 -> 207 us; step of the CIFAR topology, 40 MB 1030 -> 1022 us, no difference at 28)
        auto kern = clg_past_caches(job.total * 4, 36) ? pair_prepare_kernel<FloatOps<float>, float, float, true> : pair_prepare_kernel<FloatOps<float>, float, float, false>;
        hipLaunchKernelGGL(kern, dim3(prep + pad_blocks(job)), dim3(256), 0, st, w, sel,
                           folded_in ? (float *)nullptr : folded, table, p, g, job, (int)prep, from_logits ? 1 : 0, probs_out);
        CLG_CHECK_LAUNCH(name);
    }
    const void *fc = folded_in ? (const void *)folded_in : (const void *)folded;
    using Ops = FloatOps<float>;
    if (p.loads <= 2) return launch_pair_nl<Ops, 2>(g, p, x, fc, table, sel, y, argmax, st, name);
    if (p.loads <= 4) return launch_pair_nl<Ops, 4>(g, p, x, fc, table, sel, y, argmax, st, name);
    return launch_pair_nl<Ops, 8>(g, p, x, fc, table, sel, y, argmax, st, name);
}

int clg_forward_pair_packed(const Geom &g, const PairPlan &p, const uint64_t *x, const uint8_t *gates, const int32_t *sel, uint64_t *y, void *scratch,
                            hipStream_t st, const char *name)
{
    int32_t *table = reinterpret_cast<int32_t *>(scratch);
    const unsigned prep = (unsigned)clg_ceil_div(g.c, 256);
    if (gates != nullptr)
        hipLaunchKernelGGL((pair_prepare_kernel<BitOpsAnf, uint8_t, float, false>), dim3(prep), dim3(256), 0, st, gates, sel, (float *)nullptr, table, p, g,
                       no_pad_job<float>(), (int)prep, 0, (float *)nullptr);
    CLG_CHECK_LAUNCH(name);
    if (p.loads <= 2) return launch_pair_nl<BitOpsAnf, 2>(g, p, x, nullptr, table, sel, y, nullptr, st, name);
    if (p.loads <= 4) return launch_pair_nl<BitOpsAnf, 4>(g, p, x, nullptr, table, sel, y, nullptr, st, name);
    return launch_pair_nl<BitOpsAnf, 6>(g, p, x, nullptr, table, sel, y, nullptr, st, name);
}

extern "C" int clg_convblock_pair_plan(int dtype, const clg_conv_geom *gg, int weight_gradient, int64_t *plan)
{
    const char *name = "clg_convblock_pair_plan";
    Geom g;
    if (int e = clg_convblock_check(gg, &g, dtype, name)) return e;
    CLG_REQUIRE(plan && !(weight_gradient && dtype != CLG_F32), "%s: null pointer argument, or a weight gradient of words", name);
    PairPlan p;
    if (!clg_plan_pair(g, dtype == CLG_F64 ? 8 : 4, &p, !weight_gradient)) return 0;
    plan[0] = p.G;
    plan[1] = p.groups;
    plan[2] = p.bands;
    plan[3] = p.band_rows;
    plan[4] = (int64_t)kPairWaves * p.wave_elems * (dtype == CLG_F64 ? 8 : 4);
    plan[5] = weight_gradient ? clg_pair_grad_w_parts(g, p) : 0;
    return 1;
}
