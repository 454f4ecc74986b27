// Plan and entry points of the forward that stages two planes per wavefront (conv_pair.hip).
#pragma once

#include "conv_tile.h"

struct PairPlan {
    int G, groups;            // samples per wavefront, groups of them; or
    int bands, band_rows;     // a sample of more than 64 cells in bands of so many rows of them (bands > 0; a group is a band)
    int ct, tiles;            // kernels per workgroup, tiles of them
    int lead, pw, rs, plane, sample, wave_elems;   // LDS, in elements: zeros in front of a row, row / plane / sample stride, all of a wavefront
    int odd;                  // from a row's even columns to its odd ones where they are kept apart, else 0
    int loads;                // 16-byte pieces per lane
    uint32_t pieces;          // per plane, or per band of one
    FastDiv d_tiles, d_pieces, d_w, d_wp, d_cells, d_bands;
    size_t folded_bytes, total_bytes;   // scratch: folded coefficients | table and geometry
    int out_sample, out_cell;           // the output: elements between samples, between cells of a kernel (whose cells follow those of the kernel before)
};
// Of a tap (plane, row, column) from a window's first position: the offset of the window's first column in the low half, of its second in
// the high one; shift: what the rows' zeros put in front of column 0.
__host__ __device__ inline int32_t pair_tap(int plane, int rs, int odd, int shift, bool second, int ry, int rx)
{
    const int row = (second ? plane : 0) + ry * rs, a = rx + shift, b = a + 1;
    return (row + (a & 1) * odd + (a >> 1)) | (row + (b & 1) * odd + (b >> 1)) << 16;
}
constexpr int kPairTable = 12;          // per kernel: channel 0, channel 1 (-1: more than two), code, -, 8 taps;
                                        // behind the last one the geometry, for the rare path that needs all of it
struct PairOffsets {
    int plane, rs, odd, shift;
};
__host__ __device__ inline PairOffsets pair_offsets(const PairPlan &p) { return {p.plane, p.rs, p.odd, p.lead - p.pw}; }
#if defined(__HIPCC__)
// channels and taps of kernel q
__device__ __forceinline__ void pair_table_row(int32_t *__restrict__ table, const int32_t *__restrict__ sel, int64_t q, const PairOffsets &at, const Geom &g)
{
    const TapLimit lim = tap_limit(g);
    Tap tp[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) tp[t] = unpack_tap(sel[q * 8 + t], lim);
    const int ch0 = tp[0].ch;
    int ch1 = ch0;
#pragma unroll
    for (int t = 7; t >= 1; --t) ch1 = tp[t].ch != ch0 ? tp[t].ch : ch1;   // first channel that differs
    bool wide = false;
    int32_t *row = table + q * kPairTable;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        wide |= tp[t].ch != ch0 && tp[t].ch != ch1;
        row[4 + t] = pair_tap(at.plane, at.rs, at.odd, at.shift, tp[t].ch != ch0, tp[t].ry, tp[t].rx);
    }
    row[0] = ch0;
    row[1] = wide ? -1 : ch1;
}
#endif
// elem: 4 (float) or 8 (words).  False where the shape is another kernel's.  split: even and odd columns apart, as the forward kernels
// read them; without, as the weight gradient of floats does.
bool clg_plan_pair(const Geom &g, int elem, PairPlan *p, bool split = true);
int clg_forward_pair_f32(const Geom &g, const PairPlan &p, const float *x, const float *w, const int32_t *sel, float *y, uint8_t *argmax, void *scratch,
                         bool from_logits, float *probs_out, const float *folded_in, float *padded_out, int pad_rs, int pad_chs, int pad_sample,
                         hipStream_t st, const char *name, float *folded_out = nullptr, bool prepared = false);
// The plan of a float32 block whose forward call takes this kernel (conv_forward.hip).
int clg_forward_pair_plan(const char *name, const clg_conv_geom *gg, bool feature_major, Geom *g, PairPlan *p, bool *pair);
static inline int32_t *clg_pair_table(const PairPlan &p, void *scratch)
{
    return reinterpret_cast<int32_t *>(reinterpret_cast<unsigned char *>(scratch) + p.folded_bytes);
}
// gates: null where the table at the start of the scratch is made already
int clg_forward_pair_packed(const Geom &g, const PairPlan &p, const uint64_t *x, const uint8_t *gates, const int32_t *sel, uint64_t *y, void *scratch,
                            hipStream_t st, const char *name);
// Whether a packed block comes here when its table costs no launch of its own (conv_forward.hip).
bool clg_packed_pair(const Geom &g, PairPlan *p);

constexpr int kPairWaves = 4;
// The 28 sums per kernel of a float block's weight gradient by the same staging (conv_pair_grad.hip): partial [c][nb][28].
int clg_pair_grad_w_parts(const Geom &g, const PairPlan &p);          // nb, at most 64
bool clg_pair_grad_w_wanted(const Geom &g, const PairPlan &p);        // false where it is not the kernel to take
int clg_pair_grad_w(const Geom &g, const PairPlan &p, int nb, const float *gy, const float *x, const float *folded, const int32_t *sel,
                    const uint8_t *argmax, float *partial, hipStream_t st, const char *name);

// Both gradients: the sums as above, and the input gradient by way of gradient planes per kernel and channel (clg_pair_planes_bytes), which
// are summed per channel; nb: the parts that it has left.  count, hits: the lists of conv_block.hip.
constexpr int kHitWide = 1 << 24;                                    // of a list entry: the kernel's taps are in more than two channels
bool clg_pair_planes_fit(const Geom &g, const PairPlan &p);
size_t clg_pair_planes_bytes(const Geom &g);
int clg_pair_grads(const Geom &g, const PairPlan &p, int *nb, const float *gy, const float *x, const float *folded, const int32_t *sel,
                   const uint8_t *argmax, const int32_t *count, const int32_t *hits, float *planes, float *partial, float *gx, hipStream_t st,
                   const char *name);

#if defined(__HIPCC__)
namespace {

// LDS that the lanes of one wavefront share: its accesses complete in order, the compiler has to keep them so
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The 16-byte pieces of two planes of a group of samples on their way to LDS: fetch() requests those of two channels, store() puts them
// into the rows of the image.  ROWS: no piece crosses a row.  SPLIT: even and odd columns apart.  A lane without a piece
// reads the first one and writes behind the planes.
typedef u32x4 u32x4_any __attribute__((aligned(4)));                  // (global memory takes 16 bytes at every multiple of four)
template <typename T, int NL, bool ROWS, bool SPLIT>
struct PairPieces {
    static constexpr int PER = 16 / (int)sizeof(T);
    uint32_t from[NL], second[NL];                                   // second: all ones for a piece of channel 1
    int to[NL][ROWS ? 1 : PER];
    u32x4 piece[NL];
    __device__ __forceinline__ void place(const Geom &g, const PairPlan &p, int row_step, int g_here, int lane)
    {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t v = lane + i * kWave, pl = fdiv(v, p.d_pieces), e = (v - pl * p.pieces) * PER, s = pl >> 1, plane = pl & 1;
            const bool have = (int)s < g_here;
            second[i] = have && plane ? ~0u : 0u;
            from[i] = have ? (s * (uint32_t)(g.cin * g.h * g.w) + e) * (uint32_t)sizeof(T) : 0;
#pragma unroll
            for (int j = 0; j < (ROWS ? 1 : PER); ++j) {
                const uint32_t r = fdiv(e + j, p.d_w), col = e + j - r * (uint32_t)g.w;
                const uint32_t at = p.lead + col, place = SPLIT ? (at & 1) * p.odd + (at >> 1) : at;
                to[i][j] = have ? (int)(s * p.sample + plane * p.plane + (r + g.ph) * row_step + place) : p.wave_elems - PER - (SPLIT ? p.odd : 0) + j;
            }
        }
    }
    // a band of one sample: its rows begin at row y0 of the image, those outside it stay the zeros they are
    __device__ __forceinline__ void place_band(const Geom &g, const PairPlan &p, int row_step, int y0, int lane)
    {
        static_assert(ROWS && SPLIT, "whole pieces per row");
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t v = lane + i * kWave, plane = fdiv(v, p.d_pieces), e = (v - plane * p.pieces) * PER, r = fdiv(e, p.d_w);
            const uint32_t col = e - r * (uint32_t)g.w, at = p.lead + col;
            const int y = y0 + (int)r;
            const bool have = plane < 2 && y >= 0 && y < g.h;
            second[i] = have && plane ? ~0u : 0u;
            from[i] = have ? (uint32_t)(y * g.w + (int)col) * (uint32_t)sizeof(T) : 0;
            to[i][0] = have ? (int)(plane * p.plane + r * row_step + (at >> 1)) : p.wave_elems - PER - p.odd;
        }
    }
    // o0: bytes from the group's first sample to its channel 0, d: from there to channel 1 (modulo 2^32)
    __device__ __forceinline__ void fetch(const T *__restrict__ xg, uint32_t o0, uint32_t d)
    {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t o = from[i] + o0 + (second[i] & d);
            piece[i] = *reinterpret_cast<const u32x4_any *>(reinterpret_cast<const char *>(xg) + (size_t)o);
        }
    }
    __device__ __forceinline__ void store(T *__restrict__ image, int odd = 0)
    {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            if constexpr (ROWS && SPLIT && PER == 4) {
                *reinterpret_cast<u32x2 *>(image + to[i][0]) = u32x2{piece[i].x, piece[i].z};
                *reinterpret_cast<u32x2 *>(image + to[i][0] + odd) = u32x2{piece[i].y, piece[i].w};
            } else if constexpr (ROWS && SPLIT) {
                *reinterpret_cast<u32x2 *>(image + to[i][0]) = u32x2{piece[i].x, piece[i].y};
                *reinterpret_cast<u32x2 *>(image + to[i][0] + odd) = u32x2{piece[i].z, piece[i].w};
            } else if constexpr (ROWS) {
                *reinterpret_cast<u32x4 *>(image + to[i][0]) = piece[i];
            } else {
                T part[PER];
                __builtin_memcpy(part, &piece[i], 16);
#pragma unroll
                for (int j = 0; j < PER; ++j) image[to[i][j]] = part[j];
            }
        }
    }
};

}  // namespace
#endif
