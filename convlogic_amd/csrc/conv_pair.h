// Plan and entry points of the forward that stages two planes per wavefront (conv_pair.hip).
#pragma once

#include "conv_tile.h"

struct PairPlan {
    int G, groups;            // samples per wavefront, groups of them
    int ct, tiles;            // kernels per workgroup, tiles of them
    int lead, pw, rs, plane, sample, wave_elems;   // LDS, in elements: zeros in front of a row, row / plane / sample stride, all of a wavefront
    int loads;                // 16-byte pieces per lane
    uint32_t pieces;          // per plane
    FastDiv d_tiles, d_pieces, d_w, d_wp, d_cells;
    size_t folded_bytes, total_bytes;   // scratch: folded coefficients | table and geometry
};
// elem: 4 (float) or 8 (words).  False where the shape is another kernel's.
bool clg_plan_pair(const Geom &g, int elem, PairPlan *p);
int clg_forward_pair_f32(const Geom &g, const PairPlan &p, const float *x, const float *w, const int32_t *sel, float *y, uint8_t *argmax, void *scratch,
                         bool from_logits, float *probs_out, const float *folded_in, float *padded_out, int pad_rs, int pad_chs, int pad_sample,
                         hipStream_t st, const char *name, float *folded_out = nullptr);
int clg_forward_pair_packed(const Geom &g, const PairPlan &p, const uint64_t *x, const uint8_t *gates, const int32_t *sel, uint64_t *y, void *scratch,
                            hipStream_t st, const char *name);
