// Packed-bit inference: pack bool -> words, bitwise gate evaluation, per-class popcount.
//
// A word holds `bits` samples of one feature (sample s = bit s % bits of word s / bits, LSB first).
// Every gate is bitwise, so the evaluation kernel treats a row as a run of bytes and moves it with
// 16-byte vectors whatever the word type is; one wavefront evaluates one neuron (gate id, wiring
// and truth-table masks are wave-uniform) over a column chunk of its two input rows.
#include <stdlib.h>

#include <algorithm>

#include "clg_common.h"

namespace {

// ---------------------------------------------------------------------------------------------
// evaluation
// ---------------------------------------------------------------------------------------------
constexpr int kEvalBlock = 256;
constexpr int kEvalWaves = kEvalBlock / kWave;

// Index of the first maximum of 16 float32 logits, a NaN counting as the maximum (the rule of gate_argmax_kernel and of
// torch.argmax), computed by the whole wavefront: lane l holds logit l % 16 (`v`) as an order-preserving integer key (-0
// and +0 equal, NaN on top), the row maximum comes over DPP, the first lane that holds it names the gate.  Wave-uniform.
__device__ __forceinline__ int argmax16_uniform(float v)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, v + 0.0f);
    const uint32_t key = v != v ? 0xFFFFFFFFu : (u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u));
    const uint32_t top = row16_max(key);
    const uint32_t first = (uint32_t)__ballot(key == top) & 0xFFFFu;
    return uniform(__builtin_ctz(first));
}

// Rows are `row_vecs` vectors of type V.  blockIdx.x enumerates (column chunk, neuron group) with
// the chunk as the slow index, so that all neurons of one column chunk run back to back and the
// second read of an input row segment finds it in the last-level cache.
// LOGITS: `gate` points to float32 logits [out_dim, 16] and the wavefront takes their arg-max itself, else to uint8 gate ids.
// Rows of whole 16-byte vectors from 1 MiB on come here where there is no walk of the wiring, and rows below 16 bytes; the rest: eval_packed_rows_kernel.
template <typename V, int UNROLL, bool LOGITS>
__global__ __launch_bounds__(kEvalBlock) void eval_packed_kernel(const V *__restrict__ x, const int64_t *__restrict__ a,
                                                               const int64_t *__restrict__ b,
                                                               const void *__restrict__ gate, V *__restrict__ y,
                                                               int out_dim, int64_t row_vecs, int chunk_vecs,
                                                               int groups_per_chunk, int neurons_per_wave, int64_t in_dim)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int chunk = blockIdx.x / groups_per_chunk;
    const int group = blockIdx.x % groups_per_chunk;
    const int64_t v0 = (int64_t)chunk * chunk_vecs;
    const int64_t v1 = (v0 + chunk_vecs < row_vecs) ? v0 + chunk_vecs : row_vecs;
    const int j0 = (group * kEvalWaves + wave) * neurons_per_wave;
    for (int jj = 0; jj < neurons_per_wave; ++jj) {
        const int j = j0 + jj;
        if (j >= out_dim) break;
        const V *xa = x + clamp_index(a[j], in_dim) * row_vecs;    // (a bad index reads a wrong row; it never leaves x)
        const V *xb = x + clamp_index(b[j], in_dim) * row_vecs;
        V *yj = y + (int64_t)j * row_vecs;
        int id;
        if constexpr (LOGITS) id = argmax16_uniform(reinterpret_cast<const float *>(gate)[(int64_t)j * 16 + (lane & 15)]);
        else id = reinterpret_cast<const uint8_t *>(gate)[j];
        const Masks m = gate_masks(id);
        for (int64_t v = v0 + lane; v < v1; v += (int64_t)kWave * UNROLL) {
            V ra[UNROLL], rb[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                const int64_t vv = v + (int64_t)u * kWave;
                if (vv < v1) {
                    ra[u] = xa[vv];
                    rb[u] = xb[vv];
                }
            }
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                const int64_t vv = v + (int64_t)u * kWave;
                if (vv < v1) __builtin_nontemporal_store(gate_vec(m, ra[u], rb[u]), yj + vv);
            }
        }
    }
}

// Short rows: lanes run along the 16-byte pieces of `nj` neurons of the workgroup, all of them in flight at once, so that neither lanes without a
// piece nor one round of loads after the other are paid for; four lanes per neuron find its gate meanwhile.  Rows of any number of bytes from 16 on: the
// last piece of a row steps back to its last 16 bytes, some of which two lanes write then (the same values).  us per layer, a wavefront per neuron or a walk
// -> here: 64000 neurons on rows of 64 bytes 15.7 -> 4.1, of 252 18.3 -> 9.6, 8000 on 1280 7.7 -> 4.4; one piece of a thread at a time instead of two
// costs up to 10 %, stores that stay in the caches up to 25 (64000 on 8188: 250 us, 219).
// A row of more pieces than a workgroup has in flight is cut into parts of `per` pieces, a workgroup each: few neurons on long rows fill the chip too
// (in one workgroup each 64 on 400 KiB took 60 us, here 12.4, 1 on 4 MiB 530, 3.5, 100 on 64 KiB 8.6, 4.0).  The parts are the slow index of the launch: the neurons of one part run back to
// back and find the second use of an input row's piece in the caches.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
constexpr int kRowsMax = 64, kRowsUnroll = 2;                        // neurons of a workgroup, pieces of a thread
template <bool LOGITS>
__global__ __launch_bounds__(kEvalBlock) void eval_packed_rows_kernel(const uint8_t *__restrict__ x, const int64_t *__restrict__ a,
                                                                    const int64_t *__restrict__ b, const void *__restrict__ gate,
                                                                    uint8_t *__restrict__ y, int out_dim, int64_t row_bytes, uint32_t pieces,
                                                                    FastDiv d_pieces, int nj, FastDiv d_groups, uint32_t per, int64_t in_dim)
{
    __shared__ int ids[kRowsMax];
    const uint32_t part = fdiv(blockIdx.x, d_groups);
    const int j0 = (int)(blockIdx.x - part * d_groups.d) * nj, here = min(nj, out_dim - j0), q = threadIdx.x >> 2;
    const uint32_t total = min((uint32_t)here * pieces, (part + 1) * per);   // (more than one part: of one neuron)
    f32x4u logits = 0.f;                                              // requested ahead of the rows: vector loads return in order
    if (LOGITS && q < here) logits = reinterpret_cast<const f32x4u *>(reinterpret_cast<const float *>(gate) + (int64_t)(j0 + q) * 16)[threadIdx.x & 3];
    u32x4 ra[kRowsUnroll], rb[kRowsUnroll];
    int jn[kRowsUnroll];
    int64_t off[kRowsUnroll];
    auto request = [&](uint32_t first) {
#pragma unroll
        for (int u = 0; u < kRowsUnroll; ++u) {
            const uint32_t e = first + u * kEvalBlock + threadIdx.x, ec = e < total ? e : 0;
            jn[u] = (int)fdiv(ec, d_pieces);
            off[u] = min((int64_t)(ec - jn[u] * pieces) * 16, row_bytes - 16);
            ra[u] = *reinterpret_cast<const u32x4_any *>(x + clamp_index(a[j0 + jn[u]], in_dim) * row_bytes + off[u]);
            rb[u] = *reinterpret_cast<const u32x4_any *>(x + clamp_index(b[j0 + jn[u]], in_dim) * row_bytes + off[u]);
        }
    };
    request(part * per);
    if constexpr (LOGITS) {
        const int id = argmax16_quad(logits);
        if ((threadIdx.x & 3) == 0 && q < here) ids[q] = id;
    } else {
        if ((int)threadIdx.x < here) ids[threadIdx.x] = reinterpret_cast<const uint8_t *>(gate)[j0 + threadIdx.x];
    }
    __syncthreads();
    for (uint32_t first = part * per;;) {
#pragma unroll
        for (int u = 0; u < kRowsUnroll; ++u)
            if (first + u * kEvalBlock + threadIdx.x < total)
                __builtin_nontemporal_store((u32x4_any)gate_vec(gate_masks(ids[jn[u]]), ra[u], rb[u]),
                                            reinterpret_cast<u32x4_any *>(y + (int64_t)(j0 + jn[u]) * row_bytes + off[u]));
        first += kRowsUnroll * kEvalBlock;
        if (first >= total) return;
        request(first);
    }
}

// ---------------------------------------------------------------------------------------------
// evaluation along a precomputed walk of the wiring graph
// ---------------------------------------------------------------------------------------------
// Input rows are vertices and neurons are edges of a multigraph.  The plan lists the neurons along
// trails of that graph, so that a neuron shares one input row with its predecessor; the wavefront
// keeps that row in registers and loads only the other one.  Every row chunk is then read about once
// (plus one extra row per segment start) instead of twice.
// plan[k] = neuron | use << 28 | keep << 30
//   use : 0 nothing carried, 1 carried row is input a, 2 carried row is input b, 3 it is both
//   keep: row carried to the next step, 0 = input a, 1 = input b
// gate[j] for a wave-uniform j through the scalar cache: the aligned 32-bit word that holds it (a byte load would be a
// vector load, and the wait for it would also wait for the row loads in flight).  The last word is read bytewise when
// it reaches past the table; the table starts at a 4-byte boundary or is read bytewise altogether.
__device__ __forceinline__ int gate_id_uniform(const uint8_t *__restrict__ gate, int j, int n)
{
    if ((reinterpret_cast<uintptr_t>(gate) & 3) == 0 && (j | 3) < n) {
        const uint32_t w = reinterpret_cast<const uint32_t *>(gate)[j >> 2];
        return (int)((w >> ((j & 3) * 8)) & 0xFFu);
    }
    return gate[j];
}

// LOGITS: `gate` points to float32 logits [out_dim, 16] and the wavefront takes their arg-max itself (the layer's eval
// call then needs no launch of its own for the gate ids); else to uint8 gate ids [out_dim].
// Rows of any number of bytes from 16 on, row_vecs vectors of 16 bytes, the last of which steps back to the row's last 16 bytes.
template <int R, bool LOGITS>
__global__ __launch_bounds__(kEvalBlock) void eval_packed_walk_kernel(const uint8_t *__restrict__ x, const int64_t *__restrict__ a,
                                                                    const int64_t *__restrict__ b,
                                                                    const void *__restrict__ gate,
                                                                    const int32_t *__restrict__ plan, uint8_t *__restrict__ y,
                                                                    int steps, int seg_len, int64_t row_vecs, int64_t row_bytes, int64_t in_dim)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int k0 = (blockIdx.x * kEvalWaves + wave) * seg_len;
    if (k0 >= steps) return;
    const int k1 = k0 + seg_len < steps ? k0 + seg_len : steps;
    const int64_t col0 = (int64_t)blockIdx.y * (kWave * R) + lane;   // this lane's first vector in the row
    int64_t at[R];
#pragma unroll
    for (int r = 0; r < R; ++r) at[r] = min((col0 + r * kWave) * 16, row_bytes - 16);
    u32x4 ra[R], rb[R], carry[R];
#pragma unroll
    for (int r = 0; r < R; ++r) carry[r] = (u32x4)0u;
    for (int k = k0; k < k1; ++k) {
        const int p = plan[k];
        const int j = min(p & 0x0FFFFFFF, steps - 1), keep = (p >> 30) & 1;   // one plan entry per neuron
        const int use = k == k0 ? 0 : (p >> 28) & 3;
        const uint8_t *xa = x + clamp_index(a[j], in_dim) * row_bytes;
        const uint8_t *xb = x + clamp_index(b[j], in_dim) * row_bytes;
        float logit = 0.f;                                            // requested ahead of the rows: vector loads return in order
        if constexpr (LOGITS) logit = reinterpret_cast<const float *>(gate)[(int64_t)j * 16 + (lane & 15)];
        if (use != 1 && use != 3) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (col0 + r * kWave < row_vecs) ra[r] = *reinterpret_cast<const u32x4_any *>(xa + at[r]);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) ra[r] = carry[r];
        }
        if (use < 2) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (col0 + r * kWave < row_vecs) rb[r] = *reinterpret_cast<const u32x4_any *>(xb + at[r]);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) rb[r] = carry[r];
        }
        int id;
        if constexpr (LOGITS) id = argmax16_uniform(logit);
        else id = gate_id_uniform(reinterpret_cast<const uint8_t *>(gate), j, steps);
        const Masks m = gate_masks(id);
        uint8_t *yj = y + (int64_t)j * row_bytes;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (col0 + r * kWave < row_vecs) __builtin_nontemporal_store((u32x4_any)gate_vec(m, ra[r], rb[r]), reinterpret_cast<u32x4_any *>(yj + at[r]));
#pragma unroll
        for (int r = 0; r < R; ++r) carry[r] = keep ? rb[r] : ra[r];
    }
}

// bytewise tail / odd row sizes: one thread per byte of the output
__global__ void eval_packed_bytes_kernel(const uint8_t *__restrict__ x, const int64_t *__restrict__ a,
                                         const int64_t *__restrict__ b, const uint8_t *__restrict__ gate,
                                         uint8_t *__restrict__ y, int64_t out_dim, int64_t row_bytes, int64_t in_dim)
{
    const int64_t total = out_dim * row_bytes;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = i / row_bytes, c = i % row_bytes;
        const Masks m = gate_masks(gate[j]);
        y[i] = (uint8_t)gate_bits(m, x[clamp_index(a[j], in_dim) * row_bytes + c], x[clamp_index(b[j], in_dim) * row_bytes + c]);
    }
}

// ---------------------------------------------------------------------------------------------
// packing
// ---------------------------------------------------------------------------------------------
// 8 bool bytes (any non-zero value counts as true) -> 8 bits, byte k -> bit k.
__device__ __forceinline__ uint32_t squeeze8(uint64_t v)
{
    v |= v >> 4;
    v |= v >> 2;
    v |= v >> 1;
    v &= 0x0101010101010101ull;
    return (uint32_t)((v * 0x0102040810204080ull) >> 56);
}

// feature-major input t [F, B]: one thread per output byte (8 samples); the word type only fixes the
// padded row length, because words are little endian and samples fill them LSB first.
__global__ void pack_bits_kernel(const uint8_t *__restrict__ t, uint8_t *__restrict__ out, int64_t features, int64_t batch,
                                 int64_t row_bytes, bool aligned8)
{
    const int64_t total = features * row_bytes;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t f = i / row_bytes, c = i % row_bytes;
        const int64_t s0 = c * 8;
        const uint8_t *p = t + f * batch + s0;
        uint32_t bits = 0;
        if (aligned8 && s0 + 8 <= batch) {
            bits = squeeze8(*reinterpret_cast<const uint64_t *>(p));
        } else {
            for (int k = 0; k < 8; ++k)
                if (s0 + k < batch && p[k]) bits |= 1u << k;
        }
        out[i] = (uint8_t)bits;
    }
}

// sample-major input t [B, F]: lanes run along features (contiguous reads), each thread keeps the
// 64 samples of one feature in a 64-bit register and then stores 8 bytes of that feature's row.
// Consecutive 64-sample groups of the same features are handled by the same thread one after the
// other so that its partial-line stores merge in L2.
constexpr int kPackGroups = 16;  // 64-sample groups per thread
__global__ __launch_bounds__(256) void pack_bits_sm_kernel(const uint8_t *__restrict__ t, uint8_t *__restrict__ out,
                                                         int64_t features, int64_t batch, int64_t row_bytes)
{
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= features) return;
    const int64_t g0 = (int64_t)blockIdx.y * kPackGroups;
    for (int g = 0; g < kPackGroups; ++g) {
        const int64_t s0 = (g0 + g) * 64;
        if (s0 >= batch) break;
        uint64_t word = 0;
        const int64_t n = batch - s0 < 64 ? batch - s0 : 64;
        if (n == 64) {
#pragma unroll 16
            for (int k = 0; k < 64; ++k) word |= (uint64_t)(t[(s0 + k) * features + f] != 0) << k;
        } else {
            for (int k = 0; k < n; ++k) word |= (uint64_t)(t[(s0 + k) * features + f] != 0) << k;
        }
        uint8_t *dst = out + f * row_bytes + s0 / 8;
        const int64_t nbytes = row_bytes - s0 / 8 < 8 ? row_bytes - s0 / 8 : 8;
        if (nbytes == 8 && (row_bytes & 7) == 0) {
            *reinterpret_cast<uint64_t *>(dst) = word;
        } else {
            for (int k = 0; k < nbytes; ++k) dst[k] = (uint8_t)(word >> (8 * k));
        }
    }
}

// The same for feature counts that are multiples of 16: a lane takes 16 consecutive features, so a
// wavefront reads 1 KiB of a sample row per load.  Bytes are turned into bits four features at a time
// inside a 32-bit register: bit 7 of every byte is set where the byte is non-zero, and
// acc = (acc >> 1) | bits run over 8 samples leaves their 8 bits LSB first in every byte.
template <int V>
struct PackVec;
template <>
struct PackVec<1> {
    typedef uint32_t type;
    static __device__ __forceinline__ uint32_t get(uint32_t v, int) { return v; }
};
template <>
struct PackVec<2> {
    typedef u32x2 type;
    static __device__ __forceinline__ uint32_t get(u32x2 v, int q) { return v[q]; }
};
template <>
struct PackVec<4> {
    typedef u32x4 type;
    static __device__ __forceinline__ uint32_t get(u32x4 v, int q) { return v[q]; }
};
// V 32-bit registers (4 V features) per lane, G consecutive 64-sample groups per thread (its 8-byte stores
// to one feature row are then adjacent and merge into full lines in L2).
template <int V, int G>
__global__ __launch_bounds__(256) void pack_bits_smv_kernel(const uint8_t *__restrict__ t, uint8_t *__restrict__ out,
                                                          int64_t features, int64_t batch, int64_t row_bytes)
{
    typedef typename PackVec<V>::type Vec;
    const int64_t f0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * (4 * V);
    if (f0 >= features) return;
    const int64_t row_vecs = features / (4 * V);
    for (int g = 0; g < G; ++g) {
        const int64_t s0 = ((int64_t)blockIdx.y * G + g) * 64;
        if (s0 >= batch) break;
        const int n = batch - s0 < 64 ? (int)(batch - s0) : 64;
        const Vec *src = reinterpret_cast<const Vec *>(t + s0 * features + f0);
        uint32_t acc[8][V];
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            Vec v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = o * 8 + j < n ? src[(int64_t)(o * 8 + j) * row_vecs] : Vec(0u);
#pragma unroll
            for (int q = 0; q < V; ++q) {
                uint32_t a = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t b = PackVec<V>::get(v[j], q);
                    const uint32_t nz = (((b & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | b) & 0x80808080u;
                    a = (a >> 1) | nz;
                }
                acc[o][q] = a;
            }
        }
        const int64_t byte0 = s0 / 8;
        const int64_t nbytes = row_bytes - byte0 < 8 ? row_bytes - byte0 : 8;
#pragma unroll
        for (int q = 0; q < V; ++q) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                uint32_t lo = 0, hi = 0;
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    lo |= ((acc[o][q] >> (8 * b)) & 0xFFu) << (8 * o);
                    hi |= ((acc[4 + o][q] >> (8 * b)) & 0xFFu) << (8 * o);
                }
                uint8_t *dst = out + (f0 + 4 * q + b) * row_bytes + byte0;
                const uint64_t word = ((uint64_t)hi << 32) | lo;
                if (nbytes == 8 && (row_bytes & 7) == 0) {
                    *reinterpret_cast<uint64_t *>(dst) = word;
                } else {
                    for (int k = 0; k < nbytes; ++k) dst[k] = (uint8_t)(word >> (8 * k));
                }
            }
        }
    }
}

// The same bit gathering with the stores gone through LDS: a workgroup of FL feature lanes x SG sample groups packs
// 16 FL features x 64 SG samples, collects the words in LDS and writes SG consecutive words (8 SG bytes) of every feature
// row with consecutive lanes and streaming stores.  The 8-byte stores of the kernel above, scattered over rows, cost a
// third of its time (155 us against 100 us without them on bool [8192, 64000]).
template <int FL, int SG>
__global__ __launch_bounds__(FL *SG) void pack_bits_tile_kernel(const uint8_t *__restrict__ t, uint8_t *__restrict__ out,
                                                           int64_t features, int64_t batch, int64_t row_bytes)
{
    __shared__ uint64_t tile[FL * 16][SG + 1];
    const int fl = threadIdx.x % FL, sg = threadIdx.x / FL;
    const int64_t f0 = ((int64_t)blockIdx.x * FL + fl) * 16;
    const int64_t s0 = ((int64_t)blockIdx.y * SG + sg) * 64;
    uint32_t acc[8][4];
#pragma unroll
    for (int o = 0; o < 8; ++o)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[o][q] = 0;
    if (f0 < features && s0 < batch) {
        const int n = batch - s0 < 64 ? (int)(batch - s0) : 64;
        const int64_t row_vecs = features / 16;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(t + s0 * features + f0);
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            u32x4 v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = o * 8 + j < n ? src[(int64_t)(o * 8 + j) * row_vecs] : u32x4(0u);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t a = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t b = v[j][q];
                    const uint32_t nz = (((b & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | b) & 0x80808080u;
                    a = (a >> 1) | nz;
                }
                acc[o][q] = a;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t lo = 0, hi = 0;
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                lo |= ((acc[o][q] >> (8 * b)) & 0xFFu) << (8 * o);
                hi |= ((acc[4 + o][q] >> (8 * b)) & 0xFFu) << (8 * o);
            }
            tile[(4 * q + b) * FL + fl][sg] = ((uint64_t)hi << 32) | lo;   // feature-lane fastest: the lanes of a wavefront spread over the banks
        }
    }
    __syncthreads();
    const int64_t frow0 = (int64_t)blockIdx.x * FL * 16, grp0 = (int64_t)blockIdx.y * SG;
    for (int idx = threadIdx.x; idx < FL * 16 * SG; idx += FL * SG) {
        const int row = idx / SG, w = idx % SG;
        const int64_t f = frow0 + row, byte0 = (grp0 + w) * 8;
        if (f >= features || byte0 >= row_bytes) continue;
        const uint64_t word = tile[(row % 16) * FL + row / 16][w];
        uint8_t *dst = out + f * row_bytes + byte0;
        const int64_t nbytes = row_bytes - byte0 < 8 ? row_bytes - byte0 : 8;
        if (nbytes == 8 && (row_bytes & 7) == 0) {
            __builtin_nontemporal_store(word, reinterpret_cast<uint64_t *>(dst));
        } else {
            for (int k = 0; k < nbytes; ++k) dst[k] = (uint8_t)(word >> (8 * k));
        }
    }
}

// The same for any feature count and alignment, and for batches too small to fill the GPU with 64 samples per thread: lane =
// sample.  A wavefront reads 64 bytes of 64 consecutive rows (16 bytes per lane and load, at any alignment), and the
// comparison of one byte in all lanes IS the feature's word, which lane f keeps; SG wavefronts of consecutive sample groups then write
// runs of 8 SG bytes of every feature row.  Tiles that are neighbours along the features share lines of the input, so every
// XCD takes a contiguous run of them ([20000, 3000]: 33 -> 22 us).  Bound by latency where there is little to read
// (bool [10000, 784]: 18.5 us by tiles of 64 samples per thread, 5.9 here; [10000, 785], a byte at a time: 43, 6.2) and by the reads
// of 64-byte pieces where there is much (3 TB/s).
template <int SG>
__global__ __launch_bounds__(SG *kWave) void pack_bits_ballot_kernel(const uint8_t *__restrict__ t, uint8_t *__restrict__ out, int64_t features,
                                                                    int64_t batch, int64_t row_bytes, unsigned feature_blocks, unsigned per_xcd,
                                                                    unsigned tiles)
{
    constexpr int F = 64;
    __shared__ uint64_t tile[F][SG + 1];
    const int lane = threadIdx.x & (kWave - 1), sg = uniform((int)(threadIdx.x >> 6));
    const unsigned at = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;  // workgroups go round the XCDs
    if (at >= tiles) return;
    const int64_t f0 = (int64_t)(at % feature_blocks) * F, grp0 = (int64_t)(at / feature_blocks) * SG;
    const int64_t s = (grp0 + sg) * 64 + lane;
    const int count = features - f0 < F ? (int)(features - f0) : F;   // features of this workgroup
    u32x4 v[F / 16];
#pragma unroll
    for (int i = 0; i < F / 16; ++i) v[i] = (u32x4)0u;
    if (s < batch) {
        const uint8_t *p = t + s * features + f0;
#pragma unroll
        for (int i = 0; i < F / 16; ++i) {
            if (16 * i + 16 <= count) {                               // uniform
                __builtin_memcpy(&v[i], p + 16 * i, 16);
            } else {
#pragma unroll
                for (int b = 0; b < 16; ++b)
                    if (16 * i + b < count) v[i][b / 4] |= (uint32_t)p[16 * i + b] << (8 * (b % 4));
            }
        }
    }
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const uint64_t word = __ballot((v[f / 16][(f % 16) / 4] & (0xFFu << (8 * (f % 4)))) != 0);
        lo = lane == f ? (uint32_t)word : lo;
        hi = lane == f ? (uint32_t)(word >> 32) : hi;
    }
    tile[lane][sg] = ((uint64_t)hi << 32) | lo;
    __syncthreads();
    const int64_t byte0 = grp0 * 8, run = row_bytes - byte0 < 8 * SG ? row_bytes - byte0 : 8 * SG;
    if ((row_bytes & 3) == 0 && ((uintptr_t)out & 3) == 0) {          // runs of whole 4-byte pieces
        for (int i = threadIdx.x; i < F * 2 * SG; i += SG * kWave) {
            const int f = i / (2 * SG), piece = i % (2 * SG);
            if (f >= count || 4 * piece >= run) continue;
            const uint32_t bits = (uint32_t)(tile[f][piece / 2] >> (32 * (piece % 2)));
            *reinterpret_cast<uint32_t *>(out + (f0 + f) * row_bytes + byte0 + 4 * piece) = bits;
        }
    } else {
        for (int i = threadIdx.x; i < F * 8 * SG; i += SG * kWave) {
            const int f = i / (8 * SG), b = i % (8 * SG);
            if (f < count && b < run) out[(f0 + f) * row_bytes + byte0 + b] = (uint8_t)(tile[f][b / 8] >> (8 * (b % 8)));
        }
    }
}

template <int V, int G>
void launch_pack_smv(const uint8_t *t, void *words, int64_t features, int64_t batch, int64_t row_bytes, int64_t groups, hipStream_t st)
{
    hipLaunchKernelGGL((pack_bits_smv_kernel<V, G>), dim3((unsigned)clg_ceil_div(features / (4 * V), 256), (unsigned)clg_ceil_div(groups, G)),
                       dim3(256), 0, st, t, (uint8_t *)words, features, batch, row_bytes);
}

// ---------------------------------------------------------------------------------------------
// per-class bit counts
// ---------------------------------------------------------------------------------------------
// Lanes run along columns of type V (8-, 4- or 1-byte pieces of a row, whatever the row length and alignment allow) and,
// where a row is narrower than a wavefront or its column blocks would not fill the GPU, along rows as well: lane =
// (row phase, column), C columns x 64/C phases.  A workgroup owns C columns of one class (and one row slice); its wavefronts
// split the rows.  Every thread counts the bit positions of its column with vertical counters (plane p holds bit p of the
// running counts): four words are combined by three carry-save adders and the resulting "fours" word ripples into planes 2
// and up.  The row phases of a wavefront are added as binary numbers through lane shuffles, the wavefronts through LDS, and
// every wavefront expands its share of the bit positions into counts: no atomics and no zero fill unless a class is sliced.
// Wide rows are bound by their reads: 5.1 TB/s on [64000, 1024] 8-byte words (103 us); narrow ones by the additions of the
// counters.  Rows that are not whole 8-byte words, or shorter than 512 bytes, used to take one wavefront per 8-byte column
// that read them byte by byte and met the others in atomics: [8000, 313] 4-byte words 279 -> 7.7 us, [8000, 1251] bytes
// 281 -> 10 us, [10240, 4] 8-byte words 10.6 -> 6.4 us (the zero fill in front of the atomics included).
constexpr int kCountPlanes = 14;                                     // a workgroup counts at most 2^14 - 8 rows
template <typename V>
__device__ __forceinline__ void csa(V &hi, V &lo, V a, V b, V c)
{
    const V u = a ^ b;
    hi = (a & b) | (u & c);
    lo = u ^ c;
}
template <typename V>
__device__ __forceinline__ void count8(V (&plane)[kCountPlanes], const V (&w)[8])
{
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        V two_a, two_b, four;
        csa(two_a, plane[0], plane[0], w[4 * h], w[4 * h + 1]);
        csa(two_b, plane[0], plane[0], w[4 * h + 2], w[4 * h + 3]);
        csa(four, plane[1], plane[1], two_a, two_b);
#pragma unroll
        for (int q = 2; q < kCountPlanes; ++q) {
            const V t = plane[q] & four;
            plane[q] ^= four;
            four = t;
        }
    }
}
// plane += other, both binary numbers spread over the planes (a total above 2^14 - 1 cannot occur: the host keeps the rows of
// a workgroup below that)
template <typename V>
__device__ __forceinline__ void add_planes(V (&plane)[kCountPlanes], const V (&other)[kCountPlanes])
{
    V carry = 0;
#pragma unroll
    for (int q = 0; q < kCountPlanes; ++q) {
        const V b = other[q], u = plane[q] ^ b;
        const V c = (plane[q] & b) | (u & carry);
        plane[q] = u ^ carry;
        carry = c;
    }
}
__device__ __forceinline__ uint64_t shuffle_down(uint64_t v, int by)
{
    return ((uint64_t)(uint32_t)__shfl_down((int)(uint32_t)(v >> 32), by) << 32) | (uint32_t)__shfl_down((int)(uint32_t)v, by);
}
__device__ __forceinline__ uint32_t shuffle_down(uint32_t v, int by) { return (uint32_t)__shfl_down((int)v, by); }

// Classes of few rows: a wavefront per class and 8 bytes of its rows, lane = sample bit, so that nothing has to meet.  (The counters'
// additions above cost as much for one row as for a hundred: 100000 classes of one 8-byte word 758 us in place of 35, 10000
// classes of one row of four 74 in place of 21.)
__global__ __launch_bounds__(256) void group_bit_sum_few_kernel(const uint8_t *__restrict__ x, int32_t *__restrict__ out, int class_rows,
                                                              int64_t row_bytes, int64_t samples, int64_t k, int64_t cols8)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t item = (int64_t)blockIdx.x * 4 + uniform((int)(threadIdx.x >> 6));
    if (item >= k * cols8) return;
    const int64_t g = item / cols8, col = item - g * cols8, s = col * 64 + lane;
    if (s >= samples) return;                                         // (its byte may lie behind the row)
    const uint8_t *p = x + g * class_rows * row_bytes + (s >> 3);
    int32_t acc = 0;
    int r = 0;
    for (; r + 8 <= class_rows; r += 8, p += 8 * row_bytes) {
        uint32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[j * row_bytes];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += (v[j] >> (lane & 7)) & 1;
    }
    for (; r < class_rows; ++r, p += row_bytes) acc += (*p >> (lane & 7)) & 1;
    out[s * k + g] = acc;
}

// S: the stored piece of a row, V: the register it is counted in.  cols_log2: log2 of C.
template <typename S, typename V, int WAVES>
__global__ __launch_bounds__(WAVES *kWave) void group_bit_sum_columns_kernel(const S *__restrict__ x, int32_t *__restrict__ out,
                                                                            int64_t class_rows, int64_t row_pieces, int64_t samples,
                                                                            int k, int slices, int cols_log2, unsigned col_blocks)
{
    __shared__ V meet[WAVES][kCountPlanes][kWave];
    constexpr int kBits = 8 * (int)sizeof(S);
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    const int cols = 1 << cols_log2, phases = kWave >> cols_log2, phase = lane >> cols_log2;
    const int g = (int)(blockIdx.x / col_blocks);
    const int64_t col0 = (int64_t)(blockIdx.x - g * col_blocks) << cols_log2, col = col0 + (lane & (cols - 1));
    const int part = blockIdx.y * WAVES + wave, parts = slices * WAVES;
    const int64_t r0 = class_rows * part / parts, r1 = class_rows * (part + 1) / parts;
    const S *base = x + (int64_t)g * class_rows * row_pieces + (col < row_pieces ? col : row_pieces - 1);
    V plane[kCountPlanes];
#pragma unroll
    for (int q = 0; q < kCountPlanes; ++q) plane[q] = 0;
    // eight rows of the lane's phase per step, the next eight in flight while these are counted
    const int64_t row_step = row_pieces << (6 - cols_log2), step = 8ll << (6 - cols_log2);
    const S *p = base + (r0 + phase) * row_pieces;
    int64_t r = r0;
    if (r + step <= r1) {                                            // uniform over the wavefront
        V cur[8], nxt[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) cur[j] = (V)p[j * row_step];
        for (r += step; r + step <= r1; r += step) {
            p += 8 * row_step;
#pragma unroll
            for (int j = 0; j < 8; ++j) nxt[j] = (V)p[j * row_step];
            count8(plane, cur);
#pragma unroll
            for (int j = 0; j < 8; ++j) cur[j] = nxt[j];
        }
        count8(plane, cur);
    }
    if (r < r1) {                                                    // last, partial step: a row past the end is read from the last one and counts as zero
        V w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t at = r + phase + (int64_t)j * phases;
            w[j] = (V)base[(at < r1 ? at : r1 - 1) * row_pieces];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = r + phase + (int64_t)j * phases < r1 ? w[j] : (V)0;
        count8(plane, w);
    }
    for (int by = kWave / 2; by >= cols; by >>= 1) {                  // row phases: the first C lanes end up with the wavefront's counts
        V other[kCountPlanes];
#pragma unroll
        for (int q = 0; q < kCountPlanes; ++q) other[q] = shuffle_down(plane[q], by);
        add_planes(plane, other);
    }
#pragma unroll
    for (int q = 0; q < kCountPlanes; ++q) meet[wave][q][lane] = plane[q];
    __syncthreads();
    // thread e of the workgroup takes bit position e / C of column e % C
    const int c = threadIdx.x & (cols - 1);
    V total[kCountPlanes];
#pragma unroll
    for (int q = 0; q < kCountPlanes; ++q) total[q] = meet[0][q][c];
    for (int wv = 1; wv < WAVES; ++wv) {
        V other[kCountPlanes];
#pragma unroll
        for (int q = 0; q < kCountPlanes; ++q) other[q] = meet[wv][q][c];
        add_planes(total, other);
    }
    if (col0 + c >= row_pieces) return;
    for (int b = threadIdx.x >> cols_log2; b < kBits; b += (WAVES * kWave) >> cols_log2) {
        const int64_t s = (col0 + c) * kBits + b;
        if (s >= samples) break;
        int32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < kCountPlanes; ++q) cnt |= (int32_t)((total[q] >> b) & 1) << q;
        if (slices == 1) out[s * k + g] = cnt;
        else atomicAdd(out + s * k + g, cnt);
    }
}

__global__ void fill_zero_i32_kernel(int32_t *p, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0;
}

int small_grid(int64_t items, int block)
{
    const int64_t g = clg_ceil_div(items, block);
    return (int)(g < 1 ? 1 : (g > 65536 * 16 ? 65536 * 16 : g));
}

template <typename V, bool LOGITS>
void launch_eval(const void *x, const int64_t *a, const int64_t *b, const void *gate, void *y, int64_t out_dim,
                 int64_t row_bytes, hipStream_t st, int64_t in_dim)
{
    const int64_t row_vecs = row_bytes / (int64_t)sizeof(V);
    // column chunks of at most 4 KiB per row: both uses of a row segment fall inside one chunk pass,
    // so the working set of a pass (in_dim x 4 KiB) can stay in the last-level cache (measured best on
    // 64000 x 8 KiB rows among 0.5..8 KiB).  CLG_EVAL_CHUNK_BYTES / CLG_EVAL_NPW override for tuning.
    const char *e_chunk = clg_knob(K_EVAL_CHUNK_BYTES), *e_npw = clg_knob(K_EVAL_NPW);
    const int max_chunk_vecs = (e_chunk ? atoi(e_chunk) : 4096) / (int)sizeof(V);
    const int chunk_vecs = row_vecs < max_chunk_vecs ? (int)row_vecs : max_chunk_vecs;
    const int chunks = (int)clg_ceil_div(row_vecs, chunk_vecs);
    const int neurons_per_wave = e_npw ? atoi(e_npw) : 1;
    const int groups = (int)clg_ceil_div(out_dim, (int64_t)kEvalWaves * neurons_per_wave);
    hipLaunchKernelGGL((eval_packed_kernel<V, 2, LOGITS>), dim3((unsigned)(chunks * groups)), dim3(kEvalBlock), 0, st, (const V *)x, a,
                       b, gate, (V *)y, (int)out_dim, row_vecs, chunk_vecs, groups, neurons_per_wave, in_dim);
}

template <bool LOGITS>
void launch_rows(const void *x, const int64_t *a, const int64_t *b, const void *gate, void *y, int64_t out_dim, int64_t row_bytes, hipStream_t st,
                 int64_t in_dim)
{
    const uint32_t pieces = (uint32_t)clg_ceil_div(row_bytes, 16);
    const int nj = (int)std::max<int64_t>(1, std::min<int64_t>(kRowsMax, kRowsUnroll * kEvalBlock / pieces));
    const int64_t parts = nj > 1 ? 1 : clg_ceil_div(pieces, kRowsUnroll * kEvalBlock);
    const uint32_t per = (uint32_t)clg_ceil_div((int64_t)nj * pieces, parts);
    // (a launch is fewer than 2^32 threads; parts < 2^21, of 2^30 pieces)
    const int64_t most = ((1 << 24) - 1) / parts * nj;
    for (int64_t j = 0; j < out_dim; j += most) {
        const int64_t some = std::min(most, out_dim - j), groups = clg_ceil_div(some, nj);
        const void *gates = reinterpret_cast<const uint8_t *>(gate) + j * (LOGITS ? 64 : 1);
        hipLaunchKernelGGL(eval_packed_rows_kernel<LOGITS>, dim3((unsigned)(groups * parts)), dim3(kEvalBlock), 0, st, (const uint8_t *)x, a + j, b + j,
                           gates, (uint8_t *)y + j * row_bytes, (int)some, row_bytes, pieces, make_fastdiv(pieces), nj, make_fastdiv((uint32_t)groups), per,
                           in_dim);
    }
}

// Layers whose rows are read once along a walk of the wiring (the others twice, but all at once): us at [neurons] x bytes, lanes along several neurons' rows
// against the walk: [8000] x 3000 11.5 and 12.4, x 5000 18.5 and 17.3, [16000] x 1528 11.8 and 12.2, [32000] x 1020 15.9 and 15.3,
// [64000] x 500 17.0 and 17.5, x 768 22.3 and 20.7, [16000] x 8188 56 and 49; below 30 MB a wavefront's chain of eight neurons is what a walk takes
// ([2000] x 1280 3.9 and 7.3, [100] x 256 KiB 12.0 and 13.2, [20] x 512 KiB 5.0 and 8.7), on rows of 1 MiB and more below 20 MB ([28] x 1 MiB 14.1 and 9.9, [10] x
// 2 MiB 10.6 and 8.9, [4] x 1 MiB 3.7 and 5.3).
bool walk_pays(int64_t row_bytes, int64_t out_dim)
{
    if (const char *e = clg_knob(K_EVAL_ROWS)) return atoi(e) == 0;
    return row_bytes >= 640 && row_bytes * out_dim >= (row_bytes >= 1 << 20 ? 20'000'000 : 30'000'000);
}
// Vectors of a lane in the walk, whose grid holds 65535 column chunks of them: 268 MB of a row
int walk_vecs(int64_t row_vecs)
{
    const char *e = clg_knob(K_EVAL_WALK_R);
    int R = e ? atoi(e) : 4;
    while (R > 1 && (int64_t)kWave * (R / 2) >= row_vecs) R /= 2;
    return R;
}
constexpr int64_t kWalkChunks = 65535;
bool walk_takes(int64_t row_bytes, int64_t out_dim)
{
    const int64_t row_vecs = clg_ceil_div(row_bytes, 16);
    return row_bytes >= 16 && walk_pays(row_bytes, out_dim) && clg_ceil_div(row_vecs, (int64_t)kWave * walk_vecs(row_vecs)) <= kWalkChunks;
}

bool valid_elem(int e) { return e == 1 || e == 2 || e == 4 || e == 8; }

}  // namespace

// LOGITS: `gate` holds float32 logits; rows below 16 bytes, and from 2^34 on, must then be whole 4-byte words at 4-byte aligned addresses
template <bool LOGITS>
static int eval_packed(const char *name, int elem_size, const void *x, const int64_t *a, const int64_t *b, const void *gate, void *y,
                       int64_t in_dim, int64_t out_dim, int64_t words, void *stream)
{
    CLG_REQUIRE(valid_elem(elem_size), "%s: elem_size must be 1, 2, 4 or 8, got %d", name, elem_size);
    CLG_REQUIRE(x && a && b && gate && y, "%s: null pointer argument", name);
    CLG_REQUIRE(x != y, "%s: x and y must not overlap", name);
    CLG_REQUIRE(in_dim > 0 && out_dim > 0 && words > 0, "%s: in_dim, out_dim and words must be positive", name);
    CLG_REQUIRE(out_dim < (1ll << 31), "%s: out_dim above 2^31-1 is not supported", name);
    const int64_t row_bytes = words * elem_size;
    const uintptr_t align = (uintptr_t)x | (uintptr_t)y | (uintptr_t)row_bytes;
    hipStream_t st = clg_stream(stream);
    const int64_t blocks_needed = clg_ceil_div(row_bytes, 2048) * clg_ceil_div(out_dim, 16);
    CLG_REQUIRE(blocks_needed < (1ll << 31), "%s: problem too large for one launch (%lld blocks)", name, (long long)blocks_needed);
    // without a plan, rows of whole vectors go a wavefront per neuron and 4 KiB from 1 MiB on ([10] x 2 MiB 8.4 us, 11.4 by pieces, [10] x 16 MiB 57.7 and 62.4, [100] x
    // 4 MiB 165 and 172, [50] x 4 MiB 84.7 and 84.6; shorter ones [64000] x 8192 214.8 and 213.1, [500] x 64 KiB 16.1 and 15.1)
    const bool whole = (align & 15) == 0 && row_bytes >= 1 << 20;
    if (row_bytes >= 16 && row_bytes < (1ll << 34) && !whole) launch_rows<LOGITS>(x, a, b, gate, y, out_dim, row_bytes, st, in_dim);
    else if ((align & 15) == 0) launch_eval<u32x4, LOGITS>(x, a, b, gate, y, out_dim, row_bytes, st, in_dim);
    else if ((align & 3) == 0) launch_eval<uint32_t, LOGITS>(x, a, b, gate, y, out_dim, row_bytes, st, in_dim);
    else if constexpr (LOGITS)
        CLG_REQUIRE(false, "%s: rows must be whole 4-byte words at 4-byte aligned addresses; use clg_gate_argmax + clg_fc_eval_packed "
                    "otherwise", name);
    else
        hipLaunchKernelGGL(eval_packed_bytes_kernel, dim3(small_grid(out_dim * row_bytes, 256)), dim3(256), 0, st,
                           (const uint8_t *)x, a, b, (const uint8_t *)gate, (uint8_t *)y, out_dim, row_bytes, in_dim);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_fc_eval_packed(int elem_size, const void *x, const int64_t *a, const int64_t *b, const uint8_t *gate,
                                  void *y, int64_t in_dim, int64_t out_dim, int64_t words, void *stream)
{
    return eval_packed<false>("clg_fc_eval_packed", elem_size, x, a, b, gate, y, in_dim, out_dim, words, stream);
}

extern "C" int clg_fc_eval_packed_logits(int elem_size, const void *x, const int64_t *a, const int64_t *b, const float *logits,
                                         void *y, int64_t in_dim, int64_t out_dim, int64_t words, void *stream)
{
    CLG_REQUIRE((((uintptr_t)x | (uintptr_t)y | (uintptr_t)(words * elem_size)) & 3) == 0, "clg_fc_eval_packed_logits: rows must be whole 4-byte words at "
                "4-byte aligned addresses; use clg_gate_argmax + clg_fc_eval_packed otherwise");
    return eval_packed<true>("clg_fc_eval_packed_logits", elem_size, x, a, b, logits, y, in_dim, out_dim, words, stream);
}

static int check_pack(const void *t, void *words, int64_t features, int64_t batch, int bit_count, const char *name)
{
    CLG_REQUIRE(t && words, "%s: null pointer argument", name);
    CLG_REQUIRE(bit_count == 8 || bit_count == 16 || bit_count == 32 || bit_count == 64,
                "%s: `bit_count` has to be in { 8, 16, 32, 64 }, got %d", name, bit_count);
    CLG_REQUIRE(features > 0 && batch > 0, "%s: features and batch must be positive", name);
    return CLG_OK;
}

extern "C" int clg_pack_bits(const uint8_t *t, void *words, int64_t features, int64_t batch, int bit_count, void *stream)
{
    if (int e = check_pack(t, words, features, batch, bit_count, "clg_pack_bits")) return e;
    const int64_t row_bytes = clg_ceil_div(batch, bit_count) * (bit_count / 8);
    const bool aligned8 = (batch % 8 == 0) && (((uintptr_t)t & 7) == 0);
    hipLaunchKernelGGL(pack_bits_kernel, dim3(small_grid(features * row_bytes, 256)), dim3(256), 0, clg_stream(stream), t,
                       (uint8_t *)words, features, batch, row_bytes, aligned8);
    CLG_CHECK_LAUNCH("clg_pack_bits");
    return CLG_OK;
}

extern "C" int clg_pack_bits_sample_major(const uint8_t *t, void *words, int64_t features, int64_t batch, int bit_count,
                                          void *stream)
{
    if (int e = check_pack(t, words, features, batch, bit_count, "clg_pack_bits_sample_major")) return e;
    const int64_t row_bytes = clg_ceil_div(batch, bit_count) * (bit_count / 8);
    const int64_t groups = clg_ceil_div(batch, 64);
    // Large batches of 16-byte aligned rows: 16 features x 64 samples per thread, the words through LDS from 8 groups on (bool
    // [8192, 64000]: 155 us with direct stores, 121; CLG_PACK_TILE=0 keeps the direct stores).  What does not give these
    // kernels enough threads, or has rows that are not whole 8-byte words, is faster by ballots.  The lines, tile against
    // ballot: 67 MB as [65536, 1024] 19.0 and 20.5 us, 60 MB as [20000, 2992] 27 and 20 (rows of 4-byte words: 78 MB 34 and
    // 24, 157 MB 46 and 43), 32 MB as [2000, 16000] 14.7 and 12.2; direct stores against ballot: [128, 500000] 22 and 26,
    // [200, 200000] 20 and 15, [64, 200000] 8.5 and 12.
    const int64_t bytes = features * batch;
    const char *e_tile = clg_knob(K_PACK_TILE);
    const bool vectors = features % 16 == 0 && ((uintptr_t)t & 15) == 0 && ((uintptr_t)words & 7) == 0 && groups <= 65535;
    CLG_REQUIRE(vectors || groups <= 65535ll * kPackGroups, "clg_pack_bits_sample_major: batch above %lld samples is not supported",
                65535ll * kPackGroups * 64);
    const bool large = groups >= 8 ? bytes >= ((row_bytes & 7) == 0 ? 48ll << 20 : 160ll << 20)
                                   : bytes >= 48ll << 20 || (groups == 1 && features > 98304);
    if (vectors && (e_tile || large)) {
        const bool tiled = !e_tile || atoi(e_tile) != 0;
        // 32 feature lanes x 16 groups: 101 -> 52 us on [65536, 4096] (512 threads; 16 x 16 and 64 x 8 are 8 % slower)
        if (tiled && groups >= 16)
            hipLaunchKernelGGL((pack_bits_tile_kernel<32, 16>), dim3((unsigned)clg_ceil_div(features, 32 * 16), (unsigned)clg_ceil_div(groups, 16)),
                               dim3(512), 0, clg_stream(stream), t, (uint8_t *)words, features, batch, row_bytes);
        else if (tiled && groups >= 8)
            hipLaunchKernelGGL((pack_bits_tile_kernel<32, 8>), dim3((unsigned)clg_ceil_div(features, 32 * 16), (unsigned)clg_ceil_div(groups, 8)),
                               dim3(256), 0, clg_stream(stream), t, (uint8_t *)words, features, batch, row_bytes);
        else
            launch_pack_smv<4, 2>(t, words, features, batch, row_bytes, groups, clg_stream(stream));
    } else if (!vectors && groups <= 4 && features >= 32768) {
        // few groups of very many features fill the GPU with a thread per feature ([64, 95233]: 4.1 us, 7.3 by ballots)
        hipLaunchKernelGGL(pack_bits_sm_kernel, dim3((unsigned)clg_ceil_div(features, 256), (unsigned)clg_ceil_div(groups, kPackGroups)), dim3(256), 0,
                           clg_stream(stream), t, (uint8_t *)words, features, batch, row_bytes);
    } else {
        // eight groups per workgroup where there are plenty ([65536, 4097]: 155 us with four, 142; [10000, 784]: 5.9 and 6.7)
        const bool wide = bytes >= 96ll << 20;
        const int64_t feature_blocks = clg_ceil_div(features, 64), tiles = feature_blocks * clg_ceil_div(groups, wide ? 8 : 4), per_xcd = clg_ceil_div(tiles, 8);
        CLG_REQUIRE(tiles < (1ll << 28), "clg_pack_bits_sample_major: problem too large for one launch");
        const dim3 grid((unsigned)(8 * per_xcd));
        if (wide)
            hipLaunchKernelGGL((pack_bits_ballot_kernel<8>), grid, dim3(8 * kWave), 0, clg_stream(stream), t, (uint8_t *)words, features, batch,
                               row_bytes, (unsigned)feature_blocks, (unsigned)per_xcd, (unsigned)tiles);
        else
            hipLaunchKernelGGL((pack_bits_ballot_kernel<4>), grid, dim3(4 * kWave), 0, clg_stream(stream), t, (uint8_t *)words, features, batch,
                               row_bytes, (unsigned)feature_blocks, (unsigned)per_xcd, (unsigned)tiles);
    }
    CLG_CHECK_LAUNCH("clg_pack_bits_sample_major");
    return CLG_OK;
}

extern "C" int clg_group_bit_sum(int elem_size, const void *x, int32_t *out, int64_t features, int64_t words, int64_t pad_len,
                                 int64_t k, void *stream)
{
    CLG_REQUIRE(valid_elem(elem_size), "clg_group_bit_sum: elem_size must be 1, 2, 4 or 8, got %d", elem_size);
    CLG_REQUIRE(x && out, "clg_group_bit_sum: null pointer argument");
    CLG_REQUIRE(features > 0 && words > 0 && k > 0, "clg_group_bit_sum: features, words and k must be positive");
    CLG_REQUIRE(features % k == 0, "in_dim (%lld) has to be divisible by k (%lld) but it is not", (long long)features, (long long)k);
    const int64_t row_bytes = words * elem_size, samples = row_bytes * 8 - pad_len;
    CLG_REQUIRE(pad_len >= 0 && samples > 0, "clg_group_bit_sum: pad_len %lld leaves no samples", (long long)pad_len);
    CLG_REQUIRE(k < (1 << 20), "clg_group_bit_sum: k too large");
    const int64_t class_rows = features / k;
    hipStream_t st = clg_stream(stream);
    const uintptr_t align = (uintptr_t)x | (uintptr_t)row_bytes;
    const int piece = (align & 7) == 0 ? 8 : ((align & 3) == 0 ? 4 : 1);
    const int64_t pieces = row_bytes / piece, cols8 = clg_ceil_div(row_bytes, 8);
    // A wavefront per class and 8 bytes: up to 96 rows where the GPU is not filled by them (0.4 to 1.0 times the time of the counters, at
    // 256 rows 1.1 to 1.7 times), up to 128 or 256 where there are few columns (0.02 to 0.9), else up to 24 (0.4 to 1.0; at 64
    // 1.0 to 1.4).  Not for full GPUs of wide 8-byte rows, which the counters read 512 bytes at a time (0.8 to 1.6), unless there
    // are so many classes that what counts is the writes (0.5 to 1.1).
    const int64_t rows_max = cols8 == 1 ? (piece == 8 || k >= 1000 ? 256 : 128)
                                        : (cols8 <= 4 && piece == 8 ? 128 : (cols8 <= 8 || k * cols8 <= 4096 ? 96 : 0));
    const bool by_bit = class_rows <= rows_max || (class_rows <= 24 && (cols8 < 64 || piece == 4)) ||
                        (class_rows <= 8 && k >= 8192) || (piece == 1 && class_rows <= (cols8 < 512 ? 24 : 2));
    if (by_bit && !clg_knob(K_GSUM_SLICES)) {
        CLG_REQUIRE(clg_ceil_div(k * cols8, 4) < (1ll << 31), "clg_group_bit_sum: problem too large for one launch");
        hipLaunchKernelGGL(group_bit_sum_few_kernel, dim3((unsigned)clg_ceil_div(k * cols8, 4)), dim3(256), 0, st, (const uint8_t *)x, out,
                           (int)class_rows, row_bytes, samples, k, cols8);
        CLG_CHECK_LAUNCH("clg_group_bit_sum");
        return CLG_OK;
    }
    // Columns per workgroup: a whole wavefront of them where that gives half of the CUs a workgroup (64 lanes x 8 bytes = 512
    // contiguous bytes of a row: 103 us at [64000, 1024] 8-byte words, 135 with 32 columns), fewer -- and more row phases --
    // where it does not, as long as the columns make 64-byte runs ([81920, 64]: 95 us with 64 columns, 22 with 8), and never
    // more than the row has.
    int cols_log2 = 6;
    while (cols_log2 > 0 && (1ll << (cols_log2 - 1)) >= pieces) --cols_log2;
    while (((int64_t)piece << (cols_log2 - 1)) >= 64 && clg_ceil_div(pieces, 1ll << cols_log2) * k < 128) --cols_log2;
    const int64_t col_blocks = clg_ceil_div(pieces, 1ll << cols_log2);
    // One workgroup takes all rows of its columns and class (measured 101 us against 164 us with two row slices at 64000 x
    // 1024 8-byte words); rows are sliced only beyond the counter range of 2^14 - 8 rows per workgroup.
    const char *e_sl = clg_knob(K_GSUM_SLICES);
    int64_t slices = e_sl ? atoi(e_sl) : 1;
    if (slices > class_rows / 512) slices = class_rows / 512;
    const int64_t need = clg_ceil_div(class_rows, (1 << kCountPlanes) - 8);
    if (slices < need) slices = need;
    if (slices < 1) slices = 1;
    CLG_REQUIRE(slices <= 65535 && col_blocks * k < (1ll << 31), "clg_group_bit_sum: problem too large for one launch");
    if (slices > 1)
        hipLaunchKernelGGL(fill_zero_i32_kernel, dim3(small_grid(samples * k, 256)), dim3(256), 0, st, out, samples * k);
    const dim3 grid((unsigned)(col_blocks * k), (unsigned)slices);
#define CLG_COUNT(S, V, WAVES)                                                                                              \
    hipLaunchKernelGGL((group_bit_sum_columns_kernel<S, V, WAVES>), grid, dim3(WAVES * kWave), 0, st, (const S *)x, out, class_rows, \
                       pieces, samples, (int)k, (int)slices, cols_log2, (unsigned)col_blocks)
    // four wavefronts where eight would get less than two steps of rows each (the counters' additions at the end are then most
    // of the work: [10240, 4] 8-byte words 9.2 -> 7.3 us)
    const bool few = class_rows < (128ll << (6 - cols_log2));
    if (piece == 8) {
        if (few) CLG_COUNT(uint64_t, uint64_t, 4);
        else CLG_COUNT(uint64_t, uint64_t, 8);
    } else if (piece == 4) {
        if (few) CLG_COUNT(uint32_t, uint32_t, 4);
        else CLG_COUNT(uint32_t, uint32_t, 8);
    } else {
        CLG_COUNT(uint8_t, uint32_t, 8);
    }
#undef CLG_COUNT
    CLG_CHECK_LAUNCH("clg_group_bit_sum");
    return CLG_OK;
}

// ---- walk plan (host side) --------------------------------------------------------------------
extern "C" int clg_fc_eval_plan(const int64_t *a, const int64_t *b, int64_t in_dim, int64_t out_dim, int32_t *plan)
{
    CLG_REQUIRE(a && b && plan, "clg_fc_eval_plan: null pointer argument");
    CLG_REQUIRE(in_dim > 0 && out_dim > 0 && out_dim < (1ll << 28), "clg_fc_eval_plan: out_dim must be in 1..2^28-1");
    // adjacency: edges (neurons) incident to each vertex (input row); a self-paired neuron is listed twice
    int64_t *start = (int64_t *)calloc((size_t)in_dim + 1, sizeof(int64_t));
    int32_t *adj = (int32_t *)malloc((size_t)out_dim * 2 * sizeof(int32_t));
    int64_t *fill = (int64_t *)malloc((size_t)in_dim * sizeof(int64_t));
    uint8_t *used = (uint8_t *)calloc((size_t)out_dim, 1);
    if (!start || !adj || !fill || !used) {
        free(start); free(adj); free(fill); free(used);
        clg_set_error("clg_fc_eval_plan: out of host memory");
        return CLG_EINVAL;
    }
    for (int64_t j = 0; j < out_dim; ++j) {
        if (a[j] < 0 || a[j] >= in_dim || b[j] < 0 || b[j] >= in_dim) {
            free(start); free(adj); free(fill); free(used);
            clg_set_error("clg_fc_eval_plan: neuron %lld is wired to a feature outside 0..%lld", (long long)j, (long long)in_dim - 1);
            return CLG_EINVAL;
        }
        ++start[a[j] + 1];
        ++start[b[j] + 1];
    }
    for (int64_t v = 0; v < in_dim; ++v) start[v + 1] += start[v];
    for (int64_t v = 0; v < in_dim; ++v) fill[v] = start[v];
    for (int64_t j = 0; j < out_dim; ++j) {
        adj[fill[a[j]]++] = (int32_t)j;
        adj[fill[b[j]]++] = (int32_t)j;
    }
    for (int64_t v = 0; v < in_dim; ++v) fill[v] = start[v];       // now: scan position per vertex
    int64_t n = 0;
    // trails start at odd-degree vertices first (pass 0), then anywhere edges remain (pass 1)
    for (int pass = 0; pass < 2; ++pass) {
        for (int64_t v0 = 0; v0 < in_dim; ++v0) {
            if (pass == 0 && ((start[v0 + 1] - start[v0]) & 1) == 0) continue;
            int64_t v = v0;
            bool carried = false;
            for (;;) {
                while (fill[v] < start[v + 1] && used[adj[fill[v]]]) ++fill[v];
                if (fill[v] == start[v + 1]) break;
                const int32_t e = adj[fill[v]++];
                used[e] = 1;
                const int64_t other = a[e] == v ? b[e] : a[e];
                int use = 0;
                if (carried) use = (a[e] == v ? 1 : 0) | (b[e] == v ? 2 : 0);
                const int keep = other == b[e] ? 1 : 0;
                plan[n++] = e | (use << 28) | (keep << 30);
                v = other;
                carried = true;
            }
        }
    }
    free(start); free(adj); free(fill); free(used);
    CLG_REQUIRE(n == out_dim, "clg_fc_eval_plan: internal error, %lld of %lld neurons placed", (long long)n, (long long)out_dim);
    return CLG_OK;
}

namespace {
// rows that clg_fc_eval_packed_planned_logits promises to take: whole 16-byte vectors at 16-byte aligned addresses, at least 1 KiB long.  (The
// kernels behind it take any; clg_fc_eval_packed_layer lets them.)
bool walk_fits(int elem_size, const void *x, const void *y, int64_t words)
{
    const int64_t row_bytes = words * elem_size;
    const uintptr_t align = (uintptr_t)x | (uintptr_t)y | (uintptr_t)row_bytes;
    return (align & 15) == 0 && row_bytes >= 1024;
}

template <bool LOGITS>
int launch_walk(const char *name, int elem_size, const void *x, const int64_t *a, const int64_t *b, const void *gate, const int32_t *plan,
                void *y, int64_t in_dim, int64_t out_dim, int64_t words, void *stream)
{
    const int64_t row_bytes = words * elem_size, row_vecs = clg_ceil_div(row_bytes, 16);
    const char *e_l = clg_knob(K_EVAL_WALK_SEG);
    const int R = walk_vecs(row_vecs);
    const int seg = e_l ? atoi(e_l) : 8;
    const int64_t col_chunks = clg_ceil_div(row_vecs, (int64_t)kWave * R);
    CLG_REQUIRE(col_chunks <= kWalkChunks, "%s: rows above %lld bytes are not supported", name, (long long)kWalkChunks * kWave * R * 16);
    const dim3 grid((unsigned)clg_ceil_div(out_dim, (int64_t)kEvalWaves * seg), (unsigned)col_chunks), block(kEvalBlock);
    hipStream_t st = clg_stream(stream);
#define CLG_WALK(RR)                                                                                                          \
    hipLaunchKernelGGL((eval_packed_walk_kernel<RR, LOGITS>), grid, block, 0, st, (const uint8_t *)x, a, b, gate, plan, (uint8_t *)y, \
                       (int)out_dim, seg, row_vecs, row_bytes, in_dim)
    switch (R) {
    case 1: CLG_WALK(1); break;
    case 2: CLG_WALK(2); break;
    case 4: CLG_WALK(4); break;
    default: CLG_WALK(8); break;
    }
#undef CLG_WALK
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

}  // namespace

extern "C" int clg_fc_eval_packed_planned(int elem_size, const void *x, const int64_t *a, const int64_t *b, const uint8_t *gate,
                                          const int32_t *plan, void *y, int64_t in_dim, int64_t out_dim, int64_t words,
                                          void *stream)
{
    const char *name = "clg_fc_eval_packed_planned";
    CLG_REQUIRE(valid_elem(elem_size), "%s: elem_size must be 1, 2, 4 or 8, got %d", name, elem_size);
    CLG_REQUIRE(x && a && b && gate && plan && y, "%s: null pointer argument", name);
    CLG_REQUIRE(x != y, "%s: x and y must not overlap", name);
    CLG_REQUIRE(in_dim > 0 && out_dim > 0 && words > 0, "%s: in_dim, out_dim and words must be positive", name);
    CLG_REQUIRE(out_dim < (1ll << 28), "%s: out_dim above 2^28-1 is not supported", name);
    if (!walk_takes(words * elem_size, out_dim)) return clg_fc_eval_packed(elem_size, x, a, b, gate, y, in_dim, out_dim, words, stream);
    return launch_walk<false>(name, elem_size, x, a, b, gate, plan, y, in_dim, out_dim, words, stream);
}

extern "C" int clg_fc_eval_walk_fits(int elem_size, const void *x, const void *y, int64_t words)
{
    return valid_elem(elem_size) && x && y && words > 0 && walk_fits(elem_size, x, y, words) ? 1 : 0;
}

static int eval_packed_layer(const char *name, int elem_size, const void *x, const int64_t *a, const int64_t *b, const float *logits, const int32_t *plan,
                             void *y, int64_t in_dim, int64_t out_dim, int64_t words, void *stream, bool whole_vectors)
{
    CLG_REQUIRE(valid_elem(elem_size), "%s: elem_size must be 1, 2, 4 or 8, got %d", name, elem_size);
    CLG_REQUIRE(x && a && b && logits && plan && y, "%s: null pointer argument", name);
    CLG_REQUIRE(x != y, "%s: x and y must not overlap", name);
    CLG_REQUIRE(in_dim > 0 && out_dim > 0 && words > 0, "%s: in_dim, out_dim and words must be positive", name);
    CLG_REQUIRE(out_dim < (1ll << 28), "%s: out_dim above 2^28-1 is not supported", name);
    CLG_REQUIRE(!whole_vectors || walk_fits(elem_size, x, y, words), "%s: rows must be whole 16-byte vectors of at least 1 KiB at 16-byte aligned addresses "
                "(clg_fc_eval_walk_fits); use clg_gate_argmax + clg_fc_eval_packed_planned otherwise", name);
    const int64_t row_bytes = words * elem_size;
    CLG_REQUIRE(row_bytes >= 16 || (((uintptr_t)x | (uintptr_t)y | (uintptr_t)row_bytes) & 3) == 0, "%s: rows must be 16 bytes or more, or whole 4-byte words at "
                "4-byte aligned addresses; use clg_gate_argmax + clg_fc_eval_packed otherwise", name);
    if (walk_takes(row_bytes, out_dim)) return launch_walk<true>(name, elem_size, x, a, b, logits, plan, y, in_dim, out_dim, words, stream);
    return eval_packed<true>(name, elem_size, x, a, b, logits, y, in_dim, out_dim, words, stream);
}

extern "C" int clg_fc_eval_packed_planned_logits(int elem_size, const void *x, const int64_t *a, const int64_t *b, const float *logits,
                                                 const int32_t *plan, void *y, int64_t in_dim, int64_t out_dim, int64_t words,
                                                 void *stream)
{
    return eval_packed_layer("clg_fc_eval_packed_planned_logits", elem_size, x, a, b, logits, plan, y, in_dim, out_dim, words, stream, true);
}

extern "C" int clg_fc_eval_packed_layer(int elem_size, const void *x, const int64_t *a, const int64_t *b, const float *logits, const int32_t *plan, void *y,
                                        int64_t in_dim, int64_t out_dim, int64_t words, void *stream)
{
    return eval_packed_layer("clg_fc_eval_packed_layer", elem_size, x, a, b, logits, plan, y, in_dim, out_dim, words, stream, false);
}
