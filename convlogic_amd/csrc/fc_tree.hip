// The fully connected end of a logic network as ONE operation: a LogicLayer, two halving LogicLayers (2 out_dim = in_dim, every
// input read by exactly one neuron operand) and the GroupSum behind them (src/convlogic/model.py:49-57,102-107).
//
// Where every neuron of the first two layers is read exactly once, neuron j of the third layer is the root of a tree of
// seven gates -- four of the first layer, two of the second, itself -- over eight rows of the input, and no other root
// shares any of them.  So the three layers need no activations of their own: a wavefront reads the eight rows of a root,
// evaluates the tree in registers and adds the root's value to its class.
//   forward           8 row reads per root instead of 8 + 4 writes + 4 reads + 2 + 2 + 1 + 1 (and the GroupSum's pass)
//   backward          the tree again; the gradient of the root's row is grad_out[b][class] / tau; the 28 coefficient sums
//                     give the gradients of the seven neurons' logits, and the gradients of the eight operands go out as
//                     rows of a buffer ordered by input feature, so that
//   input gradient    is a sum of consecutive rows per feature: no wiring, no gather, no atomics, fixed order
//   packed inference  the same tree on 64 samples per word (three bit operations per gate and 32 samples), the class counts
//                     in vertical counters
// Measured, first layer to class sums (kernels of the four modules -> here): forward 36 -> 21 us and backward 58 -> 43 us on 4096
// features, 40960 / 20480 / 10240 neurons, batch 256; 1.31 -> 0.50 ms and 2.19 -> 1.63 ms on 131072 features, 2.62 M / 1.31 M /
// 655 k neurons, batch 128; packed inference of the former at 65 536 samples 273 -> 78 us.
// What bounds it: the row reads (2.7 GB of 512-byte pieces through L2 and the last-level cache in 375 us on the large shape) and,
// backward, the 2.7 GB of operand gradients written once and read once.  Keeping the first layer's output gradient instead (half
// the bytes to write) needs a gather that reads every row twice plus the other operand's row: 1133 us in place of the
// 536 us of the sum over consecutive rows.
// Activations are feature-major with a row pitch; samples from `batch` up to the pitch are computed like any other, carry no
// gradient and are not written to the result.
#include <algorithm>

#include "conv_ops.h"
#include "fc_tree.h"
#include "net_step.h"

int clg_convblock_check(const clg_conv_geom *gg, Geom *g, int dtype, const char *name);

namespace {

constexpr int kTreeWaves = 4;
constexpr int kTreeBlock = kTreeWaves * kWave;

// the samples of a lane: 1, 2 or 4 consecutive ones, so that a row of 64, 128 or 256 samples fills the wavefront and the
// root -- indices, coefficients, class -- is uniform (two roots per wavefront on rows of 128 samples need their 28
// coefficients per lane: 168 registers in the backward kernel against 115)
template <int V>
struct Samples {
    float v[V];
};
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
template <int V>
struct SamplesRaw;
template <>
struct SamplesRaw<1> { using type = float; };
template <>
struct SamplesRaw<2> { using type = f32x2u; };
template <>
struct SamplesRaw<4> { using type = f32x4u; };
template <int V, bool STREAM = false>
__device__ __forceinline__ Samples<V> load_samples(const float *p)
{
    return __builtin_bit_cast(Samples<V>, load_vec<STREAM>(reinterpret_cast<const typename SamplesRaw<V>::type *>(p)));
}
template <int V, bool STREAM = false>
__device__ __forceinline__ void store_samples(float *p, const Samples<V> &v)
{
    store_vec<STREAM>(reinterpret_cast<typename SamplesRaw<V>::type *>(p), __builtin_bit_cast(typename SamplesRaw<V>::type, v));
}
// Where the lane whose samples begin at s reads and writes: the last lane of a row whose length V does not divide steps back to the
// last V samples, which it shares with its neighbour (the same values, computed twice); lanes behind the row: 0.
template <int V>
__device__ __forceinline__ int64_t samples_at(int64_t s, int64_t pitch)
{
    return s >= pitch ? 0 : (s + V <= pitch ? s : pitch - V);
}

// ---- the trees of a wiring ----------------------------------------------------------------------------------------------
// a / b of the three layers; start / flat: the lists input feature -> neurons of the first layer, increasing in every list, the
// first operand before the second where a neuron reads a feature twice.
struct TreeWiring {
    const int64_t *a[3], *b[3], *start, *flat;
};
__global__ __launch_bounds__(256) void fc_tree_no_slots_kernel(int32_t *__restrict__ slot, int64_t n)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) slot[e] = -1;
}
// Eight lanes per root, one operand each.  An operand's place in the lists is found by bisection of its feature's list, so nothing is
// sorted: 5 us at 10240 roots and 0.6 ms at 655360, once per wiring, in place of some twenty launches of torch's (index
// arithmetic and a stable sort of 8 roots keys): first training pass of the k = 32 networks 1915 -> 1451 and 2005 -> 1759 us.  A neuron that no
// operand reads keeps slot -1: the wiring makes no trees.
__global__ __launch_bounds__(256) void fc_tree_plan_kernel(TreeWiring w, int32_t *__restrict__ rows, int32_t *__restrict__ pos,
                                                         int32_t *__restrict__ ids, int32_t *__restrict__ slot, int64_t in_dim, int roots)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x, operands = (int64_t)roots * 8;
    if (e >= operands) return;
    const int j = (int)(e >> 3), q = (int)(e & 7), leaf = q >> 1, mid = q >> 2;
    const int64_t n2 = clamp_index((mid ? w.b[2] : w.a[2])[j], 2 * (int64_t)roots);
    const int64_t n1 = clamp_index(((leaf & 1) ? w.b[1] : w.a[1])[n2], 4 * (int64_t)roots);
    const int64_t fa = clamp_index(w.a[0][n1], in_dim), fb = clamp_index(w.b[0][n1], in_dim), f = (q & 1) ? fb : fa;
    int64_t lo = clamp_index(w.start[f], operands + 1), hi = clamp_index(w.start[f + 1], operands + 1);
    while (lo < hi) {
        const int64_t at = (lo + hi) >> 1;
        if (w.flat[at] < n1) lo = at + 1;
        else hi = at;
    }
    rows[e] = (int32_t)f;
    pos[e] = (int32_t)lo + ((q & 1) && fa == fb);
    if ((q & 1) == 0) {
        ids[(int64_t)j * 8 + leaf] = (int32_t)n1;
        slot[n1] = j * 7 + leaf;
    }
    if ((q & 3) == 0) {
        ids[(int64_t)j * 8 + 4 + mid] = (int32_t)n2;
        ids[(int64_t)j * 8 + 6 + mid] = 0;
        slot[(int64_t)roots * 4 + n2] = j * 7 + 4 + mid;
    }
    if (q == 0) slot[(int64_t)roots * 6 + j] = j * 7 + 6;
}

// ---- coefficients ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ const float *tree_logits(const TreeLogits &lg, const int32_t *__restrict__ ids, int j, int q, int roots)
{
    return (q < 4 ? lg.l[0] : (q < 6 ? lg.l[1] : lg.l[2])) + tree_neuron(ids, j, q, roots) * 16;
}
__global__ __launch_bounds__(256) void fc_tree_fold_kernel(TreeFold f) { tree_fold(f, blockIdx.x); }
template <bool STREAM>
__global__ __launch_bounds__(256) void fc_tree_fold_slots_kernel(TreeFoldSlots f)
{
    tree_fold_slots<STREAM>(f, blockIdx.x);
}

// ---- forward ----------------------------------------------------------------------------------------------------------
// rows [roots][8]: the input rows of a tree.  A wavefront takes a root at a time, 64 lanes x V samples.
__device__ __forceinline__ void tree_coefs(const float *__restrict__ coef, int j, Tree<float> &t)
{
    const float4 *c = reinterpret_cast<const float4 *>(coef) + (int64_t)j * 7;
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        const float4 v = c[q];
        t.g[q] = Coef<float>{v.x, v.y, v.z, v.w};
    }
}
template <int V>
__device__ __forceinline__ void tree_rows(const float *__restrict__ x, const int32_t *__restrict__ rows, int j, int in_dim, int64_t pitch,
                                          int64_t s, Samples<V> (&v)[8])
{
    const int32_t *r = rows + (int64_t)j * 8;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = load_samples<V>(x + (int64_t)min((uint32_t)r[t], (uint32_t)in_dim - 1u) * pitch + s);
}

// grid: (slices of a class, classes, chunks of 64 V samples).  partial [slices][k][pitch]
template <int V>
__global__ __launch_bounds__(kTreeBlock) void fc_tree_forward_kernel(const float *__restrict__ x, const int32_t *__restrict__ rows,
                                                                   const float *__restrict__ coef, float *__restrict__ partial,
                                                                   int class_rows, int k, int slices, int64_t pitch, int in_dim)
{
    __shared__ Samples<V> meet[kTreeWaves][kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    const int slice = blockIdx.x, g = blockIdx.y;
    const int64_t s = ((int64_t)blockIdx.z * kWave + lane) * V, s_at = samples_at<V>(s, pitch);
    const int r0 = (int)((int64_t)class_rows * slice / slices), r1 = (int)((int64_t)class_rows * (slice + 1) / slices);
    Samples<V> acc = {};
    auto value = [&](int r, Samples<V> &y) {
        const int j = g * class_rows + r;
        Tree<float> t;
        tree_coefs(coef, j, t);
        Samples<V> v[8];
        tree_rows<V>(x, rows, j, in_dim, pitch, s_at, v);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            float tap[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) tap[q] = v[q].v[i];
            y.v[i] = eval_tree(t, tap).root;
        }
    };
    // four roots of the wavefront in flight; summed in the order of group_sum_fm_kernel
    int r = r0 + wave;
    for (; r + 12 < r1; r += 16) {
        Samples<V> y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) value(r + 4 * u, y[u]);
#pragma unroll
        for (int i = 0; i < V; ++i) acc.v[i] += (y[0].v[i] + y[1].v[i]) + (y[2].v[i] + y[3].v[i]);
    }
    for (; r < r1; r += 4) {
        Samples<V> y;
        value(r, y);
#pragma unroll
        for (int i = 0; i < V; ++i) acc.v[i] += y.v[i];
    }
    meet[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && s < pitch) {
        Samples<V> sum;
#pragma unroll
        for (int i = 0; i < V; ++i) sum.v[i] = (meet[0][lane].v[i] + meet[1][lane].v[i]) + (meet[2][lane].v[i] + meet[3][lane].v[i]);
        store_samples<V>(partial + ((int64_t)slice * k + g) * pitch + s_at, sum);
    }
}

// out[b][g] = inv_tau * sum over the slices in order, FLIGHT loads in flight
template <int FLIGHT>
__global__ __launch_bounds__(256) void fc_tree_finish_kernel(const float *__restrict__ partial, float *__restrict__ out, int slices, int k,
                                                           int64_t pitch, int64_t batch, float inv_tau)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;       // sample fastest: the loads of a wavefront are contiguous
    if (i >= batch * k) return;
    const int g = (int)(i / batch);
    const int64_t b = i - (int64_t)g * batch, step = (int64_t)k * pitch;
    const float *p = partial + (int64_t)g * pitch + b;
    float acc = 0.f;
    for (int s = 0; s < slices; s += FLIGHT) {
        float v[FLIGHT];
#pragma unroll
        for (int u = 0; u < FLIGHT; ++u) v[u] = p[(int64_t)min(s + u, slices - 1) * step];
#pragma unroll
        for (int u = 0; u < FLIGHT; ++u) acc = s + u < slices ? acc + v[u] : acc;
    }
    out[b * k + g] = acc * inv_tau;
}

// ---- backward -----------------------------------------------------------------------------------------------------------
// pos [roots][8]: the row of `rowgrad` an operand's gradient goes to: its place in the lists input feature -> operands.
// The 28 sums of a wavefront are reduced and turned round together: every exchange between lane groups halves the number of
// values a lane holds instead of repeating each value's full reduction (28 x 6 steps).  They leave as one run of 112 bytes per
// root; what remains -- 16 gates per neuron, the softmax backward -- needs the rows of seven scattered neurons and is a
// kernel of its own in neuron order (fc_tree_logit_grad_kernel): done here it held the wavefront for one more round trip and
// read and wrote 64-byte pieces all over (655360 roots x 128 samples: 1742 us, 978 without it).
// SUMS, ROWS: for the gradients of the logits, of the input (a frozen end and an input without a gradient need one of them).
template <int V, bool SUMS, bool ROWS, bool STREAM>
__global__ __launch_bounds__(kTreeBlock) void fc_tree_backward_kernel(const float *__restrict__ x, const int32_t *__restrict__ rows,
                                                                    const int32_t *__restrict__ pos, const float *__restrict__ coef,
                                                                    const float *__restrict__ grad_out,
                                                                    float *__restrict__ sums, float *__restrict__ rowgrad, int roots,
                                                                    int class_rows, int k, int64_t batch, int64_t pitch, int in_dim,
                                                                    float inv_tau)
{
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    const int64_t total_rows = (int64_t)roots * 8;
    for (int j = blockIdx.x * kTreeWaves + wave; j < roots; j += gridDim.x * kTreeWaves) {
        Tree<float> t;
        tree_coefs(coef, j, t);
        const int g = j / class_rows;
        const int32_t *pj = pos + (int64_t)j * 8;
        float acc[28];
#pragma unroll
        for (int q = 0; q < 28; ++q) acc[q] = 0.f;
        for (int64_t s0 = 0; s0 < pitch; s0 += kWave * V) {
            const int64_t s = s0 + lane * V;
            const bool live = s < pitch;
            Samples<V> v[8];
            tree_rows<V>(x, rows, j, in_dim, pitch, live ? s : 0, v);
            if (s0 + kWave * V > batch) {                             // values without a sample: zeros, whatever the row holds there
#pragma unroll
                for (int q = 0; q < 8; ++q) {
#pragma unroll
                    for (int i = 0; i < V; ++i) v[q].v[i] = s + i < batch ? v[q].v[i] : 0.f;
                }
            }
            float gy[V];
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const int64_t b = s + i;
                const float go = grad_out[(b < batch ? b : batch - 1) * k + g] * inv_tau;
                gy[i] = b < batch ? go : 0.f;
            }
#pragma unroll
            for (int i = 0; i < V; ++i) {
                float tap[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) tap[q] = v[q].v[i];
                const TreeVals<float> tv = eval_tree(t, tap);
                auto add = [&](int q, float gq, float a, float b) {
                    if constexpr (!SUMS) return;
                    const float ga = gq * a;
                    acc[4 * q] = fma_t(ga, b, acc[4 * q]);
                    acc[4 * q + 1] += ga;
                    acc[4 * q + 2] = fma_t(gq, b, acc[4 * q + 2]);
                    acc[4 * q + 3] += gq;
                };
                const float g6 = gy[i];
                add(6, g6, tv.mid[0], tv.mid[1]);
                const float gm[2] = {g6 * gate_da(t.g[6], tv.mid[1]), g6 * gate_db(t.g[6], tv.mid[0])};
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const float la = tv.leaf[2 * m], lb = tv.leaf[2 * m + 1];
                    add(4 + m, gm[m], la, lb);
                    const float gl[2] = {gm[m] * gate_da(t.g[4 + m], lb), gm[m] * gate_db(t.g[4 + m], la)};
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const int q = 2 * m + n;
                        add(q, gl[n], tap[2 * q], tap[2 * q + 1]);
                        v[2 * q].v[i] = gl[n] * gate_da(t.g[q], tap[2 * q + 1]);
                        v[2 * q + 1].v[i] = gl[n] * gate_db(t.g[q], tap[2 * q]);
                    }
                }
                // one sample at a time: interleaved, four samples take 169 registers, so 115
#pragma unroll
                for (int q = 0; q < 28; ++q) asm volatile("" : "+v"(acc[q]));
                if (i < V - 1) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) asm volatile("" : "+v"(v[q].v[i + 1]));
                }
            }
            if (ROWS && live) {
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    store_samples<V, STREAM>(rowgrad + (int64_t)min((uint64_t)(uint32_t)pj[q], (uint64_t)total_rows - 1) * pitch + s, v[q]);
            }
        }
        if constexpr (SUMS) {
            int at;
            const float sum = wave_sums28(acc, lane, at);
            if (at >= 0) sums[(int64_t)j * 28 + at] = sum;
        }
    }
}

template <bool STREAM>
__global__ __launch_bounds__(256) void fc_tree_logit_grad_kernel(TreeSums t, int64_t blocks)
{
    for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) tree_logit_grad<STREAM>(t, b);   // (28 lanes for each of 2^28 roots are no launch)
}

// gx[i] = sum of the rows start[i] .. start[i + 1] of rowgrad, eight in flight, four partial sums
template <int V, bool STREAM>
__global__ __launch_bounds__(kTreeBlock) void fc_tree_gather_kernel(const float *__restrict__ rowgrad, const int64_t *__restrict__ start,
                                                                  float *__restrict__ gx, int in_dim, int64_t pitch, int64_t total_rows)
{
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    const int i = blockIdx.x * kTreeWaves + wave;
    const int64_t s_lane = ((int64_t)blockIdx.y * kWave + lane) * V, s = samples_at<V>(s_lane, pitch);
    if (i >= in_dim || s_lane >= pitch) return;
    const int64_t beg = clamp_index(start[i], total_rows + 1), end = clamp_index(start[i + 1], total_rows + 1);
    Samples<V> part[4] = {};
    const float *p = rowgrad + beg * pitch + s;
    int64_t r = beg;
    for (; r + 8 <= end; r += 8, p += 8 * pitch) {
        Samples<V> v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load_samples<V, STREAM>(p + u * pitch);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int c = 0; c < V; ++c) part[u & 3].v[c] += v[u].v[c];
    }
    if (r < end) {
        Samples<V> v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load_samples<V, STREAM>(p + (r + u < end ? u : 0) * pitch);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int c = 0; c < V; ++c) part[u & 3].v[c] += r + u < end ? v[u].v[c] : 0.f;
    }
    Samples<V> sum;
#pragma unroll
    for (int c = 0; c < V; ++c) sum.v[c] = (part[0].v[c] + part[1].v[c]) + (part[2].v[c] + part[3].v[c]);
    store_samples<V>(gx + (int64_t)i * pitch + s, sum);
}

// The widest lanes that a row fills: a pass of 64 lanes x V samples over rows of up to 64, 128 and 256.  The kernels that only read rows and
// write whole sums take them for any row length (211 samples, 10 roots of 3200: forward 26.9 -> 23.4 us, input gradient 48.5 ->
// 32.8, in place of one sample per lane); the backward kernel, bound by the operand gradients that it writes, where V divides the row
// and the buffers are aligned (83 samples: 107 us with one sample per lane, 114 with two; 211: 77 and 75 with four).
int tree_vec(int64_t pitch) { return pitch <= 64 ? 1 : (pitch <= 128 ? 2 : 4); }
int tree_vec_dividing(int64_t pitch, const void *x, const void *rowgrad)
{
    const uintptr_t align = (uintptr_t)x | (uintptr_t)rowgrad | (uintptr_t)(pitch * 4);
    const int fit = tree_vec(pitch);
    return (align & 15) == 0 ? fit : ((align & 7) == 0 && fit > 1 ? 2 : 1);
}

// Row slices of a class, as clg_group_sum cuts them (a class sum of 65 536 values is rounded at 1e-7 of a logit in the
// thousands: the softmax of the loss then shows the order of the additions, so the order is kept).  Only one or two large classes of a
// small batch are cut into more slices than its 64, which would be the launch's only 64 or 128 workgroups.
int tree_slices(int64_t class_rows, int64_t batch, int64_t k)
{
    int64_t slices = clg_ceil_div(1024, clg_ceil_div(batch, (int64_t)kWave) * k);
    if (class_rows <= 4096) slices = 64;                              // small classes (where the GroupSum has another kernel): for the parallelism
    slices = std::min(slices, class_rows / (class_rows <= 4096 ? 16 : 64));
    return (int)std::min<int64_t>(512, std::max<int64_t>(1, slices));
}

}  // namespace

int clg_check_tree(const char *name, int64_t in_dim, int64_t roots, int64_t k)
{
    CLG_REQUIRE(in_dim > 0 && roots > 0 && k > 0 && roots % k == 0, "%s: in_dim, roots and k must be positive and k divide roots", name);
    CLG_REQUIRE(in_dim < (1ll << 31) && roots < (1ll << 28) && k <= 65535, "%s: in_dim below 2^31, roots below 2^28 and k up to 65535 only", name);
    return CLG_OK;
}

extern "C" int clg_fc_tree_plan(const int64_t *a0, const int64_t *b0, const int64_t *a1, const int64_t *b1, const int64_t *a2,
                                const int64_t *b2, const int64_t *start, const int64_t *flat, int32_t *rows, int32_t *pos, int32_t *ids,
                                int32_t *slot, int64_t in_dim, int64_t roots, void *stream)
{
    const char *name = "clg_fc_tree_plan";
    if (int e = clg_check_tree(name, in_dim, roots, 1)) return e;
    CLG_REQUIRE(a0 && b0 && a1 && b1 && a2 && b2 && start && flat && rows && pos && ids && slot, "%s: null pointer argument", name);
    const TreeWiring w = {{a0, a1, a2}, {b0, b1, b2}, start, flat};
    hipLaunchKernelGGL(fc_tree_no_slots_kernel, dim3((unsigned)clg_ceil_div(roots * 7, 256)), dim3(256), 0, clg_stream(stream), slot, roots * 7);
    CLG_CHECK_LAUNCH(name);
    hipLaunchKernelGGL(fc_tree_plan_kernel, dim3((unsigned)clg_ceil_div(roots * 8, 256)), dim3(256), 0, clg_stream(stream), w, rows, pos, ids,
                       slot, in_dim, (int)roots);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_fc_tree_fold(const float *logits0, const float *logits1, const float *logits2, const int32_t *ids, float *coef,
                                float *probs, int64_t roots, int hard, void *stream)
{
    const char *name = "clg_fc_tree_fold";
    if (int e = clg_check_tree(name, 1, roots, 1)) return e;
    CLG_REQUIRE(logits0 && logits1 && logits2 && ids && coef, "%s: null pointer argument", name);
    const TreeFold f = {{{logits0, logits1, logits2}}, ids, coef, probs, (int)roots, hard};
    hipLaunchKernelGGL(fc_tree_fold_kernel, dim3((unsigned)clg_ceil_div(roots * 7, 256)), dim3(256), 0, clg_stream(stream), f);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_fc_tree_fold_slots(const float *logits0, const float *logits1, const float *logits2, const int32_t *slot, float *coef, float *probs,
                                      int64_t roots, void *stream)
{
    const char *name = "clg_fc_tree_fold_slots";
    if (int e = clg_check_tree(name, 1, roots, 1)) return e;
    CLG_REQUIRE(logits0 && logits1 && logits2 && slot && coef, "%s: null pointer argument", name);
    const TreeFoldSlots f = {{{logits0, logits1, logits2}}, slot, coef, probs, {4 * roots, 6 * roots, 7 * roots}};
    const bool past = clg_past_caches(7 * roots * 64, 100);
    hipLaunchKernelGGL((past ? fc_tree_fold_slots_kernel<true> : fc_tree_fold_slots_kernel<false>), dim3((unsigned)clg_ceil_div(roots * 7, 256)), dim3(256), 0,
                       clg_stream(stream), f);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int64_t clg_fc_tree_partial_elems(int64_t roots, int64_t k, int64_t batch, int64_t pitch)
{
    if (roots <= 0 || k <= 0 || batch <= 0 || pitch < batch) return -1;
    return (int64_t)tree_slices(roots / k, batch, k) * k * pitch;
}

extern "C" int clg_fc_tree_forward(const float *x, const int32_t *rows, const float *coef, float *partial, float *out, int64_t in_dim,
                                   int64_t roots, int64_t k, int64_t batch, int64_t pitch, double tau, void *stream)
{
    const char *name = "clg_fc_tree_forward";
    if (int e = clg_check_tree(name, in_dim, roots, k)) return e;
    CLG_REQUIRE(x && rows && coef && partial && out, "%s: null pointer argument", name);
    CLG_REQUIRE(batch > 0 && pitch >= batch && pitch < (1ll << 28) && tau != 0.0, "%s: the row pitch must hold the batch, tau must not be zero",
                name);
    const int slices = tree_slices(roots / k, batch, k);
    int vec = tree_vec(pitch);                                        // fewer samples per lane where the launch would have less than four wavefronts per SIMD
    while (vec > 1 && (int64_t)slices * k * clg_ceil_div(pitch, (int64_t)kWave * vec) * kTreeWaves < 4096) vec /= 2;
    const dim3 grid((unsigned)slices, (unsigned)k, (unsigned)clg_ceil_div(pitch, (int64_t)kWave * vec));
    CLG_REQUIRE(grid.z <= 65535, "%s: batch too large", name);
    hipStream_t st = clg_stream(stream);
#define CLG_TREE_F(V)                                                                                                        \
    hipLaunchKernelGGL((fc_tree_forward_kernel<V>), grid, dim3(kTreeBlock), 0, st, x, rows, coef, partial, (int)(roots / k), (int)k, \
                       slices, pitch, (int)in_dim)
    if (vec == 1) CLG_TREE_F(1);
    else if (vec == 2) CLG_TREE_F(2);
    else CLG_TREE_F(4);
#undef CLG_TREE_F
    CLG_CHECK_LAUNCH(name);
#define CLG_TREE_S(FLIGHT)                                                                                                    \
    hipLaunchKernelGGL((fc_tree_finish_kernel<FLIGHT>), dim3((unsigned)clg_ceil_div(batch * k, 256)), dim3(256), 0, st, (const float *)partial, \
                       out, slices, (int)k, pitch, batch, 1.f / (float)tau)
    if (slices > 8) CLG_TREE_S(32);
    else CLG_TREE_S(8);
#undef CLG_TREE_S
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

static int tree_backward(const char *name, const float *x, const int32_t *rows, const int32_t *pos, const int32_t *slot, const float *coef,
                         const float *grad_out, const float *probs, float *grad0, float *grad1, float *grad2, float *rowgrad, float *sums,
                         const int64_t *start, float *grad_x, int64_t in_dim, int64_t roots, int64_t k, int64_t batch, int64_t pitch, double tau, void *stream_,
                         clg_late_sums *late)
{
    if (int e = clg_check_tree(name, in_dim, roots, k)) return e;
    const bool logits = grad0 || grad1 || grad2;
    CLG_REQUIRE(x && rows && coef && grad_out && (logits || grad_x), "%s: null pointer argument", name);
    CLG_REQUIRE(!logits || (slot && probs && sums), "%s: gradients of logits need slot, probs and sums", name);
    CLG_REQUIRE(!grad_x || (pos && rowgrad && start), "%s: the gradient of x needs pos, rowgrad and start", name);
    CLG_REQUIRE(batch > 0 && pitch >= batch && pitch < (1ll << 28) && tau != 0.0, "%s: the row pitch must hold the batch, tau must not be zero",
                name);
    const int vec = tree_vec_dividing(pitch, x, rowgrad), gvec = tree_vec(pitch);
    hipStream_t st = clg_stream(stream_);
    // Operand gradients: replayed step of the CIFAR topology, us through the caches and past them: 60 to 82 MB within 1 % but for 274 and 267 (k = 64, 128 images, 80 MB),
    // 94 MB 345 and 328, 100 MB 332 and 318, 125 MB 419 and 395, 160 MB 479 and 460, rows of 512 bytes 2.7 GB 4722 and 4550.  Pieces of lines at the ends of rows cost what that gives: rows of 400 bytes, MNIST
    // topology, 98 MB 229 and 232, 250 MB 519 and 495; of 508 bytes, which lanes write four at a time, 79 MB 194 and 216, of 804 294 MB 934 and 1002.
    const bool stream = pitch % 4 == 0 && clg_past_caches(roots * 8 * pitch * 4, pitch % 16 == 0 ? 48 : 200);
    const TreeGrads gr = {{grad0, grad1, grad2}, {4 * roots, 6 * roots, 7 * roots}};
    const dim3 grid((unsigned)clg_ceil_div(roots, kTreeWaves));
    const dim3 ggrid((unsigned)clg_ceil_div(in_dim, kTreeWaves), (unsigned)clg_ceil_div(pitch, (int64_t)kWave * gvec));
    CLG_REQUIRE(ggrid.y <= 65535, "%s: batch too large", name);
#define CLG_TREE_K(V, SUMS, ROWS)                                                                                                \
    hipLaunchKernelGGL((ROWS && stream ? fc_tree_backward_kernel<V, SUMS, ROWS, ROWS> : fc_tree_backward_kernel<V, SUMS, ROWS, false>), grid, \
                       dim3(kTreeBlock), 0, st, x, rows, pos, coef, grad_out, sums, rowgrad, \
                       (int)roots, (int)(roots / k), (int)k, batch, pitch, (int)in_dim, 1.f / (float)tau)
#define CLG_TREE_B(V)                                                                                                            \
    do {                                                                                                                         \
        if (logits && grad_x) CLG_TREE_K(V, true, true);                                                                         \
        else if (logits) CLG_TREE_K(V, true, false);                                                                             \
        else CLG_TREE_K(V, false, true);                                                                                         \
    } while (0)
#define CLG_TREE_G(V)                                                                                                            \
    hipLaunchKernelGGL((stream ? fc_tree_gather_kernel<V, true> : fc_tree_gather_kernel<V, false>), ggrid, dim3(kTreeBlock), 0, st, \
                       (const float *)rowgrad, start, grad_x, (int)in_dim, pitch, roots * 8)
    if (vec == 1) CLG_TREE_B(1);
    else if (vec == 2) CLG_TREE_B(2);
    else CLG_TREE_B(4);
    if (grad_x) {
        if (gvec == 1) CLG_TREE_G(1);
        else if (gvec == 2) CLG_TREE_G(2);
        else CLG_TREE_G(4);
    }
#undef CLG_TREE_G
#undef CLG_TREE_B
#undef CLG_TREE_K
    CLG_CHECK_LAUNCH(name);
    if (!logits) return CLG_OK;
    const TreeSums t = {gr, probs, sums, slot, 7 * roots};
    const int64_t blocks = clg_ceil_div(7 * roots * 4, 256);
    const bool stream_logits = clg_past_caches(7 * roots * 64, 100);
    if (late != nullptr && !stream_logits) {
        *late = clg_late(kLateTree, (int)blocks, t);
        return CLG_OK;
    }
    hipLaunchKernelGGL((stream_logits ? fc_tree_logit_grad_kernel<true> : fc_tree_logit_grad_kernel<false>), dim3((unsigned)std::min<int64_t>(blocks, 1 << 23)),
                       dim3(256), 0, st, t, blocks);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_fc_tree_backward(const float *x, const int32_t *rows, const int32_t *pos, const int32_t *slot, const float *coef,
                                    const float *grad_out, const float *probs, float *grad0, float *grad1, float *grad2, float *rowgrad,
                                    float *sums, const int64_t *start, float *grad_x, int64_t in_dim, int64_t roots, int64_t k, int64_t batch,
                                    int64_t pitch, double tau, void *stream)
{
    return tree_backward("clg_fc_tree_backward", x, rows, pos, slot, coef, grad_out, probs, grad0, grad1, grad2, rowgrad, sums, start, grad_x,
                         in_dim, roots, k, batch, pitch, tau, stream, nullptr);
}

extern "C" int clg_fc_tree_backward_late(const float *x, const int32_t *rows, const int32_t *pos, const int32_t *slot, const float *coef,
                                         const float *grad_out, const float *probs, float *grad0, float *grad1, float *grad2, float *rowgrad,
                                         float *sums, const int64_t *start, float *grad_x, int64_t in_dim, int64_t roots, int64_t k, int64_t batch,
                                         int64_t pitch, double tau, clg_late_sums *late, void *stream)
{
    CLG_REQUIRE(late, "clg_fc_tree_backward_late: null pointer argument");
    *late = {};
    return tree_backward("clg_fc_tree_backward_late", x, rows, pos, slot, coef, grad_out, probs, grad0, grad1, grad2, rowgrad, sums, start, grad_x,
                         in_dim, roots, k, batch, pitch, tau, stream, late);
}

// ---- packed inference ---------------------------------------------------------------------------------------------------
// x int64 words [in_dim, words], 64 samples per word.  codes [roots] = tree_code() of the arg-max gates: three bits per gate
// and the root's constant, so that a gate is three 3-input bit operations with one mask each.
//
// Lanes run along words and, where a row has fewer than 64, along roots as well (cols_log2: log2 of the words a workgroup
// takes); a lane counts the 64 bit positions of its word over its roots in vertical counters, the workgroup adds the counters
// as binary numbers and writes (or, with several slices of a class, atomically adds: integers, any order) the class counts.
// WIDE (64 words): the root is uniform, rows and masks come through the scalar cache.  Workgroups are numbered so that an XCD
// works on one block of 64 words at a time: in_dim x 512 bytes of input then stay in its L2.
// 4096 features, 10240 roots, 65 536 samples: 671 MB of row reads from L2 in 78 us = 8.6 TB/s (the three evaluation kernels and
// the counting kernel: 273 us).
namespace {

// The blocks in front of the trees: the same launch finds the gate ids of their kernels (in the workgroups from tree_blocks on), or the table
// of kernels and taps that a block's own kernel reads -- one launch for a network in place of one of 4 us per block and another of 2 to
// 4 us per table.  Four lanes per gate, 16 bytes each: a lane that read the 16 logits of a gate by itself waited for one
// after the other (75520 roots: 87 us, now 18).
constexpr int kMaxNetBlocks = 16;
struct NetBlock {
    const float *logits;
    const int32_t *sel;
    uint8_t *ids;                 // gate ids [c, 7], or
    int32_t *table;               // rows of conv_pair.h
    int end;                      // kernels up to and including the block's
    int plane, rs, odd, shift;    // of the table's offsets
    Geom geom;
};
struct NetGates {
    NetBlock block[kMaxNetBlocks];
    int blocks, tree_blocks;
};
// 32 lanes per kernel, four per gate; the kernel's eight taps are the first eight lanes'
__device__ __forceinline__ void net_kernel(const NetBlock &b, int64_t c, int lane)
{
    const int part = lane & 3, q = (lane >> 2) & 7, half = lane & 32, t = lane & 31;
    const int32_t tap = b.sel[c * 8 + (t & 7)];                       // (on its way while the gates are found)
    int id = 0;
    if (q < 7) id = argmax16_quad(reinterpret_cast<const f32x4u *>(b.logits + (c * 7 + q) * 16)[part]);
    if (b.table == nullptr) {
        if (q < 7 && part == 0) b.ids[c * 7 + q] = (uint8_t)id;
        return;
    }
    uint8_t gate[7];
#pragma unroll
    for (int u = 0; u < 7; ++u) gate[u] = (uint8_t)__shfl(id, half + 4 * u, kWave);
    const Tap tp = unpack_tap(tap, tap_limit(b.geom));
    const int ch0 = __shfl(tp.ch, half, kWave);
    const uint32_t differ = (uint32_t)(__ballot(tp.ch != ch0) >> half) & 0xFFu;
    const int ch1 = __shfl(tp.ch, half + (differ ? __builtin_ctz(differ) : 0), kWave);
    const bool wide = ((uint32_t)(__ballot(tp.ch != ch0 && tp.ch != ch1) >> half) & 0xFFu) != 0;
    int32_t *row = b.table + c * kPairTable;
    if (t < 8) row[4 + t] = pair_tap(b.plane, b.rs, b.odd, b.shift, tp.ch != ch0, tp.ry, tp.rx);
    if (t == 0) {
        row[0] = ch0;
        row[1] = wide ? -1 : ch1;
        row[2] = (int32_t)tree_code(gate);
        if (c == 0) *reinterpret_cast<Geom *>(b.table + (int64_t)b.geom.c * kPairTable) = b.geom;
    }
}
__global__ __launch_bounds__(256) void fc_tree_codes_kernel(TreeLogits lg, const int32_t *__restrict__ ids, uint32_t *__restrict__ codes,
                                                          int roots, int32_t *__restrict__ counts, int64_t n_counts, NetGates net)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t i = e; i < n_counts; i += (int64_t)gridDim.x * 256) counts[i] = 0;   // (for the counting kernel's atomics)
    const int part = threadIdx.x & 3;
    if ((int)blockIdx.x >= net.tree_blocks) {
        const int64_t at = (e - (int64_t)net.tree_blocks * 256) >> 5;
        int first = 0;
        for (int b = 0; b < net.blocks; ++b) {                        // (32 lanes together)
            if (at >= first && at < net.block[b].end) net_kernel(net.block[b], at - first, threadIdx.x & (kWave - 1));
            first = net.block[b].end;
        }
        return;
    }
    const int q = (threadIdx.x >> 2) & 7;                             // 32 lanes per root, four per gate
    for (int j0 = blockIdx.x * 8; j0 < roots; j0 += net.tree_blocks * 8) {
        const int j = j0 + (int)(threadIdx.x >> 5);
        int id = 0;
        if (j < roots && q < 7) id = argmax16_quad(reinterpret_cast<const f32x4u *>(tree_logits(lg, ids, j, q, roots))[part]);
        uint8_t gate[7];
#pragma unroll
        for (int t = 0; t < 7; ++t) gate[t] = (uint8_t)__shfl(id, (threadIdx.x & 32) + 4 * t, kWave);
        if (j < roots && q == 0 && part == 0) codes[j] = tree_code(gate);
    }
}

constexpr int kTreePlanes = 14;                                      // a workgroup takes at most 2^14 - 1 roots
__device__ __forceinline__ void carry_save(uint32_t &hi, uint32_t &lo, uint32_t a, uint32_t b, uint32_t c)
{
    const uint32_t u = a ^ b;
    hi = (a & b) | (u & c);
    lo = u ^ c;
}
__device__ __forceinline__ void add_counts(uint32_t (&plane)[kTreePlanes], const uint32_t (&other)[kTreePlanes])
{
    uint32_t carry = 0;
#pragma unroll
    for (int q = 0; q < kTreePlanes; ++q) {
        const uint32_t b = other[q], u = plane[q] ^ b, c = (plane[q] & b) | (u & carry);
        plane[q] = u ^ carry;
        carry = c;
    }
}

// Slices of a class meet in atomics on `out`, or, where the caller has room, in partial [slices][k][samples] that fc_tree_meet_kernel
// adds: 985 000 atomics of 52 slices were half of the time at 75520 roots and 1894 samples (97 us, now 23 and 5; 10240
// roots and 256 samples 14 -> 9 us).
template <bool WIDE, int WAVES>
__global__ __launch_bounds__(WAVES *kWave) void fc_tree_packed_kernel(const uint32_t *__restrict__ x, const int32_t *__restrict__ rows,
                                                                            const uint32_t *__restrict__ codes, int32_t *__restrict__ out,
                                                                            float *__restrict__ sums, float inv_tau, int32_t *__restrict__ partial,
                                                                            int class_rows, int k, int slices, uint32_t words,
                                                                            int64_t samples, int in_dim, int cols_log2, unsigned col_blocks)
{
    __shared__ uint32_t meet[WAVES][kTreePlanes][kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = uniform((int)(threadIdx.x >> 6));
    const int cols = WIDE ? kWave : 1 << cols_log2, phases = WIDE ? 1 : kWave >> cols_log2, phase = WIDE ? 0 : lane >> cols_log2;
    // block -> (class, slice, column block): eight column blocks at a time, one per XCD, over all classes and slices
    const unsigned per_cb = (unsigned)k * slices, group = blockIdx.x / (8 * per_cb), in_group = blockIdx.x - group * 8 * per_cb;
    const unsigned wide = min(8u, col_blocks - group * 8);           // column blocks of this group
    const unsigned cs = in_group / wide, cb = group * 8 + in_group % wide;
    const int g = (int)(cs / slices), slice = (int)(cs % slices);
    const uint32_t col0 = cb * cols, col = col0 + (lane & (cols - 1)), at = col < words ? col : words - 1;
    const int part = slice * WAVES + wave, parts = slices * WAVES;
    const int r0 = (int)((int64_t)class_rows * part / parts), r1 = (int)((int64_t)class_rows * (part + 1) / parts);
    uint32_t plane[kTreePlanes];
#pragma unroll
    for (int q = 0; q < kTreePlanes; ++q) plane[q] = 0;
    for (int r = r0; r < r1; r += 4 * phases) {                      // four roots of a lane per step
        uint32_t w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int rr = r + phase + u * phases;
            const bool ok = rr < r1;
            int j = g * class_rows + (ok ? rr : r1 - 1);
            if constexpr (WIDE) j = uniform(j);
            const int32_t *row = rows + (int64_t)j * 8;
            uint32_t v[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = x[(uint64_t)min((uint32_t)row[t], (uint32_t)in_dim - 1u) * words + at];
            const BitOpsAnf::Params pr = BitOpsAnf::unpack(codes[j]);
            uint32_t leaf[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) leaf[q] = BitOpsAnf::gate32(pr, q, v[2 * q], v[2 * q + 1]);
            const uint32_t y = BitOpsAnf::gate32(pr, 6, BitOpsAnf::gate32(pr, 4, leaf[0], leaf[1]), BitOpsAnf::gate32(pr, 5, leaf[2], leaf[3]));
            w[u] = ok ? y ^ pr.inv : 0;
        }
        uint32_t two_a, two_b, four;
        carry_save(two_a, plane[0], plane[0], w[0], w[1]);
        carry_save(two_b, plane[0], plane[0], w[2], w[3]);
        carry_save(four, plane[1], plane[1], two_a, two_b);
#pragma unroll
        for (int q = 2; q < kTreePlanes; ++q) {
            const uint32_t t = plane[q] & four;
            plane[q] ^= four;
            four = t;
        }
    }
    if constexpr (!WIDE) {
        for (int by = kWave / 2; by >= cols; by >>= 1) {             // root phases: the first lanes end up with the wavefront's counts
            uint32_t other[kTreePlanes];
#pragma unroll
            for (int q = 0; q < kTreePlanes; ++q) other[q] = (uint32_t)__shfl_down((int)plane[q], by);
            add_counts(plane, other);
        }
    }
#pragma unroll
    for (int q = 0; q < kTreePlanes; ++q) meet[wave][q][lane] = plane[q];
    __syncthreads();
    // the wavefronts' counts in two rounds: wavefront w < 4 adds every fourth of them, then a thread per column those four
    if constexpr (WAVES > 4) {
        if (wave < 4) {
            for (int wv = 4; wv < WAVES; wv += 4) {
                uint32_t other[kTreePlanes];
#pragma unroll
                for (int q = 0; q < kTreePlanes; ++q) other[q] = meet[wave + wv][q][lane];
                add_counts(plane, other);
            }
#pragma unroll
            for (int q = 0; q < kTreePlanes; ++q) meet[wave][q][lane] = plane[q];
        }
        __syncthreads();
    }
    if (wave == 0) {
#pragma unroll
        for (int wv = 1; wv < 4; ++wv) {
            uint32_t other[kTreePlanes];
#pragma unroll
            for (int q = 0; q < kTreePlanes; ++q) other[q] = meet[wv][q][lane];
            add_counts(plane, other);
        }
#pragma unroll
        for (int q = 0; q < kTreePlanes; ++q) meet[0][q][lane] = plane[q];
    }
    __syncthreads();
    // consecutive threads take consecutive samples
    const int b = threadIdx.x & 31;
    for (int c = threadIdx.x >> 5; c < cols; c += WAVES * 2) {
        const int64_t s = (int64_t)(col0 + c) * 32 + b;
        if (s >= samples) break;                                      // (so is every later one; columns past the row as well)
        int32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < kTreePlanes; ++q) cnt |= (int32_t)((meet[0][q][c] >> b) & 1) << q;
        if (partial != nullptr) partial[((int64_t)slice * k + g) * samples + s] = cnt;
        else if (slices > 1) atomicAdd(out + s * k + g, cnt);
        else if (sums != nullptr) sums[s * k + g] = (float)cnt * inv_tau;
        else out[s * k + g] = cnt;
    }
}

// out or sums [samples][k] = sum over the slices of partial [slices][k][samples]
__global__ __launch_bounds__(256) void fc_tree_meet_kernel(const int32_t *__restrict__ partial, int32_t *__restrict__ out, float *__restrict__ sums,
                                                         int slices, int k, int64_t samples, float inv_tau)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x, n = samples * k;
    if (e >= n) return;
    const int64_t g = e / samples, s = e - g * samples;
    int32_t cnt = 0;
    int i = 0;
    for (; i + 8 <= slices; i += 8) {
        int32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = partial[(i + u) * n + e];
#pragma unroll
        for (int u = 0; u < 8; ++u) cnt += v[u];
    }
    for (; i < slices; ++i) cnt += partial[i * n + e];
    if (sums != nullptr) sums[s * k + g] = (float)cnt * inv_tau;
    else out[s * k + g] = cnt;
}

// How a launch is cut: columns of 32-bit words per workgroup, slices of a class, wavefronts of a workgroup
struct PackedCut {
    int cols_log2, waves;
    int64_t col_blocks, slices;
};
// meet: the slices meet in a partial buffer, not in atomics
PackedCut cut_packed(int64_t roots, int64_t k, int64_t words, bool meet)
{
    const int64_t class_rows = roots / k, halves = words * 2;        // 32-bit words of a row: a lane takes one
    PackedCut c;
    c.cols_log2 = 6;
    while (c.cols_log2 > 0 && (1ll << (c.cols_log2 - 1)) >= halves) --c.cols_log2;
    c.col_blocks = clg_ceil_div(halves, 1ll << c.cols_log2);
    // One workgroup takes all roots of its columns and class where that gives half of the CUs one; else the classes are sliced
    // down to two steps of roots per wavefront, two workgroups per CU (what LDS holds of them).  (Twelve slices of a class at 65 536
    // samples: 7.9 M atomics, 385 us instead of 66.)  A workgroup takes at most 2^14 - 4 roots.
    const int64_t phases = 64 >> c.cols_log2, per_slice = k * c.col_blocks;
    c.waves = 16;
    int64_t slices = per_slice >= 128 ? 1 : (meet ? 512 / per_slice : clg_ceil_div(512, per_slice));
    slices = std::min(slices, class_rows / (8 * phases * c.waves));
    if (meet && std::max<int64_t>(slices, 1) * per_slice < 64) {      // small classes: workgroups of four wavefronts, one step each
        c.waves = 4;
        slices = std::min<int64_t>(512 / per_slice, class_rows / (4 * phases * c.waves));
    }
    c.slices = std::max<int64_t>(std::max<int64_t>(slices, clg_ceil_div(class_rows, (1 << kTreePlanes) - 4)), 1);
    return c;
}

// counts (int32) or sums (float, counts / tau) of packed words; partial: room for slices x k x samples, or null
int count_packed(const char *name, const int64_t *x, const int32_t *rows, const uint32_t *codes, int32_t *counts, float *sums, float inv_tau,
                 int32_t *partial, int64_t in_dim, int64_t roots, int64_t k, int64_t words, int64_t samples, const PackedCut &c, hipStream_t st)
{
    if (c.slices == 1) partial = nullptr;
#define CLG_TREE_P(WIDE, WAVES)                                                                                               \
    hipLaunchKernelGGL((fc_tree_packed_kernel<WIDE, WAVES>), dim3((unsigned)(k * c.slices * c.col_blocks)), dim3(WAVES * kWave), 0, st, \
                       (const uint32_t *)x, rows, codes, counts, sums, inv_tau, partial, (int)(roots / k), (int)k, (int)c.slices, \
                       (uint32_t)(words * 2), samples, (int)in_dim, c.cols_log2, (unsigned)c.col_blocks)
    if (c.waves == 4 && c.cols_log2 == 6) CLG_TREE_P(true, 4);
    else if (c.waves == 4) CLG_TREE_P(false, 4);
    else if (c.cols_log2 == 6) CLG_TREE_P(true, 16);
    else CLG_TREE_P(false, 16);
#undef CLG_TREE_P
    CLG_CHECK_LAUNCH(name);
    if (partial != nullptr) {
        hipLaunchKernelGGL(fc_tree_meet_kernel, dim3((unsigned)clg_ceil_div(samples * k, 256)), dim3(256), 0, st, (const int32_t *)partial, counts,
                           sums, (int)c.slices, (int)k, samples, inv_tau);
        CLG_CHECK_LAUNCH(name);
    }
    return CLG_OK;
}

int make_codes(const char *name, const TreeLogits &lg, const int32_t *ids, uint32_t *codes, int64_t roots, int32_t *counts, int64_t n_counts,
               NetGates &net, hipStream_t st)
{
    // 2^18 workgroups fill the GPU many times over; a launch of 32 lanes for each of 2^27 roots would be of more threads than there can be
    net.tree_blocks = (int)std::min<int64_t>(clg_ceil_div(roots * 32, 256), 1 << 18);
    const int64_t gate_blocks = net.blocks ? clg_ceil_div((int64_t)net.block[net.blocks - 1].end * 32, 256) : 0;
    hipLaunchKernelGGL(fc_tree_codes_kernel, dim3((unsigned)(net.tree_blocks + gate_blocks)), dim3(256), 0, st, lg, ids, codes, (int)roots,
                       counts, n_counts, net);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

int check_packed(const char *name, int64_t k, int64_t words, const PackedCut &c)
{
    CLG_REQUIRE(k * c.slices * c.col_blocks < (1ll << 28) && words < (1ll << 30), "%s: problem too large for one launch", name);
    return CLG_OK;
}

}  // namespace

extern "C" int clg_fc_tree_packed(const int64_t *x, const int32_t *rows, const int32_t *ids, const float *logits0, const float *logits1,
                                  const float *logits2, uint32_t *codes, int32_t *out, int64_t in_dim, int64_t roots, int64_t k,
                                  int64_t words, int64_t samples, void *stream)
{
    const char *name = "clg_fc_tree_packed";
    if (int e = clg_check_tree(name, in_dim, roots, k)) return e;
    CLG_REQUIRE(x && rows && ids && logits0 && logits1 && logits2 && codes && out, "%s: null pointer argument", name);
    CLG_REQUIRE(words > 0 && samples > 0 && samples <= words * 64 && words < (1ll << 31), "%s: words %lld, samples %lld", name,
                (long long)words, (long long)samples);
    const PackedCut c = cut_packed(roots, k, words, false);
    if (int e = check_packed(name, k, words, c)) return e;
    hipStream_t st = clg_stream(stream);
    const TreeLogits lg = {{logits0, logits1, logits2}};
    NetGates none{};
    if (int e = make_codes(name, lg, ids, codes, roots, out, c.slices > 1 ? samples * k : (int64_t)0, none, st)) return e;
    return count_packed(name, x, rows, codes, out, nullptr, 0.f, nullptr, in_dim, roots, k, words, samples, c, st);
}

// ---- a whole network on packed words -----------------------------------------------------------------------------------------
// Blocks, flattening and trees in one call: the launches of the modules without the host's work between them, and the gate ids
// of all blocks and trees in one launch.
namespace {

size_t net_up(size_t v) { return (v + 255) & ~(size_t)255; }
struct NetLayout {
    size_t gates_off[kMaxNetBlocks], codes_off, partial_off, ping_off, pong_off, ws_off, total;
};

// a block's geometry in a network and, where it is staged two planes at a time, its plan; the last one writes its words feature-major
int net_pair(const char *name, const clg_packed_block *blocks, int n_blocks, int b, Geom *g, PairPlan *p, bool *pair)
{
    if (int e = clg_convblock_check(&blocks[b].geom, g, CLG_F64, name)) return e;
    g->y_fm = b == n_blocks - 1 ? 1 : 0;
    *pair = clg_packed_pair(*g, p);
    if (!*pair) g->y_fm = 0;
    return CLG_OK;
}

// checks the blocks against each other and lays the scratch out: gate ids or tables | codes | slices' counts | two activations | a block's scratch
int net_layout(const char *name, const clg_packed_block *blocks, int n_blocks, int64_t in_dim, int64_t roots, int64_t k, int64_t samples,
               NetLayout *l)
{
    CLG_REQUIRE(blocks && n_blocks > 0 && n_blocks <= kMaxNetBlocks, "%s: 1 to %d blocks", name, kMaxNetBlocks);
    size_t at = 0, act[2] = {0, 0}, ws = 0;
    int64_t c = 0, h = 0, w = 0;
    for (int b = 0; b < n_blocks; ++b) {
        const clg_conv_geom &gg = blocks[b].geom;
        CLG_REQUIRE(b == 0 || (gg.n == blocks[0].geom.n && gg.c_in == c && gg.h == h && gg.w == w), "%s: block %d does not take the output of the one before",
                    name, b);
        const int64_t need = clg_convblock_eval_packed_scratch_bytes(&gg);
        if (need < 0) return CLG_EINVAL;
        ws = std::max(ws, (size_t)need);
        c = gg.c_out;
        h = ((gg.h + 2 * gg.pad_h - gg.kernel_h) / gg.stride_h + 1) / 2;
        w = ((gg.w + 2 * gg.pad_w - gg.kernel_w) / gg.stride_w + 1) / 2;
        l->gates_off[b] = at;
        Geom g;
        PairPlan p;
        bool pair = false;
        if (int e = net_pair(name, blocks, n_blocks, b, &g, &p, &pair)) return e;
        at += net_up(pair ? p.total_bytes : (size_t)c * 7);
        act[b & 1] = std::max(act[b & 1], (size_t)gg.n * c * h * w * 8);
    }
    CLG_REQUIRE(c * h * w == in_dim, "%s: the last block gives %lld features, the trees take %lld", name, (long long)(c * h * w), (long long)in_dim);
    const PackedCut cut = cut_packed(roots, k, blocks[0].geom.n, true);
    l->codes_off = at;
    l->partial_off = l->codes_off + net_up((size_t)roots * 4);
    l->ping_off = l->partial_off + (cut.slices > 1 ? net_up((size_t)cut.slices * samples * k * 4) : 0);
    l->pong_off = l->ping_off + net_up(act[0]);
    l->ws_off = l->pong_off + net_up(act[1]);
    l->total = l->ws_off + net_up(ws);
    return CLG_OK;
}

}  // namespace

extern "C" int64_t clg_net_packed_scratch_bytes(const clg_packed_block *blocks, int n_blocks, int64_t in_dim, int64_t roots, int64_t k,
                                                int64_t samples)
{
    const char *name = "clg_net_packed_scratch_bytes";
    if (clg_check_tree(name, in_dim, roots, k)) return -1;
    NetLayout l;
    return net_layout(name, blocks, n_blocks, in_dim, roots, k, samples, &l) ? -1 : (int64_t)l.total;
}

extern "C" int clg_net_packed(const clg_packed_block *blocks, int n_blocks, const int64_t *x, const int32_t *rows, const int32_t *ids,
                              const float *logits0, const float *logits1, const float *logits2, int64_t *features, int32_t *counts, float *sums,
                              double tau, int64_t in_dim, int64_t roots, int64_t k, int64_t samples, void *scratch, void *stream)
{
    const char *name = "clg_net_packed";
    if (int e = clg_check_tree(name, in_dim, roots, k)) return e;
    NetLayout l;
    if (int e = net_layout(name, blocks, n_blocks, in_dim, roots, k, samples, &l)) return e;
    const int64_t words = blocks[0].geom.n;
    CLG_REQUIRE(x && rows && ids && logits0 && logits1 && logits2 && features && scratch && (counts != nullptr) != (sums != nullptr),
                "%s: null pointer argument, or both or neither of counts and sums", name);
    CLG_REQUIRE(samples > 0 && samples <= words * 64 && (sums == nullptr || tau != 0.0), "%s: words %lld, samples %lld, tau %g", name,
                (long long)words, (long long)samples, tau);
    const PackedCut c = cut_packed(roots, k, words, true);
    if (int e = check_packed(name, k, words, c)) return e;
    unsigned char *base = reinterpret_cast<unsigned char *>(scratch);
    NetGates net{};
    net.blocks = n_blocks;
    PairPlan plan[kMaxNetBlocks];
    int64_t kernels = 0;
    for (int b = 0; b < n_blocks; ++b) {
        CLG_REQUIRE(blocks[b].logits && blocks[b].selection, "%s: null pointer in block %d", name, b);
        NetBlock &nb = net.block[b];
        bool pair = false;
        if (int e = net_pair(name, blocks, n_blocks, b, &nb.geom, &plan[b], &pair)) return e;
        nb.logits = blocks[b].logits;
        nb.sel = blocks[b].selection;
        kernels += nb.geom.c;
        CLG_REQUIRE(kernels < (1ll << 28), "%s: problem too large for one launch", name);
        nb.end = (int)kernels;
        if (pair) {
            nb.table = reinterpret_cast<int32_t *>(base + l.gates_off[b]);
            nb.plane = plan[b].plane;
            nb.rs = plan[b].rs;
            nb.odd = plan[b].odd;
            nb.shift = plan[b].lead - plan[b].pw;
        } else {
            nb.ids = base + l.gates_off[b];
        }
    }
    hipStream_t st = clg_stream(stream);
    const TreeLogits lg = {{logits0, logits1, logits2}};
    uint32_t *codes = reinterpret_cast<uint32_t *>(base + l.codes_off);
    if (int e = make_codes(name, lg, ids, codes, roots, nullptr, 0, net, st)) return e;
    const uint64_t *in = reinterpret_cast<const uint64_t *>(x);
    bool flat = false;                                                // the last block wrote its words feature-major
    for (int b = 0; b < n_blocks; ++b) {
        const clg_packed_block &bl = blocks[b];
        uint64_t *out = reinterpret_cast<uint64_t *>(base + ((b & 1) ? l.pong_off : l.ping_off));
        const NetBlock &nb = net.block[b];
        const bool last = b == n_blocks - 1, pair = nb.table != nullptr;
        flat = last && (pair || clg_convblock_eval_packed_fm_supported(&bl.geom));
        if (flat) out = reinterpret_cast<uint64_t *>(features);
        const int e = pair ? clg_forward_pair_packed(nb.geom, plan[b], in, nullptr, bl.selection, out, nb.table, st, name)
                           : (flat ? clg_convblock_eval_packed_fm(&bl.geom, in, nb.ids, bl.selection, out, stream)
                                   : clg_convblock_eval_packed_ws(&bl.geom, in, nb.ids, bl.selection, out, base + l.ws_off, stream));
        if (e) return e;
        in = out;
    }
    if (!flat)
        if (int e = clg_transpose_2d(8, in, features, words, in_dim, stream)) return e;
    return count_packed(name, features, rows, codes, counts, sums, sums != nullptr ? 1.f / (float)tau : 0.f,
                        reinterpret_cast<int32_t *>(base + l.partial_off), in_dim, roots, k, words, samples, c, st);
}
