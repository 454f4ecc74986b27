// Input binarisation in front of the logic layers: every pixel is compared with L thresholds and the
// results become L times as many {0,1} channels, threshold-major (channel l * c0 + c), either as floats
// for training or directly as packed words for inference (64 samples per word, group-major images --
// the layout the packed conv-logic block reads).
#include "clg_common.h"

namespace {

template <int SAMPLES>
struct PartWord;
template <>
struct PartWord<64> {
    typedef uint64_t type;
};
template <>
struct PartWord<16> {
    typedef uint16_t type;
};

constexpr int kLevelsPerPass = 8;

// Thresholds that the host has at hand travel in the kernel's arguments (no copy to the device, nothing to wait for)
constexpr int kHostLevels = 64;
struct HostThresholds {
    float t[kHostLevels];
};

// A workgroup takes 256 / SPLIT elements of the [c0, h*w] plane set (blockIdx.x) of one group of 64 samples (blockIdx.y) and up to
// L thresholds (blockIdx.z); wavefront lanes read consecutive pixels of one sample (coalesced).  SPLIT threads share an
// element, 64 / SPLIT samples each, and meet in LDS.  Bound by the read of the images; L is the number of thresholds where it is
// small, so that none is compared in vain (an L of 4 for all cost 165 us at 3 levels, and from 5 levels on a second read of the
// images).
// BINARY: images that hold 0 and 1 already (any other value is a 1 and sets *bad).
template <int L, int SPLIT, bool BINARY = false>
__global__ __launch_bounds__(256) void threshold_pack_kernel(const float *__restrict__ x, const float *__restrict__ thr, const HostThresholds host,
                                                           uint64_t *__restrict__ words, int64_t n, int64_t plane_elems, int levels,
                                                           int32_t *__restrict__ bad = nullptr)
{
    constexpr int kElems = 256 / SPLIT, kSamples = 64 / SPLIT, kBatch = 16;
    typedef typename PartWord<kSamples>::type Part;
    __shared__ Part part[SPLIT > 1 ? SPLIT : 1][SPLIT > 1 ? L : 1][SPLIT > 1 ? kElems : 1];
    const int lane = threadIdx.x % kElems, q = uniform((int)threadIdx.x / kElems);
    const int64_t e = (int64_t)blockIdx.x * kElems + lane;
    const bool live = e < plane_elems;
    const int64_t g = blockIdx.y;
    const int l0 = blockIdx.z * kLevelsPerPass;
    float t[L];
#pragma unroll
    for (int l = 0; l < L; ++l) t[l] = l0 + l < levels ? (thr ? thr[l0 + l] : host.t[l0 + l]) : 0.0f;
    Part w[L];
#pragma unroll
    for (int l = 0; l < L; ++l) w[l] = 0;
    const int64_t s0 = g * 64 + q * kSamples, left = n - s0;
    const float *src = x + s0 * plane_elems + e;
    bool other = false;
    auto bit = [&](float v, float threshold) {
        if constexpr (BINARY) {
            other = other || (v != 0.f && v != 1.f);
            return v != 0.f;
        } else {
            return v > threshold;
        }
    };
    if (live && left >= kSamples) {
#pragma unroll
        for (int s = 0; s < kSamples; s += kBatch) {
            float v[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) v[j] = src[(int64_t)(s + j) * plane_elems];
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
#pragma unroll
                for (int l = 0; l < L; ++l) w[l] |= (Part)(bit(v[j], t[l]) ? 1 : 0) << (s + j);
        }
    } else if (live) {
        for (int s = 0; s < left; ++s) {
            const float v = src[(int64_t)s * plane_elems];
#pragma unroll
            for (int l = 0; l < L; ++l) w[l] |= (Part)(bit(v, t[l]) ? 1 : 0) << s;
        }
    }
    if (BINARY && other) *bad = 1;
    if constexpr (SPLIT == 1) {
        if (!live) return;
#pragma unroll
        for (int l = 0; l < L; ++l)
            if (l0 + l < levels) __builtin_nontemporal_store((uint64_t)w[l], &words[(g * levels + l0 + l) * plane_elems + e]);
    } else {
#pragma unroll
        for (int l = 0; l < L; ++l) part[q][l][lane] = w[l];
        __syncthreads();
        for (int i = threadIdx.x; i < L * kElems; i += 256) {
            const int l = i / kElems, el = i % kElems;
            const int64_t at = (int64_t)blockIdx.x * kElems + el;
            if (l0 + l >= levels || at >= plane_elems) continue;
            uint64_t word = 0;
#pragma unroll
            for (int j = 0; j < SPLIT; ++j) word |= (uint64_t)part[j][l][el] << (j * kSamples);
            __builtin_nontemporal_store(word, &words[(g * levels + l0 + l) * plane_elems + at]);
        }
    }
}

__global__ __launch_bounds__(256) void threshold_float_kernel(const float *__restrict__ x, const float *__restrict__ thr,
                                                            float *__restrict__ out, int64_t n, int64_t plane_elems, int levels)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n * plane_elems) return;
    const int64_t s = i / plane_elems, e = i - s * plane_elems;
    const float v = x[i];
    for (int l = 0; l < levels; ++l) out[(s * levels + l) * plane_elems + e] = v > thr[l] ? 1.0f : 0.0f;
}

int check_threshold_args(const void *x, const void *thr, const void *out, int64_t n, int64_t c0, int64_t hw, int64_t levels,
                         const char *name)
{
    CLG_REQUIRE(x && thr && out, "%s: null pointer argument", name);
    CLG_REQUIRE(n > 0 && c0 > 0 && hw > 0 && levels > 0, "%s: n, channels, pixels and levels must be positive", name);
    CLG_REQUIRE(levels <= 4096 && c0 * hw < (1ll << 31), "%s: at most 4096 levels and 2^31-1 elements per sample", name);
    return CLG_OK;
}

}  // namespace

namespace {
template <int L>
void launch_threshold_pack(const float *x, const float *thr, const HostThresholds &host, uint64_t *words, int64_t n, int64_t plane_elems,
                           int levels, int64_t groups, hipStream_t st)
{
    const unsigned passes = (unsigned)clg_ceil_div(levels, kLevelsPerPass);
    // Four threads per element: 161 -> 153 us on [65536, 3, 32, 32] with 3 levels (5.8 TB/s), 9.0 -> 4.8 us with 256 images;
    // one where a level's words alone leave LDS nothing to save and the elements fill the GPU (36 against 40 us on
    // [65536, 1, 28, 28] with 1 level), and where four would be more threads than a launch can have.
    const bool split = (levels > 1 || clg_ceil_div(plane_elems, 256) * groups < 2048) && clg_ceil_div(plane_elems, 64) < (1 << 24);
    if (split)
        hipLaunchKernelGGL((threshold_pack_kernel<L, 4>), dim3((unsigned)clg_ceil_div(plane_elems, 64), (unsigned)groups, passes), dim3(256), 0, st,
                           x, thr, host, words, n, plane_elems, levels, (int32_t *)nullptr);
    else
        hipLaunchKernelGGL((threshold_pack_kernel<L, 1>), dim3((unsigned)clg_ceil_div(plane_elems, 256), (unsigned)groups, passes), dim3(256), 0, st,
                           x, thr, host, words, n, plane_elems, levels, (int32_t *)nullptr);
}

int threshold_pack(const char *name, const float *x, const float *thr, const HostThresholds &host, uint64_t *words, int64_t n, int64_t c0,
                   int64_t hw, int64_t levels, void *stream)
{
    const int64_t groups = clg_ceil_div(n, 64), plane_elems = c0 * hw;
    CLG_REQUIRE(groups <= 65535 * 64ll, "%s: batch too large for one launch", name);
    // the grid's y extent is limited to 65535: larger batches go in slabs of 65535 groups
    for (int64_t g0 = 0; g0 < groups; g0 += 65535) {
        const int64_t gs = groups - g0 < 65535 ? groups - g0 : 65535, left = n - g0 * 64;
        const float *xs = x + g0 * 64 * plane_elems;
        uint64_t *ws = words + g0 * levels * plane_elems;
        if (levels == 1) launch_threshold_pack<1>(xs, thr, host, ws, left, plane_elems, (int)levels, gs, clg_stream(stream));
        else if (levels == 2) launch_threshold_pack<2>(xs, thr, host, ws, left, plane_elems, (int)levels, gs, clg_stream(stream));
        else if (levels == 3) launch_threshold_pack<3>(xs, thr, host, ws, left, plane_elems, (int)levels, gs, clg_stream(stream));
        else if (levels <= 5) launch_threshold_pack<5>(xs, thr, host, ws, left, plane_elems, (int)levels, gs, clg_stream(stream));
        else launch_threshold_pack<kLevelsPerPass>(xs, thr, host, ws, left, plane_elems, (int)levels, gs, clg_stream(stream));
        CLG_CHECK_LAUNCH(name);
    }
    return CLG_OK;
}
}  // namespace

extern "C" int clg_threshold_pack_images(const float *x, const float *thresholds, uint64_t *words, int64_t n, int64_t c0,
                                         int64_t hw, int64_t levels, void *stream)
{
    const char *name = "clg_threshold_pack_images";
    if (int e = check_threshold_args(x, thresholds, words, n, c0, hw, levels, name)) return e;
    return threshold_pack(name, x, thresholds, HostThresholds{}, words, n, c0, hw, levels, stream);
}

extern "C" int clg_threshold_pack_images_host(const float *x, const float *thresholds, uint64_t *words, int64_t n, int64_t c0,
                                              int64_t hw, int64_t levels, void *stream)
{
    const char *name = "clg_threshold_pack_images_host";
    if (int e = check_threshold_args(x, thresholds, words, n, c0, hw, levels, name)) return e;
    CLG_REQUIRE(levels <= kHostLevels, "%s: at most %d levels", name, kHostLevels);
    HostThresholds host{};
    for (int64_t l = 0; l < levels; ++l) host.t[l] = thresholds[l];
    return threshold_pack(name, x, nullptr, host, words, n, c0, hw, levels, stream);
}

extern "C" int clg_pack_binary_images(const float *x, uint64_t *words, int64_t n, int64_t c0, int64_t hw, int32_t *not_binary, void *stream)
{
    const char *name = "clg_pack_binary_images";
    if (int e = check_threshold_args(x, not_binary, words, n, c0, hw, 1, name)) return e;
    const int64_t groups = clg_ceil_div(n, 64), plane_elems = c0 * hw;
    CLG_REQUIRE(groups <= 65535, "%s: batch too large for one launch", name);
    if (clg_ceil_div(plane_elems, 256) * groups < 2048)              // (the split as for one threshold)
        hipLaunchKernelGGL((threshold_pack_kernel<1, 4, true>), dim3((unsigned)clg_ceil_div(plane_elems, 64), (unsigned)groups), dim3(256), 0,
                           clg_stream(stream), x, (const float *)nullptr, HostThresholds{}, words, n, plane_elems, 1, not_binary);
    else
        hipLaunchKernelGGL((threshold_pack_kernel<1, 1, true>), dim3((unsigned)clg_ceil_div(plane_elems, 256), (unsigned)groups), dim3(256), 0,
                           clg_stream(stream), x, (const float *)nullptr, HostThresholds{}, words, n, plane_elems, 1, not_binary);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_threshold_images(const float *x, const float *thresholds, float *out, int64_t n, int64_t c0, int64_t hw,
                                    int64_t levels, void *stream)
{
    if (int e = check_threshold_args(x, thresholds, out, n, c0, hw, levels, "clg_threshold_images")) return e;
    const int64_t total = n * c0 * hw;
    CLG_REQUIRE(clg_ceil_div(total, 256) < (1ll << 31), "clg_threshold_images: batch too large for one launch");
    hipLaunchKernelGGL(threshold_float_kernel, dim3((unsigned)clg_ceil_div(total, 256)), dim3(256), 0, clg_stream(stream), x,
                       thresholds, out, n, c0 * hw, (int)levels);
    CLG_CHECK_LAUNCH("clg_threshold_images");
    return CLG_OK;
}
