// Autograd nodes of the float32 training path in C++: the same calls of the C ABI, tensors and checks as the Python functions of
// the modules (difflogic/difflogic.py, difflogic/fc_tree.py, convlogic/convlogic_layer.py), which serve every other case.
// What they are for: the backward pass runs on autograd's device thread, where a Python function first has to take the
// interpreter from the thread that waits for it, and an eager step of a small network is bound by that and by the interpreter's time
// per launch.  Forward and backward of one block 82 us on a quiet host and 146 with the hand-off by the Python
// functions, of a LogicLayer 64 and 124.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/utils/pybind.h>

#include "convlogic_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc)
{
    TORCH_CHECK(rc == CLG_OK, clg_last_error());
}
void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const int64_t *idx(const Tensor &t) { return static_cast<const int64_t *>(t.data_ptr()); }
Tensor floats(const Tensor &like, at::IntArrayRef shape) { return at::empty(shape, like.options()); }
Tensor bytes(const Tensor &like, int64_t n)
{
    TORCH_CHECK(n >= 0, clg_last_error());
    return at::empty({n < 8 ? 8 : n}, like.options().dtype(at::kByte));
}
// what the kernels read as raw float32 memory of `like`'s device
void need(const Tensor &t, const Tensor &like, const char *name, at::IntArrayRef shape)
{
    TORCH_CHECK(t.device() == like.device(), "all tensors must be on one device, got ", like.device(), " and ", t.device());
    TORCH_CHECK(t.scalar_type() == at::kFloat, name, " must have dtype torch.float32, got ", t.scalar_type());
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes());
}
Tensor transposed(const Tensor &x)
{
    Tensor out = at::empty({x.size(1), x.size(0)}, x.options());
    if (out.numel()) check(clg_transpose_2d((int)x.element_size(), x.data_ptr(), out.data_ptr(), x.size(0), x.size(1), stream_of(x)));
    return out;
}
Tensor contiguous_2d(const Tensor &t)
{
    if (t.is_contiguous()) return t;
    if (t.is_cuda() && t.dim() == 2 && t.transpose(0, 1).is_contiguous()) return transposed(t.transpose(0, 1));
    return t.contiguous();
}

// ---- layouts -----------------------------------------------------------------------------------------------------------
// [batch, features] -> contiguous [features, batch], and the same for the gradient
struct FeatureMajor : torch::autograd::Function<FeatureMajor> {
    static Tensor forward(AutogradContext *, const Tensor &x) { return transposed(x); }
    static variable_list backward(AutogradContext *, variable_list grads)
    {
        const Tensor &g = grads[0];
        return {g.is_cuda() && g.is_contiguous() ? transposed(g) : g.transpose(0, 1)};
    }
};
Tensor feature_major(const Tensor &x) { return FeatureMajor::apply(x); }

// ---- LogicLayer ------------------------------------------------------------------------------------------------------------
struct FcLayer : torch::autograd::Function<FcLayer> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_in, const Tensor &a, const Tensor &b, const Tensor &logits, const Tensor &start,
                          const Tensor &flat, bool sole, bool sample_major)
    {
        const int64_t out_dim = logits.size(0), in_dim = x_in.size(sample_major ? 1 : 0), batch = x_in.size(sample_major ? 0 : 1);
        Tensor y = floats(x_in, {out_dim, batch}), probs = floats(x_in, {out_dim, 16}), folded = floats(x_in, {out_dim, 4}), x = x_in;
        if (sample_major) {
            x = floats(x_in, {in_dim, batch});
            check(clg_fc_forward_logits_ex(CLG_F32, x_in.data_ptr(), idx(a), idx(b), logits.data_ptr(), probs.data_ptr(), folded.data_ptr(),
                                           y.data_ptr(), in_dim, out_dim, batch, CLG_FC_X_SAMPLE_MAJOR, x.data_ptr(), stream_of(x)));
        } else {
            check(clg_fc_forward_logits(CLG_F32, x.data_ptr(), idx(a), idx(b), logits.data_ptr(), probs.data_ptr(), folded.data_ptr(), y.data_ptr(),
                                        in_dim, out_dim, batch, stream_of(x)));
        }
        ctx->save_for_backward({x, a, b, probs, folded, start, flat});
        ctx->saved_data["sole"] = sole;
        ctx->saved_data["sample_major"] = sample_major;
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &a = saved[1], &b = saved[2], &probs = saved[3], &folded = saved[4], &start = saved[5], &flat = saved[6];
        const bool sole = ctx->saved_data["sole"].toBool(), sample_major = ctx->saved_data["sample_major"].toBool();
        const bool need_x = ctx->needs_input_grad(0), need_l = ctx->needs_input_grad(3);
        const int64_t in_dim = x.size(0), batch = x.size(1), out_dim = folded.size(0);
        const bool fused = !sole && need_x && need_l && clg_fc_backward_fused_fits(CLG_F32, batch);
        Tensor gy = grads[0], gx, gl;
        // a gradient that arrives as a transposed view: its feature-major copy is made by the call that computes both gradients
        const bool gy_sample_major = fused && !gy.is_contiguous() && gy.is_cuda() && gy.dim() == 2 && gy.transpose(0, 1).is_contiguous();
        if (gy_sample_major) {
            gy = gy.transpose(0, 1);
            need(gy, x, "grad_y", {batch, out_dim});
        } else {
            gy = contiguous_2d(gy);
            need(gy, x, "grad_y", {out_dim, batch});
        }
        if (need_l) gl = floats(x, {out_dim, 16});
        if (fused) {
            gx = sample_major ? floats(x, {batch, in_dim}) : floats(x, {in_dim, batch});
            Tensor copy;
            if (gy_sample_major) copy = floats(x, {out_dim, batch});
            check(clg_fc_backward_fused_ex(CLG_F32, x.data_ptr(), idx(a), idx(b), folded.data_ptr(), probs.data_ptr(), gy.data_ptr(), idx(start),
                                           idx(flat), gx.data_ptr(), gl.data_ptr(), in_dim, out_dim, batch,
                                           (sample_major ? CLG_FC_GX_SAMPLE_MAJOR : 0) | (gy_sample_major ? CLG_FC_GY_SAMPLE_MAJOR : 0), ptr(copy),
                                           stream_of(x)));
            return {gx, Tensor(), Tensor(), gl, Tensor(), Tensor(), Tensor(), Tensor()};
        }
        if (need_x) gx = at::empty_like(x);
        if (sole && need_x && need_l) {
            check(clg_fc_backward_sole(CLG_F32, x.data_ptr(), idx(a), idx(b), folded.data_ptr(), probs.data_ptr(), gy.data_ptr(), gx.data_ptr(),
                                       gl.data_ptr(), in_dim, out_dim, batch, stream_of(x)));
        } else {
            if (need_x)
                check(clg_fc_backward_x_folded(CLG_F32, x.data_ptr(), idx(a), idx(b), folded.data_ptr(), gy.data_ptr(), idx(start), idx(flat),
                                               gx.data_ptr(), in_dim, out_dim, batch, stream_of(x)));
            if (need_l)
                check(clg_fc_backward_logits(CLG_F32, x.data_ptr(), idx(a), idx(b), probs.data_ptr(), gy.data_ptr(), gl.data_ptr(), in_dim, out_dim,
                                             batch, stream_of(x)));
        }
        if (sample_major && need_x) gx = transposed(gx);
        return {gx, Tensor(), Tensor(), gl, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};
// x [batch, in] where sample_major, else [in, batch]; -> [batch, out], a transposed view of [out, batch]
Tensor fc_layer(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &logits, const Tensor &start, const Tensor &flat, bool sole,
                bool sample_major)
{
    need(logits, x, "weights", {a.numel(), 16});
    return FcLayer::apply(x, a, b, logits, start, flat, sole, sample_major).transpose(0, 1);
}

// ---- complete blocks -----------------------------------------------------------------------------------------------------
struct Conv {                                                         // stride, padding and kernel of a block
    int64_t sh, sw, ph, pw, kh, kw;
    clg_conv_geom geom(at::IntArrayRef x, int64_t c_out) const
    {
        return {(int32_t)x[0], (int32_t)x[1], (int32_t)x[2], (int32_t)x[3], (int32_t)c_out, (int32_t)sh, (int32_t)sw, (int32_t)ph, (int32_t)pw,
                (int32_t)kh, (int32_t)kw};
    }
    clg_conv_geom geom(const Tensor &x, int64_t c_out) const { return geom(x.sizes(), c_out); }
    c10::IValue saved(std::vector<int64_t> more) const
    {
        std::vector<int64_t> l{sh, sw, ph, pw, kh, kw};
        l.insert(l.end(), more.begin(), more.end());
        return c10::IValue(std::move(l));
    }
    static Conv from(const std::vector<int64_t> &l) { return {l[0], l[1], l[2], l[3], l[4], l[5]}; }
};
std::vector<int64_t> pooled(const clg_conv_geom &g)
{
    const int64_t ho = (g.h + 2 * g.pad_h - g.kernel_h) / g.stride_h + 1, wo = (g.w + 2 * g.pad_w - g.kernel_w) / g.stride_w + 1;
    return {g.n, g.c_out, std::max<int64_t>(ho, 0) / 2, std::max<int64_t>(wo, 0) / 2};
}

// What a block keeps of its forward pass, in the order in which it is saved.
struct BlockState {
    Tensor x, probs, sel, argmax, folded, padded;
    static constexpr int kTensors = 6;
    void save(variable_list &list) const { list.insert(list.end(), {x, probs, sel, argmax, folded, padded}); }
    static BlockState from(const Tensor *t) { return {t[0], t[1], t[2], t[3], t[4], t[5]}; }
};
// What clg_train_prepare has filled for a float32 block: probabilities and coefficients, and the scratch of its forward call.
struct Prepared {
    Tensor probs, scratch;
    static Prepared room(const Tensor &like, const clg_conv_geom &g)
    {
        return {floats(like, {(int64_t)g.c_out * (112 + 28)}), bytes(like, clg_convblock_forward_scratch_bytes(CLG_F32, &g))};
    }
};
// Sums that the backward calls of a network's layers leave for one launch, and the buffers their parts are in -- those alone, a layer's scratch
// is the next one's: operand gradients and gradient planes of all layers held together were twice the memory of a step (CIFAR topology, k =
// 100, 1024 images: 3.07 GB, 1.88 like this and by the modules).
struct Late {
    std::vector<clg_late_sums> sums;
    Tensor parts, histogram;                                          // (of a binary block: the only one's scratch)
    int64_t used = 0, block = 0;                                      // block: bytes of the parts of the block at hand
    static int64_t aligned(int64_t n) { return (n + 255) & ~(int64_t)255; }
    void *take(int64_t n)                                             // of parts, which hold as much as all layers take
    {
        TORCH_CHECK(used + n <= parts.numel(), "late sums: more parts than room");
        void *at = static_cast<char *>(parts.data_ptr()) + used;
        used += aligned(n);
        return at;
    }
    clg_late_sums *next()
    {
        sums.push_back({});
        return &sums.back();
    }
    void run(void *stream)
    {
        if (!sums.empty()) check(clg_late_sums_run(sums.data(), (int)sums.size(), stream));
    }
};
// signature: that of the layer's backward plan.  pair: probabilities and folded coefficients [c, 7, 16], [c, 7, 4] in one buffer
// that a network made for all its layers (or null).  fm (in): the output may be feature-major; (out): it is, [c, h, w, n].
Tensor block_forward(const Tensor &x_in, const Tensor &logits, const Tensor &sel_in, const Conv &conv, bool &fm, int64_t signature,
                     const std::pair<Tensor, Tensor> *pair, bool need_x, BlockState &state, const Prepared *made = nullptr)
{
    const Tensor x = x_in.contiguous(), sel = sel_in.contiguous();
    const int64_t c = logits.size(0);
    const clg_conv_geom g = conv.geom(x, c);
    const auto s = pooled(g);
    fm = fm && clg_convblock_fm_supported(CLG_F32, &g);
    Tensor y = fm ? floats(x, {s[1], s[2], s[3], s[0]}) : floats(x, s), argmax = at::empty(s, x.options().dtype(at::kByte));
    Tensor probs, folded;                                             // without a pair: probabilities and coefficients in one tensor, no folded
    if (pair != nullptr) {
        probs = pair->first, folded = pair->second;
        need(probs, x, "prefolded probabilities", {c, 7, 16});
        need(folded, x, "prefolded coefficients", {c, 7, 4});
        TORCH_CHECK(folded.data_ptr<float>() == probs.data_ptr<float>() + probs.numel(),
                    "prefolded: the folded coefficients must follow the probabilities in one buffer (fold_many)");
    } else if (made == nullptr) {
        probs = floats(x, {c * (112 + 28)});
    } else {
        probs = made->probs;
    }
    const Tensor scratch = made != nullptr ? made->scratch : bytes(x, clg_convblock_forward_scratch_bytes(CLG_F32, &g));
    const int flags = CLG_FWD_W_LOGITS | (fm ? CLG_FWD_Y_FEATURE_MAJOR : 0) | CLG_FWD_FOLDED_OUT |
                      (made != nullptr ? CLG_FWD_FOLDED_IN | CLG_FWD_PREPARED : (pair != nullptr ? CLG_FWD_FOLDED_IN : 0));
    Tensor padded;
    if (need_x && !fm) {                                              // the copy of x that the forward kernels stage and the backward reads
        const int64_t elems = clg_convblock_padded_elems_planned(CLG_F32, &g, 1, signature);
        if (elems > 0) padded = floats(x, {elems});
    }
    const int32_t *selection = static_cast<const int32_t *>(sel.data_ptr());
    uint8_t *codes = static_cast<uint8_t *>(argmax.data_ptr());
    if (padded.defined())
        check(clg_convblock_forward_padded(CLG_F32, &g, x.data_ptr(), logits.data_ptr(), selection, y.data_ptr(), codes, probs.data_ptr(), flags,
                                           scratch.data_ptr(), padded.data_ptr(), stream_of(x)));
    else
        check(clg_convblock_forward_ex(CLG_F32, &g, x.data_ptr(), logits.data_ptr(), selection, y.data_ptr(), codes, probs.data_ptr(), flags,
                                       scratch.data_ptr(), stream_of(x)));
    state = {x, probs, sel, argmax, folded, padded};
    return y;
}
// -> gradients of x and of the logits; fm: the forward pass was feature-major
std::pair<Tensor, Tensor> block_backward(const BlockState &state, const Conv &conv, bool fm, const Tensor &plan, int64_t signature, Tensor gy, bool need_x,
                                         bool need_l, Late *late = nullptr)
{
    const Tensor &x = state.x, &probs = state.probs, &sel = state.sel;
    const int64_t c = sel.size(0);
    const float *folded = state.folded.defined() ? state.folded.data_ptr<float>() : probs.data_ptr<float>() + c * 112;
    const int32_t *selection = static_cast<const int32_t *>(sel.data_ptr());
    const uint8_t *codes = static_cast<const uint8_t *>(state.argmax.data_ptr());
    const clg_conv_geom g = conv.geom(x, c);
    Tensor gx, gl;
    if (need_x) gx = at::empty_like(x);
    if (need_l) {
        fm = fm && !gy.is_contiguous() && gy.permute({1, 2, 3, 0}).is_contiguous();
        const auto s = pooled(g);
        if (fm) {
            gy = gy.permute({1, 2, 3, 0});
            need(gy, x, "grad_y", {s[1], s[2], s[3], s[0]});
        } else {
            gy = gy.contiguous();
            need(gy, x, "grad_y", s);
        }
        gl = floats(x, {c, 7, 16});
        const Tensor scratch = bytes(x, need_x ? clg_convblock_backward_planned_scratch_bytes(CLG_F32, &g, signature)
                                              : clg_convblock_backward_planned_w_scratch_bytes(CLG_F32, &g));
        const Tensor padded = fm || !need_x ? Tensor() : state.padded;
        const int flags = CLG_BWD_WRT_LOGITS | (fm ? CLG_BWD_GY_FEATURE_MAJOR : 0);
        if (late != nullptr)
            check(clg_convblock_backward_planned_late(CLG_F32, &g, gy.data_ptr(), x.data_ptr(), probs.data_ptr(), folded, ptr(padded), selection, codes,
                                                      plan.data_ptr(), signature, ptr(gx), gl.data_ptr(), flags, scratch.data_ptr(),
                                                      late->take(late->block), late->next(), stream_of(x)));
        else if (padded.defined())
            check(clg_convblock_backward_planned_padded(CLG_F32, &g, gy.data_ptr(), x.data_ptr(), probs.data_ptr(), folded, padded.data_ptr(),
                                                        selection, codes, plan.data_ptr(), signature, gx.data_ptr(), gl.data_ptr(), flags,
                                                        scratch.data_ptr(), stream_of(x)));
        else
            check(clg_convblock_backward_planned(CLG_F32, &g, gy.data_ptr(), x.data_ptr(), probs.data_ptr(), folded, selection, codes,
                                                 plan.data_ptr(), signature, ptr(gx), gl.data_ptr(), flags, scratch.data_ptr(), stream_of(x)));
    } else if (need_x) {
        gy = gy.contiguous();
        need(gy, x, "grad_y", pooled(g));
        const Tensor scratch = bytes(x, clg_convblock_backward_x_scratch_bytes(CLG_F32, &g));
        check(clg_convblock_backward_x(CLG_F32, &g, gy.data_ptr(), x.data_ptr(), probs.data_ptr(), selection, codes, gx.data_ptr(),
                                       scratch.data_ptr(), stream_of(x)));
    }
    return {gx, gl};
}
struct Block : torch::autograd::Function<Block> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &logits, const Tensor &sel, const Conv *conv, bool want_fm,
                          const Tensor *plan, int64_t signature, const std::pair<Tensor, Tensor> *pair, bool need_x)
    {
        BlockState state;
        const Tensor y = block_forward(x, logits, sel, *conv, want_fm, signature, pair, need_x, state);
        variable_list saved;
        state.save(saved);
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["conv"] = conv->saved({want_fm, signature});
        ctx->saved_data["plan"] = *plan;
        return want_fm ? y.permute({3, 0, 1, 2}) : y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const auto ints = ctx->saved_data["conv"].toIntVector();
        const auto g = block_backward(BlockState::from(saved.data()), Conv::from(ints), ints[6], ctx->saved_data["plan"].toTensor(), ints[7], grads[0],
                                      ctx->needs_input_grad(0), ctx->needs_input_grad(1));
        return {g.first, g.second, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};
Tensor block(const Tensor &x, const Tensor &logits, const Tensor &sel, std::array<int64_t, 6> conv, bool want_fm, const Tensor &plan,
             int64_t signature, const std::optional<std::pair<Tensor, Tensor>> &prefolded)
{
    need(logits, x, "weights", {sel.size(0), 7, 16});
    const Conv cv{conv[0], conv[1], conv[2], conv[3], conv[4], conv[5]};
    return Block::apply(x, logits, sel, &cv, want_fm, &plan, signature, prefolded ? &*prefolded : nullptr, at::GradMode::is_enabled() && x.requires_grad());
}

// The block on 0/1 inputs, from the logits.  flag: device address of the layer's BinaryFlag.  It keeps taps and keep; x itself is not needed
// again.  made: clg_train_prepare has filled keep.
Tensor binary_forward(const Tensor &x_in, const Tensor &logits, const Tensor &sel_in, const Conv &conv, int64_t flag, Tensor &taps, Tensor &keep,
                      bool made = false)
{
    const Tensor x = x_in.contiguous(), sel = sel_in.contiguous();
    const clg_conv_geom g = conv.geom(x, logits.size(0));
    if (!made) keep = bytes(x, clg_convblock_bin_ctx_bytes(CLG_F32, &g));
    const auto s = pooled(g);
    Tensor y = floats(x, s);
    taps = at::empty(s, x.options().dtype(at::kShort));
    check(clg_convblock_bin_forward(CLG_F32, &g, x.data_ptr(), logits.data_ptr(), static_cast<const int32_t *>(sel.data_ptr()), y.data_ptr(),
                                    static_cast<uint16_t *>(taps.data_ptr()), keep.data_ptr(), CLG_FWD_W_LOGITS | (made ? CLG_FWD_PREPARED : 0),
                                    reinterpret_cast<int32_t *>(flag), stream_of(x)));
    return y;
}
// xs: shape of x
std::pair<Tensor, Tensor> binary_backward(const Tensor &taps, const Tensor &keep, const Conv &cv, at::IntArrayRef xs, const Tensor &grad, bool need_x, bool need_l,
                                          Late *late = nullptr)
{
    const Tensor gy = grad.contiguous();
    TORCH_CHECK(gy.is_cuda(), "grad_y must be a CUDA tensor");
    TORCH_CHECK(gy.device() == taps.device(), "all tensors must be on one device, got ", taps.device(), " and ", gy.device());
    need(gy, gy, "grad_y", taps.sizes());
    const int64_t c = gy.size(1);
    const clg_conv_geom g = {(int32_t)xs[0], (int32_t)xs[1], (int32_t)xs[2], (int32_t)xs[3], (int32_t)c, (int32_t)cv.sh, (int32_t)cv.sw,
                             (int32_t)cv.ph, (int32_t)cv.pw, (int32_t)cv.kh, (int32_t)cv.kw};
    Tensor gx, gl, scratch;
    if (need_x) gx = floats(gy, xs);
    if (need_l) {
        gl = floats(gy, {c, 7, 16});
        scratch = bytes(gy, clg_convblock_bin_backward_scratch_bytes(CLG_F32, &g));
    }
    if (need_l && late != nullptr) {
        late->histogram = scratch;
        check(clg_convblock_bin_backward_late(CLG_F32, &g, gy.data_ptr(), static_cast<const uint16_t *>(taps.data_ptr()), keep.data_ptr(), ptr(gx), ptr(gl),
                                              CLG_BWD_WRT_LOGITS, ptr(scratch), late->next(), stream_of(gy)));
    } else if (need_x || need_l)
        check(clg_convblock_bin_backward(CLG_F32, &g, gy.data_ptr(), static_cast<const uint16_t *>(taps.data_ptr()), keep.data_ptr(), ptr(gx), ptr(gl),
                                         CLG_BWD_WRT_LOGITS, ptr(scratch), stream_of(gy)));
    return {gx, gl};
}
struct BinaryBlock : torch::autograd::Function<BinaryBlock> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &logits, const Tensor &sel, const Conv *conv, int64_t flag)
    {
        Tensor taps, keep;
        const Tensor y = binary_forward(x, logits, sel, *conv, flag, taps, keep);
        ctx->save_for_backward({taps, keep});
        ctx->saved_data["conv"] = conv->saved(x.sizes().vec());
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const auto ints = ctx->saved_data["conv"].toIntVector();
        const auto g = binary_backward(saved[0], saved[1], Conv::from(ints), at::IntArrayRef(ints).slice(6), grads[0], ctx->needs_input_grad(0),
                                       ctx->needs_input_grad(1));
        return {g.first, g.second, Tensor(), Tensor(), Tensor()};
    }
};
Tensor binary_block(const Tensor &x, const Tensor &logits, const Tensor &sel, std::array<int64_t, 6> conv, int64_t flag)
{
    need(logits, x, "weights", {sel.size(0), 7, 16});
    const Conv cv{conv[0], conv[1], conv[2], conv[3], conv[4], conv[5]};
    return BinaryBlock::apply(x, logits, sel, &cv, flag);
}

// ---- three LogicLayers and a GroupSum as trees --------------------------------------------------------------------------------
// wiring: indices_0 and indices_1 of the three layers, saved for autograd's check that they were not written in between;
// rows, pos, ids, slot: the tables of the wiring.
struct TreeArgs {
    Tensor start, rows, pos, ids, slot;
    std::vector<Tensor> wiring;
    int64_t roots, k;
    double tau;
};
const int32_t *i32(const Tensor &v) { return static_cast<const int32_t *>(v.data_ptr()); }
float *f32(const Tensor &v) { return static_cast<float *>(ptr(v)); }
// x feature-major -> class sums; coef and (need_l) probs are kept, and made here unless coef is there
Tensor trees_forward(const Tensor &x, const Tensor &l0, const Tensor &l1, const Tensor &l2, const TreeArgs &t, bool need_l, Tensor &coef, Tensor &probs)
{
    const int64_t in_dim = x.size(0), batch = x.size(1);
    if (!coef.defined()) {
        coef = floats(x, {t.roots, 28});
        if (need_l) probs = floats(x, {7 * t.roots, 16});             // (the logits may be updated between forward and backward)
        check(clg_fc_tree_fold_slots(l0.data_ptr<float>(), l1.data_ptr<float>(), l2.data_ptr<float>(), i32(t.slot), f32(coef), f32(probs), t.roots,
                                     stream_of(x)));
    }
    const int64_t elems = clg_fc_tree_partial_elems(t.roots, t.k, batch, batch);
    Tensor out = floats(x, {batch, t.k}), partial = floats(x, {elems < 0 ? 0 : elems});
    check(clg_fc_tree_forward(f32(x), i32(t.rows), f32(coef), f32(partial), f32(out), in_dim, t.roots, t.k, batch, batch, t.tau, stream_of(x)));
    return out;
}
// -> gradients of x and of the three layers' logits, those that are wanted.  tables: rows, pos, slot
std::array<Tensor, 4> trees_backward(const Tensor &x, const Tensor &start, const Tensor &coef, const Tensor &probs, const std::vector<Tensor> &tables, int64_t k,
                                     double tau, const Tensor &grad, std::array<bool, 4> wanted, Late *late = nullptr)
{
    const int64_t in_dim = x.size(0), batch = x.size(1), roots = coef.size(0);
    const Tensor go = grad.contiguous();
    need(go, x, "grad_out", {batch, k});
    std::array<Tensor, 4> g;
    if (wanted[0]) g[0] = at::empty_like(x);
    const int64_t neurons[3] = {4 * roots, 2 * roots, roots};
    for (int i = 0; i < 3; ++i)
        if (wanted[1 + i]) g[1 + i] = floats(x, {neurons[i], 16});
    const int64_t rows = g[0].defined() ? 8 * roots * batch : 0;
    const Tensor scratch = floats(x, {rows + (late ? 0 : 28 * roots)});   // operand gradients, then sums
    float *sums = late ? static_cast<float *>(late->take(112 * roots)) : f32(scratch) + rows;
    if (late != nullptr)
        check(clg_fc_tree_backward_late(f32(x), i32(tables[0]), i32(tables[1]), i32(tables[2]), f32(coef), f32(go), f32(probs), f32(g[1]), f32(g[2]),
                                        f32(g[3]), f32(scratch), sums, idx(start), f32(g[0]), in_dim, roots, k, batch, batch, tau, late->next(),
                                        stream_of(x)));
    else
        check(clg_fc_tree_backward(f32(x), i32(tables[0]), i32(tables[1]), i32(tables[2]), f32(coef), f32(go), f32(probs), f32(g[1]), f32(g[2]), f32(g[3]),
                                   f32(scratch), sums, idx(start), f32(g[0]), in_dim, roots, k, batch, batch, tau, stream_of(x)));
    return g;
}
struct Trees : torch::autograd::Function<Trees> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &l0, const Tensor &l1, const Tensor &l2, const TreeArgs *t, bool need_l)
    {
        Tensor coef, probs;
        const Tensor out = trees_forward(x, l0, l1, l2, *t, need_l, coef, probs);
        variable_list saved = {x, t->start, coef, probs};
        saved.insert(saved.end(), t->wiring.begin(), t->wiring.end());
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["tables"] = std::vector<Tensor>{t->rows, t->pos, t->slot};
        ctx->saved_data["k"] = t->k;
        ctx->saved_data["tau"] = t->tau;
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const auto g = trees_backward(saved[0], saved[1], saved[2], saved[3], ctx->saved_data["tables"].toTensorVector(), ctx->saved_data["k"].toInt(),
                                      ctx->saved_data["tau"].toDouble(), grads[0],
                                      {ctx->needs_input_grad(0), ctx->needs_input_grad(1), ctx->needs_input_grad(2), ctx->needs_input_grad(3)});
        return {g[0], g[1], g[2], g[3], Tensor(), Tensor()};
    }
};
Tensor trees(const Tensor &x, const Tensor &l0, const Tensor &l1, const Tensor &l2, const Tensor &start, std::vector<Tensor> wiring, const Tensor &rows,
             const Tensor &pos, const Tensor &ids, const Tensor &slot, int64_t roots, int64_t k, double tau)
{
    need(l0, x, "weights", {4 * roots, 16});
    need(l1, x, "weights", {2 * roots, 16});
    need(l2, x, "weights", {roots, 16});
    const TreeArgs t{start, rows, pos, ids, slot, std::move(wiring), roots, k, tau};
    return Trees::apply(x, l0, l1, l2, &t, at::GradMode::is_enabled() && (l0.requires_grad() || l1.requires_grad() || l2.requires_grad()));
}

// ---- a network: blocks, flattening, trees -------------------------------------------------------------------------------------
// One node for what the modules' nodes do one after the other, with the same kernels: a step of a small network is bound by the
// host, which takes longer from node to node (module calls in Python, views, the engine's queue) than for the launches of one.  MNIST
// topology, k = 32, 100 images, a step with its loss: 344 -> 285 us, with the set-up and the sums of all layers in a launch each 273; CIFAR, 256
// images: 352 -> 330, 296.
struct NetBlock {
    Tensor sel, plan;
    Conv conv;
    int64_t signature, flag;                                          // flag: not 0 for a block on 0/1 inputs, which has no plan
    bool fm;
};
struct NetArgs {
    std::vector<NetBlock> blocks;
    TreeArgs trees;
    std::vector<bool> wanted;                                         // of x and every logits
};
struct Network : torch::autograd::Function<Network> {
    // per block and for the trees in front of their wiring: as many saved tensors
    static constexpr int kEach = BlockState::kTensors, kTrees = 4;
    static constexpr size_t kTogether = 16;                           // blocks that clg_train_prepare and clg_late_sums_run take
    static Tensor forward(AutogradContext *ctx, const Tensor &x, at::TensorList logits, const NetArgs *a)
    {
        const size_t n = a->blocks.size();
        const bool need_l = a->wanted[1 + n] || a->wanted[2 + n] || a->wanted[3 + n];
        // the set-up of all layers in one launch
        Tensor coef, probs;
        std::vector<Prepared> made(n);                                // (a binary block's: its keep)
        const bool together = n <= kTogether;
        if (together) {
            std::vector<clg_train_block> first(n);
            at::DimVector shape(x.sizes());
            for (size_t i = 0; i < n; ++i) {
                const NetBlock &b = a->blocks[i];
                const clg_conv_geom g = b.conv.geom(shape, b.sel.size(0));
                const auto next = pooled(g);
                const bool binary = b.flag != 0;
                if (binary) made[i].probs = bytes(x, clg_convblock_bin_ctx_bytes(CLG_F32, &g));
                else made[i] = Prepared::room(x, g);
                first[i] = {g, binary ? f32(x) : nullptr, f32(logits[i]), i32(b.sel), binary ? nullptr : f32(made[i].probs),
                            binary ? ptr(made[i].probs) : ptr(made[i].scratch), reinterpret_cast<int32_t *>(b.flag),
                            !binary && b.fm && clg_convblock_fm_supported(CLG_F32, &g)};
                shape.assign(next.begin(), next.end());
            }
            coef = floats(x, {a->trees.roots, 28});
            if (need_l) probs = floats(x, {7 * a->trees.roots, 16});
            check(clg_train_prepare(first.data(), (int)n, f32(logits[n]), f32(logits[n + 1]), f32(logits[n + 2]), i32(a->trees.ids), f32(coef), f32(probs),
                                    a->trees.roots, stream_of(x)));
        }
        variable_list saved;
        std::vector<int64_t> ints;
        std::vector<Tensor> plans;
        Tensor h = x;
        bool some = a->wanted[0], fm = false;                         // whether a gradient is wanted of what the block takes
        for (size_t i = 0; i < n; ++i) {
            const NetBlock &b = a->blocks[i];
            BlockState state;
            const auto shape = h.sizes().vec();
            fm = b.fm;
            if (b.flag != 0) {
                fm = false;
                state.probs = made[i].probs;
                h = binary_forward(h, logits[i], b.sel, b.conv, b.flag, state.x, state.probs, together);
            } else {
                h = block_forward(h, logits[i], b.sel, b.conv, fm, b.signature, nullptr, some, state, together ? &made[i] : nullptr);
            }
            made[i] = {};
            state.save(saved);
            const std::vector<int64_t> own{b.conv.sh, b.conv.sw, b.conv.ph, b.conv.pw, b.conv.kh, b.conv.kw, shape[0], shape[1], shape[2], shape[3],
                                           b.flag != 0, b.signature, fm};
            ints.insert(ints.end(), own.begin(), own.end());
            plans.push_back(b.plan);
            some = some || a->wanted[1 + i];
        }
        // features [c h w, n]
        const int64_t batch = x.size(0);
        h = fm ? h.view({-1, batch}) : transposed(h.view({batch, -1}));
        const Tensor out = trees_forward(h, logits[n], logits[n + 1], logits[n + 2], a->trees, need_l, coef, probs);
        saved.insert(saved.end(), {h, a->trees.start, coef, probs});
        saved.insert(saved.end(), a->trees.wiring.begin(), a->trees.wiring.end());
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["blocks"] = std::move(ints);
        ctx->saved_data["plans"] = std::move(plans);
        ctx->saved_data["tables"] = std::vector<Tensor>{a->trees.rows, a->trees.pos, a->trees.slot};
        ctx->saved_data["k"] = a->trees.k;
        ctx->saved_data["tau"] = a->trees.tau;
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        constexpr int kInts = 13;
        const auto saved = ctx->get_saved_variables();
        const auto ints = ctx->saved_data["blocks"].toIntVector();
        const auto plans = ctx->saved_data["plans"].toTensorVector();
        const size_t n = plans.size();
        const auto wanted = [&](size_t i) { return ctx->needs_input_grad(i); };
        std::vector<bool> below(n + 1);                               // whether a gradient is wanted of what block i, or the trees, take
        below[0] = wanted(0);
        for (size_t i = 0; i < n; ++i) below[i + 1] = below[i] || wanted(1 + i);
        variable_list out(1 + n + 3 + 1);
        const Tensor *t = saved.data() + n * kEach;
        Late sums, *late = n <= kTogether ? &sums : nullptr;
        std::vector<int64_t> parts_of(n);
        if (late != nullptr) {
            int64_t parts = Late::aligned(112 * t[2].size(0));
            for (size_t i = 0; i < n; ++i) {
                const int64_t *own = ints.data() + i * kInts;
                if (own[10] != 0 || !wanted(1 + i)) continue;
                const clg_conv_geom geom = Conv{own[0], own[1], own[2], own[3], own[4], own[5]}.geom(at::IntArrayRef(own + 6, 4), saved[i * kEach + 2].size(0));
                parts += Late::aligned(parts_of[i] = clg_convblock_late_sums_bytes(CLG_F32, &geom));
            }
            sums.parts = bytes(t[0], parts);
        }
        auto g = trees_backward(t[0], t[1], t[2], t[3], ctx->saved_data["tables"].toTensorVector(), ctx->saved_data["k"].toInt(),
                                ctx->saved_data["tau"].toDouble(), grads[0], {below[n], wanted(1 + n), wanted(2 + n), wanted(3 + n)}, late);
        for (size_t i = 0; i < 3; ++i) out[1 + n + i] = g[1 + i];
        Tensor h = g[0];
        for (size_t i = n; i-- > 0 && (below[i] || wanted(1 + i));) {
            const int64_t *own = ints.data() + i * kInts;
            const Conv conv{own[0], own[1], own[2], own[3], own[4], own[5]};
            const Tensor *kept = saved.data() + i * kEach;
            const bool binary = own[10] != 0, fm = own[12] != 0;
            if (i + 1 == n) {                                         // from [features, batch]
                const auto s = pooled({(int32_t)own[6], (int32_t)own[7], (int32_t)own[8], (int32_t)own[9], (int32_t)(binary ? kept[0].size(1) : kept[2].size(0)),
                                       (int32_t)own[0], (int32_t)own[1], (int32_t)own[2], (int32_t)own[3], (int32_t)own[4], (int32_t)own[5]});
                h = fm ? h.view({s[1], s[2], s[3], s[0]}).permute({3, 0, 1, 2}) : transposed(h).view(s);
            }
            sums.block = parts_of[i];
            const auto gi = binary ? binary_backward(kept[0], kept[1], conv, at::IntArrayRef(own + 6, 4), h, below[i], wanted(1 + i), late)
                                   : block_backward(BlockState::from(kept), conv, fm, plans[i], own[11], h, below[i], wanted(1 + i), late);
            h = gi.first;
            out[1 + i] = gi.second;
        }
        if (below[0]) out[0] = h;
        sums.run(stream_of(t[0]));
        return out;
    }
};
// blocks: selection, stride / padding / kernel, plan, its signature, feature-major output, flag; logits of the blocks and of the three layers
using NetBlockTuple = std::tuple<Tensor, std::array<int64_t, 6>, Tensor, int64_t, bool, int64_t>;
Tensor network(const Tensor &x, const std::vector<Tensor> &logits, const std::vector<NetBlockTuple> &blocks, const Tensor &start, std::vector<Tensor> wiring,
               const Tensor &rows, const Tensor &pos, const Tensor &ids, const Tensor &slot, int64_t roots, int64_t k, double tau)
{
    const size_t n = blocks.size();
    TORCH_CHECK(n > 0 && logits.size() == n + 3, "logits of ", n, " blocks and three layers are needed, got ", logits.size());
    NetArgs a{{}, {start, rows, pos, ids, slot, std::move(wiring), roots, k, tau}, {x.requires_grad()}};
    for (size_t i = 0; i < n; ++i) {
        const auto &[sel, cv, plan, signature, fm, flag] = blocks[i];
        need(logits[i], x, "weights", {sel.size(0), 7, 16});
        a.blocks.push_back({sel, plan, {cv[0], cv[1], cv[2], cv[3], cv[4], cv[5]}, signature, flag, fm});
    }
    for (int i = 0; i < 3; ++i) need(logits[n + i], x, "weights", {(4 >> i) * roots, 16});
    for (const Tensor &l : logits) a.wanted.push_back(l.requires_grad());
    return Network::apply(x, at::TensorList(logits), &a);
}

// grad_fn of a node's output in Python: a type of the name that the Python function's node has
template <typename F>
void name_node(const char *name)
{
    static PyTypeObject type;
    torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
    torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<F>), &type);
}

}  // namespace

// (the interpreter is given up while a node works: the launches wait for nothing, but another thread may)
PYBIND11_MODULE(_nodes, m)
{
    const auto no_gil = py::call_guard<py::gil_scoped_release>();
    name_node<FeatureMajor>("_FeatureMajorBackward");
    name_node<FcLayer>("_LogicLayerLogitsFunctionBackward");
    name_node<Block>("_FullConvLogicLogitsFunctionBackward");
    name_node<BinaryBlock>("_FullConvLogicBinaryFunctionBackward");
    name_node<Trees>("_TreeFunctionBackward");
    name_node<Network>("_TreeNetworkFunctionBackward");
    m.def("feature_major", &feature_major, no_gil);
    m.def("fc_layer", &fc_layer, no_gil);
    m.def("block", &block, no_gil);
    m.def("binary_block", &binary_block, no_gil);
    m.def("trees", &trees, no_gil);
    m.def("network", &network, no_gil);
}
