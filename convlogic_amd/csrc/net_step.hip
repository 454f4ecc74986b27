// The first and the last launch of a training step of a small network.  Every layer has a set-up of its own (softmax and folding of its logits, tables, the
// bit rows of a binary first block) and sums that end its weight gradient; none of them depends on another layer, and a launch of
// either kind is 4 to 6 us of one round trip to memory after the other, whatever it does.  Here one launch makes the set-up of all layers and another one
// the sums: CIFAR topology, k = 32, 256 images: 26 us in five launches -> 9.9, 19.3 us in four -> 7.7
// (replayed step 321 -> 301 us); MNIST topology, 100 images: 21 in four -> 7.8, 17 in four -> 6.2.
#include "conv_binary.h"
#include "conv_pair.h"
#include "fc_tree.h"
#include "net_step.h"

namespace {

constexpr int kMaxStepBlocks = 16;

// A float block: probabilities [c, 7, 16] and folded coefficients [c, 7, 4], and the table of its forward kernel where it reads one
struct BlockPrepare {
    const float *logits;
    const int32_t *sel;
    float *probs;
    int32_t *table;
    int end;                                                         // workgroups up to and including the block's
    PairOffsets at;
    Geom g;
};
struct StepPrepare {
    int bin_end, tree_end, blocks;                                   // workgroups of a binary block (the longest chain), of the trees behind them
    BlockPrepare block[kMaxStepBlocks];
};

__global__ __launch_bounds__(256) void step_prepare_kernel(TreeFold trees, PrepArgs bin, Geom bin_geom, StepPrepare a)
{
    const int b = blockIdx.x;
    if (b < a.bin_end) {
        bin_prepare(bin, bin_geom, b, a.bin_end);
        return;
    }
    if (b < a.tree_end) {
        tree_fold(trees, b - a.bin_end);
        return;
    }
    int first = a.tree_end, i = 0;
    while (i < a.blocks - 1 && b >= a.block[i].end) first = a.block[i++].end;
    const BlockPrepare &p = a.block[i];
    const int64_t q = (int64_t)(b - first) * 256 + threadIdx.x;
    if (q < (int64_t)p.g.c * 7) fold_gate<float, float>(p.logits, q, true, p.probs, p.probs + (int64_t)p.g.c * 112);
    if (p.table != nullptr) {
        if (q == 0) *reinterpret_cast<Geom *>(p.table + (int64_t)p.g.c * kPairTable) = p.g;
        if (q < p.g.c) pair_table_row(p.table, p.sel, q, p.at, p.g);
    }
}

constexpr int kMaxLate = kMaxStepBlocks + 1;
struct StepSums {
    clg_late_sums late[kMaxLate];                                    // (blocks: workgroups up to and including the entry's)
    int n;
};
__global__ __launch_bounds__(256) void step_sums_kernel(StepSums s)
{
    const int b = blockIdx.x;
    int first = 0, i = 0;
    while (i < s.n - 1 && b >= s.late[i].blocks) first = s.late[i++].blocks;
    const clg_late_sums &l = s.late[i];
    if (l.kind == kLateBin) bin_sums(reinterpret_cast<const BinSums &>(l.field), b - first);
    else if (l.kind == kLateTree) tree_logit_grad<false>(reinterpret_cast<const TreeSums &>(l.field), b - first);
    else reduce_coef_partials(reinterpret_cast<const CoefSums<float> &>(l.field), b - first);
}

}  // namespace

extern "C" int clg_train_prepare(const clg_train_block *blocks, int n_blocks, const float *logits0, const float *logits1, const float *logits2,
                                 const int32_t *ids, float *coef, float *probs, int64_t roots, void *stream)
{
    const char *name = "clg_train_prepare";
    if (int e = clg_check_tree(name, 1, roots, 1)) return e;
    CLG_REQUIRE(blocks && n_blocks > 0 && n_blocks <= kMaxStepBlocks, "%s: 1 to %d blocks", name, kMaxStepBlocks);
    CLG_REQUIRE(logits0 && logits1 && logits2 && ids && coef, "%s: null pointer argument", name);
    StepPrepare a = {};
    PrepArgs bin_args = {};
    Geom bin_geom = {};
    const TreeFold trees = {{{logits0, logits1, logits2}}, ids, coef, probs, (int)roots, 0};
    int64_t end = 0;
    const clg_train_block *bin = nullptr;
    for (int i = 0; i < n_blocks; ++i) {
        const clg_train_block &b = blocks[i];
        if (b.not_binary == nullptr) continue;
        CLG_REQUIRE(bin == nullptr, "%s: one binary block at most", name);
        bin = &b;
        int count = 0;
        if (int e = clg_bin_prepare_args(name, CLG_F32, &b.geom, b.x, b.logits, b.selection, b.scratch, true, b.not_binary, &bin_geom, &bin_args, &count))
            return e;
        a.bin_end = (int)(end += count);
    }
    end += clg_ceil_div(roots * 7, 256);
    CLG_REQUIRE(end < (1 << 23), "%s: problem too large for one launch", name);
    a.tree_end = (int)end;
    for (int i = 0; i < n_blocks; ++i) {
        const clg_train_block &b = blocks[i];
        if (&b == bin) continue;
        CLG_REQUIRE(b.logits && b.selection && b.probs && b.scratch, "%s: null pointer in block %d", name, i);
        BlockPrepare &p = a.block[a.blocks++];
        PairPlan plan;
        bool pair = false;
        if (int e = clg_forward_pair_plan(name, &b.geom, b.feature_major != 0, &p.g, &plan, &pair)) return e;
        p.logits = b.logits;
        p.sel = b.selection;
        p.probs = b.probs;
        if (pair) {
            p.table = clg_pair_table(plan, b.scratch);
            p.at = pair_offsets(plan);
        }
        end += clg_ceil_div((int64_t)p.g.c * 7, 256);
        CLG_REQUIRE(end < (1 << 23), "%s: problem too large for one launch", name);
        p.end = (int)end;
    }
    hipLaunchKernelGGL(step_prepare_kernel, dim3((unsigned)end), dim3(256), 0, clg_stream(stream), trees, bin_args, bin_geom, a);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}

extern "C" int clg_late_sums_run(const clg_late_sums *late, int n, void *stream)
{
    const char *name = "clg_late_sums_run";
    CLG_REQUIRE(n >= 0 && n <= kMaxLate && (late || n == 0), "%s: 0 to %d entries", name, kMaxLate);
    StepSums s = {};
    int64_t end = 0;
    for (int i = n - 1; i >= 0; --i) {                                // (a binary block, whose sums take longest, comes last in a backward pass)
        if (late[i].kind == kLateNone) continue;
        CLG_REQUIRE(late[i].kind >= kLateCoef && late[i].kind <= kLateTree && late[i].blocks > 0, "%s: entry %d is not what a backward call left", name, i);
        s.late[s.n] = late[i];
        end += late[i].blocks;
        CLG_REQUIRE(end < (1 << 24), "%s: problem too large for one launch", name);
        s.late[s.n++].blocks = (int)end;
    }
    if (s.n == 0) return CLG_OK;
    hipLaunchKernelGGL(step_sums_kernel, dim3((unsigned)end), dim3(256), 0, clg_stream(stream), s);
    CLG_CHECK_LAUNCH(name);
    return CLG_OK;
}
