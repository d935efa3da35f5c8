// Gate fusion (lgh_fused.hip): pass scheduling and fused forward / adjoint
// passes.  Internal to liblgh.so.
#pragma once

#include <functional>
#include <memory>
#include <vector>

#include "lgh_internal.hpp"

namespace lgh {

// One fused pass: gates (indices into the compiled op list, in execution
// order) whose dense targets are lane bits or register bits.  Lane position
// p (bit p of the lane id) carries index bit lane_bits[p]; the lowest lane
// positions always carry the lowest index bits, so that every load covers
// whole runs of consecutive amplitudes.  A standalone pass holds one gate
// that the fused kernels cannot run.
struct Pass {
    bool standalone = false;
    int lane_bits[6] = {0, 1, 2, 3, 4, 5};
    int reg_bits[4] = {0, 0, 0, 0}; // the first rb entries are used
    std::vector<int> ops;
};

void set_fusion(int enabled);
// register bits of forward and adjoint passes (3 or 4 each)
void set_tile_bits(int forward, int adjoint);
int fusion_enabled();
// caps on the wavefronts of the forward and adjoint passes' grids (0: default)
void set_pass_waves(int64_t forward, int64_t adjoint);
// rb: register bits of the passes (tile = 2^(6 + rb) amplitudes per wavefront)
bool fusable(const KOp &k, int n, int rb);
// trainable_slot[i] >= 0 marks gates whose generator overlap is accumulated
// (at most max_slots per pass: kMaxSlots for the batched kernels,
// kMaxSlotsSv for the single-state adjoint kernel); empty for the forward
// direction.
// fixed_lanes: the lane positions 0..fixed_lanes-1 carry index bits
// 0..fixed_lanes-1 in every pass; the scheduler chooses the index bits of the
// other lane positions per pass, like the register bits (6: all lane bits
// fixed).  max_slots does not matter without trainable gates.
std::vector<Pass> schedule_passes(const std::vector<KOp> &ops, int n, const std::vector<int> &trainable_slot,
                                  int rb, int fixed_lanes, int max_slots);
// schedule_passes through a cache keyed by the gates' structure (the
// schedule does not depend on parameter values).
std::shared_ptr<const std::vector<Pass>> schedule_passes_cached(const std::vector<KOp> &ops, int n,
                                                                const std::vector<int> &trainable_slot, int rb,
                                                                int fixed_lanes, int max_slots);
// lgh_set_lean_passes: passes of lean gate forms run in the lean kernels
bool lean_enabled();
// Host-side plan of the fused passes a gate sequence gets (no device use):
// forward passes, or adjoint passes with every parametric gate trainable.
struct FusionPlan {
    int32_t passes = 0, standalone = 0, runs = 0, run_members = 0, lean = 0;
};
FusionPlan plan_passes(const lgh_op *ops, int64_t num_ops, int n, bool adjoint, lgh_dtype dtype);

// Forward application of a compiled op list through fused passes.
void fused_apply(lgh_sv *sv, const std::vector<KOp> &kops);

// One observable's reverse sweep.
struct AdjSweep {
    lgh_sv *lam;         // lambda: written by every pass
    const void *lam_src; // where the first pass reads it (null: lam's own contents)
    lgh_sv *bra;         // the observable's state
    double *jac_row;     // device row of the Jacobian
    // An observable state that the sweep forms itself: bra = Z-word(zmask)
    // lambda, inside the first reverse pass when that pass is fused; otherwise
    // `materialize` forms it before lambda first changes.
    bool bra_from_z = false;
    uint64_t zmask = 0;
    std::function<void()> materialize;
};

// One sweep's arrays.  A launch of several sweeps reads them from a device
// table, one entry per sweep; a launch of one has them as kernel arguments (a
// table pointer of null), which saves a copy per call and a chain of two reads
// from memory at the start of every kernel.
struct AdjArrays {
    const void *lam_src; // lambda's starting values
    void *lam, *bra;
    uint64_t zmask;
    double *jac_row;
};

// A reverse step of a gate that mixes pairs of basis states (KOp::npair), on
// lambda and the observable state of `count` sweeps (lgh_adjoint.hip): with a
// generator, workgroup b of sweep y leaves its share of Im<bra|G lambda> in
// partials[y * stride + b].
unsigned adj_pairs_blocks(int n, const KOp &udag);
void launch_adj_pairs(StreamCtx *ctx, lgh_dtype dtype, int n, const KOp &udag, const KGen *gen, const AdjArrays &one,
                      const AdjArrays *table, int count, double *partials, uint64_t stride);

// Applies U^dagger of one non-fusable gate to a sweep's lambda and observable
// state; with a generator, stores factor * Im<bra|G lambda> into jac_row[col].
using StandaloneStep =
    std::function<void(const AdjSweep &sweep, const KOp &udag, const KGen *gen, int64_t col, double factor)>;

// The fused reverse passes of a circuit, scheduled once.  A pass is built and
// uploaded in the first run, just before its launch, so that the host works on
// it while the device runs the pass before.  again: more than one run follows;
// the descriptors are then kept on the device.  udag: the ops in forward order
// compiled as U^dagger; slot_col[i]: Jacobian column of a trainable gate or
// -1; factor[i] = -2 s (inverse ? -1 : 1).
class AdjPasses {
  public:
    AdjPasses(const lgh_sv *like, const std::vector<KOp> &udag, const std::vector<KGen> &gens,
              const std::vector<int> &slot_col, const std::vector<double> &factor, bool again);
    ~AdjPasses();
    AdjPasses(const AdjPasses &) = delete;
    // Runs the sweeps side by side, one launch per pass for all of them.
    // partials: count * fused_partials_bytes() bytes; table: count *
    // kTableBytes bytes, both on the device and the call's own.
    static constexpr size_t kTableBytes = 64;
    void run(const AdjSweep *sweeps, int count, double *partials, void *table, const StandaloneStep &standalone);

  private:
    // A fused pass, a gate on its own, or a run of gates that mix pairs of
    // basis states, whose overlaps are summed and stored together at its end.
    struct Step {
        std::vector<int> pairs;   // that run's gates, in execution order
        int op = -1;              // a gate on its own, or -1
        unsigned blocks = 0;      // workgroups of each of the run's trainable gates
        const unsigned char *dev = nullptr; // descriptors; offsets into them:
        size_t o_ops = 0, o_gens = 0, o_cols = 0, o_facs = 0;
        int row = 0;              // a fused pass's first row of partials
        int pending = 0;          // slots whose columns and factors are in dev: its own and those of passes before it
        bool store = false;       // they are stored after this step
        int level = 0;
    };
    struct Blob; // host copy of a step's descriptors
    template <class R>
    void run_t(const AdjSweep *sweeps, int count, double *partials, void *table, const StandaloneStep &s);
    const unsigned char *to_device(const Blob &blob);
    const std::vector<KOp> &udag_;
    const std::vector<KGen> &gens_;
    const std::vector<int> &slot_col_;
    const std::vector<double> &factor_;
    StreamCtx *ctx_;
    int n_, device_, rb_, waves_per_cu_;
    lgh_dtype dtype_;
    bool again_, built_ = false;
    std::shared_ptr<const std::vector<Pass>> passes_;
    std::vector<Step> steps_;                    // in execution order
    std::vector<std::pair<void *, size_t>> kept_; // descriptors of every step, where runs follow the first
};
size_t fused_partials_bytes(int n, int device);

} // namespace lgh
