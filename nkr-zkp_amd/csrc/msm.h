// Pippenger multi-scalar multiplication over G1 and G2 for gfx950.
//
// Design (MI355X-first):
//  * Proving-key bases are fixed per circuit, so `prepare` stores, for every
//    signed-digit window w, the shifted copy 2^(c*w) * P_i (affine, 64 B for
//    G1 / 128 B for G2).  All windows then share ONE set of B = 2^(c-1)
//    buckets: no per-window bucket reduction and no doubling chain at the end.
//    The copies cost W*n bases of HBM (about 1 GiB for a 2^20-point G1 key),
//    which a 288 GB device affords.
//  * Scalars are recoded into signed c-bit digits; a counting sort groups the
//    (window, point, sign) entries by bucket: about one workgroup per CU
//    histograms a contiguous slice of scalars in LDS and writes its counts as
//    one row of a (workgroups x B) matrix, a column scan turns the matrix into
//    per-(workgroup, bucket) offsets, and an LDS-cursor scatter places the
//    entries -- no global atomics, no inter-workgroup waiting and no host
//    round trip.
//  * Several MSMs run as one batch ("jobs"): every stage below is a single
//    launch over all jobs, so the latency of each reduction level is paid
//    once per batch, not once per MSM.
//      1. accumulate: every lane sums an equally long run of the sorted
//         entries, one partial sum per bucket it meets (mixed affine
//         additions into XYZZ);
//      2. fold: buckets left with more than 128 partial sums (skewed digit
//         distributions, e.g. witnesses that are mostly 0 or 1) are folded
//         64:1, a wave per sum, until they are not; others are untouched;
//      3. complete: 1..16 lane groups per bucket, strided partial sums then
//         a shuffle tree, give the bucket sums S_m;
//      4. bit planes: a log-depth tree merges bucket blocks into
//         U_j = sum over m with bit j of S_m (c points per job), several
//         levels per launch inside LDS.
//    Stages 2-4 are chains of additions with few in flight, so each addition
//    is shared by a group of lanes (coop29.h); which buckets need what is
//    planned from the schedules in one launch before the accumulation.
//    The host combines sum_j 2^j U_j (c doublings) and normalises.
// The reference computes the same sums with libff multi_exp<BDLO12>
// (third_party/.../libff/algebra/scalar_multiplication/multiexp.tcc:165-282);
// the affine result is unique, so it matches the reference bit for bit.
#pragma once

#include <algorithm>
#include <type_traits>
#include <vector>

#include "curve.h"
#include "curve29.h"
#include "msm_plan.h"
#include "runtime.h"

namespace nkr {

// Process-wide MSM tuning knobs: the accumulation lanes of a launch
// (2^target_log, 10 .. 22; at kMsmTargetDefault, which it starts at, MsmLanes'
// own) and the most lane groups that complete one bucket (1 .. 16, a power of
// two).  Set them before proving, not while proofs run.
void msm_set_shape(uint32_t target_pieces_log, uint32_t complete_lanes_cap);
// The lanes of a group's launches (msm_lanes_of) for a target_log, or (0) for
// the process-wide setting.
MsmLanes msm_lanes(bool g2, uint32_t target_log = 0);
uint32_t msm_complete_lanes_cap();
// Both process-wide knobs in one word: launches captured under one value are
// not replayed under another.
uint64_t msm_shape_key();

// Device bytes of an MsmBatch that runs jobs of these totals
// (msm_schedule_sizes has a schedule's).
template <class F>
uint64_t msm_batch_bytes(const MsmTotals &jobs);

// Window-shifted affine bases of one proving-key vector.
template <class F>
class MsmBases {
public:
    // `jacobian` is a device array of n reference-layout Jacobian points
    // (any Z, infinity as Z = 0); `perm` optionally reorders them
    // (base i = jacobian[perm[i]]).
    void prepare(const Jacobian<F> *jacobian, const uint32_t *perm, const MsmPlan &plan, hipStream_t stream);
    const Affine<F> *data() const { return pts_.get(); }
    const MsmPlan &plan() const { return plan_; }
    size_t bytes() const { return pts_.bytes(); }

private:
    MsmPlan plan_;
    DeviceBuffer<Affine<F>> pts_;
};

// The terms i < n for which a[i] or b[i] (device arrays) is not infinity, in
// order.  Synchronises the stream.
void msm_finite_terms(const g1_jac *a, const g2_jac *b, uint32_t n, std::vector<uint32_t> &terms, hipStream_t stream);

// Signed-digit recoding and bucket sort of one scalar vector; shared by every
// MSM that uses the same scalars (the witness drives four of the five).
// Entirely asynchronous on `stream`.
class MsmSchedule {
public:
    // pick: optional device list of plan.n scalar numbers; term i's scalar is
    // then scalars_mont[pick[i]] (for bases prepared with the same list).
    void build(const fr_t *scalars_mont, const uint32_t *pick, const MsmPlan &plan, hipStream_t stream,
               StageTimer *timer = nullptr);
    // Sizes the buffers for `plan`; returns the scalars per sort workgroup.
    uint32_t prepare(const MsmPlan &plan);
    const MsmPlan &plan() const { return plan_; }
    // Device counter: entries (non-zero digits).
    const uint32_t *totals() const { return bucket_start_.get() + plan_.B; }
    // Device bytes held, and their release (the next prepare reallocates).
    uint64_t device_bytes() const
    {
        return sorted_.bytes() + bucket_start_.bytes() + in_tile_.bytes() + tile_total_.bytes() +
               block_count_.bytes();
    }
    void release_device()
    {
        sorted_.release();
        bucket_start_.release();
        in_tile_.release();
        tile_total_.release();
        block_count_.release();
    }

    MsmPlan plan_;
    uint32_t blocks_ = 0;
    DeviceBuffer<uint32_t> sorted_;        // entries: sign << 31 | (w * n + i)
    DeviceBuffer<uint32_t> bucket_start_;  // B + 1, the last the entry count
    DeviceBuffer<uint32_t> in_tile_;       // B: bucket starts within 64-bucket tiles
    DeviceBuffer<uint32_t> tile_total_;    // entries of each tile
    DeviceBuffer<uint32_t> block_count_;   // blocks x B: per-workgroup counts, then offsets
};

// Many schedules with one launch per sort phase (histogram, scan, scatter)
// instead of three launches per schedule.  Same result as
// MsmSchedule::build for each of them.
class MsmScheduleBatch {
public:
    struct Item {
        MsmSchedule *sched;
        const fr_t *scalars_mont;
        const uint32_t *pick;
        MsmPlan plan;
    };
    // graph: the launches are being captured into a graph that is replayed
    // later, so nothing here may wait on the host (no staging event is
    // recorded; the caller synchronises its streams before the staging
    // buffers are written again).
    void build(const std::vector<Item> &items, hipStream_t stream, bool graph = false);
    uint64_t device_bytes() const { return table_.bytes(); }
    void release_device() { table_.release(); }

private:
    PinnedStaging<uint8_t> stage_;
    DeviceBuffer<uint8_t> table_;
};

// The form of the partial sums between the accumulation and the bit planes:
// the reduced-radix form (curve29.h) through fold, completion and tree, so
// no addition converts.  The bit planes handed to the host are canonical.
template <class F>
struct MsmPartial;
template <>
struct MsmPartial<fq_t> {
    using type = Xyzz29<FqParams>;
};
template <>
struct MsmPartial<fq2_t> {
    using type = Xyzz2_29<FqParams>;
};
template <class F>
using partial_t = typename MsmPartial<F>::type;

// Stage indices used with StageTimer by the MSM code.
enum MsmStage { kStageSort = 3, kStageAccumulate = 4, kStageFold = 5, kStageAccumulateG2 = 7 };

template <class F>
struct MsmJob {
    const MsmBases<F> *bases;
    const MsmSchedule *sched;
    Xyzz<F> *planes;   // device output: c points U_0 .. U_{c-1}
    uint32_t piece_min = 1;  // shortest run of an accumulation lane of this job
};

// Runs a batch of MSMs of one group (all with the same window width).
template <class F>
class MsmBatch {
public:
    // The lanes of the batch's accumulations (msm_lanes), instead of the
    // process-wide setting as of each layout.
    void set_lanes(const MsmLanes &lanes)
    {
        own_lanes_ = lanes;
        have_lanes_ = true;
    }
    // graph: as MsmScheduleBatch::build.
    void run(const std::vector<MsmJob<F>> &jobs, hipStream_t stream, StageTimer *timer = nullptr,
             bool graph = false);
    // Device bytes held by the batch's work buffers, and their release (the
    // next run reallocates what it needs).
    uint64_t device_bytes() const
    {
        return seg_base_.bytes() + seg_count_.bytes() + class_count_.bytes() + class_list_.bytes() +
               jobs_dev_.bytes() + lane_base_.bytes() + pool_.bytes() + sums_.bytes() + reg_start_.bytes() +
               reg_count_.bytes() + recs_.bytes() + state_.bytes() + tree_[0].bytes() + tree_[1].bytes();
    }
    void release_device()
    {
        seg_base_.release();
        seg_count_.release();
        class_count_.release();
        class_list_.release();
        jobs_dev_.release();
        lane_base_.release();
        pool_.release();
        sums_.release();
        tree_[0].release();
        tree_[1].release();
        reg_start_.release();
        reg_count_.release();
        recs_.release();
        state_.release();
        key_.clear();  // the layout cache refers to the released buffers
    }

    // The jobs' layout, and the lanes it was sized for, are those the batch's
    // buffers already hold.
    bool layout_matches(const std::vector<MsmJob<F>> &jobs) const;

private:
    MsmLanes wanted_lanes() const { return have_lanes_ ? own_lanes_ : msm_lanes(std::is_same<F, fq2_t>::value); }
    void layout(const std::vector<MsmJob<F>> &jobs, hipStream_t stream);
    std::vector<const void *> key_;
    MsmSizes sizes_;                 // as of the layout
    MsmLanes lanes_{}, own_lanes_{};               // lanes_: as of the layout
    bool have_lanes_ = false;
    DeviceBuffer<uint32_t> seg_base_, seg_count_, class_count_, class_list_, lane_base_;
    DeviceBuffer<uint8_t> jobs_dev_, recs_, state_;
    PinnedStaging<uint8_t> jobs_stage_;
    DeviceBuffer<partial_t<F>> pool_, sums_, tree_[2];
    DeviceBuffer<uint32_t> reg_start_, reg_count_;
};

// Host: sum_j 2^j U_j, then the reference's affine form (Z = 1, or (0, 1, 0)).
template <class F>
Jacobian<F> msm_finish(const Xyzz<F> *planes_host, uint32_t c);
// The same sum left in XYZZ form (not normalised).
template <class F>
Xyzz<F> msm_sum(const Xyzz<F> *planes_host, uint32_t c);

// Whole-vector convenience used by the standalone operator API.
template <class F>
class MsmContext {
public:
    MsmContext(const Jacobian<F> *bases_dev, uint32_t n, uint32_t c_override, hipStream_t stream);
    Jacobian<F> run(const fr_t *scalars_dev, hipStream_t stream);
    const MsmPlan &plan() const { return bases_.plan(); }

private:
    MsmBases<F> bases_;
    MsmSchedule sched_;
    MsmBatch<F> batch_;
    DeviceBuffer<Xyzz<F>> planes_;
};

}  // namespace nkr
