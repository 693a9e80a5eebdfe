// MSM sizing: window choice, accumulation lanes, folds, and the bounds the
// device buffers are sized from.  No HIP, so that a CPU test can check every
// one of them; what the planning kernel uses as well is constexpr.
#pragma once

#include <algorithm>
#include <cstdint>

#include "error.h"

namespace nkr {

// Accumulation lanes.  A batch's E sorted entries (non-zero digits, known on
// the device) are split evenly: each lane sums ceil(E / lanes) consecutive
// ones, a serial chain, and leaves about one partial sum to the bucket
// reduction, whose additions have a quarter (G2: an eighth) of the chip's
// lanes' parallelism but only 2.5 us (3.8 us) of latency.  lanes[i] applies
// while E is below below[i] (lanes[3] from below[2] on):
//   one wave per SIMD (65536 lanes) while the chain is short: 4.6 us per
//   addition at G1, 13 us at G2, with single entries at the smallest sizes;
//   more waves (G1 up to three per SIMD, G2 two) once what they gain in
//   throughput (G1 5.0 -> 4.0 us per wave and SIMD, G2 13 -> 12.2) is more
//   than the reduction of their partials costs (10 and 29 us per 65536);
//   two full rounds of those for the largest, whose last round then ends
//   early where another stream's kernels took some of the slots.
// One MSM on MI355X, us, just below and above each limit (2^16, 2^17 and 2^18
// lanes; 6 * 2^16 in the last figure):
//   G1  2^22: 561, 541, 553 and 580, 556, 576 (the lines cross above 2^21)
//       2^24: 1688, 1569, 1556 and 1765, 1642, 1622
//       2^25: 3202, 2996, 2996 and 3372, 3168, 3125 against 3098
//   G2  2^21: 759, 794, 840 and 768, 823, 883 (they cross below 2^22: 1230, 1158)
//       2^23: 2140, 2022, 2033 and 2299, 2160, 2174
struct MsmLanes {
    uint32_t lanes[4];
    uint64_t below[3];
    bool operator==(const MsmLanes &o) const
    {
        return std::equal(lanes, lanes + 4, o.lanes) && std::equal(below, below + 3, o.below);
    }
};
// More entries never mean fewer lanes: a bound on the entries bounds the lanes.
constexpr bool msm_lanes_ascend(const MsmLanes &r)
{
    return r.lanes[0] <= r.lanes[1] && r.lanes[1] <= r.lanes[2] && r.lanes[2] <= r.lanes[3] &&
           r.below[0] <= r.below[1] && r.below[1] <= r.below[2];
}
constexpr MsmLanes kMsmLanesG1 = {{1u << 16, 2u << 16, 4u << 16, 6u << 16}, {1u << 22, 1u << 24, 1u << 25}};
constexpr MsmLanes kMsmLanesG2 = {{1u << 16, 1u << 16, 2u << 16, 4u << 16}, {1u << 19, 1u << 21, 1u << 23}};
static_assert(msm_lanes_ascend(kMsmLanesG1) && msm_lanes_ascend(kMsmLanesG2), "lane rule");
// The default of the lane setting (2^target_log lanes for every launch): the
// group's own lanes above.
constexpr uint32_t kMsmTargetDefault = 19;

// The lanes of a group's launches for a setting of target_log.
inline MsmLanes msm_lanes_of(bool g2, uint32_t target_log)
{
    MsmLanes r = g2 ? kMsmLanesG2 : kMsmLanesG1;
    if (target_log != kMsmTargetDefault)
        for (uint32_t &l : r.lanes) l = 1u << target_log;
    return r;
}

// The planning kernel's rules (constexpr: host and device run the same code).
// Lanes of a launch over `entries` entries.
constexpr uint32_t msm_launch_lanes(const MsmLanes &r, uint64_t entries)
{
    uint32_t lanes = r.lanes[3];
    for (int i = 2; i >= 0; --i)
        if (entries < r.below[i]) lanes = r.lanes[i];
    return lanes;
}
// Entries per lane of a launch over `entries` entries, and of one of its jobs,
// whose runs may have a minimum of their own.
constexpr uint32_t msm_piece(const MsmLanes &r, uint64_t entries)
{
    const uint32_t lanes = msm_launch_lanes(r, entries);
    return entries == 0 ? 1u : (uint32_t)((entries + lanes - 1) / lanes);
}
constexpr uint32_t msm_job_piece(uint32_t piece, uint32_t piece_min) { return piece < piece_min ? piece_min : piece; }
// Largest bucket count (c <= 16): the histograms and bucket scans hold B
// counts in one workgroup's LDS (128 KiB of gfx950's 160 KiB).
constexpr uint32_t kMsmMaxBuckets = 1u << 15;

// Folds: a launch turns the partial sums of every bucket that has more than
// kMsmDirectMax into one per kMsmFoldSpan.  8 lane groups complete kMsmDirectMax
// in fewer additions of latency than a fold and a completion take.
constexpr uint32_t kMsmFoldSpan = 64;
constexpr uint32_t kMsmDirectMax = 128;
constexpr uint32_t kMsmMaxFoldLaunches = 4;
constexpr bool msm_folds(uint64_t partials) { return partials > kMsmDirectMax; }
constexpr uint64_t msm_folded(uint64_t partials) { return (partials + kMsmFoldSpan - 1) / kMsmFoldSpan; }
// Fold launches for buckets of at most `partials` partial sums.
constexpr uint32_t msm_fold_launches(uint64_t partials)
{
    uint32_t launches = 0;
    for (; msm_folds(partials); partials = msm_folded(partials)) ++launches;
    return launches;
}
static_assert(msm_fold_launches((1ull << 24) + 1) <= kMsmMaxFoldLaunches, "the most lanes a launch may have");

// Completion classes: 1, 2, 4, 8 or 16 lane groups per bucket (G2: up to 8, the
// groups of one wave), at most 64 lanes.
constexpr uint32_t kMsmCompleteClasses = 5;

// What the device buffers of a batch of jobs hold at most: the lanes of its
// accumulation, and from them the partial sums, the folds and the completion.
struct MsmSizes {
    uint64_t lanes = 0;    // accumulation lanes
    uint64_t buckets = 0;  // of all jobs
    uint32_t fold_launches = 0;
    // the pool of partial sums: one per (lane, bucket) at slot lane + bucket,
    // then each fold launch's outputs from fold_base on, fold_cap of them at most
    uint64_t fold_base[kMsmMaxFoldLaunches] = {}, fold_cap[kMsmMaxFoldLaunches] = {};
    uint64_t pool = 0;
    uint64_t records = 0;         // fold records of one launch
    uint64_t complete_lanes = 0;  // 64 per bucket, and each segment's padding
};
// For `jobs` jobs with `buckets` buckets and up to `entries` sorted entries in
// all, of a launch of `launch_lanes`.  A job's last lane may be a short one, so
// every job adds one; a bucket has at most a partial per lane of its job.
inline MsmSizes msm_sizes(uint64_t jobs, uint64_t entries, uint64_t buckets, uint64_t launch_lanes)
{
    MsmSizes s;
    const uint64_t job_lanes = std::min(entries, launch_lanes) + 1;
    s.lanes = job_lanes - 1 + jobs;
    s.buckets = buckets;
    s.fold_launches = msm_fold_launches(job_lanes);
    NKR_REQUIRE(s.fold_launches <= kMsmMaxFoldLaunches, "MSM launch with too many lanes to fold");
    // a launch folds buckets of more than kMsmDirectMax partials, to fewer than
    // a 32nd of them
    const uint64_t partials = s.lanes + buckets;
    uint64_t left = partials;
    s.pool = partials;
    for (uint32_t L = 0; L < kMsmMaxFoldLaunches; ++L) {
        left = left / 32 + 1;
        s.fold_base[L] = s.pool;
        s.fold_cap[L] = left;
        s.pool += left;
    }
    s.records = partials / (kMsmDirectMax + 1) + 1;
    s.complete_lanes = (buckets + jobs * kMsmCompleteClasses) * 64;
    return s;
}

struct MsmPlan {
    uint32_t n = 0;         // number of bases / scalars
    uint32_t c = 0;         // window width in bits
    uint32_t W = 0;         // windows (signed digits), c*W >= 255
    uint32_t B = 0;         // buckets 1..B, B = 2^(c-1)

    // ~3/4 log2 n bits (16 from 2^20 terms up), or c_override when non-zero.
    static MsmPlan choose(uint32_t n, uint32_t c_override = 0)
    {
        NKR_REQUIRE(n > 0, "MSM needs at least one term");
        MsmPlan p;
        p.n = n;
        uint32_t c = c_override;
        if (c == 0) {
            const unsigned lg = ceil_log2(n);
            // 16 bits from 2^20 terms up: 16 windows instead of 17, and its
            // 128 KiB bucket histogram still fits one workgroup's LDS.
            c = lg >= 20 ? 16u : std::max(4u, std::min(15u, (lg * 3 + 2) / 4));
            // Scalars have 254 bits; a top window with only a few of them sends
            // a whole window's entries to a handful of buckets (long serial
            // chains), so move to a neighbouring width whose top window keeps
            // at least 4 bits.
            if (top_bits(c) < 4) {
                if (c < 16 && top_bits(c + 1) >= 4)
                    c += 1;
                else if (c > 4 && top_bits(c - 1) >= 4)
                    c -= 1;
            }
        }
        NKR_REQUIRE(c >= 2 && c <= 16, "MSM window must be 2..16 bits");
        p.c = c;
        p.W = (255 + c - 1) / c;
        p.B = 1u << (c - 1);
        NKR_REQUIRE((uint64_t)p.W * n < (1ull << 31), "MSM too large for 31-bit entry indices");
        return p;
    }
    // Bits of a 254-bit scalar left for the top window of width cc.
    static uint32_t top_bits(uint32_t cc) { return 254 - cc * ((255 + cc - 1) / cc - 1); }

    uint64_t max_entries() const { return (uint64_t)n * W; }
};

// The plan of the witness's MSMs over n columns: at most 15 bits, whose
// schedule is built beside the transforms.
inline MsmPlan msm_witness_plan(uint32_t n, uint32_t c_override = 0)
{
    const MsmPlan p = MsmPlan::choose(n, c_override);
    return p.c > 15 ? MsmPlan::choose(n, 15) : p;
}

// The plan of bs1 and bs2 when `finite` of the witness's columns have a finite
// point: the witness's own, or, where at least a quarter of the columns go, one
// for the columns that stay.  A width the caller asked for was for all of the
// columns; these may be a hundredth of them.
inline MsmPlan msm_b_plan(const MsmPlan &witness, uint32_t finite)
{
    const uint32_t n = std::max(1u, finite);  // an MSM has at least one term
    if (n == witness.n || n > witness.n - witness.n / 4) return witness;
    return msm_witness_plan(n);
}

// What the sizes of a batch's jobs of one group depend on; the totals of several
// batches add up to those of their union.
struct MsmTotals {
    uint64_t jobs = 0, entries = 0, buckets = 0;
    void add(const MsmPlan &p)
    {
        ++jobs;
        entries += p.max_entries();
        buckets += p.B;
    }
    void add(const MsmTotals &o)
    {
        jobs += o.jobs;
        entries += o.entries;
        buckets += o.buckets;
    }
    MsmSizes sizes(const MsmLanes &rule) const
    {
        return msm_sizes(jobs, entries, buckets, msm_launch_lanes(rule, entries));
    }
};

// Sort workgroups: about one per CU, each histogramming a contiguous slice of
// at least kMsmSortMinPerBlock scalars.
constexpr uint32_t kMsmSortBlocksTarget = 256;
constexpr uint32_t kMsmSortMinPerBlock = 256;
inline uint32_t msm_sort_blocks(uint32_t n)
{
    return std::max<uint32_t>(1, std::min<uint32_t>(kMsmSortBlocksTarget, div_up(n, kMsmSortMinPerBlock)));
}
// The words of a schedule's buffers.
struct MsmScheduleSizes {
    uint64_t sorted, bucket_start, in_tile, tile_total, block_count;
    uint64_t bytes() const { return 4 * (sorted + bucket_start + in_tile + tile_total + block_count); }
};
inline MsmScheduleSizes msm_schedule_sizes(const MsmPlan &p)
{
    const uint64_t entries = (p.max_entries() + 3) & ~uint64_t(3);  // read in blocks of four
    return {entries, uint64_t(p.B) + 1, p.B, div_up(p.B, 64), uint64_t(msm_sort_blocks(p.n)) * p.B};
}

}  // namespace nkr
