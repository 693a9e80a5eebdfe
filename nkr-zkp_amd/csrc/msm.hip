// Pippenger MSM kernels for gfx950 (see msm.h for the design).
#include "msm.h"

#include "block_inverse.h"
#include "coop29.h"
#include "curve29.h"

#include <algorithm>
#include <array>
#include <cstring>
#include <mutex>
#include <type_traits>

namespace nkr {

namespace {

constexpr uint32_t kEntryMask = 0x7fffffffu;
constexpr uint32_t kSortThreads = 1024;
// Column scan tile: 64 buckets x kScanGroups row groups per workgroup.
constexpr uint32_t kScanGroups = 16;
// LDS per tree workgroup (two buffers of 2^h blocks): two workgroups per CU.
constexpr size_t kTreeLds = 64 * 1024;
constexpr uint32_t kTreeThreads = 256;
constexpr uint32_t kPlanThreads = 1024;
// Lane groups of an addition per wave (coop29.h).
template <class F>
constexpr uint32_t kWaveGroups = 64 / Coop<F>::kLanes;

// One bucket to fold at one level: its partials at pool[src .. src + cnt)
// become ceil(cnt / kMsmFoldSpan) sums, the level's outputs `start` ...
struct FoldRec {
    uint32_t start, src, cnt;
};

// A batch's reduction plan on the device (k_reduce_plan).  `ticket` and
// `fold_ctr` are zero between launches; fold_count holds their last values.
struct ReduceState {
    uint32_t ticket;
    uint32_t piece;  // entries per accumulation lane (msm_piece)
    unsigned long long fold_ctr[kMsmMaxFoldLaunches];  // records << 32 | outputs
    unsigned long long fold_count[kMsmMaxFoldLaunches];
};

template <class F>
struct JobDev {
    const Affine<F> *bases;
    const uint32_t *sorted;
    const uint32_t *bucket_start;  // B + 1
    uint32_t *reg_start;           // B: where bucket k's partials to complete live in the pool
    uint32_t *reg_count;           // B
    partial_t<F> *sums;            // B: S_{k+1}
    partial_t<F> *tree[2];         // B each
    Xyzz<F> *planes;               // c (canonical)
    uint32_t B, c;
    uint32_t b_off;  // buckets of the jobs before this one
    uint32_t piece_min;
};

// ------------------------------------------------------------ digit recoding
// Signed c-bit digits of an integer scalar (< 2^254): d_w in [-2^(c-1), 2^(c-1)],
// top window unsigned so that c*W >= 255 suffices.
template <class Fn>
__device__ __forceinline__ void for_each_digit(const fr_t &s, uint32_t c, uint32_t W, Fn fn)
{
    const uint32_t half = 1u << (c - 1);
    const uint32_t full = 1u << c;
    const uint32_t mask = full - 1u;
    uint32_t carry = 0;
    for (uint32_t w = 0; w < W; ++w) {
        const uint32_t off = w * c;
        const uint32_t word = off >> 5, sh = off & 31u;
        // selects instead of s.l[word]: a dynamically indexed register array
        // would live in scratch memory
        uint64_t lo = 0, hi = 0;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            lo = k == word ? s.l[k] : lo;
            hi = k == word + 1 ? s.l[k] : hi;
        }
        uint32_t v = (uint32_t)(((hi << 32) | lo) >> sh) & mask;
        v += carry;
        int32_t d;
        if (w + 1 < W && v >= half) {
            d = (int32_t)v - (int32_t)full;
            carry = 1;
        } else {
            d = (int32_t)v;
            carry = 0;
        }
        if (d != 0) {
            // Canonical scalars (< r) never exceed 2^(c-1); the clamp keeps a
            // malformed input inside the bucket arrays instead of faulting.
            const int32_t lim = (int32_t)half;
            fn(w, d > lim ? lim : (d < -lim ? -lim : d));
        }
    }
}

// Histogram of the bucket magnitudes of scalars [b * per_block, ...) in LDS,
// written as row b of the (blocks x B) count matrix.
// Term i's scalar is scalars[pick[i]], or scalars[i] without a list.
__device__ __forceinline__ void hist_block(uint32_t *hist, const fr_t *__restrict__ scalars,
                                          const uint32_t *__restrict__ pick, uint32_t n, uint32_t c, uint32_t W,
                                          uint32_t B, uint32_t per_block, uint32_t b,
                                          uint32_t *__restrict__ block_count)
{
    for (uint32_t k = threadIdx.x; k < B; k += blockDim.x) hist[k] = 0;
    __syncthreads();
    const uint32_t beg = b * per_block;
    const uint32_t end = min(n, beg + per_block);
    for (uint32_t i = beg + threadIdx.x; i < end; i += blockDim.x) {
        const fr_t s = fp_from_mont(scalars[pick ? pick[i] : i]);
        for_each_digit(s, c, W, [&](uint32_t, int32_t d) {
            const uint32_t m = (uint32_t)(d < 0 ? -d : d);
            atomicAdd(&hist[m - 1], 1u);
        });
    }
    __syncthreads();
    uint32_t *row = block_count + (size_t)b * B;
    for (uint32_t k = threadIdx.x; k < B; k += blockDim.x) row[k] = hist[k];
}

// Exclusive prefix of f(0) .. f(len - 1) into out[0 .. len], by one workgroup
// (whole waves).
template <class Fn>
__device__ void group_prefix(uint32_t len, uint32_t *__restrict__ out, Fn f)
{
    __shared__ uint32_t wave_sum[16];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    uint32_t base = 0;
    for (uint32_t k0 = 0; k0 < len; k0 += blockDim.x) {
        const uint32_t k = k0 + threadIdx.x;
        const uint32_t v = k < len ? f(k) : 0u;
        uint32_t incl = v;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, off);
            if (lane >= (uint32_t)off) incl += y;
        }
        if (lane == 63) wave_sum[wave] = incl;
        __syncthreads();
        uint32_t run = base;
        for (uint32_t w = 0; w < waves; ++w) {
            if (w < wave) run += wave_sum[w];
            base += wave_sum[w];
        }
        if (k < len) out[k] = run + incl - v;
        __syncthreads();
    }
    if (threadIdx.x == 0) out[len] = base;
    __syncthreads();
}

// Column scan of the count matrix for buckets [64 tile, 64 tile + 64): row b
// of block_count becomes the offset of workgroup b's entries inside each
// bucket (the sum of the rows above it), and the columns' totals the buckets'
// starts within the tile (in_tile) and the tile's total; the scatter adds the
// tiles' prefix.  64 x kScanGroups threads: each row group sums its rows, the
// groups' sums are scanned in LDS, then each group rewrites its rows as
// offsets, and the last group scans its totals.
__device__ __forceinline__ void colscan_tile(uint32_t *__restrict__ block_count, uint32_t blocks, uint32_t B,
                                            uint32_t tile, uint32_t *__restrict__ in_tile,
                                            uint32_t *__restrict__ tile_total)
{
    __shared__ uint32_t part[kScanGroups][64];
    const uint32_t kk = threadIdx.x & 63u, g = threadIdx.x >> 6;
    const uint32_t k = tile * 64 + kk;
    const uint32_t rows = (blocks + kScanGroups - 1) / kScanGroups;
    const uint32_t r0 = min(blocks, g * rows), r1 = min(blocks, r0 + rows);
    uint32_t sum = 0;
    if (k < B)
        for (uint32_t r = r0; r < r1; ++r) sum += block_count[(size_t)r * B + k];
    part[g][kk] = sum;
    __syncthreads();
    uint32_t run = 0;
    for (uint32_t h = 0; h < g; ++h) run += part[h][kk];
    if (k < B) {
        for (uint32_t r = r0; r < r1; ++r) {
            uint32_t *p = block_count + (size_t)r * B + k;
            const uint32_t v = *p;
            *p = run;
            run += v;
        }
    }
    if (g == kScanGroups - 1) {
        const uint32_t v = k < B ? run : 0u;
        uint32_t incl = v;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, off);
            if (kk >= (uint32_t)off) incl += y;
        }
        if (k < B) in_tile[k] = incl - v;
        if (kk == 63) tile_total[tile] = incl;
    }
}

// Every workgroup scans the (at most kMsmMaxBuckets / 64) tile totals for its
// own cursors, which costs less than a launch that would do it once; the
// first one writes the bucket starts for the kernels after it.
__device__ __forceinline__ void scatter_block(uint32_t *cursor, const fr_t *__restrict__ scalars,
                                             const uint32_t *__restrict__ pick, uint32_t n, uint32_t c, uint32_t W,
                                             uint32_t B, uint32_t per_block, uint32_t b,
                                             const uint32_t *__restrict__ in_tile,
                                             const uint32_t *__restrict__ tile_total,
                                             const uint32_t *__restrict__ block_off,
                                             uint32_t *__restrict__ bucket_start, uint32_t *__restrict__ sorted)
{
    __shared__ uint32_t tile_base[kMsmMaxBuckets / 64 + 1];
    group_prefix((B + 63) / 64, tile_base, [&](uint32_t t) { return tile_total[t]; });
    const uint32_t *row = block_off + (size_t)b * B;
    for (uint32_t k = threadIdx.x; k < B; k += blockDim.x) {
        const uint32_t start = in_tile[k] + tile_base[k / 64];
        cursor[k] = start + row[k];
        if (b == 0) bucket_start[k] = start;
    }
    if (b == 0 && threadIdx.x == 0) bucket_start[B] = tile_base[(B + 63) / 64];
    __syncthreads();
    const uint32_t beg = b * per_block;
    const uint32_t end = min(n, beg + per_block);
    for (uint32_t i = beg + threadIdx.x; i < end; i += blockDim.x) {
        const fr_t s = fp_from_mont(scalars[pick ? pick[i] : i]);
        for_each_digit(s, c, W, [&](uint32_t w, int32_t d) {
            const uint32_t m = (uint32_t)(d < 0 ? -d : d);
            const uint32_t pos = atomicAdd(&cursor[m - 1], 1u);
            sorted[pos] = (d < 0 ? 0x80000000u : 0u) | (w * n + i);
        });
    }
}

__global__ __launch_bounds__(kSortThreads) void k_hist(const fr_t *__restrict__ scalars,
                                                       const uint32_t *__restrict__ pick, uint32_t n, uint32_t c,
                                                       uint32_t W, uint32_t B, uint32_t per_block,
                                                       uint32_t *__restrict__ block_count)
{
    extern __shared__ uint32_t lds[];
    hist_block(lds, scalars, pick, n, c, W, B, per_block, blockIdx.x, block_count);
}

__global__ __launch_bounds__(64 * kScanGroups) void k_colscan(uint32_t *__restrict__ block_count, uint32_t blocks,
                                                              uint32_t B, uint32_t *__restrict__ in_tile,
                                                              uint32_t *__restrict__ tile_total)
{
    colscan_tile(block_count, blocks, B, blockIdx.x, in_tile, tile_total);
}

__global__ __launch_bounds__(kSortThreads) void k_scatter(const fr_t *__restrict__ scalars,
                                                          const uint32_t *__restrict__ pick, uint32_t n, uint32_t c,
                                                          uint32_t W, uint32_t B, uint32_t per_block,
                                                          const uint32_t *__restrict__ in_tile,
                                                          const uint32_t *__restrict__ tile_total,
                                                          const uint32_t *__restrict__ block_off,
                                                          uint32_t *__restrict__ bucket_start,
                                                          uint32_t *__restrict__ sorted)
{
    extern __shared__ uint32_t lds[];
    scatter_block(lds, scalars, pick, n, c, W, B, per_block, blockIdx.x, in_tile, tile_total, block_off, bucket_start,
                  sorted);
}

// Last index k in [0, len) with starts[k] <= p (starts[0] <= p < starts[len]).
__device__ __forceinline__ uint32_t find_segment(const uint32_t *starts, uint32_t len, uint32_t p)
{
    uint32_t lo = 0, hi = len;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (starts[mid] <= p)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// One schedule of a batched sort.
struct SortJob {
    const fr_t *scalars;
    const uint32_t *pick;
    uint32_t n, c, W, B, blocks, per_block;
    uint32_t *block_count, *in_tile, *tile_total, *bucket_start, *sorted;
};

// Workgroup blockIdx.x is sort block (blockIdx.x - block_off[j]) of job j.
__global__ __launch_bounds__(kSortThreads) void k_hist_batch(const SortJob *__restrict__ jobs,
                                                             const uint32_t *__restrict__ block_off, uint32_t J)
{
    extern __shared__ uint32_t lds[];
    const uint32_t j = find_segment(block_off, J, blockIdx.x);
    const SortJob &jb = jobs[j];
    hist_block(lds, jb.scalars, jb.pick, jb.n, jb.c, jb.W, jb.B, jb.per_block, blockIdx.x - block_off[j], jb.block_count);
}

__global__ __launch_bounds__(64 * kScanGroups) void k_colscan_batch(const SortJob *__restrict__ jobs)
{
    const SortJob &jb = jobs[blockIdx.y];
    if (blockIdx.x * 64 >= jb.B) return;
    colscan_tile(jb.block_count, jb.blocks, jb.B, blockIdx.x, jb.in_tile, jb.tile_total);
}

__global__ __launch_bounds__(kSortThreads) void k_scatter_batch(const SortJob *__restrict__ jobs,
                                                                const uint32_t *__restrict__ block_off, uint32_t J)
{
    extern __shared__ uint32_t lds[];
    const uint32_t j = find_segment(block_off, J, blockIdx.x);
    const SortJob &jb = jobs[j];
    scatter_block(lds, jb.scalars, jb.pick, jb.n, jb.c, jb.W, jb.B, jb.per_block, blockIdx.x - block_off[j], jb.in_tile,
                  jb.tile_total, jb.block_count, jb.bucket_start, jb.sorted);
}

// Accumulation lanes of a job.
template <class F>
__device__ __forceinline__ uint32_t job_lanes(const JobDev<F> &jb, uint32_t launch_piece)
{
    const uint32_t piece = msm_job_piece(launch_piece, jb.piece_min);
    return (jb.bucket_start[jb.B] + piece - 1) / piece;
}

// The plan of a batch, from the schedules' bucket starts: one launch before
// the accumulation instead of several small ones around it.
//   * the accumulation gives every lane L consecutive entries of a job's
//     sorted list, L = msm_piece of all jobs' entries or, where that is more,
//     the job's minimum; a bucket of the
//     entries [a, b) therefore gets a partial from each of the lanes a / L ..
//     (b - 1) / L, and lane l's partial of bucket k is number l + k of the job
//     (two lanes share a bucket, or one lane two buckets, never both), at
//     lanes and buckets of the jobs before it in the pool;
//   * a bucket with more than kMsmDirectMax partials gets a fold record per
//     level that brings it below (kMsmFoldSpan : 1 each); any bucket's final
//     partials become reg_start / reg_count;
//   * completion classes: a bucket with m partials is completed by 2^c lane
//     groups, the smallest c with m <= serial << c.  With the partials spread
//     over the chip's lane groups a group has (lanes + buckets) / groups of
//     them; half as many again keep most buckets in one group (the shuffle
//     levels of more idle half of them or more), and only the longer ones
//     take several.  An empty bucket's sum is infinity;
//   * the last workgroup to finish turns the counts into offsets:
//     lane_base[j] = accumulation lanes of the jobs before j, seg_base[s] =
//     lanes of the completion segments before s = kMsmCompleteClasses * j + c,
//     each padded to whole waves, and clears the counters for the next launch.
template <class F>
__global__ __launch_bounds__(kPlanThreads) void k_reduce_plan(const JobDev<F> *__restrict__ jobs, uint32_t J,
                                                     MsmLanes rule, uint32_t buckets, uint32_t max_class,
                                                     ReduceState *__restrict__ st, FoldRec *__restrict__ recs,
                                                     uint32_t rec_cap, const uint32_t *__restrict__ fold_base,
                                                     uint32_t *__restrict__ class_count,
                                                     uint32_t *__restrict__ class_list,
                                                     uint32_t *__restrict__ lane_base,
                                                     uint32_t *__restrict__ seg_count,
                                                     uint32_t *__restrict__ seg_base)
{
    const uint32_t j = blockIdx.y;
    const JobDev<F> &jb = jobs[j];
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    __shared__ unsigned long long entries;
    if (threadIdx.x == 0) entries = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < J; i += blockDim.x)
        atomicAdd(&entries, (unsigned long long)jobs[i].bucket_start[jobs[i].B]);
    __syncthreads();
    const uint32_t launch_piece = msm_piece(rule, entries);
    __shared__ uint32_t lanes_before;
    if (threadIdx.x == 0) lanes_before = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < j; i += blockDim.x)
        atomicAdd(&lanes_before, job_lanes(jobs[i], launch_piece));
    __syncthreads();
    const uint32_t piece = msm_job_piece(launch_piece, jb.piece_min);
    uint32_t m = 0;
    if (k < jb.B) {
        const uint32_t beg = jb.bucket_start[k], end = jb.bucket_start[k + 1];
        uint32_t src = lanes_before + jb.b_off + beg / piece + k;
        if (beg < end) m = (end - 1) / piece - beg / piece + 1;
        for (uint32_t L = 0; msm_folds(m); ++L) {
            const uint32_t n = (uint32_t)msm_folded(m);
            const unsigned long long at = atomicAdd(&st->fold_ctr[L], (1ull << 32) | n);
            const uint32_t start = (uint32_t)at;
            recs[(size_t)L * rec_cap + (uint32_t)(at >> 32)] = FoldRec{start, src, m};
            src = fold_base[L] + start;
            m = n;
        }
        jb.reg_start[k] = src;
        jb.reg_count[k] = m;
        if (m == 0) jb.sums[k] = partial_t<F>::infinity();
    }
    // one atomic per workgroup and class: ballots rank the lanes of a wave, and
    // the waves' counts are scanned in LDS
    __shared__ uint32_t count[kMsmCompleteClasses][kPlanThreads / 64], list_at[kMsmCompleteClasses];
    constexpr uint32_t groups = 65536 / Coop<F>::kLanes;
    const uint32_t serial = 1 + (uint32_t)(3 * (entries / launch_piece + buckets) / (2 * groups));
    uint32_t c = 0;
    while (c < max_class && (serial << c) < m) ++c;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    uint32_t rank = 0;
    for (uint32_t cc = 0; cc < kMsmCompleteClasses; ++cc) {
        const uint64_t mask = __ballot(m > 0 && c == cc);
        if (c == cc) rank = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
        if (lane == 0) count[cc][wave] = (uint32_t)__popcll(mask);
    }
    __syncthreads();
    if (threadIdx.x < kMsmCompleteClasses) {
        uint32_t sum = 0;
        for (uint32_t w = 0; w < waves; ++w) {
            const uint32_t n = count[threadIdx.x][w];
            count[threadIdx.x][w] = sum;
            sum += n;
        }
        if (sum) list_at[threadIdx.x] = atomicAdd(&class_count[kMsmCompleteClasses * j + threadIdx.x], sum);
    }
    __syncthreads();
    if (m > 0)
        class_list[((size_t)jb.b_off * kMsmCompleteClasses + (size_t)c * jb.B) + list_at[c] + count[c][wave] + rank] = k;

    // The last workgroup reads what the others left in the counters, which are
    // only touched by atomics; each of its own has returned here.
    __shared__ uint32_t last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        last = atomicAdd(&st->ticket, 1u) + 1u == gridDim.x * gridDim.y ? 1u : 0u;
        if (last) st->ticket = 0;
    }
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0) st->piece = launch_piece;
    group_prefix(J, lane_base, [&](uint32_t i) { return job_lanes(jobs[i], launch_piece); });
    group_prefix(kMsmCompleteClasses * J, seg_base, [&](uint32_t s) {
        const uint32_t n = atomicExch(&class_count[s], 0u);
        seg_count[s] = n;
        return ((n * Coop<F>::kLanes << (s % kMsmCompleteClasses)) + 63u) & ~63u;
    });
    if (threadIdx.x < kMsmMaxFoldLaunches) st->fold_count[threadIdx.x] = atomicExch(&st->fold_ctr[threadIdx.x], 0ull);
}

// The G2 accumulator of one lane with X and ZZ in registers and Y and ZZZ in
// LDS: each of Y and ZZZ is used twice per addition, far apart, and holding
// them (36 registers) across the products would push the addition's working
// set past the 256 registers a lane has at two waves per SIMD.  LDS holds
// limb i of a coordinate's 18 at [i * kAccThreads + lane], so a wave's access
// to one limb is 64 consecutive words (no bank conflicts).  The accesses are
// volatile so that the compiler neither merges the two reads of a coordinate
// nor keeps it in registers between them.
// The pointers carry the LDS address space so that the accesses compile to
// ds_read/ds_write rather than flat instructions.
constexpr uint32_t kAccThreads = 256;
typedef __attribute__((address_space(3))) volatile uint32_t lds_word_t;

template <class P>
struct Xyzz2_29Lds {
    Fq2_29<P> x, zz;
    lds_word_t *y, *zzz;  // this lane's column of each coordinate's 18 x kAccThreads words

    __device__ static Fq2_29<P> load(const lds_word_t *s)
    {
        Fq2_29<P> r;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            r.c0.l[i] = s[i * kAccThreads];
            r.c1.l[i] = s[(9 + i) * kAccThreads];
        }
        return r;
    }
    __device__ static void store(lds_word_t *s, const Fq2_29<P> &v)
    {
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            s[i * kAccThreads] = v.c0.l[i];
            s[(9 + i) * kAccThreads] = v.c1.l[i];
        }
    }
    __device__ bool is_inf() const { return zz.is_exact_zero(); }
    __device__ Fq2_29<P> X() const { return x; }
    __device__ Fq2_29<P> Y() const { return load(y); }
    __device__ Fq2_29<P> ZZ() const { return zz; }
    __device__ Fq2_29<P> ZZZ() const { return load(zzz); }
    __device__ void set(const Fq2_29<P> &X, const Fq2_29<P> &Y, const Fq2_29<P> &ZZ, const Fq2_29<P> &ZZZ)
    {
        x = X;
        zz = ZZ;
        store(y, Y);
        store(zzz, ZZZ);
    }
    __device__ void set(const Xyzz2_29<P> &q) { set(q.X, q.Y, q.ZZ, q.ZZZ); }
    __device__ Xyzz2_29<P> get() const { return {x, load(y), zz, load(zzz)}; }
};

// What a lane keeps of its run between the entries: in registers, or (Lds) in
// a column of LDS words, read where it is used.  The G1 addition needs all
// 168 registers that three waves per SIMD leave it, and a spilled one would
// cost more than its reload: scratch loads return in order behind the direct
// loads of the next base, so each addition would wait for that one's latency
// (4.6 against 4.1 us per addition at two waves per SIMD).
enum LaneWord { kBucket, kNextEnd, kSlot, kBuckets, kStarts, kStarts1, kSorted, kSorted1, kFirst, kLast, kBases, kBases1,
                kLaneWords };
template <bool Lds>
struct LaneWords {
    uint32_t w[kLaneWords];
    __device__ LaneWords(uint32_t *) {}
    __device__ uint32_t get(int i) const { return w[i]; }
    __device__ void set(int i, uint32_t v) { w[i] = v; }
};
template <>
struct LaneWords<true> {
    lds_word_t *w;  // word i of the lane at w[i * kAccThreads]
    __device__ LaneWords(uint32_t *lds) : w((lds_word_t *)(lds + threadIdx.x)) {}
    __device__ uint32_t get(int i) const { return w[i * kAccThreads]; }
    __device__ void set(int i, uint32_t v) { w[i * kAccThreads] = v; }
};
template <class T, bool Lds>
__device__ __forceinline__ const T *lane_ptr(const LaneWords<Lds> &lw, int i)
{
    return reinterpret_cast<const T *>((uint64_t)lw.get(i + 1) << 32 | lw.get(i));
}
template <class T, bool Lds>
__device__ __forceinline__ void set_lane_ptr(LaneWords<Lds> &lw, int i, const T *p)
{
    lw.set(i, (uint32_t)(uint64_t)p);
    lw.set(i + 1, (uint32_t)((uint64_t)p >> 32));
}

// A lane's walk over its run of a job's sorted entries.
template <bool Lds>
struct RunCursor {
    uint32_t e, e1;  // next entry, end of the run
    uint32_t end;    // end of entry e's bucket
    LaneWords<Lds> &lw;

    // lane: of the job; lane0: lanes and buckets of the jobs before it
    __device__ RunCursor(LaneWords<Lds> &words, const uint32_t *__restrict__ starts, uint32_t B, uint32_t lane0,
                         uint32_t lane, uint32_t piece)
        : lw(words)
    {
        e = lane * piece;
        e1 = min(e + piece, starts[B]);
        const uint32_t k = find_segment(starts, B, e);
        end = starts[k + 1];
        lw.set(kBucket, k);
        lw.set(kNextEnd, starts[min(k + 2, B)]);  // loaded ahead
        lw.set(kSlot, lane0 + lane + k);
        lw.set(kBuckets, B);
        set_lane_ptr(lw, kStarts, starts);
    }
    // where this lane's partial of the current bucket goes
    __device__ __forceinline__ uint32_t slot() const { return lw.get(kSlot); }
    // Past the last entry of the bucket: on to the bucket of entry e.
    __device__ __forceinline__ void advance()
    {
        const uint32_t *starts = lane_ptr<uint32_t>(lw, kStarts);
        const uint32_t B = lw.get(kBuckets), k0 = lw.get(kBucket);
        uint32_t k = k0, next = lw.get(kNextEnd);
        do {
            ++k;
            end = next;
            next = starts[min(k + 2, B)];
        } while (end == e);
        lw.set(kBucket, k);
        lw.set(kNextEnd, next);
        lw.set(kSlot, lw.get(kSlot) + k - k0);
    }
};

// The bases of a lane's run, one entry ahead of the additions.  They are
// gathered (64 or 128 bytes anywhere in a gigabyte), so a load is microseconds
// away, and neither holding the next base in registers (16 or 32 of them, a
// wave per SIMD less) nor waiting for it behind three waves pays.  Instead a
// lane's loads go straight to LDS while it adds: each 16-byte part of the
// wave's 64 bases is one direct load, lane i's at part[i].  The sorted indices
// come the same way, four at a time (one by one, a line of them would have
// left the caches before its next use), in two blocks used in turn.
//
// A direct load writes at one LDS address for the whole wave plus the lane's
// place, so the row must be the same for all lanes that load together.  The
// lanes of a wave take their entries in step; the blocks are therefore counted
// from each lane's first one, and those that go on to another block at the
// same step go on to one of the same number.
template <class F, bool Lds>
struct BaseStream {
    static constexpr uint32_t kParts = sizeof(Affine<F>) / sizeof(uint4);
    static constexpr uint32_t kRows = kParts + 2;  // rows of 64 x 16 bytes per wave
    uint4 (*rows)[64];                             // this wave's
    LaneWords<Lds> &lw;
    uint32_t v = 0;  // index of the base on its way

    __device__ static void load(const uint4 *from, uint4 *row)
    {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                         (__attribute__((address_space(3))) void *)row, 16, 0, 0);
    }
    // Direct loads so far have arrived / LDS reads so far are done.
    __device__ static void arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
    __device__ static void read_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

    // the run's block number t (counted in the list) of four indices
    __device__ __forceinline__ void load_block(uint32_t t)
    {
        load(lane_ptr<uint4>(lw, kSorted) + min(t, lw.get(kLast)),
             rows[kParts + __builtin_amdgcn_readfirstlane((t - lw.get(kFirst)) & 1u)]);
    }
    __device__ __forceinline__ uint32_t index(uint32_t e) const
    {
        const uint4 *block = &rows[kParts + (((e >> 2) - lw.get(kFirst)) & 1u)][threadIdx.x & 63u];
        return reinterpret_cast<const uint32_t *>(block)[e & 3u];
    }
    __device__ __forceinline__ void load_base()
    {
        const uint4 *b = reinterpret_cast<const uint4 *>(lane_ptr<Affine<F>>(lw, kBases) + (v & kEntryMask));
#pragma unroll
        for (uint32_t k = 0; k < kParts; ++k) load(b + k, rows[k]);
    }
    // Starts the run at entry e of a list of `entries`.
    __device__ BaseStream(uint4 (*wave_rows)[64], LaneWords<Lds> &words, const Affine<F> *bases,
                          const uint32_t *sorted, uint32_t e, uint32_t entries)
        : rows(wave_rows), lw(words)
    {
        set_lane_ptr(lw, kBases, bases);
        set_lane_ptr(lw, kSorted, sorted);
        lw.set(kFirst, e >> 2);
        lw.set(kLast, (entries - 1) >> 2);
        load_block(e >> 2);
        load_block((e >> 2) + 1);
        arrived();
        v = index(e);
        load_base();
    }
    // Entry e's base and sign.  The next entry's is on its way when this
    // returns (at the end of the run, e + 1 = e1, entry e's again).
    __device__ __forceinline__ Affine<F> take(uint32_t e, uint32_t e1, bool &negative)
    {
        Affine<F> P;
        arrived();
        uint4 *out = reinterpret_cast<uint4 *>(&P);
#pragma unroll
        for (uint32_t k = 0; k < kParts; ++k) out[k] = rows[k][threadIdx.x & 63u];
        negative = v >> 31;
        const bool more = e + 1 < e1;
        v = index(more ? e + 1 : e);
        read_done();
        load_base();
        if (more && ((e + 1) & 3u) == 0) load_block(((e + 1) >> 2) + 1);
        return P;
    }
};

// Accumulation over all jobs: a lane sums its run of L consecutive sorted
// entries (k_reduce_plan) of signed bases into one partial per bucket it
// meets.  Every lane has the same number of additions whatever the buckets'
// sizes, so waves end together and a launch of resident size is even; the
// store at a bucket's end costs a wave a few lanes' time once every bucket.
template <class F>
__device__ __forceinline__ void accumulate_body(const JobDev<F> *__restrict__ jobs,
                                                const uint32_t *__restrict__ lane_base, uint32_t J,
                                                const ReduceState *__restrict__ st, partial_t<F> *__restrict__ pool)
{
    constexpr bool kLds = !std::is_same<F, fq2_t>::value;
    using Stream = BaseStream<F, kLds>;
    __shared__ uint4 stage[kAccThreads / 64][Stream::kRows][64];
    __shared__ uint32_t words[kLds ? kLaneWords * kAccThreads : 1];
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= lane_base[J]) return;
    const uint32_t j = find_segment(lane_base, J, g);
    const JobDev<F> &jb = jobs[j];
    LaneWords<kLds> lw(words);
    RunCursor<kLds> c(lw, jb.bucket_start, jb.B, lane_base[j] + jb.b_off, g - lane_base[j],
                      msm_job_piece(st->piece, jb.piece_min));
    Stream in(stage[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)], lw, jb.bases, jb.sorted, c.e,
              jb.bucket_start[jb.B]);
    if constexpr (std::is_same<F, fq2_t>::value) {
        // G2: the accumulator in the reduced-radix form as for G1 (curve29.h,
        // Fq2 bounds), stored in it; Y and ZZZ in LDS between their uses.
        __shared__ uint32_t side[36 * kAccThreads];
        Xyzz2_29Lds<FqParams> acc{Fq2_29<FqParams>{}, Fq2_29<FqParams>{}, (lds_word_t *)(side + threadIdx.x),
                                  (lds_word_t *)(side + 18 * kAccThreads + threadIdx.x)};
        acc.set(Xyzz2_29<FqParams>::infinity());
#pragma unroll 1
        for (; c.e < c.e1; ++c.e) {
            if (c.e == c.end) {
                pool[c.slot()] = acc.get();
                acc.set(Xyzz2_29<FqParams>::infinity());
                c.advance();
            }
            bool negative;
            const Affine<F> P = in.take(c.e, c.e1, negative);
            if (!affine_is_inf(P)) {
                const F y = negative ? FieldOps<F>::neg(P.y) : P.y;
                xyzz2_29_madd<FqParams>(acc, fq2_29_from<FqParams>(P.x), fq2_29_from<FqParams>(y));
            }
        }
        pool[c.slot()] = acc.get();
    } else {
        // G1: the accumulator stays in the reduced-radix form (curve29.h: one
        // v_mad_u64_u32 per product term, no carries) for the whole run and is
        // stored in it; bases are converted as they arrive.
        Xyzz29<FqParams> acc = Xyzz29<FqParams>::infinity();
#pragma unroll 1
        for (; c.e < c.e1; ++c.e) {
            // The addition's 1,473 multiply-adds are 8 bytes long and issue more
            // slowly where they straddle an 8-byte boundary, and where the loop
            // begins decides how many do: 372 from 4 bytes past a boundary
            // here, 1,101 from the boundary (the launch of a 2^20 proof 1145
            // and 1175 us).
            asm volatile(".p2align 3\n\ts_nop 0");
            if (c.e == c.end) {
                pool[c.slot()] = acc;
                acc = Xyzz29<FqParams>::infinity();
                c.advance();
            }
            bool negative;
            const Affine<F> P = in.take(c.e, c.e1, negative);
            if (!affine_is_inf(P)) {
                const F y = negative ? FieldOps<F>::neg(P.y) : P.y;
                acc = xyzz29_add_affine(acc, fp29_from_mont(P.x), fp29_from_mont(y));
            }
        }
        pool[c.slot()] = acc;
    }
    // no direct load may be in flight when the workgroup gives its LDS back
    Stream::arrived();
}

// G1: at most 168 registers, three waves per SIMD.
template <class F>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_accumulate(const JobDev<F> *__restrict__ jobs,
                                                    const uint32_t *__restrict__ lane_base, uint32_t J,
                                                    const ReduceState *__restrict__ st,
                                                    partial_t<F> *__restrict__ pool)
{
    accumulate_body<F>(jobs, lane_base, J, st, pool);
}

// The G2 addition's working set exceeds 256 registers, which would leave one
// wave per SIMD; held to two waves, its spills cost less than the second wave
// gains (G2 accumulation of the dense 2^20 Poseidon-style proof 10.3 -> 8.5
// ms on MI355X), and with the accumulator's Y and ZZZ in LDS (36 KiB per
// workgroup) the spills fell from 280 to 80 bytes per lane (112 with the run's
// state).
template <>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_accumulate<fq2_t>(
    const JobDev<fq2_t> *__restrict__ jobs, const uint32_t *__restrict__ lane_base, uint32_t J,
    const ReduceState *__restrict__ st, partial_t<fq2_t> *__restrict__ pool)
{
    accumulate_body<fq2_t>(jobs, lane_base, J, st, pool);
}

// Sum over the lane groups of aligned runs of `groups` groups: every group of
// a run ends with its run's sum.
template <class F>
__device__ __forceinline__ Coop<F> coop_reduce(Coop<F> acc, uint32_t groups)
{
#pragma unroll 1
    for (uint32_t off = groups >> 1; off >= 1; off >>= 1) acc = coop_add(acc, coop_shfl_xor(acc, off));
    return acc;
}

// pool[src + i] for i = first, first + step, ... < cnt, summed by one lane
// group (infinity when there is none); the next partial is loaded before the
// addition that precedes it.
template <class F>
__device__ __forceinline__ Coop<F> coop_sum(const partial_t<F> *__restrict__ pool, uint32_t src, uint32_t cnt,
                                            uint32_t first, uint32_t step)
{
    Coop<F> acc = first < cnt ? coop_load<F>(pool, (size_t)src + first) : Coop<F>::infinity();
    uint32_t i = first + step;
    Coop<F> next = i < cnt ? coop_load<F>(pool, (size_t)src + i) : Coop<F>::infinity();
#pragma unroll 1
    while (i < cnt) {
        const Coop<F> cur = next;
        i += step;
        if (i < cnt) next = coop_load<F>(pool, (size_t)src + i);
        acc = coop_add(acc, cur);
    }
    return acc;
}

// Fold launch L: a wave sums up to kMsmFoldSpan partials of one record into one
// output; 7 (G1) or 10 (G2) additions deep.
template <class F>
__global__ __launch_bounds__(256) void k_fold(const ReduceState *__restrict__ st, const FoldRec *__restrict__ recs,
                                              uint32_t L, uint32_t out_base, partial_t<F> *__restrict__ pool)
{
    const unsigned long long n = st->fold_count[L];
    const uint32_t total = (uint32_t)n, nrec = (uint32_t)(n >> 32);
    const uint32_t group = (threadIdx.x & 63u) / Coop<F>::kLanes;
#pragma unroll 1
    for (uint32_t t = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64; t < total;
         t += gridDim.x * (blockDim.x / 64)) {
        uint32_t lo = 0, hi = nrec;  // the last record with start <= t
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (recs[mid].start <= t)
                lo = mid;
            else
                hi = mid;
        }
        const FoldRec r = recs[lo];
        const uint32_t off = (t - r.start) * kMsmFoldSpan;
        const uint32_t cnt = min(kMsmFoldSpan, r.cnt - off);
        const Coop<F> acc =
            coop_reduce(coop_sum<F>(pool, r.src + off, cnt, group, kWaveGroups<F>), kWaveGroups<F>);
        if (group == 0) coop_store<F>(pool, (size_t)out_base + t, acc);
    }
}

// Bucket completion: the 2^c lane groups of a class-c bucket stride over its
// partials, then a shuffle tree of c levels; grid-stride over all segments.
template <class F>
__global__ __launch_bounds__(256) void k_complete(const JobDev<F> *__restrict__ jobs,
                                                  const partial_t<F> *__restrict__ pool,
                                                  const uint32_t *__restrict__ seg_count,
                                                  const uint32_t *__restrict__ class_list,
                                                  const uint32_t *__restrict__ seg_base, uint32_t S)
{
    const uint32_t total = seg_base[S];
#pragma unroll 1
    for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < total; g += gridDim.x * blockDim.x) {
        const uint32_t s = find_segment(seg_base, S, g);
        const uint32_t j = s / kMsmCompleteClasses, c = s % kMsmCompleteClasses;
        const JobDev<F> &jb = jobs[j];
        const uint32_t local = (g - seg_base[s]) / Coop<F>::kLanes;
        const uint32_t idx = local >> c, group = local & ((1u << c) - 1u);
        const bool live = idx < seg_count[s];
        const uint32_t k =
            live ? class_list[(size_t)jb.b_off * kMsmCompleteClasses + (size_t)c * jb.B + idx] : 0u;
        Coop<F> acc = coop_sum<F>(pool, live ? jb.reg_start[k] : 0u, live ? jb.reg_count[k] : 0u, group, 1u << c);
        acc = coop_reduce(acc, 1u << c);
        if (live && group == 0) coop_store<F>(jb.sums, k, acc);
    }
}

// Bit-plane tree.  A level-t block covers buckets [b*2^t, (b+1)*2^t) and
// holds P_0..P_{t-1} (the sums of its buckets with that bit set) and T (its
// total); level 0 is S_m itself (S_0 = infinity).  Merging blocks 2b and
// 2b+1 into level t+1: P_e = P_e(2b) + P_e(2b+1) for e < t, P_t = T(2b+1),
// T = T(2b) + T(2b+1).  At the last level (t+1 = c-1) the merged P_e are the
// bit planes U_e, and U_{c-1} = S_B (bucket B = 2^(c-1) alone has bit c-1).
//
// One launch runs up to h levels from level t0: a workgroup loads 2^h
// level-t0 blocks of one job into LDS and merges them level by level, a lane
// group per addition, with a barrier in between (one addition of latency per
// level, no launch or global round trip), then stores the merged block to the
// other global tree buffer (`src` names the one it reads).  Jobs whose tree
// ends earlier run fewer levels; jobs already done return.  LDS accesses are
// one component (9 words, an odd stride) per lane: no bank conflicts.
template <class F>
__global__ __launch_bounds__(kTreeThreads) void k_tree_lds(const JobDev<F> *__restrict__ jobs, uint32_t t0,
                                                           uint32_t h, uint32_t src)
{
    extern __shared__ uint8_t tree_lds[];
    const JobDev<F> &jb = jobs[blockIdx.y];
    if (t0 + 1 > jb.c - 1) return;
    const uint32_t lv = min(h, jb.c - 1 - t0);
    if (blockIdx.x >= (jb.B >> (t0 + lv))) return;
    const uint32_t cap = (1u << h) * (t0 + 1);
    partial_t<F> *buf[2] = {reinterpret_cast<partial_t<F> *>(tree_lds),
                            reinterpret_cast<partial_t<F> *>(tree_lds) + cap};
    const uint32_t group = threadIdx.x / Coop<F>::kLanes, groups = blockDim.x / Coop<F>::kLanes;

    const uint32_t nin = (1u << lv) * (t0 + 1);
    const uint32_t first = (blockIdx.x << lv) * (t0 + 1);
    for (uint32_t idx = group; idx < nin; idx += groups) {
        Coop<F> v = Coop<F>::infinity();
        if (t0 != 0)
            v = coop_load<F>(jb.tree[src], first + idx);
        else if (first + idx != 0)
            v = coop_load<F>(jb.sums, first + idx - 1);
        coop_store<F>(buf[0], idx, v);
    }
    __syncthreads();
    for (uint32_t s = 0; s < lv; ++s) {
        const uint32_t t = t0 + s, E = t + 2;
        const bool last = (t + 1 == jb.c - 1);
        const partial_t<F> *in = buf[s & 1];
        partial_t<F> *out = buf[(s + 1) & 1];
        const uint32_t adds = (1u << (lv - s - 1)) * (t + 1);
        for (uint32_t idx = group; idx < adds; idx += groups) {
            const uint32_t b = idx / (t + 1), e = idx % (t + 1);
            const Coop<F> l = coop_load<F>(in, (size_t)(2 * b) * (t + 1) + e);
            const Coop<F> r = coop_load<F>(in, (size_t)(2 * b + 1) * (t + 1) + e);
            const bool top = e == t;  // T: the sum goes behind P_t, which is r itself
            const Coop<F> o = last && top ? coop_load<F>(jb.sums, jb.B - 1) : coop_add(l, r);
            if (last) {
                coop_store_plane<F>(jb.planes + (top ? t + 1 : e), o);
                if (top) coop_store_plane<F>(jb.planes + t, r);
            } else {
                coop_store<F>(out, (size_t)b * E + (top ? t + 1 : e), o);
                if (top) coop_store<F>(out, (size_t)b * E + t, r);
            }
        }
        __syncthreads();
    }
    const uint32_t t1 = t0 + lv;
    if (t1 < jb.c - 1)
        for (uint32_t e = group; e <= t1; e += groups)
            coop_store<F>(jb.tree[src ^ 1u], (size_t)blockIdx.x * (t1 + 1) + e, coop_load<F>(buf[lv & 1], e));
}

// finite[i] = 1 if a[i] or b[i] is not infinity.
__global__ __launch_bounds__(256) void k_finite(const g1_jac *__restrict__ a, const g2_jac *__restrict__ b, uint32_t n,
                                                uint8_t *__restrict__ finite)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) finite[i] = !a[i].Z.is_zero() || !b[i].Z.is_zero() ? 1 : 0;
}

// Base preparation: normalise the reference-layout Jacobian point and store
// 2^(c*w) * P for every window w (affine, infinity flagged).  Each window's
// points share one inversion per workgroup (an inversion of its own cost every
// point more than twice its c doublings).
constexpr uint32_t kPrepareThreads = 128;
template <class F>
__global__ __launch_bounds__(kPrepareThreads) void k_prepare_bases(const Jacobian<F> *__restrict__ in,
                                                                  const uint32_t *__restrict__ perm, uint32_t n,
                                                                  uint32_t c, uint32_t W, Affine<F> *__restrict__ out)
{
    __shared__ fq_t node[2 * kPrepareThreads];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Xyzz<F> P = i < n ? jacobian_to_xyzz(in[perm ? perm[i] : i]) : Xyzz<F>::infinity();
    for (uint32_t w = 0; w < W; ++w) {
        if (w)
            for (uint32_t t = 0; t < c; ++t) P = xyzz_dbl(P);
        const Affine<F> a = block_to_affine<kPrepareThreads>(P, node);
        if (i < n) out[(size_t)w * n + i] = a;
    }
}

// Workgroups of 256 threads of `kernel` the device keeps resident at once
// (all CUs at the kernel's occupancy), times two so that grid-stride loops
// end evenly.  Computed once per kernel.
template <auto Kernel>
uint64_t resident_blocks()
{
    static const uint64_t blocks = [] {
        int dev = 0, cus = 0, per_cu = 0;
        NKR_HIP(hipGetDevice(&dev));
        NKR_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        NKR_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, Kernel, 256, 0));
        return (uint64_t)std::max(1, cus) * std::max(1, per_cu) * 2;
    }();
    return blocks;
}

uint32_t g_target_log = kMsmTargetDefault;
uint32_t g_lanes_cap = 16;

}  // namespace

void msm_set_shape(uint32_t target_pieces_log, uint32_t complete_lanes_cap)
{
    NKR_REQUIRE(target_pieces_log >= 10 && target_pieces_log <= 22, "MSM target pieces must be 2^10 .. 2^22");
    NKR_REQUIRE(complete_lanes_cap >= 1 && complete_lanes_cap <= 16 &&
                    (complete_lanes_cap & (complete_lanes_cap - 1)) == 0,
                "MSM completion lanes must be a power of two in 1 .. 16");
    g_target_log = target_pieces_log;
    g_lanes_cap = complete_lanes_cap;
}


MsmLanes msm_lanes(bool g2, uint32_t target_log)
{
    return msm_lanes_of(g2, target_log ? target_log : g_target_log);
}
uint32_t msm_complete_lanes_cap() { return g_lanes_cap; }
uint64_t msm_shape_key() { return (uint64_t)g_target_log << 32 | g_lanes_cap; }

template <class F>
uint64_t msm_batch_bytes(const MsmTotals &jobs)
{
    if (jobs.jobs == 0) return 0;
    const MsmSizes s = jobs.sizes(msm_lanes(std::is_same<F, fq2_t>::value));
    // partial sums and their folds; per bucket: sums and two tree levels, region
    // start and count, the completion class lists; fold records; and the fixed
    // records (job table, class counters, lane offsets, plan state)
    return s.pool * sizeof(partial_t<F>) + s.buckets * (3 * sizeof(partial_t<F>) + 8 + 4 * kMsmCompleteClasses) +
           s.records * kMsmMaxFoldLaunches * sizeof(FoldRec) + 1024 * jobs.jobs;
}

void msm_finite_terms(const g1_jac *a, const g2_jac *b, uint32_t n, std::vector<uint32_t> &terms, hipStream_t stream)
{
    DeviceBuffer<uint8_t> dev(n);
    std::vector<uint8_t> host(n);
    k_finite<<<div_up(n, 256), 256, 0, stream>>>(a, b, n, dev.get());
    NKR_LAUNCH_CHECK();
    NKR_HIP(hipMemcpyAsync(host.data(), dev.get(), n, hipMemcpyDeviceToHost, stream));
    NKR_HIP(hipStreamSynchronize(stream));
    terms.clear();
    for (uint32_t i = 0; i < n; ++i)
        if (host[i]) terms.push_back(i);
}

template <class F>
void MsmBases<F>::prepare(const Jacobian<F> *jacobian, const uint32_t *perm, const MsmPlan &plan,
                          hipStream_t stream)
{
    plan_ = plan;
    pts_.allocate((size_t)plan.W * plan.n);
    k_prepare_bases<F><<<div_up(plan.n, kPrepareThreads), kPrepareThreads, 0, stream>>>(jacobian, perm, plan.n, plan.c,
                                                                                     plan.W, pts_.get());
    NKR_LAUNCH_CHECK();
}

// The sort kernels hold B counts in dynamic LDS: up to 128 KiB for c = 16,
// above the 64 KiB a launch gets without asking.
static void allow_sort_lds()
{
    static std::once_flag once;
    std::call_once(once, [] {
        const int bytes = (int)(kMsmMaxBuckets * sizeof(uint32_t));
        NKR_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_hist),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        NKR_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_scatter),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        NKR_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_hist_batch),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        NKR_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_scatter_batch),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    });
}

uint32_t MsmSchedule::prepare(const MsmPlan &plan)
{
    allow_sort_lds();
    NKR_REQUIRE(plan.B <= kMsmMaxBuckets, "MSM window too wide for the bucket scans");
    plan_ = plan;
    blocks_ = msm_sort_blocks(plan.n);
    const MsmScheduleSizes sizes = msm_schedule_sizes(plan);
    sorted_.ensure(sizes.sorted);
    bucket_start_.ensure(sizes.bucket_start);
    in_tile_.ensure(sizes.in_tile);
    tile_total_.ensure(sizes.tile_total);
    block_count_.ensure(sizes.block_count);
    return div_up(plan.n, blocks_);
}

void MsmSchedule::build(const fr_t *scalars_mont, const uint32_t *pick, const MsmPlan &plan, hipStream_t stream,
                        StageTimer *timer)
{
    const uint32_t per_block = prepare(plan);
    const uint32_t n = plan.n, B = plan.B;
    const size_t lds = (size_t)B * sizeof(uint32_t);
    const uint32_t threads = std::min<uint32_t>(kSortThreads, (per_block + 63) & ~63u);
    if (timer) timer->begin(kStageSort, stream);
    k_hist<<<blocks_, threads, lds, stream>>>(scalars_mont, pick, n, plan.c, plan.W, B, per_block, block_count_.get());
    NKR_LAUNCH_CHECK();
    k_colscan<<<div_up(B, 64), 64 * kScanGroups, 0, stream>>>(block_count_.get(), blocks_, B, in_tile_.get(),
                                                              tile_total_.get());
    NKR_LAUNCH_CHECK();
    k_scatter<<<blocks_, threads, lds, stream>>>(scalars_mont, pick, n, plan.c, plan.W, B, per_block, in_tile_.get(),
                                                 tile_total_.get(), block_count_.get(), bucket_start_.get(),
                                                 sorted_.get());
    NKR_LAUNCH_CHECK();
    if (timer) timer->end(kStageSort, stream);
}

void MsmScheduleBatch::build(const std::vector<Item> &items, hipStream_t stream, bool graph)
{
    const uint32_t J = (uint32_t)items.size();
    if (J == 0) return;
    NKR_REQUIRE(J <= 65535, "a schedule batch holds at most 65535 schedules");
    const size_t jobs_bytes = (sizeof(SortJob) * J + 15) & ~size_t(15);
    const size_t total = jobs_bytes + sizeof(uint32_t) * (J + 1);
    uint8_t *st = graph ? stage_.reuse_unsynced(total) : stage_.reuse(total);
    table_.ensure(total);
    SortJob *jobs = reinterpret_cast<SortJob *>(st);
    uint32_t *off = reinterpret_cast<uint32_t *>(st + jobs_bytes);
    uint32_t Bmax = 0, threads = 64;
    uint64_t blocks = 0;
    for (uint32_t j = 0; j < J; ++j) {
        MsmSchedule &s = *items[j].sched;
        const MsmPlan &p = items[j].plan;
        const uint32_t per_block = s.prepare(p);
        jobs[j] = SortJob{items[j].scalars_mont, items[j].pick, p.n, p.c, p.W, p.B, s.blocks_, per_block, s.block_count_.get(),
                          s.in_tile_.get(), s.tile_total_.get(), s.bucket_start_.get(), s.sorted_.get()};
        off[j] = (uint32_t)blocks;
        blocks += s.blocks_;
        Bmax = std::max(Bmax, p.B);
        threads = std::max(threads, std::min<uint32_t>(kSortThreads, (per_block + 63) & ~63u));
    }
    NKR_REQUIRE(blocks < (1ull << 31), "schedule batch too large");
    off[J] = (uint32_t)blocks;
    NKR_HIP(hipMemcpyAsync(table_.get(), st, total, hipMemcpyHostToDevice, stream));
    if (!graph) stage_.uploaded(stream);
    const SortJob *dj = reinterpret_cast<const SortJob *>(table_.get());
    const uint32_t *doff = reinterpret_cast<const uint32_t *>(table_.get() + jobs_bytes);
    const size_t lds = (size_t)Bmax * sizeof(uint32_t);
    k_hist_batch<<<(uint32_t)blocks, threads, lds, stream>>>(dj, doff, J);
    NKR_LAUNCH_CHECK();
    k_colscan_batch<<<dim3(div_up(Bmax, 64), J), 64 * kScanGroups, 0, stream>>>(dj);
    NKR_LAUNCH_CHECK();
    k_scatter_batch<<<(uint32_t)blocks, threads, lds, stream>>>(dj, doff, J);
    NKR_LAUNCH_CHECK();
}

template <class F>
static std::vector<const void *> layout_key(const std::vector<MsmJob<F>> &jobs)
{
    std::vector<const void *> key;
    for (const auto &jb : jobs) {
        key.push_back(jb.bases->data());
        key.push_back(jb.sched->sorted_.get());
        key.push_back(jb.sched->bucket_start_.get());
        key.push_back(jb.planes);
        key.push_back(reinterpret_cast<const void *>((uintptr_t)jb.sched->plan().max_entries()));
        key.push_back(reinterpret_cast<const void *>((uintptr_t)jb.sched->plan().B));
        key.push_back(reinterpret_cast<const void *>((uintptr_t)jb.piece_min));
    }
    return key;
}

template <class F>
bool MsmBatch<F>::layout_matches(const std::vector<MsmJob<F>> &jobs) const
{
    return layout_key(jobs) == key_ && wanted_lanes() == lanes_;
}

template <class F>
void MsmBatch<F>::layout(const std::vector<MsmJob<F>> &jobs, hipStream_t stream)
{
    if (layout_matches(jobs)) return;
    std::vector<const void *> key = layout_key(jobs);
    key_.clear();  // until the new layout is whole
    lanes_ = wanted_lanes();
    const uint32_t J = (uint32_t)jobs.size();
    // where each job's buckets lie in the per-bucket arrays
    std::vector<uint64_t> b_off(J + 1, 0);
    MsmTotals totals;
    for (uint32_t j = 0; j < J; ++j) {
        const MsmPlan &p = jobs[j].sched->plan();
        NKR_REQUIRE(jobs[j].bases->plan().n == p.n && jobs[j].bases->plan().c == p.c,
                    "MSM bases and schedule disagree");
        totals.add(p);
        b_off[j + 1] = b_off[j] + p.B;
    }
    sizes_ = totals.sizes(lanes_);
    NKR_REQUIRE(sizes_.pool < (1ull << 32), "MSM partial pool exceeds 32-bit indexing");
    NKR_REQUIRE(sizes_.complete_lanes < (1ull << 32), "MSM batch too large for 32-bit work indices");
    uint32_t fold_base[kMsmMaxFoldLaunches];
    for (uint32_t L = 0; L < kMsmMaxFoldLaunches; ++L) fold_base[L] = (uint32_t)sizes_.fold_base[L];
    // grow-only: a batch whose composition changes from call to call reuses them
    pool_.ensure(sizes_.pool);
    sums_.ensure(b_off[J]);
    tree_[0].ensure(b_off[J]);
    tree_[1].ensure(b_off[J]);
    reg_start_.ensure(b_off[J]);
    reg_count_.ensure(b_off[J]);

    static_assert(std::is_trivially_copyable<JobDev<F>>::value, "job records are raw-copied");
    const size_t jobs_bytes = (sizeof(JobDev<F>) * J + 15) & ~size_t(15);
    const size_t table_bytes = jobs_bytes + sizeof(fold_base);
    uint8_t *st = jobs_stage_.reuse(table_bytes);
    JobDev<F> *host = reinterpret_cast<JobDev<F> *>(st);
    for (uint32_t j = 0; j < J; ++j) {
        const MsmJob<F> &jb = jobs[j];
        JobDev<F> &d = host[j];
        d.bases = jb.bases->data();
        d.sorted = jb.sched->sorted_.get();
        d.bucket_start = jb.sched->bucket_start_.get();
        d.reg_start = reg_start_.get() + b_off[j];
        d.reg_count = reg_count_.get() + b_off[j];
        d.sums = sums_.get() + b_off[j];
        d.tree[0] = tree_[0].get() + b_off[j];
        d.tree[1] = tree_[1].get() + b_off[j];
        d.planes = jb.planes;
        d.B = jb.sched->plan().B;
        d.c = jb.sched->plan().c;
        d.b_off = (uint32_t)b_off[j];
        d.piece_min = std::max(1u, jb.piece_min);
    }
    std::memcpy(st + jobs_bytes, fold_base, sizeof(fold_base));
    seg_base_.ensure(kMsmCompleteClasses * J + 1);
    seg_count_.ensure(kMsmCompleteClasses * J);
    class_count_.ensure(kMsmCompleteClasses * J);
    class_list_.ensure(kMsmCompleteClasses * b_off[J]);
    recs_.ensure(sizes_.records * kMsmMaxFoldLaunches * sizeof(FoldRec));
    state_.ensure(sizeof(ReduceState));
    jobs_dev_.ensure(table_bytes);
    lane_base_.ensure(J + 1);  // filled on the device per run
    // k_reduce_plan leaves its counters cleared; new buffers start so (never
    // inside a captured graph, which reuses the layout of an eager run)
    NKR_HIP(hipMemsetAsync(class_count_.get(), 0, class_count_.bytes(), stream));
    NKR_HIP(hipMemsetAsync(state_.get(), 0, sizeof(ReduceState), stream));
    NKR_HIP(hipMemcpyAsync(jobs_dev_.get(), st, table_bytes, hipMemcpyHostToDevice, stream));
    jobs_stage_.uploaded(stream);
    key_ = key;
}

template <class F>
void MsmBatch<F>::run(const std::vector<MsmJob<F>> &jobs, hipStream_t stream, StageTimer *timer, bool graph)
{
    if (jobs.empty()) return;
    NKR_REQUIRE(!graph || layout_matches(jobs), "a captured MSM batch must reuse the layout of its eager run");
    layout(jobs, stream);
    const uint32_t J = (uint32_t)jobs.size();
    uint32_t Bmax = 0, cmax = 0;
    for (const auto &jb : jobs) {
        Bmax = std::max(Bmax, jb.sched->plan().B);
        cmax = std::max(cmax, jb.sched->plan().c);
    }
    const uint8_t *table = jobs_dev_.get();
    const JobDev<F> *jd = reinterpret_cast<const JobDev<F> *>(table);
    const uint32_t *fold_base_dev =
        reinterpret_cast<const uint32_t *>(table + ((sizeof(JobDev<F>) * J + 15) & ~size_t(15)));
    ReduceState *state = reinterpret_cast<ReduceState *>(state_.get());
    FoldRec *recs = reinterpret_cast<FoldRec *>(recs_.get());

    // A launch that fails half way leaves the plan's counters unknown: the
    // next run lays the batch out again.
    struct Relayout {
        std::vector<const void *> *key;
        ~Relayout()
        {
            if (key) key->clear();
        }
    } relayout{&key_};

    uint32_t max_class = 0;
    while ((2u << max_class) <= std::min(msm_complete_lanes_cap(), kWaveGroups<F>)) ++max_class;
    const uint32_t S = kMsmCompleteClasses * J;
    const uint32_t plan_threads = std::min<uint32_t>(kPlanThreads, std::max<uint32_t>(256, (Bmax + 63) & ~63u));
    k_reduce_plan<F><<<dim3(div_up(Bmax, plan_threads), J), plan_threads, 0, stream>>>(
        jd, J, lanes_, (uint32_t)sizes_.buckets, max_class, state, recs, (uint32_t)sizes_.records, fold_base_dev, class_count_.get(),
        class_list_.get(), lane_base_.get(), seg_count_.get(), seg_base_.get());
    NKR_LAUNCH_CHECK();
    // the accumulation stage brackets exactly the k_accumulate launch
    const int acc_stage = std::is_same<F, fq2_t>::value ? kStageAccumulateG2 : kStageAccumulate;
    if (timer) timer->begin(acc_stage, stream);
    k_accumulate<F><<<(uint32_t)div_up(sizes_.lanes, kAccThreads), kAccThreads, 0, stream>>>(
        jd, lane_base_.get(), J, state, pool_.get());
    NKR_LAUNCH_CHECK();
    if (timer) {
        timer->end(acc_stage, stream);
        timer->begin(kStageFold, stream);
    }
    // as many fold launches as one bucket with every lane's partial would
    // need (2 from 8193 lanes to 2^19): an empty one costs less than the host's
    // wait for the largest count
    for (uint32_t L = 0; L < sizes_.fold_launches; ++L) {
        const uint64_t blocks = std::min<uint64_t>(div_up(sizes_.fold_cap[L], 4), 1024);
        k_fold<F><<<(uint32_t)blocks, 256, 0, stream>>>(state, recs + (size_t)L * sizes_.records, L, (uint32_t)sizes_.fold_base[L],
                                                      pool_.get());
        NKR_LAUNCH_CHECK();
    }
    {
        const uint64_t blocks = std::min<uint64_t>(div_up(sizes_.complete_lanes, 256), resident_blocks<k_complete<F>>());
        k_complete<F><<<(uint32_t)std::max<uint64_t>(blocks, 1), 256, 0, stream>>>(
            jd, pool_.get(), seg_count_.get(), class_list_.get(), seg_base_.get(), S);
    }
    NKR_LAUNCH_CHECK();
    // bit-plane tree: as many levels per launch as two LDS buffers of 2^h
    // level-t blocks allow; a workgroup has a lane group per addition of its
    // widest level (whole waves, at most kTreeThreads)
    for (uint32_t t = 0, src = 0; t + 1 <= cmax - 1; src ^= 1u) {
        uint32_t h = 1;
        while (t + h < cmax - 1 && 2 * (size_t(2) << h) * (t + 1) * sizeof(partial_t<F>) <= kTreeLds) ++h;
        const size_t lds = 2 * (size_t(1) << h) * (t + 1) * sizeof(partial_t<F>);
        uint32_t widest = 0;
        for (uint32_t s = 0; s < h; ++s) widest = std::max(widest, (1u << (h - 1 - s)) * (t + s + 1));
        const uint32_t lanes =
            std::min<uint32_t>(kTreeThreads, (uint32_t)div_up(widest * Coop<F>::kLanes, 64) * 64);
        k_tree_lds<F><<<dim3(Bmax >> (t + h), J), lanes, lds, stream>>>(jd, t, h, src);
        NKR_LAUNCH_CHECK();
        t += h;
    }
    if (timer) timer->end(kStageFold, stream);
    relayout.key = nullptr;
}

template <class F>
Xyzz<F> msm_sum(const Xyzz<F> *planes, uint32_t c)
{
    Xyzz<F> acc = planes[c - 1];
    for (int j = (int)c - 2; j >= 0; --j) {
        acc = xyzz_dbl(acc);
        acc = xyzz_add(acc, planes[j]);
    }
    return acc;
}

template <class F>
Jacobian<F> msm_finish(const Xyzz<F> *planes, uint32_t c)
{
    return xyzz_to_jacobian_affine(msm_sum(planes, c));
}

template <class F>
MsmContext<F>::MsmContext(const Jacobian<F> *bases_dev, uint32_t n, uint32_t c_override, hipStream_t stream)
{
    const MsmPlan plan = MsmPlan::choose(n, c_override);
    bases_.prepare(bases_dev, nullptr, plan, stream);
    planes_.allocate(plan.c);
}

template <class F>
Jacobian<F> MsmContext<F>::run(const fr_t *scalars_dev, hipStream_t stream)
{
    const MsmPlan &plan = bases_.plan();
    sched_.build(scalars_dev, nullptr, plan, stream);
    batch_.run({MsmJob<F>{&bases_, &sched_, planes_.get()}}, stream);
    std::vector<Xyzz<F>> host(plan.c);
    NKR_HIP(hipMemcpyAsync(host.data(), planes_.get(), plan.c * sizeof(Xyzz<F>), hipMemcpyDeviceToHost, stream));
    NKR_HIP(hipStreamSynchronize(stream));
    return msm_finish(host.data(), plan.c);
}

template class MsmBases<fq_t>;
template class MsmBases<fq2_t>;
template class MsmBatch<fq_t>;
template class MsmBatch<fq2_t>;
template class MsmContext<fq_t>;
template class MsmContext<fq2_t>;
template Jacobian<fq_t> msm_finish(const Xyzz<fq_t> *, uint32_t);
template Jacobian<fq2_t> msm_finish(const Xyzz<fq2_t> *, uint32_t);
template Xyzz<fq_t> msm_sum(const Xyzz<fq_t> *, uint32_t);
template Xyzz<fq2_t> msm_sum(const Xyzz<fq2_t> *, uint32_t);
template uint64_t msm_batch_bytes<fq_t>(const MsmTotals &);
template uint64_t msm_batch_bytes<fq2_t>(const MsmTotals &);

}  // namespace nkr
