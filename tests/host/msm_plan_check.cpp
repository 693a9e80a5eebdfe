// CPU check of the MSM sizing arithmetic (nkr-zkp_amd/csrc/msm_plan.h).
// stdin: one request per line,
//   plan n c_override     -> "c W B" or "error <message>"
//   schedule n c_override -> the words of a schedule's buffers and their bytes
//   lanes g2 target_log   -> the lane rule: 4 lane counts, 3 limits
//   piece g2 target_log piece_min entries... -> per entry count, the launch's
//                            entries per lane and those of a job with that minimum
//   bplan cols c_override finite -> "n c" of bs1 and bs2
//   sizes g2 target_log jobs entries buckets -> the bounds msm_sizes gives a launch
//                            under that lane rule: lanes pool records complete_lanes
//                            launches, then each fold launch's base and cap
//   launches partials     -> fold launches for buckets of at most that many
//   divup a b             -> ceil(a / b) or "error <message>"
// Errors are reported, never turned into a crash: a zero divisor must raise
// nkr::Error instead of ending the process with SIGFPE.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <iostream>
#include <sstream>
#include <string>

#include "msm_plan.h"

using namespace nkr;

int main()
{
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string op;
        in >> op;
        try {
            if (op == "plan") {
                uint64_t n, c;
                in >> n >> c;
                const MsmPlan p = MsmPlan::choose((uint32_t)n, (uint32_t)c);
                std::printf("%u %u %u\n", p.c, p.W, p.B);
            } else if (op == "schedule") {
                uint64_t n, c;
                in >> n >> c;
                const MsmScheduleSizes s = msm_schedule_sizes(MsmPlan::choose((uint32_t)n, (uint32_t)c));
                std::printf("%llu %llu %llu %llu %llu %llu\n", (unsigned long long)s.sorted,
                            (unsigned long long)s.bucket_start, (unsigned long long)s.in_tile,
                            (unsigned long long)s.tile_total, (unsigned long long)s.block_count,
                            (unsigned long long)s.bytes());
            } else if (op == "lanes") {
                uint64_t g2, tl;
                in >> g2 >> tl;
                const MsmLanes r = msm_lanes_of(g2 != 0, (uint32_t)tl);
                for (uint32_t l : r.lanes) std::printf("%u ", l);
                for (uint64_t b : r.below) std::printf("%llu ", (unsigned long long)b);
                std::printf("\n");
            } else if (op == "piece") {
                uint64_t g2, tl, pm, e;
                in >> g2 >> tl >> pm;
                const MsmLanes r = msm_lanes_of(g2 != 0, (uint32_t)tl);
                while (in >> e) std::printf("%u %u ", msm_piece(r, e), msm_job_piece(msm_piece(r, e), (uint32_t)pm));
                std::printf("\n");
            } else if (op == "bplan") {
                uint64_t cols, c, finite;
                in >> cols >> c >> finite;
                const MsmPlan p = msm_b_plan(msm_witness_plan((uint32_t)cols, (uint32_t)c), (uint32_t)finite);
                std::printf("%u %u\n", p.n, p.c);
            } else if (op == "sizes") {
                uint64_t g2, tl, jobs, entries, buckets;
                in >> g2 >> tl >> jobs >> entries >> buckets;
                const MsmLanes r = msm_lanes_of(g2 != 0, (uint32_t)tl);
                MsmTotals totals;
                totals.add(MsmTotals{jobs, entries, buckets});
                const MsmSizes s = totals.sizes(r);
                std::printf("%llu %llu %llu %llu %u", (unsigned long long)s.lanes, (unsigned long long)s.pool,
                            (unsigned long long)s.records, (unsigned long long)s.complete_lanes, s.fold_launches);
                for (uint32_t L = 0; L < kMsmMaxFoldLaunches; ++L)
                    std::printf(" %llu %llu", (unsigned long long)s.fold_base[L], (unsigned long long)s.fold_cap[L]);
                std::printf("\n");
            } else if (op == "launches") {
                uint64_t k;
                in >> k;
                std::printf("%u\n", msm_fold_launches(k));
            } else if (op == "divup") {
                uint64_t a, b;
                in >> a >> b;
                std::printf("%u\n", div_up(a, b));
            } else {
                std::printf("error unknown request\n");
            }
        } catch (const Error &e) {
            std::printf("error %s\n", e.what());
        }
        std::fflush(stdout);
    }
    return 0;
}
