// CPU check of the MSM sizing arithmetic (nkr-zkp_amd/csrc/msm_plan.h).
// stdin: one request per line,
//   plan n c_override target_log piece_lo piece_hi
//       -> "c W B max_pieces capacity levels" or "error <message>"
//   folds partials        -> fold levels for one bucket with that many partials
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
                uint64_t n, c, tl, lo, hi;
                in >> n >> c >> tl >> lo >> hi;
                MsmPlan p = MsmPlan::choose((uint32_t)n, (uint32_t)c);
                p.piece_lo = (uint32_t)lo;
                p.piece_hi = (uint32_t)hi;
                const uint64_t pieces = p.max_pieces((uint32_t)tl);
                uint32_t levels = 0;
                const uint64_t cap = msm_partial_capacity(p, pieces, &levels, nullptr);
                std::printf("%u %u %u %llu %llu %u\n", p.c, p.W, p.B, (unsigned long long)pieces,
                            (unsigned long long)cap, levels);
            } else if (op == "folds") {
                uint64_t k;
                in >> k;
                std::printf("%u\n", msm_fold_levels(k));
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
                const MsmSizes s = msm_sizes(jobs, entries, buckets, msm_launch_lanes(r, entries));
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
