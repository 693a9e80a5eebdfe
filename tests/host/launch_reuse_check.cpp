// CPU walk through the states of LaunchReuse (nkr-zkp_amd/csrc/launch_reuse.h).
// stdin: one step per line,
//   call <allowed 0|1> <outcome ok|fail> key...  -> eager, capture or replay.  A
//          call that succeeds finishes, and a capture is in a graph then; one that
//          fails throws before either.
//   drop | forget                                -> the word itself
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "launch_reuse.h"

using namespace nkr;

int main()
{
    LaunchReuse reuse;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string op, outcome;
        in >> op;
        if (op == "drop") {
            reuse.dropped();
            std::puts("drop");
        } else if (op == "forget") {
            reuse.forget();
            std::puts("forget");
        } else {
            int allowed = 0;
            in >> allowed >> outcome;
            std::vector<uint64_t> key;
            for (uint64_t k; in >> k;) key.push_back(k);
            const LaunchReuse::Mode m = reuse.begin(key, allowed != 0);
            if (outcome == "ok") {
                if (m == LaunchReuse::Mode::kCapture) reuse.captured();
                reuse.finish();
            }
            std::puts(m == LaunchReuse::Mode::kEager ? "eager" : m == LaunchReuse::Mode::kCapture ? "capture" : "replay");
        }
    }
    return 0;
}
