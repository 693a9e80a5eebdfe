// Which calls of a batch are captured into a HIP graph and which replay it.
// Host logic only (no HIP), so that a CPU test can walk its states.
//
// A call is named by a key (what its launches refer to and depend on).  A call
// that repeats the one before it is captured, and from then on the graph is
// replayed while the key stays the same; any other call runs eagerly and drops
// the graph, since it may move what the graph's launches refer to.  A call
// counts as the one before only once it has succeeded: one that failed half
// way may have left the work buffers without the layout that a capture relies
// on, so the call after it is eager whatever its key.
#pragma once

#include <cstdint>
#include <utility>
#include <vector>

namespace nkr {

class LaunchReuse {
public:
    enum class Mode { kEager, kCapture, kReplay };

    // The mode of a call with this key.
    Mode begin(std::vector<uint64_t> key, bool capture_allowed)
    {
        const bool repeats = done_ && key == call_;
        done_ = false;
        call_ = std::move(key);
        if (captured_ && call_ == graph_) return Mode::kReplay;
        captured_ = false;
        return repeats && capture_allowed ? Mode::kCapture : Mode::kEager;
    }
    // The call's launches are in a graph.
    void captured()
    {
        graph_ = call_;
        captured_ = true;
    }
    // The call has succeeded.
    void finish() { done_ = true; }
    // The graph is gone.
    void dropped() { captured_ = false; }
    // The buffers are gone too: the next call is eager.
    void forget()
    {
        captured_ = false;
        done_ = false;
    }

private:
    std::vector<uint64_t> call_;   // the latest call's key
    std::vector<uint64_t> graph_;  // the graph's
    bool done_ = false;            // the latest call succeeded
    bool captured_ = false;        // there is a graph
};

}  // namespace nkr
