// Which recorded steps run as graphs (host only, no device code, so that it can be driven from a CPU test).
//
// A step of one token a session is some 120 launches, which leave the host more slowly than small models run them: from its second time on a step of as many rows is one
// graph launch.  The first, launch by launch, has loaded every kernel.  Where all places are taken the step that has not come for the longest time gives up its own: emptied as a
// whole, the places of a course that goes round among more numbers of rows than there are places never came to be used.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace tmk {

template<class Graph>
class StepGraphs {
    struct Step {
        int    rows, want, seen;
        size_t used;
        Graph  graph;
    };
    std::vector<Step> steps_;
    size_t            most_ = 32, now_ = 0;

public:
    // places for `slots` sessions: every number of rows with and without logits, up to 256 (a graph of 120 launches takes some 15 KB of host memory and 0.2 ms to make)
    void set_slots(int slots)
    {
        most_ = std::min<size_t>(2 * (size_t)std::max(slots, 1), 256);
    }
    size_t size() const
    {
        return steps_.size();
    }
    // Runs a step of `rows` rows, `want`: with their logits.  on: graphs are in use; launch() -> rc runs it launch by launch, capture(Graph*) -> rc makes its graph,
    // replay(Graph) -> rc runs that, destroy(Graph) frees it (every step has ended by then).  A step that cannot be captured is one of launches for good
    template<class Launch, class Capture, class Replay, class Destroy>
    int run(int rows, int want, bool on, Launch launch, Capture capture, Replay replay, Destroy destroy)
    {
        if (!on) {
            return launch();
        }
        size_t i = 0;
        while (i < steps_.size() && (steps_[i].rows != rows || steps_[i].want != want)) {
            ++i;
        }
        if (i == steps_.size()) {
            if (i < most_) {
                steps_.push_back(Step{});
            }
            else {
                i = std::min_element(steps_.begin(), steps_.end(), [](const Step& a, const Step& b) { return a.used < b.used; }) - steps_.begin();
                if (steps_[i].graph) {
                    destroy(steps_[i].graph);
                }
            }
            steps_[i] = Step{rows, want, 0, 0, Graph{}};
        }
        Step& s = steps_[i];
        s.used  = ++now_;
        if (s.seen < 2 && ++s.seen == 2 && capture(&s.graph) != 0) {
            s.graph = Graph{};
        }
        return s.graph ? replay(s.graph) : launch();
    }
    template<class Destroy>
    void clear(Destroy destroy)
    {
        for (Step& s : steps_) {
            if (s.graph) {
                destroy(s.graph);
            }
        }
        steps_.clear();
    }
};

}  // namespace tmk
