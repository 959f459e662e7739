// Which recorded steps run as graphs (host only, no device code, so that it can be driven from a CPU test).
//
// A step of one token a session is some 120 launches, which leave the host more slowly than small models run them: from its second time on a step of as many rows is one
// graph launch.  The first, launch by launch, has loaded every kernel.
#pragma once
#include <cstddef>
#include <vector>

namespace tmk {

template<class Graph>
class StepGraphs {
    struct Step {
        int   rows, want, seen;
        Graph graph;
    };
    std::vector<Step> steps_;
    size_t            most_;

public:
    explicit StepGraphs(size_t most): most_(most) {}
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
            if (i >= most_) {
                clear(destroy);
                i = 0;
            }
            steps_.push_back(Step{rows, want, 0, Graph{}});
        }
        Step& s = steps_[i];
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
