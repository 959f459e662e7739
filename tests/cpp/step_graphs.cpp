// CPU-only harness for lmdeploy_amd/csrc/step_graphs.h: which steps run as graphs, counted with a stand-in for a graph.  Built and run by
// tests/test_step_graphs.py.
#include "../../lmdeploy_amd/csrc/step_graphs.h"

#include <cstdio>
#include <cstdlib>
#include <set>

using namespace tmk;

#define CHECK(c)                                                                     \
    do {                                                                             \
        if (!(c)) {                                                                  \
            std::fprintf(stderr, "%s:%d: CHECK(%s) failed\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                                            \
        }                                                                            \
    } while (0)

struct Counts {
    int           launches = 0, captures = 0, replays = 0, made = 0;
    bool          fails = false;
    std::set<int> live;
};

static int step(StepGraphs<int>& g, Counts& c, int rows, int want = 1, bool on = true)
{
    return g.run(
        rows, want, on, [&] { return ++c.launches, 0; },
        [&](int* graph) {
            ++c.captures;
            if (c.fails) {
                *graph = 99;  // (whatever a failed call leaves)
                return 3;
            }
            c.live.insert(*graph = ++c.made);
            return 0;
        },
        [&](int graph) {
            CHECK(c.live.count(graph));
            return ++c.replays, 0;
        },
        [&](int graph) { CHECK(c.live.erase(graph) == 1); });
}

int main()
{
    {  // the first by launches, the others as a graph; logits wanted or not are steps of their own
        StepGraphs<int> g;
        Counts          c;
        g.set_slots(2);
        for (int i = 0; i < 5; ++i) {
            CHECK(step(g, c, 3) == 0 && step(g, c, 3, 0) == 0);
        }
        CHECK(c.launches == 2 && c.captures == 2 && c.replays == 8 && c.live.size() == 2);
        CHECK(step(g, c, 3, 1, false) == 0 && c.launches == 3);  // not in use: by launches
        g.clear([&](int graph) { CHECK(c.live.erase(graph) == 1); });
        CHECK(c.live.empty() && g.size() == 0);
    }
    {  // a step that cannot be captured runs, and is not tried again
        StepGraphs<int> g;
        Counts          c;
        g.set_slots(2);
        c.fails = true;
        for (int i = 0; i < 5; ++i) {
            CHECK(step(g, c, 7) == 0);
        }
        CHECK(c.launches == 5 && c.captures == 1 && c.replays == 0);
        g.clear([&](int) { CHECK(false); });
    }
    {  // more numbers of rows than places: one gives way, the others stay; a course through all rows of the slots keeps every graph
        StepGraphs<int> g;
        Counts          c;
        g.set_slots(20);
        for (int pass = 0; pass < 3; ++pass) {
            for (int rows = 20; rows > 0; --rows) {
                CHECK(step(g, c, rows) == 0 && step(g, c, rows, 0) == 0);
            }
        }
        CHECK(c.launches == 40 && c.captures == 40 && c.replays == 80 && g.size() == 40 && c.live.size() == 40);
        CHECK(step(g, c, 20) == 0);  // the oldest, used again: its neighbour, 20 rows without logits, is the oldest now
        CHECK(step(g, c, 21) == 0 && c.launches == 41 && g.size() == 40 && c.live.size() == 39);
        CHECK(step(g, c, 20) == 0 && step(g, c, 19) == 0 && c.captures == 40 && c.replays == 83);
        CHECK(step(g, c, 20, 0) == 0 && c.launches == 42 && c.live.size() == 38);  // in the place of 19 rows without logits
        g.clear([&](int graph) { CHECK(c.live.erase(graph) == 1); });
        CHECK(c.live.empty());
        g.set_slots(1000);
        for (int rows = 1; rows <= 1000; ++rows) {
            step(g, c, rows), step(g, c, rows);
        }
        CHECK(g.size() == 256 && c.live.size() == 256);
    }
    std::puts("ok");
    return 0;
}
