// row_rule.h -- when the plain step takes 16 lanes per agent (row_kernels.h);
// host code only.
#pragma once

#include <algorithm>

namespace ecm {

// Crowds up to which the step, and its attraction pass, take 16 lanes.
constexpr int kRowAgents = 160000, kRowAttrAgents = 16000;

struct RowRule {
    bool step = false, attr = false;
    int agents = 0;                 // agents the row step's grid is sized for

    // shape: a plain step in the default launch shape; other shapes say how
    // agents are laid out.
    void update(bool shape, int n) {
        // a crowd near a limit keeps the form it has: changing it captures the
        // step graphs anew
        auto small = [&](bool now, int limit) { return n <= (now ? limit + limit / 4 : limit); };
        step = shape && small(step, kRowAgents);
        attr = shape && small(attr, kRowAttrAgents);
        // The kernel strides over its grid, so any count is covered: the grid
        // is made larger when the crowd outgrows it and smaller when it falls
        // well below.  One that followed the count in steps of 4,096 captured
        // the graphs anew at every crossing (a crowd around 4,096, read after
        // every step: 94 us a step instead of 66).
        if (!step) agents = 0;
        else if (n > agents || n < agents - std::max(8192, agents / 4)) agents = (n + 4095) / 4096 * 4096;
    }
};

}  // namespace ecm
