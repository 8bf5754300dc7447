// row_rule.h -- when the plain step takes 16 lanes per agent (row_kernels.h);
// host code only.
#pragma once

#include <algorithm>

namespace ecm {

// The largest crowd whose step takes 16 lanes per agent, where one lane per
// agent becomes the faster form.  The row form's time grows with the agents,
// the one-lane form's with k: its list and unrolled constraints fill a
// wavefront's lanes whatever the crowd, and past k 10 its ORCA pass leaves the
// registers.  us for 20 steps, one lane / row, of a jam (4 agents a square
// metre) and of a crowd at 0.15 a square metre:
//   k 1,  100,000: 1400 / 1448, 1347 / 1386     120,000: 1433 / 1638, 1386 / 1591
//   k 5,  100,000: 2108 / 2468, 1682 / 1590     120,000: 2179 / 2835, 1722 / 1813
//   k 6,  120,000: 2738 / 2960, 2137 / 1853     160,000: 2905 / 3646, 2224 / 2281
//   k 10, 120,000: 3442 / 3269, 2439 / 2038     160,000: 3754 / 4000, 2648 / 2491
//   k 11, 160,000: 5061 / 4094, 3263 / 2570     190,000: 5284 / 4649, 3332 / 2843
// The line is the crossing of the crowd that is not jammed.
constexpr int row_agents_max(int k) { return k <= 5 ? 112000 : k <= 10 ? 160000 : 200000; }
// The same for the attraction pass alone, which knows no k.
constexpr int kRowAttrAgents = 16000;

struct RowRule {
    bool step = false, attr = false;
    int agents = 0;                 // agents the row step's grid is sized for
    bool step_fits = true, attr_fits = true;

    // shape: a plain step in the default launch shape; other shapes say how
    // agents are laid out.
    void update(bool shape, int k, int n) {
        // A crowd that outgrew a limit comes back once it is an eighth below:
        // changing the form captures the step graphs anew.  Not the other way
        // about: above the limit the row form is the slower one (a crowd grown
        // to 195,000, k 5: 4115 us for 20 steps, 2410 with one lane).
        auto small = [&](bool now, int limit) { return n <= (now ? limit : limit - limit / 8); };
        step_fits = small(step_fits, row_agents_max(k));
        attr_fits = small(attr_fits, kRowAttrAgents);
        step = shape && step_fits;
        attr = shape && attr_fits;
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
