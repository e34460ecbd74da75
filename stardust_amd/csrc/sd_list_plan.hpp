// Host side of the lists that steps run on (near lists of sphere contexts,
// partner lists of clump contexts): how many steps of which kind to queue in one
// launch sequence, from what the last one left. Plain C++.
#pragma once

#include <algorithm>
#include <cmath>

namespace sd {

// Margin of a clump context's lists: 40 steps of the last movement, within these
// shares of the mean body size. (constexpr: the build computes them on the device.)
constexpr float CL_MARGIN_STEPS = 40.0f, CL_MARGIN_MIN = 0.005f, CL_MARGIN_MAX = 0.05f;
constexpr float clump_widest(float size) { return CL_MARGIN_MAX * size; }
constexpr float clump_margin(float last, float size) {
    const float m = CL_MARGIN_STEPS * last, lo = CL_MARGIN_MIN * size, hi = clump_widest(size);
    return m > hi ? hi : (m > lo ? m : lo);
}
// What rounding of coordinates up to `far` can take from a margin, and the share
// of the margin that the limit on the movement keeps.
constexpr float clump_rounding(float far, float margin) { return 5e-7f * (far + margin); }
constexpr float CL_MARGIN_KEPT = 0.98f;
// The largest movement that lists allow.
constexpr float clump_largest(float size) { return CL_MARGIN_KEPT * clump_widest(size); }
constexpr float clump_limit(float margin, float far) { return CL_MARGIN_KEPT * margin - clump_rounding(far, margin); }
// The margin of a build: wider by what rounding takes, as far as the widest
// goes. Far enough from the origin (about 100,000 body sizes) that leaves
// nothing, and the plan rests the lists. Planned without it, every step built a
// tree and queued 64 that were dropped: 2,000 slow bodies of 8 cm 2 km from the
// origin 258 us a step, now 10; at 30 km 258, now 119 (no lists there).
constexpr float clump_build_margin(float last, float size, float far) {
    const float m = clump_margin(last, size) + 1.05f * clump_rounding(far, clump_widest(size));
    return m < clump_widest(size) ? m : clump_widest(size);
}

// Steps queued between two looks at how long the lists last, or whether they
// would do.
constexpr int LIST_REST = 64;

// What a launch sequence left, as its context reads it back.
struct ListReport {
    int ran = 0;             // steps that ran
    bool given_up = false;   // a step was given up
    bool crowded = false;    // some list did not hold all it had to
    float last = 0.0f;       // largest movement of a step
    float budget = 0.0f;     // movement that the lists allow, from their build
    float used = 0.0f;       // of it, up to the last step that ran
    float lost = 0.0f;       // what rounding took from the budget
};

// Steps to queue, in this order: on no lists (then nothing else), or one that
// builds them and some that use them.
struct ListRun {
    int none = 0, build = 0, use = 0;
};

struct ListPlan {
    int steps = 0;         // steps that the lists are expected to last (0: build them next)
    int rest = 0;          // steps to run without lists before they are tried again
    float last = -1.0f;    // largest movement of a step as last read back (negative: not known)
    float lost = -1.0f;    // what rounding takes from a build's budget (negative: not known)
    bool crowded = false;  // the last lists were too short

    // Steps that lists last with `left` of their budget, a tenth short of what
    // the last movement says (a shortfall costs a given-up launch sequence, a
    // surplus a build a few steps early).
    static int life(float left, float last) {
        const float s = 0.9f * left / std::fmax(last, 1e-30f);
        return s >= (float)LIST_REST ? LIST_REST : (s > 0.0f ? (int)s : 0);  // (not a number: 0)
    }

    // Whether lists pay: not where the largest budget, less what rounding takes
    // from it, would last fewer than 4 steps.
    bool pays(float largest) const { return 4.0f * last <= largest - std::fmax(lost, 0.0f); }

    // left: steps still to run; on: lists are possible and pay; rebuild: the
    // lists cannot be used whatever they hold; largest, fresh: the largest budget,
    // and that of a build at the last movement.
    ListRun next(int left, bool on, bool rebuild, float largest, float fresh) {
        ListRun r;
        if (!on || rest > 0) {
            r.none = std::min(left, LIST_REST);
            steps = 0;
            return r;
        }
        if (rebuild || steps < std::min(left, 2)) {
            // of unknown speed or rounding, or too short the last time: a look first
            const bool look = crowded || last < 0.0f || lost < 0.0f;
            steps = look ? 2 : life(std::fmin(fresh, largest - lost), last);
            r.build = 1;
        }
        r.use = std::min(left - r.build, steps);
        return r;
    }

    // used: the sequence was one of lists. Lists that were too short, or that
    // would pay but for what rounding takes from their budget, are tried again
    // after a long rest.
    void read(const ListReport& p, bool used, float largest) {
        last = std::isfinite(p.last) ? p.last : 3.4e38f;
        steps = 0;
        if (!used) {
            rest = std::max(0, rest - p.ran);
            return;
        }
        // (the movement of the step to come is not in yet: counted as the last one)
        if (!p.given_up) steps = life(p.budget - p.used - p.last, p.last);
        crowded = p.crowded;
        lost = p.lost;
        if (crowded || (4.0f * last <= largest && !pays(largest))) {
            steps = 0;
            rest = 4 * LIST_REST;
            lost = -1.0f;
        }
    }
};

}  // namespace sd
