#pragma once
// How the SGD steps that one block takes are dealt to launches.  In a header of its own, so that it can be checked without
// a GPU up to the largest number of steps a call may ask for (2^31 - 1: sums of steps do not fit an int).
#include <cstdint>

namespace xad_linreg {

// Launch k of 0 .. step_launches() - 1 takes the steps first .. first + steps - 1 and gathers the samples of the `gather`
// steps from `coming` on, those of launch k + 1; launch -1 does nothing but gather.
struct StepLaunch {
    std::int64_t first, coming;
    int steps, gather;
};

inline std::int64_t step_launches(int epochs, int per_launch) {
    return (static_cast<std::int64_t>(epochs) + per_launch - 1) / per_launch;
}

inline StepLaunch step_launch(std::int64_t k, int epochs, int per_launch) {
    auto up_to_a_launch = [&](std::int64_t left) { return static_cast<int>(left < 0 ? 0 : (left < per_launch ? left : per_launch)); };
    StepLaunch l{};
    l.first = k * per_launch;
    l.coming = l.first + per_launch;
    l.steps = k < 0 ? 0 : up_to_a_launch(epochs - l.first);
    l.gather = up_to_a_launch(epochs - l.coming);
    return l;
}

}  // namespace xad_linreg
