// oxr_steps.h -- a lane's bounce steps on their way to the launch counter (64 bits).
#pragma once
#include <stdint.h>

namespace oxd {

// In the persistent form a lane sums over every photon it takes, and max_bounce has no limit
// of its own: the lane keeps 32 bits (a register across the whole loop) and hands them over
// once they reach 2^31. A photon's own steps are below 2^31, so the sum never wraps.
// (constexpr: for the host and the device)
template <class Hand>
__attribute__((always_inline)) constexpr void add_steps(uint32_t& steps, int bounces, Hand hand) {
    steps += uint32_t(bounces);
    if (steps >> 31) {
        hand(steps);
        steps = 0;
    }
}

} // namespace oxd
