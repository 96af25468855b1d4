// Test-only envs of many observation and head widths, odd ones among them: the
// operands that the policy kernels pair up, pad or stage by width. A position
// that drifts with the action; float k of the observation is a line in it.
#pragma once
#include "mg/env.h"

template <uint32_t O, uint32_t A>
struct RampBase {
    struct State {
        float x;
        uint32_t steps;
    };
    using Action = int;
    struct Obs {
        float v[O];
    };
    static constexpr uint32_t OBS_DIM = O;
    static constexpr uint32_t ACT_DIM = A;

    MG_HD static void reset(State& s, uint32_t& rng) {
        s.x = rngUniform(rng, -1.0f, 1.0f);
        s.steps = rngInt(rng, 8);
    }
    MG_HD static void step(State& s, Action a, Obs& obs, float& reward, uint8_t& done) {
        s.x = 0.875f * s.x + 0.0625f * (float)(a + 1);
        s.steps += 1;
        reward = -s.x;
        done = s.steps >= 10 ? 1 : 0;
        for (uint32_t k = 0; k < O; ++k) obs.v[k] = (k & 1 ? -1.0f : 1.0f) * s.x + 0.0625f * (float)k;
    }
};
struct Ramp1 : RampBase<1, 2> { static constexpr const char* KERNEL = "rollout_test_ramp1"; };
struct Ramp3 : RampBase<3, 4> { static constexpr const char* KERNEL = "rollout_test_ramp3"; };
struct Ramp15 : RampBase<15, 15> { static constexpr const char* KERNEL = "rollout_test_ramp15"; };
struct Ramp33 : RampBase<33, 7> { static constexpr const char* KERNEL = "rollout_test_ramp33"; };
struct Ramp63 : RampBase<63, 15> { static constexpr const char* KERNEL = "rollout_test_ramp63"; };
