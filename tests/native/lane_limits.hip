// Prints the deepest policy that each fp32 lane collect has LDS for
// (collect_lane_bytes, include/mg/device/collect.h): "env shares blocks".
// Host code only: nothing is launched.
#include <stdio.h>

#include "mg/device/env_kernels.h"
#include "mg/envs/cartpole.h"
#include "mg/envs/cartpole_continuous.h"
#include "mg/envs/voxelnav.h"
#include "mg/envs/voxelnav16.h"

extern "C" int mg_env_register(const mg_env_desc*) { return 0; }

template <typename Env, int HS>
void deepest(const char* name) {
    uint32_t l = 0;
    while (l < MG_MAX_LAYERS && mg::dev::collect_lane_bytes<Env, MG_PRECISION_FP32, HS>(l + 1)) ++l;
    printf("%s %d %u\n", name, HS, l);
}
template <typename Env>
void both(const char* name) {
    deepest<Env, 1>(name);
    deepest<Env, 2>(name);
}
int main() {
    both<CartPole>("cartpole");
    both<CartPoleContinuous>("cartpole_continuous");
    both<VoxelNav16>("voxelnav16");
    both<VoxelNav>("voxelnav");
    return 0;
}
