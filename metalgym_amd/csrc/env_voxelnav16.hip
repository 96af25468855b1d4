// Built-in env: VoxelNav16, the gather-heavy 16^3 voxel navigation env.
#include "mg/device/env_kernels.h"
#include "mg/device/rollout_voxelnav16.h"

MG_DEFINE_ENV(VoxelNav16)
