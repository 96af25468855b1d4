// One row's head in the fp32 tiles' arithmetic (tile_row_head, policy_lane.h;
// split_row_head, policy_pair.h) for every row of an array, for the test that
// holds them against the tiles bit for bit.
#include <hip/hip_runtime.h>

#include "mg/device/collect.h"

using namespace mg::dev;

template <int CPT, int O, int HD>
__global__ void __launch_bounds__(64) tile_rows(const mg_policy_view pv, const float* obs, float* head) {
    __shared__ __align__(16) float lds[kLaneRowLds];
    __shared__ float h[HD];
    tile_row_head<CPT, O, HD>(pv, obs + (size_t)blockIdx.x * O, lds, h);
    if (threadIdx.x < HD) head[(size_t)blockIdx.x * HD + threadIdx.x] = h[threadIdx.x];
}

template <int O, int HD>
__global__ void __launch_bounds__(64 * kPairW) split_rows(const mg_policy_view pv, const float* obs, float* head) {
    extern __shared__ __align__(16) float lds[];  // scratch, then the row and its head
    float* row = lds + pv.hidden + 10 * kEmbed + 32;
    float* h = row + O;
    if (threadIdx.x < O) row[threadIdx.x] = obs[(size_t)blockIdx.x * O + threadIdx.x];
    split_row_head<O, HD>(pv, small_params(pv), row, blockIdx.x / kSplitRows, lds, h);
    if (threadIdx.x < HD) head[(size_t)blockIdx.x * HD + threadIdx.x] = h[threadIdx.x];
}

// tile: 16, 32 or 64 rows. Device pointers; blocking. A hipError_t, or -1 for a
// policy it does not have.
extern "C" int mg_test_row_heads(const mg_policy_view* pv, const float* obs, uint32_t rows, uint32_t tile, float* head) {
    const dim3 grid(rows);
    const size_t lds = (pv->hidden + 10 * kEmbed + 32 + 64) * 4;
    if (pv->obs_dim == 4 && pv->head_dim == 3 && tile == 16)
        hipLaunchKernelGGL((split_rows<4, 3>), grid, dim3(64 * kPairW), lds, 0, *pv, obs, head);
    else if (pv->obs_dim == 4 && pv->head_dim == 3 && tile == 32)
        hipLaunchKernelGGL((tile_rows<16, 4, 3>), grid, dim3(64), 0, 0, *pv, obs, head);
    else if (pv->obs_dim == 4 && pv->head_dim == 3 && tile == 64)
        hipLaunchKernelGGL((tile_rows<32, 4, 3>), grid, dim3(64), 0, 0, *pv, obs, head);
    else if (pv->obs_dim == 30 && pv->head_dim == 7 && tile == 32)
        hipLaunchKernelGGL((tile_rows<16, 30, 7>), grid, dim3(64), 0, 0, *pv, obs, head);
    else if (pv->obs_dim == 30 && pv->head_dim == 7 && tile == 64)
        hipLaunchKernelGGL((tile_rows<32, 30, 7>), grid, dim3(64), 0, 0, *pv, obs, head);
    else
        return -1;
    if (hipError_t e = hipGetLastError()) return (int)e;
    return (int)hipDeviceSynchronize();
}
