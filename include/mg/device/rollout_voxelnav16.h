// VoxelNav16's rollout with the grid at one bit per cell: a wave owns E envs,
// one per lane, their grids in LDS as 256 rows of 16 bits (516 bytes an env in
// the place of 4 KB).
//
// rollout_split_kernel, still the faster for what takes() leaves to it, stages
// the grids as bytes, of which LDS holds 36 to 38 per CU, and spreads a step's 27
// gathers over threads behind two barriers. As
// bits, 256 envs fit a CU: a step is a lane's own (nine 16-bit row reads give
// its 27 cells) and needs no barrier, and the observations leave through a
// wave's LDS tile as 16-byte stores. A reset's 256 draws are spread over the
// wave: xorshift32 is linear over GF(2), so lane j starts at draw 4 j by a
// product with a power of the step's matrix (kJump) and draws its four rows;
// on one lane the fill took 5.6 K instructions.
//
// Same draws, order and floats as rollout_kernel. Bound by the grids (4 KB read
// once per env and launch: one step at 65536 envs takes 47 us, 5.7 TB/s) and then
// by the 129 bytes a step of slots, written at 2.9 TB/s (the launch's 540 MB are
// past the Infinity Cache).
#pragma once
#include "../envs/voxelnav16.h"
#include "rollout.h"

namespace mg {
namespace dev {

// kJump.col[b][j]: the xorshift32 state 4 j draws after 1 << b.
struct XorshiftJump {
    uint32_t col[32][64];
};
constexpr XorshiftJump make_xorshift_jump() {
    XorshiftJump t{};
    for (int b = 0; b < 32; ++b) {
        uint32_t s = 1u << b;
        for (int j = 0; j < 64; ++j) {
            t.col[b][j] = s;
            for (int k = 0; k < 4; ++k) {
                s ^= s << 13;
                s ^= s >> 17;
                s ^= s << 5;
            }
        }
    }
    return t;
}
static __device__ const XorshiftJump kJump = make_xorshift_jump();

constexpr uint32_t kVnRows = 256;          // 16-bit rows of a grid: row 16 z + y, x from bit 0
constexpr uint32_t kVnLd = kVnRows + 2;    // halfwords per env, an odd number of dwords against bank conflicts
constexpr int kVnObs = VoxelNav16::OBS_DIM;

// One env's bits.
struct VnBits {
    uint16_t* r;
    __device__ __forceinline__ uint32_t row(uint32_t i) const { return r[i]; }
    __device__ __forceinline__ bool cell(uint32_t c) const { return (r[c >> 4] >> (c & 15u)) & 1u; }
    __device__ __forceinline__ void clear(uint32_t c) { r[c >> 4] &= (uint16_t)~(1u << (c & 15u)); }
};

// VoxelNav16::draw_free_cell on bits.
__device__ __forceinline__ int vn_free_cell(VnBits g, uint32_t& rng, int avoid) {
    int c = 0;
    for (int t = 0; t < VoxelNav16::MAX_TRIES; ++t) {
        c = (int)(rngNext(rng) & (uint32_t)(VoxelNav16::CELLS - 1));
        if (!g.cell((uint32_t)c) && c != avoid) return c;
    }
    if (c == avoid) c = (c + 1) & (VoxelNav16::CELLS - 1);
    g.clear((uint32_t)c);
    return c;
}

// 16 occupancy bytes as 16 bits, set where the byte is not 0.
__device__ __forceinline__ uint32_t vn_pack(const uint32_t (&x)[4]) {
    uint32_t t[4];  // 128 in each byte that is not 0
#pragma unroll
    for (int q = 0; q < 4; ++q) t[q] = (((x[q] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x[q]) & 0x80808080u;
    const uint32_t lo = __builtin_amdgcn_udot4(t[1], 0x80402010u, __builtin_amdgcn_udot4(t[0], 0x08040201u, 0u, false), false);
    const uint32_t hi = __builtin_amdgcn_udot4(t[3], 0x80402010u, __builtin_amdgcn_udot4(t[2], 0x08040201u, 0u, false), false);
    return (hi << 1) | (lo >> 7);
}

__device__ __forceinline__ void vn_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// E envs per wave, on its first E lanes; every lane takes part in the loads,
// the resets and the observation stores.
template <int MODE, int E>
__global__ void __launch_bounds__(64) rollout_voxelnav16_kernel(const mg_rollout_args a) {
    using State = VoxelNav16::State;
    static_assert(E % 4 == 0 && E <= 64, "four envs per load batch, one lane each");
    __shared__ uint16_t rowsL[E * kVnLd];
    __shared__ __align__(16) float obsL[E * kVnObs];
    const uint32_t lane = threadIdx.x, n = a.n, e0 = blockIdx.x * E;
    const uint32_t ne = n - e0 < (uint32_t)E ? n - e0 : (uint32_t)E;
    State* states = static_cast<State*>(a.state) + e0;
    const bool live = lane < ne;
    const uint32_t me = live ? lane : 0;  // lanes past the end load the first env again and store nothing
    int32_t* head = reinterpret_cast<int32_t*>(states + me);
    int px = head[0], py = head[1], pz = head[2], gx = head[3], gy = head[4], gz = head[5];
    uint32_t steps = (uint32_t)head[6];
    uint32_t rng = a.rng[e0 + me];
    uint32_t done = live ? a.done[e0 + me] : 0u;
    const VnBits mine{rowsL + me * kVnLd};
    uint32_t jump[32];  // this lane's column of each power of the step's matrix
#pragma unroll
    for (int b = 0; b < 32; ++b) jump[b] = kJump.col[b][lane];

    // grids to bits: a lane takes rows lane + 64 u of four envs at a time, the
    // next four envs' 16 loads in flight
    uint32_t v[2][4][4][4];
    auto load = [&](uint32_t (&x)[4][4][4], uint32_t e) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t* g = reinterpret_cast<const uint32_t*>(states[e + k < ne ? e + k : ne - 1].grid);
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) x[k][u][q] = g[4 * (lane + 64 * u) + q];
        }
    };
    auto put = [&](const uint32_t (&x)[4][4][4], uint32_t e) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
                rowsL[(e + k < ne ? e + k : ne - 1) * kVnLd + lane + 64 * u] = (uint16_t)vn_pack(x[k][u]);
    };
    load(v[0], 0);
    for (uint32_t e = 0; e < ne; e += 8) {
        load(v[1], e + 4);
        put(v[0], e);
        if (e + 4 >= ne) break;
        load(v[0], e + 8);
        put(v[1], e + 4);
    }
    vn_fence();

    uint64_t reset_in = 0;  // envs reset during the launch
    for (uint32_t t = 0; t < a.steps; ++t) {
        const size_t k = (size_t)t * n + e0 + lane;
        int act;
        if constexpr (MODE == MG_ACTIONS_RANDOM) {
            act = random_action<VoxelNav16>(rng);
            if (a.actions_out && live) static_cast<int*>(a.actions_out)[k] = act;
        } else {
            act = live ? static_cast<const int*>(a.actions_in)[k] : 0;
        }
        uint64_t again = __ballot(done != 0);
        reset_in |= again;
        for (; again; again &= again - 1) {
            const int e = __builtin_ctzll(again);
            const uint32_t s0 = (uint32_t)__builtin_amdgcn_readlane((int)rng, e);
            uint32_t s = 0;
#pragma unroll
            for (int b = 0; b < 32; ++b) s ^= (0u - ((s0 >> b) & 1u)) & jump[b];
            uint16_t* fresh = rowsL + e * kVnLd + 4 * lane;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t r = rngNext(s);
                // bit 2 c of x is set iff the 2-bit field c of r is 3; the even bits packed
                uint32_t x = r & (r >> 1) & 0x55555555u;
                x = (x | x >> 1) & 0x33333333u;
                x = (x | x >> 2) & 0x0F0F0F0Fu;
                x = (x | x >> 4) & 0x00FF00FFu;
                fresh[d] = (uint16_t)(x | x >> 8);
            }
            const uint32_t after = (uint32_t)__builtin_amdgcn_readlane((int)s, 63);  // after all 256 draws
            vn_fence();
            if ((int)lane == e) {
                rng = after;
                const int c = vn_free_cell(mine, rng, -1);
                const int g = vn_free_cell(mine, rng, c);
                px = c % 16, py = (c / 16) % 16, pz = c / 256;
                gx = g % 16, gy = (g / 16) % 16, gz = g / 256;
                steps = 0;
            }
            vn_fence();
        }
        // VoxelNav16::stepState
        const int m = act < 0 ? 0 : (act > 5 ? 5 : act), sign = (m & 1) ? -1 : 1, axis = m >> 1;
        const int nx = px + (axis == 0 ? sign : 0), ny = py + (axis == 1 ? sign : 0), nz = pz + (axis == 2 ? sign : 0);
        const bool in = ((nx | ny | nz) & ~15) == 0;
        const uint32_t there = mine.row(in ? (uint32_t)(16 * nz + ny) : 0u);
        const bool blocked = !in || ((there >> (nx & 15)) & 1u);
        px = blocked ? px : nx, py = blocked ? py : ny, pz = blocked ? pz : nz;
        steps += 1;
        const bool atGoal = px == gx && py == gy && pz == gz;
        const float reward = atGoal ? 1.0f : (blocked ? -0.1f : -0.01f);
        done = (live && (atGoal || steps >= VoxelNav16::MAX_STEPS)) ? 1u : 0u;
        if (live) {
            if (a.reward_out) a.reward_out[k] = reward;
            if (a.done_out) a.done_out[k] = (uint8_t)done;
        }
        if (a.obs_out) {
            if (lane < (uint32_t)E) {
                uint32_t r[9];
#pragma unroll
                for (int p = 0; p < 9; ++p) {  // rows of the 3 x 3 neighbourhood in z, y
                    const int y = py + p % 3 - 1, z = pz + p / 3 - 1;
                    r[p] = mine.row(((y | z) & ~15) == 0 ? (uint32_t)(16 * z + y) : 0u);
                }
                float o[kVnObs];
                // an agent that the caller put outside the grid may be anywhere
                const int sh = (px < -2 ? -2 : px > 17 ? 17 : px) + 2;
#pragma unroll
                for (int p = 0; p < 9; ++p) {
                    const int y = py + p % 3 - 1, z = pz + p / 3 - 1;
                    const uint32_t row = ((y | z) & ~15) == 0 ? r[p] : 0xFFFFu;
                    const uint32_t c = ((row << 3) | 0xFFF80007u) >> sh;  // cells px - 1 .. px + 1, out-of-grid ones set
#pragma unroll
                    for (int d = 0; d < 3; ++d) o[3 * p + d] = (float)((c >> d) & 1u);
                }
                o[27] = VoxelNav16::div15(gx - px);
                o[28] = VoxelNav16::div15(gy - py);
                o[29] = VoxelNav16::div15(gz - pz);
                float2* ol = reinterpret_cast<float2*>(obsL + lane * kVnObs);
#pragma unroll
                for (int p = 0; p < kVnObs / 2; ++p) ol[p] = make_float2(o[2 * p], o[2 * p + 1]);
            }
            vn_fence();
            float* out = a.obs_out + ((size_t)t * n + e0) * kVnObs;
            const uint32_t words = ne * kVnObs;
            if ((reinterpret_cast<uintptr_t>(out) & 15u) == 0 && words % 4 == 0) {
#pragma unroll
                for (uint32_t u = 0; u < (E * kVnObs / 4 + 63) / 64; ++u) {
                    const uint32_t q = lane + 64 * u;
                    if (4 * q < words) reinterpret_cast<float4*>(out)[q] = reinterpret_cast<const float4*>(obsL)[q];
                }
            } else {
#pragma unroll
                for (uint32_t u = 0; u < (E * kVnObs + 63) / 64; ++u) {
                    const uint32_t q = lane + 64 * u;
                    if (q < words) out[q] = obsL[q];
                }
            }
            vn_fence();  // the tile is read before the next step writes it
        }
    }
    if (live) {
        head[0] = px, head[1] = py, head[2] = pz, head[3] = gx, head[4] = gy, head[5] = gz;
        head[6] = (int32_t)steps;
        a.rng[e0 + lane] = rng;
        a.done[e0 + lane] = (uint8_t)done;
    }
    for (; reset_in; reset_in &= reset_in - 1) {  // a grid that changed, back to bytes
        const int e = __builtin_ctzll(reset_in);
        uint32_t* g = reinterpret_cast<uint32_t*>(states[e].grid);
        const VnBits b{rowsL + e * kVnLd};
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t r = b.row(lane + 64 * u);
            uint32_t* p = g + 4 * (lane + 64 * u);
#pragma unroll
            for (int q = 0; q < 4; ++q) p[q] = (((r >> (4 * q)) & 15u) * 0x00204081u) & 0x01010101u;
        }
    }
}

template <>
struct PackedRollout<VoxelNav16> {
    static constexpr bool OK = true;
    // Not the observations of a few envs, which the split kernel computes on more
    // lanes: us a launch of 32 random steps, it against this, 24 / 29 for one env,
    // 27 / 29.5 for 4, 32 / 30 for 8. Nor few steps of very many envs, which are the
    // stream of their grids alone: one step 121 / 120 at 131072 envs, 147 / 152 at
    // 163840, 229 / 241 at 262144; two 190 / 190 at 196544, 248 / 254 at 262144;
    // four 208 / 208 and 270 / 274; eight 317 / 311.
    static bool takes(const mg_rollout_args* a) {
        const uint32_t many = a->steps == 1u ? 131073u : a->steps <= 4u ? 196608u : 0xFFFFFFFFu;
        return !(a->n < 8u && a->obs_out) && a->n < many;
    }
    template <int E>
    static void launch_e(const mg_rollout_args* a, hipStream_t st) {
        const dim3 grid((a->n + E - 1) / E), block(64);
        if (a->mode == MG_ACTIONS_RANDOM)
            hipLaunchKernelGGL((rollout_voxelnav16_kernel<MG_ACTIONS_RANDOM, E>), grid, block, 0, st, *a);
        else
            hipLaunchKernelGGL((rollout_voxelnav16_kernel<MG_ACTIONS_GIVEN, E>), grid, block, 0, st, *a);
    }
    // Few envs per wave while that spreads a short chain over more CUs, up to
    // half a wave where the GPU is full (a whole one leaves one wave per SIMD).
    // us a launch of 32 random steps, the split kernel against this, over 256
    // launches: 52 / 40 at 64 envs, 61 / 40 at 256, 64 / 40 at 1024, 312 / 163 at
    // 65536. Without the launches in which the step cap resets every env, the
    // split kernel against 8 / 16 / 32 / 64 envs per wave: 56 against 41 / 44 /
    // 48 / 56 at 4096 envs, 94 against 58 / 53 / 54 / 59 at 16384, 222 against
    // 183 / 162 / 144 / 146 at 65536, 716 against 590 / 535 / 546 / 573 at 262144.
    static void launch(const mg_rollout_args* a, hipStream_t st) {
        if (a->n < 1024u)
            launch_e<4>(a, st);
        else if (a->n < 8192u)
            launch_e<8>(a, st);
        else if (a->n < 32768u)
            launch_e<16>(a, st);
        else
            launch_e<32>(a, st);
    }
};

}  // namespace dev
}  // namespace mg
