// Env-agnostic policy kernels: forward over arbitrary obs rows (forward()),
// per-row sampling (act() and teacher-forced parity), GAE and the per-block
// advantage statistics used by the PPO loss.
#include "kernels.h"
#include "mg/device/policy_bf16.h"
#include "mg/device/policy_lane.h"
#include "mg/device/policy_pair.h"
#include "mg/device/sample.h"

namespace mg {
namespace dev {

constexpr int kMaxObs = 64;   // OBS_DIM limit of the staged forward
constexpr int kMaxHead = 64;  // ACT_DIM + 1 limit (model/ppo.h:117)

// model/ppo.h:575-626 on `rows` obs rows; rows past the end compute on zeros
// and are not stored.
template <int M, bool BF16>
__global__ void __launch_bounds__(256) forward_kernel(const mg_policy_view pv, const float* __restrict__ obs,
                                                      uint32_t rows, float* __restrict__ head) {
    __shared__ typename std::conditional<BF16, FwdSmemB<M>, FwdSmem<M>>::type sm;
    __shared__ float obsL[M * kMaxObs];
    __shared__ float headL[M * kMaxHead];
    FwdRegs<M> R;
    const int O = (int)pv.obs_dim, HD = (int)pv.head_dim;
    const uint32_t row0 = blockIdx.x * M;
    for (int idx = threadIdx.x; idx < M * O; idx += 256) {
        const uint32_t r = row0 + idx / O;
        obsL[idx] = r < rows ? obs[(size_t)row0 * O + idx] : 0.0f;
    }
    __syncthreads();
    if constexpr (BF16)
        policy_forward_b<M>(pv, small_params(pv), sm, R, obsL, O, headL, HD);
    else
        policy_forward<M>(pv, small_params(pv), sm, R, obsL, O, headL, HD);
    for (int idx = threadIdx.x; idx < M * HD; idx += 256) {
        const uint32_t r = row0 + idx / HD;
        if (r < rows) head[(size_t)row0 * HD + idx] = headL[idx];
    }
}

// The same with a row in a pair of lanes (policy_lane.h), kLaneTile rows per
// workgroup. HC, OC: bounds of the head's and the observation's width.
template <int PREC, int HC, int OC>
__global__ void __launch_bounds__(kLaneNT, 2) forward_lane_kernel(const mg_policy_view pv,
                                                                  const float* __restrict__ obs, uint32_t rows,
                                                                  float* __restrict__ head) {
    extern __shared__ __align__(16) float lane_lds_f[];
    const LaneLds L = lane_lds<PREC, HC, 1>(pv.layers, 0, 0);
    LaneParams<HC> P;
    LaneRing<PREC, 1> ring;
    const int O = (int)pv.obs_dim, HD = (int)pv.head_dim;
    const int lane = threadIdx.x & 63, q = lane >> 5;
    const uint32_t r = blockIdx.x * kLaneTile + (uint32_t)(kLaneRows * (threadIdx.x >> 6) + (lane & 31));
    const float* o = obs + (size_t)(r < rows ? r : rows - 1) * O;
    float ob[(OC + 1) / 2];
#pragma unroll
    for (int s = 0; s < (OC + 1) / 2; ++s) {
        const float v = o[2 * s + q < O ? 2 * s + q : 0];
        ob[s] = 2 * s + q < O ? v : 0.0f;
    }
    lane_start<PREC, HC>(pv, lane_lds_f, L, 0, P, ring);
    float hv[HC];
    lane_forward<PREC, HC, OC, false>(pv, P, ring, O, ob, hv);
    if (r < rows && q == 0) {
#pragma unroll
        for (int j = 0; j < HC; ++j)
            if (j < HD) head[(size_t)r * HD + j] = hv[j];
    }
}

// The same in 16-row tiles with the fp32 products on pairs (policy_pair.h), one
// workgroup per CU. Dynamic LDS: the small parameters, the observations and the
// heads.
__host__ __device__ constexpr uint32_t forward_pair_floats(uint32_t O, uint32_t HD, uint32_t layers) {
    return O * kEmbed + kEmbed + (layers + 1) * 2 * kEmbed + kEmbed * HD + kSplitRows * (O + HD);
}
__global__ void __launch_bounds__(64 * kPairW, 1) forward_pair_kernel(const mg_policy_view pv,
                                                                      const float* __restrict__ obs, uint32_t rows,
                                                                      float* __restrict__ head) {
    constexpr int NT = 64 * kPairW, M = kSplitRows;
    __shared__ PairFwdSmem sm;
    extern __shared__ __align__(16) float pair_lds[];
    const int tid = threadIdx.x, O = (int)pv.obs_dim, HD = (int)pv.head_dim;
    const int lnf = (int)(pv.layers + 1) * 2 * kEmbed;
    PairFwd F;
    F.start(pv);
    SmallParams sp = small_params(pv);
    float* win = pair_lds;
    float* bin = win + O * kEmbed;
    float* ln = bin + kEmbed;
    float* wh = ln + lnf;
    float* obsL = wh + kEmbed * HD;
    float* headL = obsL + M * O;
    const uint32_t row0 = blockIdx.x * M;
#pragma unroll 4
    for (int k = tid; k < O * kEmbed; k += NT) win[k] = sp.win[k];
    for (int k = tid; k < kEmbed; k += NT) bin[k] = sp.bin[k];
    for (int k = tid; k < lnf; k += NT) ln[k] = sp.ln[k];
#pragma unroll 4
    for (int k = tid; k < kEmbed * HD; k += NT) wh[k] = sp.wh[k];
    for (int k = tid; k < M * O; k += NT) obsL[k] = row0 + k / O < rows ? obs[(size_t)row0 * O + k] : 0.0f;
    if (tid < 2 * MG_MAX_LAYERS) sm.exps[tid] = pair_scale(pv.frag_fwd16_bf, pv.count)->cur[tid];
    sp = {win, bin, ln, wh};
    __syncthreads();
    pair_forward<0>(pv, sp, sm, F, obsL, O, headL, HD);
    for (int k = tid; k < M * HD; k += NT)
        if (row0 + k / HD < rows) head[(size_t)row0 * HD + k] = headL[k];
}

// model/sample.metal:18-47 / model/gaussian.metal:42-71, one thread per row.
__global__ void __launch_bounds__(256) sample_kernel(const mg_policy_view pv, const float* __restrict__ head,
                                                     uint32_t rows, uint32_t* __restrict__ rng, void* actions,
                                                     float* __restrict__ logp, float* __restrict__ value) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int A = (int)pv.act_dim, HD = (int)pv.head_dim;
    const float* h = head + (size_t)r * HD;
    uint32_t s = rng[r];
    float lp;
    if (pv.continuous) {
        sample_gaussian(h, pv.params + pv.off_log_std, A, s, static_cast<float*>(actions) + (size_t)r * A, lp);
    } else {
        static_cast<int*>(actions)[r] = sample_categorical(h, A, s, lp);
    }
    rng[r] = s;
    logp[r] = lp;
    value[r] = h[A];
}

// model/gae.metal:14-36: one thread per env, reverse scan over the horizon.
// The [t][n] loads of a lane are independent of the scan, so they are issued
// in batches of 8 ahead of the dependent arithmetic.
__global__ void __launch_bounds__(256) gae_kernel(const float* __restrict__ reward, const uint8_t* __restrict__ done,
                                                  const float* __restrict__ value, const float* __restrict__ head,
                                                  uint32_t head_dim, uint32_t act_dim, uint32_t n, uint32_t horizon,
                                                  float gamma, float lambda, float* __restrict__ adv,
                                                  float* __restrict__ ret) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float lastAdv = 0.0f;
    float nextValue = head[(size_t)i * head_dim + act_dim];
    int t = (int)horizon - 1;
    for (; t >= 7; t -= 8) {
        float r[8], v[8];
        uint8_t d[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t k = (size_t)(t - u) * n + i;
            r[u] = reward[k];
            v[u] = value[k];
            d[u] = done[k];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t k = (size_t)(t - u) * n + i;
            const float nonTerminal = d[u] ? 0.0f : 1.0f;
            const float delta = r[u] + gamma * nextValue * nonTerminal - v[u];
            lastAdv = delta + gamma * lambda * nonTerminal * lastAdv;
            adv[k] = lastAdv;
            ret[k] = lastAdv + v[u];
            nextValue = v[u];
        }
    }
    for (; t >= 0; --t) {
        const size_t k = (size_t)t * n + i;
        const float nonTerminal = done[k] ? 0.0f : 1.0f;
        const float delta = reward[k] + gamma * nextValue * nonTerminal - value[k];
        lastAdv = delta + gamma * lambda * nonTerminal * lastAdv;
        adv[k] = lastAdv;
        ret[k] = lastAdv + value[k];
        nextValue = value[k];
    }
}

// model/gae.metal:42-77 for every minibatch block at once: one workgroup per
// block, two passes (mean, then population variance), deterministic tree sums.
__global__ void __launch_bounds__(256) adv_stats_kernel(const float* __restrict__ adv, uint32_t n,
                                                        uint32_t minibatch, float* __restrict__ stats) {
    __shared__ float red[256];
    const uint32_t b = blockIdx.x, perSlot = n / minibatch;
    const float* a = adv + (size_t)(b / perSlot) * n + (size_t)(b % perSlot) * minibatch;
    float s = 0.0f;
    for (uint32_t r = threadIdx.x; r < minibatch; r += 256) s += a[r];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    const float mean = red[0] / (float)minibatch;
    __syncthreads();
    float q = 0.0f;
    for (uint32_t r = threadIdx.x; r < minibatch; r += 256) {
        const float d = a[r] - mean;
        q += d * d;
    }
    red[threadIdx.x] = q;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const float var = red[0] / (float)minibatch;
        stats[2 * b] = mean;
        stats[2 * b + 1] = 1.0f / (sqrtf(var) + 1e-8f);
    }
}

}  // namespace dev

namespace {
template <int PREC, int HC, int OC>
bool try_forward_lane(hipStream_t st, const mg_policy_view& pv, const float* obs, uint32_t rows, float* head) {
    if (pv.head_dim > (uint32_t)HC || pv.obs_dim > (uint32_t)OC) return false;
    const size_t lds = (size_t)dev::lane_lds<PREC, HC, 1>(pv.layers, 0, 0).total * 4;
    if (lds > 163840 / 2) return false;
    hipLaunchKernelGGL((dev::forward_lane_kernel<PREC, HC, OC>), dim3((rows + dev::kLaneTile - 1) / dev::kLaneTile),
                       dim3(dev::kLaneNT), lds, st, pv, obs, rows, head);
    return true;
}
// Over 8192 rows (65 workgroups): a workgroup takes the time of its chain of
// stages however few there are, so smaller tiles are as fast where they fit the
// GPU once. us a call, CartPole: fp32, forward_kernel / this, 92 / 56 at 8193
// rows, 98 / 56 at 16384, 544 / 176 at 100003 (forward_pair_kernel 44 at 8192);
// bf16 29.8 at 8192, 35.9 / 32 at 8193, 38 / 32 at 16384, 162 / 77 at 100003.
template <int PREC>
bool launch_forward_lane(hipStream_t st, const mg_policy_view& pv, const float* obs, uint32_t rows, float* head) {
    if (rows <= 8192u) return false;
    return try_forward_lane<PREC, 4, 4>(st, pv, obs, rows, head) ||
           try_forward_lane<PREC, 8, 32>(st, pv, obs, rows, head) ||
           try_forward_lane<PREC, 16, 64>(st, pv, obs, rows, head);
}
// An fp32 forward of fewer rows, or of a policy that the lane kernel does not
// take, in the place of forward_kernel's 32-row tiles. Past 4096 rows (a
// workgroup of 16 per CU) only for heads up to 8 columns: the head's columns are
// added one after the other, twice there. us a call, forward_kernel / this, at
// 4096 and 8192 rows, 1 block of hidden 128: 16 / 10 and 16 / 15 (3 columns), 22
// / 12 and 22 / 19 (7), 28 / 23 and 29 / 43 (16), 75 / 68 and 77 / 132 (64); 8
// blocks, at 100003 rows, 646 / 550 (7 columns) and 716 / 830 (16).
bool launch_forward_pair(hipStream_t st, const mg_policy_view& pv, const float* obs, uint32_t rows, float* head) {
    if (rows > 4096u && pv.head_dim > 8) return false;
    static_assert(dev::forward_pair_floats(dev::kMaxObs, dev::kMaxHead, MG_MAX_LAYERS) * 4 + sizeof(dev::PairFwdSmem) <=
                      163840, "the largest policy fits");
    const size_t lds = (size_t)dev::forward_pair_floats(pv.obs_dim, pv.head_dim, pv.layers) * 4;
    hipLaunchKernelGGL(dev::forward_pair_kernel, dim3((rows + dev::kSplitRows - 1) / dev::kSplitRows),
                       dim3(64 * dev::kPairW), lds, st, pv, obs, rows, head);
    return true;
}
}  // namespace

int launch_forward(hipStream_t st, const mg_policy_view& pv, const float* obs, uint32_t rows, float* head) {
    MG_CHECK(pv.obs_dim <= (uint32_t)dev::kMaxObs && pv.head_dim <= (uint32_t)dev::kMaxHead, MG_ERR_INVALID,
             "forward: OBS_DIM must be <= %d and ACT_DIM + 1 <= %d", dev::kMaxObs, dev::kMaxHead);
    if (rows == 0) return MG_OK;
    const dim3 tiles((rows + 31) / 32);
    if (pv.precision == MG_PRECISION_BF16) {
        if (!launch_forward_lane<MG_PRECISION_BF16>(st, pv, obs, rows, head))
            hipLaunchKernelGGL((dev::forward_kernel<32, true>), tiles, dim3(256), 0, st, pv, obs, rows, head);
    } else if (!launch_forward_lane<MG_PRECISION_FP32>(st, pv, obs, rows, head) &&
               !launch_forward_pair(st, pv, obs, rows, head)) {
        hipLaunchKernelGGL((dev::forward_kernel<32, false>), tiles, dim3(256), 0, st, pv, obs, rows, head);
    }
    MG_HIP(hipGetLastError(), "forward launch");
    return MG_OK;
}

int launch_sample(hipStream_t st, const mg_policy_view& pv, const float* head, uint32_t rows, uint32_t* rng,
                  void* actions, float* logp, float* value) {
    if (rows == 0) return MG_OK;
    hipLaunchKernelGGL(dev::sample_kernel, dim3((rows + 255) / 256), dim3(256), 0, st, pv, head, rows, rng, actions,
                       logp, value);
    MG_HIP(hipGetLastError(), "sample launch");
    return MG_OK;
}

int launch_gae(hipStream_t st, const float* reward, const uint8_t* done, const float* value, const float* head,
               uint32_t head_dim, uint32_t act_dim, uint32_t n, uint32_t horizon, float gamma, float lambda,
               float* adv, float* ret) {
    MG_CHECK(act_dim < head_dim, MG_ERR_INVALID, "gae: value column %u outside head width %u", act_dim, head_dim);
    if (n == 0 || horizon == 0) return MG_OK;
    hipLaunchKernelGGL(dev::gae_kernel, dim3((n + 255) / 256), dim3(256), 0, st, reward, done, value, head, head_dim,
                       act_dim, n, horizon, gamma, lambda, adv, ret);
    MG_HIP(hipGetLastError(), "gae launch");
    return MG_OK;
}

int launch_adv_stats(hipStream_t st, const float* adv, uint32_t n, uint32_t horizon, uint32_t minibatch,
                     float* stats) {
    MG_CHECK(minibatch > 0 && n % minibatch == 0, MG_ERR_INVALID, "adv stats: minibatch must divide n");
    const uint32_t blocks = horizon * (n / minibatch);
    hipLaunchKernelGGL(dev::adv_stats_kernel, dim3(blocks), dim3(256), 0, st, adv, n, minibatch, stats);
    MG_HIP(hipGetLastError(), "adv stats launch");
    return MG_OK;
}

}  // namespace mg
