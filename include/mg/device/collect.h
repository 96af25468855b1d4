// collect<Env>: the whole rollout of model/ppo.h:716-751 (minus GAE) in one
// launch. Each workgroup (4 waves; 8 for 16-row tiles) owns M envs for all T steps:
//
//   for t in 0..T:  policy forward on the staged obs (MFMA, see policy.h)
//                   t <  T: env lanes sample from the head with their own RNG,
//                           reset-if-done, Env::step, write the [T][n] slots
//                   t == T: write the bootstrap head (model/ppo.h:735)
//
// Env lanes are threads 0..M-1 (one wave). A small State lives in registers of
// its lane for the whole rollout; a larger one is staged in LDS for the T steps
// when the tile's envs fit beside the forward's LDS (copied in and out by the
// whole workgroup), else it is updated in place in device memory. Per env and
// step the RNG order is: sample draw(s), reset draws if done, then step
// (model/ppo.h:728-730, rollout.h:46-47). An env that declares a split
// observation (OBS_SPLIT, env.h) has its states stepped by the env lanes,
// which also write the observation's other floats; after a barrier all threads
// of the workgroup compute the tile's OBS_SPLIT parts per env.
#pragma once
#include "policy_bf16.h"
#include "policy_lane.h"
#include "policy_pair.h"
#include "policy_split.h"
#include "sample.h"

namespace mg {
namespace dev {

// Launch shape per tile height: 64- and 32-row tiles run 4 waves and two
// workgroups per CU (one when the env lane holds more than 32 observation
// floats, which do not fit beside the weights at two, unless WIDE); 16-row
// tiles (runs of at most 512 workgroups, one per CU) of envs with up to 16
// observation floats run 8 waves, 16 output columns each (a wider observation
// held by the env lane would not fit the register budget of 8 waves).
// WIDE: an env with a split observation whose states stay in device memory,
// two workgroups per CU (VoxelNav's 40 observation floats: 231 VGPRs, no
// spills), so one workgroup's env phase overlaps the other's GEMMs.
template <int M, int O, bool WIDE = false>
struct CollectShape {
    static constexpr int W = M == 16 && O <= 16 ? 8 : 4;
    static constexpr int NT = 64 * W;
    static constexpr int MIN_WG = M == 16 || (O > 32 && !WIDE) ? 1 : 2;  // workgroups per CU
};

// The forward of a tile: fp32 16-row tiles on 8 waves run the split layout
// (split_forward16: no barrier per chunk, and the relu'd hidden chunk never
// goes through LDS); the others stage each hidden chunk in LDS (policy.h,
// policy_bf16.h).
template <int M, int O, bool BF16>
struct CollectFwd {
    static constexpr bool SPLIT = !BF16 && M == 16 && CollectShape<M, O>::W == 8;
    using Smem = std::conditional_t<SPLIT, SplitFwdSmem<8>, std::conditional_t<BF16, FwdSmemB<M>, FwdSmem<M>>>;
};

// The tile's LDS: the forward's, then the staged observations and the head.
// Outside the split forward the observations ([M][O]) and the head ([M][HD])
// share the forward's hidden-chunk buffer: the observations are read only by
// the embed, before the first chunk is written (LN0's barriers between), and
// the head is written after the final LN's first barrier, when every wave is
// done with the last chunk; the env phase that reads the head and writes the
// next observations ends before the next forward. That leaves room at two
// workgroups per CU for VoxelNav16's small parameters but W_in (SmallStage).
// 16-byte aligned in size as well, so the dynamic LDS after the static
// arrays (the staged small parameters, read as float4s) starts 16-byte
// aligned: at 4 bytes past a 16-byte boundary the CartPole collect ran 8%
// slower, bf16 41%.
template <int M, int O, int HD, bool BF16>
struct alignas(16) CollectSmem {
    using Fwd = typename CollectFwd<M, O, BF16>::Smem;
    static constexpr size_t IO = (size_t)M * (O + HD);  // floats: obs, then head
    static constexpr bool ALIAS = !CollectFwd<M, O, BF16>::SPLIT && IO * 4 <= (BF16 ? (size_t)M * kLdsB * 2
                                                                                       : (size_t)M * kLds * 4);
    Fwd fwd;
    float io[ALIAS ? 1 : IO];
    __device__ __forceinline__ float* obs() {
        if constexpr (ALIAS) {
            if constexpr (BF16)
                return reinterpret_cast<float*>(&fwd.vb[0][0]);
            else
                return &fwd.vs[0][0];
        } else {
            return io;
        }
    }
    __device__ __forceinline__ float* head() { return obs() + M * O; }
};

// LDS staging of a State too large for registers: the tile's M states at an
// odd stride of dwords (env e at dword e * STRIDE), so the lanes' accesses to
// one field fall in different banks. Used when the states fit beside the
// forward's LDS at the kernel's workgroups per CU; gathers from a state (a
// VoxelNav heightmap's ray march) then cost an LDS round trip instead of a
// cache miss.
template <typename Env, int M, bool BF16, bool WIDE = false>
struct LdsState {
    using State = typename Env::State;
    static constexpr uint32_t SD = sizeof(State) / 4;           // dwords per state
    static constexpr uint32_t STRIDE = SD % 2 ? SD : SD + 1;   // odd dword stride
    static constexpr size_t BYTES = (size_t)M * STRIDE * 4;
    static constexpr int O = Env::OBS_DIM, HD = Env::ACT_DIM + 1;
    // 256 bytes of headroom for the compiler's alignment padding between the
    // two static LDS arrays
    static constexpr bool USE = !WIDE && !EnvTraits<Env>::STATE_IN_REGISTERS && sizeof(State) % 4 == 0 &&
                                alignof(State) <= 4 &&
                                sizeof(CollectSmem<M, O, HD, BF16>) + BYTES + 256 <=
                                    (size_t)163840 / CollectShape<M, O>::MIN_WG;
};

// LDS copies of the forward's small parameters for the T + 1 forwards of a
// collect (W_in, b_in, the layers + 1 LNs' gamma and beta, W_head), in the
// kernel's dynamic LDS: the embed, LN and head phases then read them without
// an L2 round trip (at one workgroup per CU no other workgroup's MFMAs overlap
// that latency; at two, 64-row tiles, it took the 262144-env CartPole collect
// from 36.0 to 35.4 ms). Used when they fit beside the kernel's static LDS at
// its workgroups per CU (kAll); else all but W_in where those fit (kNoWin:
// W_in is read once per step, by the embed's MFMAs), else none and the forward
// reads the arena. The launcher decides from the static size the compiler gave
// the kernel (padding included) and passes the decision as the kernel's
// second argument.
template <typename Env, int M, bool BF16>
struct SmallStage {
    static constexpr int O = Env::OBS_DIM, HD = Env::ACT_DIM + 1;
    static constexpr int WIN = O * kEmbed, BIN = kEmbed, WH = kEmbed * HD;
    static constexpr uint32_t kNone = 0, kAll = 1, kNoWin = 2;
    __host__ __device__ static constexpr uint32_t floats(uint32_t layers, uint32_t mode = kAll) {
        return (mode == kAll ? WIN : 0) + BIN + (layers + 1) * 2 * kEmbed + WH;
    }
};

// BF16: the policy forward multiplies bfloat16 operands (policy_bf16.h).
template <typename Env, int M, bool BF16, bool WIDE>
__global__ void __launch_bounds__((CollectShape<M, Env::OBS_DIM, WIDE>::NT),
                                  (CollectShape<M, Env::OBS_DIM, WIDE>::MIN_WG))
    collect_kernel(const mg_collect_args a, const uint32_t stage_small) {
    using Tr = EnvTraits<Env>;
    using State = typename Env::State;
    using Action = typename Env::Action;
    using Obs = typename Env::Obs;
    using CS = CollectShape<M, Env::OBS_DIM, WIDE>;
    using LS = LdsState<Env, M, BF16, WIDE>;
    constexpr int O = Env::OBS_DIM, A = Env::ACT_DIM, HD = A + 1;
    // the embed's observation width at compile time (its unrolled k loop reads
    // a row's floats together: VoxelNav at 262144 envs 70.8 -> 66.0 ms) at
    // 64-row and WIDE tiles; the others' register budgets it would overflow
    // (VoxelNav's 32-row tiles with states in LDS: 44 VGPRs spilled)
    constexpr int OE = M == 64 || WIDE ? O : 0;
    // parts of a split observation per env, spread over the whole workgroup
    // when the states sit in LDS or (WIDE) in device memory (0: the env lanes
    // call step()). A State held in registers is written back only at the end,
    // so the other threads could not read it: such an env always calls step().
    constexpr uint32_t KS = LS::USE || (WIDE && !Tr::STATE_IN_REGISTERS) ? Tr::OBS_SPLIT : 0;
    __shared__ CollectSmem<M, O, HD, BF16> sm;
    static_assert(sizeof(CollectSmem<M, O, HD, BF16>) % 16 == 0, "the staged small parameters start 16-byte aligned");
    __shared__ uint32_t lds_state[LS::USE ? M * LS::STRIDE : 1];
    using SS = SmallStage<Env, M, BF16>;
    extern __shared__ __align__(16) float small_lds[];  // SS::floats(layers, stage_small) floats
    FwdRegs<M, CS::W> R;
    std::conditional_t<CollectFwd<M, O, BF16>::SPLIT, SkStream<8 / CS::W>, char> wst;  // split forward's weights

    const int tid = threadIdx.x;
    const uint32_t n = a.n, T = a.horizon;
    const uint32_t i = blockIdx.x * M + (uint32_t)tid;
    const bool envLane = tid < M;
    State* states = static_cast<State*>(a.state);
    Action* actSlots = static_cast<Action*>(a.action_slots);
    const float* logStd = a.policy.params + a.policy.off_log_std;

    uint32_t rng = 0;
    uint8_t done = 0;
    // A small State lives in this register copy; a larger one in LDS or, if it
    // does not fit there, in place in device memory.
    std::conditional_t<Tr::STATE_IN_REGISTERS, State, char> sreg;
    auto S = [&]() -> State& {
        if constexpr (Tr::STATE_IN_REGISTERS)
            return sreg;
        else if constexpr (LS::USE)
            return *reinterpret_cast<State*>(lds_state + tid * LS::STRIDE);
        else
            return states[i];
    };
    if constexpr (LS::USE) {
        // the tile's states are contiguous in device memory: dword k of the run
        // is dword k % SD of env k / SD
        const uint32_t* gin = reinterpret_cast<const uint32_t*>(states + (size_t)blockIdx.x * M);
        states_to_lds<LS::SD, LS::STRIDE, M, CS::NT>(lds_state, gin, M);
        __syncthreads();
    }
    float obs[O];

    SmallParams sp = small_params(a.policy);
    // a runtime choice: a template parameter instead (LDS instructions for the
    // small parameters) measured slower at 4096 and 262144 envs, fp32 and bf16
    if (stage_small) {  // ordered before the forwards by the barrier below
        const int lnf = (int)(a.policy.layers + 1) * 2 * kEmbed;
        const bool all = stage_small == SS::kAll;
        float* win = small_lds;
        float* bin = win + (all ? SS::WIN : 0);
        float* ln = bin + SS::BIN;
        float* wh = ln + lnf;
        if (all)
            for (int k = tid; k < SS::WIN; k += CS::NT) win[k] = sp.win[k];
        for (int k = tid; k < SS::BIN; k += CS::NT) bin[k] = sp.bin[k];
        for (int k = tid; k < lnf; k += CS::NT) ln[k] = sp.ln[k];
        for (int k = tid; k < SS::WH; k += CS::NT) wh[k] = sp.wh[k];
        sp = {all ? win : sp.win, bin, ln, wh};
    }

    if (envLane) {
        rng = a.rng[i];
        done = a.done[i];
        if constexpr (Tr::STATE_IN_REGISTERS) sreg = states[i];
        if (a.first) {  // model/ppo.h:720-722: one step with action 0 into slot 0
            Action act{};
            if (done) Env::reset(S(), rng);
            Obs o{};
            float r = 0.0f;
            Env::step(S(), act, o, r, done);
            const float* of = reinterpret_cast<const float*>(&o);
#pragma unroll
            for (int k = 0; k < O; ++k) obs[k] = of[k];
            store_floats<O>(a.obs_slots + (size_t)i * O, obs);
            a.reward_slots[i] = r;
        } else {  // model/ppo.h:724: obs[T] -> obs[0]
            load_floats<O>(obs, a.obs_slots + ((size_t)T * n + i) * O);
            store_floats<O>(a.obs_slots + (size_t)i * O, obs);
        }
#pragma unroll
        for (int k = 0; k < O; ++k) sm.obs()[tid * O + k] = obs[k];
    }
    __syncthreads();

    for (uint32_t t = 0; t <= T; ++t) {
        if constexpr (CollectFwd<M, O, BF16>::SPLIT)
            split_forward16<CS::W, O>(a.policy, sp, sm.fwd, wst, t == 0, sm.obs(), sm.head(), HD);
        else if constexpr (BF16)
            policy_forward_b<M, CS::W, HD, OE>(a.policy, sp, sm.fwd, R, sm.obs(), O, sm.head(), HD);
        else
            // global weight loads when the env states sit in LDS: there the
            // buffer loads' scalar descriptors cost the heightmap env more
            // spilling than they save (VoxelNav at 262144 envs, 135 -> 151 ms)
            policy_forward<M, CS::W, !LS::USE, HD, OE>(a.policy, sp, sm.fwd, R, sm.obs(), O, sm.head(), HD);
        if (envLane) {
            const float* h = sm.head() + tid * HD;
            if (t == T) {  // bootstrap head for GAE and headValue()
#pragma unroll
                for (int j = 0; j < HD; ++j) a.head_out[(size_t)i * HD + j] = h[j];
            } else {
                const size_t k = (size_t)t * n + i;
                Action act;
                float lp;
                if constexpr (Tr::CONTINUOUS)
                    sample_gaussian(h, logStd, A, rng, reinterpret_cast<float*>(&act), lp);
                else
                    act = (Action)sample_categorical(h, A, rng, lp);
                actSlots[k] = act;
                a.logp_slots[k] = lp;
                a.value_slots[k] = h[A];
                if (done) Env::reset(S(), rng);
                Obs o{};
                float r = 0.0f;
                const float* of = reinterpret_cast<const float*>(&o);
                if constexpr (KS > 0) {  // the floats from KS on; the parts after the barrier below
                    Env::stepState(S(), act, r, done);
                    Env::observeRest(S(), o);
#pragma unroll
                    for (int q = KS; q < O; ++q) {
                        a.obs_slots[(k + n) * O + q] = of[q];
                        sm.obs()[tid * O + q] = of[q];
                    }
                } else {
                    Env::step(S(), act, o, r, done);
#pragma unroll
                    for (int q = 0; q < O; ++q) obs[q] = of[q];
                    store_floats<O>(a.obs_slots + (k + n) * O, obs);
#pragma unroll
                    for (int q = 0; q < O; ++q) sm.obs()[tid * O + q] = obs[q];
                }
                a.reward_slots[k] = r;
                a.done_slots[k] = done;
            }
        }
        if constexpr (KS > 0) {
            if (t < T) {
                __syncthreads();  // every env lane's state is stepped
                // part p of env e, consecutive threads on consecutive parts
                const size_t row0 = ((size_t)(t + 1) * n + (size_t)blockIdx.x * M) * O;
                for (uint32_t q = tid; q < M * KS; q += CS::NT) {
                    const uint32_t e = q / KS, p = q % KS;
                    const State& se = LS::USE ? *reinterpret_cast<const State*>(lds_state + e * LS::STRIDE)
                                              : states[(size_t)blockIdx.x * M + e];
                    const float v = Env::observePart(se, p);
                    sm.obs()[e * O + p] = v;
                    a.obs_slots[row0 + (size_t)e * O + p] = v;
                }
            }
        }
        __syncthreads();
    }
    if (envLane) {
        if constexpr (Tr::STATE_IN_REGISTERS) states[i] = sreg;
        a.rng[i] = rng;
        a.done[i] = done;
    }
    if constexpr (LS::USE) {  // every env lane's last step is before the loop's final barrier
        uint32_t* gout = reinterpret_cast<uint32_t*>(states + (size_t)blockIdx.x * M);
        states_from_lds<LS::SD, LS::STRIDE, M, CS::NT>(lds_state, gout, M);
    }
}

// collect on the row-per-lane-pair forward (policy_lane.h): four waves, lanes
// 0 .. 31 of a wave of share 0 its env lanes. With one share a workgroup has 128
// envs and two of them a CU; observations pass between the lanes of a wave, so
// the only barriers are the weight ring's, and a wave's LN, head and env phases
// run beside the other workgroup's products. With two shares a workgroup has 64
// envs and a CU to itself; share 1 gets the observations through LDS.
template <typename Env, int PREC, int HS>
struct CollectLane {
    using Tr = EnvTraits<Env>;
    static constexpr int O = Env::OBS_DIM, HD = Env::ACT_DIM + 1;
    static constexpr int HC = (HD + 3) / 4 * 4;  // head columns, padded
    // parts of a split observation: lane (n, q) computes the parts p = 2 s + q
    // of row n, which are its embed operands
    static constexpr uint32_t KS = Tr::STATE_IN_REGISTERS ? 0 : Tr::OBS_SPLIT;
    static constexpr int NOB = (O + 1) / 2;
    static constexpr uint32_t WIN = O <= 16 * HS ? O * kEmbed : 0;  // W_in in LDS
    // a wave's heads; an fp32 policy's categorical draws near an edge also need
    // a row's scratch (tile_row_head)
    static constexpr bool EDGE = PREC == MG_PRECISION_FP32 && !Tr::CONTINUOUS && Env::ACT_DIM > 1;
    static constexpr uint32_t ROW = (kLaneRows * HD + 3) / 4 * 4;
    static constexpr uint32_t IO = ROW + (EDGE ? kLaneRowLds : 0);
    static constexpr bool OK = HD <= 16;  // the head's columns are registers
};

template <typename Env, int PREC, int HS>
__global__ void __launch_bounds__(kLaneNT, LaneShape<HS>::WG) collect_lane_kernel(const mg_collect_args a) {
    using CL = CollectLane<Env, PREC, HS>;
    using Ring = LaneRing<PREC, HS>;
    constexpr int RG = LaneShape<HS>::RG;
    using Tr = EnvTraits<Env>;
    using State = typename Env::State;
    using Action = typename Env::Action;
    using Obs = typename Env::Obs;
    constexpr int O = CL::O, A = Env::ACT_DIM, HD = CL::HD, HC = CL::HC, NOB = CL::NOB;
    constexpr uint32_t KS = CL::KS;
    extern __shared__ __align__(16) float lane_lds_f[];
    const LaneLds L = lane_lds<PREC, HC, HS>(a.policy.layers, CL::WIN, CL::IO);
    LaneParams<HC> P;
    Ring ring;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, row = lane & 31, q = lane >> 5;
    const bool lead = HS == 1 || wave < RG;  // share 0, which has the envs
    const uint32_t n = a.n, T = a.horizon;
    const uint32_t i0 = blockIdx.x * LaneShape<HS>::TILE + (uint32_t)(kLaneRows * rg);
    // n is a multiple of 64, so a wave's rows are all there or none; a wave of
    // none still moves its share of the weights, on row 0's values
    const bool valid = i0 < n;
    const uint32_t i = valid ? i0 + (uint32_t)row : (uint32_t)row;
    const bool envLane = valid && q == 0 && lead;
    const bool wide = n >= 64u * 512u;  // the tile height that launch_collect_tiles would take
    float* ioL = lane_lds_f + L.io + rg * (int)CL::IO;
    float* headL = ioL + row * HD;
    State* states = static_cast<State*>(a.state);
    Action* actSlots = static_cast<Action*>(a.action_slots);
    const float* logStd = a.policy.params + a.policy.off_log_std;

    uint32_t rng = 0;
    uint8_t done = 0;
    std::conditional_t<Tr::STATE_IN_REGISTERS, State, char> sreg;
    auto S = [&]() -> State& {
        if constexpr (Tr::STATE_IN_REGISTERS)
            return sreg;
        else
            return states[i];
    };
    float ob[NOB];  // this lane's embed operands: observation floats 2 s + q of its row
    // Steps the env lanes with act and passes the observation on: to its slot
    // and to the lanes' embed operands.
    auto env_step = [&](const Action& act, size_t slot, float& r) {
        if constexpr (KS > 0) {
            if (envLane) {
                if (done) Env::reset(S(), rng);
                Env::stepState(S(), act, r, done);
            }
            // the stepped state is read by both lanes of the row
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            const State& s = states[i];
            Obs o{};
            Env::observeRest(s, o);
            const float* of = reinterpret_cast<const float*>(&o);
#pragma unroll
            for (int u = 0; u < NOB; ++u) {
                constexpr int K = (int)KS;
                float v = 0.0f;
                if (2 * u + 1 < K) {
                    v = Env::observePart(s, 2 * u + q);
                } else {
                    const float e = 2 * u < K ? 0.0f : of[2 * u];
                    const float d = 2 * u + 1 < O ? of[2 * u + 1 < O ? 2 * u + 1 : 0] : 0.0f;
                    v = q ? d : e;
                    if (2 * u < K) {
                        if (q == 0) v = Env::observePart(s, 2 * u);
                    }
                }
                ob[u] = v;
                if (valid && 2 * u + q < O) a.obs_slots[slot * O + 2 * u + q] = v;
            }
        } else {
            float obs[2 * NOB];
#pragma unroll
            for (int k = 0; k < 2 * NOB; ++k) obs[k] = 0.0f;
            if (envLane) {
                if (done) Env::reset(S(), rng);
                Obs o{};
                Env::step(S(), act, o, r, done);
                const float* of = reinterpret_cast<const float*>(&o);
#pragma unroll
                for (int k = 0; k < O; ++k) obs[k] = of[k];
                store_floats<O>(a.obs_slots + slot * O, obs);
            }
#pragma unroll
            for (int u = 0; u < NOB; ++u) ob[u] = lane_give(obs[2 * u], obs[2 * u + 1]);
        }
    };

    lane_start<PREC, HC>(a.policy, lane_lds_f, L, CL::WIN, P, ring);
    if (envLane) {
        rng = a.rng[i];
        done = a.done[i];
        if constexpr (Tr::STATE_IN_REGISTERS) sreg = states[i];
    }
    // the observations to share 1
    auto share = [&]() {
        if constexpr (HS > 1) {
            static_assert(NOB * 64 <= 2048 * LaneEx<PREC>::N, "a row group's observations fit");
            float* at = reinterpret_cast<float*>(LaneEx<PREC>::at(ring, rg)) + lane;
            if (lead)
#pragma unroll
                for (int u = 0; u < NOB; ++u) at[64 * u] = ob[u];
            Ring::barrier();
            if (!lead)
#pragma unroll
                for (int u = 0; u < NOB; ++u) ob[u] = at[64 * u];
        }
    };
    if (!lead) {
    } else if (a.first) {  // model/ppo.h:720-722: one step with action 0 into slot 0
        Action act{};
        float r = 0.0f;
        env_step(act, i, r);
        if (envLane) a.reward_slots[i] = r;
    } else {  // model/ppo.h:724: obs[T] -> obs[0]
#pragma unroll
        for (int u = 0; u < NOB; ++u) {
            const bool in = 2 * u + q < O;
            const float v = a.obs_slots[((size_t)T * n + i) * O + (in ? 2 * u + q : 0)];
            ob[u] = in ? v : 0.0f;
            if (valid && in) a.obs_slots[(size_t)i * O + 2 * u + q] = v;
        }
    }

    share();

    for (uint32_t t = 0; t <= T; ++t) {
        float hv[HC];
        lane_forward<PREC, HC, O, (CL::WIN > 0)>(a.policy, P, ring, O, ob, hv);
        if (t == T) {  // bootstrap head for GAE and headValue()
            if (envLane) {
#pragma unroll
                for (int j = 0; j < HD; ++j) a.head_out[(size_t)i * HD + j] = hv[j];
            }
            break;
        }
        if (lead) {
            const size_t k = (size_t)t * n + i;
            Action act{};
            float r = 0.0f, lp = 0.0f, edge = 1.0f;
            const uint32_t rng0 = rng;
            if (envLane) {
    #pragma unroll
                for (int j = 0; j < HD; ++j) headL[j] = hv[j];  // the samplers index the row
                if constexpr (Tr::CONTINUOUS)
                    sample_gaussian(headL, logStd, A, rng, reinterpret_cast<float*>(&act), lp);
                else
                    act = (Action)sample_categorical(headL, A, rng, lp, CL::EDGE ? &edge : nullptr);
            }
            if constexpr (CL::EDGE) {
                for (uint64_t near = __ballot(envLane && edge <= kLaneEdge); near; near &= near - 1) {
                    const int e = __builtin_ctzll(near);
                    const float* ep = a.obs_slots + ((size_t)t * n + i0 + (uint32_t)e) * O;
                    if (wide)
                        tile_row_head<32, O, HD>(a.policy, ep, ioL + CL::ROW, ioL + e * HD);
                    else
                        tile_row_head<16, O, HD>(a.policy, ep, ioL + CL::ROW, ioL + e * HD);
                    if (lane == e) {
                        const float mine = lp;
                        uint32_t s = rng0;
                        const Action own = act;
                        act = (Action)sample_categorical(headL, A, s, lp);
                        if (act == own) lp = mine;
                    }
                }
            }
            if (envLane) {
                actSlots[k] = act;
                a.logp_slots[k] = lp;
                a.value_slots[k] = hv[A];
            }
            env_step(act, k + n, r);
            if (envLane) {
                a.reward_slots[k] = r;
                a.done_slots[k] = done;
            }
        }
        share();
    }
    if (envLane) {
        if constexpr (Tr::STATE_IN_REGISTERS) states[i] = sreg;
        a.rng[i] = rng;
        a.done[i] = done;
    }
}

// collect of 16-row tiles with the forward on pairs (pair_forward): eight
// waves, one workgroup per CU, env lanes 0 .. 15 of wave 0.
template <typename Env>
struct CollectPair {
    static constexpr int O = Env::OBS_DIM, HD = Env::ACT_DIM + 1;
    static constexpr bool OK = O <= 16 && HD <= 16 && EnvTraits<Env>::STATE_IN_REGISTERS;
    static constexpr bool EDGE = !EnvTraits<Env>::CONTINUOUS && Env::ACT_DIM > 1;
    // floats of the small parameters, each array a multiple of 4
    __host__ __device__ static constexpr uint32_t small(uint32_t layers) {
        return O * kEmbed + kEmbed + (layers + 1) * 2 * kEmbed + kEmbed * HD;
    }
};

template <typename Env>
__global__ void __launch_bounds__(64 * kPairW, 1) collect_pair_kernel(const mg_collect_args a) {
    using CP = CollectPair<Env>;
    using Tr = EnvTraits<Env>;
    using State = typename Env::State;
    using Action = typename Env::Action;
    using Obs = typename Env::Obs;
    constexpr int M = kSplitRows, NT = 64 * kPairW, O = CP::O, A = Env::ACT_DIM, HD = CP::HD;
    __shared__ PairFwdSmem sm;
    __shared__ float obsL[M * O];
    __shared__ float headL[M * HD];
    __shared__ float edgeHead[HD];
    __shared__ uint32_t near;  // env lanes whose draw fell near an edge
    extern __shared__ __align__(16) float small_lds[];

    const int tid = threadIdx.x;
    const uint32_t n = a.n, T = a.horizon, i = blockIdx.x * M + (uint32_t)tid;
    const bool envLane = tid < M;
    State* states = static_cast<State*>(a.state);
    Action* actSlots = static_cast<Action*>(a.action_slots);
    const float* logStd = a.policy.params + a.policy.off_log_std;

    PairFwd F;
    F.start(a.policy);
    SmallParams sp = small_params(a.policy);
    {
        const int lnf = (int)(a.policy.layers + 1) * 2 * kEmbed;
        float* win = small_lds;
        float* bin = win + O * kEmbed;
        float* ln = bin + kEmbed;
        float* wh = ln + lnf;
        for (int k = tid; k < O * kEmbed; k += NT) win[k] = sp.win[k];
        for (int k = tid; k < kEmbed; k += NT) bin[k] = sp.bin[k];
        for (int k = tid; k < lnf; k += NT) ln[k] = sp.ln[k];
        for (int k = tid; k < kEmbed * HD; k += NT) wh[k] = sp.wh[k];
        sp = {win, bin, ln, wh};
        if (tid < 2 * MG_MAX_LAYERS) sm.exps[tid] = pair_scale(a.policy.frag_fwd16_bf, a.policy.count)->cur[tid];
    }
    uint32_t rng = 0;
    uint8_t done = 0;
    State st;
    auto env_step = [&](const Action& act, size_t slot, float& r) {
        if (done) Env::reset(st, rng);
        Obs o{};
        Env::step(st, act, o, r, done);
        const float* of = reinterpret_cast<const float*>(&o);
        float obs[O];
#pragma unroll
        for (int k = 0; k < O; ++k) obs[k] = of[k];
        store_floats<O>(a.obs_slots + slot * O, obs);
#pragma unroll
        for (int k = 0; k < O; ++k) obsL[tid * O + k] = obs[k];
    };
    if (envLane) {
        rng = a.rng[i];
        done = a.done[i];
        st = states[i];
        if (a.first) {  // model/ppo.h:720-722: one step with action 0 into slot 0
            Action act{};
            float r = 0.0f;
            env_step(act, i, r);
            a.reward_slots[i] = r;
        } else {  // model/ppo.h:724: obs[T] -> obs[0]
            float obs[O];
            load_floats<O>(obs, a.obs_slots + ((size_t)T * n + i) * O);
            store_floats<O>(a.obs_slots + (size_t)i * O, obs);
#pragma unroll
            for (int k = 0; k < O; ++k) obsL[tid * O + k] = obs[k];
        }
    }
    __syncthreads();

    for (uint32_t t = 0; t <= T; ++t) {
        pair_forward<O>(a.policy, sp, sm, F, obsL, O, headL, HD);
        if (t == T) {  // bootstrap head for GAE and headValue()
            if (envLane) {
#pragma unroll
                for (int j = 0; j < HD; ++j) a.head_out[(size_t)i * HD + j] = headL[tid * HD + j];
            }
            break;
        }
        const size_t k = (size_t)t * n + i;
        const uint32_t rng0 = rng;
        Action act{};
        float r = 0.0f, lp = 0.0f, edge = 1.0f;
        if (envLane) {
            const float* h = headL + tid * HD;
            if constexpr (Tr::CONTINUOUS)
                sample_gaussian(h, logStd, A, rng, reinterpret_cast<float*>(&act), lp);
            else
                act = (Action)sample_categorical(h, A, rng, lp, CP::EDGE ? &edge : nullptr);
        }
        if constexpr (CP::EDGE) {
            // draws near an edge take the action of the fp32 tiles' arithmetic
            // (policy_lane.h): of the 32-row tile from 8192 envs, else of
            // split_forward16
            if (tid < 64) {
                const uint64_t b = __ballot(envLane && edge <= kLaneEdge);
                if (tid == 0) near = (uint32_t)b;
            }
            __syncthreads();
            for (uint32_t rest = near; rest; rest &= rest - 1) {
                const int e = __builtin_ctz(rest);
                if (n >= 32u * 256u) {
                    if (tid < 64) tile_row_head<16, O, HD>(a.policy, obsL + e * O, &sm.red[0][0], edgeHead);
                    __syncthreads();
                } else {
                    split_row_head<O, HD>(a.policy, sp, obsL + e * O, blockIdx.x, &sm.red[0][0], edgeHead);
                }
                if (tid == e) {
                    const float mine = lp;
                    uint32_t s = rng0;
                    const Action own = act;
                    act = (Action)sample_categorical(edgeHead, A, s, lp);
                    if (act == own) lp = mine;
                }
                __syncthreads();  // edgeHead and red are free again
            }
        }
        if (envLane) {
            actSlots[k] = act;
            a.logp_slots[k] = lp;
            a.value_slots[k] = headL[tid * HD + A];
            env_step(act, k + n, r);
            a.reward_slots[k] = r;
            a.done_slots[k] = done;
        }
        __syncthreads();
    }
    if (envLane) {
        states[i] = st;
        a.rng[i] = rng;
        a.done[i] = done;
    }
}

// Runs the collect on collect_pair_kernel where that is the faster: to 8192 envs
// (two workgroups per CU, one after the other) of an env with at most 16
// observation floats and a register-held State. ms a collect of 32 steps,
// CartPole, split_forward16 or the 32-row tiles against this: 0.63 / 0.40 at 64
// envs, 0.65 / 0.42 at 4096, 1.34 / 0.83 at 8192 (collect_lane_kernel 1.06),
// 2.32 / 1.22 at 12288 (1.10). A step takes 14 us at 4096 envs, of
// which the weights' 1 MB through each CU's L1 is about 11. At exactly 8192 the
// steps between the products of the smallest network, one block of 128 units,
// cost more than the products gain: 8 steps of CartPole 80 us on the tiles, 86 here.
// So does a wide head, whose columns the 16 env lanes of a workgroup take one after
// the other: past 8 columns only networks of 1024 hidden units and more come
// here, and fewer than 8192 envs. us a collect of 3 steps of 15 floats and 16
// columns, tiles / this, at 64, 4096, 6144 and 8192 envs: 94 / 100, 98 / 114, 187 /
// 199 and 83 / 145 (1 block of 128), 149 / 129, 160 / 150, 301 / 267 and 215 /
// 320 (2 of 512); 16 steps of 4096 envs, 5 columns, 1 of 128, 103 / 107.
template <typename Env>
bool launch_collect_pair(const mg_collect_args* a, hipStream_t st) {
    using CP = CollectPair<Env>;
    if constexpr (CP::OK) {
        const uint32_t units = a->policy.layers * a->policy.hidden;
        if (a->policy.precision != MG_PRECISION_FP32 || !a->policy.frag_fwd16_bf) return false;
        if (a->n > (CP::HD > 8 || units <= 128u ? 8191u : 8192u)) return false;
        if (CP::HD > 4 && units <= 128u) return false;
        if (CP::HD > 8 && (units < 1024u || a->policy.hidden < 512u)) return false;
        hipLaunchKernelGGL((collect_pair_kernel<Env>), dim3(a->n / kSplitRows), dim3(64 * kPairW),
                           CP::small(a->policy.layers) * 4, st, *a);
        return true;
    } else {
        return false;
    }
}

// The kernel's static LDS as the compiler laid it out (SIZE_MAX if the
// runtime cannot tell, which turns the small-parameter staging off).
template <typename Env, int M, bool BF16, bool WIDE>
size_t collect_static_lds() {
    static const size_t bytes = [] {
        hipFuncAttributes attr{};
        if (hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&collect_kernel<Env, M, BF16, WIDE>)) !=
            hipSuccess) {
            (void)hipGetLastError();  // not this launch's error
            return (size_t)SIZE_MAX;
        }
        return (size_t)attr.sharedSizeBytes;
    }();
    return bytes;
}

template <typename Env, int M, bool BF16, bool WIDE>
void launch_collect_mw(const mg_collect_args* a, hipStream_t st) {
    using SS = SmallStage<Env, M, BF16>;
    constexpr size_t kPerWg = (size_t)163840 / CollectShape<M, Env::OBS_DIM, WIDE>::MIN_WG;  // LDS per workgroup
    const size_t stat = collect_static_lds<Env, M, BF16, WIDE>();
    const size_t all = (size_t)SS::floats(a->policy.layers, SS::kAll) * 4;
    const size_t nowin = (size_t)SS::floats(a->policy.layers, SS::kNoWin) * 4;
    const size_t room = stat <= kPerWg ? kPerWg - stat : 0;
    const uint32_t stage = all <= room ? SS::kAll : nowin <= room ? SS::kNoWin : SS::kNone;
    const size_t dyn = stage == SS::kAll ? all : stage == SS::kNoWin ? nowin : 0;
    const dim3 grid(a->n / M), block(CollectShape<M, Env::OBS_DIM, WIDE>::NT);
    hipLaunchKernelGGL((collect_kernel<Env, M, BF16, WIDE>), grid, block, dyn, st, *a, stage);
}

// An env with a split observation runs WIDE where the grid has at least two
// workgroups per CU (VoxelNav, ms per collect of 32 steps, WIDE against its
// states in LDS at one workgroup per CU: 70.9 / 77.9 at 262144 envs, 4.53 /
// 5.47 at 16384; at 8192 envs, 256 workgroups, 3.23 / 2.81).
template <typename Env, int M, bool BF16>
void launch_collect_m(const mg_collect_args* a, hipStream_t st) {
    if constexpr (EnvTraits<Env>::OBS_SPLIT > 0 && M >= 32) {
        if (a->n / M >= 512) {
            launch_collect_mw<Env, M, BF16, true>(a, st);
            return;
        }
    }
    launch_collect_mw<Env, M, BF16, false>(a, st);
}

// The LDS bytes of a workgroup of collect_lane_kernel; 0 where that is more than
// its share of a CU's. In fp32 the small parameters of a deep policy do not fit
// beside the ring: one share takes up to 4 blocks of CartPole and 2 of VoxelNav
// and VoxelNav16, two shares 8, and 7 of VoxelNav16.
template <typename Env, int PREC, int HS>
size_t collect_lane_bytes(uint32_t layers) {
    using CL = CollectLane<Env, PREC, HS>;
    const size_t lds = (size_t)lane_lds<PREC, CL::HC, HS>(layers, CL::WIN, CL::IO).total * 4;
    return lds > 163840 / LaneShape<HS>::WG ? 0 : lds;
}

template <typename Env, int PREC, int HS>
bool launch_collect_lane_as(const mg_collect_args* a, hipStream_t st) {
    using Sh = LaneShape<HS>;
    if constexpr (CollectLane<Env, PREC, HS>::OK) {
        const size_t lds = collect_lane_bytes<Env, PREC, HS>(a->policy.layers);
        if (!a->policy.frag_fwd32_bf || lds == 0) return false;
        hipLaunchKernelGGL((collect_lane_kernel<Env, PREC, HS>), dim3((a->n + Sh::TILE - 1) / Sh::TILE), dim3(kLaneNT),
                           lds, st, *a);
        return true;
    } else {
        return false;
    }
}

// Runs the collect on collect_lane_kernel where that is the faster, for heads of
// up to 16 columns. With 128 envs a workgroup (one share) a step takes the time
// of one workgroup's stages up to 32768 envs, one per CU, and 1.15 PFLOP/s of
// binary16 products from 65536 (what the library's 8192^3 binary16 product
// reaches here); at 16384 half the CUs have none, so there two shares take 64
// envs a workgroup. ms a collect of 32 steps, CartPole, fp32, the tiles below (to
// 12288 envs the 16-row tiles on pairs) / two shares / one: 0.83 / 1.06 / 1.32 at
// 8192 envs, 1.22 / 1.10 / 1.37 at 12288, 2.30 / 1.14 / 1.38 at 16384, 3.26 /
// 2.08 / 1.43 at 24576, 8.44 / 4.18 / 2.86 at 65536. VoxelNav16, 16 steps: 0.83 /
// 0.75 / 0.98 at 8192, 1.34 / 0.80 / 1.02 at 16384. bf16, 0.56 / 0.62 / 0.62 at
// 16384, 0.71 / 1.20 / 0.63 at 20480, 0.87 / 1.21 / 0.68 at 32768: one share only.
// An env of more than 32 observation floats spends its step on computing them
// (VoxelNav's 32 ray marches), which the tiles spread over more threads, until
// the grid is full: 16 steps, tiles / one share, fp32 2.37 / 3.16 at 16384 and
// 4.09 / 3.32 at 32768; bf16 2.34 / 2.93 at 32768, and 8 steps of 65536 2.48 /
// 1.92. A policy too deep for the LDS (collect_lane_bytes) runs on the tiles.
// Small networks stay on the tiles where those fill the GPU evenly (8192 envs are
// one 32-row workgroup per CU, 16384 two, 32768 two of 64 rows) and the products
// are too few to pay for the observations' slower way. us a collect of 8 steps,
// tiles / lanes: VoxelNav16 at 8192 149 / 180 (1 block of 128), 275 / 288 (2 of
// 256), 353 / 356 (2 of 384), 433 / 404 (2 of 512), but 402 / 289 (2 of 256) at
// 8256; 1 of 128 at 8256 181 / 182 (one step 44 / 50), at 12288 199 / 193, at 16384
// 189 / 198; 4 steps of VoxelNav at 32768 817 / 889 (1 of 128), 891 / 900 (1 of
// 256). Heads of more than 8 columns likewise at 8192: 16 columns, 2 of 512, 215 /
// 223 for 3 steps and 463 / 414 for 8.
template <typename Env, int PREC>
bool launch_collect_lane(const mg_collect_args* a, hipStream_t st) {
    constexpr bool F32 = PREC == MG_PRECISION_FP32;
    const bool least = a->policy.layers * a->policy.hidden <= 128u;
    if constexpr (Env::OBS_DIM > 32) {
        if (a->n < (F32 ? (least ? 32769u : 32768u) : 65536u)) return false;
    }
    if (a->n > 16384u) return launch_collect_lane_as<Env, PREC, 1>(a, st);
    if constexpr (F32) {
        if (Env::OBS_DIM > 16 && least) return false;
        const bool even = a->policy.hidden >= 512u && Env::ACT_DIM + 1 <= 8;
        return a->n >= (even ? 8192u : 8193u) && launch_collect_lane_as<Env, PREC, 2>(a, st);
    } else {
        return false;
    }
}

template <typename Env, bool BF16>
int launch_collect_tiles(const mg_collect_args* a) {
    hipStream_t st = static_cast<hipStream_t>(a->stream);
    if (launch_collect_pair<Env>(a, st)) return (int)hipGetLastError();
    if (launch_collect_lane<Env, BF16 ? MG_PRECISION_BF16 : MG_PRECISION_FP32>(a, st)) return (int)hipGetLastError();
    // 64-row tiles reuse each weight fragment across the most rows; they need
    // n / 64 >= 512 workgroups (2 per CU) to fill the chip. Smaller runs use
    // 32-row, then 16-row tiles for more workgroups.
    if (a->n >= 64u * 512u)
        launch_collect_m<Env, 64, BF16>(a, st);
    else if (a->n >= 32u * 256u)
        launch_collect_m<Env, 32, BF16>(a, st);
    else
        launch_collect_m<Env, 16, BF16>(a, st);
    return (int)hipGetLastError();
}

template <typename Env>
int launch_collect(const mg_collect_args* a) {
    if (!a || a->n == 0 || a->n % 64 != 0 || a->horizon == 0) return MG_ERR_INVALID;
    if (a->policy.obs_dim != Env::OBS_DIM || a->policy.act_dim != Env::ACT_DIM ||
        a->policy.embed != (uint32_t)kEmbed || a->policy.hidden % kChunk != 0 || a->policy.layers == 0 ||
        a->policy.layers > MG_MAX_LAYERS)
        return MG_ERR_INVALID;
    if (a->policy.precision == MG_PRECISION_BF16 && (!a->policy.frag_fwd32_bf || !a->policy.frag_fwd16_bf))
        return MG_ERR_INVALID;
    return a->policy.precision == MG_PRECISION_BF16 ? launch_collect_tiles<Env, true>(a)
                                                      : launch_collect_tiles<Env, false>(a);
}

}  // namespace dev
}  // namespace mg
