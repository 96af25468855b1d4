// The hidden-unit split of a 16-row tile (policy_split.h) on pairs of binary16
// values: the fp32 row pass of a PPO minibatch with both block GEMMs on
// v_mfma_f32_16x16x32_f16, three products per fp32 product (policy_lane.h has
// the split, its accuracy and its range).
//
// The hidden units go to the waves in groups of 32: wave w owns groups w, w +
// 8, ... and runs them without synchronising. Of a group, two 16-unit strips:
// strip s holds units 8 (r / 4) + 4 s + r % 4, so that the two results of the
// first GEMM, V^T strips of 16 units x 16 rows (the weights are the A operand,
// the block input X the B operand), leave each lane with 8 consecutive units
// of its row, which are one A operand (K = 32) of the second GEMM. That adds
// V W1 to the wave's private 16 x 128 partial of the block output; the partials
// are added in LDS once per block, as in policy_split.h.
//
// Weights: 4 bytes each, as the fp32 copies, hi and lo halves in operand order.
// Role 0 (first GEMM, K = 128 embed columns): group p at 8192 p halves, then
// (strip, k-group of 32, plane) runs of 64 lanes x 8 (1 KB): lane 16 q + r
// holds unit r of the strip, k = 8 q .. + 7. Role 1 (second GEMM, K = the
// group's 32 units): group p at 8192 p, then (16-column strip, plane) runs:
// lane 16 q + c holds column c, units 8 q .. + 7. One group of one role is 16
// KB of consecutive memory.
#pragma once
#include "policy_lane.h"
#include "policy_split.h"

namespace mg {
namespace dev {

constexpr int kPairW = 8;          // waves
constexpr uint32_t kPairGroup = 32;  // hidden units of a group
constexpr int kPairLd = kEmbed + 8;  // halves per LDS row of a plane
constexpr int kPairRowTarget = 11;   // |x| < 2^11 in a scaled block input row: |V| < 128 2^11 2^13 < 2^32
constexpr int kPairTiles = 128;      // most 32 x 32 tiles of a block matrix

// The scales of the planes, after frag_fwd16_bf's 2 count halves. A matrix's
// exponent follows its largest finite magnitude, which an Adam step changes:
// Adam writes its planes with `next`, records it in `cur` and leaves each tile's
// largest finite magnitude in tilemax; the next row pass makes `next` from those and
// from what one more Adam step can add. |m| <= 7.27 sqrt(v) for Adam's moments
// (Cauchy-Schwarz over their weights, beta 0.9 and 0.999, both from 0) and the
// bias corrections only shrink that ratio, so a step moves no weight by more
// than 7.27 lr. All of it stays on the device, in stream order, so a captured
// train step replays correctly. tilemax also gives the collects' exponents
// after a train call (derive_blocks_kernel).
constexpr float kAdamReach = 7.3f;
struct PairScale {
    int cur[2 * MG_MAX_LAYERS];  // per block matrix (up, down per layer): the planes' exponent
    int next[2 * MG_MAX_LAYERS];
    float tilemax[2 * MG_MAX_LAYERS][kPairTiles];
};
__host__ __device__ __forceinline__ size_t pair_elems(uint32_t count) {
    return 2 * (size_t)count + sizeof(PairScale) / 2;
}
__host__ __device__ __forceinline__ PairScale* pair_scale(uint16_t* planes, uint32_t count) {
    return reinterpret_cast<PairScale*>(planes + 2 * (size_t)count);
}
// The exponent of a matrix whose largest magnitude is m.
__device__ __forceinline__ int pair_exp(float m) { return split_min(kMatTarget - pow2_above(m), 40); }

// A wave's position in the forward's blocks and then the backward's (FWD_ONLY:
// the forward's, again and again).
struct PairPos {
    int bwd, l, k;
};
template <bool FWD_ONLY = false>
struct PairSeq {
    const uint16_t* fwd;  // frag_fwd16_bf + 2 float_group: up in role 0, down in role 1
    const uint16_t* bwd;  // frag_bwd16_bf + 2 float_group: up in role 1, down in role 0
    int L, nk, wave, rot;  // nk: this wave's groups per block
    uint32_t EH;           // 128 hidden
    __device__ __forceinline__ int group(const PairPos& p) const {
        const int k = p.k + rot;
        return wave + kPairW * (k < nk ? k : k - nk);
    }
    __device__ __forceinline__ const uint16_t* role(const PairPos& p, int r) const {
        const size_t m = 2 * (size_t)(2 * p.l + (p.bwd ? 1 - r : r)) * EH;
        return (p.bwd ? bwd : fwd) + m + 8192u * (size_t)group(p);
    }
    __device__ __forceinline__ PairPos next(PairPos p) const {
        if (++p.k < nk) return p;
        p.k = 0;
        if (!p.bwd) {
            if (++p.l < L) return p;
            if (FWD_ONLY) return PairPos{0, 0, 0};
            p.bwd = 1;
            p.l = L - 1;
            return p;
        }
        if (--p.l >= 0) return p;
        return PairPos{1, 0, nk - 1};  // past the end: the last group again
    }
};

__device__ __forceinline__ f32x4 mfma16x16x32h(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The operand registers of both roles, each refilled for the same role of the
// next group right after its MFMAs.
struct PairStream {
    f16x8 w0[2][4][2];  // strip, k-group, plane
    f16x8 w1[8][2];     // column strip, plane

    __device__ __forceinline__ static f16x8 load(const uint16_t* p, uint32_t run) {
        return __builtin_bit_cast(f16x8, buffer_load16(p, 16 * (threadIdx.x & 63), 1024 * run));
    }
    __device__ __forceinline__ void start(const uint16_t* a, const uint16_t* b) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int p = 0; p < 2; ++p) w0[s][g][p] = load(a, 2 * (4 * s + g) + p);
#pragma unroll
        for (int ct = 0; ct < 8; ++ct)
#pragma unroll
            for (int p = 0; p < 2; ++p) w1[ct][p] = load(b, 2 * ct + p);
    }
    // acc[s] += strip s . xb: lane l register r = unit 8 (l / 16) + 4 s + r of
    // the group, row l % 16
    __device__ __forceinline__ void gemm0(f32x4 (&acc)[2], const f16x8 (&xb)[4][2], const uint16_t* nx) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int s = 0; s < 2; ++s) acc[s] = mfma16x16x32h(w0[s][g][0], xb[g][1], acc[s]);
#pragma unroll
            for (int s = 0; s < 2; ++s) acc[s] = mfma16x16x32h(w0[s][g][1], xb[g][0], acc[s]);
#pragma unroll
            for (int s = 0; s < 2; ++s) acc[s] = mfma16x16x32h(w0[s][g][0], xb[g][0], acc[s]);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int p = 0; p < 2; ++p) w0[s][g][p] = load(nx, 2 * (4 * s + g) + p);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // hp[ct] += v W1: hp[ct] lane l register r = row 4 (l / 16) + r, column 16
    // ct + l % 16
    __device__ __forceinline__ void gemm1(f32x4 (&hp)[8], const f16x8 (&v)[2], const uint16_t* nx) {
#pragma unroll
        for (int c2 = 0; c2 < 8; c2 += 2) {
#pragma unroll
            for (int ct = c2; ct < c2 + 2; ++ct) hp[ct] = mfma16x16x32h(v[0], w1[ct][1], hp[ct]);
#pragma unroll
            for (int ct = c2; ct < c2 + 2; ++ct) hp[ct] = mfma16x16x32h(v[1], w1[ct][0], hp[ct]);
#pragma unroll
            for (int ct = c2; ct < c2 + 2; ++ct) hp[ct] = mfma16x16x32h(v[0], w1[ct][0], hp[ct]);
#pragma unroll
            for (int ct = c2; ct < c2 + 2; ++ct)
#pragma unroll
                for (int p = 0; p < 2; ++p) w1[ct][p] = load(nx, 2 * ct + p);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// The block input's planes in LDS, and what takes a row's first product back
// to its own units.
struct alignas(16) PairInput {
    uint16_t x[2][kSplitRows * kPairLd];
    int unit[kSplitRows];  // exponent of the row's V: its own plus the first matrix's
};

// A row's block input (NV float4s per thread, TPR threads) to planes, scaled
// by the row's own power of two; returns its exponent. An infinite element is in
// the low plane alone, as an infinite weight (LaneOps::pack_weights).
template <int TPR, int NV>
__device__ __forceinline__ int pair_store_input(PairInput& in, const RowVec<NV>& x, int row, int lk, int e0) {
    static_assert(NV == 1, "four columns per thread");
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) m = fmaxf(m, fabsf(x[c]));
    m = group_max<TPR>(m);
    const int e = split_min(kPairRowTarget - pow2_above(m), 40);
    const float f = pow2i(e < -126 ? -126 : e);
    f16x2 h0, l0, h1, l1;
    split_f16_scaled(x[0], x[1], opaque_v(f), h0, l0);
    split_f16_scaled(x[2], x[3], opaque_v(f), h1, l1);
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    f16x4 hi = {h0[0], h0[1], h1[0], h1[1]}, lo = {l0[0], l0[1], l1[0], l1[1]};
    // one branch in the chain from LN to the products: the selects alone took 0.1 us
    if (__any(m == __builtin_huge_valf())) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (__builtin_isinf((float)hi[c])) lo[c] = hi[c], hi[c] = (_Float16)0.0f;
    }
    *reinterpret_cast<f16x4*>(&in.x[0][row * kPairLd + 4 * lk]) = hi;
    *reinterpret_cast<f16x4*>(&in.x[1][row * kPairLd + 4 * lk]) = lo;
    if (lk == 0) in.unit[row] = e + e0;
    return e;
}
__device__ __forceinline__ void pair_load_input(const PairInput& in, f16x8 (&xb)[4][2]) {
    const int lane = threadIdx.x & 63, at = (lane & 15) * kPairLd + 8 * (lane >> 4);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int p = 0; p < 2; ++p) xb[g][p] = *reinterpret_cast<const f16x8*>(&in.x[p][at + 32 * g]);
}

// Eight values times 2^kHiddenExp as planes.
__device__ __forceinline__ void pair_pack(const float (&x)[8], f16x8 (&p)[2]) {
    const float f = opaque(1.0f / (float)(1 << -kHiddenExp));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f16x2 hi, lo;
        split_f16_scaled(x[2 * j], x[2 * j + 1], f, hi, lo);
        p[0][2 * j] = hi[0], p[0][2 * j + 1] = hi[1];
        p[1][2 * j] = lo[0], p[1][2 * j + 1] = lo[1];
    }
}

// LDS of pair_forward: the block input, the waves' partials of a block output
// (scratch for split_row_head between the forwards) and the planes' exponents.
struct alignas(16) PairFwdSmem {
    PairInput in;
    float red[kPairW][kSplitRows * kLds];
    int exps[2 * MG_MAX_LAYERS];
};

// A wave's weight stream, carried from one forward to the next: the last
// group's refills are the next forward's first operands.
struct PairFwd {
    PairStream wst;
    PairSeq<true> seq;
    PairPos pos;
    __device__ __forceinline__ void start(const mg_policy_view& pv) {
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int nk = ((int)(pv.hidden / kPairGroup) - wave + kPairW - 1) / kPairW;
        const int rot = nk > 0 ? (wave + (int)(blockIdx.x >> 3)) % nk : 0;
        seq = PairSeq<true>{pv.frag_fwd16_bf + 2 * (size_t)pv.float_group, nullptr, (int)pv.layers, nk, wave, rot,
                            (uint32_t)kEmbed * pv.hidden};
        pos = PairPos{0, 0, 0};
        if (nk > 0) wst.start(seq.role(pos, 0), seq.role(pos, 1));
    }
};

// split_forward16 (policy_split.h) with the block GEMMs on pairs: obs staged in
// obsL ([16][O], LDS) -> head in headL ([16][HD], LDS), ending with a barrier.
// OC: O where it is known at compile time, else 0.
template <int OC>
__device__ __forceinline__ void pair_forward(const mg_policy_view& pv, const SmallParams& sp, PairFwdSmem& sm,
                                             PairFwd& F, const float* obsL, int O, float* headL, int HD) {
    constexpr int TPR = 64 * kPairW / kSplitRows;  // 32 threads per row, four columns each
    constexpr int kUnroll = OC > 0 ? OC : 4;
    const int tid = threadIdx.x, wave = F.seq.wave, On = OC > 0 ? OC : O;
    const int row = tid / TPR, lk = tid % TPR, c0 = 4 * lk, NL = (int)pv.layers;
    RowVec<1> h = rv_load<1>(sp.bin + c0);  // model/input.metal:11-27
#pragma unroll kUnroll
    for (int k = 0; k < On; ++k) {
        const float ok = obsL[row * On + k];
        const RowVec<1> w = rv_load<1>(sp.win + k * kEmbed + c0);
#pragma unroll
        for (int c = 0; c < 4; ++c) h[c] = __builtin_fmaf(ok, w[c], h[c]);
    }
    RowVec<1> x, xn;
    float sd;
    for (int l = 0; l < NL; ++l) {
        sk_layernorm<TPR>(h, sp.ln + l * 2 * kEmbed, sp.ln + l * 2 * kEmbed + kEmbed, c0, x, xn, sd);
        const int unit = pair_store_input<TPR>(sm.in, x, row, lk, 0) + sm.exps[2 * l] + kHiddenExp + sm.exps[2 * l + 1];
        __syncthreads();  // X complete; every wave is past its reads of red
        f16x8 xb[4][2];
        pair_load_input(sm.in, xb);
        f32x4 hp[8];
#pragma unroll
        for (int ct = 0; ct < 8; ++ct) hp[ct] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = 0; k < F.seq.nk; ++k) {  // model/mlp.metal:18-86 for one of this wave's groups
            const PairPos nx = F.seq.next(F.pos);
            f32x4 v[2] = {};
            F.wst.gemm0(v, xb, F.seq.role(nx, 0));
            float t[8];
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r) t[4 * s + r] = v[s][r];
            f16x8 vb[2];
            LaneOps<MG_PRECISION_FP32>::pack_hidden(t, vb);
            F.wst.gemm1(hp, vb, F.seq.role(nx, 1));
            F.pos = nx;
        }
        RowVec<1> d = sk_reduce_buf<kPairW, 1>(&sm.red[0][0], hp, wave, row, c0);
#pragma unroll
        for (int c = 0; c < 4; ++c) h[c] += __builtin_ldexpf(d[c], -unit);  // model/elementwise.metal:4-13
    }
    sk_layernorm<TPR>(h, sp.ln + NL * 2 * kEmbed, sp.ln + NL * 2 * kEmbed + kEmbed, c0, x, xn, sd);
    for (int j = 0; j < HD; ++j) {  // model/linear.metal:17-37
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc = __builtin_fmaf(x[c], sp.wh[(c0 + c) * HD + j], acc);
        acc = group_sum<TPR>(acc);
        if (lk == 0) headL[row * HD + j] = acc;
    }
    __syncthreads();
}

// One row's head as split_forward16 computes it, bit for bit, by the whole
// workgroup of 8 waves (policy_lane.h says what for): V one unit per thread,
// then wave w adds its units' products into its partial, two columns per lane.
// Orders: an MFMA's k = 16 g + 4 q + j over g, j, q; the second GEMM's units 4
// q + j of a strip over j, q, the wave's chunks from its rotation; a row's sums
// over four columns, then 32 threads as group_sum does; the partials in wave
// order. block: the tile's workgroup index there. lds: scratch of (hidden + 8 *
// 128 + 2 * 128 + 32) floats, dead otherwise. Starts and ends with a barrier.
template <int OC, int HD>
__device__ __forceinline__ void split_row_head(const mg_policy_view& pv, const SmallParams& sp, const float* obs,
                                               uint32_t block, float* lds, float* head) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = (int)pv.hidden, NC = H / kChunk;
    float* vs = lds;               // [hidden]
    float* part = lds + H;         // [8][128]
    float* hs = part + 8 * kEmbed;  // [128] residual stream
    float* xs = hs + kEmbed;       // [128] LN output
    float* rs = xs + kEmbed;       // [32]
    __syncthreads();
    if (tid < kEmbed) {
        float h = sp.bin[tid];
        for (int k = 0; k < OC; ++k) h += obs[k] * sp.win[k * kEmbed + tid];
        hs[tid] = h;
    }
    // sum over the row of f(column): four columns per thread in order, then the
    // 32 threads' pairing of group_sum<32>; every thread computes it
    auto row_sum = [&](auto f) {
        __syncthreads();
        if (tid < 32) {
            float s = f(4 * tid);
#pragma unroll
            for (int c = 1; c < 4; ++c) s += f(4 * tid + c);
            rs[tid] = s;
        }
        __syncthreads();
        float q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = (rs[4 * i] + rs[4 * i + 1]) + (rs[4 * i + 2] + rs[4 * i + 3]);
        return ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
    };
    auto layernorm = [&](int l) {
        const float mean = row_sum([&](int c) { return hs[c]; }) / (float)kEmbed;
        const float q = row_sum([&](int c) {
            const float d = hs[c] - mean;
            return d * d;
        });
        const float rstd = 1.0f / sqrtf(q / (float)kEmbed + 1e-5f);
        if (tid < kEmbed) {
            const float xn = (hs[tid] - mean) * rstd;
            xs[tid] = sp.ln[2 * kEmbed * l + tid] * xn + sp.ln[2 * kEmbed * l + kEmbed + tid];
        }
        __syncthreads();
    };
    for (int l = 0; l < (int)pv.layers; ++l) {
        layernorm(l);
        for (int u = tid; u < H; u += 64 * kPairW) {
            const float* up = pv.params + pv.off_up[l] + u;
            float v = 0.0f;
#pragma unroll 1
            for (int g = 0; g < 8; ++g) {
                float w[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) w[k] = up[(size_t)(16 * g + k) * H];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) v = __builtin_fmaf(w[4 * q + j], xs[16 * g + 4 * q + j], v);
            }
            vs[u] = v > 0.0f ? v : 0.0f;
        }
        __syncthreads();
        float p[2] = {0.0f, 0.0f};
        const int rot = (wave + (int)(block >> 3)) % NC;
#pragma unroll 1
        for (int k = 0; k < NC; ++k) {
            const int c = k + rot < NC ? k + rot : k + rot - NC;
            const int u0 = kChunk * c + 16 * wave;
            const float* dn = pv.params + pv.off_down[l] + (size_t)u0 * kEmbed + lane;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        p[i] = __builtin_fmaf(vs[u0 + 4 * q + j], dn[(4 * q + j) * kEmbed + 64 * i], p[i]);
        }
        part[wave * kEmbed + lane] = p[0], part[wave * kEmbed + 64 + lane] = p[1];
        __syncthreads();
        if (tid < kEmbed) {
            float s = part[tid];
            for (int w = 1; w < kPairW; ++w) s += part[w * kEmbed + tid];
            hs[tid] = hs[tid] + s;
        }
    }
    layernorm((int)pv.layers);
    for (int j = 0; j < HD; ++j) {
        const float s = row_sum([&](int c) { return xs[c] * sp.wh[c * HD + j]; });
        if (tid == 0) head[j] = s;
    }
    __syncthreads();
}

// Where element (unit u of a matrix's hidden index, column k of the embed) of a
// block matrix sits in the role-0 or role-1 order, in halves of the hi plane
// (lo: 512 later).
__host__ __device__ constexpr uint32_t pair_index0(uint32_t u, uint32_t k) {
    return (u / 32) * 8192u + 2u * ((((u >> 2) & 1u) * 4u + k / 32) * 512u) + (((k % 32) >> 3) * 16u +
           4u * ((u % 32) >> 3) + (u & 3u)) * 8u + (k & 7u);
}
__host__ __device__ constexpr uint32_t pair_index1(uint32_t u, uint32_t c) {
    return (u / 32) * 8192u + 2u * ((c / 16) * 512u) + (((u % 32) >> 3) * 16u + (c % 16)) * 8u + (u & 7u);
}

}  // namespace dev
}  // namespace mg
