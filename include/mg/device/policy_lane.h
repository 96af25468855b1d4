// The policy forward with a row in a pair of lanes: every wave owns 32 rows,
// and lanes n and n + 32 hold row n's residual stream, LN output and hidden
// activations in registers from the embed to the head.
//
// Each product is computed transposed, D = W^T X^T on 32 x 32 x 16 matrix
// instructions with the weights as the A operand and the activations as the B
// operand, so a result register already sits in the lane that needs it as the
// next product's B operand: no activation goes through LDS, LayerNorm reduces
// over 64 registers and one lane swap, and the head is a plain dot product per
// lane. What the waves share is the weights: a stage of one 32-unit hidden
// tile (its Up^T strip and its Down^T columns) is staged in LDS once per
// workgroup of 128 rows, double-buffered, with one barrier per stage, the
// stage after next already in flight in registers. A stage is bound by the
// matrix instructions (48 of 32 cycles in fp32) where a SIMD has two waves; with
// one, everything a wave does between them counts, so each operand is read one
// step ahead of its product and the next stage's LDS writes and loads are spread
// over the first eight: 1.47 -> 1.12 us a stage at one wave per SIMD (16384
// rows), a step of 65536 envs 93 -> 86 us.
//
// Where 128 rows a workgroup leave CUs idle the four waves are two row groups of
// two waves each (shares): a wave does half of the hidden units of its 32 rows,
// the two sums meet in LDS after a block (LaneEx), and LN, embed and head are
// done by both. A step of 16384 envs (hidden 512, 2 blocks) 42 -> 34 us.
//
// Precision MG_PRECISION_FP32: each fp32 operand as two binary16 halves, x =
// hi + lo (22 bits and the sign of lo), and hi hi + hi lo + lo hi accumulated
// in fp32: three v_mfma_f32_32x32x16_f16 in the place of eight
// v_mfma_f32_32x32x2_f32, which take 5.3 times as long. Against 64 bits this is
// closer than the fp32 instructions (relative 2-norm of a product of normal
// rows and uniform weights: 1.43e-7 against 2.04e-7 over 128 terms, 2.59e-7
// against 4.06e-7 over 512), since a sum of 16 products is rounded once where
// the fp32 chain rounds after every two. A split into three bfloat16 needs six
// products for 1.63e-7 and 3.39e-7, and is worse than fp32 on rectified
// inputs (3.26e-7 against 2.87e-7).
// binary16's range is met by powers of two, which change no bit of a result:
// the weights are stored scaled (SplitScale, from each matrix's largest
// magnitude), gamma and beta are staged scaled so that no LN output row is
// longer than 2^15 (a normalised row of 128 is at most sqrt(128) long), hence
// |V| <= 2^15 sqrt(128) 2^13 < 2^31.6 whatever the observation, which 2^-16 takes
// into range, and the residual stream is kept in the units of the block's
// product. Weights down to 2^-15 of their matrix's largest and LN outputs and
// hidden units down to 2^-16 of their bounds keep all 22 bits; below that
// their error is 2^-38 of the largest.
// Infinities come out as in fp32: a weight that is not finite is in its low
// plane alone (pack_weights), so it meets the other operand's high half only,
// and a hidden unit at infinity, which pack_hidden's clamp holds at 2^32, leaves
// binary16's range again in the conversion.
//
// MG_PRECISION_BF16: one bfloat16 plane, as policy_bf16.h.
#pragma once
#include "policy_bf16.h"

namespace mg {
namespace dev {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kLaneRows = 32;  // rows of a wave

constexpr int kLaneWaves = 4;  // waves of a workgroup
constexpr int kLaneNT = 64 * kLaneWaves;
// HS waves share the hidden units of 32 rows: wave h RG + g is share h of row
// group g of RG = 4 / HS.
template <int HS>
struct LaneShape {
    static constexpr int RG = kLaneWaves / HS, TILE = kLaneRows * RG;
    static constexpr int WG = HS == 1 ? 2 : 1;  // workgroups per CU: the ring is 64 HS KB
};
constexpr int kLaneTile = LaneShape<1>::TILE;

// The binary16 planes of an fp32 policy (mg_policy_view.frag_fwd32_bf with
// MG_PRECISION_FP32): up^T and down^T in the order of the bf16 copies, each
// element times its matrix's power of two (split_exp), the hi halves at the
// arena offsets and the lo halves `count` elements later; after both,
// SplitScale: per matrix the least e with every finite |element| < 2^e.
struct SplitScale {
    int up[MG_MAX_LAYERS];
    int down[MG_MAX_LAYERS];
};
__host__ __device__ __forceinline__ size_t split_elems(uint32_t count) {
    return 2 * (size_t)count + sizeof(SplitScale) / 2;
}
__host__ __device__ __forceinline__ const SplitScale* split_scale(const uint16_t* planes, uint32_t count) {
    return reinterpret_cast<const SplitScale*>(planes + 2 * (size_t)count);
}

// 2^e for -126 <= e <= 127.
__device__ __forceinline__ float pow2i(int e) { return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23); }
// The least e with m < 2^e, for a finite m >= 0 (0 and denormals: -126).
__device__ __forceinline__ int pow2_above(float m) {
    return (int)((__builtin_bit_cast(uint32_t, m) >> 23) & 0xFFu) - 126;
}
// The exponents of a block's powers of two: |up| and |down| < 2^13 after them,
// an LN output row shorter than 2^15, hidden units times 2^-16. Small matrices
// are scaled up only so far that the residual stream, in units of the block's
// product, stays under 2^60 of itself; a down matrix may be as small as its up
// matrix is large.
constexpr int kMatTarget = 13, kRowTarget = 15, kHiddenExp = -16;
__host__ __device__ __forceinline__ int split_min(int a, int b) { return a < b ? a : b; }
__host__ __device__ __forceinline__ int split_exp_up(int up) { return split_min(kMatTarget - up, 49); }
__host__ __device__ __forceinline__ int split_exp_down(int up, int down) {
    return split_min(split_min(kMatTarget - down, 49 - split_exp_up(up)), 126);
}

// x = hi + lo in binary16, both rounded to nearest even; the remainder x - hi
// is exact in fp32. minus1 is -1 in a scalar register, opaque to the compiler,
// which then takes the half straight into v_fma_mix_f32 instead of converting
// it and subtracting: two instructions per element, three fewer.
__device__ __forceinline__ void split_f16(float x0, float x1, float minus1, f16x2& hi, f16x2& lo) {
    hi = f16x2{(_Float16)x0, (_Float16)x1};
    lo = f16x2{(_Float16)__builtin_fmaf((float)hi[0], minus1, x0), (_Float16)__builtin_fmaf((float)hi[1], minus1, x1)};
}
// The same of x f, f a power of two (opaque like minus1): the product is part
// of the conversion (v_fma_mixlo_f16 / v_fma_mixhi_f16) and of the remainder.
__device__ __forceinline__ void split_f16_scaled(float x0, float x1, float f, f16x2& hi, f16x2& lo) {
    hi = f16x2{(_Float16)__builtin_fmaf(x0, f, 0.0f), (_Float16)__builtin_fmaf(x1, f, 0.0f)};
    lo = f16x2{(_Float16)__builtin_fmaf(x0, f, -(float)hi[0]), (_Float16)__builtin_fmaf(x1, f, -(float)hi[1])};
}
// v in a scalar register, unknown to the compiler.
__device__ __forceinline__ float opaque(float v) {
    asm("" : "+s"(v));
    return v;
}

// The same in a vector register.
__device__ __forceinline__ float opaque_v(float v) {
    asm("" : "+v"(v));
    return v;
}

template <int PREC>
struct LaneOps;
template <>
struct LaneOps<MG_PRECISION_FP32> {
    using V = f16x8;
    static constexpr int PL = 2;  // planes
    __device__ static __forceinline__ void pack(const float (&x)[8], V (&p)[2]) {
        const float m1 = opaque(-1.0f);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f16x2 hi, lo;
            split_f16(x[2 * j], x[2 * j + 1], m1, hi, lo);
            p[0][2 * j] = hi[0], p[0][2 * j + 1] = hi[1];
            p[1][2 * j] = lo[0], p[1][2 * j + 1] = lo[1];
        }
    }
    // The planes of weights. inf = inf + (inf - inf) would make every product
    // NaN, and the relu a 0 of that; as 0 + inf it is infinity times the high
    // half of the other operand, with the fp32 product's sign (and NaN times 0).
    __device__ static __forceinline__ void pack_weights(const float (&x)[8], V (&p)[2]) {
        pack(x, p);
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(x[j]));
        if (m < 65520.0f) return;  // a NaN stays in both
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (!(fabsf(x[j]) < 65520.0f)) p[0][j] = (_Float16)0.0f, p[1][j] = (_Float16)x[j];
    }
    // relu of hidden units, times 2^kHiddenExp: 2^-32 takes them under 1, where
    // the multiplication's own clamp is the relu (0 for NaN, as x > 0 ? x : 0),
    // and the conversion takes them up again (from the clamp's 1, an infinite
    // unit, to 2^16: infinity in binary16)
    __device__ static __forceinline__ void pack_hidden(const float (&x)[8], V (&p)[2]) {
        const float f = opaque((float)(1 << (32 + kHiddenExp)));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f16x2 hi, lo;
            const float x0 = __builtin_amdgcn_fmed3f(x[2 * j] * 0x1p-32f, 0.0f, 1.0f);
            const float x1 = __builtin_amdgcn_fmed3f(x[2 * j + 1] * 0x1p-32f, 0.0f, 1.0f);
            split_f16_scaled(x0, x1, f, hi, lo);
            p[0][2 * j] = hi[0], p[0][2 * j + 1] = hi[1];
            p[1][2 * j] = lo[0], p[1][2 * j + 1] = lo[1];
        }
    }
    // the small products first: their sum is rounded at its own size where the
    // accumulator starts at zero
    __device__ static __forceinline__ f32x16 mma(const V (&a)[2], const V (&b)[2], f32x16 c) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], b[1], c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], b[0], c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], b[0], c, 0, 0, 0);
    }
};
template <>
struct LaneOps<MG_PRECISION_BF16> {
    using V = bf16x8;
    static constexpr int PL = 1;
    __device__ static __forceinline__ void pack(const float (&x)[8], V (&p)[1]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[0][j] = (__bf16)x[j];
    }
    __device__ static __forceinline__ void pack_hidden(const float (&x)[8], V (&p)[1]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[0][j] = (__bf16)fmaxf(x[j], 0.0f);
    }
    __device__ static __forceinline__ f32x16 mma(const V (&a)[1], const V (&b)[1], f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], c, 0, 0, 0);
    }
};

// Row m of the A operand that lands where the D layout's register order is a
// run of consecutive rows per lane: D register 8 b + j of half-wave q is row
// 16 b + 8 (j / 4) + 4 q + j % 4 of the product; with A's rows permuted by pi
// it is row 16 b + 8 q + j of the matrix, the K order of the weight copies.
__device__ __forceinline__ int lane_pi(int m) { return (m & 0x13) | ((m & 4) << 1) | ((m & 8) >> 1); }

// The weights of one forward as a cycle of stages (layer l, hidden tile ht of
// each share) through two LDS buffers of 32 (fp32) or 16 KB (bf16) per share.
template <int PREC, int HS>
struct LaneRing {
    using Ops = LaneOps<PREC>;
    static constexpr int PL = Ops::PL;
    static constexpr int T4 = 1024 * PL;   // float4s of a hidden tile
    static constexpr int F4 = T4 * HS;     // of a stage
    static constexpr int NL = F4 / kLaneNT;  // loads per thread
    const uint16_t* planes;
    f32x4* buf;  // LDS, 2 F4
    uint32_t count, group, EH, H;
    int tiles, layers;  // hidden tiles per layer and share
    int nl, nt;         // the stage in flight
    f32x4 st[NL];

    // Load k of stage (nl, nt) into st[k]: of each share's tile (h tiles + nt)
    // up^T's strip of 32 hidden units (8 KB a plane, contiguous) and the two
    // k-groups of down^T's four strips (2 KB each).
    __device__ __forceinline__ void load(int k) {
        const int tid = threadIdx.x, h = k / (4 * PL), r = k % (4 * PL), p = r / 2 % PL, u = r % 2;
        const uint32_t t = (uint32_t)(nt + h * tiles);
        const uint32_t up = group + 2u * (uint32_t)nl * EH + 4096u * t;
        const uint32_t dn = group + (2u * (uint32_t)nl + 1u) * EH + 1024u * t;
        if (r < 2 * PL) {
            st[k] = buffer_load16(planes, 16u * tid, 2u * (up + p * count + 2048u * u));
        } else {
            const uint32_t vd = (uint32_t)(tid >> 7) * 64u * H + 16u * (uint32_t)(tid & 127);
            st[k] = buffer_load16(planes, vd, 2u * (dn + p * count + 64u * u * H));
        }
    }
    __device__ __forceinline__ void store(int b, int k) { buf[b * F4 + kLaneNT * k + threadIdx.x] = st[k]; }
    __device__ __forceinline__ void next() {
        if (++nt == tiles) {
            nt = 0;
            if (++nl == layers) nl = 0;
        }
    }
    // Stage 0 in buffer 0 and stage 1 in flight; the caller's next barrier
    // makes buffer 0 readable.
    __device__ __forceinline__ void start(const mg_policy_view& pv, f32x4* lds) {
        planes = pv.frag_fwd32_bf, buf = lds;
        count = pv.count, group = pv.float_group, H = pv.hidden, EH = (uint32_t)kEmbed * H;
        tiles = (int)H / (32 * HS), layers = (int)pv.layers;
        nl = nt = 0;
#pragma unroll
        for (int k = 0; k < NL; ++k) load(k);
        next();
#pragma unroll
        for (int k = 0; k < NL; ++k) store(0, k);
#pragma unroll
        for (int k = 0; k < NL; ++k) load(k);
        next();
    }
    // Beside the products of buffer b's stage, part i of 8: the stage in flight
    // goes to the other buffer, which every wave finished reading before the
    // last barrier, and the one after it leaves; then finish().
    __device__ __forceinline__ void pass(int b, int i) {
#pragma unroll
        for (int k = i; k < NL; k += 8) {
            store(b ^ 1, k);
            load(k);
        }
    }
    __device__ __forceinline__ void finish() {
        next();
        barrier();
    }
    __device__ static __forceinline__ void barrier() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
};

// Small parameters in LDS. ln: gamma, beta per LN (the blocks' scaled by
// xs[l]); wh: W_head, HC columns a row, zero past the head's width.
template <int HC>
struct LaneParams {
    const float* ln;
    const float* bin;
    const float* wh;
    const float* win;  // LDS, or the arena
    const float* scale;  // per block: the exponent (int) of the residual stream's unit, then the unit's inverse
};

// The exponent of the power of two for an LN's gamma and beta, from their 128
// values each: a wave-wide computation. poison: an element is infinite and none
// is NaN, so that fp32 arithmetic has infinite inputs of every row (a NaN makes
// every hidden unit of the block NaN, and the relu a 0 of it, in both).
__device__ __forceinline__ int lane_row_exp(const float* gamma, const float* beta, bool& poison) {
    const int lane = threadIdx.x & 63;
    const float g0 = gamma[lane], g1 = gamma[lane + 64], b0 = beta[lane], b1 = beta[lane + 64];
    const float g = group_max<64>(fmaxf(fabsf(g0), fabsf(g1)));
    const float b = group_max<64>(fmaxf(fabsf(b0), fabsf(b1)));
    // sqrt(128) (max |gamma| + max |beta|), rounded up, times 2^-8 against overflow
    const float len = 11.4f * (0x1p-8f * g + 0x1p-8f * b);
    poison = len == __builtin_huge_valf() && !__any(g0 != g0 || g1 != g1 || b0 != b0 || b1 != b1);
    return split_min(kRowTarget - 8 - pow2_above(len), 28);
}

// Row sums over the lane pair.
__device__ __forceinline__ float lane_sum(float v) {
    float lo, hi;
    lane_pair<32>(v, lo, hi);
    return lo + hi;
}

// a in lanes 0 .. 31 and, in lanes 32 .. 63, the b of the lane 32 below. Every
// lane of the wave must be active.
__device__ __forceinline__ float lane_give(float a, float b) {
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return a;
}

// The residual stream of a wave's 32 rows: register 8 b + j of tile mt in lane
// (n, q) is column 32 mt + 16 b + 8 q + j of row n.
struct LaneRows {
    f32x16 h[4];
};

// Mean and reciprocal deviation of the rows (model/layernorm.metal:10-71); the
// stream times inv, a power of two, is the residual stream, so h inv - mean is
// rounded once.
__device__ __forceinline__ void lane_stats(const LaneRows& R, float inv, float& mean, float& rstd) {
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = R.h[0][j] + R.h[0][8 + j];
#pragma unroll
    for (int i = 2; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] += R.h[i >> 1][8 * (i & 1) + j];
    mean = lane_sum(tree_sum(s)) * ((1.0f / (float)kEmbed) * inv);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float d = __builtin_fmaf(R.h[0][j], inv, -mean);
        s[j] = d * d;
    }
#pragma unroll
    for (int i = 1; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float d = __builtin_fmaf(R.h[i >> 1][8 * (i & 1) + j], inv, -mean);
            s[j] = __builtin_fmaf(d, d, s[j]);
        }
    const float var = lane_sum(tree_sum(s)) * (1.0f / (float)kEmbed);
    rstd = 1.0f / sqrtf(var + 1e-5f);
}

// Eight consecutive floats of LDS.
__device__ __forceinline__ void lane_read8(const float* p, float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = a[j], v[4 + j] = b[j];
}

// What passes between the two shares of a row group, in ring buffer 1, which is
// free from the last stage of a block to the first of the next: N of a wave's
// tiles a time, 4 KB each.
template <int PREC>
struct LaneEx {
    using Ring = LaneRing<PREC, 2>;
    static constexpr int N = PREC == MG_PRECISION_FP32 ? 4 : 2;
    static_assert(LaneShape<2>::RG * 2 * 256 * N <= Ring::F4, "fits the buffer");
    __device__ static __forceinline__ f32x4* at(const Ring& ring, int rg) { return ring.buf + Ring::F4 + 512 * N * rg; }
    // The two shares' sums, in both. Starts and ends where every wave has
    // finished with the memory.
    __device__ static __forceinline__ void join(LaneRows& R, f32x4* ex, int half, int lane) {
        f32x4 *mine = ex + 256 * N * half + lane, *other = ex + 256 * N * (half ^ 1) + lane;
#pragma unroll
        for (int m0 = 0; m0 < 4; m0 += N) {
#pragma unroll
            for (int m = 0; m < N; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const f32x16 h = R.h[m0 + m];
                    mine[64 * (4 * m + r)] = f32x4{h[4 * r], h[4 * r + 1], h[4 * r + 2], h[4 * r + 3]};
                }
            Ring::barrier();
#pragma unroll
            for (int m = 0; m < N; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const f32x4 v = other[64 * (4 * m + r)];
#pragma unroll
                    for (int j = 0; j < 4; ++j) R.h[m0 + m][4 * r + j] += v[j];
                    if (r == 3) __builtin_amdgcn_sched_barrier(0);
                }
            Ring::barrier();
        }
    }
};

// model/ppo.h:575-626 for the wave's 32 rows. ob[s]: this lane's embed
// operand, observation float 2 s + q of row n (0 past the last). The head (HC
// columns, both lanes of a row) goes to hv, of share 0 where there are two.
// O <= OC: the observation width (OC itself where it is known at compile
// time); WINL: W_in is in LDS.
template <int PREC, int HC, int OC, bool WINL, int HS>
__device__ __forceinline__ void lane_forward(const mg_policy_view& pv, const LaneParams<HC>& P,
                                             LaneRing<PREC, HS>& ring, int O, const float (&ob)[(OC + 1) / 2],
                                             float (&hv)[HC]) {
    using Ring = LaneRing<PREC, HS>;
    constexpr int NOB = (OC + 1) / 2;
    using Ops = LaneOps<PREC>;
    using V = typename Ops::V;
    constexpr int PL = Ops::PL;
    const int lane = threadIdx.x & 63, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int half = HS > 1 ? wave / LaneShape<HS>::RG : 0;
    const int slot = lane_pi(lane & 31) + 32 * q + half * Ring::T4;
    LaneRows R;
    // model/input.metal:11-27 on v_mfma_f32_32x32x2_f32
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float v[8];
            lane_read8(P.bin + 32 * mt + 16 * b + 8 * q, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) R.h[mt][8 * b + j] = v[j];
        }
    const int wl = q * kEmbed + lane_pi(lane & 31);  // this lane's element of W_in's rows 2 s, 2 s + 1
#pragma unroll
    for (int s = 0; s < NOB; ++s) {
        if (2 * s >= O) break;
        // where row 2 s is the last the second operand is row 2 s again, times 0
        const bool pad = 2 * s + 1 >= O;
        const int at = pad ? wl - q * kEmbed : wl;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            float w;
            if constexpr (WINL)
                w = P.win[at + 2 * s * kEmbed + 32 * mt];
            else
                w = buffer_load4(P.win, 4u * (uint32_t)at, 4u * (2 * s * kEmbed + 32 * mt));
            if (pad) w = q ? 0.0f : w;
            R.h[mt] = mfma32x32x2(w, ob[s], R.h[mt]);
        }
        // at most 16 weights in flight: all 60 of VoxelNav16's spill
        if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (HS > 1) Ring::barrier();  // the observations' LDS is read
    float inv = 1.0f;
    float near = 1.0f;  // fp32: 0 for a row too large for the units of a block, NaN for one that is not finite
    int exp = 0;        // of the stream's unit
    for (uint32_t l = 0; l < pv.layers; ++l) {
        float mean, rstd;
        lane_stats(R, inv, mean, rstd);
        V xb[8][PL];
        const float* gm = P.ln + 2 * kEmbed * l + 8 * q;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            float g[8], b[8], x[8];
            lane_read8(gm + 16 * s, g);
            lane_read8(gm + kEmbed + 16 * s, b);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = __builtin_fmaf(g[j], __builtin_fmaf(R.h[s >> 1][8 * (s & 1) + j], inv, -mean) * rstd, b[j]);
            Ops::pack(x, xb[s]);
        }
        if constexpr (PREC == MG_PRECISION_FP32) {
            // the stream to this block's units (in share 0's sum). They hold rows
            // under 2^67; larger ones have a deviation of infinity, so LN gives
            // them beta, here and in all that follows: as it does a stream of 0.
            if (!(rstd > 0.0f && fabsf(mean) <= 0x1p66f)) near = 0.0f * rstd;
            const int e = __builtin_bit_cast(int, P.scale[2 * l]);
            const int by = half || near == 0.0f ? -1000 : e - exp;
            exp = e;
            inv = P.scale[2 * l + 1] * near;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int r = 0; r < 16; ++r) R.h[mt][r] = __builtin_ldexpf(R.h[mt][r], by);
        } else if constexpr (HS > 1) {
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int r = 0; r < 16; ++r) R.h[mt][r] = half ? 0.0f : R.h[mt][r];
        }
        for (int ht = 0; ht < ring.tiles; ++ht) {  // tiles is even: hidden is a multiple of 128
            const f32x4* w = ring.buf + (ht & 1) * Ring::F4 + slot;
            // model/mlp.metal:18-86: V^T = relu(Up^T x^T) for 32 units, then h^T += Down^T V^T
            f32x16 v = f32x16{};
            V a[2][PL];
            auto fetch = [&](int i) {  // operand i of 8 + 8
                const int at = i < 8 ? 64 * i : 512 * PL + 128 * (i & 3) + 64 * ((i - 8) >> 2);
#pragma unroll
                for (int p = 0; p < PL; ++p) a[i & 1][p] = __builtin_bit_cast(V, w[512 * p + at]);
            };
            fetch(0);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                fetch(s + 1);
                v = Ops::mma(a[s & 1], xb[s], v);
                ring.pass(ht & 1, s);
                __builtin_amdgcn_sched_barrier(0);  // or the loads, and their waits, are moved together
            }
            V vb[2][PL];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float t[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) t[j] = v[8 * b + j];
                Ops::pack_hidden(t, vb[b]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (i < 7) fetch(i + 9);
                R.h[i & 3] = Ops::mma(a[i & 1], vb[i >> 2], R.h[i & 3]);
            }
            ring.finish();
        }
        if constexpr (HS > 1) {
            LaneEx<PREC>::join(R, LaneEx<PREC>::at(ring, wave % LaneShape<HS>::RG), half, lane);
        }
    }
    float mean, rstd;
    lane_stats(R, inv, mean, rstd);
    const float* gm = P.ln + 2 * kEmbed * pv.layers + 8 * q;
    // model/linear.metal:17-37
#pragma unroll
    for (int j = 0; j < HC; ++j) hv[j] = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        float g[8], b[8];
        lane_read8(gm + 16 * s, g);
        lane_read8(gm + kEmbed + 16 * s, b);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = __builtin_fmaf(g[j], __builtin_fmaf(R.h[s >> 1][8 * (s & 1) + j], inv, -mean) * rstd, b[j]);
            const float* wr = P.wh + (16 * s + 8 * q + j) * HC;
#pragma unroll
            for (int c = 0; c < HC; c += 4) {
                const f32x4 wv = *reinterpret_cast<const f32x4*>(wr + c);
#pragma unroll
                for (int i = 0; i < 4; ++i) hv[c + i] = __builtin_fmaf(x, wv[i], hv[c + i]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < HC; ++j) hv[j] = lane_sum(hv[j]);
}

// ---- one row in the fp32 tiles' arithmetic --------------------------------------
// The split product's head differs from the fp32 tiles' (policy.h) in its last
// bits, so a draw that falls within rounding of an edge of the CDF could pick
// another action, and the env's rollout would go its own way from there. Such
// draws (edge <= kLaneEdge, one in 2^18 per edge) are decided by the row's
// head as the tiles compute it, bit for bit: a seeded fp32 collect of a
// categorical policy takes the same actions whichever kernel runs it, as long as
// the two heads' edges are that close. Of a policy whose logits have a standard
// deviation of 1 they are: the logits differ by at most 5.5e-6 over 2^21 rows,
// an edge by a quarter of that. That grows with the head's weights: at 20, 2 of
// 2^21 draws were decided otherwise. Gaussian and bfloat16 collects, and samples
// of a forward's head, follow their own kernel's rounding. One wave recomputes one row, weights from
// the arena, every sum in the tiles' order: an MFMA adds its k in order with
// one rounding each (v_mfma_f32_32x32x2_f32 equals the chain of FMAs, checked
// on 65536 sums of 128), the k of a group of 8 in the order 0, 4, 1, 5, 2, 6, 3,
// 7 (policy.h's K-order permutation), a row's LN and head sums as trees over
// CPT columns (32 in a 64-row tile, 16 in a 32-row tile), then over its threads.
constexpr float kLaneEdge = 0x1p-19f;
constexpr int kLaneRowLds = 2 * kEmbed + 16;  // floats of scratch per wave

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Sum over a row of 128 floats in LDS, f of each: CPT columns as a tree (or G
// at a time, in order), then the threads' sums pairwise. parts: 8 floats.
template <int CPT, int G, class F>
__device__ __forceinline__ float tile_row_sum(int lane, float* parts, F f) {
    constexpr int TPR = kEmbed / CPT;
    if (lane < TPR) {
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < CPT; g += G) {
            float t[G];
#pragma unroll
            for (int c = 0; c < G; ++c) t[c] = f(CPT * lane + g + c);
            const float s = tree_sum(t);
            acc = g == 0 ? s : acc + s;
        }
        parts[lane] = acc;
    }
    wave_lds_fence();
    float q = (parts[0] + parts[1]) + (parts[2] + parts[3]);
    if constexpr (TPR == 8) q = q + ((parts[4] + parts[5]) + (parts[6] + parts[7]));
    wave_lds_fence();
    return q;
}

template <int CPT, int O, int HD>
__device__ __forceinline__ void tile_row_head(const mg_policy_view& pv, const float* obs, float* lds, float* head) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // or every address below is formed, and spilled, before the rollout's loop
    float *xs = lds, *vs = lds + kEmbed, *parts = lds + 2 * kEmbed;
    const uint32_t H = pv.hidden;
    float h[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int c = lane + 64 * u;
        h[u] = pv.params[pv.off_in_b + c];
        for (int k = 0; k < O; ++k) h[u] = __builtin_fmaf(obs[k], pv.params[pv.off_in_w + k * kEmbed + c], h[u]);
    }
    const float* lnp = pv.params + pv.off_ln_gamma[0];
    // LN l of h into xs
    auto layernorm = [&](uint32_t l) {
        xs[lane] = h[0], xs[lane + 64] = h[1];
        wave_lds_fence();
        const float mean = tile_row_sum<CPT, CPT>(lane, parts, [&](int c) { return xs[c]; }) / (float)kEmbed;
        const float q = tile_row_sum<CPT, CPT>(lane, parts, [&](int c) {
            const float d = xs[c] - mean;
            return d * d;
        });
        const float rstd = 1.0f / sqrtf(q / (float)kEmbed + 1e-5f);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = lane + 64 * u;
            const float xn = (h[u] - mean) * rstd;
            xs[c] = lnp[2 * kEmbed * l + c] * xn + lnp[2 * kEmbed * l + kEmbed + c];
        }
        wave_lds_fence();
    };
    // acc[u] += sum over k < 128 of a[k] w[k ld + 64 u], k in the tiles' order
    auto chain = [&](float (&acc)[2], const float* a, const float* w, uint32_t ld) {
#pragma unroll 2
        for (int g = 0; g < kEmbed; g += 8) {
            float x[8], wv[8][2];
            lane_read8(a + g, x);
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int u = 0; u < 2; ++u) wv[k][u] = w[(size_t)(g + k) * ld + 64 * u];
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int kk = 4 * (k & 1) + (k >> 1);
                    acc[u] = __builtin_fmaf(x[kk], wv[kk][u], acc[u]);
                }
        }
    };
    for (uint32_t l = 0; l < pv.layers; ++l) {
        layernorm(l);
        const float* up = pv.params + pv.off_up[l] + lane;
        const float* dn = pv.params + pv.off_down[l] + lane;
        for (uint32_t c = 0; c < H; c += kChunk) {
            float v[2] = {0.0f, 0.0f};
            chain(v, xs, up + c, H);
            vs[lane] = v[0] > 0.0f ? v[0] : 0.0f;
            vs[lane + 64] = v[1] > 0.0f ? v[1] : 0.0f;
            wave_lds_fence();
            chain(h, vs, dn + (size_t)c * kEmbed, kEmbed);
            wave_lds_fence();
        }
    }
    layernorm(pv.layers);
    const float* wh = pv.params + pv.off_head;
    constexpr int G = HD == 4 && CPT == 32 ? 16 : CPT;  // fwd_head_regs' column groups
    for (int j = 0; j < HD; ++j) {
        const float s = tile_row_sum<CPT, G>(lane, parts, [&](int c) { return xs[c] * wh[c * HD + j]; });
        if (lane == 0) head[j] = s;
    }
    wave_lds_fence();
}

// A workgroup's LDS, in floats: the ring, the small parameters (W_in where
// win), then io floats per row group.
struct LaneLds {
    uint32_t ln, bin, scale, wh, win, io, total;
};
template <int PREC, int HC, int HS>
__host__ __device__ __forceinline__ LaneLds lane_lds(uint32_t layers, uint32_t win, uint32_t io_per_wave) {
    LaneLds L;
    uint32_t o = 2u * LaneRing<PREC, HS>::F4 * 4u;
    L.ln = o, o += (layers + 1) * 2 * kEmbed;
    L.bin = o, o += kEmbed;
    L.scale = o, o += 2 * MG_MAX_LAYERS;
    L.wh = o, o += kEmbed * HC;
    L.win = o, o += win;
    L.io = o, o += LaneShape<HS>::RG * ((io_per_wave + 3u) & ~3u);
    L.total = o;
    return L;
}

// Stages the small parameters (the blocks' gamma and beta scaled) and starts
// the ring. Ends with a barrier. win: floats of W_in to stage (0: read from
// the arena).
template <int PREC, int HC, int HS>
__device__ __forceinline__ void lane_start(const mg_policy_view& pv, float* lds, const LaneLds& L, uint32_t win,
                                           LaneParams<HC>& P, LaneRing<PREC, HS>& ring) {
    const int tid = threadIdx.x;
    ring.start(pv, reinterpret_cast<f32x4*>(lds));
    const float* lnp = pv.params + pv.off_ln_gamma[0];
    const int nl = (int)pv.layers, HD = (int)pv.head_dim;
    for (int k = tid; k < kEmbed; k += kLaneNT) lds[L.bin + k] = pv.params[pv.off_in_b + k];
    for (int k = tid; k < kEmbed * HC; k += kLaneNT) {
        const int c = k / HC, j = k % HC;
        const float w = pv.params[pv.off_head + c * HD + (j < HD ? j : 0)];
        lds[L.wh + k] = j < HD ? w : 0.0f;
    }
    for (uint32_t k = tid; k < win; k += kLaneNT) lds[L.win + k] = pv.params[pv.off_in_w + k];
    for (int l = 0; l <= nl; ++l) {
        float xs = 1.0f;
        if constexpr (PREC == MG_PRECISION_FP32) {
            if (l < nl) {
                const SplitScale& ss = *split_scale(pv.frag_fwd32_bf, pv.count);
                bool poison;
                const int ex = lane_row_exp(lnp + 2 * kEmbed * l, lnp + 2 * kEmbed * l + kEmbed, poison);
                xs = pow2i(ex);
                // the unit of block l's product (at 2^-126 the products are past fp32's range)
                int e = ex + split_exp_up(ss.up[l]) + kHiddenExp + split_exp_down(ss.up[l], ss.down[l]);
                e = e < -126 ? -126 : e;
                // poison: an infinite input's planes are inf and NaN, which the relu would
                // turn into a block output of 0
                if (tid == 0)
                    lds[L.scale + 2 * l] = __builtin_bit_cast(float, e),
                    lds[L.scale + 2 * l + 1] = poison ? __builtin_nanf("") : pow2i(-e);
            }
        }
        if (tid < 2 * kEmbed) lds[L.ln + 2 * kEmbed * l + tid] = xs * lnp[2 * kEmbed * l + tid];
    }
    P.ln = lds + L.ln, P.bin = lds + L.bin, P.wh = lds + L.wh, P.scale = lds + L.scale;
    P.win = win ? lds + L.win : pv.params + pv.off_in_w;
    __syncthreads();
}

}  // namespace dev
}  // namespace mg
