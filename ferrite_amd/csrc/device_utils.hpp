// Device-side helpers shared by several translation units.
#pragma once
#include <hip/hip_runtime.h>

#include "numerics.hpp"

namespace fe {

// Activation scales are kept in the order the MFMA scale operand wants them: the e8m0 byte of the 32-wide k
// block b (k step kt = b/4, quarter g = b%4) sits at byte scale_pos(b) of its row, so that lane (column, g)
// reads the four k steps kt4*4 .. kt4*4+3 of its quarter as one dword at 16*kt4 + 4*g and selects the step
// with op_sel.  Rows are scale_pitch(K) bytes long.
__host__ __device__ __forceinline__ int scale_pos(int b) {
    const int kt = b >> 2, g = b & 3;
    return (kt >> 2) * 16 + g * 4 + (kt & 3);
}
__host__ __device__ __forceinline__ int scale_pitch(int K) { return ((K / 128 + 3) / 4) * 16; }

// Four floats to four packed e4m3 codes (byte i = value i) with the hardware converter (round to nearest even),
// made to agree with e4m3_encode(): magnitudes are clamped to 448 first, and the reference's subnormal rule
// (quant.rs:98-124: |x| in [7.5, 8) * 2^-9 encodes as 7, not as the smallest normal) is applied by moving such
// values onto 7 * 2^-9 before the conversion.  Anything that is not <= 448 in magnitude, NaN included, becomes
// +-448 as in e4m3_encode().
__device__ __forceinline__ float e4m3_prepare(float x) {
    const float ax = fabsf(x);
    x = (ax >= 0x1.ep-7f && ax < 0x1p-6f) ? copysignf(0x1.cp-7f, x) : x;
    return ax <= 448.0f ? x : copysignf(448.0f, x);
}
__device__ __forceinline__ uint32_t e4m3_encode4_hw(float a, float b, float c, float d) {
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(e4m3_prepare(a), e4m3_prepare(b), 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(e4m3_prepare(c), e4m3_prepare(d), w, true);
    return (uint32_t)w;
}

// The same for finite values of magnitude <= 448 (a block divided by its own scale): below 2^-6 the step is 2^-9, and
// a value held to +-7 * 2^-9 rounds to the code that the rule asks for.
__device__ __forceinline__ float e4m3_prepare_finite(float x) {
    const float small = __builtin_amdgcn_fmed3f(x, -0x1.cp-7f, 0x1.cp-7f);
    return fabsf(x) < 0x1p-6f ? small : x;
}
__device__ __forceinline__ uint32_t e4m3_encode4_finite(float a, float b, float c, float d) {
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(e4m3_prepare_finite(a), e4m3_prepare_finite(b), 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(e4m3_prepare_finite(c), e4m3_prepare_finite(d), w, true);
    return (uint32_t)w;
}

// Blocks whose largest magnitude lies below this are the finite ones.  From 248 * 2^120 on, the midpoint of the codes 240 and
// 256, code times scale is 2^128: the first term's product is infinite, and so is what it leaves over.
constexpr float E4M3_FINITE_AMAX = 0x1.fp127f;

// What four codes leave over of the values they were made from, in a finite block: v - decode(code) * scale.  The product is
// exact (four significant bits times a power of two, below 2^128), so one fused operation rounds as the subtraction alone does.
__device__ __forceinline__ void e4m3_residual4(uint32_t codes, float scale, float* v) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)codes, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)codes, true);
    v[0] = fmaf(-lo[0], scale, v[0]);
    v[1] = fmaf(-lo[1], scale, v[1]);
    v[2] = fmaf(-hi[0], scale, v[2]);
    v[3] = fmaf(-hi[1], scale, v[3]);
}

// Larger magnitude, NaN if either is (fmaxf would drop it).
__device__ __forceinline__ float amax_nan(float amax, float x) { return __builtin_elementwise_maximum(amax, fabsf(x)); }

// Clamped SwiGLU (cpu.rs:192-201) for the MFMA mode, whose results are rounded to e4m3 right afterwards: the
// hardware exponential and reciprocal (a few ulp) instead of the bit-exact expf and division of swiglu_ref().
__device__ __forceinline__ float swiglu_fast(float g, float u, float limit) {
    // compare-and-select like swiglu_ref (cpu.rs:192-201), not fminf / fmaxf: those return the non-NaN operand and
    // would turn a NaN accumulator into +-limit
    const float gi = g > limit ? limit : g;
    const float ui = u < -limit ? -limit : (u > limit ? limit : u);
    return gi * __builtin_amdgcn_rcpf(1.0f + __expf(-gi)) * ui;
}

// The same for limit >= 0: NaN-propagating minimum and maximum are the two selects.
__device__ __forceinline__ float swiglu_fast_min(float g, float u, float limit) {
    const float gi = __builtin_elementwise_minimum(g, limit);
    const float ui = __builtin_elementwise_maximum(__builtin_elementwise_minimum(u, limit), -limit);
    return gi * __builtin_amdgcn_rcpf(1.0f + __expf(-gi)) * ui;
}

// 32 consecutive f32 / bf16 values (32- / 16-byte aligned) into registers.
template <typename XT>
__device__ __forceinline__ void load_block32(const XT* __restrict__ src, float (&v)[32]) {
    if constexpr (sizeof(XT) == 4) {
        const float4* p = reinterpret_cast<const float4*>(src);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float4 t = p[i];
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
    } else {
        const uint4* p = reinterpret_cast<const uint4*>(src);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint4 t = p[i];
            uint32_t wds[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[8 * i + 2 * j] = u2f(wds[j] << 16);          // bf16 -> f32 is exact
                v[8 * i + 2 * j + 1] = u2f(wds[j] & 0xffff0000u);
            }
        }
    }
}

// act_quant_fp8 of one block of 32 values held in registers (crates/ferrite-models/src/dsv41/quant.rs:190-214,
// power-of-two scale): 32 e4m3 codes to q (32-byte aligned) and the e8m0 scale byte as the return value.
// kResidual: v is replaced by what the codes leave over, v - decode(code) * scale (one f32 multiply by a power of
// two and one f32 subtraction per value), the input of the second term of a two-term quantisation.
template <bool kResidual>
__device__ __forceinline__ uint32_t encode_block32(float (&v)[32], uint8_t* __restrict__ q) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) amax = amax_nan(amax, v[i]);
    uint32_t out[8], sb;
    if (amax < E4M3_FINITE_AMAX) {
        sb = block_scale_e8m0(amax);
        const float inv = u2f((254u - sb) << 23);   // 2^(127 - sb): exact reciprocal of the power-of-two scale
        const float sc = u2f(sb << 23);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            out[i] = e4m3_encode4_finite(v[4 * i] * inv, v[4 * i + 1] * inv, v[4 * i + 2] * inv, v[4 * i + 3] * inv);
            if constexpr (kResidual) e4m3_residual4(out[i], sc, &v[4 * i]);
        }
    } else {   // NaN or infinities in the block, or in what it leaves over
        amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(v[i]));
        sb = block_scale_e8m0(amax);
        const float inv = u2f((254u - sb) << 23);
        const float sc = u2f(sb << 23);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            out[i] = e4m3_encode4_hw(v[4 * i] * inv, v[4 * i + 1] * inv, v[4 * i + 2] * inv, v[4 * i + 3] * inv);
            if constexpr (kResidual) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[4 * i + j] = fadd(v[4 * i + j], -fmul(e4m3_decode((out[i] >> (8 * j)) & 0xffu), sc));
            }
        }
    }
    uint4* o = reinterpret_cast<uint4*>(q);
    o[0] = make_uint4(out[0], out[1], out[2], out[3]);
    o[1] = make_uint4(out[4], out[5], out[6], out[7]);
    return sb;
}

// act_quant_fp8 of one block of 32 consecutive values in memory.
template <typename XT>
__device__ __forceinline__ uint32_t quant_block32(const XT* __restrict__ src, uint8_t* __restrict__ q) {
    float v[32];
    load_block32(src, v);
    return encode_block32<false>(v, q);
}

// Two-term quantisation of one block: x ~ decode(q1) * 2^(s1-127) + decode(q2) * 2^(s2-127), where the second
// term is act_quant_fp8 of the residual of the first.  Returns s1 | s2 << 8.
template <typename XT>
__device__ __forceinline__ uint32_t quant_block32_x2(const XT* __restrict__ src, uint8_t* __restrict__ q1,
                                                     uint8_t* __restrict__ q2) {
    float v[32];
    load_block32(src, v);
    const uint32_t s1 = encode_block32<true>(v, q1);
    const uint32_t s2 = encode_block32<false>(v, q2);
    return s1 | (s2 << 8);
}

// Block b (of bpr per row) of the layer's input, codes row-major, scales in operand order.
template <typename XT>
__device__ __forceinline__ void quant_block_operand_order(const XT* __restrict__ x, long b, int bpr, uint8_t* __restrict__ q,
                                                          uint8_t* __restrict__ scale, uint8_t* __restrict__ q2,
                                                          uint8_t* __restrict__ scale2) {
    const size_t at = (size_t)(b / bpr) * scale_pitch(bpr * 32) + scale_pos((int)(b % bpr));
    if (q2) {
        const uint32_t sb = quant_block32_x2(x + b * 32, q + b * 32, q2 + b * 32);
        scale[at] = (uint8_t)(sb & 0xffu);
        scale2[at] = (uint8_t)(sb >> 8);
    } else {
        scale[at] = (uint8_t)quant_block32(x + b * 32, q + b * 32);
    }
}

// The left-to-right f32 sum (separately rounded adds, the reference's rmsnorm order: cpu.rs:124-143) of the n4 float4 at
// s4 in LDS, continued from ss.  Every lane reads the same addresses and holds the same running sum.  For short rows.
// Straight-line pieces of eight batches (256 values): a batch of eight 16-byte reads is in flight while the 32
// dependent adds of the batch before it run, and nothing is in flight at the end of a piece.  With the two
// register buffers carried around a loop instead, the compiler copied one buffer into the other every iteration and
// waited for every outstanding read at the top of a batch: 15 us for 4096 values against 10 us this way.
constexpr int SUMSQ_SHORT = 384;   // float4; beyond that sumsq_walk is sooner through
__device__ __forceinline__ float sumsq_piece(const float4* p, float ss) {
    constexpr int NB = 8;
    float4 r[2][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[0][j] = p[j];
#pragma unroll
    for (int g = 0; g < NB; ++g) {
        if (g + 1 < NB) {
#pragma unroll
            for (int j = 0; j < 8; ++j) r[(g + 1) & 1][j] = p[(g + 1) * 8 + j];
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC87F);   // lgkmcnt <= 8: everything but the batch just issued
        } else {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC07F);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float4 q = r[g & 1][j];
            ss = fadd(ss, q.x);
            ss = fadd(ss, q.y);
            ss = fadd(ss, q.z);
            ss = fadd(ss, q.w);
        }
        // pins the batch's adds in front of the next batch's reads (the optimiser otherwise hoists all 64 reads of
        // the piece to its top, 256 registers) and the reads behind it
        asm volatile("" : "+v"(ss) : : "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    return ss;
}

__device__ __forceinline__ float sumsq_chain(const float4* s4, int n4, float ss) {
    const int pieces = n4 >> 6;
    for (int i = 0; i < pieces; ++i) ss = sumsq_piece(s4 + i * 64, ss);
    for (int j = pieces * 64; j < n4; ++j) {
        const float4 q = s4[j];
        ss = fadd(ss, q.x);
        ss = fadd(ss, q.y);
        ss = fadd(ss, q.z);
        ss = fadd(ss, q.w);
    }
    return ss;
}

// A wave's inclusive scan: of sums, or of steps (see sumsq_walk), where a lane's step is taken behind those before it.
// row_shr 1, 2, 4, 8 within rows of 16; lane 15 of rows 0, 2 to rows 1, 3; lane 31 to rows 2 and 3.  Lanes without a
// source get 0, the step that changes nothing.
#define FE_WAVE_SCAN(STEP) \
    STEP(0x111, 0xf, true) STEP(0x112, 0xf, true) STEP(0x114, 0xf, true) STEP(0x118, 0xf, true) STEP(0x142, 0xa, false) STEP(0x143, 0xc, false)
__device__ __forceinline__ int wave_prefix(int v) {
#define FE_STEP(CTRL, ROWS, BOUND) v += __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, BOUND);
    FE_WAVE_SCAN(FE_STEP)
#undef FE_STEP
    return v;
}
__device__ __forceinline__ void wave_prefix_steps(int& even, int& odd) {
#define FE_STEP(CTRL, ROWS, BOUND)                                                                                             \
    {                                                                                                                          \
        const int e = __builtin_amdgcn_update_dpp(0, even, CTRL, ROWS, 0xf, BOUND);                                             \
        const int o = __builtin_amdgcn_update_dpp(0, odd, CTRL, ROWS, 0xf, BOUND);                                              \
        const int ne = e + ((e & 1) ? odd : even), no = o + ((o & 1) ? even : odd);                                            \
        even = ne;                                                                                                             \
        odd = no;                                                                                                              \
    }
    FE_WAVE_SCAN(FE_STEP)
#undef FE_STEP
}
#undef FE_WAVE_SCAN

// The same sum for long rows, all values >= +0 or NaN and ss >= 0; called by a whole wave.
// The chain is serial, but most of it can be worked out in parallel with the same bits.  While the running sum s stays
// within one binade it is M ulp with M in [2^23, 2^24), and adding q rounds to M + rint(q / ulp), whatever M is, unless
// q / ulp lies halfway between two integers (a tie): then the even neighbour of the exact sum is taken, which depends on
// M's parity.  So a lane takes 16 consecutive values of a chunk of 1024 and adds their integers; a prefix sum over the
// lanes says up to which lane s stays in its binade.  What does not fit - the first 128 values and sums below 2^-100, the
// 16 values in which s passes a power of two - is walked value by value: every lane adds its own 16 to s, and the result
// of the lane whose turn it is counts.  So are lanes with a tie while they are few; where they are many (rows of values
// that were rounded to bf16 or fp8) every lane works out the step that its values make from an even M and from an odd
// one, and the scan composes steps.  Zeros are passed over; a chunk that has been left ten times is walked to its end.
//
// us of rmsnorm, 192 rows           2048: normal bf16    4096: normal bf16 zeros     7168: normal bf16
//   chain alone                           8.0    8.0           14.3   14.2   14.4          23.7   23.8
//   without steps, zeros walked           8.5   27.9           10.7   31.4   26.0          13.5   80.2
//   this way                              8.3    8.4           11.0   10.7    3.9          13.4   15.0
// At 1024 values the chain takes 5.0 us, this way 6.2 to 7.3; at 8192 rows of 2048 45 and 37.  With steps from 3 / 5 / 9 / 13
// tied lanes on (one run): 4096 bf16 10.8 / 11.5 / 12.7 / 13.4, 7168 normal 14.6 / 14.0 / 13.9 / 13.8.
constexpr int SUMSQ_TIES = 4;
__device__ __forceinline__ float sumsq_walk(const float4* s4, int n4, float ss) {
    const int lane = threadIdx.x & 63;
    uint32_t sb = (uint32_t)__builtin_amdgcn_readfirstlane((int)f2u(ss));
#pragma unroll 1
    for (int base = 0; base < n4; base += 256) {
        const float4* p = s4 + base + lane * 4;
        float4 v[4];
        if (base + 256 <= n4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = p[i];
        } else {   // values past the end are +0: adding them changes nothing
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (base + lane * 4 + i < n4) v[i] = p[i];
            }
        }
        const float q[16] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w,
                             v[2].x, v[2].y, v[2].z, v[2].w, v[3].x, v[3].y, v[3].z, v[3].w};
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) bits |= f2u(q[i]);
        unsigned long long todo = __ballot(bits != 0);   // lanes that are not in s yet; zeros need not be
        int ex_of = -1, left = 0;
        int even = 0, odd = 0;   // the lane's step in ulp of ex_of; 2^24, past any binade's end, where it has none
        bool ties = false;
#pragma unroll 1
        while (todo != 0) {
            int first = __builtin_ctzll(todo);
            const int ex = (int)(sb >> 23);
            int walk = 8;   // lanes that are walked next
            if (ex >= 27 && ex < 255) {
                if (ex != ex_of) {
                    const float scale = u2f((uint32_t)(277 - ex) << 23);   // 1 / ulp
                    float total = 0.0f, off = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        const float t0 = q[i] * scale, t1 = q[i + 1] * scale, r0 = rintf(t0), r1 = rintf(t1);
                        off = fmaxf(off, fmaxf(fabsf(t0 - r0), fabsf(t1 - r1)));
                        total += r0 + r1;   // exact up to 2^24
                    }
                    const bool none = !(total <= 16777216.0f);   // NaN too
                    const bool tied = !none && off == 0.5f;
                    ties = __builtin_popcountll(__ballot(tied) & todo) > SUMSQ_TIES;
                    if (ties) {
                        float again = scale;          // the quotients are worked out a second time: kept, they take
                        asm("" : "+v"(again));        // 32 registers, which cost the rows' kernels a block per CU
                        even = 0;
                        odd = 1;
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const float t = q[i] * again, r = rintf(t), f = fabsf(t - r) == 0.5f ? t : r;
                            const int twice = (int)(f + f), whole = twice >> 1, half = twice & 1;
                            even += whole;
                            even += even & half;   // a half that follows an odd number makes it even, else it is dropped
                            odd += whole;
                            odd += odd & half;
                        }
                        odd -= 1;
                        if (none) even = odd = 1 << 24;
                    } else {
                        even = (none || tied) ? 1 << 24 : (int)total;
                    }
                    ex_of = ex;
                }
                const int m = (int)((sb & 0x7fffffu) | 0x800000u);
                int at = lane >= first ? even : 0;
                if (ties) {
                    int from_odd = lane >= first ? odd : 0;
                    wave_prefix_steps(at, from_odd);
                    if (m & 1) at = from_odd;
                } else {
                    at = wave_prefix(at);
                }
                at += m;   // where s stands behind this lane
                const unsigned long long stop = __ballot(at > 0xffffff);
                if (stop == 0) {
                    sb = ((uint32_t)ex << 23) | ((uint32_t)__builtin_amdgcn_readlane(at, 63) & 0x7fffffu);
                    break;
                }
                first = __builtin_ctzll(stop);
                if (first > 0) sb = ((uint32_t)ex << 23) | ((uint32_t)__builtin_amdgcn_readlane(at, first - 1) & 0x7fffffu);
                walk = ++left > 10 ? 64 : 1;
            }
#pragma unroll 1
            do {
                float t = u2f(sb);
#pragma unroll
                for (int i = 0; i < 16; ++i) t = fadd(t, q[i]);
                sb = (uint32_t)__builtin_amdgcn_readlane((int)f2u(t), first++);
            } while (--walk > 0 && first < 64);
            todo = first < 64 ? todo >> first << first : 0;
        }
    }
    return u2f(sb);
}

}  // namespace fe
