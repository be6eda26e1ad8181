// MXFP4 -> f32 dequantisation and e4m3-per-32 activation quantisation.  Both are bit-exact restatements of
// crates/ferrite-models/src/dsv41/quant.rs (dequant_fp4_row32 :260-278, act_quant_fp8 :190-214) and are
// bound by HBM traffic: every thread moves 128-bit vectors.
#include "internal.hpp"
#include "device_utils.hpp"
#include "numerics.hpp"

namespace fe {

// One thread dequantises 32 columns of one row: 16 code bytes (one 128-bit load) and one scale byte in,
// 32 floats (eight 128-bit stores) out.
__global__ __launch_bounds__(256) void mxfp4_dequant_kernel(const uint8_t* __restrict__ w,
                                                            const uint8_t* __restrict__ scale, int64_t nblocks,
                                                            float* __restrict__ dst) {
    int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    uint4 c = *reinterpret_cast<const uint4*>(w + b * 16);
    float s = ue8m0_decode(scale[b]);
    uint32_t words[4] = {c.x, c.y, c.z, c.w};
    float4* o = reinterpret_cast<float4*>(dst + b * 32);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t v = words[q];
        float4 lo, hi;
        lo.x = e2m1_decode(v & 15u) * s;         lo.y = e2m1_decode((v >> 4) & 15u) * s;
        lo.z = e2m1_decode((v >> 8) & 15u) * s;  lo.w = e2m1_decode((v >> 12) & 15u) * s;
        hi.x = e2m1_decode((v >> 16) & 15u) * s; hi.y = e2m1_decode((v >> 20) & 15u) * s;
        hi.z = e2m1_decode((v >> 24) & 15u) * s; hi.w = e2m1_decode((v >> 28) & 15u) * s;
        o[2 * q] = lo;
        o[2 * q + 1] = hi;
    }
}

// One thread quantises one block of 32 consecutive values of a row; with q2 / scale2, a second term from the
// residual of the first (quant_block32_x2).  Scales are row-major (the layer's own quantisation writes them in operand
// order: quant_block_operand_order).
template <typename XT>
__global__ __launch_bounds__(256) void act_quant_kernel(const XT* __restrict__ x, int64_t nblocks,
                                                        uint8_t* __restrict__ q, uint8_t* __restrict__ scale,
                                                        uint8_t* __restrict__ q2, uint8_t* __restrict__ scale2) {
    int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    if (q2) {
        const uint32_t sb = quant_block32_x2(x + b * 32, q + b * 32, q2 + b * 32);
        scale[b] = (uint8_t)(sb & 0xffu);
        scale2[b] = (uint8_t)(sb >> 8);
    } else {
        scale[b] = (uint8_t)quant_block32(x + b * 32, q + b * 32);
    }
}

// Weights to MXFP4 per block of 32 consecutive values of a row (quant.rs:217-238 with the power-of-two scale of :190-198
// against the e2m1 maximum 6): 16 code bytes, low nibble = even column, and the e8m0 byte of the scale.  Nearest magnitude,
// a tie going to the smaller one (quant.rs:40-55 keeps the first candidate of a strictly-smaller search); the sign bit
// is set for negative quotients even when they round to zero.
// The scale's exponent is that of amax / 6 rounded up to a power of two, from the bits of amax: 6 = 1.5 * 2^2 (the rounded
// quotient of a mantissa next to 1.5 never reaches or leaves a power of two: 0.67 ulp above 1, 1.33 ulp below 2).
FE_HD uint32_t block_scale_fp4_e8m0(float amax) {
    const uint32_t bits = f2u(amax);                        // amax >= 0, not NaN
    if (bits >= 0x7f800000u) return 255u;
    const uint32_t e = (bits + 0x3fffffu) >> 23;
    return e < 3u ? 1u : e - 2u;
}
FE_HD uint32_t e2m1_encode(float x) {
    float a = fabsf(x);
    a = a > 6.0f ? 6.0f : a;
    const uint32_t m = (uint32_t)(a > 0.25f) + (uint32_t)(a > 0.75f) + (uint32_t)(a > 1.25f) + (uint32_t)(a > 1.75f) +
                       (uint32_t)(a > 2.5f) + (uint32_t)(a > 3.5f) + (uint32_t)(a > 5.0f);
    return m | (x < 0.0f ? 8u : 0u);
}

// Four neighbouring lanes share a block, eight values each, so that a wave's loads and stores are whole lines.  The hardware
// converts, rounding to nearest even, where the quotient by the power-of-two scale (an exact product) is finite: of the
// seven ties 0.75, 1.75 and 3.5 would go up, so a value with at most four significant bits is moved towards zero by an ulp
// or two first, which leaves the code of every one that is no tie as it is; adding zero drops the sign of a zero quotient.
// Bound by the launch and HBM at the sizes of an expert (4096 x 1536 bf16: 12.6 MB in, 3.3 MB out); with seven compares and
// a division per value and 64 bytes per thread it was 9.7 us of vector instructions, now 5.1.
template <typename XT>
__global__ __launch_bounds__(256) void mxfp4_quant_kernel(const XT* __restrict__ x, int64_t nblocks,
                                                          uint8_t* __restrict__ codes, uint8_t* __restrict__ scale) {
    const int64_t i8 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // eight values; a block's four lanes are all live or none is
    if (i8 >= nblocks * 4) return;
    float v[8];
    if constexpr (sizeof(XT) == 4) {
        const float4* p = reinterpret_cast<const float4*>(x + i8 * 8);
        const float4 t0 = p[0], t1 = p[1];
        v[0] = t0.x; v[1] = t0.y; v[2] = t0.z; v[3] = t0.w;
        v[4] = t1.x; v[5] = t1.y; v[6] = t1.z; v[7] = t1.w;
    } else {
        const uint4 t = *reinterpret_cast<const uint4*>(x + i8 * 8);
        const uint32_t wds[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[2 * j] = u2f(wds[j] << 16);
            v[2 * j + 1] = u2f(wds[j] & 0xffff0000u);
        }
    }
    // two maxima: NaN kept (is the block finite?) and NaN dropped (what the scale is made from)
    float nan_max = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) nan_max = amax_nan(nan_max, v[i]);
    auto quad = [](float a, auto pick) {
        const float b = pick(a, u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(a), 0xB1, 0xf, 0xf, false)));
        return pick(b, u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(b), 0x4E, 0xf, 0xf, false)));
    };
    float amax = quad(nan_max, [](float a, float b) { return amax_nan(a, b); });
    uint32_t out = 0, sb;
    if (amax < __builtin_inff()) {   // the same for the four lanes
        sb = block_scale_fp4_e8m0(amax);
        const float inv = u2f((254u - sb) << 23);
        float t[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float q = v[i] * inv;
            const float nudged = q * (1.0f - 0x1p-23f);
            q = (f2u(q) & 0xfffffu) == 0u ? nudged : q;
            t[i] = q + 0.0f;
        }
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, t[0], t[1], 1.0f, 0);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, t[2], t[3], 1.0f, 1);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, t[4], t[5], 1.0f, 2);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, t[6], t[7], 1.0f, 3);
    } else {
        amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float a = fabsf(v[i]);
            amax = a > amax ? a : amax;
        }
        amax = quad(amax, [](float a, float b) { return fmaxf(a, b); });
        sb = block_scale_fp4_e8m0(amax);
        const float sc = u2f(sb << 23);
#pragma unroll
        for (int i = 0; i < 8; ++i) out |= e2m1_encode(fdiv(v[i], sc)) << (4 * i);
    }
    *reinterpret_cast<uint32_t*>(codes + i8 * 4) = out;
    if ((threadIdx.x & 3) == 0) scale[i8 >> 2] = (uint8_t)sb;
}

int launch_act_quant(const void* x, int x_dtype, int64_t rows, int cols, uint8_t* q, uint8_t* scale, uint8_t* q2,
                     uint8_t* scale2, hipStream_t st) {
    if (rows < 0 || cols < 0 || cols % 32 != 0 || (q2 == nullptr) != (scale2 == nullptr)) return FERRITE_ERR_INVALID_ARG;
    int64_t nblocks = rows * (cols / 32);
    if (nblocks == 0) return FERRITE_OK;
    unsigned grid = (unsigned)((nblocks + 255) / 256);
    if (x_dtype == FERRITE_DT_F32)
        act_quant_kernel<float><<<grid, 256, 0, st>>>((const float*)x, nblocks, q, scale, q2, scale2);
    else if (x_dtype == FERRITE_DT_BF16)
        act_quant_kernel<uint16_t><<<grid, 256, 0, st>>>((const uint16_t*)x, nblocks, q, scale, q2, scale2);
    else
        return FERRITE_ERR_INVALID_ARG;
    return check_launch("act_quant");
}

}  // namespace fe

using namespace fe;

extern "C" int ferrite_mxfp4_dequant(const uint8_t* w, const uint8_t* scale, int64_t rows, int64_t cols, float* dst,
                                     ferrite_stream_t stream) {
    if (rows < 0 || cols < 0 || cols % 32 != 0) return FERRITE_ERR_INVALID_ARG;
    int64_t nblocks = rows * (cols / 32);
    if (nblocks == 0) return FERRITE_OK;
    if (!w || !scale || !dst) return FERRITE_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(w) & 15) || (reinterpret_cast<uintptr_t>(dst) & 15)) return FERRITE_DECLINED;
    mxfp4_dequant_kernel<<<(unsigned)((nblocks + 255) / 256), 256, 0, as_stream(stream)>>>(w, scale, nblocks, dst);
    return check_launch("mxfp4_dequant");
}

// Blocks of 32 values a launch: four threads each, and a launch holds fewer than 2^32 threads.
constexpr int64_t kMxQuantBlocks = int64_t(1) << 29;

extern "C" int ferrite_mxfp4_quant(const void* x, int x_dtype, int64_t rows, int64_t cols, uint8_t* codes,
                                   uint8_t* scale, ferrite_stream_t stream) {
    if (rows < 0 || cols < 0 || cols % 32 != 0) return FERRITE_ERR_INVALID_ARG;
    const int64_t nblocks = rows * (cols / 32);
    if (nblocks == 0) return FERRITE_OK;
    if (!x || !codes || !scale) return FERRITE_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(codes) & 15)) return FERRITE_DECLINED;
    if (x_dtype != FERRITE_DT_F32 && x_dtype != FERRITE_DT_BF16) return FERRITE_ERR_INVALID_ARG;
    for (int64_t b0 = 0; b0 < nblocks; b0 += kMxQuantBlocks) {
        const int64_t nb = nblocks - b0 < kMxQuantBlocks ? nblocks - b0 : kMxQuantBlocks;
        const unsigned grid = (unsigned)((nb * 4 + 255) / 256);
        if (x_dtype == FERRITE_DT_F32)
            mxfp4_quant_kernel<float><<<grid, 256, 0, as_stream(stream)>>>((const float*)x + b0 * 32, nb, codes + b0 * 16, scale + b0);
        else
            mxfp4_quant_kernel<uint16_t><<<grid, 256, 0, as_stream(stream)>>>((const uint16_t*)x + b0 * 32, nb, codes + b0 * 16, scale + b0);
        if (int rc = check_launch("mxfp4_quant")) return rc;
    }
    return FERRITE_OK;
}

extern "C" int ferrite_act_quant_fp8(const void* x, int x_dtype, int64_t rows, int cols, uint8_t* q, uint8_t* scale,
                                     ferrite_stream_t stream) {
    if (rows > 0 && cols > 0 && (!x || !q || !scale)) return FERRITE_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(q) & 15)) return FERRITE_DECLINED;
    return launch_act_quant(x, x_dtype, rows, cols, q, scale, nullptr, nullptr, as_stream(stream));
}

extern "C" int ferrite_act_quant_fp8_x2(const void* x, int x_dtype, int64_t rows, int cols, uint8_t* q1, uint8_t* scale1,
                                        uint8_t* q2, uint8_t* scale2, ferrite_stream_t stream) {
    if (rows > 0 && cols > 0 && (!x || !q1 || !scale1 || !q2 || !scale2)) return FERRITE_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(q1) & 15) ||
        (reinterpret_cast<uintptr_t>(q2) & 15))
        return FERRITE_DECLINED;
    return launch_act_quant(x, x_dtype, rows, cols, q1, scale1, q2, scale2, as_stream(stream));
}
