// f32 mode of the expert FFN: activations stay f32, MXFP4 weights are dequantised exactly in registers, products and sums
// are f32.  It serves the shapes that the block-scaled MFMA modes decline and is what the layer is compared with the f32
// CPU golden in at 1e-5 (crates/ferrite-exec/src/lib.rs:1316-1332 for the expert, :1154-1164 for the combine).
//
// Rows are addressed in the grouped order of the permutation: row g < n*topk is assignment gather_src[g]
// (token = that / topk, expert = ids[that]); rows n*topk + t are the shared expert applied to token t.
#include "internal.hpp"
#include "numerics.hpp"

namespace fe {

typedef float fx_f2 __attribute__((ext_vector_type(2)));
typedef float fx_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int fx_u4 __attribute__((ext_vector_type(4), aligned(4)));   // checkpoint pointers promise no more

// Both GEMMs run on v_mfma_f32_16x16x4_f32 (f32 inputs, f32 accumulation) over the 16-row units of the permutation: an
// expert's weights are read and decoded once for up to 16 of its tokens.  A wave owns two tiles of 16 weight rows (gate
// and up rows of the same 16 outputs, or 32 rows of down) against the unit's rows; operands of one MFMA:
//   A: lane (r, g) = (lane % 16, lane / 16) holds weight row r at k = 128 s + 32 g + j, B: the same k of activation row r
// so a lane's 32 steps of a block of 128 k are the 16 code bytes and one scale byte of one 32-column block of its row.
// The activations go through LDS in windows of FX_WIN k, rows 16 bytes out of step so that 16 rows at one k touch
// different banks.  Every block of 128 k is summed in f32, by four accumulators per tile and a tree of three adds, and added
// to a sum in f64: 4.6e-7 from the 64-bit layer with f32 accumulators over the whole of K (27 tokens, hidden 2080), 2.5e-7
// this way, 2.6e-7 with the lane-wise sums that this kernel replaced (one wave per output row and token, the weights
// read again for every token: 283 + 157 us there, 58 + 32 us this way).
// Most of the time goes to the matrix pipe, padding of the units to 16 rows included: it is busy in 50 % of the cycles that
// a CU is busy at that shape (32 cycles per MFMA), vector instructions (1.5 per weight for the decoding) in 25 %.
constexpr int FX_WIN = 512, FX_PITCH = FX_WIN + 4, FX_SETS = 4;

struct FxArgs {
    const uint8_t *codes[2], *scales[2];         // routed experts: gate and up, or down (twice)
    const uint8_t *sh_codes[2], *sh_scales[2];   // shared expert
    const float* src;                            // x [n][K], or act [rows][src_ld]
    const int32_t* gather_src;
    const int32_t *unit_expert, *unit_row0, *unit_rows, *n_units;
    float* dst;                                  // act [rows][dst_ld], or y [rows][dst_ld]
    int n, topk, n_experts, max_units, groups;
    int rows, K, sh_rows, sh_K;                  // weight rows and reduction length, routed / shared
    int src_ld, dst_ld;
    float limit;
};

struct FxWeights {
    fx_u4 code[2];
    uint32_t scale[2];
};

// kSplit: the four waves of a block share a pair of tiles, each takes every fourth block of 128 k.
template <bool kGateUp, bool kSplit>
__global__ __launch_bounds__(256, 2) void experts_f32_kernel(FxArgs a) {
    __shared__ __align__(32) float xs[16 * FX_PITCH];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u = blockIdx.x / a.groups, ig = blockIdx.x % a.groups;
    if (u >= min(*a.n_units, a.max_units)) return;
    const int e = a.unit_expert[u], row0 = a.unit_row0[u], nrows = a.unit_rows[u];
    const int nk = a.n * a.topk;
    const bool shared = e == a.n_experts;
    // tables of an uninitialised workspace must not cause a fault
    if (nrows < 1 || nrows > 16 || row0 < 0 || e < 0 || e > a.n_experts) return;
    if (shared ? (a.sh_rows <= 0 || row0 < nk || row0 + nrows > nk + a.n) : row0 + nrows > nk) return;
    const int K = shared ? a.sh_K : a.K, rows = shared ? a.sh_rows : a.rows, nb = K / 32;
    constexpr int STEP = kGateUp ? 16 : 32;                  // output rows per pair of tiles
    const int pairs = rows / STEP, pair = kSplit ? ig : ig * 4 + wave;
    if ((kSplit ? ig : ig * 4) >= pairs) return;             // the whole block
    const int h0 = min(pair, pairs - 1) * STEP;              // a wave without a pair repeats the last one, unstored
    const size_t expert = shared ? 0 : (size_t)e * rows;
    const uint8_t *cp[2], *sp[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const size_t row = expert + h0 + (kGateUp ? 0 : 16 * t) + r;
        cp[t] = (shared ? a.sh_codes : a.codes)[t] + row * (size_t)(K / 2);
        sp[t] = (shared ? a.sh_scales : a.scales)[t] + row * (size_t)nb;
    }
    const int kblocks = (nb + 3) / 4;   // blocks of 128 k, the last one padded with zero weights
    auto load = [&](FxWeights& w, int kb) {
        const int b = kb * 4 + g, bc = min(b, nb - 1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            w.code[t] = *reinterpret_cast<const fx_u4*>(cp[t] + (size_t)bc * 16);
            w.scale[t] = b < nb ? (uint32_t)sp[t][bc] : 0u;   // byte 0 decodes to 0.0
        }
    };
    constexpr int KSTRIDE = kSplit ? 4 : 1;
    const int kfirst = kSplit ? wave : 0;
    FxWeights w;
    if (kfirst < kblocks) load(w, kfirst);
    auto token_row = [&](int c) -> const float* {
        const int gr = row0 + c;
        if (!kGateUp) return a.src + (size_t)gr * a.src_ld;
        int t = gr - nk;
        if (!shared) {
            const int i = a.gather_src[gr];
            t = (i < 0 || i >= nk) ? 0 : i / a.topk;
        }
        return a.src + (size_t)t * a.src_ld;
    };
    typedef double fx_d4 __attribute__((ext_vector_type(4)));
    fx_d4 total[2] = {{0., 0., 0., 0.}, {0., 0., 0., 0.}};

    // staging: 16 threads per row, each every 16th 16-byte piece of it
    const int sr = threadIdx.x >> 4, sj = threadIdx.x & 15;
    const float* srow = token_row(min(sr, nrows - 1));
    for (int w0 = 0; w0 < K; w0 += FX_WIN) {
        const int wk = min(FX_WIN, (K - w0 + 127) & ~127);
        if (w0 > 0) __syncthreads();   // every wave is done with the window in LDS
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            fx_f4 v[FX_WIN / 128];
#pragma unroll
            for (int i = 0; i < FX_WIN / 128; ++i) {
                const int k = ((h * (FX_WIN / 128) + i) * 16 + sj) * 4;
                v[i] = (fx_f4){0.f, 0.f, 0.f, 0.f};
                if (k < wk && w0 + k < K) v[i] = *reinterpret_cast<const fx_f4*>(srow + w0 + k);
            }
#pragma unroll
            for (int i = 0; i < FX_WIN / 128; ++i) {
                const int k = ((h * (FX_WIN / 128) + i) * 16 + sj) * 4;
                if (k < wk) *reinterpret_cast<fx_f4*>(&xs[sr * FX_PITCH + k]) = v[i];
            }
        }
        __syncthreads();
        const int kb_end = (w0 + wk) / 128;
#pragma unroll 1
        for (int kb = w0 / 128 + kfirst; kb < kb_end; kb += KSTRIDE) {   // FX_WIN / 128 is a multiple of KSTRIDE
            FxWeights next;
            load(next, min(kb + KSTRIDE, kblocks - 1));
            const fx_f4* xr = reinterpret_cast<const fx_f4*>(&xs[r * FX_PITCH + kb * 128 - w0 + 32 * g]);
            float sc[2];
            fx_f4 acc[2][FX_SETS];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                sc[t] = ue8m0_decode(w.scale[t]);
#pragma unroll
                for (int i = 0; i < FX_SETS; ++i) acc[t][i] = (fx_f4){0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const fx_f4 x0 = xr[2 * q], x1 = xr[2 * q + 1];
                const float xv[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                float wv[2][8];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    // two codes a conversion; the e2m1 value times a power of two is exact (byte 0 and NaN scales are
                    // the multiplication's business: the conversion itself runs at scale 1)
                    const uint32_t c = w.code[t][q];
                    const fx_f2 p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 0), p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 1),
                                p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 2), p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 3);
                    const float p[8] = {p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
#pragma unroll
                    for (int b = 0; b < 8; ++b) wv[t][b] = p[b] * sc[t];
                }
#pragma unroll
                for (int b = 0; b < 8; ++b)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[t][b % FX_SETS] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][b], xv[b], acc[t][b % FX_SETS], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const fx_f4 sum = (acc[t][0] + acc[t][1]) + (acc[t][2] + acc[t][3]);
                total[t] += __builtin_convertvector(sum, fx_d4);
            }
            w = next;
        }
    }
    if constexpr (kSplit) {
        __syncthreads();
        fx_d4* part = reinterpret_cast<fx_d4*>(xs);   // [wave][tile][lane]: 16 KiB
#pragma unroll
        for (int t = 0; t < 2; ++t) part[(wave * 2 + t) * 64 + lane] = total[t];
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int t = 0; t < 2; ++t)
            total[t] = (part[t * 64 + lane] + part[(2 + t) * 64 + lane]) + (part[(4 + t) * 64 + lane] + part[(6 + t) * 64 + lane]);
    } else if (pair >= pairs) {
        return;
    }
    const fx_f4 sum[2] = {__builtin_convertvector(total[0], fx_f4), __builtin_convertvector(total[1], fx_f4)};
    // D: lane (r, g) holds rows 4 g + v of the tile for activation row r
    if (r >= nrows) return;
    float* dst = a.dst + (size_t)(row0 + r) * a.dst_ld + h0 + 4 * g;
    if constexpr (kGateUp) {
        fx_f4 o;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = swiglu_ref(sum[0][v], sum[1][v], a.limit);
        *reinterpret_cast<fx_f4*>(dst) = o;
    } else {
        *reinterpret_cast<fx_f4*>(dst) = sum[0];
        *reinterpret_cast<fx_f4*>(dst + 16) = sum[1];
    }
}

// out[t] = sum_j (ascending) probs[t,j] * y[perm_map[t*k+j]]  then  + y[n*k + t]   (exec/lib.rs:1154-1164:
// a rounded product and a rounded add per slot, the shared expert last)
// One 16-byte piece of a y row: four f32, or eight bf16 widened (exact).
template <typename YT>
struct YPiece {
    static constexpr int N = 16 / sizeof(YT);
    uint4 raw;
    __device__ __forceinline__ float at(int i) const {
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
        if constexpr (sizeof(YT) == 4) return u2f(w[i]);
        else return u2f((i & 1) ? (w[i >> 1] & 0xffff0000u) : (w[i >> 1] << 16));
    }
};

// f32 -> bf16, round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint32_t combine_bf16(float f) {
    const uint32_t u = f2u(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// A thread owns 16 bytes of every y row of its token (4 or 8 columns).  The slots are walked in batches of eight:
// first the eight table entries, then the eight row pieces - all loads of a batch are in flight together - then the
// products and sums in slot order.
// With hc.residual set (f32 output only) the token's combined row x is not stored: the hyper-connection update that
// follows the layer (KernelBackend::hc_post, cpu.rs:788-807) is applied to it in registers and its nh rows
// out[t,i,:] = post[t,i] * x + sum_k comb[t,k,i] * residual[t,k,:] (k ascending, multiply and add rounded
// separately) are what goes to memory.
template <typename OT, typename YT>
__global__ __launch_bounds__(256) void combine_kernel(const YT* __restrict__ y, const float* __restrict__ probs,
                                                      const int32_t* __restrict__ perm_map, int n, int topk,
                                                      int H, int has_shared, OT* __restrict__ out, HcPostArgs hc) {
    constexpr int N = YPiece<YT>::N;
    const int t = blockIdx.y;
    const int h = (blockIdx.x * blockDim.x + threadIdx.x) * N;
    if (h >= H) return;
    float o[N];
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = 0.0f;
    const int nk = n * topk;
    for (int j0 = 0; j0 < topk; j0 += 8) {
        int g[8];
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool in = j0 + j < topk;
            g[j] = in ? perm_map[(size_t)t * topk + j0 + j] : -1;
            p[j] = in ? probs[(size_t)t * topk + j0 + j] : 0.0f;
        }
        YPiece<YT> v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // tables of an uninitialised workspace must not cause a fault: such slots are skipped
            const bool ok = g[j] >= 0 && g[j] < nk;
            v[j].raw = ok ? *reinterpret_cast<const uint4*>(y + (size_t)g[j] * H + h) : make_uint4(0u, 0u, 0u, 0u);
            g[j] = ok ? 1 : 0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (g[j]) {
#pragma unroll
                for (int i = 0; i < N; ++i) o[i] = fadd(o[i], fmul(p[j], v[j].at(i)));
            }
        }
    }
    if (has_shared) {
        YPiece<YT> v;
        v.raw = *reinterpret_cast<const uint4*>(y + ((size_t)nk + t) * H + h);
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = fadd(o[i], v.at(i));
    }
    OT* dst = out + (size_t)t * H + h;
    if constexpr (sizeof(OT) == 4) {
        if (hc.residual != nullptr) {
            // the thread's columns of all nh residual streams first, as hc_post_kernel does: out may then be the
            // residual buffer itself (the in-place update of the streams)
            constexpr int MAX_NH = 8;
            const int nh = hc.nh;
            float rv[MAX_NH][N];
#pragma unroll
            for (int k = 0; k < MAX_NH; ++k) {
                if (k < nh) {
                    const float* r = hc.residual + ((size_t)t * nh + k) * H + h;
#pragma unroll
                    for (int c = 0; c < N; c += 4) {
                        const float4 q = *reinterpret_cast<const float4*>(r + c);
                        rv[k][c] = q.x; rv[k][c + 1] = q.y; rv[k][c + 2] = q.z; rv[k][c + 3] = q.w;
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < MAX_NH; ++i) {
                if (i >= nh) break;
                const float p = hc.post[(size_t)t * nh + i];
                float acc[N];
#pragma unroll
                for (int c = 0; c < N; ++c) acc[c] = fmul(p, o[c]);
#pragma unroll
                for (int k = 0; k < MAX_NH; ++k) {
                    if (k < nh) {
                        const float cf = hc.comb[((size_t)t * nh + k) * nh + i];
#pragma unroll
                        for (int c = 0; c < N; ++c) acc[c] = fadd(acc[c], fmul(cf, rv[k][c]));
                    }
                }
                float* od = reinterpret_cast<float*>(out) + ((size_t)t * nh + i) * H + h;
#pragma unroll
                for (int c = 0; c < N; c += 4)
                    *reinterpret_cast<float4*>(od + c) = make_float4(acc[c], acc[c + 1], acc[c + 2], acc[c + 3]);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < N; i += 4) *reinterpret_cast<float4*>(dst + i) = make_float4(o[i], o[i + 1], o[i + 2], o[i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < N; i += 4)
            *reinterpret_cast<uint2*>(dst + i) = make_uint2(combine_bf16(o[i]) | (combine_bf16(o[i + 1]) << 16),
                                                            combine_bf16(o[i + 2]) | (combine_bf16(o[i + 3]) << 16));
    }
}

template <bool kGateUp>
static int launch_experts_f32(FxArgs a, const UnitTables& units, hipStream_t st) {
    if (units.unit_rows_cap != 16) return FERRITE_ERR_INVALID_ARG;
    a.unit_expert = units.unit_expert; a.unit_row0 = units.unit_row0; a.unit_rows = units.unit_rows;
    a.n_units = units.n_units; a.max_units = units.max_units;
    const int pairs = (a.rows > a.sh_rows ? a.rows : a.sh_rows) / (kGateUp ? 16 : 32);
    const bool split = f32_split(a.n, a.topk, a.n_experts, units.max_units, a.rows, a.sh_rows, a.K, !kGateUp) != 0;
    a.groups = split ? pairs : (pairs + 3) / 4;
    const long blocks = (long)units.max_units * a.groups;
    if (blocks > 0x7fffffffL) return FERRITE_DECLINED;
    if (split) experts_f32_kernel<kGateUp, true><<<(unsigned)blocks, 256, 0, st>>>(a);
    else experts_f32_kernel<kGateUp, false><<<(unsigned)blocks, 256, 0, st>>>(a);
    return check_launch("experts_f32");
}

int launch_gate_up_f32(const ferrite_moe_shape& s, const ferrite_moe_weights& w, const float* x, int n,
                       const int32_t* gather_src, const UnitTables& units, float* act, hipStream_t st) {
    FxArgs a{};
    a.codes[0] = w.gate_w; a.codes[1] = w.up_w; a.scales[0] = w.gate_s; a.scales[1] = w.up_s;
    a.sh_codes[0] = w.sh_gate_w; a.sh_codes[1] = w.sh_up_w; a.sh_scales[0] = w.sh_gate_s; a.sh_scales[1] = w.sh_up_s;
    a.src = x; a.gather_src = gather_src; a.dst = act;
    a.n = n; a.topk = s.topk; a.n_experts = s.n_experts;
    a.rows = s.inter; a.sh_rows = s.shared_inter; a.K = a.sh_K = s.hidden;
    a.src_ld = s.hidden; a.dst_ld = s.inter > s.shared_inter ? s.inter : s.shared_inter;
    a.limit = s.swiglu_limit;
    return launch_experts_f32<true>(a, units, st);
}

int launch_down_f32(const ferrite_moe_shape& s, const ferrite_moe_weights& w, const float* act, int n,
                    const UnitTables& units, float* y, hipStream_t st) {
    FxArgs a{};
    a.codes[0] = a.codes[1] = w.down_w; a.scales[0] = a.scales[1] = w.down_s;
    a.sh_codes[0] = a.sh_codes[1] = w.sh_down_w; a.sh_scales[0] = a.sh_scales[1] = w.sh_down_s;
    a.src = act; a.dst = y;
    a.n = n; a.topk = s.topk; a.n_experts = s.n_experts;
    a.rows = s.hidden; a.sh_rows = s.shared_inter > 0 ? s.hidden : 0; a.K = s.inter; a.sh_K = s.shared_inter;
    a.src_ld = s.inter > s.shared_inter ? s.inter : s.shared_inter; a.dst_ld = s.hidden;
    return launch_experts_f32<false>(a, units, st);
}

int launch_combine(const void* y, int y_dtype, const float* probs, const int32_t* perm_map, int n, int topk,
                   int hidden, int has_shared, void* out, int out_dtype, hipStream_t st, const HcPostArgs* hcp) {
    const HcPostArgs hc = hcp ? *hcp : HcPostArgs{nullptr, nullptr, nullptr, 0};
    if (hc.residual && (out_dtype != FERRITE_DT_F32 || hc.nh < 1 || hc.nh > 8 || !hc.post || !hc.comb)) return FERRITE_ERR_INVALID_ARG;
    const bool of32 = out_dtype == FERRITE_DT_F32, yf32 = y_dtype == FERRITE_DT_F32;
    const int per_thread = yf32 ? 4 : 8;   // columns per thread: 16 bytes of a y row
    if (hidden % per_thread) return FERRITE_ERR_INVALID_ARG;
    dim3 grid((hidden / per_thread + 255) / 256, n);
    if ((!of32 && out_dtype != FERRITE_DT_BF16) || (!yf32 && y_dtype != FERRITE_DT_BF16)) return FERRITE_ERR_INVALID_ARG;
    if (of32 && yf32)
        combine_kernel<float, float><<<grid, 256, 0, st>>>((const float*)y, probs, perm_map, n, topk, hidden, has_shared, (float*)out, hc);
    else if (of32)
        combine_kernel<float, uint16_t><<<grid, 256, 0, st>>>((const uint16_t*)y, probs, perm_map, n, topk, hidden, has_shared, (float*)out, hc);
    else if (yf32)
        combine_kernel<uint16_t, float><<<grid, 256, 0, st>>>((const float*)y, probs, perm_map, n, topk, hidden, has_shared, (uint16_t*)out, hc);
    else
        combine_kernel<uint16_t, uint16_t><<<grid, 256, 0, st>>>((const uint16_t*)y, probs, perm_map, n, topk, hidden, has_shared, (uint16_t*)out, hc);
    return check_launch("combine");
}

}  // namespace fe
