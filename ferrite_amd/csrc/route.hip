// Router logits (bit-exact sequential-k f32 GEMM), noaux-tc sigmoid group-limited top-k, and the stable
// token permutation by expert.  gfx950, wave64.
#include "internal.hpp"
#include "device_utils.hpp"
#include "numerics.hpp"

namespace fe {

// ------------------------------------------------------------------------------------------------
// x . w^T with the reference's arithmetic (crates/ferrite-kernel/src/cpu.rs:106-111): for every output one
// chain s = 0; s = fl(s + fl(x[l] * w[l])) in ascending l.  The chain cannot be re-associated, its adds stay on the
// vector ALU.  Three kernels; all stage x and w through LDS as f32 in chunks of 64 k, the first two with the fetches of
// several chunks in flight in registers and one barrier per chunk.
//
// chain_mfma_kernel, for enough chains: the products come from the matrix cores (an f32 MFMA on a zero accumulator
// gives the correctly rounded product; -0 comes out as +0, which a chain that starts at +0 cannot see).  A wave owns
// 16 tokens x 16 outputs.  v_mfma_f32_16x16x1_4b is four outer products of 16 x 16, and its four blocks take the same
// tokens and outputs at four different k: lane l = (q = l / 16, r = l % 16) holds x[t0 + r] and w[o0 + r] at
// k = 16 s + 4 q .. + 3, the MFMA of component c leaves in register 4 b + v the product of token 4 q + v, output r at
// k = 16 s + 4 b + c.  A step of 16 k is two 16-byte LDS reads per lane, four MFMAs and 64 adds (four chains per lane);
// the products of step s + 1 are made while the adds of step s run.  Bound by the adds: of the cycles that a CU is busy
// (4096 x 128, counters) vector instructions issue in 78 %, nine tenths of them adds; the matrix pipe is busy in 34 % (32
// cycles per MFMA), nothing waits for LDS banks.
//
// chain_valu_kernel, for few chains, where a chain's own length is the time: one chain per lane (8 tokens x 8 outputs per
// wave), multiply and add on the vector ALU.  A lone wave issues one instruction per four cycles.
//
// chain_rows_kernel, for a few rows of x against very many outputs, where w's way through memory is the time: a wave has one
// row, a lane one output, so that the chip is not occupied with padding rows.
//
// us:                                                   before    mfma    valu
//   router 8192 tokens x 256, H 7168 (bf16 x)              735     648     -       (valu, 4 x 4 chains per lane: 620;
//                                                                                   nowhere else faster, not kept)
//   router 4096 x 128, H 4096 (bf16 x)                     149     105     -       (2 x 2 chains per lane: 125)
//   router 2047 x 128, H 4096 (f32 x)                      146      76     -       (2 x 2: 101)
//   router 509 x 128, H 4096 (bf16 x)                       47      50     42
//   100 x 3072, k 4096 / 100 x 4096, k 1536             168 / 78   91 / 40  -      (2 x 2: 109 / 47)
//   100 x 128, k 4096 / 27 x 32, k 2080                  70 / 37   46 / 25  35 / 20
// The lines between them, us:                          mfma    valu    rows
//   384 / 512 tiles (32 x 3072, 1024 x 128), k 4096      64      46
//   560 / 672 / 768 tiles                                64      63 / 63 / 66
//   784 / 1024 tiles                                     64 / 65 79 / 84
//   512 / 640 / 768 tiles, k 7168                       109      76 / 106 / 109
//   4 x 17000 / 32768 / 65536, k 4096              86 / 127 / 238  82 / 174 / 332  67 / 123 / 199
//   4 x 32768 / 65536, k 256                          9.8 / 20  12 / 22  7.0 / 13
//   8 x 65536, k 4096 / 256                           236 / 21  341 / 22  384 / 23 (two passes over w)
// Also built: x through DPP broadcasts or v_readlane instead of LDS (161 and 177 us for the second line: both instructions
// cost several plain ones); operands read from memory in MFMA order without LDS (64 requests per load to the address
// unit: 121 us for 100 x 3072); one chunk in flight instead of three (51 against 46 us for 100 x 128).
// ------------------------------------------------------------------------------------------------
typedef float ch_f16 __attribute__((ext_vector_type(16)));
typedef float ch_f4 __attribute__((ext_vector_type(4)));
typedef ch_f4 ch_f4u __attribute__((aligned(4)));   // x of the stand-alone op may be aligned to its elements only
typedef unsigned int ch_u2 __attribute__((ext_vector_type(2)));

constexpr int CH_T = 16;              // rows of x and of w per staged tile
constexpr int CH_KC = 64;             // k per chunk
constexpr int CH_PIECES = CH_KC / 4;  // 16-byte pieces of a row's chunk
constexpr int CH_TILE = CH_T * CH_PIECES;

struct ChainArgs {
    const void* x;       // [n][k]
    const float* w;      // [o][k], or the k-blocked transpose [k/4][w_pitch][4] of the packed router weight
    const float* bias;   // [o] or NULL
    float* out;          // [n][o]
    int n, k, o, w_pitch;
    int x_major;         // which operand's tiles are dealt to the XCDs
};

// Block -> (token tile of 16, output group of OT tiles).  Hardware deals consecutive blocks round-robin over the 8 XCDs,
// so the blocks that read the same tile of the larger operand (x of thousands of tokens, or the weight of a wide matmul)
// get block numbers 8 apart: one L2 fetches that tile once.  Returns false for blocks without work.
template <int OT>
__device__ __forceinline__ bool chain_block(const ChainArgs& a, int& t0, int& o0) {
    const int tg = (a.n + CH_T - 1) / CH_T, og = (a.o + OT * CH_T - 1) / (OT * CH_T);
    const int minor = a.x_major ? og : tg, majors = a.x_major ? tg : og;
    const int slot = blockIdx.x >> 3;
    const int mj = (slot / minor) * 8 + (blockIdx.x & 7), mn = slot % minor;
    t0 = (a.x_major ? mj : mn) * CH_T;
    o0 = (a.x_major ? mn : mj) * OT * CH_T;
    return mj < majors;
}

// A thread's part of the block's staging: one piece of x and WN of w per chunk.  Of a row-major operand 16 lanes fetch
// the 16 pieces of a row, of the transposed weight 16 rows of a piece (256 contiguous bytes either way); w tile `tile`
// of the block, its rows or pieces group * 4 * WN .. are fetched by the calling wave.  Piece j of row r sits at slot
// 16 r + (j ^ r) of its tile: the sixteen neighbouring lanes of a write and of a read touch different banks.  Rows past
// the end repeat the last one, pieces past K are zero (they add +0 to the chains).
template <typename XT, bool kPackedW, int WN, bool kShort>
struct ChainFetch {
    const XT* xrow;
    const float* wrow[WN];
    int xslot, wslot[WN], pj, K, nchunk, w_pitch;
    struct Set {
        ch_f4 x, w[WN];
    };
    __device__ __forceinline__ ChainFetch(const ChainArgs& a, int t0, int o_tile, int group) : pj(threadIdx.x & 15), K(a.k) {
        const int pr = threadIdx.x >> 4, r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
        nchunk = (K + CH_KC - 1) / CH_KC;
        w_pitch = a.w_pitch;
        xrow = static_cast<const XT*>(a.x) + (size_t)min(t0 + pr, a.n - 1) * K;
        xslot = pr * CH_PIECES + (pj ^ pr);
#pragma unroll
        for (int i = 0; i < WN; ++i) {
            const int m = (group * WN + i) * 4 + q;
            if constexpr (kPackedW) {
                wrow[i] = a.w + ((size_t)m * a.w_pitch + min(o_tile + r, a.w_pitch - 1)) * 4;
                wslot[i] = r * CH_PIECES + (m ^ r);
            } else {
                wrow[i] = a.w + (size_t)min(o_tile + m, a.o - 1) * K;
                wslot[i] = m * CH_PIECES + (r ^ m);
            }
        }
    }
    __device__ __forceinline__ void load(Set& f, int c) const {   // past the end the last chunk again, never used
        if (kShort && c >= nchunk) return;
        c = min(c, nchunk - 1);
        const int k = min(c * CH_KC + pj * 4, K - 4);
        if constexpr (sizeof(XT) == 4) {
            f.x = *reinterpret_cast<const ch_f4u*>(xrow + k);
        } else {
            const ch_u2 v = *reinterpret_cast<const ch_u2*>(xrow + k);
            f.x[0] = u2f(v[0]);
            f.x[1] = u2f(v[1]);
        }
#pragma unroll
        for (int i = 0; i < WN; ++i)
            f.w[i] = *reinterpret_cast<const ch_f4*>(wrow[i] + (kPackedW ? (size_t)c * CH_PIECES * 4 * w_pitch : (size_t)k));
    }
    __device__ __forceinline__ void store(const Set& f, int c, ch_f4* xs, ch_f4* ws) const {
        if (kShort && c >= nchunk) return;
        const bool in = min(c, nchunk - 1) * CH_KC + pj * 4 < K;   // the transposed weight comes with K % 64 == 0
        const ch_f4 zero = {0.f, 0.f, 0.f, 0.f};
        ch_f4 xv = f.x;
        if constexpr (sizeof(XT) == 2) {
            const uint32_t lo = f2u(xv[0]), hi = f2u(xv[1]);
            xv = (ch_f4){u2f(lo << 16), u2f(lo & 0xffff0000u), u2f(hi << 16), u2f(hi & 0xffff0000u)};
        }
        xs[xslot] = in ? xv : zero;
#pragma unroll
        for (int i = 0; i < WN; ++i) ws[wslot[i]] = (kPackedW || in) ? f.w[i] : zero;
    }
};

// Block = 4 waves: 16 tokens x 64 outputs.  Chunks c and c + 1 are readable while chunk c is walked, chunk c + 2 is
// written at its start; three more chunks are on their way.
template <typename XT, bool kPackedW, bool kShort>
__global__ __launch_bounds__(256, 2) void chain_mfma_kernel(ChainArgs a) {
    __shared__ ch_f4 xs[3][CH_TILE];
    __shared__ ch_f4 ws[4][3][CH_TILE];
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t0, o0;
    if (!chain_block<4>(a, t0, o0)) return;   // the whole block
    o0 += wave * CH_T;                        // may lie past o: such a wave works on the last row
    const ChainFetch<XT, kPackedW, 4, kShort> src(a, t0, o0, 0);
    const int nchunk = src.nchunk;
    ch_f4 xo[2], wo[2];
    auto read = [&](int at, int u, int to) {
        xo[to] = xs[at][r * CH_PIECES + ((4 * u + q) ^ r)];
        wo[to] = ws[wave][at][r * CH_PIECES + ((4 * u + q) ^ r)];
    };
    ch_f16 p[2][4];
    const ch_f16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float acc[4] = {0.f, 0.f, 0.f, 0.f};

    typename ChainFetch<XT, kPackedW, 4, kShort>::Set f[3];   // f[c % 3]: chunk c
    src.load(f[0], 0);
    src.load(f[1], 1);
    src.load(f[2], 2);
    src.store(f[0], 0, xs[0], ws[wave][0]);
    src.load(f[0], 3);
    src.store(f[1], 1, xs[1], ws[wave][1]);
    src.load(f[1], 4);
    __syncthreads();
    read(0, 0, 0);
    read(0, 1, 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) p[0][c] = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[0][c], wo[0][c], zero, 0, 0, 0);
#pragma unroll 1
    for (int c0 = 0; c0 < nchunk; c0 += 3) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (c0 + j >= nchunk) break;   // uniform
            const int c = c0 + j, at = j, at1 = (j + 1) % 3, at2 = (j + 2) % 3;   // slots of chunks c, c + 1, c + 2
            if (c) __syncthreads();   // chunk c + 1 is complete; nobody reads the slot of chunk c - 1 any more
            src.store(f[at2], c + 2, xs[at2], ws[wave][at2]);
            __builtin_amdgcn_sched_barrier(0);
            src.load(f[at2], c + 5);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                // adds of step 4 c + u, products of the next one, operands of the one after
                read(u < 2 ? at : at1, (u + 2) & 3, u & 1);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    p[(u + 1) & 1][b] = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[(u + 1) & 1][b], wo[(u + 1) & 1][b], zero, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[v] = fadd(acc[v], p[u & 1][cc][4 * b + v]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
    const int col = o0 + r;
    if (col < a.o) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = t0 + 4 * q + v;
            if (t < a.n) a.out[(size_t)t * a.o + col] = a.bias ? fadd(acc[v], a.bias[col]) : acc[v];
        }
    }
}

// Block = 4 waves, two by two: 16 tokens x 16 outputs.  Chunk c + 1 is written while chunk c is walked; three more are
// on their way.
template <typename XT, bool kPackedW, bool kShort>
__global__ __launch_bounds__(256, 2) void chain_valu_kernel(ChainArgs a) {
    constexpr int FD = 4;   // even: a register set's LDS slot is a constant
    __shared__ ch_f4 xs[2][CH_TILE], ws[2][CH_TILE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t0, o0;
    if (!chain_block<1>(a, t0, o0)) return;   // the whole block
    const ChainFetch<XT, kPackedW, 1, kShort> src(a, t0, o0, wave);
    const int nchunk = src.nchunk;
    const int xr = (wave >> 1) * 8 + (lane >> 3), wr = (wave & 1) * 8 + (lane & 7);
    float acc = 0.0f;
    typename ChainFetch<XT, kPackedW, 1, kShort>::Set f[FD];   // f[c % FD]: chunk c
#pragma unroll
    for (int i = 0; i < FD; ++i) src.load(f[i], i);
    src.store(f[0], 0, xs[0], ws[0]);
    src.load(f[0], FD);
#pragma unroll 1
    for (int c0 = 0; c0 < nchunk; c0 += FD) {
#pragma unroll
        for (int h = 0; h < FD; ++h) {
            const int c = c0 + h;
            if (c >= nchunk) break;   // uniform
            __syncthreads();   // chunk c is complete; nobody reads the slot of chunk c - 1 any more
            src.store(f[(h + 1) % FD], c + 1, xs[(h + 1) & 1], ws[(h + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
            src.load(f[(h + 1) % FD], c + 1 + FD);
            __builtin_amdgcn_sched_barrier(0);
            ch_f4 xv[2], wv[2];
            auto read = [&](int p, int to) {
                xv[to] = xs[h & 1][xr * CH_PIECES + (p ^ xr)];
                wv[to] = ws[h & 1][wr * CH_PIECES + (p ^ wr)];
            };
            read(0, 0);
#pragma unroll
            for (int p = 0; p < CH_PIECES; ++p) {
                if (p + 1 < CH_PIECES) read(p + 1, (p + 1) & 1);
#pragma unroll
                for (int q = 0; q < 4; ++q) acc = fadd(acc, fmul(xv[p & 1][q], wv[p & 1][q]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const int t = t0 + xr, col = o0 + wr;
    if (t < a.n && col < a.o) a.out[(size_t)t * a.o + col] = a.bias ? fadd(acc, a.bias[col]) : acc;
}

// Block = 4 waves: up to 4 rows x 64 outputs, w transposed in LDS so that a lane reads four consecutive k of its row
// at once, two buffers.
constexpr int CR_ROWS = 4, CR_OUTS = 64;

__global__ __launch_bounds__(256, 4) void chain_rows_kernel(ChainArgs a) {
    __shared__ ch_f4 ws[2][CH_PIECES][CR_OUTS + 1];
    __shared__ ch_f4 xs[2][CR_ROWS][CH_PIECES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int o0 = blockIdx.x * CR_OUTS, K = a.k;
    const int nchunk = (K + CH_KC - 1) / CH_KC;
    const int pr = tid >> 4, pj = tid & 15;   // a thread stages piece pj of w rows pr, pr + 16, .. and of x row pr
    const float* xrow = static_cast<const float*>(a.x) + (size_t)min(pr, a.n - 1) * K;
    const ch_f4 zero = {0.f, 0.f, 0.f, 0.f};
    ch_f4 w[4], x = zero;
    auto fetch = [&](int c) {   // pieces past K are zero, rows past the end repeat the last one
        const int k = c * CH_KC + pj * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            w[i] = k < K ? *reinterpret_cast<const ch_f4*>(a.w + (size_t)min(o0 + pr + 16 * i, a.o - 1) * K + k) : zero;
        if (pr < CR_ROWS) x = k < K ? *reinterpret_cast<const ch_f4u*>(xrow + k) : zero;
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ws[buf][pj][pr + 16 * i] = w[i];
        if (pr < CR_ROWS) xs[buf][pr][pj] = x;
    };
    float acc = 0.0f;
    fetch(0);
    stash(0);
    __syncthreads();
    for (int c = 0; c < nchunk; ++c) {
        const int buf = c & 1;
        if (c + 1 < nchunk) fetch(c + 1);
#pragma unroll 4
        for (int j = 0; j < CH_PIECES; ++j) {
            const ch_f4 wv = ws[buf][j][lane], xv = xs[buf][wave][j];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc = fadd(acc, fmul(xv[q], wv[q]));
        }
        if (c + 1 < nchunk) stash(buf ^ 1);
        __syncthreads();
    }
    const int col = o0 + lane;
    if (wave < a.n && col < a.o) a.out[(size_t)wave * a.o + col] = a.bias ? fadd(acc, a.bias[col]) : acc;
}

// Which kernel (figures at the top): 512 tiles of 16 x 16 chains are two waves of the one-chain-per-lane kernel for each of
// the chip's 1024 SIMDs; beyond that its multiplies and LDS reads bound it, and below that the matrix-core kernel leaves SIMDs idle.  Up to
// four rows against more than 1024 tiles of outputs take the kernel that has no padding rows.
// Up to 128 k the fetches that run ahead are not made past the end: they would be most of all fetches (24 x 65536, k 64:
// 15 -> 11 us; 1 x 12288: 4.3 -> 3.7).  At 256 k, and with it in the loop of longer chains, the waits that the conditional loads
// need cost more than the fetches (131072 outputs, k 256: 35 -> 38; 32768, k 4096: 127 -> 143).
constexpr int CH_SHORT = 128, CH_ROWS_TILES = 1024;

template <typename XT, bool kPackedW>
static int launch_chain(ChainArgs a, hipStream_t st) {
    const long tg = ((long)a.n + CH_T - 1) / CH_T, ot = ((long)a.o + CH_T - 1) / CH_T;
    if constexpr (sizeof(XT) == 4 && !kPackedW) {
        if (a.n <= CR_ROWS && ot > CH_ROWS_TILES) {
            chain_rows_kernel<<<(unsigned)((a.o + CR_OUTS - 1) / CR_OUTS), 256, 0, st>>>(a);
            return check_launch("chain_rows");
        }
    }
    const bool mfma = tg * ot > 512;
    const long og = mfma ? (ot + 3) / 4 : ot;
    a.x_major = (size_t)a.n * sizeof(XT) >= (size_t)a.o * sizeof(float);
    const long blocks = ((a.x_major ? tg : og) + 7) / 8 * 8 * (a.x_major ? og : tg);
    if (blocks > 0x7fffffffL) return FERRITE_DECLINED;
    auto go = [&](auto kernel) { kernel<<<(unsigned)blocks, 256, 0, st>>>(a); };
    if (a.k <= CH_SHORT) mfma ? go(chain_mfma_kernel<XT, kPackedW, true>) : go(chain_valu_kernel<XT, kPackedW, true>);
    else mfma ? go(chain_mfma_kernel<XT, kPackedW, false>) : go(chain_valu_kernel<XT, kPackedW, false>);
    return check_launch("chain");
}

int launch_matmul_exact(const void* x, int x_dtype, const float* w, const float* bias, float* out, int n, int k,
                        int o, hipStream_t st) {
    if (n < 0 || k < 0 || o < 0) return FERRITE_ERR_INVALID_ARG;
    if (n == 0 || o == 0) return FERRITE_OK;
    // four consecutive k per load: the weight's rows are whole, 16-byte aligned pieces of four
    if (k < 4 || (k & 3) != 0 || (reinterpret_cast<uintptr_t>(w) & 15) != 0) return FERRITE_DECLINED;
    ChainArgs a{x, w, bias, out, n, k, o, 0, 0};
    if (x_dtype == FERRITE_DT_F32) return launch_chain<float, false>(a, st);
    if (x_dtype == FERRITE_DT_BF16) return launch_chain<uint16_t, false>(a, st);
    return FERRITE_ERR_INVALID_ARG;
}

// Any-k variant: one lane per output straight from global memory (small or unaligned problems).
__global__ void matmul_exact_simple_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                           const float* __restrict__ bias, float* __restrict__ out, int n, int k,
                                           int o) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)n * o) return;
    int t = (int)(idx / o), j = (int)(idx % o);
    float s = 0.0f;
    for (int l = 0; l < k; ++l) s = fadd(s, fmul(x[(size_t)t * k + l], w[(size_t)j * k + l]));
    if (bias) s = fadd(s, bias[j]);
    out[idx] = s;
}

// ------------------------------------------------------------------------------------------------
// clamped SwiGLU (cpu.rs:178-203)
// ------------------------------------------------------------------------------------------------
__global__ void swiglu_kernel(const float* __restrict__ gate_up, float limit, float* __restrict__ out, int n,
                              int inter) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)n * inter) return;
    size_t i = idx / inter, j = idx % inter;
    out[idx] = swiglu_ref(gate_up[i * 2 * inter + j], gate_up[i * 2 * inter + inter + j], limit);
}

// ------------------------------------------------------------------------------------------------
// Routing: one wave per token.  sigmoid -> +bias -> (group top-2 sums -> keep topk_group groups) -> the topk-th
// largest choice as a threshold, found bit by bit -> the candidates at or above it, ranked among themselves under
// (choice desc, index asc), are the selection, in order -> renormalised weights from the raw sigmoid.
// Semantics and operation order follow cpu.rs:546-569; ties -> lower index (cpu.rs:560).
// ------------------------------------------------------------------------------------------------
constexpr int RT_MAX_E = 512;
constexpr int RT_MAX_K = 32;
constexpr int RT_RANK_E = RT_MAX_K;   // experts up to which a token's are ranked against each other (route_wave_ni): RouteScratch::sel_key

__device__ __forceinline__ uint32_t ordered_u32(float f) {
    uint32_t u = f2u(f);
    return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}

// LDS scratch of one routing wave
struct RouteScratch {
    float choice[RT_MAX_E];
    float score[64];
    unsigned long long sel_key[RT_MAX_K];
    float pre_sig[RT_MAX_K];
    float sel_sig[RT_MAX_K];
    int sel_id[RT_MAX_K];
};

// Loads that must observe stores made by other workgroups of the same kernel.
__device__ __forceinline__ float load_coherent(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int load_coherent(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders a wave's own LDS traffic: its lanes' earlier writes are visible to its later reads.  The LDS unit
// executes one wave's instructions in order, so only the compiler has to be kept from reordering.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// v of the lane that `kCtrl` pairs with this one inside its row of 16 (quad_perm, row_half_mirror, row_mirror).
template <int kCtrl>
__device__ __forceinline__ float dpp_pair(float v) {
    return u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(v), kCtrl, 0xf, 0xf, false));
}

// The two largest of a group of 2^lg neighbouring lanes, each of which brings m1 (m2 = -inf) and gets the group's.
__device__ __forceinline__ void group_top2(float& m1, float& m2, int lg) {
    auto merge = [&](float o1, float o2) {
        m2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
        m1 = fmaxf(m1, o1);
    };
    if (lg > 0) merge(dpp_pair<0xB1>(m1), dpp_pair<0xB1>(m2));     // lane ^ 1
    if (lg > 1) merge(dpp_pair<0x4E>(m1), dpp_pair<0x4E>(m2));     // lane ^ 2
    if (lg > 2) merge(dpp_pair<0x141>(m1), dpp_pair<0x141>(m2));   // the other quad of eight (quads hold one value by now)
    if (lg > 3) merge(dpp_pair<0x140>(m1), dpp_pair<0x140>(m2));   // the other half of sixteen
    if (lg > 4) merge(__shfl_xor(m1, 16, 64), __shfl_xor(m2, 16, 64));
    if (lg > 5) merge(__shfl_xor(m1, 32, 64), __shfl_xor(m2, 32, 64));
}

// One wave routes one token.  `lg` = the token's e logits, or lane j's is in `own` (kOwn, e <= 64).  The scratch is private
// to the wave, so waves of a block may call this independently of each other.
// NI = expert slots per lane (ceil(e / 64) rounded up to 1, 2, 4 or 8): everything below costs in proportion to it.
// A lone wave issues an instruction every four cycles, so the count of instructions bounds this: the topk-th largest
// choice is found bit by bit (two or three instructions per slot and bit, about 20 bits until exactly topk keys are at or
// above it) instead of ranking every expert against every other, only the selected ones are ranked, and a group's two largest
// meet by lane exchanges.  Against the ranking loops, us: head of one token 27.2 -> 25.7, 32 tokens 29.4 -> 27.6, 192 48.0 -> 45.5,
// 200 tokens of 64 experts in one group 37.0 -> 25.9; moe_route_kernel, 4096 tokens x 128 experts 11.7 -> 8.3, 8192 x 256 50.5 -> 17.5.
// Up to 32 experts the bits are more than the experts, and ranking stays (moe_route_kernel, 100 tokens, ranking / threshold: 8
// experts 2.8 / 3.2, 16 3.1 / 3.4, 32 3.3 / 3.6, 48 3.5 / 3.6, 64 3.6 / 3.5).
template <bool kCoherent, bool kOwn, int NI>
__device__ __forceinline__ void route_wave_ni(const float* __restrict__ lg, float own, const float* __restrict__ bias, bool live,
                                           int e, int topk, int n_group, int topk_group, float scaling,
                                           RouteScratch& sc, float* __restrict__ probs, float* __restrict__ ids_f32,
                                           int32_t* __restrict__ ids_i32) {
    const int lane = threadIdx.x & 63;
    const int ni = (e + 63) >> 6;
    float sg[NI], ch[NI];
    bool ok[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int j = lane + 64 * i;
        ok[i] = live && i < ni && j < e;
        float l = 0.0f;
        if constexpr (kOwn) l = ok[i] ? own : 0.0f;
        else if (ok[i]) l = kCoherent ? load_coherent(lg + j) : lg[j];
        sg[i] = sigmoid_ref(l);
        ch[i] = ok[i] ? fadd(sg[i], bias ? bias[j] : 0.0f) : 0.0f;
        // A NaN score (NaN logit or bias) is never selected, as in the reference's device router, whose arg-max
        // comparisons are false for NaN (kernels/cuda/ferrite_kernels.cu:1233-1241); slots that no finite score
        // can fill keep id -1 and weight 0 (ferrite_kernels.cu:1255-1270).  CpuBackend panics instead (cpu.rs:560).
        if (ch[i] != ch[i]) ok[i] = false;
    }
    if (lane < RT_MAX_K) { sc.sel_id[lane] = -1; sc.sel_sig[lane] = 0.0f; }

    if (n_group > 1) {
        const int gs = e / n_group;
        const bool pow2 = (gs & (gs - 1)) == 0 && gs <= 64;   // groups are aligned runs of lanes
        const int lgs = pow2 ? __builtin_ctz(gs) : 0;
        // score of a group: largest + second largest choice (largest first; the order of equal ones does not show)
        float gscore = 0.0f;
        if (pow2) {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (i >= ni) break;
                const int j = lane + 64 * i;
                const float ninf = u2f(0xff800000u);
                float m1 = j < e && ch[i] == ch[i] ? ch[i] : ninf, m2 = ninf;
                group_top2(m1, m2, lgs);
                if (j < e && (lane & (gs - 1)) == 0) sc.score[j >> lgs] = gs > 1 ? fadd(m1, m2) : m1;
            }
            wave_sync();
            if (lane < n_group) gscore = sc.score[lane];
        } else {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                int j = lane + 64 * i;
                if (i < ni && j < e) sc.choice[j] = ch[i];
            }
            wave_sync();
            if (lane < n_group) {   // lane g scores group g
                float m1 = u2f(0xff800000u), m2 = u2f(0xff800000u);
                for (int j = lane * gs; j < (lane + 1) * gs; ++j) {
                    float c = sc.choice[j];
                    if (c > m1) { m2 = m1; m1 = c; }
                    else if (c > m2) m2 = c;
                }
                gscore = fadd(m1, m2);
            }
        }
        // rank of group g under (score desc, index asc)
        int rank = 0;
        for (int g2 = 0; g2 < n_group; ++g2) {
            const float s2 = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(gscore), g2));
            rank += (s2 > gscore || (s2 == gscore && g2 < lane)) ? 1 : 0;
        }
        const unsigned long long keep = __ballot(lane < n_group && rank < topk_group);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int j = lane + 64 * i, g = pow2 ? j >> lgs : j / gs;
            if (!((keep >> (g & 63)) & 1ull)) ok[i] = false;
        }
    }

    // order-preserving bits of the choices; 0 = not selectable (-inf is 0x007fffff)
    uint32_t key[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) key[i] = ok[i] ? ordered_u32(ch[i]) : 0u;
    if (NI == 1 && e <= RT_RANK_E) {   // every expert against every other
        // larger = earlier in the reference's sort (choice desc, index asc)
        const unsigned long long mine = key[0] != 0u ? ((unsigned long long)key[0] << 32) | (0xFFFFFFFFu - (uint32_t)lane) : 0ull;
        if (lane < e) sc.sel_key[lane] = mine;
        wave_sync();
        int rank = 0;
        for (int j2 = 0; j2 < e; ++j2) rank += sc.sel_key[j2] > mine ? 1 : 0;   // same address in every lane: an LDS broadcast
        if (mine != 0ull && rank < topk) {
            sc.sel_id[rank] = lane;
            sc.sel_sig[rank] = sg[0];
        }
        wave_sync();
    } else {
        uint32_t thr = 0;   // the largest value that at least topk keys reach, or one that exactly topk reach
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = thr | (1u << bit);
            int cnt = 0;
#pragma unroll
            for (int i = 0; i < NI; ++i) cnt += __popcll(__ballot(key[i] >= cand));
            if (cnt >= topk) {
                thr = cand;
                if (cnt == topk) break;
            }
        }
        // selected: every key above thr, and of those equal to it the first ones by index
        int above = 0;
#pragma unroll
        for (int i = 0; i < NI; ++i) above += __popcll(__ballot(key[i] > thr));
        const unsigned long long below_me = (1ull << lane) - 1ull;
        int ties = 0, m = 0;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const bool tie = key[i] == thr && key[i] != 0u;
            const unsigned long long tmask = __ballot(tie);
            const bool sel = key[i] > thr || (tie && ties + __popcll(tmask & below_me) < topk - above);
            const unsigned long long smask = __ballot(sel);
            if (sel) {
                const int at = m + __popcll(smask & below_me);
                const uint32_t j = lane + 64 * i;
                // larger = earlier in the reference's sort (choice desc, index asc)
                sc.sel_key[at] = ((unsigned long long)key[i] << 32) | (0xFFFFFFFFu - j);
                sc.pre_sig[at] = sg[i];
            }
            ties += __popcll(tmask);
            m += __popcll(smask);
        }
        wave_sync();
        if (lane < m) {
            const unsigned long long mine = sc.sel_key[lane];
            int rank = 0;
            for (int r = 0; r < m; ++r) rank += sc.sel_key[r] > mine ? 1 : 0;
            sc.sel_id[rank] = (int)(0xFFFFFFFFu - (uint32_t)mine);
            sc.sel_sig[rank] = sc.pre_sig[lane];
        }
        wave_sync();
    }
    // cpu.rs:562-568: sum in selection order, then sig / (sum + f32::EPSILON) * scale
    const int slot = lane < RT_MAX_K ? lane : 0;
    const float my_sig = sc.sel_sig[slot];
    const int my_id = sc.sel_id[slot];
    float sum = 0.0f;
    for (int r = 0; r < topk; ++r) sum = fadd(sum, u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(my_sig), r)));
    if (live && lane < topk) {
        probs[lane] = fmul(fdiv(my_sig, fadd(sum, 1.1920928955078125e-07f)), scaling);
        if (ids_f32) ids_f32[lane] = (float)my_id;
        if (ids_i32) ids_i32[lane] = my_id;
    }
}

template <bool kCoherent>
__device__ __forceinline__ void route_wave(const float* __restrict__ lg, const float* __restrict__ bias, bool live,
                                           int e, int topk, int n_group, int topk_group, float scaling,
                                           RouteScratch& sc, float* __restrict__ probs, float* __restrict__ ids_f32,
                                           int32_t* __restrict__ ids_i32) {
    if (e <= 64) route_wave_ni<kCoherent, false, 1>(lg, 0.0f, bias, live, e, topk, n_group, topk_group, scaling, sc, probs, ids_f32, ids_i32);
    else if (e <= 128) route_wave_ni<kCoherent, false, 2>(lg, 0.0f, bias, live, e, topk, n_group, topk_group, scaling, sc, probs, ids_f32, ids_i32);
    else if (e <= 256) route_wave_ni<kCoherent, false, 4>(lg, 0.0f, bias, live, e, topk, n_group, topk_group, scaling, sc, probs, ids_f32, ids_i32);
    else route_wave_ni<kCoherent, false, 8>(lg, 0.0f, bias, live, e, topk, n_group, topk_group, scaling, sc, probs, ids_f32, ids_i32);
}

// Blocks below route_blocks route four tokens each, a wave per token; the others quantise x (as act_quant_kernel in operand
// order), which needs nothing of the routing: latency bounds the former, HBM the latter, so side by side they take little
// more than the longer of the two.  Layer with two launches / one, us: hidden 2048, 64 experts, 300 tokens 86.5 / 84.4, 1000 tokens two
// terms 135.9 / 132.6; hidden 4096, 128 experts, 300 303.8 / 301.6, 509 two terms 351.0 / 346.6, 2047 723 / 718, 4096 830 / 827.
struct RouteQuant {
    const void* x;
    ActPlanes xq;
    long nblocks;    // of 32 values, 0: none
    int bpr;         // per row
    int route_blocks;
};

template <typename XT, bool kQuant>
__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ logits,
                                                        const float* __restrict__ bias, int n, int e, int topk,
                                                        int n_group, int topk_group, float scaling,
                                                        float* __restrict__ probs, float* __restrict__ ids_f32,
                                                        int32_t* __restrict__ ids_i32, RouteQuant rq) {
    __shared__ RouteScratch scratch[4];
    if (kQuant && (int)blockIdx.x >= rq.route_blocks) {
        const long b = (long)((int)blockIdx.x - rq.route_blocks) * 256 + threadIdx.x;
        if (b < rq.nblocks)
            quant_block_operand_order(static_cast<const XT*>(rq.x), b, rq.bpr, rq.xq.q, rq.xq.s, rq.xq.q2, rq.xq.s2);
        return;
    }
    const int wave = threadIdx.x >> 6;
    const int t = blockIdx.x * 4 + wave;
    const bool live = t < n;
    const size_t tt = live ? t : 0;
    route_wave<false>(logits + tt * e, bias, live, e, topk, n_group, topk_group, scaling, scratch[wave],
                      probs + tt * topk, ids_f32 ? ids_f32 + tt * topk : nullptr,
                      ids_i32 ? ids_i32 + tt * topk : nullptr);
}

// Routing of n tokens and, with xq.q set, the quantisation of their rows of H values.  Parameters as checked by the callers.
int launch_route(const float* logits, const float* bias, int n, int e, int topk, int n_group, int topk_group, float scaling,
                 float* probs, float* ids_f32, int32_t* ids_i32, const void* x, int x_dtype, int H, const ActPlanes& xq, hipStream_t st) {
    const int g = (n_group < 1 || topk_group == n_group) ? 1 : n_group;   // every group kept: the ungrouped router
    RouteQuant rq{x, xq, xq.q ? (long)n * (H / 32) : 0, H / 32, (n + 3) / 4};
    const unsigned grid = (unsigned)(rq.route_blocks + (rq.nblocks + 255) / 256);
    auto go = [&](auto kernel) { kernel<<<grid, 256, 0, st>>>(logits, bias, n, e, topk, g, topk_group, scaling, probs, ids_f32, ids_i32, rq); };
    if (!xq.q) go(moe_route_kernel<float, false>);   // half the registers: 1 us less for a few tokens
    else if (x_dtype == FERRITE_DT_BF16) go(moe_route_kernel<uint16_t, true>);
    else go(moe_route_kernel<float, true>);
    return check_launch("moe_route");
}

// ------------------------------------------------------------------------------------------------
// Stable permutation by expert.  Every token holds each expert at most once, so the assignments of expert e
// in ascending flat index are its tokens in ascending order: rank = number of earlier tokens that chose e.
// Tokens are cut into chunks of 64; per (expert, chunk) a 64-bit membership mask is built with LDS atomics;
// a per-expert prefix over chunks plus a popcount below the token's bit gives the rank, and an exclusive
// scan of the per-expert totals gives the expert's first grouped row.  No global atomics and no dependence
// on scheduling: the tables are a pure function of ids.
//   phase A: masks    phase B: per-expert chunk prefixes, expert scan, active list, unit tables
//   phase C: scatter
// Small n runs A,B,C in one block with the masks in LDS; larger n uses three launches with the masks in the
// caller's scratch.
// ------------------------------------------------------------------------------------------------
constexpr int PM_MAX_E = 512;
constexpr int PM_SMALL_N = 1024;

struct PermArgs {
    const int32_t* ids;
    int n, topk, n_experts;
    int32_t *counts, *starts, *perm_map, *gather_src, *active, *n_active;
    int32_t *unit_expert, *unit_row0, *unit_rows, *unit_first, *unit_count, *n_units;
    int unit_cap, max_units, has_shared;
};

// How an expert's c rows are cut into `units` = ceil(c / cap) units.  With 16-row units the cut is every cap rows.
// The tiled kernels' units are balanced in whole 16-row tiles instead (the first `rem` units hold one tile more than
// the others): the blocks that work on the units of one expert then run at the same pace and fetch the expert's
// weights together, where a nearly empty last unit runs ahead of the full ones and both miss L2.
struct UnitCut {
    int c, cap, base, rem;   // base, rem: tiles per unit and units with one more (tiled kernels only)
    __device__ __forceinline__ UnitCut(int c_, int cap_, int units) : c(c_), cap(cap_), base(0), rem(0) {
        if (cap > 16 && units > 0) {
            const int tiles = (c + 15) >> 4;
            base = tiles / units;
            rem = tiles - base * units;
        }
    }
    __device__ __forceinline__ void span(int i, int& r0, int& rows) const {
        if (cap <= 16) {
            r0 = i * cap;
            rows = min(cap, c - r0);
        } else {
            r0 = (i * base + min(i, rem)) * 16;
            rows = min(c, r0 + (base + (i < rem ? 1 : 0)) * 16) - r0;
        }
    }
};

// wave 0 of a block: exclusive scan over experts + active list. cnt[] readable by the wave; starts_lds [E + 1] and
// first_lds [E + 1] (an expert's first unit) are left for the rest of the block.
__device__ __forceinline__ void perm_expert_scan(const PermArgs& a, const int32_t* cnt, int32_t* starts_lds, int32_t* first_lds) {
    const int lane = threadIdx.x & 63;
    const int E = a.n_experts;
    const int per = (E + 63) >> 6;            // experts per lane (<= 8)
    const int e0 = lane * per;
    const int cap_log = a.unit_cap > 0 ? __builtin_ctz(a.unit_cap) : 0;   // 16, 64 or 128
    int tot = 0, nact = 0, ntile = 0;
    for (int i = 0; i < per; ++i) {
        int e = e0 + i;
        if (e < E) {
            int c = cnt[e];
            tot += c;
            nact += c > 0;
            if (a.unit_cap > 0) ntile += (c + a.unit_cap - 1) >> cap_log;
        }
    }
    const int s_tot = wave_prefix(tot), s_act = wave_prefix(nact), s_tile = wave_prefix(ntile);
    int run = s_tot - tot, ract = s_act - nact, rtile = s_tile - ntile;
    const int total = __builtin_amdgcn_readlane(s_tot, 63), total_act = __builtin_amdgcn_readlane(s_act, 63),
              total_tile = __builtin_amdgcn_readlane(s_tile, 63);
    for (int i = 0; i < per; ++i) {
        int e = e0 + i;
        if (e < E) {
            int c = cnt[e];
            a.counts[e] = c;
            a.starts[e] = run;
            starts_lds[e] = run;
            first_lds[e] = rtile;
            if (c > 0 && a.active) a.active[ract] = e;
            ract += c > 0;
            if (a.unit_cap > 0) rtile += (c + a.unit_cap - 1) >> cap_log;
            run += c;
        }
    }
    if (lane == 0) {
        a.starts[E] = total;
        starts_lds[E] = total;
        first_lds[E] = total_tile;
        if (a.n_active) *a.n_active = total_act;
    }
    if (a.active)
        for (int i = total_act + lane; i < E; i += 64) a.active[i] = -1;
}

// The unit tables, a thread per unit: the expert whose units hold unit u is found in first_lds.  (With the units written by
// the lane that owns their expert, a popular expert's lane wrote dozens while 63 waited: 8192 skewed tokens, 256 experts
// 26.9 -> 21.3 us for the phase.)
__device__ __forceinline__ void perm_units(const PermArgs& a, const int32_t* cnt, const int32_t* starts_lds, const int32_t* first_lds,
                                           int tid, int nthr) {
    if (a.unit_cap <= 0) return;
    const int E = a.n_experts, cap_log = __builtin_ctz(a.unit_cap);
    const int routed = first_lds[E];
    const int shared = a.has_shared ? (a.n + a.unit_cap - 1) >> cap_log : 0;   // all n tokens, rows from n * topk on
    const int total = min(routed + shared, a.max_units);
    for (int u = tid; u < total; u += nthr) {
        int e = E, first = routed, count = shared, rows_all = a.n, row0 = a.n * a.topk;
        if (u < routed) {
            int lo = 0, hi = E;   // the last expert with first_lds <= u (experts without units share their successor's)
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (first_lds[mid] <= u) lo = mid;
                else hi = mid;
            }
            e = lo; first = first_lds[e]; rows_all = cnt[e]; row0 = starts_lds[e];
            count = (rows_all + a.unit_cap - 1) >> cap_log;
        }
        int r0, rows;
        UnitCut(rows_all, a.unit_cap, count).span(u - first, r0, rows);
        a.unit_expert[u] = e;
        a.unit_row0[u] = row0 + r0;
        a.unit_rows[u] = rows;
        if (a.unit_first) { a.unit_first[u] = first; a.unit_count[u] = count; }
    }
    if (tid == 0) *a.n_units = total;
}

// The tables of a single token, by the wave that routed it: lane j < topk holds the j-th selected expert (-1: none).  Every
// selected expert has one row, and its place among them is the number of smaller ids.  Spares the hand-over between blocks and
// the block-wide phases: head of one token 25.5 -> 23.3 us.
__device__ __forceinline__ void permute_one_token(const PermArgs& a, int id) {
    const int lane = threadIdx.x & 63, E = a.n_experts, k = a.topk;
    const bool valid = lane < k && id >= 0 && id < E;
    if (!valid) id = -1;
    const int total = __popcll(__ballot(valid));
    int place = 0;
    for (int q = 0; q < k; ++q) {
        const int other = __builtin_amdgcn_readlane(id, q);
        place += other >= 0 && other < id ? 1 : 0;
    }
    if (lane < k) a.perm_map[lane] = valid ? place : -1;
    if (valid) a.gather_src[place] = lane;
    if (lane >= total && lane < k) a.gather_src[lane] = -1;
    for (int e = lane; e < E; e += 64) {
        int before = 0, count = 0;
        for (int q = 0; q < k; ++q) {
            const int other = __builtin_amdgcn_readlane(id, q);
            before += other >= 0 && other < e ? 1 : 0;
            count += other == e ? 1 : 0;
        }
        a.counts[e] = count;
        a.starts[e] = before;
        if (a.active && e >= total) a.active[e] = -1;
    }
    if (valid && a.active) a.active[place] = id;
    if (lane == 0) {
        a.starts[E] = total;
        if (a.n_active) *a.n_active = total;
    }
    if (a.unit_cap > 0) {
        const int units = total + (a.has_shared ? 1 : 0);
        const bool shared = lane == k && a.has_shared;   // lane k writes the shared expert's unit (k < 64)
        const int u = shared ? total : place;
        if ((valid || shared) && u < a.max_units) {
            a.unit_expert[u] = shared ? E : id;
            a.unit_row0[u] = shared ? k : place;
            a.unit_rows[u] = 1;
            if (a.unit_first) { a.unit_first[u] = u; a.unit_count[u] = 1; }
        }
        if (lane == 0) *a.n_units = min(units, a.max_units);
    }
}

static inline size_t perm_block_lds_bytes(int n, int n_experts) {
    size_t nchunk = ((size_t)n + 63) / 64;
    return (size_t)n_experts * nchunk * 12 + (size_t)(3 * n_experts + 2) * 4;
}

// The whole permutation by one workgroup (any multiple of 64 threads).  lds: perm_block_lds_bytes.
template <bool kCoherent>
__device__ __forceinline__ void permute_in_block(const PermArgs& a, unsigned long long* lds) {
    const int E = a.n_experts, n = a.n, k = a.topk;
    const int nchunk = (n + 63) >> 6;
    unsigned long long* mask = lds;                                      // [E][nchunk]
    int32_t* offs = reinterpret_cast<int32_t*>(mask + (size_t)E * nchunk);  // [E][nchunk]
    int32_t* cnt = offs + (size_t)E * nchunk;                            // [E]
    int32_t* starts_lds = cnt + E;                                       // [E+1]
    int32_t* first_lds = starts_lds + E + 1;                             // [E+1]
    const int tid = threadIdx.x, nthr = blockDim.x;
    auto id_at = [&](int i) -> int { return kCoherent ? load_coherent(a.ids + i) : a.ids[i]; };
    for (int i = tid; i < E * nchunk; i += nthr) mask[i] = 0ull;
    __syncthreads();
    for (int i = tid; i < n * k; i += nthr) {
        int t = i / k;
        int e = id_at(i);
        if (e >= 0 && e < E) atomicOr(&mask[(size_t)e * nchunk + (t >> 6)], 1ull << (t & 63));
    }
    __syncthreads();
    for (int e = tid; e < E; e += nthr) {
        int run = 0;
        for (int c = 0; c < nchunk; ++c) {
            offs[(size_t)e * nchunk + c] = run;
            run += __popcll(mask[(size_t)e * nchunk + c]);
        }
        cnt[e] = run;
    }
    __syncthreads();
    if (tid < 64) perm_expert_scan(a, cnt, starts_lds, first_lds);
    __syncthreads();
    perm_units(a, cnt, starts_lds, first_lds, tid, nthr);
    const int total = starts_lds[E];
    for (int i = tid; i < n * k; i += nthr) {
        int t = i / k;
        int e = id_at(i);
        if (e < 0 || e >= E) { a.perm_map[i] = -1; continue; }
        unsigned long long m = mask[(size_t)e * nchunk + (t >> 6)];
        int g = starts_lds[e] + offs[(size_t)e * nchunk + (t >> 6)] + __popcll(m & ((1ull << (t & 63)) - 1ull));
        a.perm_map[i] = g;
        a.gather_src[g] = i;
    }
    for (int g = total + tid; g < n * k; g += nthr) a.gather_src[g] = -1;
}

__global__ __launch_bounds__(1024) void permute_small_kernel(PermArgs a) {
    extern __shared__ unsigned long long pm_lds[];
    permute_in_block<false>(a, pm_lds);
}

// large-n phase A: one wave per 64-token chunk
__global__ __launch_bounds__(256) void permute_mask_kernel(PermArgs a, unsigned long long* __restrict__ gmask) {
    extern __shared__ unsigned long long pm_lds[];
    const int E = a.n_experts, n = a.n, k = a.topk;
    const int nchunk = (n + 63) >> 6;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunk = blockIdx.x * 4 + wave;
    unsigned long long* m = pm_lds + (size_t)wave * E;
    for (int e = lane; e < E; e += 64) m[e] = 0ull;
    __syncthreads();
    int t = chunk * 64 + lane;
    if (chunk < nchunk && t < n)
        for (int j = 0; j < k; ++j) {
            int e = a.ids[(size_t)t * k + j];
            if (e >= 0 && e < E) atomicOr(&m[e], 1ull << lane);
        }
    __syncthreads();
    if (chunk < nchunk)
        for (int e = lane; e < E; e += 64) gmask[(size_t)chunk * E + e] = m[e];
}

// large-n phase B: one block; thread e walks its chunks.  Masks and prefixes are [chunk][expert], so that neighbouring
// threads touch neighbouring words, sixteen loads in flight: memory latency is what the walk costs (8192 tokens, 256
// experts 21.3 -> 9.6 us against [expert][chunk] with eight).
__global__ __launch_bounds__(512) void permute_scan_kernel(PermArgs a, const unsigned long long* __restrict__ gmask,
                                                           int32_t* __restrict__ goffs) {
    __shared__ int32_t cnt[PM_MAX_E];
    __shared__ int32_t starts_lds[PM_MAX_E + 1], first_lds[PM_MAX_E + 1];
    const int E = a.n_experts;
    const int nchunk = (a.n + 63) >> 6;
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        int run = 0;
        int c = 0;
        for (; c + 16 <= nchunk; c += 16) {
            unsigned long long m[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) m[j] = gmask[(size_t)(c + j) * E + e];
#pragma unroll
            for (int j = 0; j < 16; ++j) { goffs[(size_t)(c + j) * E + e] = run; run += __popcll(m[j]); }
        }
        for (; c < nchunk; ++c) { goffs[(size_t)c * E + e] = run; run += __popcll(gmask[(size_t)c * E + e]); }
        cnt[e] = run;
    }
    __syncthreads();
    if (threadIdx.x < 64) perm_expert_scan(a, cnt, starts_lds, first_lds);
    __syncthreads();
    perm_units(a, cnt, starts_lds, first_lds, threadIdx.x, blockDim.x);
}

// large-n phase C
__global__ __launch_bounds__(256) void permute_scatter_kernel(PermArgs a, const unsigned long long* __restrict__ gmask,
                                                              const int32_t* __restrict__ goffs) {
    const int E = a.n_experts, n = a.n, k = a.topk;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)n * k) return;
    const int total = a.starts[E];
    if ((int)i >= total) a.gather_src[i] = -1;   // positions no assignment reaches (distinct from any g below)
    int t = (int)(i / k);
    int e = a.ids[i];
    if (e < 0 || e >= E) { a.perm_map[i] = -1; return; }
    const size_t at = (size_t)(t >> 6) * E + e;
    unsigned long long m = gmask[at];
    int g = a.starts[e] + goffs[at] + __popcll(m & ((1ull << (t & 63)) - 1ull));
    a.perm_map[i] = g;
    a.gather_src[g] = (int)i;
}

// ------------------------------------------------------------------------------------------------
// The head of the layer as ONE launch (decode-sized batches).
// Workgroups have eight waves.
//   blocks (eb, tg), eb < eblocks: router logits of the tokens of group tg for experts [64 eb, 64 eb + 64): the reference's
//                                  sequential chain, one lane of wave 0 per expert.  A lone wave issues one
//                                  instruction every four cycles, loads and address arithmetic included, so the
//                                  chain wave is left with nothing but the adds: six producer waves fetch the router
//                                  weight (k-blocked transpose [H/4][Epad][4], four chunks ahead), multiply it
//                                  with x[t] (the products are order-independent and each rounded once, as in
//                                  the reference) and hand the products over through a two-buffer LDS ring;
//                                  wave 0 reads them back and adds them in k order.  When one token per
//                                  block would need more than one round of blocks, a block takes two tokens
//                                  (two interleaved chains in wave 0, the weights fetched once for both)
//   blocks (eblocks, t)          : e4m3-per-32 quantisation of x[t] (off the critical path)
//   last logits block of a token : its wave 0 routes the token (arrival counter per token)
//   last routed token            : its block builds the permutation and unit tables with all of its waves (the
//                                  others have been waiting at a barrier for the chain wave's verdict) and clears
//                                  the counters so the next launch (or graph replay) starts clean
// counters[0] = routed tokens, counters[1 + t] = logits blocks of token t that have arrived; all zero on entry.
// ------------------------------------------------------------------------------------------------
constexpr int HEAD_MAX_N = 256;
constexpr int HD_NP = 6;                               // producer waves

struct HeadArgs {
    const void* x;
    const float* wt;      // [H/4][Epad][4]
    const float* bias;
    int n, H, E, Epad, topk, n_group, topk_group;
    float scaling;
    float *logits, *probs, *ids_f32;
    int32_t* ids;
    ActPlanes xq;         // q may be NULL: no quantisation blocks are launched then; q2 set: two-term
    int32_t* counters;    // [1 + n]
    const float* norm_w;  // not NULL: x is the un-normalised f32 stream and every block applies rmsnorm(x, norm_w, eps)
    float eps;            // to its token(s) first (cpu.rs:124-143), so the normalised activations never go through HBM
    PermArgs perm;
};

// T = tokens per block, W = product groups (of four k, all tokens together) per ring buffer.
//   up to 256 blocks (one per CU)  : T 1, W 32 - 64 KiB of ring, the fewest barriers per chain
//   up to 512 blocks               : T 1, W 16 - 32 KiB of ring and under 128 registers, so two blocks share a CU and
//                                    their chain waves run side by side (192 tokens x 2 expert blocks: 44.7 us
//                                    against 60.6 us for two interleaved chains per block)
//   more                           : T 2, W 32 - two interleaved chains per block, the weights fetched once
template <int T, int W>
struct HeadCfg {
    static constexpr int CH = W / T;                         // groups of four k per chunk and token
    static constexpr int PW = (CH + HD_NP - 1) / HD_NP;      // groups per producer wave and chunk
    static constexpr size_t RING_BYTES = 2 * (size_t)W * 1024;
};

template <int T, int W>
struct HeadSet {
    float4 w[HeadCfg<T, W>::PW];
};

// Producer P (0..HD_NP-1) owns groups P, P+HD_NP, ... of every chunk.  Chunks past the end re-read the last one
// (never consumed), which keeps every load unconditional.
template <int T, int W, int P>
__device__ __forceinline__ void head_pload(HeadSet<T, W>& st, const float4* __restrict__ wp, int Epad, int c, int nch) {
    constexpr int CH = HeadCfg<T, W>::CH;
    const float4* base = wp + (size_t)min(c, nch - 1) * CH * Epad;
#pragma unroll
    for (int i = 0; i < HeadCfg<T, W>::PW; ++i)
        if (P + HD_NP * i < CH) st.w[i] = base[(size_t)(P + HD_NP * i) * Epad];
}

// products of the chunk's group j for token ti go to slot (j*T + ti)*64 + lane of the ring buffer
template <int T, int W, int P>
__device__ __forceinline__ void head_pmul(const HeadSet<T, W>& st, const float4* xl, int nk4, int c, float4* buf, int lane) {
    constexpr int CH = HeadCfg<T, W>::CH;
#pragma unroll
    for (int i = 0; i < HeadCfg<T, W>::PW; ++i) {
        const int j = P + HD_NP * i;
        if (j < CH) {
            const float4 wv = st.w[i];
#pragma unroll
            for (int ti = 0; ti < T; ++ti) {
                const float4 xv = xl[ti * nk4 + c * CH + j];
                buf[(j * T + ti) * 64 + lane] =
                    make_float4(fmul(xv.x, wv.x), fmul(xv.y, wv.y), fmul(xv.z, wv.z), fmul(xv.w, wv.w));
            }
        }
    }
}

// rmsnorm of the block's token in place of the first barrier ("x is in LDS") of every wave's role.  On entry every
// thread has staged its share of the raw row in xl and of its squares (each rounded once) in sq.  The reference sums
// the squares of a row left to right in f32 (cpu.rs:124-143): a serial chain, which wave 0 works out (sumsq_chain,
// sumsq_walk) while the producer waves' first weight loads are already in flight.
// Then all waves scale xl to (x * inv) * w, which is what the router chain and the quantisation see.
struct HeadNorm {
    const float* w;
    float eps;
    float4* xl;
    const float4* sq;
    float* inv;   // in LDS
    int nk4;
};

__device__ __forceinline__ void head_first_sync(const HeadNorm& nm) {
    __syncthreads();   // x (and with a norm the squares) are in LDS
    if (nm.w == nullptr) return;
    const int tid = threadIdx.x;
    if (tid < 64) {
        float ss = nm.nk4 <= SUMSQ_SHORT ? sumsq_chain(nm.sq, nm.nk4, 0.0f) : sumsq_walk(nm.sq, nm.nk4, 0.0f);
        ss = fdiv(ss, (float)(nm.nk4 * 4));
        const float inv = fdiv(1.0f, fsqrt(fadd(ss, nm.eps)));
        if (tid == 0) *nm.inv = inv;
    }
    __syncthreads();
    const float iv = *nm.inv;
    for (int i = tid; i < nm.nk4; i += blockDim.x) {
        const float4 v = nm.xl[i], g = reinterpret_cast<const float4*>(nm.w)[i];
        nm.xl[i] = make_float4(fmul(fmul(v.x, iv), g.x), fmul(fmul(v.y, iv), g.y), fmul(fmul(v.z, iv), g.z),
                               fmul(fmul(v.w, iv), g.w));
    }
    __syncthreads();   // the normalised row is in place and the squares' space is free for the products
}

// Products of chunk c+1 are made while the chain consumes chunk c; register set c%4 holds the weights of chunk c
// and is reloaded for chunk c+4 as soon as it has been used.
template <int T, int W, int P>
__device__ __forceinline__ void head_producer(const float4* __restrict__ wp, int Epad, int nk4, const float4* xl,
                                              float4* ring, int lane, const HeadNorm& nm) {
    constexpr int CH = HeadCfg<T, W>::CH;
    const int nch = nk4 / CH;
    float4* b0 = ring;
    float4* b1 = ring + CH * T * 64;
    HeadSet<T, W> s0, s1, s2, s3;
    head_pload<T, W, P>(s0, wp, Epad, 0, nch);
    head_pload<T, W, P>(s1, wp, Epad, 1, nch);
    head_pload<T, W, P>(s2, wp, Epad, 2, nch);
    head_pload<T, W, P>(s3, wp, Epad, 3, nch);
    head_first_sync(nm);   // x is in LDS
    head_pmul<T, W, P>(s0, xl, nk4, 0, b0, lane);
    head_pload<T, W, P>(s0, wp, Epad, 4, nch);
    __syncthreads();
    for (int c = 0; c < nch; c += 4) {
        head_pmul<T, W, P>(s1, xl, nk4, min(c + 1, nch - 1), b1, lane);
        head_pload<T, W, P>(s1, wp, Epad, c + 5, nch);
        __syncthreads();
        head_pmul<T, W, P>(s2, xl, nk4, min(c + 2, nch - 1), b0, lane);
        head_pload<T, W, P>(s2, wp, Epad, c + 6, nch);
        __syncthreads();
        head_pmul<T, W, P>(s3, xl, nk4, min(c + 3, nch - 1), b1, lane);
        head_pload<T, W, P>(s3, wp, Epad, c + 7, nch);
        __syncthreads();
        head_pmul<T, W, P>(s0, xl, nk4, min(c + 4, nch - 1), b0, lane);
        head_pload<T, W, P>(s0, wp, Epad, c + 8, nch);
        __syncthreads();
    }
}

// The chains over one chunk of products: batches of eight LDS reads (8/T groups of four k for each of the T
// tokens), one wait per batch (0xC87F: lgkmcnt <= 8, i.e. everything but the batch just issued; 0xC07F: lgkmcnt 0),
// 32 adds per batch, dependent within a token's chain.
template <int T, int W>
__device__ __forceinline__ void head_consume(float (&s)[T], const float4* buf, int lane) {
    constexpr int NB = HeadCfg<T, W>::CH * T / 8;   // batches per chunk (4)
    float4 r[2][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[0][j] = buf[j * 64 + lane];
#pragma unroll
    for (int g = 0; g < NB; ++g) {
        if (g + 1 < NB) {
#pragma unroll
            for (int j = 0; j < 8; ++j) r[(g + 1) & 1][j] = buf[((g + 1) * 8 + j) * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC87F);
        } else {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC07F);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {   // slot order is (group, token): j % T is the token
            const float4 p = r[g & 1][j];
            float a = s[j % T];
            a = fadd(a, p.x);
            a = fadd(a, p.y);
            a = fadd(a, p.z);
            a = fadd(a, p.w);
            s[j % T] = a;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Barriers pair one to one with head_producer's.
template <int T, int W>
__device__ __forceinline__ void head_consumer(float (&s)[T], int nk4, const float4* ring, int lane, const HeadNorm& nm) {
    constexpr int CH = HeadCfg<T, W>::CH;
    const int nch = nk4 / CH;
    const float4* b0 = ring;
    const float4* b1 = ring + CH * T * 64;
    __builtin_amdgcn_s_setprio(3);   // ahead of another block's producer waves on the same SIMD
    head_first_sync(nm);
    __syncthreads();
    for (int c = 0; c < nch; c += 4) {
        head_consume<T, W>(s, b0, lane);
        __syncthreads();
        if (c + 1 < nch) head_consume<T, W>(s, b1, lane);
        __syncthreads();
        if (c + 2 < nch) head_consume<T, W>(s, b0, lane);
        __syncthreads();
        if (c + 3 < nch) head_consume<T, W>(s, b1, lane);
        __syncthreads();
    }
    __builtin_amdgcn_s_setprio(0);
}

// The barriers of head_producer / head_consumer and nothing else.
template <int T, int W>
__device__ __forceinline__ void head_bystander(int nk4, const HeadNorm& nm) {
    const int nch = nk4 / HeadCfg<T, W>::CH;
    head_first_sync(nm);
    __syncthreads();
    for (int c = 0; c < nch; c += 4) {
        __syncthreads();
        __syncthreads();
        __syncthreads();
        __syncthreads();
    }
}

template <typename XT, int T, int W>
__global__ __launch_bounds__(512) void moe_head_kernel(HeadArgs a) {
    extern __shared__ __align__(16) unsigned char head_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int eb = blockIdx.x, t0 = blockIdx.y * T;
    const int eblocks = a.Epad >> 6;
    const int H = a.H;
    constexpr bool kNorm = sizeof(XT) == 4 && T == 1 && W == 32;   // see head_norm_supported
    if (eb == eblocks) {
        for (int ti = 0; ti < T; ++ti) {
            const int t = t0 + ti;
            if (t >= a.n) break;
            const XT* xrow = static_cast<const XT*>(a.x) + (size_t)t * H;
            if constexpr (kNorm) {
                if (a.norm_w) {
                    // normalise the row in LDS first (the same three steps as in the logits blocks), quantise from there
                    float4* row = reinterpret_cast<float4*>(head_lds + HeadCfg<T, W>::RING_BYTES);
                    float4* sq = reinterpret_cast<float4*>(head_lds);
                    float* inv = reinterpret_cast<float*>(head_lds + HeadCfg<T, W>::RING_BYTES + (size_t)T * H * 4);
                    __syncthreads();   // the previous token's quantisation has read its row
                    for (int i = tid; i < H / 4; i += 512) {
                        const float4 v = reinterpret_cast<const float4*>(xrow)[i];
                        row[i] = v;
                        sq[i] = make_float4(fmul(v.x, v.x), fmul(v.y, v.y), fmul(v.z, v.z), fmul(v.w, v.w));
                    }
                    head_first_sync(HeadNorm{a.norm_w, a.eps, row, sq, inv, H / 4});
                    xrow = reinterpret_cast<const XT*>(row);
                }
            }
            for (int b = tid; b < H / 32; b += 512) {   // the row may be the normalised one in LDS
                const size_t at = (size_t)t * scale_pitch(H) + scale_pos(b), qo = (size_t)t * H + b * 32;
                if (a.xq.q2) {
                    const uint32_t sb = quant_block32_x2(xrow + b * 32, a.xq.q + qo, a.xq.q2 + qo);
                    a.xq.s[at] = (uint8_t)(sb & 0xffu);
                    a.xq.s2[at] = (uint8_t)(sb >> 8);
                } else {
                    a.xq.s[at] = (uint8_t)quant_block32(xrow + b * 32, a.xq.q + qo);
                }
            }
        }
        return;
    }
    float4* ring = reinterpret_cast<float4*>(head_lds);
    float4* xl = reinterpret_cast<float4*>(head_lds + HeadCfg<T, W>::RING_BYTES);   // [T][H/4]
    const int nk4 = H / 4;   // a multiple of 32 (H % 128 == 0)
    const float4* wp = reinterpret_cast<const float4*>(a.wt) + (size_t)eb * 64 + lane;
    for (int i = tid; i < T * nk4; i += 512) {
        const int ti = i / nk4, k4 = i - ti * nk4;
        const XT* xrow = static_cast<const XT*>(a.x) + (size_t)min(t0 + ti, a.n - 1) * H;
        float4 v;
        if constexpr (sizeof(XT) == 4) {
            v = reinterpret_cast<const float4*>(xrow)[k4];
        } else {
            uint2 q = reinterpret_cast<const uint2*>(xrow)[k4];
            v = make_float4(u2f(q.x << 16), u2f(q.x & 0xffff0000u), u2f(q.y << 16), u2f(q.y & 0xffff0000u));
        }
        xl[i] = v;
        if constexpr (kNorm) {
            if (a.norm_w) ring[i] = make_float4(fmul(v.x, v.x), fmul(v.y, v.y), fmul(v.z, v.z), fmul(v.w, v.w));
        }
    }
    const HeadNorm nm{kNorm ? a.norm_w : nullptr, a.eps, xl, ring,
                      reinterpret_cast<float*>(head_lds + HeadCfg<T, W>::RING_BYTES + (size_t)T * H * 4), nk4};
    // wave 0 chains; wave 4 would share its SIMD (and its VALU issue slots) and only keeps the barriers company; the
    // others produce
    float s[T];
#pragma unroll
    for (int ti = 0; ti < T; ++ti) s[ti] = 0.0f;
    switch (wave) {
        case 0: head_consumer<T, W>(s, nk4, ring, lane, nm); break;
        case 1: head_producer<T, W, 0>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        case 2: head_producer<T, W, 1>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        case 3: head_producer<T, W, 2>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        case 5: head_producer<T, W, 3>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        case 6: head_producer<T, W, 4>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        case 7: head_producer<T, W, 5>(wp, a.Epad, nk4, xl, ring, lane, nm); break;
        default: head_bystander<T, W>(nk4, nm); break;
    }
    // From here on wave 0 works alone (LDS is free for its scratch); the other waves wait at the barrier below and join
    // in if this block turns out to be the one that routed the last token.
    __shared__ int perm_here;
    int do_perm = 0;
    if (wave == 0) {
        const int e = eb * 64 + lane;
#pragma unroll
        for (int ti = 0; ti < T; ++ti) {
            const int t = t0 + ti;
            if (t >= a.n) break;
            if (e < a.E) a.logits[(size_t)t * a.E + e] = s[ti];
            RouteScratch& sc = *reinterpret_cast<RouteScratch*>(head_lds);
            float *probs = a.probs + (size_t)t * a.topk, *ids_f32 = a.ids_f32 + (size_t)t * a.topk;
            int32_t* ids = a.ids + (size_t)t * a.topk;
            int last = 0;
            if (T == 1 && eblocks == 1) {   // the token's logits are this wave's: nobody to wait for (two tokens a block: eblocks > 2)
                wave_sync();
                route_wave_ni<false, true, 1>(nullptr, s[ti], a.bias, true, a.E, a.topk, a.n_group, a.topk_group, a.scaling, sc, probs,
                                              ids_f32, ids);
            } else {
                // arrival: the stores above are made visible before the counter moves
                __threadfence();
                if (lane == 0) last = atomicAdd(&a.counters[1 + t], 1) == eblocks - 1;
                last = __shfl(last, 0, 64);
                if (!last) continue;
                __threadfence();
                wave_sync();
                route_wave<true>(a.logits + (size_t)t * a.E, a.bias, true, a.E, a.topk, a.n_group, a.topk_group,
                                 a.scaling, sc, probs, ids_f32, ids);
            }
            if (a.n == 1) {   // the tables follow from what this wave holds: no other block has a part in them
                if (eblocks > 1 && lane < 2) a.counters[lane] = 0;
                permute_one_token(a.perm, lane < RT_MAX_K ? sc.sel_id[lane] : -1);
                continue;
            }
            __threadfence();
            last = 0;
            if (lane == 0) last = atomicAdd(&a.counters[0], 1) == a.n - 1;
            last = __shfl(last, 0, 64);
            if (!last) continue;
            __threadfence();
            wave_sync();
            do_perm = 1;
            for (int i = lane; i < a.n + 1; i += 64) a.counters[i] = 0;
        }
        if (lane == 0) perm_here = do_perm;
    }
    __syncthreads();
    if (perm_here) permute_in_block<true>(a.perm, reinterpret_cast<unsigned long long*>(head_lds));
}

// tokens per block: two when one per block would not fit the chip's 256 CUs in one round
// (tokens per block, ring width) for n tokens x eblocks blocks of 64 experts: see HeadCfg.
struct HeadShape { int T, W; };
static HeadShape head_shape(int n, int eblocks) {
    const long blocks = (long)n * eblocks;
    // (the quantisation blocks, one more per token, are short but take a block slot each while they run: 96 tokens
    // x 2 blocks run in one round beside theirs, 37 us; 128 x 2 did not, 58 us against 44 us with the narrow ring)
    if (blocks + n / 2 <= 256) return {1, 32};
    if (blocks <= 512) return {1, 16};
    return {2, 32};
}

static size_t head_lds_bytes(int n, int H, int E) {
    const HeadShape hs = head_shape(n, (E + 63) / 64);
    size_t b = 2 * (size_t)hs.W * 1024 + (size_t)hs.T * H * 4 + 64;   // ring, x rows, the rows' 1/rms
    if (b < sizeof(RouteScratch)) b = sizeof(RouteScratch);
    const size_t p = perm_block_lds_bytes(n, E);
    if (p > b) b = p;
    return b;
}

// The fused rmsnorm keeps the squares of the block's row where the product ring will be.  Every block of a token
// works out that token's sum of squares again, which pays while each block has a CU to itself (32 tokens, H 4096: the
// block call 4 us shorter than with rmsnorm as a launch of its own).  With two blocks on a CU it gains and loses (H 4096,
// 128 experts: 128 tokens 99 against 103 us, 192 tokens 109 and 111 against 110 and 111, 250 tokens 131 against 128):
// offered for the one-block-per-CU shape only.
bool head_norm_supported(int n, int H, int E) {
    if (!head_supported(n, H, E)) return false;
    const HeadShape hs = head_shape(n, (E + 63) / 64);
    return hs.T == 1 && hs.W == 32 && (size_t)hs.T * H * 4 <= 2 * (size_t)hs.W * 1024;
}

bool head_supported(int n, int H, int E) {
    return n <= HEAD_MAX_N && E <= RT_MAX_E && (H % 128) == 0 && head_lds_bytes(n, H, E) <= 160 * 1024 - 64;   // 64: the kernel's static LDS
}

template <typename XT, int T, int W>
static int launch_head_tt(const HeadArgs& a, int quant, size_t lds, hipStream_t st) {
    int rc = LdsLimit<&moe_head_kernel<XT, T, W>>::ensure(lds);
    if (rc) return rc;
    dim3 grid(a.Epad / 64 + quant, (a.n + T - 1) / T);
    moe_head_kernel<XT, T, W><<<grid, 512, lds, st>>>(a);
    return check_launch("moe_head");
}

template <typename XT>
static int launch_head_t(const HeadArgs& a, int quant, size_t lds, hipStream_t st) {
    const HeadShape hs = head_shape(a.n, a.Epad / 64);
    if (hs.T == 2) return launch_head_tt<XT, 2, 32>(a, quant, lds, st);
    if (hs.W == 16) return launch_head_tt<XT, 1, 16>(a, quant, lds, st);
    return launch_head_tt<XT, 1, 32>(a, quant, lds, st);
}

int launch_moe_head(const void* x, int x_dtype, const float* router_t, const float* bias, const ferrite_moe_shape& s,
                    int n, float* logits, float* probs, float* ids_f32, int32_t* ids, const ActPlanes& xq,
                    int32_t* counters, int32_t* counts, int32_t* starts, int32_t* perm_map, int32_t* gather_src,
                    int32_t* active, int32_t* n_active, const UnitTables& units, const float* norm_w,
                    float eps, hipStream_t st) {
    if (!head_supported(n, s.hidden, s.n_experts)) return FERRITE_DECLINED;
    if (norm_w && (x_dtype != FERRITE_DT_F32 || !head_norm_supported(n, s.hidden, s.n_experts))) return FERRITE_DECLINED;
    HeadArgs a{};
    a.x = x; a.wt = router_t; a.bias = bias;
    a.n = n; a.H = s.hidden; a.E = s.n_experts; a.Epad = (s.n_experts + 63) / 64 * 64; a.topk = s.topk;
    a.n_group = (s.n_group > 1 && s.topk_group < s.n_group) ? s.n_group : 1;
    a.topk_group = s.topk_group; a.scaling = s.routed_scaling;
    a.logits = logits; a.probs = probs; a.ids_f32 = ids_f32; a.ids = ids; a.xq = xq; a.counters = counters;
    a.norm_w = norm_w; a.eps = eps;
    PermArgs& p = a.perm;
    p.ids = ids; p.n = n; p.topk = s.topk; p.n_experts = s.n_experts;
    p.counts = counts; p.starts = starts; p.perm_map = perm_map; p.gather_src = gather_src;
    p.active = active; p.n_active = n_active; p.has_shared = s.shared_inter > 0;
    p.unit_expert = units.unit_expert; p.unit_row0 = units.unit_row0; p.unit_rows = units.unit_rows;
    p.unit_first = units.unit_first; p.unit_count = units.unit_count;
    p.n_units = units.n_units; p.unit_cap = units.unit_rows_cap; p.max_units = units.max_units;
    const size_t lds = head_lds_bytes(n, s.hidden, s.n_experts);
    if (x_dtype == FERRITE_DT_F32) return launch_head_t<float>(a, xq.q ? 1 : 0, lds, st);
    if (x_dtype == FERRITE_DT_BF16) return launch_head_t<uint16_t>(a, xq.q ? 1 : 0, lds, st);
    return FERRITE_ERR_INVALID_ARG;
}

// What every routing kernel here assumes of its parameters, for the stand-alone op and for the fused head alike:
// argument errors first (the reference returns Err for them, cpu.rs:539-545), then the limits of these kernels
// (eight slots of 64 experts and an LDS array of RT_MAX_E choices, RT_MAX_K selections, one lane per group) as FERRITE_DECLINED.
int check_routing_params(int e, int topk, int n_group, int topk_group) {
    if (e <= 0 || topk <= 0 || topk > e) return FERRITE_ERR_INVALID_ARG;
    if (n_group > 1) {
        if (e % n_group != 0 || topk_group < 1 || topk_group > n_group) return FERRITE_ERR_INVALID_ARG;
        if (topk > topk_group * (e / n_group)) return FERRITE_ERR_INVALID_ARG;
        if (n_group > 64) return FERRITE_DECLINED;
    }
    if (e > RT_MAX_E || topk > RT_MAX_K) return FERRITE_DECLINED;
    return FERRITE_OK;
}

template <typename XT>
static int warmup_head() {
    const size_t cap = kLdsCap - 64;   // 64: the kernel's static LDS
    int rc;
    if ((rc = LdsLimit<&moe_head_kernel<XT, 1, 32>>::ensure(cap))) return rc;
    if ((rc = LdsLimit<&moe_head_kernel<XT, 1, 16>>::ensure(cap))) return rc;
    return LdsLimit<&moe_head_kernel<XT, 2, 32>>::ensure(cap);
}

int warmup_route() {
    int rc;
    if ((rc = warmup_head<float>())) return rc;
    return warmup_head<uint16_t>();
}

// Router GEMM alone from the transposed weight (any n): logits only.
int launch_router_chain(const void* x, int x_dtype, const float* router_t, int n, int H, int E, float* logits,
                        hipStream_t st) {
    if (H % 128 != 0 || n <= 0 || n > 65535) return FERRITE_DECLINED;
    ChainArgs a{x, router_t, nullptr, logits, n, H, E, (E + 63) / 64 * 64, 0};
    if (x_dtype == FERRITE_DT_F32) return launch_chain<float, true>(a, st);
    if (x_dtype == FERRITE_DT_BF16) return launch_chain<uint16_t, true>(a, st);
    return FERRITE_ERR_INVALID_ARG;
}

// router weight [E][H] -> k-blocked transpose [H/4][Epad][4], zero padded
__global__ __launch_bounds__(256) void router_transpose_kernel(const float* __restrict__ w, int E, int Epad, int H,
                                                               float4* __restrict__ dst) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)(H / 4) * Epad) return;
    int e = (int)(idx % Epad);
    size_t k4 = idx / Epad;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (e < E) v = *reinterpret_cast<const float4*>(w + (size_t)e * H + k4 * 4);
    dst[idx] = v;
}

int launch_router_transpose(const float* w, int E, int H, float* dst, hipStream_t st) {
    const int Epad = (E + 63) / 64 * 64;
    size_t total = (size_t)(H / 4) * Epad;
    router_transpose_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>(w, E, Epad, H, reinterpret_cast<float4*>(dst));
    return check_launch("router_transpose");
}

__global__ void zero_i32_kernel(int32_t* p, int count) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = 0;
}

int launch_zero_i32(int32_t* p, int count, hipStream_t st) {
    if (count <= 0) return FERRITE_OK;
    zero_i32_kernel<<<(count + 255) / 256, 256, 0, st>>>(p, count);
    return check_launch("zero_i32");
}

size_t perm_scratch_bytes(int n, int n_experts) {
    size_t nchunk = ((size_t)n + 63) / 64;
    return (size_t)n_experts * nchunk * (8 + 4) + 64;
}

int launch_permute(const int32_t* ids, int n, int topk, int n_experts, int32_t* counts, int32_t* starts,
                   int32_t* perm_map, int32_t* gather_src, int32_t* active, int32_t* n_active, void* scratch,
                   size_t scratch_bytes, const UnitTables* units, int has_shared, hipStream_t st) {
    if (n <= 0 || topk <= 0 || n_experts <= 0 || n_experts > PM_MAX_E) return FERRITE_ERR_INVALID_ARG;
    PermArgs a{};
    a.ids = ids; a.n = n; a.topk = topk; a.n_experts = n_experts;
    a.counts = counts; a.starts = starts; a.perm_map = perm_map; a.gather_src = gather_src;
    a.active = active; a.n_active = n_active; a.has_shared = has_shared;
    if (units) {
        a.unit_expert = units->unit_expert; a.unit_row0 = units->unit_row0; a.unit_rows = units->unit_rows;
        a.unit_first = units->unit_first; a.unit_count = units->unit_count;
        a.n_units = units->n_units; a.unit_cap = units->unit_rows_cap; a.max_units = units->max_units;
    }
    const int nchunk = (n + 63) / 64;
    const size_t lds = perm_block_lds_bytes(n, n_experts);
    // one block while its masks, prefixes, counts and starts take at most 60 KiB: such calls need no scratch.  With the
    // units' starts, E + 1 words more, 64 KiB are enough for every E up to PM_MAX_E.
    static_assert(60 * 1024 + (PM_MAX_E + 1) * 4 <= 64 * 1024, "the block's tables fit the LDS of a plain launch");
    if (n <= PM_SMALL_N && lds - (size_t)(n_experts + 1) * 4 <= 60 * 1024) {
        permute_small_kernel<<<1, 1024, lds, st>>>(a);
        return check_launch("permute_small");
    }
    if (scratch == nullptr || scratch_bytes < perm_scratch_bytes(n, n_experts)) return FERRITE_ERR_WORKSPACE;
    unsigned long long* gmask = reinterpret_cast<unsigned long long*>(scratch);
    int32_t* goffs = reinterpret_cast<int32_t*>(gmask + (size_t)n_experts * nchunk);
    permute_mask_kernel<<<(nchunk + 3) / 4, 256, (size_t)4 * n_experts * 8, st>>>(a, gmask);
    int rc = check_launch("permute_mask");
    if (rc) return rc;
    permute_scan_kernel<<<1, 512, 0, st>>>(a, gmask, goffs);
    rc = check_launch("permute_scan");
    if (rc) return rc;
    size_t na = (size_t)n * topk;
    permute_scatter_kernel<<<(unsigned)((na + 255) / 256), 256, 0, st>>>(a, gmask, goffs);
    return check_launch("permute_scatter");
}

}  // namespace fe

using namespace fe;

extern "C" int ferrite_matmul_f32(const float* x, const float* w, const float* bias, float* out, int n, int k,
                                  int o, ferrite_stream_t stream) {
    if (n < 0 || k < 0 || o < 0) return FERRITE_ERR_INVALID_ARG;
    if (n == 0 || o == 0) return FERRITE_OK;
    if ((n > 0 && !x) || !w || !out) return FERRITE_ERR_INVALID_ARG;
    hipStream_t st = as_stream(stream);
    if (k > 0 && (k & 3) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && (size_t)n * o >= 1024)
        return launch_matmul_exact(x, FERRITE_DT_F32, w, bias, out, n, k, o, st);
    size_t total = (size_t)n * o;
    matmul_exact_simple_kernel<<<(unsigned)((total + 63) / 64), 64, 0, st>>>(x, w, bias, out, n, k, o);
    return check_launch("matmul_exact_simple");
}

extern "C" int ferrite_swiglu_limited_f32(const float* gate_up, float limit, float* out, int n, int inter,
                                          ferrite_stream_t stream) {
    if (n < 0 || inter < 0) return FERRITE_ERR_INVALID_ARG;
    size_t total = (size_t)n * inter;
    if (total == 0) return FERRITE_OK;
    if (!gate_up || !out) return FERRITE_ERR_INVALID_ARG;
    swiglu_kernel<<<(unsigned)((total + 255) / 256), 256, 0, as_stream(stream)>>>(gate_up, limit, out, n, inter);
    return check_launch("swiglu");
}

extern "C" int ferrite_moe_route(const float* logits, const float* bias, int n, int e, int topk, int n_group,
                                 int topk_group, float routed_scaling, float* probs, float* ids_f32,
                                 int32_t* ids_i32, ferrite_stream_t stream) {
    if (n < 0 || !logits || !probs) return FERRITE_ERR_INVALID_ARG;
    if (int rc = check_routing_params(e, topk, n_group, topk_group)) return rc;
    if (n == 0) return FERRITE_OK;
    return launch_route(logits, bias, n, e, topk, n_group, topk_group, routed_scaling, probs, ids_f32, ids_i32, nullptr, FERRITE_DT_F32, 0,
                        ActPlanes{nullptr, nullptr, nullptr, nullptr}, as_stream(stream));
}

extern "C" size_t ferrite_moe_permute_scratch_bytes(int n, int topk, int n_experts) {
    if (n <= 0 || topk <= 0 || n_experts <= 0 || (long long)n * topk > 0x3fffffffLL) return 0;
    return perm_scratch_bytes(n * topk, n_experts);
}

extern "C" int ferrite_moe_permute(const int32_t* ids, int n, int topk, int n_experts, int32_t* counts,
                                   int32_t* starts, int32_t* perm_map, int32_t* gather_src, int32_t* active,
                                   int32_t* n_active, void* scratch, size_t scratch_bytes,
                                   ferrite_stream_t stream) {
    if (!ids || !counts || !starts || !perm_map || !gather_src) return FERRITE_ERR_INVALID_ARG;
    if (n <= 0 || topk <= 0 || (long long)n * topk > 0x3fffffffLL) return FERRITE_ERR_INVALID_ARG;
    // The kernels rank an assignment by the earlier *tokens* that chose its expert, which is right when a token
    // holds each expert at most once (what a router emits).  This stand-alone op promises nothing about its ids
    // (the reference's own vector, chain_dev.rs:25042, lists an expert twice in one token), so it runs them with
    // every assignment as a token of its own: flat index, tables and order are the same, duplicates rank by slot.
    return launch_permute(ids, n * topk, 1, n_experts, counts, starts, perm_map, gather_src, active, n_active, scratch,
                          scratch_bytes, nullptr, 0, as_stream(stream));
}
