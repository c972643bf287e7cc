// Linear-layer kernels for MI355X (gfx950): weight gradients, weight casts and the SwiGLU activation.
//
// Weight gradients: dW = dY^T X, fp32 sums and result.
// The contraction runs over the tokens, which are the rows of both operands, so both MFMA operands are columns of
// row-major tiles: tiles move global -> LDS by DMA (tiles.h) and are read with ds_read_b64_tr_b16; nothing is
// transposed in memory. A weight gradient of this model is a small matrix with a long contraction (768 x 768 over
// 8192 tokens): its 128 x 128 tiles are 36 blocks for 256 CUs, so the tokens are split over `nsplit` blocks per tile,
// whose fp32 partials wgrad_sum_kernel adds in split order (no atomics).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <string>

#include "nanonemo_linear.h"
#include "tiles.h"

#define NNLIN_API extern "C" __attribute__((visibility("default")))

namespace {

constexpr int kTN = 128, kTK = 128, kTT = 64;  // a block's tile of dW, and the tokens of one stage
constexpr int kSub = kTT * 64;                  // elements of a 64-column half of an operand's stage

struct Outs {
    float* p[3];
    int end[3];  // rows below end[0] go to p[0], then to p[1], p[2]
};
__device__ inline float* out_row(const Outs& o, int n, int K) {
    const int i = n < o.end[0] ? 0 : n < o.end[1] ? 1 : 2;
    return o.p[i] + (size_t)(n - (i ? o.end[i - 1] : 0)) * K;
}

// One operand of a block: 128 columns of a row-major matrix, copied kTT rows at a time. The address and the extent of
// readable memory advance by scalar adds (recomputed from the stage's index, with branches for the edges, they took
// longer than the stage's products). The extent ends at the last row's last column; what lies past it reads as zeros,
// and so does a half whose columns lie past the matrix's width. Columns past the width before the last row read the
// next row's values: they only reach rows and columns of dW that are not stored.
struct Operand {
    uint64_t at;      // the first half's first element of the next stage
    uint32_t step;    // bytes from a stage to the next
    int ld2;          // bytes of a row
    int width[2];     // bytes from the half's first column to the end of a row (very negative: no such column)
    __device__ void init(const u16* p, long long ld, int t0, int col, int cols) {
        at = reinterpret_cast<uint64_t>(p + t0 * ld + col);
        ld2 = (int)ld * 2;
        step = kTT * ld2;
        width[0] = 2 * (cols - col);
        width[1] = cols > col + 64 ? 2 * (cols - col - 64) : -(1 << 30);
    }
    // This wave's copies of the next stage into two half tiles, and on to the one after. left: rows from the stage's
    // first to the end (0 or less: none).
    __device__ void copy(int left, u16* lds, int wave, const DmaOffs<64, kTT, 8>& fo) {
#if defined(__HIP_DEVICE_COMPILE__)
        const int body = __builtin_amdgcn_readfirstlane((min(left, kTT) - 1) * ld2);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32)), lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
        const uint64_t base = ((uint64_t)hi << 32) | lo;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            void* g = reinterpret_cast<void*>(base + 128 * h);
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(g, 0, left > 0 ? max(0, body + width[h]) : 0, kBufWord3);
#pragma unroll
            for (int it = 0; it < DmaOffs<64, kTT, 8>::N; ++it)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_AS(void, lds + h * kSub + (it * 8 + wave) * 512), 16, fo.o[it], 0, 0, 0);
        }
        at = base + step;
#endif
    }
};

// Block = 8 waves on one 128 x 128 tile of dW: waves 0-3 take the first 32 tokens of every 64-token stage and
// waves 4-7 the other 32 (two waves per SIMD on one tile's copies; the halves are added through LDS at the end), each
// wave a 64 x 64 quarter as 2 x 2 products of 32 x 32. A = columns of dY (rows of dW), B = columns of X, so that a
// store instruction covers 32 consecutive floats of two rows. Four stages of 32 KB, three in flight.
// Bound: a stage is 512 MFMA cycles per SIMD beside 64 KB of transposing LDS reads (about 580 cycles per CU) and the
// scalar work of its copies; it takes about 1300. Measured with the sum kernel, against the library's bf16 product
// and cast, 8192 tokens: 768 x 768 22 us (51), 1280 x 768 27 (54), 4096 x 768 61 (82), 768 x 2048 38 (65); an earlier
// form with two 64 KB buffers and branching edge tests: 24, 30, 77, 48.
template <int DT>
__global__ __launch_bounds__(512, 2) void wgrad_kernel(const u16* __restrict__ dY, long long ldy,
                                                       const u16* __restrict__ X, long long ldx, int T, int N, int K,
                                                       int ntk, int tiles, int nsplit, float* __restrict__ part,
                                                       Outs outs) {
    using E = Elem<DT>;
    __shared__ __attribute__((aligned(16))) u16 b0[4 * kSub];  // a stage: two halves of dY, two of X
    __shared__ __attribute__((aligned(16))) u16 b1[4 * kSub];
    __shared__ __attribute__((aligned(16))) u16 b2[4 * kSub];
    __shared__ __attribute__((aligned(16))) u16 b3[4 * kSub];
    // Blocks go to the 8 XCDs round-robin; each XCD takes a run of consecutive work items, ordered by split, so that
    // the tiles that read the same tokens share them in that XCD's L2.
    const int nb = tiles * nsplit, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int item = xcd * (nb >> 3) + min(xcd, nb & 7) + slot;
    const int sp = item / tiles, tile = item - sp * tiles;
    const int n0 = tile / ntk * kTN, k0 = tile % ntk * kTK;
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5, g16 = (lane >> 4) & 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, wn = (wave >> 1) & 1, wk = wave & 1;
    // This split's stages [first, last): whole groups of four, so that the loop has no exits (only the last group can
    // run past T).
    const int ng = (T + 4 * kTT - 1) / (4 * kTT);
    const int first = 4 * (int)((long long)sp * ng / nsplit), last = 4 * (int)((long long)(sp + 1) * ng / nsplit);

    const DmaOffs<64, kTT, 8> yo = dma_offsets<64, kTT, 8>(lane, wave, (int)ldy);
    const DmaOffs<64, kTT, 8> xo = dma_offsets<64, kTT, 8>(lane, wave, (int)ldx);
    constexpr int kOps = 4 * DmaOffs<64, kTT, 8>::N;  // copy instructions of a stage per wave
    Operand oy, ox;
    oy.init(dY, ldy, first * kTT, n0, N);
    ox.init(X, ldx, first * kTT, k0, K);
    int left = min(T, last * kTT) - first * kTT;  // rows from the next stage's first to the split's end
    auto issue = [&](u16* st) {
        oy.copy(left, st, wave, yo);
        ox.copy(left, st + 2 * kSub, wave, xo);
        left -= kTT;
    };
    int coff[2][2];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int x = 0; x < 2; ++x) coff[dt][x] = col_off<64>(8 * x + 4 * hh, 32 * dt + 16 * g16, lane) + kTT / 2 * 64 * grp;

    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = f32x16{};
    auto compute = [&](const u16* st) {
        const u16 *yw = st + wn * kSub, *xw = st + (2 + wk) * kSub;
#pragma unroll
        for (int c = 0; c < kTT / 32; ++c) {
            u16x8 a[2], b[2];
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) {
                a[dt] = cat4(ld_tr(yw + 16 * c * 64 + coff[dt][0]), ld_tr(yw + 16 * c * 64 + coff[dt][1]));
                b[dt] = cat4(ld_tr(xw + 16 * c * 64 + coff[dt][0]), ld_tr(xw + 16 * c * 64 + coff[dt][1]));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = E::mfma(a[i], b[j], acc[i][j]);
        }
    };
    // One stage: wait for its copies (issued three stages ago; copies complete in issue order, so those of the two
    // stages after it stay in flight), meet the other waves, start the third stage after it into the buffer that every
    // wave has now finished reading, and compute. The barrier orders LDS only. Stages past the end copy zeros.
    auto stage = [&](const u16* cur, u16* next) {
        wait_vmem_keep<2 * kOps>();
        barrier_lds();
        issue(next);
        compute(cur);
    };
    issue(b0);
    issue(b1);
    issue(b2);
    for (int it = first; it < last; it += 4) {
        stage(b0, b3);
        stage(b1, b0);
        stage(b2, b1);
        stage(b3, b2);
    }
    wait_vmem();

    // The two token halves: each wave hands the other group's wave of its quarter one of its two 32-row slabs (waves
    // 0-3 keep slab 0) and adds the one it receives, first half plus second in both. A slab is 32 floats per lane;
    // the slabs of a group fill 32 KB, so the groups use one tile array each.
    __syncthreads();
    float* mine = reinterpret_cast<float*>(grp ? b1 : b0) + (wave & 3) * 2048;
    const float* theirs = reinterpret_cast<const float*>(grp ? b0 : b1) + (wave & 3) * 2048;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x16& v = grp ? acc[0][j] : acc[1][j];
            reinterpret_cast<f32x4*>(mine)[(4 * j + g) * 64 + lane] = f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
        }
    __syncthreads();
    const int nrow = n0 + 64 * wn + 32 * grp, kcol = k0 + 64 * wk + l32;
    float* pb = part + (size_t)sp * N * K;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 o = reinterpret_cast<const f32x4*>(theirs)[(4 * j + g) * 64 + lane];
            const f32x16& v = grp ? acc[1][j] : acc[0][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = nrow + 8 * g + 4 * hh + e, k = kcol + 32 * j;
                if (n < N && k < K) {
                    float* row = nsplit > 1 ? pb + (size_t)n * K : out_row(outs, n, K);
                    row[k] = v[4 * g + e] + o[e];
                }
            }
        }
}

// dW = the sum over splits s = 0, 1, ... of part[s], four values per thread.
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const float* __restrict__ part, int nsplit, int N, int K,
                                                        Outs outs) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // N K / 4 fits in 31 bits
    const int kq = K / 4;
    if (i >= N * kq) return;
    const int n = i / kq, k = (i - n * kq) * 4;
    const size_t per = (size_t)N * K;
    const float* p = part + (size_t)n * K + k;
    f32x4 acc = *reinterpret_cast<const f32x4*>(p);
    int s = 1;
    for (; s + 4 <= nsplit; s += 4) {  // four loads in flight, added in split order
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4*>(p + (s + u) * per);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += v[u];
    }
    for (; s < nsplit; ++s) acc += *reinterpret_cast<const f32x4*>(p + s * per);
    *reinterpret_cast<f32x4*>(out_row(outs, n, K) + k) = acc;
}

// A layer's fp32 weights to 16 bits, round to nearest even, eight elements per thread. One launch for up to four
// weights: each is a few MB (0.8 us of traffic), so the launches would cost more than the copies.
struct Casts {
    const float* src[4];
    u16* dst[4];
    int end[4];  // vectors of 8 up to the end of array i
};
template <int DT>
__global__ __launch_bounds__(256) void cast_kernel(Casts c) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= c.end[3]) return;
    const int a = i < c.end[0] ? 0 : i < c.end[1] ? 1 : i < c.end[2] ? 2 : 3;
    const int v = i - (a ? c.end[a - 1] : 0);
    const f32x4* s = reinterpret_cast<const f32x4*>(c.src[a]) + 2 * (size_t)v;
    const f32x4 x = s[0], y = s[1];
    reinterpret_cast<u32x4*>(c.dst[a])[v] = u32x4{Elem<DT>::pack2(x[0], x[1]), Elem<DT>::pack2(x[2], x[3]),
                                                  Elem<DT>::pack2(y[0], y[1]), Elem<DT>::pack2(y[2], y[3])};
}

// The same with a transposed copy beside each, for a training step: the products for the inputs' gradients contract over
// the weights' rows, and the library's products are the faster ones where that is the contiguous dimension of both
// operands. 8192 tokens, bf16, rows against transposed: 4096 x 768 64 us to 51, 768 x 2048 29 to 25, 1280 x 768 24.5 to
// 21.8, 768 x 768 18.5 to 15.5; 512 tokens 19.5 to 13.7, 8.2 to 6.9, 9.2 to 7.0, 7.1 to 6.1; 50304 x 768 542 to 488. It
// was the faster one at every size measured, 128 to 16384 tokens. HBM-bound, one read and two
// writes: an MLP of 768 x 2048 6.6 us (38 MB, 5.7 TB/s; without the transposed copy 4.5), 50304 x 768 52 us (309 MB,
// 5.9 TB/s; 33).
// A block turns a 64 x 64 tile through LDS, rows padded to 66 elements: a wave's transposing stores (8 rows, 8 columns
// apart) then fall into 64 different banks.
struct Turns {
    const float* src[4];
    u16 *dst[4], *dst_t[4];
    int rows[4], cols[4], ldt[4];
    int end[4];  // tiles up to the end of array i
};
template <int DT>
__global__ __launch_bounds__(256) void cast_both_kernel(Turns c) {
    constexpr int kLd = 66;
    __shared__ uint32_t tile[64 * kLd / 2];
    u16* const t = reinterpret_cast<u16*>(tile);
    const int b = blockIdx.x, a = b < c.end[0] ? 0 : b < c.end[1] ? 1 : b < c.end[2] ? 2 : 3;
    const int i = b - (a ? c.end[a - 1] : 0), rows = c.rows[a], cols = c.cols[a], ntc = (cols + 63) / 64;
    const int r0 = i / ntc * 64, c0 = i % ntc * 64;
    const int hi = threadIdx.x >> 3, lo = (threadIdx.x & 7) * 8;
#pragma unroll
    for (int p = 0; p < 64; p += 32) {
        const int r = p + hi;
        if (r0 + r >= rows || c0 + lo >= cols) continue;  // both are multiples of 8
        const size_t at = (size_t)(r0 + r) * cols + c0 + lo;
        const f32x4 x = *reinterpret_cast<const f32x4*>(c.src[a] + at), y = *reinterpret_cast<const f32x4*>(c.src[a] + at + 4);
        const u32x4 v = {Elem<DT>::pack2(x[0], x[1]), Elem<DT>::pack2(x[2], x[3]), Elem<DT>::pack2(y[0], y[1]),
                         Elem<DT>::pack2(y[2], y[3])};
        *reinterpret_cast<u32x4*>(c.dst[a] + at) = v;
        const u16x8 e = __builtin_bit_cast(u16x8, v);
#pragma unroll
        for (int k = 0; k < 8; ++k) t[(lo + k) * kLd + r] = e[k];
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 64; p += 32) {
        const int col = p + hi;
        if (c0 + col >= cols || r0 + lo >= rows) continue;
        const uint32_t* w = tile + (col * kLd + lo) / 2;
        *reinterpret_cast<u32x4*>(c.dst_t[a] + (size_t)(c0 + col) * c.ldt[a] + r0 + lo) = u32x4{w[0], w[1], w[2], w[3]};
    }
}

// SwiGLU forward and backward, eight columns per thread: every input is read once and every output written once, where
// PyTorch's silu, mul and their backwards move 2.5 times the bytes (8192 x 2048: 34 us forward and 50 backward).
// HBM-bound; 8192 x 2048: forward 15 us (100 MB, 6.8 TB/s, partly from the last-level cache), backward 24 us (168 MB, 7.0);
// 32768 x 2048: 68 us (5.9 TB/s) and 116 us (5.8); a 1 GiB device copy runs at 5.1 TB/s.
template <int DT>
__device__ inline void widen8(const u16* p, float* v) {
    const u16x8 w = ld8(p);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = Elem<DT>::to_f32(w[e]);
}
template <int DT>
__device__ inline void round8(u16* p, const float* v) {
    *reinterpret_cast<u32x4*>(p) = u32x4{Elem<DT>::pack2(v[0], v[1]), Elem<DT>::pack2(v[2], v[3]),
                                         Elem<DT>::pack2(v[4], v[5]), Elem<DT>::pack2(v[6], v[7])};
}
__device__ inline float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

template <int DT>
__global__ __launch_bounds__(256) void swiglu_fwd_kernel(const u16* __restrict__ gu, u16* __restrict__ h, int n, int vpr) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int row = i / vpr;
    const u16* p = gu + ((size_t)i + (size_t)row * vpr) * 8;  // row 2 F + column
    float g[8], u[8];
    widen8<DT>(p, g);
    widen8<DT>(p + (size_t)vpr * 8, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = g[e] * sigmoid(g[e]) * u[e];
    round8<DT>(h + (size_t)i * 8, g);
}

template <int DT>
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const u16* __restrict__ dh, const u16* __restrict__ gu,
                                                         u16* __restrict__ dgu, int n, int vpr) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int row = i / vpr;
    const size_t at = ((size_t)i + (size_t)row * vpr) * 8, up = at + (size_t)vpr * 8;
    float d[8], g[8], u[8];
    widen8<DT>(dh + (size_t)i * 8, d);
    widen8<DT>(gu + at, g);
    widen8<DT>(gu + up, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float s = sigmoid(g[e]);
        const float dg = d[e] * u[e] * (s * fmaf(g[e], 1.f - s, 1.f));  // silu'(g) = s (1 + g (1 - s))
        u[e] = d[e] * (g[e] * s);
        g[e] = dg;
    }
    round8<DT>(dgu + at, g);
    round8<DT>(dgu + up, u);
}

// ------------------------------------------------------------------------------------------
// Host side.
// ------------------------------------------------------------------------------------------
thread_local std::string g_err;

int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
int fail(const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return -1;
}

int launched(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_err = std::string(what) + " launch failed: " + hipGetErrorString(e);
        return (int)e;
    }
    return 0;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

constexpr int64_t kCus = 256, kMaxSplit = 32;
// Splits of the tokens: the count with the least estimated time, from a block's time for four stages (2.0 us, measured
// at 4096 x 768, one block per CU), its fixed time (3 us) and, split, the sum's launch (3 us) and the partials' round
// trip at 5 TB/s.
int wgrad_split(int64_t T, int64_t N, int64_t K) {
    const int64_t tiles = ((N + kTN - 1) / kTN) * ((K + kTK - 1) / kTK), nt = (T + 4 * kTT - 1) / (4 * kTT);  // groups of four stages
    int best = 1;
    double best_us = 1e30;
    for (int64_t s = 1; s <= std::min(kMaxSplit, std::max<int64_t>(nt, 1)); ++s) {
        const double rounds = (double)((tiles * s + kCus - 1) / kCus), per = (double)((nt + s - 1) / s);
        const double us = rounds * (per * 2.0 + 3.0) + (s > 1 ? 3.0 + 8e-6 * s * N * K / 5.0 : 0.0);
        if (us < best_us) best_us = us, best = (int)s;
    }
    return best;
}

}  // namespace

NNLIN_API const char* nn_linear_last_error(void) { return g_err.c_str(); }

NNLIN_API size_t nn_linear_wgrad_workspace_size(int64_t T, int64_t N, int64_t K) {
    if (T <= 0 || N <= 0 || K <= 0) return 0;
    const int s = wgrad_split(T, N, K);
    return s > 1 ? (size_t)s * N * K * 4 : 0;
}

NNLIN_API int nn_linear_wgrad(const void* dy, int64_t ldy, const void* x, int64_t ldx, int64_t T, int64_t N, int64_t K,
                              int nout, float* const* out, const int64_t* rows, void* workspace,
                              size_t workspace_bytes, int dtype, void* stream) {
    g_err.clear();
    if (T < 0 || N < 1 || K < 1 || N % 8 || K % 8) return fail("N and K must be positive multiples of 8");
    if (ldy < N || ldx < K || ldy % 8 || ldx % 8) return fail("row strides must be multiples of 8, at least the width");
    if (dtype != kF16 && dtype != kBF16) return fail("dtype must be float16 or bfloat16");
    if (T >= (1 << 30) || N * K >= ((int64_t)1 << 31) || kTT * ldy >= (1 << 29) || kTT * ldx >= (1 << 29)) return fail("sizes too large");
    if (nout < 1 || nout > 3 || !out || !rows) return fail("1 to 3 outputs");
    Outs o{};
    int64_t end = 0;
    for (int i = 0; i < 3; ++i) {
        if (i < nout) {
            if (rows[i] < 1 || !out[i] || !aligned16(out[i])) return fail("outputs must be non-empty and 16-byte aligned");
            end += rows[i];
            o.p[i] = out[i];
        }
        o.end[i] = (int)end;
    }
    if (end != N) return fail("the outputs' rows must add up to N");
    if (T && (!dy || !x || !aligned16(dy) || !aligned16(x))) return fail("inputs must be 16-byte aligned");
    const int s = T ? wgrad_split(T, N, K) : 1;
    if (s > 1 && (!workspace || !aligned16(workspace) || workspace_bytes < (size_t)s * N * K * 4)) return fail("workspace too small or misaligned");
    hipStream_t st = (hipStream_t)stream;
    const int ntk = (int)((K + kTK - 1) / kTK), tiles = (int)((N + kTN - 1) / kTN) * ntk;
    auto go = [&](auto kern) {
        kern<<<dim3((unsigned)(tiles * s)), dim3(512), 0, st>>>((const u16*)dy, (long long)ldy, (const u16*)x, (long long)ldx, (int)T, (int)N,
                                                                (int)K, ntk, tiles, s, (float*)workspace, o);
        return launched("wgrad_kernel");
    };
    if (int e = dtype == kBF16 ? go(wgrad_kernel<kBF16>) : go(wgrad_kernel<kF16>)) return e;
    if (s == 1) return 0;
    wgrad_sum_kernel<<<dim3((unsigned)((N * K / 4 + 255) / 256)), dim3(256), 0, st>>>((const float*)workspace, s, (int)N, (int)K, o);
    return launched("wgrad_sum_kernel");
}

NNLIN_API int nn_linear_cast(int n, const float* const* src, void* const* dst, const int64_t* count, int dtype,
                             void* stream) {
    g_err.clear();
    if (n < 1 || n > 4 || !src || !dst || !count) return fail("1 to 4 arrays");
    if (dtype != kF16 && dtype != kBF16) return fail("dtype must be float16 or bfloat16");
    Casts c{};
    int64_t end = 0;
    for (int i = 0; i < 4; ++i) {
        if (i < n) {
            if (count[i] < 0 || count[i] % 8) return fail("counts must be multiples of 8");
            if (count[i] && (!src[i] || !dst[i] || !aligned16(src[i]) || !aligned16(dst[i]))) return fail("arrays must be 16-byte aligned");
            end += count[i] / 8;
            if (end >= (1 << 30)) return fail("sizes too large");
            c.src[i] = src[i];
            c.dst[i] = (u16*)dst[i];
        }
        c.end[i] = (int)end;
    }
    if (end == 0) return 0;
    const dim3 grid((unsigned)((end + 255) / 256));
    if (dtype == kBF16)
        cast_kernel<kBF16><<<grid, dim3(256), 0, (hipStream_t)stream>>>(c);
    else
        cast_kernel<kF16><<<grid, dim3(256), 0, (hipStream_t)stream>>>(c);
    return launched("cast_kernel");
}

NNLIN_API int nn_linear_cast_both(int n, const float* const* src, void* const* dst, void* const* dst_t, const int64_t* rows,
                                  const int64_t* cols, const int64_t* ldt, int dtype, void* stream) {
    g_err.clear();
    if (n < 1 || n > 4 || !src || !dst || !dst_t || !rows || !cols || !ldt) return fail("1 to 4 arrays");
    if (dtype != kF16 && dtype != kBF16) return fail("dtype must be float16 or bfloat16");
    Turns c{};
    int64_t end = 0;
    for (int i = 0; i < 4; ++i) {
        if (i < n) {
            if (rows[i] < 0 || cols[i] < 0 || rows[i] % 8 || cols[i] % 8 || ldt[i] % 8 || ldt[i] < rows[i])
                return fail("rows, columns and the transposed stride must be multiples of 8");
            if (rows[i] >= (1 << 30) || cols[i] >= (1 << 30) || ldt[i] >= (1 << 30)) return fail("sizes too large");
            if (rows[i] && cols[i] && (!src[i] || !dst[i] || !dst_t[i] || !aligned16(src[i]) || !aligned16(dst[i]) || !aligned16(dst_t[i])))
                return fail("arrays must be 16-byte aligned");
            end += ((rows[i] + 63) / 64) * ((cols[i] + 63) / 64);
            if (end >= (1 << 30)) return fail("sizes too large");
            c.src[i] = src[i];
            c.dst[i] = (u16*)dst[i];
            c.dst_t[i] = (u16*)dst_t[i];
            c.rows[i] = (int)rows[i], c.cols[i] = (int)cols[i], c.ldt[i] = (int)ldt[i];
        }
        c.end[i] = (int)end;
    }
    if (end == 0) return 0;
    if (dtype == kBF16)
        cast_both_kernel<kBF16><<<dim3((unsigned)end), dim3(256), 0, (hipStream_t)stream>>>(c);
    else
        cast_both_kernel<kF16><<<dim3((unsigned)end), dim3(256), 0, (hipStream_t)stream>>>(c);
    return launched("cast_both_kernel");
}

namespace {
int check_swiglu(int64_t T, int64_t F, int dtype, const void* a, const void* b, const void* c) {
    g_err.clear();
    if (T < 0 || F < 8 || F % 8) return fail("F must be a positive multiple of 8");
    if (dtype != kF16 && dtype != kBF16) return fail("dtype must be float16 or bfloat16");
    if (T * (F / 8) >= ((int64_t)1 << 31) - 256) return fail("sizes too large");
    if (T && (!a || !b || !c || !aligned16(a) || !aligned16(b) || !aligned16(c))) return fail("tensors must be 16-byte aligned");
    return 0;
}
}  // namespace

NNLIN_API int nn_swiglu_fwd(const void* gu, void* h, int64_t T, int64_t F, int dtype, void* stream) {
    if (int e = check_swiglu(T, F, dtype, gu, h, h)) return e;
    if (T == 0) return 0;
    const int n = (int)(T * (F / 8));
    auto go = [&](auto kern) {
        kern<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>((const u16*)gu, (u16*)h, n, (int)(F / 8));
        return launched("swiglu_fwd_kernel");
    };
    return dtype == kBF16 ? go(swiglu_fwd_kernel<kBF16>) : go(swiglu_fwd_kernel<kF16>);
}

NNLIN_API int nn_swiglu_bwd(const void* dh, const void* gu, void* dgu, int64_t T, int64_t F, int dtype, void* stream) {
    if (int e = check_swiglu(T, F, dtype, dh, gu, dgu)) return e;
    if (T == 0) return 0;
    const int n = (int)(T * (F / 8));
    auto go = [&](auto kern) {
        kern<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>((const u16*)dh, (const u16*)gu, (u16*)dgu, n, (int)(F / 8));
        return launched("swiglu_bwd_kernel");
    };
    return dtype == kBF16 ? go(swiglu_bwd_kernel<kBF16>) : go(swiglu_bwd_kernel<kF16>);
}
