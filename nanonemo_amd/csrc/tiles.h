// Building blocks of the MFMA kernels for MI355X (gfx950): element types and their 32x32x16 products, swizzled LDS tiles
// filled by DMA, row and column operands read from them, and the waits that go with the copies.
//
// MFMA 32x32x16 register layouts (lane l, l32 = l % 32, hh = l / 32):
//   A (32x16, M x K): lane l supplies A[l32][8*hh + j], j = 0..7
//   B (16x32, K x N): lane l supplies B[8*hh + j][l32]
//   C (32x32):        lane l holds C[(i/4)*8 + 4*hh + (i%4)][l32] in element i = 0..15
// A and B agree on which (half-wave, element) carries which k, so a product may permute the
// contraction index freely as long as both operands use the same permutation.
//
// ds_read_b64_tr_b16 (per 16-lane group, lane i, result element j) returns element i%4 of the
// 4-element vector addressed by lane 4j + i/4 of the same group. If lane i' of a group
// addresses row r0 + i'/4, columns c0 + 4*(i'%4) .. +3 of a row-major tile, lane i receives
// rows r0..r0+3 of column c0 + i: a column operand for the MFMA.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

using u16 = unsigned short;
typedef u16 u16x8 __attribute__((ext_vector_type(8)));
typedef u16 u16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kF16 = 0;
constexpr int kBF16 = 1;

#define LDS_AS(T, p) ((__attribute__((address_space(3))) T*)(p))

template <int DT>
struct Elem;

template <>
struct Elem<kBF16> {
    __device__ static inline f32x16 mfma(u16x8 a, u16x8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
    }
    // Round-to-nearest-even conversion of two fp32 values into one packed dword (lo first).
    __device__ static inline uint32_t pack2(float lo, float hi) {
        bf16x2 v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    // acc + lo + hi of a packed pair.
    __device__ static inline float add_pair(uint32_t pair, float acc) {
        const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), one, acc, false);
    }
    __device__ static inline float to_f32(u16 x) { return __uint_as_float((uint32_t)x << 16); }
};

template <>
struct Elem<kF16> {
    __device__ static inline f32x16 mfma(u16x8 a, u16x8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    __device__ static inline uint32_t pack2(float lo, float hi) {
        f16x2 v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    __device__ static inline float add_pair(uint32_t pair, float acc) {
        const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pair), one, acc, false);
    }
    __device__ static inline float to_f32(u16 x) { return (float)__builtin_bit_cast(_Float16, x); }
};

// Elements [base, base+8) of an accumulator, rounded to 16 bits and packed as an MFMA operand.
template <int DT>
__device__ inline u16x8 pack8(const f32x16& a, int base) {
    u32x4 r = {Elem<DT>::pack2(a[base + 0], a[base + 1]), Elem<DT>::pack2(a[base + 2], a[base + 3]),
               Elem<DT>::pack2(a[base + 4], a[base + 5]), Elem<DT>::pack2(a[base + 6], a[base + 7])};
    return __builtin_bit_cast(u16x8, r);
}

__device__ inline u16x8 cat4(u16x4 a, u16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
typedef float f32x8 __attribute__((ext_vector_type(8)));
__device__ inline f32x16 cat16(f32x4 a, f32x4 b, f32x4 c, f32x4 d) {
    const f32x8 ab = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    const f32x8 cd = __builtin_shufflevector(c, d, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_shufflevector(ab, cd, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
}
__device__ inline u16x8 ld8(const u16* p) { return *reinterpret_cast<const u16x8*>(p); }

// Row-major LDS tiles of W 16-bit columns store 16-byte chunk c of row r at chunk position
// swz_chunk(r, c). The XOR pattern depends only on row bits 1..3 (W = 64) or 2..3 (W = 32), so
// it repeats every 16 rows, and it keeps both access patterns free of bank conflicts:
//   * ds_read_b128 of one logical chunk from 16 consecutive rows (row operands);
//   * ds_read_b64_tr_b16 of 4 consecutive rows x 4 aligned chunks per 32 lanes (column operands).
// It is an involution, so the DMA uses the same map to place chunks.
template <int W>
__device__ inline int swz_chunk(int row, int c) {
    static_assert(W == 64 || W == 32, "tile width");
    if constexpr (W == 64)
        return c ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
    else
        return c ^ ((row >> 2) & 3);
}
template <int W>
__device__ inline int swz(int row, int col) {
    return row * W + (swz_chunk<W>(row, col >> 3) << 3) + (col & 7);
}

// Per-lane offset of a row operand: 8 columns col0 + 8*hh .. of row `row` (rows 16k + row read
// the same chunk positions, so callers add 16k * W).
template <int W>
__device__ inline int row_off(int row, int col) { return swz<W>(row, col); }

// Per-lane offset of a column operand for ds_read_b64_tr_b16: lane i (of its 16-lane group)
// addresses row r0 + i/4, columns c0 + 4*(i%4) .. +3, and receives rows r0..r0+3 of column
// c0 + i. r0 % 4 == 0 and c0 % 16 == 0; rows 16k + r0 reuse the offset plus 16k * W.
template <int W>
__device__ inline int col_off(int r0, int c0, int lane) {
    const int i = lane & 15;
    return swz<W>(r0 + (i >> 2), c0 + 4 * (i & 3));
}
__device__ inline u16x4 ld_tr(const u16* p) {
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_AS(s16x4, const_cast<u16*>(p))));
}

// Per-lane part of the DMA addressing of a W-column tile (computed once per kernel): the lane's
// row within one copy instruction (a copy instruction moves 64 chunks of 16 bytes, i.e.
// 64 / (W / 8) rows) and its swizzled chunk byte offset. An instruction's rows start at a
// multiple of 64 / (W / 8); the swizzle reads row bits 1..3 (W = 64), of which that start
// contributes only bit 3 (cB1 applies to odd instructions), or bits 2..3 (W = 32), which it never
// touches.
struct DmaLane {
    uint32_t rl, cB0, cB1;
};
template <int W>
__device__ inline DmaLane dma_lane(int lane) {
    constexpr int CH = W / 8;
    const int rl = lane / CH, cl = lane % CH;
    return {(uint32_t)rl, (uint32_t)swz_chunk<W>(rl, cl) * 16, (uint32_t)swz_chunk<W>(rl + 8, cl) * 16};
}

// Per-lane byte offsets of the copy instructions (this wave's share) of a [ROWS][W] tile with row
// stride `ld` elements, relative to the tile's first row: computed once per kernel, so that a copy
// of a tile that does not reach past row T - 1 costs no per-lane address arithmetic.
template <int W, int ROWS, int NW>
struct DmaOffs {
    static constexpr int N = ROWS * (W / 8) / (64 * NW);
    uint32_t o[N];
};
template <int W, int ROWS, int NW>
__device__ inline DmaOffs<W, ROWS, NW> dma_offsets(int lane, int wave, int ld) {
    constexpr int CH = W / 8;
    const DmaLane dl = dma_lane<W>(lane);
    DmaOffs<W, ROWS, NW> r;
#pragma unroll
    for (int it = 0; it < DmaOffs<W, ROWS, NW>::N; ++it) {
        const int k = it * NW + wave;  // copy instruction index within the tile
        r.o[it] = (dl.rl + (uint32_t)(k * (64 / CH))) * (uint32_t)ld * 2 + ((W == 64 && (k & 1)) ? dl.cB1 : dl.cB0);
    }
    return r;
}

// Buffer resource word 3 for raw (unswizzled, stride 0) buffer access on gfx9-family parts.
constexpr int kBufWord3 = 0x00020000;

// Copies ROWS rows of W columns at g, row stride `ld` elements, into a swizzled row-major LDS tile, 16
// bytes per lane; `left` rows (at least 1) remain in the matrix. `g`, `ld`, `left`, `lds` and `wave` are
// wave-uniform, and `fo` holds this lane's offsets for stride `ld` (dma_offsets). The copies are
// buffer loads: the tile's base and extent live in a scalar buffer descriptor and each lane adds its
// 32-bit offset, so they cost no per-lane address arithmetic. The descriptor's extent ends at the last
// row, so rows past it read as zeros (their results are masked by the callers). The LDS
// destination of a copy is the uniform base + 16 * lane.
template <int W, int ROWS, int NW>
__device__ inline void dma_tile(const u16* __restrict__ g, int ld, int left, u16* lds, int wave,
                                const DmaOffs<W, ROWS, NW>& fo) {
    constexpr int CH = W / 8, NCH = ROWS * CH;
    static_assert(NCH % (64 * NW) == 0 && 64 % CH == 0, "tile must split evenly over the block's waves");
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer descriptor type exists in the device pass only
    const int wu = __builtin_amdgcn_readfirstlane(wave);
    // readfirstlane yields an int: each half goes through uint32_t before widening, or a low word with
    // bit 31 set would sign-extend into the high word.
    const uint64_t ga = reinterpret_cast<uint64_t>(g);
    const uint32_t ghi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(ga >> 32));
    const uint32_t glo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)ga);
    void* gt = reinterpret_cast<void*>(((uint64_t)ghi << 32) | glo);
    const int nbytes = __builtin_amdgcn_readfirstlane(min(left, ROWS) * ld * 2);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(gt, 0, nbytes, kBufWord3);
#pragma unroll
    for (int it = 0; it < NCH / (64 * NW); ++it) {
        const int k = it * NW + wu;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_AS(void, lds + k * 64 * 8), 16, fo.o[it], 0, 0, 0);
    }
#endif
}
// The same for rows [r0, r0 + ROWS) of a [T][W] matrix at g.
template <int W, int ROWS, int NW>
__device__ inline void dma_rows(const u16* __restrict__ g, int ld, int r0, int T, u16* lds, int wave,
                                const DmaOffs<W, ROWS, NW>& fo) {
    dma_tile<W, ROWS, NW>(g + (size_t)r0 * ld, ld, T - r0, lds, wave, fo);
}

// Wait until this wave's vector-memory operations (including LDS DMA) have completed.
__device__ inline void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// Wait until at most N of this wave's vector-memory operations are outstanding (they complete in
// issue order, so everything issued before the last N has landed). gfx9 encoding: vmcnt in bits
// 3:0 and 15:14; expcnt and lgkmcnt left at their maxima.
template <int N>
__device__ inline void wait_vmem_keep() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Block barrier that orders LDS only: this wave's LDS accesses complete, then s_barrier. Vector-memory
// operations (global loads and stores, LDS DMA) may stay in flight across it, so it must only be used
// where no wave reads, before its own vmcnt wait, LDS that such an operation writes. (__syncthreads
// also waits for every vector-memory operation.) The memory clobber keeps the compiler from moving
// memory accesses across it.
__device__ inline void barrier_lds() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace
