// Index arithmetic and split rules of the contractions as plain functions: which elements of its operands a thread of the
// fp32 contraction (gemm_f32_split_kernel in gemm.hip) touches, and into how many parts a reduction is split.  The
// kernels and their launches call them; tests/gemm_bounds.cpp walks them on the CPU.
#ifndef PCCNN_GEMM_TILES_H
#define PCCNN_GEMM_TILES_H

#include <stddef.h>
#include <stdint.h>

#ifdef __HIPCC__
#define GEMM_HD __host__ __device__ __forceinline__
#else
#define GEMM_HD inline
#endif

#define GS_K 32            // reduction elements per step of the split kernel

// One operand of the split kernel: its tile of X rows (or columns) is loaded in units of 8 consecutive k, unit
// threadIdx.x + 256 i by pass i of a thread.  KC: the reduction index is the contiguous one.  Offsets are in elements.
//
// Rows past the tile's or the operand's edge read rows inside it (their results are not stored): a unit of W rows that
// begins past the edge reads the last W.  A unit of two rows that begins on the last one (odd extents only) reads the
// next k's first row too, which exists in every step but the last.  There, and where a step is not whole, units are read
// whole only where each is (the empty ones read the step's first), else element by element, each inside the operand.
template <bool KC, int X> struct GemmUnits {
    static constexpr int W = (!KC && X >= 96) ? 2 : 1;              // rows per unit load
    static constexpr int UNITS = X * (GS_K / 8) / W;
    static constexpr int PASSES = (UNITS + 255) / 256;

    static GEMM_HD bool active(int thread, int i) { return UNITS % 256 == 0 || thread + 256 * i < UNITS; }
    static GEMM_HD void unit(int thread, int i, int &x, int &k8)
    {
        const int u = thread + 256 * i;
        if (KC) { x = u / (GS_K / 8); k8 = u % (GS_K / 8); }
        else { k8 = u / (X / W); x = (u % (X / W)) * W; }
    }
    static GEMM_HD int rows_left(int64_t x0, int64_t x_end) { return (int)((x_end - x0) < X ? (x_end - x0) : X); }
    static GEMM_HD int64_t origin(int64_t x0, int64_t k0, int64_t ld) { return KC ? x0 * ld + k0 : k0 * ld + x0; }
    static GEMM_HD int64_t advance(int64_t ld) { return KC ? GS_K : GS_K * ld; }
    // First element of a unit, from the step's origin; its others: KC the next 7, else for each of its eight k (ld
    // apart) W neighbors.
    static GEMM_HD unsigned offset(int x, int k8, int x_left, unsigned ld)
    {
        const unsigned xc = (unsigned)(x < x_left ? x : (x_left >= W ? x_left - W : 0)), kk = (unsigned)(k8 * 8);
        return KC ? xc * ld + kk : kk * ld + xc;
    }
    // Whether the units of a step of which k_left elements of the reduction are left are all whole or empty.
    static GEMM_HD bool whole_units(int x_left, int k_left) { return k_left % 8 == 0 && (W == 1 || x_left % 2 == 0); }
    // Element (x, k) of a step of which k_left elements of the reduction are left, or one inside the operand for it.
    static GEMM_HD int64_t checked(int x, int k, int x_left, int k_left, int64_t ld)
    {
        const int64_t xc = x < x_left ? x : x_left - 1, kc = k < k_left ? k : k_left - 1;
        return KC ? xc * ld + kc : kc * ld + xc;
    }
};

// Whether the byte offsets of a tile of `rows` rows (or columns) fit into 32 bits.
inline bool gemm_tile_fits(int rows, int64_t ld) { return ld < (((int64_t)1 << 32) - 256) / 4 / (rows < GS_K ? GS_K : rows); }

// Steps of a reduction of `count` elements, and how many of them, from the first, are loaded without checks: all where
// the last one is whole and no unit of two rows (w) straddles an edge.  An empty reduction has no step of either kind.
GEMM_HD int64_t gemm_steps(int64_t count) { return (count + GS_K - 1) / GS_K; }
GEMM_HD int64_t gemm_steps_unchecked(int64_t count, int w_a, int64_t rows, int w_b, int64_t cols)
{
    if (count == 0) return 0;
    const bool whole = count % GS_K == 0 && (w_a == 1 || rows % 2 == 0) && (w_b == 1 || cols % 2 == 0);
    return whole ? gemm_steps(count) : gemm_steps(count) - 1;
}

// Split of the sample dimension for d_weights = P^T x dOut with bf16 operands (tiles of 64 x 128 or, from 1024 workgroups
// of those on, 128 x 128): a product bound by its operand traffic, whose output has few tiles.  As many parts as fit on
// the chip at once, four workgroups per CU, and not one more: 720 x 16 x 65 536 takes 40 us with 1020 workgroups and 55
// with 1152; parts of 64 samples or more; from 30 000 samples on 64 parts even where they do not fit at once, for the
// taller tile (2560 x 160 x 120 000: 330 us, 400 with 12 parts; 1920 x 256 x 65 536: 165, 196 with 12), but not
// before, where the partial sums weigh more than that gains (1920 x 256 x 8192: 58 us with 64 parts, 43 with 17;
// 2560 x 256 x 20 000: 109 and 78).
inline int gemm_bf16_split(int64_t rows, int64_t cols, int64_t inner, int batch, size_t workspace_floats)
{
    const int64_t tiles = (rows + 63) / 64 * ((cols + 127) / 128) * batch;
    const int64_t room = (int64_t)(workspace_floats / ((size_t)rows * cols * batch));
    int64_t split = 1024 / tiles;
    if (split < 64 && inner >= 30000) split = 64;
    if (split > inner / 64) split = inner / 64;
    if (split > room) split = room;
    return split < 1 ? 1 : (int)split;
}

#endif
