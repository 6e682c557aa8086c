// fp32 GEMM on the CDNA matrix cores: the [M, K*Cin] x [K*Cin, Cout] contraction of the convolutions and its two
// transposes.
//
// Two kernels.  gemm_f32_split_kernel takes the products that can fill the chip: every fp32 operand is carried as
// three bf16 terms and multiplied on the bf16 matrix pipe (v_mfma_f32_32x32x16_bf16), whose rate is sixteen times
// that of the fp32 matrix instructions and beside which vector instructions run (beside the fp32 ones they do not).
// gemm_f32_short_kernel takes the small ones, which are bound by latency, on the fp32 matrix instructions.  Split-K
// writes partial products to a workspace that a further kernel sums in a fixed order.
//
// The three terms lose nothing: x = h1 + h2 + h3 exactly, with h1 = x rounded to bf16 (8 significant bits), h2 the
// rest rounded to bf16, h3 what is left (at most 8 bits of the 24 remain).  A product of two terms is exact in fp32
// (16 bits), and the sums are fp32.  Of the nine products of a pair x y the three smallest, h2 h3', h3 h2' and
// h3 h3', are left out: together at most 2^-24 |x y|, what rounding the product once to fp32 loses.  Error against
// float64, relative to the result's norm, this kernel / the fp32 matrix instructions: reduction of 128: 1.6e-7 /
// 2.0e-7, 1024: 4.9e-7 / 5.7e-7, 1920: 2.6e-7 / 7.8e-7, 3855 of 65 536: 3.9e-7 / 1.1e-6.
//
// Measured, before (128 x 128 and 64 x 128 tiles of fp32 matrix instructions) and now, launches in a row, us: 65 536 x
// 128 x 1024 174 -> 118, its transposes 171 -> 126 and 162 -> 130; 65 536 x 256 x 1920 493 -> 384 (168 TFLOP/s; the
// fp32 instructions' peak is 157), transposes 533 -> 369 and 512 -> 397; 120 000 x 64 x 1920 536 -> 249; 37 675 x 96 x
// 720 89 -> 60; 40 000 x 205 x 645 (odd leading dimension) 169 -> 97; 24 x 33 x 7327 136 -> 9; 346 x 256 x 1024 51 -> 11.
// The large ones fill no pipe: counters give 47 to 60 % of the SIMD cycles to the matrix pipe and 31 to 42 % to vector
// instructions, at a clock of about 1.8 GHz; a wavefront splits, hands over and multiplies in turn, and the two or
// three of a SIMD overlap in part.  The six products run at 1.0 PFLOP/s.
#include <type_traits>

#include "common.h"
#include "gemm_tiles.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));      // dword-aligned 16-byte access
typedef float floatx2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define GS_PLANES 3
// Operands are scaled by 2^16 (exact) on their way into terms and results back by 2^-32: a third term of the smallest
// normal number then still is a bf16 number, and even subnormal operands are carried exactly.  What overflows on the
// way (operands from 2^112, sums from 2^96) is computed again at the end of the kernel.
#define GS_SCALE 65536.0f
// Longer reductions keep the sum of the largest products h1 h1' apart from that of the five smaller ones, so that the
// large sum is rounded once and not six times per 16 elements (error at 1920: 6.8e-7 -> 2.6e-7 of the result's norm).
// The second sum costs registers and with them a wavefront per SIMD where the reduction is short (65 536 x 1024 x 128,
// B transposed: 121 -> 130 us), and there one sum is as precise as it need be.
#define GS_ONE_SUM 1024
#define GS_STAGE_LD 36     // floats per row of a staged output tile

struct GemmArgs {
    const float *a, *b;
    float *c;
    int64_t rows, cols, inner;
    int64_t lda, ldb, ldc;
    int64_t stride_a, stride_b, stride_c;
    int split_k;
    int64_t k_chunk;       // inner elements per split
    int tiles_x, tiles_y;  // workgroup tiles along the columns / rows
    int64_t total_wg;      // tiles_x * tiles_y * batch * split_k
};

// Workgroups are handed to the 8 XCDs round-robin by their linear id, and each XCD has its own L2.  The
// launch is one-dimensional and padded to a multiple of 8; workgroup i works on logical tile
// (i % 8) * (padded / 8) + i / 8, so every XCD owns one contiguous run of logical tiles.  Logical tiles are
// ordered column tile fastest, then row tile, then batch / split: neighbours in that order share their A
// row tile (or, with one column tile, their B chunk), which is then fetched from HBM by one XCD, once.
#define GEMM_XCDS 8

struct GemmTile {
    int64_t bm, bn, k_begin, k_end;
    int batch, split;
    bool valid;
};

template <int BM, int BN>
__device__ __forceinline__ GemmTile gemm_tile(const GemmArgs &g)
{
    GemmTile t;
    const int64_t per_xcd = (int64_t)gridDim.x / GEMM_XCDS;
    const int64_t tile = (int64_t)(blockIdx.x % GEMM_XCDS) * per_xcd + blockIdx.x / GEMM_XCDS;
    t.valid = tile < g.total_wg;                                    // false: padding of the launch
    const int tx = (int)(tile % g.tiles_x);
    const int ty = (int)((tile / g.tiles_x) % g.tiles_y);
    const int tz = (int)(tile / ((int64_t)g.tiles_x * g.tiles_y));
    t.batch = tz / g.split_k;
    t.split = tz % g.split_k;
    t.bm = (int64_t)ty * BM;
    t.bn = (int64_t)tx * BN;
    t.k_begin = (int64_t)t.split * g.k_chunk;
    t.k_end = (t.k_begin + g.k_chunk < g.inner) ? t.k_begin + g.k_chunk : g.inner;
    return t;
}

__device__ __forceinline__ float *gemm_output(const GemmArgs &g, const GemmTile &t, float *partial, int64_t &ldc)
{
    if (g.split_k > 1) {
        ldc = g.cols;
        return partial + ((int64_t)t.batch * g.split_k + t.split) * g.rows * g.cols;
    }
    ldc = g.ldc;
    return g.c + (int64_t)t.batch * g.stride_c;
}

// A 32 x 32 tile of the product by one wavefront on the fp32 matrix instructions, operands straight from memory (`a` and
// `b`: this lane's row and column; `h`: its half, which takes k = 4 h + e of every eight).  Ends early once every sum
// that is wanted (bit v: register v of this lane) is NaN.  Few registers rather than many loads in flight: it must not
// cost the kernel around it a wavefront.
template <bool AT, bool BT>
__device__ __forceinline__ floatx16 gemm_tile_f32(const float *__restrict__ a, const float *__restrict__ b, int64_t lda,
                                                  int64_t ldb, int h, int64_t k_begin, int64_t k_end, unsigned wanted)
{
    constexpr int AHEAD = 2;
    floatx16 s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.0f;
#pragma unroll 1
    for (int64_t k0 = k_begin; k0 < k_end; k0 += 8 * AHEAD) {
        float fa[4 * AHEAD], fb[4 * AHEAD];
#pragma unroll
        for (int e = 0; e < 4 * AHEAD; ++e) {
            const int64_t k = k0 + 8 * (e / 4) + 4 * h + e % 4;
            const bool in = k < k_end;
            const int64_t kc = in ? k : k_end - 1;
            fa[e] = a[AT ? kc * lda : kc];
            fb[e] = b[BT ? kc : kc * ldb];
            if (!in) fa[e] = fb[e] = 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 4 * AHEAD; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], s, 0, 0, 0);
        bool done = true;
#pragma unroll
        for (int v = 0; v < 16; ++v) done = done && (s[v] != s[v] || !(wanted >> v & 1));
        if (__all(done)) break;
    }
    return s;
}

// ---------------------------------------------------------------------------------------------------------------
// Split kernel.  Workgroup: 4 wavefronts, WM x WN of them, each TM x TN MFMA tiles of 32 x 32; inner step 32.
//
// An operand tile of X rows (or columns) sits in LDS as 16-byte units of 8 consecutive k of one row, one plane per
// term: unit (term, k / 8, x) in slot gs_slot(x, k / 8).  A fragment of the MFMA is one unit per lane, 32 consecutive
// x: one ds_read_b128 without bank conflicts.  A thread makes whole units: it loads 8 k of a row (XC with 96 or more
// rows: of two neighboring rows) and splits them in registers.
//   KC (reduction index contiguous in memory): unit u = (x = u / 4, k / 8 = u % 4), two 16-byte loads;
//   XC (row / column index contiguous): unit u = (k / 8 = u / (X / W), x = W (u % (X / W))), eight loads of W floats.
// The wide loads are dword-aligned: any leading dimension.  Which elements they touch is in gemm_tiles.h.
//
// One LDS buffer and two barriers per step, the next step's loads in flight in registers: the two or three workgroups
// of a CU fill each other's gaps.  Tried and not taken: two steps of loads ahead (no difference); two LDS buffers of
// 16 with one barrier and the split between the MFMAs of the same wavefront (361 against 364 us at 65 536 x 256 x
// 1920, slower on narrow tiles and spilling with both operands XC); 256 x 128 tiles everywhere (faster there, 324
// against 364, slower at 65 536 x 128 x 1024, 118 against 107, and with both operands XC, 483 against 368).
__device__ __forceinline__ int gs_slot(int x, int k8) { return x ^ ((x >> 3) & 1) ^ (k8 << 1); }

__device__ __forceinline__ uint32_t gs_pack(float lo, float hi)
{
    const floatx2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// The three terms of eight values, packed in order.
__device__ __forceinline__ void gs_split(const float (&x)[8], uint4 (&term)[GS_PLANES])
{
    uint32_t t[GS_PLANES][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float lo = x[2 * i] * GS_SCALE, hi = x[2 * i + 1] * GS_SCALE;
#pragma unroll
        for (int p = 0; p < GS_PLANES; ++p) {
            const uint32_t w = gs_pack(lo, hi);
            t[p][i] = w;
            if (p + 1 < GS_PLANES) {
                lo -= __uint_as_float(w << 16);
                hi -= __uint_as_float(w & 0xffff0000u);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < GS_PLANES; ++p) term[p] = make_uint4(t[p][0], t[p][1], t[p][2], t[p][3]);
}

template <bool KC, int X> struct SplitOperand : GemmUnits<KC, X> {
    typedef GemmUnits<KC, X> Units;
    static constexpr int W = Units::W, PASSES = Units::PASSES;
    const float *base;                                              // uniform: origin of the current step
    int64_t ld;
    unsigned off[PASSES];                                           // this thread's units, in bytes
    int x_left;                                                     // rows of the operand from the tile's first on
    struct Regs { float v[PASSES][8 * W]; };

    __device__ __forceinline__ static bool active(int i) { return Units::active(threadIdx.x, i); }
    __device__ __forceinline__ static void unit(int i, int &x, int &k8) { Units::unit(threadIdx.x, i, x, k8); }
    __device__ __forceinline__ void init(const float *origin, int64_t ld_, int64_t x0, int64_t x_end, int64_t k0)
    {
        ld = ld_;
        base = origin + Units::origin(x0, k0, ld);
        x_left = Units::rows_left(x0, x_end);
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            int x, k8;
            unit(i, x, k8);
            off[i] = Units::offset(x, k8, x_left, (unsigned)ld) * 4u;
        }
    }
    // the unit of pass i at `bytes` from the step's origin
    __device__ __forceinline__ void load_unit(Regs &r, int i, unsigned bytes)
    {
        if (KC) {
            const floatx4u lo = *(const floatx4u *)((const char *)base + bytes);
            const floatx4u hi = *(const floatx4u *)((const char *)(base + 4) + bytes);
#pragma unroll
            for (int e = 0; e < 4; ++e) { r.v[i][e] = lo[e]; r.v[i][4 + e] = hi[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const char *p = (const char *)(base + e * ld) + bytes;
                if (W == 2) {
                    const floatx2u q = *(const floatx2u *)p;
                    r.v[i][2 * e] = q[0];
                    r.v[i][2 * e + W - 1] = q[1];
                } else {
                    r.v[i][e] = *(const float *)p;
                }
            }
        }
    }
    // the step at `base`, which moves on
    __device__ __forceinline__ void load(Regs &r)
    {
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (!active(i)) break;
            load_unit(r, i, off[i]);
        }
        base += Units::advance(ld);
    }
    // the last step: k_left elements of the reduction, zeros past them.  Whole units where there are no others (65 536 x
    // 128 x 48: 14.5 us, 17.0 element by element; 32 768 x 1024 x 16, B transposed: 27 and 33, x 48: 33 and 46)
    __device__ __forceinline__ void load_last(Regs &r, int k_left)
    {
        if (Units::whole_units(x_left, k_left)) {                   // uniform
#pragma unroll
            for (int i = 0; i < PASSES; ++i) {
                if (!active(i)) break;
                int x, k8;
                unit(i, x, k8);
                const bool in = k8 * 8 < k_left;
                load_unit(r, i, Units::offset(x, in ? k8 : 0, x_left, (unsigned)ld) * 4u);
#pragma unroll
                for (int e = 0; e < 8 * W; ++e) r.v[i][e] = in ? r.v[i][e] : 0.0f;
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (!active(i)) break;
            int x, k8;
            unit(i, x, k8);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool in = k8 * 8 + e < k_left;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const float q = base[Units::checked(x + w, k8 * 8 + e, x_left, k_left, ld)];
                    r.v[i][e * W + w] = in ? q : 0.0f;
                }
            }
        }
    }
    __device__ __forceinline__ static void park(const Regs &r, uint4 (*lds)[GS_K / 8][X])
    {
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (!active(i)) break;
            int x, k8;
            unit(i, x, k8);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                float q[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) q[e] = r.v[i][e * W + w];
                uint4 term[GS_PLANES];
                gs_split(q, term);
#pragma unroll
                for (int p = 0; p < GS_PLANES; ++p) lds[p][k8][gs_slot(x + w, k8)] = term[p];
            }
        }
    }
};

template <bool AT, bool BT, int WM, int WN, int TM, int TN, bool LOW>
__global__ void __launch_bounds__(256, 2)
gemm_f32_split_kernel(GemmArgs g, float *__restrict__ partial)
{
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    __shared__ uint4 lds[GS_PLANES * (GS_K / 8) * (BM + BN)];
    uint4 (*As)[GS_K / 8][BM] = (uint4 (*)[GS_K / 8][BM])lds;
    uint4 (*Bs)[GS_K / 8][BN] = (uint4 (*)[GS_K / 8][BN])(lds + GS_PLANES * (GS_K / 8) * BM);
    const int lane = pccnn_lane();
    const int wave = threadIdx.x >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int r = lane & 31, h = lane >> 5;
    const GemmTile t = gemm_tile<BM, BN>(g);
    if (!t.valid) return;
    const float *a = g.a + (int64_t)t.batch * g.stride_a;
    const float *b = g.b + (int64_t)t.batch * g.stride_b;

    floatx16 acc[TM][TN], low[LOW ? TM : 1][LOW ? TN : 1];          // LOW: h1 h1', and the five smaller products
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[i][j][v] = 0.0f;
                if (LOW) low[i][j][v] = 0.0f;
            }

    SplitOperand<!AT, BM> oa;
    SplitOperand<BT, BN> ob;
    oa.init(a, g.lda, t.bm, g.rows, t.k_begin);
    ob.init(b, g.ldb, t.bn, g.cols, t.k_begin);
    typename SplitOperand<!AT, BM>::Regs va;
    typename SplitOperand<BT, BN>::Regs vb;
    const int64_t nk = gemm_steps(t.k_end - t.k_begin);
    const int nf = (int)gemm_steps_unchecked(t.k_end - t.k_begin, SplitOperand<!AT, BM>::W, g.rows,
                                             SplitOperand<BT, BN>::W, g.cols);
    // this wave's LDS traffic is complete, then everyone's (the global loads stay in flight)
    auto lds_barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto multiply = [&](int k_left) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < GS_K / 16; ++ks) {
            if (16 * ks >= k_left) break;                           // uniform; zeros
            const int k8 = 2 * ks + h;
            bf16x8 fa[GS_PLANES][TM], fb[GS_PLANES][TN];
#pragma unroll
            for (int p = 0; p < GS_PLANES; ++p) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    fa[p][i] = __builtin_bit_cast(bf16x8, As[p][k8][gs_slot(wm * (TM * 32) + i * 32 + r, k8)]);
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    fb[p][j] = __builtin_bit_cast(bf16x8, Bs[p][k8][gs_slot(wn * (TN * 32) + j * 32 + r, k8)]);
            }
            // the operands are swapped (see the store below)
            constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
            for (int n = 0; n < 6; ++n)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        floatx16 &sum = LOW && n < 5 ? low[LOW ? i : 0][LOW ? j : 0] : acc[i][j];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[PB[n]][j], fa[PA[n]][i], sum, 0, 0, 0);
                    }
        }
    };
    if (nf > 0) {
        oa.load(va);
        ob.load(vb);
    }
    for (int kt = 0; kt < nf; ++kt) {
        if (kt > 0) lds_barrier();                                  // everyone has read the previous step
        SplitOperand<!AT, BM>::park(va, As);
        SplitOperand<BT, BN>::park(vb, Bs);
        lds_barrier();
        if (kt + 1 < nf) {
            oa.load(va);
            ob.load(vb);
        }
        multiply(GS_K);
    }
    if (nf < nk) {                                                  // the last step, with checks
        const int k_left = (int)(t.k_end - t.k_begin - (int64_t)nf * GS_K);
        oa.load_last(va, k_left);
        ob.load_last(vb, k_left);
        lds_barrier();
        SplitOperand<!AT, BM>::park(va, As);
        SplitOperand<BT, BN>::park(vb, Bs);
        lds_barrier();
        multiply(k_left);
    }

    // With the operands swapped a tile of the accumulator is the transpose of the output tile: lane l holds output
    // row l % 32 and, in registers 4 g .. 4 g + 3, the four consecutive columns 8 g + 4 (l / 32) + 0..3.  A tile goes
    // through the wavefront's own piece of LDS so that a store writes eight whole 128-byte rows.
    int64_t ldc;
    float *cbase = gemm_output(g, t, partial, ldc);
    lds_barrier();                                                  // the fragments of the last step have been read
    float *stage = (float *)lds + wave * (32 * GS_STAGE_LD);
    const int srow = lane >> 3, scol = (lane & 7) * 4;
    unsigned bad = 0;                                               // uniform: tiles with a result that is not finite
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bool finite = true;
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                floatx4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = acc[i][j][4 * gq + e];
                    if (LOW) v[e] += low[LOW ? i : 0][LOW ? j : 0][4 * gq + e];
                    v[e] *= 1.0f / (GS_SCALE * GS_SCALE);
                    finite = finite && fabsf(v[e]) <= 3.402823466e38f;
                }
                *(floatx4 *)(stage + r * GS_STAGE_LD + 8 * gq + 4 * h) = v;
            }
            if (__any(!finite)) bad |= 1u << (i * TN + j);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int64_t col = t.bn + (wn * TN + j) * 32 + scol;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t row = t.bm + (wm * TM + i) * 32 + q * 8 + srow;
                const floatx4 v = *(const floatx4 *)(stage + (q * 8 + srow) * GS_STAGE_LD + scol);
                if (row < g.rows && col + 4 <= g.cols) {
                    *(floatx4u *)(cbase + row * ldc + col) = v;
                } else if (row < g.rows) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < g.cols) cbase[row * ldc + col + e] = v[e];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    // An infinite operand (or one that rounds up to infinity as bf16) makes its terms' products infinity times zero.
    // Results that are not finite are computed again, a tile at a time, by the fp32 matrix instructions, which give what
    // fp32 arithmetic gives.  65 536 x 128 x 1024 (116 us): with one infinite weight 340 us, with an infinite column of
    // them 130 (its results are NaN at once), with infinities everywhere 660; one lane for one element took 640, 130
    // and 18 000.
    if (bad != 0) {
        __threadfence_block();
#pragma unroll 1
        for (int tile = 0; tile < TM * TN; ++tile) {
            if (!(bad >> tile & 1)) continue;
            const int64_t row0 = t.bm + (wm * TM + tile / TN) * 32, col0 = t.bn + (wn * TN + tile % TN) * 32;
            const int64_t row = row0 + r < g.rows ? row0 + r : g.rows - 1, col = col0 + r < g.cols ? col0 + r : g.cols - 1;
            // register v of lane l: row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32 of the tile
            unsigned wanted = 0;
#pragma unroll 2
            for (int v = 0; v < 16; ++v) {
                const int64_t orow = row0 + 8 * (v / 4) + 4 * h + v % 4;
                if (orow < g.rows && col0 + r < g.cols && !(fabsf(cbase[orow * ldc + col0 + r]) <= 3.402823466e38f))
                    wanted |= 1u << v;
            }
            const floatx16 s = gemm_tile_f32<AT, BT>(a + (AT ? row : row * g.lda), b + (BT ? col * g.ldb : col), g.lda,
                                                     g.ldb, h, t.k_begin, t.k_end, wanted);
            int64_t ld = ldc;
            asm volatile("" : "+s"(ld));                            // the addresses anew, not kept over the loop
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (wanted >> v & 1) cbase[(row0 + 8 * (v / 4) + 4 * h + v % 4) * ld + col0 + r] = s[v];
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Short kernel: products too small to fill the chip with the tiles above (up to 128 of them; 2048 x 32 x 480: 27 -> 7
// us, where 16 workgroups of the wide tile take 17; long reductions with 32 to 128 tiles, before and now: 1000 x 256 x
// 2560 120 -> 23, 2048 x 256 x 1920 70 -> 37, 4096 x 128 x 2560 92 -> 46).  A workgroup of 8 wavefronts owns 32 rows
// and 32 TN columns and splits the reduction: wavefront w takes the groups of eight k number w, w + 8, ...  Operands
// go straight from memory to the fp32 MFMAs (v_mfma_f32_32x32x2_f32: lane half h takes k = 4 h + e of a group in the
// e-th of its four MFMAs), four groups requested together; the partial tiles meet in LDS, added in order.
#define GSH_WAVES 8

// k = kg + 4 h .. + 3 of one row or column (elements `step` apart in memory), zeros from k_end on
template <bool KC>
__device__ __forceinline__ void gsh_load(const float *__restrict__ p, int64_t step, int64_t kg, int h, int64_t k_end,
                                         float (&out)[4])
{
    const int64_t kq = kg + 4 * h;
    if (kg + 8 <= k_end) {
        if (KC) {
            const floatx4u v = *(const floatx4u *)(p + kq);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = p[(kq + e) * step];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = kq + e < k_end;
            const float v = p[(in ? kq + e : k_end - 1) * step];
            out[e] = in ? v : 0.0f;
        }
    }
}

template <bool AT, bool BT, int TN>
__global__ void __launch_bounds__(GSH_WAVES * 64)
gemm_f32_short_kernel(GemmArgs g, float *__restrict__ partial)
{
    constexpr int BN = 32 * TN;
    constexpr int AHEAD = 4;
    __shared__ float part[GSH_WAVES][32 * BN];
    const int lane = pccnn_lane();
    const int wave = threadIdx.x >> 6;
    const int r = lane & 31, h = lane >> 5;
    const GemmTile t = gemm_tile<32, BN>(g);
    if (!t.valid) return;
    const int64_t row = t.bm + r < g.rows ? t.bm + r : g.rows - 1;
    const float *a = g.a + (int64_t)t.batch * g.stride_a + (AT ? row : row * g.lda);
    const float *b = g.b + (int64_t)t.batch * g.stride_b;
    const float *bc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int64_t col = t.bn + 32 * j + r < g.cols ? t.bn + 32 * j + r : g.cols - 1;
        bc[j] = b + (BT ? col * g.ldb : col);
    }
    floatx16 acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.0f;

    for (int64_t k0 = t.k_begin + wave * 8; k0 < t.k_end; k0 += AHEAD * GSH_WAVES * 8) {
        float fa[AHEAD][4], fb[AHEAD][TN][4];
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            const int64_t kg = k0 + q * (GSH_WAVES * 8);            // uniform over the wavefront
            if (kg >= t.k_end) break;
            gsh_load<!AT>(a, AT ? g.lda : 1, kg, h, t.k_end, fa[q]);
#pragma unroll
            for (int j = 0; j < TN; ++j) gsh_load<BT>(bc[j], BT ? 1 : g.ldb, kg, h, t.k_end, fb[q][j]);
        }
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            if (k0 + q * (GSH_WAVES * 8) >= t.k_end) break;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[q][e], fb[q][j][e], acc[j], 0, 0, 0);
        }
    }
    // register v of lane l: row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32 of the tile
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) part[wave][(8 * (v / 4) + 4 * h + v % 4) * BN + 32 * j + r] = acc[j][v];
    __syncthreads();
    int64_t ldc;
    float *cbase = gemm_output(g, t, partial, ldc);
    for (int e = threadIdx.x; e < 32 * BN; e += GSH_WAVES * 64) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < GSH_WAVES; ++w) s += part[w][e];
        const int64_t orow = t.bm + e / BN, ocol = t.bn + e % BN;
        if (orow < g.rows && ocol < g.cols) cbase[orow * ldc + ocol] = s;
    }
}

// Sums the partial products in a fixed order.  LANES threads share an output element (each adds every LANES-th run of
// splits, eight loads in flight) and meet in LDS: with few elements and many splits one thread's chain of loads would
// be the whole time.
template <int LANES>
__global__ void __launch_bounds__(256)
splitk_reduce_kernel(const float *__restrict__ partial, float *__restrict__ c, int64_t rows, int64_t cols, int64_t ldc,
                     int64_t stride_c, int split_k, int batch_count)
{
    constexpr int COLS = 256 / LANES;
    __shared__ float part[LANES][COLS];
    const int64_t per = rows * cols;
    const int64_t total = per * batch_count;
    const int col = threadIdx.x % COLS, lane = threadIdx.x / COLS;
    const int run = (split_k + LANES - 1) / LANES;
    const int k0 = lane * run, k1 = k0 + run < split_k ? k0 + run : split_k;
    for (int64_t base = (int64_t)blockIdx.x * COLS; base < total; base += (int64_t)gridDim.x * COLS) {
        const int64_t i = base + col;
        const int64_t bi = i / per, e = i % per;
        float s = 0.0f;
        if (i < total) {
            const float *src = partial + bi * split_k * per + e;
            int k = k0;
            for (; k + 8 <= k1; k += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = src[(int64_t)(k + u) * per];
#pragma unroll
                for (int u = 0; u < 8; ++u) s += v[u];
            }
            for (; k < k1; ++k) s += src[(int64_t)k * per];
        }
        if (LANES > 1) {
            part[lane][col] = s;
            __syncthreads();
            if (lane == 0) {
#pragma unroll
                for (int l = 1; l < LANES; ++l) s += part[l][col];
            }
            __syncthreads();
        }
        if (lane == 0 && i < total) c[bi * stride_c + (e / cols) * ldc + (e % cols)] = s;
    }
}

int pccnn_splitk_reduce(const float *partial, float *c, int64_t rows, int64_t cols, int64_t ldc, int64_t stride_c,
                        int split_k, int batch, hipStream_t s)
{
    const int64_t total = rows * cols * batch;
    // one thread per element when that fills the chip, two when it nearly does (64 parts of 480 x 256, whole products of
    // 20 000 samples: 28.6 us with one, 28.3 with two, 30.6 with eight; 512 x 128: 23.3 with one, 22.2 with eight)
    const int lanes = total >= (1 << 17) || split_k <= 8 ? 1 : (total > (1 << 16) ? 2 : 8);
    int64_t blocks = pccnn_ceil_div(total * lanes, 256);
    if (blocks > 4096) blocks = 4096;
    if (lanes == 1)
        splitk_reduce_kernel<1><<<(unsigned)blocks, 256, 0, s>>>(partial, c, rows, cols, ldc, stride_c, split_k, batch);
    else if (lanes == 2)
        splitk_reduce_kernel<2><<<(unsigned)blocks, 256, 0, s>>>(partial, c, rows, cols, ldc, stride_c, split_k, batch);
    else
        splitk_reduce_kernel<8><<<(unsigned)blocks, 256, 0, s>>>(partial, c, rows, cols, ldc, stride_c, split_k, batch);
    PCCNN_LAUNCH_CHECK();
    return PCCNN_OK;
}

// Which tile a product takes: (rows, columns) of a workgroup's tile; `is_short`: the short kernel.
struct GemmPlan {
    int bm, bn;
    bool is_short;
};

static int64_t gemm_tiles(int64_t rows, int64_t cols, int bm, int bn)
{
    return pccnn_ceil_div(rows, bm) * pccnn_ceil_div(cols, bn);
}

// `copies`: how many times the tiles of one product are in the launch (batch x split).
static GemmPlan gemm_plan(int64_t rows, int64_t cols, int64_t copies, int64_t lda, int64_t ldb)
{
    // the wide tile that pads the columns least, weighted with what a column costs in it (65 536 x 256 x 1920: 352 us
    // with 128 columns, 392 with 64)
    GemmPlan p = {128, 128, false};
    if (cols <= 32) p.bn = 32;
    else if (cols <= 64) p.bn = 64;
    else {
        const double c128 = 1.0 * pccnn_ceil_div(cols, 128) * 128, c96 = 1.08 * pccnn_ceil_div(cols, 96) * 96,
                     c64 = 1.12 * pccnn_ceil_div(cols, 64) * 64;
        p.bn = c128 <= c96 && c128 <= c64 ? 128 : (c96 <= c64 ? 96 : 64);
    }
    // nearly two workgroups per CU (of the 96-column tile one) or the 64 x 64 tile: 14 065 x 64 x 512 20 us with 110
    // workgroups of 128 x 64, 16 with 220; 12 000 x 250 x 200 17.7 with 376, 16.1 with 752; 37 675 x 96 x 720 51 with
    // 295 workgroups of 128 x 96, 56 with 1178
    if (p.bn > 32 && gemm_tiles(rows, cols, 128, p.bn) * copies < (p.bn == 96 ? 256 : 448)) p.bm = p.bn = 64;
    // (rows of 9 000 000, 256 x 128 in 64 parts: 5.5 ms with 64 x 64 tiles, 8.6 in the short kernel)
    if (!gemm_tile_fits(128, lda) || !gemm_tile_fits(128, ldb)) p.bm = p.bn = 64;
    if (gemm_tiles(rows, cols, p.bm, p.bn) * copies <= 128 || !gemm_tile_fits(64, lda) || !gemm_tile_fits(64, ldb)) {
        p.is_short = true;
        p.bm = 32;
        p.bn = cols > 32 && gemm_tiles(rows, cols, 32, 64) * copies > 256 ? 64 : 32;
    }
    return p;
}

// A split of the reduction for a product whose output has few tiles (d_weights = P^T x dOut): two workgroups per CU of
// the wide tile with 512 or more of the reduction each, else of the 64 x 64 tile with 128 or more.  What
// the split writes and the last kernel reads again is bounded by the workspace.
int pccnn_gemm_f32_split(int64_t rows, int64_t cols, int64_t inner, int batch, size_t workspace_floats)
{
    if (inner < 512 || rows < 1 || cols < 1) return 1;
    const int64_t room = (int64_t)(workspace_floats / ((size_t)rows * cols * batch));
    const int64_t most = room < 512 ? room : 512;
    const GemmPlan wide = gemm_plan(rows, cols, 1 << 20, 1, 1);
    // (not more than two per CU: 540 workgroups of 1920 x 256 x 65 536 take 485 us, 510 take 386)
    int64_t split = 512 / (gemm_tiles(rows, cols, 128, wide.bn) * batch);
    if (split < 1) split = 1;
    if (split > most || inner / split < 512) {
        split = 512 / (gemm_tiles(rows, cols, wide.bn > 32 ? 64 : 128, wide.bn > 32 ? 64 : 32) * batch);
        if (split > inner / 128) split = inner / 128;
        if (split > most) split = most;
    }
    return split < 1 ? 1 : (int)split;
}

extern "C" int pccnn_gemm_f32(const float *a, const float *b, float *c, int64_t rows, int64_t cols, int64_t inner,
                              int a_trans, int b_trans, int64_t lda, int64_t ldb, int64_t ldc, int batch,
                              int64_t stride_a, int64_t stride_b, int64_t stride_c, int split_k, void *workspace,
                              size_t workspace_bytes, void *stream)
{
    PCCNN_REQUIRE(rows >= 0 && cols >= 0 && inner >= 0 && batch >= 1, PCCNN_ERR_INVALID,
                  "pccnn_gemm_f32: rows=%lld cols=%lld inner=%lld batch=%d", (long long)rows, (long long)cols,
                  (long long)inner, batch);
    if (rows == 0 || cols == 0) return PCCNN_OK;
    PCCNN_REQUIRE(a && b && c, PCCNN_ERR_INVALID, "pccnn_gemm_f32: null pointer");
    PCCNN_REQUIRE(lda >= (a_trans ? rows : inner) && ldb >= (b_trans ? inner : cols) && ldc >= cols, PCCNN_ERR_INVALID,
                  "pccnn_gemm_f32: leading dimension too small (lda=%lld ldb=%lld ldc=%lld)", (long long)lda,
                  (long long)ldb, (long long)ldc);
    if (split_k < 1) split_k = 1;
    GemmPlan plan = gemm_plan(rows, cols, (int64_t)batch * split_k, lda, ldb);
    GemmArgs g;
    g.a = a; g.b = b; g.c = c;
    g.rows = rows; g.cols = cols; g.inner = inner;
    g.lda = lda; g.ldb = ldb; g.ldc = ldc;
    g.stride_a = stride_a; g.stride_b = stride_b; g.stride_c = stride_c;
    const int unit = plan.is_short ? GSH_WAVES * 8 : GS_K;
    const int64_t chunk = pccnn_ceil_div(pccnn_ceil_div(inner > 0 ? inner : 1, split_k), unit) * unit;
    split_k = (int)pccnn_ceil_div(inner > 0 ? inner : 1, chunk);
    g.split_k = split_k;
    g.k_chunk = chunk;
    float *partial = nullptr;
    if (split_k > 1) {
        size_t need = (size_t)batch * split_k * rows * cols * sizeof(float);
        PCCNN_REQUIRE(workspace && workspace_bytes >= need, PCCNN_ERR_WORKSPACE,
                      "pccnn_gemm_f32: split-k workspace of %zu bytes, need %zu", workspace_bytes, need);
        partial = (float *)workspace;
    }
    hipStream_t s = (hipStream_t)stream;
    g.tiles_x = (int)pccnn_ceil_div(cols, plan.bn);
    g.tiles_y = (int)pccnn_ceil_div(rows, plan.bm);
    g.total_wg = (int64_t)g.tiles_x * g.tiles_y * batch * split_k;
    PCCNN_REQUIRE(g.total_wg < (1ll << 31) - GEMM_XCDS, PCCNN_ERR_UNSUPPORTED, "pccnn_gemm_f32: grid too large");
    dim3 grid((unsigned)(pccnn_ceil_div(g.total_wg, GEMM_XCDS) * GEMM_XCDS));
    {
        PccnnTimed timed(PCCNN_T_GEMM, s);
#define SPLIT_GO(AT, BT, WM, WN, TM, TN)                                                                          \
    do {                                                                                                          \
        if (chunk > GS_ONE_SUM) gemm_f32_split_kernel<AT, BT, WM, WN, TM, TN, true><<<grid, 256, 0, s>>>(g, partial); \
        else gemm_f32_split_kernel<AT, BT, WM, WN, TM, TN, false><<<grid, 256, 0, s>>>(g, partial);                 \
    } while (0)
#define GEMM_GO(AT, BT)                                                                                           \
    do {                                                                                                          \
        if (plan.is_short) {                                                                                      \
            if (plan.bn == 64) gemm_f32_short_kernel<AT, BT, 2><<<grid, GSH_WAVES * 64, 0, s>>>(g, partial);      \
            else gemm_f32_short_kernel<AT, BT, 1><<<grid, GSH_WAVES * 64, 0, s>>>(g, partial);                    \
        } else if (plan.bm == 64) SPLIT_GO(AT, BT, 2, 2, 1, 1);                                                   \
        else if (plan.bn == 128) SPLIT_GO(AT, BT, 2, 2, 2, 2);                                                    \
        else if (plan.bn == 96) SPLIT_GO(AT, BT, 4, 1, 1, 3);                                                     \
        else if (plan.bn == 64) SPLIT_GO(AT, BT, 2, 2, 2, 1);                                                     \
        else SPLIT_GO(AT, BT, 4, 1, 1, 1);                                                                        \
    } while (0)
        if (!a_trans && !b_trans) GEMM_GO(false, false);
        else if (!a_trans && b_trans) GEMM_GO(false, true);
        else if (a_trans && !b_trans) GEMM_GO(true, false);
        else GEMM_GO(true, true);
#undef GEMM_GO
#undef SPLIT_GO
    }
    PCCNN_LAUNCH_CHECK();
    if (split_k > 1) return pccnn_splitk_reduce(partial, c, rows, cols, ldc, stride_c, split_k, batch, s);
    return PCCNN_OK;
}
