// Walks the loads of one operand of the fp32 contraction's split kernel on the CPU, in the order of SplitOperand (init,
// load, load_last): every thread of the first and last tile, every split, the first and last step without checks and
// the checked one.
#include "../pccnn_lib_amd/csrc/gemm_tiles.h"

namespace {

struct Operand {
    int64_t extent, inner, ld;
    bool kc;
    // one past the last element that the matrix has
    int64_t size() const { return kc ? (extent - 1) * ld + inner : (inner - 1) * ld + extent; }
    int64_t at(int64_t x, int64_t k) const { return kc ? x * ld + k : k * ld + x; }
};

struct Tally {
    int64_t outside = 0, wrong = 0;
    void see(const Operand &o, int64_t element, int64_t x, int64_t k, int64_t k_end)
    {
        if (element < 0 || element >= o.size()) ++outside;
        if (x < o.extent && k < k_end && element != o.at(x, k)) ++wrong;
    }
};

template <bool KC, int X>
void walk(const Operand &o, int other_w, int64_t other_extent, int64_t k_chunk, Tally &tally)
{
    typedef GemmUnits<KC, X> U;
    const int64_t last_tile = (o.extent - 1) / X * X;
    for (int64_t x0 = 0; x0 <= last_tile; x0 += last_tile > 0 ? last_tile : 1) {
        for (int64_t k0 = 0; k0 == 0 || k0 < o.inner; k0 += k_chunk) {
            const int64_t k_end = k0 + k_chunk < o.inner ? k0 + k_chunk : o.inner;
            const int64_t steps = gemm_steps(k_end - k0);
            const int64_t unchecked = gemm_steps_unchecked(k_end - k0, U::W, o.extent, other_w, other_extent);
            if (unchecked < 0) { ++tally.wrong; continue; }
            const int x_left = U::rows_left(x0, o.extent);
            for (int64_t step = 0; step < steps; ++step) {
                if (step != 0 && step < unchecked - 1) continue;
                const int64_t base = U::origin(x0, k0, o.ld) + step * U::advance(o.ld), k = k0 + step * GS_K;
                for (int thread = 0; thread < 256; ++thread)
                    for (int i = 0; i < U::PASSES && U::active(thread, i); ++i) {
                        int x, k8;
                        U::unit(thread, i, x, k8);
                        // the kernel's offsets are 32-bit bytes
                        const uint64_t bytes = 4 * ((uint64_t)(KC ? X - 1 : 24) * (uint64_t)o.ld + GS_K + X);
                        if (gemm_tile_fits(X, o.ld) && bytes >> 32) ++tally.outside;
                        for (int e = 0; e < 8; ++e)
                            for (int w = 0; w < U::W; ++w) {
                                const int k_left = (int)(k_end - k), in = step < unchecked || k8 * 8 < k_left;
                                const int64_t element =
                                    step < unchecked || U::whole_units(x_left, k_left)
                                        ? base + U::offset(x, in ? k8 : 0, x_left, (unsigned)o.ld) + (KC ? e : e * o.ld + w)
                                        : base + U::checked(x + w, k8 * 8 + e, x_left, k_left, o.ld);
                                // (a row that lies in the next tile belongs to that tile)
                                tally.see(o, element, x + w < x_left ? x0 + x + w : o.extent, k + k8 * 8 + e, k_end);
                            }
                    }
            }
        }
    }
}

}  // namespace

// Elements read outside the operand, and elements of it read from the wrong place, for `extent` rows (or columns) in
// tiles of `tile`.
extern "C" void gemm_bounds(int kc, int tile, int64_t extent, int64_t inner, int64_t ld, int other_w, int64_t other_extent,
                            int64_t k_chunk, int64_t *outside, int64_t *wrong)
{
    const Operand o = {extent, inner, ld, kc != 0};
    Tally tally;
    switch (tile) {
    case 128: kc ? walk<true, 128>(o, other_w, other_extent, k_chunk, tally) : walk<false, 128>(o, other_w, other_extent, k_chunk, tally); break;
    case 96: kc ? walk<true, 96>(o, other_w, other_extent, k_chunk, tally) : walk<false, 96>(o, other_w, other_extent, k_chunk, tally); break;
    case 64: kc ? walk<true, 64>(o, other_w, other_extent, k_chunk, tally) : walk<false, 64>(o, other_w, other_extent, k_chunk, tally); break;
    default: kc ? walk<true, 32>(o, other_w, other_extent, k_chunk, tally) : walk<false, 32>(o, other_w, other_extent, k_chunk, tally);
    }
    *outside = tally.outside;
    *wrong = tally.wrong;
}

extern "C" int bf16_split(int64_t rows, int64_t cols, int64_t inner, int batch, int64_t workspace_floats)
{
    return gemm_bf16_split(rows, cols, inner, batch, (size_t)workspace_floats);
}

extern "C" int tile_fits(int rows, int64_t ld) { return gemm_tile_fits(rows, ld); }
