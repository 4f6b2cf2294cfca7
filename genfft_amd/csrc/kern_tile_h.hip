// kern_tile_h.hip -- 16-bit storage tile kernels (FP16 and BF16 pairs, FP32
// arithmetic in LDS).
//
// The LDS shapes are the complex64 ones (rows up to L = 1024, column tiles up
// to L = 2048, transposing rows up to L = 4096): the LDS tile is FP32 in both
// cases, so the tile sizes that fit are the same; only the HBM side narrows
// to four bytes per element.  Rows from 128 points on are held in registers.
#include "gfft_registry.h"

namespace gfft {
namespace {
constexpr int R_ = PAT_ROW, C_ = PAT_COL, S_ = LAY_SEQ, E_ = LAY_ELEM;

template <class S>
struct HalfTable {
    static constexpr KernelEntry tab[] = {
        // --- batched rows ---
        make_entry_h<S, 2, 1024, 128, S_, R_, R_, 2>(),
        make_entry_h<S, 4, 1024, 256, S_, R_, R_, 4>(),
        make_entry_h<S, 8, 512, 256, S_, R_, R_, 8>(),
        make_entry_h<S, 16, 256, 256, S_, R_, R_, 16>(),
        make_entry_h<S, 32, 128, 256, S_, R_, R_, 8, 4>(),
        make_entry_h<S, 64, 64, 256, S_, R_, R_, 8, 8>(),
        make_variant_h<S, 128, 32, 256, S_, R_, R_, 16, 8>(),
        make_variant_h<S, 256, 16, 256, S_, R_, R_, 16, 16>(),
        make_variant_h<S, 512, 8, 256, S_, R_, R_, 8, 8, 8>(),
        make_variant_h<S, 1024, 4, 256, S_, R_, R_, 16, 16, 4>(),
        // --- column tiles ---
        make_entry_h<S, 2, 512, 64, E_, C_, C_, 2>(),
        make_entry_h<S, 4, 256, 64, E_, C_, C_, 4>(),
        make_entry_h<S, 8, 128, 64, E_, C_, C_, 8>(),
        make_entry_h<S, 16, 64, 64, E_, C_, C_, 16>(),
        make_entry_h<S, 32, 64, 128, E_, C_, C_, 8, 4>(),
        make_entry_h<S, 64, 64, 256, E_, C_, C_, 8, 8>(),
        make_entry_h<S, 128, 32, 256, E_, C_, C_, 16, 8>(),
        make_entry_h<S, 256, 16, 256, E_, C_, C_, 16, 16>(),
        make_entry_h<S, 512, 16, 512, E_, C_, C_, 8, 8, 8>(),
        make_entry_h<S, 1024, 16, 1024, E_, C_, C_, 16, 16, 4>(),
        make_entry_h<S, 2048, 8, 1024, E_, C_, C_, 16, 16, 8>(),
        // --- transposing rows ---
        make_entry_h<S, 64, 64, 256, S_, R_, C_, 8, 8>(),
        make_entry_h<S, 128, 32, 256, S_, R_, C_, 16, 8>(),
        make_entry_h<S, 256, 16, 256, S_, R_, C_, 16, 16>(),
        make_entry_h<S, 512, 16, 512, S_, R_, C_, 8, 8, 8>(),
        make_entry_h<S, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>(),
        make_entry_h<S, 2048, 8, 1024, S_, R_, C_, 16, 16, 8>(),
        make_entry_h<S, 4096, 4, 1024, S_, R_, C_, 16, 16, 16>(),
        // --- persistent pipelined forms of the 2^20 four-step passes ---
        make_pipe_entry_h<S, 1024, 16, 1024, E_, C_, C_, 8, 8, 16>(),
        make_pipe_entry_h<S, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>(),
        // --- rows held in registers, whole rows, so that the automatic scale
        // needs no pass over the input of its own.  MI355X, us per call, LDS
        // tiles -> these, scaled / unscaled: 1024 points x 1024 125 -> 6.1 /
        // 6.4 -> 5.9; 4096 x 4096 59.0 -> 38.3 / 38.6 -> 36.1; 4096 x 32768 399
        // -> 270 / 288 -> 243; 16384 x 8192 565 -> 314 / 444 -> 302.  8-byte
        // lanes of rows of 32 or 64 points fetch 32-byte pieces: those keep the
        // LDS tiles past the Infinity Cache (64 x 2^21 213 against 254 us) ---
        make_reg_cached_h<S, HINT_NONE, 32, 32, 128, 4, 2, 4>(),
        make_reg_cached_h<S, HINT_NONE, 64, 16, 64, 8, 8>(),
        make_reg_rows_h<S, HINT_ST, 128, 8, 64, 8, 2, 8>(),
        make_reg_rows_h<S, HINT_ST, 256, 4, 64, 8, 4, 8>(),
        make_reg_rows_h<S, HINT_ST, 512, 4, 128, 8, 8, 8>(),
        make_reg_rows_h<S, HINT_ST, 1024, 2, 128, 8, 16, 8>(),
        make_reg_rows_h<S, HINT_ST, 2048, 1, 128, 8, 4, 8, 8>(),
        make_reg_rows_h<S, HINT_ST, 4096, 1, 256, 8, 8, 8, 8>(),
        make_reg_rows_h<S, HINT_ST, 8192, 1, 512, 8, 16, 8, 8>(),
        make_reg_rows_h<S, HINT_ST, 16384, 1, 512, 16, 8, 8, 16>(),
    };
};
}  // namespace

const KernelEntry *tile_kernels_f16(int *count)
{
    *count = (int)(sizeof(HalfTable<st_f16>::tab) / sizeof(KernelEntry));
    return HalfTable<st_f16>::tab;
}

const KernelEntry *tile_kernels_bf16(int *count)
{
    *count = (int)(sizeof(HalfTable<st_bf16>::tab) / sizeof(KernelEntry));
    return HalfTable<st_bf16>::tab;
}

}  // namespace gfft
