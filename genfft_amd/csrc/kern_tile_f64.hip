// kern_tile_f64.hip -- complex128 tile-kernel shapes.
//
// Same three families as complex64 (rows, column tiles, transposing rows)
// with half the elements per tile, since each element is 16 bytes: rows hold
// 2048 complex (32 KB) up to L = 128 and are held in registers from L = 256 on
// (gfft_regtile.h); column tiles are >= 8 columns (128-byte segments) where
// LDS allows.
#include "gfft_registry.h"

namespace gfft {
namespace {
using T = double;
constexpr int R_ = PAT_ROW, C_ = PAT_COL, S_ = LAY_SEQ, E_ = LAY_ELEM;

const KernelEntry kTable[] = {
    // --- batched rows ---
    make_entry<T, 2, 512, 64, S_, R_, R_, 2>(),
    make_entry<T, 4, 512, 128, S_, R_, R_, 4>(),
    make_entry<T, 8, 256, 128, S_, R_, R_, 8>(),
    make_entry<T, 16, 128, 128, S_, R_, R_, 16>(),
    make_entry<T, 32, 64, 128, S_, R_, R_, 8, 4>(),
    make_entry<T, 64, 32, 128, S_, R_, R_, 8, 8>(),
    make_entry<T, 128, 16, 128, S_, R_, R_, 16, 8>(),
    // tuner alternatives to the register-held rows below, and the kernels of
    // layouts past their 32-bit offsets; radix <= 8 and 8 elements per thread:
    // an FP64 radix-16 butterfly holds 64 VGPRs of data plus 60 of twiddles
    // (148-190 VGPRs per kernel); the radix-8 forms use 83-116 and run 25-30%
    // faster (MI355X, 1 GiB batches: L = 1024 0.624 -> 0.449 ms, 8192 0.787 ->
    // 0.569 ms)
    make_variant<T, 256, 8, 256, S_, R_, R_, 8, 8, 4>(),
    make_variant<T, 512, 4, 256, S_, R_, R_, 8, 8, 8>(),
    make_variant<T, 1024, 2, 256, S_, R_, R_, 8, 4, 8, 4>(),
    make_variant<T, 2048, 1, 256, S_, R_, R_, 8, 8, 8, 4>(),
    make_variant<T, 4096, 1, 512, S_, R_, R_, 8, 8, 8, 8>(),
    make_variant<T, 8192, 1, 1024, S_, R_, R_, 8, 8, 8, 8, 2>(),
    // --- column tiles ---
    make_entry<T, 2, 256, 64, E_, C_, C_, 2>(),
    make_entry<T, 4, 256, 64, E_, C_, C_, 4>(),
    make_entry<T, 8, 128, 64, E_, C_, C_, 8>(),
    make_entry<T, 16, 64, 64, E_, C_, C_, 16>(),
    make_entry<T, 32, 32, 64, E_, C_, C_, 8, 4>(),
    make_entry<T, 64, 32, 128, E_, C_, C_, 8, 8>(),
    make_entry<T, 128, 16, 128, E_, C_, C_, 16, 8>(),
    make_entry<T, 256, 8, 128, E_, C_, C_, 16, 16>(),
    make_entry<T, 512, 8, 256, E_, C_, C_, 8, 8, 8>(),
    make_entry<T, 1024, 8, 512, E_, C_, C_, 16, 16, 4>(),
    make_entry<T, 2048, 4, 512, E_, C_, C_, 16, 8, 16>(),  // c128 2^22 column pass 0.62-0.63 ms (16*16*8: 0.64)
    // --- transposing rows ---
    make_entry<T, 64, 32, 128, S_, R_, C_, 8, 8>(),
    make_entry<T, 128, 16, 128, S_, R_, C_, 16, 8>(),
    make_entry<T, 256, 8, 128, S_, R_, C_, 16, 16>(),
    make_entry<T, 512, 8, 256, S_, R_, C_, 8, 8, 8>(),
    make_entry<T, 1024, 8, 512, S_, R_, C_, 16, 16, 4>(),
    make_entry<T, 2048, 4, 512, S_, R_, C_, 16, 16, 8>(),
    make_entry<T, 4096, 2, 512, S_, R_, C_, 16, 16, 16>(),
    // --- persistent pipelined forms of the 2^20 four-step passes ---
    make_pipe_entry<T, 1024, 8, 512, E_, C_, C_, 16, 16, 4>(),
    make_pipe_entry<T, 1024, 8, 512, S_, R_, C_, 16, 16, 4>(),
    // --- autotuner alternatives ---
    make_variant<T, 1024, 4, 256, S_, R_, R_, 16, 16, 4>(),
    make_variant<T, 1024, 2, 128, S_, R_, R_, 4, 16, 16>(),
    make_variant<T, 2048, 2, 256, S_, R_, R_, 16, 16, 8>(),
    make_variant<T, 1024, 4, 512, S_, R_, R_, 8, 4, 8, 4>(),
    make_variant<T, 2048, 2, 512, S_, R_, R_, 8, 8, 8, 4>(),
    // the radix-16 forms
    make_variant<T, 256, 8, 128, S_, R_, R_, 16, 16>(),
    make_variant<T, 512, 4, 128, S_, R_, R_, 8, 8, 8>(),
    make_variant<T, 1024, 2, 128, S_, R_, R_, 16, 16, 4>(),
    make_variant<T, 2048, 1, 128, S_, R_, R_, 16, 16, 8>(),
    make_variant<T, 4096, 1, 256, S_, R_, R_, 16, 16, 16>(),
    make_variant<T, 8192, 1, 512, S_, R_, R_, 16, 16, 8, 4>(),
    // --- rows held in registers.  MI355X against the LDS tiles above, 1 GiB
    // batches (streaming loads) / 256 MiB batches (plain loads) / one row:
    // 256 points 0.374 -> 0.350 ms / 0.101 -> 0.063 ms / 4.1 -> 3.9 us, 1024
    // 0.378 -> 0.349 / 0.101 -> 0.068 / 4.9 -> 4.6, 4096 0.417 -> 0.362 /
    // 0.116 -> 0.090 / 7.5 -> 6.2, 8192 0.579 -> 0.345 / 0.157 -> 0.083 /
    // 12.8 -> 10.3; 16384 points against the four-step 0.77 -> 0.435 ms ---
    make_reg_entry<T, 256, 8, 256, R_, R_, 8, 4, 8>(),
    make_reg_wide<T, 256, 8, 256, 8, 4, 8>(),
    make_reg_entry<T, 512, 4, 256, R_, R_, 8, 8, 8>(),
    make_reg_wide<T, 512, 4, 256, 8, 8, 8>(),
    make_reg_entry<T, 1024, 2, 256, R_, R_, 8, 4, 4, 8>(),
    make_reg_wide<T, 1024, 2, 256, 8, 4, 4, 8>(),
    make_reg_entry<T, 2048, 1, 128, R_, R_, 16, 16, 8>(),
    make_reg_wide<T, 2048, 1, 128, 16, 16, 8>(),
    make_reg_entry<T, 4096, 1, 256, R_, R_, 16, 16, 16>(),
    make_reg_wide<T, 4096, 1, 256, 16, 16, 16>(),
    make_reg_entry<T, 8192, 1, 512, R_, R_, 8, 16, 8, 8>(),
    make_reg_wide<T, 8192, 1, 512, 8, 16, 8, 8>(),
    make_reg_long<T, 16384, 1024, HINT_ST, 16, 16, 8, 8>(),
    make_reg_long<T, 16384, 1024, HINT_LD | HINT_ST, 16, 16, 8, 8>(),
    // --- column tiles held in registers: 2^22 x 16 four-step columns of 2048
    // 0.612 -> 0.529 ms, transposing rows 0.563 -> 0.427; whole columns: 512 x
    // 999 8.6 -> 6.8 us, 1024 x 4999 61 -> 48, 2048 x 2048 35 -> 28 (the
    // pipelined 1024-row tile stays the four-step's: 0.469 against 0.496).  512
    // rows whose pitch is no multiple of a line stay on the LDS tile past 128
    // MiB: 16387 columns 66 against 70, 65539 249 against 290 ---
    make_reg_many<T, 2048, 8, 1024, C_, C_, 16, 8, 16>(1),
    make_reg_cols<T, 128, 8, 128, 8, 2, 8>(),
    make_reg_cols<T, 128, 16, 256, 8, 2, 8>(),
    make_reg_cols<T, 256, 4, 128, 8, 4, 8>(),
    make_reg_cols<T, 256, 8, 256, 8, 4, 8>(),
    make_reg_cols<T, 512, 4, 256, 8, 8, 8>(0, (int64_t)128 << 20),
    make_reg_cols<T, 512, 8, 512, 8, 8, 8>(0, (int64_t)128 << 20),
    make_reg_cols<T, 1024, 4, 256, 16, 4, 16>(),
    make_reg_cols<T, 1024, 8, 512, 16, 4, 16>(),
    make_reg_cols<T, 2048, 4, 512, 16, 8, 16>(),
    make_reg_cols<T, 2048, 8, 1024, 16, 8, 16>(),
    // --- transposing rows held in registers ---
    make_reg_many<T, 2048, 8, 1024, R_, C_, 16, 16, 8>(1),
    // --- short rows and columns held in registers.  Rows, us, one row / 1 MiB /
    // 32 MiB / 128 MiB, LDS -> register tile: 16 points 3.9 -> 3.0 / 5.5 -> 3.2 /
    // 14.5 -> 14.6 / LDS, 32 4.7 -> 3.4 / 6.3 -> 3.6 / 16.1 -> 12.8 / 60 -> 57,
    // 64 4.8 -> 3.5 / 6.4 -> 3.6 / 16.3 -> 12.6 / 61 -> 55, 128 4.6 -> 3.9 /
    // 6.1 -> 4.1 / 16.0 -> 13.3 / 59 -> 56; 512 MiB (streaming loads) 64 points
    // 195 -> 188, 128 193 -> 184, 32 195 -> 206 (LDS).  Columns: 32 rows x 1000
    // 4.9 -> 3.4, x 262144 54 -> 41, 64 x 300 5.2 -> 3.6, x 131072 57 -> 41 ---
    make_reg_cached<T, 16, 16, 64, 4, 4>((int64_t)64 << 20),
    make_reg_cached<T, 32, 16, 64, 8, 4>(),
    make_reg_cached<T, 64, 8, 64, 8, 8>(),
    make_reg_wide<T, 64, 8, 64, 8, 8>(),
    make_reg_cached<T, 128, 8, 128, 8, 2, 8>(),
    make_reg_wide<T, 128, 8, 128, 8, 2, 8>(),
    make_reg_cols<T, 32, 16, 64, 8, 4>(),
    make_reg_cols<T, 32, 32, 128, 8, 4>(),
    make_reg_cols<T, 64, 8, 64, 8, 8>(),
    make_reg_cols<T, 64, 32, 256, 8, 8>(),
};
// The 2^20 four-step's two pipelined passes paired in one launch (column pass
// of chunk k, transposing row pass of chunk k - 1).
using ColPass = PipeShape<T, 1024, 8, 512, E_, C_, C_, 16, 16, 4>;
using RowPass = PipeShape<T, 1024, 8, 512, S_, R_, C_, 16, 16, 4>;
const DualEntry kDual[] = {
    make_dual<ColPass, RowPass>(&tile_fft_pipe_kernel<T, 1024, 8, 512, E_, C_, C_, 16, 16, 4>,
                                &tile_fft_pipe_kernel<T, 1024, 8, 512, S_, R_, C_, 16, 16, 4>),
};
}  // namespace

const KernelEntry *tile_kernels_f64(int *count)
{
    *count = (int)(sizeof(kTable) / sizeof(kTable[0]));
    return kTable;
}

const DualEntry *dual_kernels_f64(int *count)
{
    *count = (int)(sizeof(kDual) / sizeof(kDual[0]));
    return kDual;
}

}  // namespace gfft
