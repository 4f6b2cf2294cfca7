// kern_tile_f32.hip -- complex64 tile-kernel shapes.
//
// Rows (PAT_ROW -> PAT_ROW, sequence-major LDS): batched 1D transforms and
// the 2D row pass; a tile holds 4096 complex (32 KB)
// up to L = 2048.
// Columns (PAT_COL -> PAT_COL, element-major LDS): the first pass of a
// four-step transform and the 2D column pass; M adjacent columns give
// >= 64-byte contiguous row segments.
// Transposing rows (PAT_ROW -> PAT_COL): the second four-step pass, writing
// element k of row k1 to k1 + N1*k, M rows wide.
// Every default LDS shape keeps 16 elements per thread, so radix-16 butterflies
// live entirely in registers (the radix-32 alternatives hold 32).  Rows
// within the Infinity Cache and from 4096 points on are held in registers
// (gfft_regtile.h).
#include "gfft_registry.h"

namespace gfft {
namespace {
using T = float;
constexpr int R_ = PAT_ROW, C_ = PAT_COL, S_ = LAY_SEQ, E_ = LAY_ELEM;

const KernelEntry kTable[] = {
    // --- batched rows ---
    make_entry<T, 2, 1024, 128, S_, R_, R_, 2>(),
    make_entry<T, 4, 1024, 256, S_, R_, R_, 4>(),
    make_entry<T, 8, 512, 256, S_, R_, R_, 8>(),
    make_entry<T, 16, 256, 256, S_, R_, R_, 16>(),
    make_entry<T, 32, 128, 256, S_, R_, R_, 8, 4>(),
    make_entry<T, 64, 64, 256, S_, R_, R_, 8, 8>(),
    make_variant<T, 128, 32, 256, S_, R_, R_, 16, 8>(),
    make_entry<T, 256, 16, 256, S_, R_, R_, 16, 16>(),
    make_entry<T, 512, 8, 256, S_, R_, R_, 8, 8, 8>(),
    make_variant<T, 1024, 4, 256, S_, R_, R_, 16, 16, 4>(),
    make_entry<T, 2048, 2, 256, S_, R_, R_, 16, 16, 8>(),
    make_variant<T, 4096, 1, 256, S_, R_, R_, 16, 16, 16>(),
    make_variant<T, 8192, 1, 512, S_, R_, R_, 16, 16, 8, 4>(),
    make_variant<T, 16384, 1, 1024, S_, R_, R_, 16, 16, 16, 4>(),
    // --- column tiles ---
    make_entry<T, 2, 512, 64, E_, C_, C_, 2>(),
    make_entry<T, 4, 256, 64, E_, C_, C_, 4>(),
    make_entry<T, 8, 128, 64, E_, C_, C_, 8>(),
    make_entry<T, 16, 64, 64, E_, C_, C_, 16>(),
    make_entry<T, 32, 64, 128, E_, C_, C_, 8, 4>(),
    make_entry<T, 64, 64, 256, E_, C_, C_, 8, 8>(),
    make_entry<T, 128, 32, 256, E_, C_, C_, 16, 8>(),
    make_entry<T, 256, 16, 256, E_, C_, C_, 16, 16>(),
    make_variant<T, 512, 16, 512, E_, C_, C_, 8, 8, 8>(),
    make_entry<T, 1024, 16, 1024, E_, C_, C_, 16, 16, 4>(),
    make_entry<T, 1024, 8, 512, E_, C_, C_, 16, 16, 4>(),
    make_entry<T, 2048, 8, 1024, E_, C_, C_, 16, 8, 16>(),  // c64 2^22 column pass 0.550 ms (16*16*8: 0.592, 8*16*16: 0.565)
    make_entry<T, 4096, 4, 1024, E_, C_, C_, 16, 16, 16>(),  // 32-byte rows: column transforms only, not four-step
    // --- transposing rows ---
    make_entry<T, 64, 64, 256, S_, R_, C_, 8, 8>(),
    make_entry<T, 128, 32, 256, S_, R_, C_, 16, 8>(),
    make_entry<T, 256, 16, 256, S_, R_, C_, 16, 16>(),
    make_entry<T, 512, 16, 512, S_, R_, C_, 8, 8, 8>(),
    make_entry<T, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>(),
    make_entry<T, 1024, 8, 512, S_, R_, C_, 16, 16, 4>(),
    make_entry<T, 2048, 8, 1024, S_, R_, C_, 16, 16, 8>(),
    make_entry<T, 4096, 4, 1024, S_, R_, C_, 16, 16, 16>(),
    // --- persistent pipelined forms, kept where they measured faster on
    // MI355X (c64 2^20 x 128: column pass 0.565 -> 0.524 ms, transposing row
    // pass 0.462 -> 0.392 ms); the L = 512 / 2048 and M = 8 forms fall to
    // one workgroup per CU and lose to the plain kernels (c64 2^22 x 32,
    // L = 2048, M = 8: column pass 0.63-0.72 ms pipelined, with or without
    // tile runs, against 0.59; transposing row pass 0.55 against 0.50) ---
    // column pass, radix 16 * 4 * 16: measured on c64 2^20 x 128 against the
    // other orders at 1024 threads, 0.440-0.443 ms (8*8*16: 0.464, 4*16*16:
    // 0.479, 16*16*4: 0.493; the transposing row pass does not move with order)
    make_pipe_entry<T, 1024, 16, 1024, E_, C_, C_, 16, 4, 16>(),
    make_pipe_entry<T, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>(),
    // (tuner alternative) single 16384-point sequences (tile: 136 KB of LDS);
    // radix 16*4*16*16:
    // c64 2^14 x 8192 0.500 ms with the pass twiddles read from global memory
    // (16*16*16*4: 0.509, 16*16*4*16: 0.502, 4*16*16*16: 0.521), 0.442 ms with
    // the last pass's twiddles generated from a 4 KB table in LDS
    // (PassTw::GEN: the first three passes' 8 KB of tables fit beside it)
    make_pipe_variant<T, 16384, 1, 1024, S_, R_, R_, 16, 4, 16, 16>(),
    // --- autotuner alternatives: radix order, tile width, threads per tile.
    // The double-width row tiles (64 KB, 512 threads; make_wide_variant) are
    // also the planner's choice for batches of >= 512 MiB: measured on MI355X
    // through the autotuner, 1 GiB batches ran 3-5% faster on them (L = 256:
    // 0.385 -> 0.372 ms, 512: 0.385 -> 0.365, 1024: 0.379 -> 0.365, 2048:
    // 0.388 -> 0.367), 256 MiB batches (within the Infinity Cache) 0-12% slower ---
    make_wide_variant<T, 256, 32, 512, S_, R_, R_, 16, 16>(),
    make_variant<T, 512, 8, 256, S_, R_, R_, 16, 8, 4>(),
    make_wide_variant<T, 512, 16, 512, S_, R_, R_, 8, 8, 8>(),
    make_variant<T, 1024, 4, 256, S_, R_, R_, 4, 16, 16>(),
    make_variant<T, 1024, 4, 256, S_, R_, R_, 8, 8, 16>(),
    make_wide_variant<T, 1024, 8, 512, S_, R_, R_, 16, 16, 4>(),
    make_variant<T, 1024, 2, 128, S_, R_, R_, 16, 16, 4>(),
    make_variant<T, 1024, 4, 128, S_, R_, R_, 32, 32>(),   // two radix-32 passes, 32 elements per thread
    make_variant<T, 1024, 8, 256, S_, R_, R_, 32, 32>(),
    make_variant<T, 2048, 2, 256, S_, R_, R_, 8, 16, 16>(),
    make_wide_variant<T, 2048, 4, 512, S_, R_, R_, 16, 16, 8>(),
    make_variant<T, 4096, 2, 512, S_, R_, R_, 16, 16, 16>(),
    make_variant<T, 4096, 1, 512, S_, R_, R_, 8, 8, 8, 8>(),
    make_variant<T, 8192, 1, 512, S_, R_, R_, 16, 16, 16, 2>(),
    make_variant<T, 16384, 1, 1024, S_, R_, R_, 16, 16, 8, 8>(),
    // one wavefront per 1024-point row, lanes exchanged by DPP / permlane swaps
    make_wave_entry<256>(),
    // --- rows held in registers.  Short ones: few elements per thread and no
    // load, store or pass sweep through LDS, so a small batch's one round of
    // tiles ends sooner and within the Infinity Cache the loads and stores of
    // more workgroups overlap.  Past it the LDS tiles' 16-byte accesses win up
    // to 2048 points.  MI355X, us per call, one row / 4 MiB / 64 MiB, LDS tile
    // -> register tile: 64 points 4.9 -> 3.5 / 5.4 -> 4.1 (8192 rows; LDS
    // beyond), 256: 4.9 -> 4.2 / 5.5 -> 4.8 / 25.8 -> 24.1, 512: 5.3 -> 4.3 /
    // 5.8 -> 4.9 / 25.9 -> 24.1, 2048: 6.1 -> 4.7 / 6.4 -> 5.4 / 27.1 -> 24.1,
    // 4096: 5.9 -> 5.5 / 6.6 -> 6.1 / 28.5 -> 25.0.  Long ones (LDS plane 34 /
    // 69 / 135 KB: four / two / one workgroup per CU), 1 GiB batches with
    // streaming loads: 4096 points 0.392 -> 0.369 ms, 8192 0.427 -> 0.352,
    // 16384 0.435 -> 0.378, 32768 0.72 -> 0.46 (four-step); 256 MiB batches:
    // 8192 0.087 -> 0.067, 16384 0.104 -> 0.080.  The streaming 16384-point
    // tile runs 16*4*16*16 with 1024 threads, the order of the LDS tile before
    // it: 0.387 ms (32*32*16 with 512: 0.375) ---
    make_reg_narrow<T, 16, 32, 64, 4, 4>(),
    make_reg_narrow<T, 32, 16, 64, 8, 4>(),
    make_reg_narrow<T, 64, 8, 64, 8, 8>(),
    make_reg_entry<T, 128, 16, 256, R_, R_, 8, 2, 8>(),
    make_reg_cached<T, 256, 8, 256, 8, 4, 8>(),
    make_reg_cached<T, 512, 4, 256, 8, 8, 8>(),
    make_reg_narrow<T, 1024, 2, 128, 16, 4, 16>(),
    make_reg_entry<T, 1024, 4, 256, R_, R_, 16, 8, 8>(),
    make_reg_cached<T, 2048, 1, 128, 16, 8, 16>(),
    make_reg_entry<T, 4096, 1, 256, R_, R_, 16, 16, 16>(),
    make_reg_wide<T, 4096, 1, 256, 16, 16, 16>(),
    make_reg_entry<T, 8192, 1, 512, R_, R_, 16, 8, 8, 8>(),
    make_reg_wide<T, 8192, 1, 512, 8, 16, 8, 8>(),
    make_reg_entry<T, 16384, 1, 512, R_, R_, 32, 32, 16>(),
    make_reg_wide<T, 16384, 1, 1024, 16, 4, 16, 16>(),
    make_reg_long<T, 32768, 1024, HINT_ST, 32, 32, 32>(),
    make_reg_long<T, 32768, 1024, HINT_LD | HINT_ST, 32, 32, 32>(),
    // --- column tiles held in registers.  Four-step passes (MI355X, 1 GiB a
    // pass): 512 rows 0.476 -> 0.421 ms (from 4 tiles per CU on; below, the
    // LDS tile: 2^19 x 4 25 against 28 us), 2048 rows of 16 columns 0.540 ->
    // 0.48-0.49 (8 columns are as much as the LDS holds: 64-byte runs), from one
    // tile per CU on (real 2^21 x 2, 64 of them against 128 of 8 columns: 67.7 /
    // 62.9 us; 2^21 x 8, 256 of them: 134 / 146).  Whole
    // column transforms, by width (Builder::col_variant), us, LDS -> register
    // tile: 512 x 999 8.0 -> 5.7, 1024 x 513 12.6 -> 7.2, 1024 x 4999 32 -> 20
    // (the pipelined 16-column tile left 2 rounds of 256 workgroups, the second
    // 22% full), 1024^2 x 16 images' columns 55 -> 42, 2048 x 2048 19.8 -> 17.1,
    // 4096 x 2049 58 -> 40, 4096 x 6000 154 -> 110.  4096 rows past 96 MiB
    // want 8 columns: two 4-column tiles per CU keep 8 MB of quarter lines in
    // flight per XCD, twice its L2 (4096 x 4096: 135 us, LDS tile 105); so do
    // widths whose 8-column tiles are one round (x 2048 55 / 37.5, x 1400 31.1 /
    // 26.8; x 2100, a second round of 7 tiles, 55.4 / 59.4) ---
    make_reg_many<T, 512, 16, 512, C_, C_, 16, 2, 16>(4),
    make_reg_many<T, 2048, 16, 1024, C_, C_, 16, 8, 16>(1),
    make_reg_cols<T, 64, 16, 128, 8, 8>(),
    make_reg_cols<T, 128, 8, 128, 8, 2, 8>(),
    make_reg_cols<T, 256, 8, 256, 8, 4, 8>(),
    make_reg_cols<T, 512, 8, 512, 8, 8, 8>(),
    make_reg_cols<T, 1024, 4, 256, 16, 4, 16>(),
    make_reg_cols<T, 1024, 8, 512, 16, 4, 16>(),
    make_reg_cols<T, 1024, 16, 512, 32, 32>(),
    make_reg_cols<T, 2048, 4, 512, 16, 8, 16>(),
    make_reg_cols<T, 2048, 8, 1024, 16, 8, 16>(),
    make_reg_cols<T, 4096, 4, 512, 16, 16, 16>((int64_t)96 << 20),
    make_reg_cols_big<T, 4096, 8, 1024, 16, 16, 16>((int64_t)96 << 20),
    // --- transposing rows held in registers: 2048 points, 2^22 x 32 0.505 ->
    // 0.456 ms (128-byte runs instead of 64) ---
    make_reg_many<T, 2048, 16, 1024, R_, C_, 16, 16, 8>(1),
    make_reg_many<T, 4096, 8, 1024, R_, C_, 16, 16, 16>(1),
    // --- more column tiles of whole column transforms.  Few rows, us, LDS ->
    // register tile: 32 x 16 4.5 -> 3.3, x 32768 5.3 -> 4.5, 64 x 300 5.1 ->
    // 3.8, x 32768 7.5 -> 6.5, 128 x 32768 12.2 -> 11.1, 256 x 4096 5.8 -> 5.2,
    // x 131072 112 -> 104, 512 x 8192 14.3 -> 12.8, x 131072 243 -> 219.  The
    // columns of images, read from the Infinity Cache, want the LDS tiles'
    // fewer threads past 64 MiB (256 rows: 46.2 against 46.5 us there, 134.9
    // against 130.8 at 160 MiB) and 32 MiB (512 rows: 26.9 against 29.3, 47.5
    // against 45.5 at 64 MiB) ---
    make_reg_cols<T, 32, 16, 64, 8, 4>(),
    make_reg_cols<T, 32, 64, 256, 8, 4>(),
    make_reg_cols<T, 64, 64, 512, 8, 8>(),
    make_reg_cols<T, 128, 32, 512, 8, 2, 8>(),
    make_reg_cols<T, 256, 16, 512, 8, 4, 8>((int64_t)64 << 20),
    make_reg_cols_big<T, 256, 16, 512, 8, 4, 8>(0),
    make_reg_cols<T, 512, 16, 1024, 8, 8, 8>((int64_t)32 << 20),
    make_reg_cols_big<T, 512, 16, 1024, 8, 8, 8>(0),
};
// The 2^20 four-step's two pipelined passes paired in one launch (column pass
// of chunk k, transposing row pass of chunk k - 1).
using ColPass = PipeShape<T, 1024, 16, 1024, E_, C_, C_, 16, 4, 16>;
using RowPass = PipeShape<T, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>;
const DualEntry kDual[] = {
    make_dual<ColPass, RowPass>(&tile_fft_pipe_kernel<T, 1024, 16, 1024, E_, C_, C_, 16, 4, 16>,
                                &tile_fft_pipe_kernel<T, 1024, 16, 1024, S_, R_, C_, 16, 16, 4>),
};
}  // namespace

const KernelEntry *tile_kernels_f32(int *count)
{
    *count = (int)(sizeof(kTable) / sizeof(kTable[0]));
    return kTable;
}

const DualEntry *dual_kernels_f32(int *count)
{
    *count = (int)(sizeof(kDual) / sizeof(kDual[0]));
    return kDual;
}

}  // namespace gfft
