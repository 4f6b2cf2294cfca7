// gfft_registry.h -- the table of compiled tile-kernel shapes.
//
// Every instantiation of gfft::tile_fft_kernel is described by one entry;
// the planner (plan.cpp) picks entries by (precision, L, input pattern,
// output pattern) and launches them through the function pointer.
#pragma once
#include <type_traits>

#include "gfft_device.h"
#include "gfft_regtile.h"
#include "gfft_wave.h"

namespace gfft {

struct KernelEntry {
    int prec;      // 0 = complex64, 1 = complex128
    int L;         // sequence length
    int M;         // sequences per tile
    int NT;        // threads per workgroup
    int layout;    // LAY_SEQ / LAY_ELEM
    int inp, outp; // PAT_ROW / PAT_COL
    int nrad;
    int rad[8];
    int lds_bytes;
    int persistent;  // 1: tile_fft_pipe_kernel (grid sized to the device, loops over tiles)
    int tune_only;   // 1: an alternative (radix order / tile width / threads) only the autotuner selects
    void (*fn)(TileArgs);
    void (*fn_plain)(TileArgs);  // reg: the same with plain stores, where one is compiled
    int store;       // 0: complex T in memory; 1: FP16 pairs; 2: BF16 pairs (FP32 arithmetic)
    int gen_tw;      // 1: the last pass builds its twiddles from TileArgs::gen_lo / gen_hi (W_L)
    int wave;        // 1: one wavefront per row, lanes exchanged without LDS (wave_rows1024_kernel)
    int reg;         // 1: tile held in registers (reg_tile_kernel); its own pass twiddle table layout
    int many;        // tiles per CU from which this one is taken instead of the LDS tile of its width
    int64_t most;    // cols, cached: bytes a side up to which it is taken (0: any)
    int64_t most_odd;  // cols: the same where rows of the matrix share lines
    int64_t least;   // cols: bytes a side from which it is taken
    int one_round;   // cols: 1: also below, where its tiles are one full round of the CUs
    int cols;        // 1: column tile for whole column transforms only; 2: but not those of complex 2D planes
    int cached;      // 1: row tile the planner takes for batches within the Infinity Cache
    int long_row;    // 1: a row longer than the LDS row tiles (the planner takes it by its own rule)
    int wide;        // 1: double-width row tile the planner takes for batches past the Infinity Cache
};

// Shape of a tile entry, without its kernel: each make_* below takes the
// address of exactly the kernel it registers, so no translation unit
// instantiates kernels of another table.
template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry entry_shape()
{
    static_assert(((RS * ...) == L), "radices must multiply to L");
    static_assert((M * L) % NT == 0, "tile must split evenly over threads");
    static_assert(NT % 64 == 0 && NT <= 1024, "whole wavefronts, at most 1024 threads");
    using G = TileGeom<L, M, LAY, INP, OUTP>;
    static_assert(G::ELEMS * sizeof(cx<T>) <= 160 * 1024, "tile exceeds gfx950 LDS");
    KernelEntry e{};
    e.prec = sizeof(T) == 8 ? 1 : 0;
    e.L = L;
    e.M = M;
    e.NT = NT;
    e.layout = LAY;
    e.inp = INP;
    e.outp = OUTP;
    e.nrad = sizeof...(RS);
    const int r[] = {RS...};
    for (int i = 0; i < (int)sizeof...(RS); i++) e.rad[i] = r[i];
    e.lds_bytes = (int)(G::ELEMS * sizeof(cx<T>));
    e.persistent = 0;
    e.tune_only = 0;
    e.fn = nullptr;
    return e;
}

template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_entry()
{
    KernelEntry e = entry_shape<T, L, M, NT, LAY, INP, OUTP, RS...>();
    e.fn = &tile_fft_kernel<T, L, M, NT, LAY, INP, OUTP, RS...>;
    return e;
}

template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_variant()
{
    KernelEntry e = make_entry<T, L, M, NT, LAY, INP, OUTP, RS...>();
    e.tune_only = 1;
    return e;
}

// A tuning alternative the planner also takes by itself for batches larger
// than the Infinity Cache (KernelEntry::wide).
template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_wide_variant()
{
    KernelEntry e = make_variant<T, L, M, NT, LAY, INP, OUTP, RS...>();
    e.wide = 1;
    return e;
}

// Persistent, software-pipelined variant (same tile math, LDS-resident pass
// twiddles, next tile prefetched into registers).
template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry pipe_shape()
{
    KernelEntry e = entry_shape<T, L, M, NT, LAY, INP, OUTP, RS...>();
    using S = PipeLds<T, L, M, NT, LAY, INP, OUTP, RS...>;
    e.lds_bytes = (int)((S::TILE_A + S::TW) * sizeof(cx<T>));
    e.gen_tw = S::P::GEN ? 1 : 0;
    e.persistent = 1;
    return e;
}

// One wavefront per 1024-point complex64 row, no LDS (wave_rows1024_kernel),
// radix stages (16, 16, 4); twiddles generated from the two-level table of W_1024.
template <int NT>
constexpr KernelEntry make_wave_entry()
{
    KernelEntry e = entry_shape<float, 1024, NT / 64, NT, LAY_SEQ, PAT_ROW, PAT_ROW, 16, 16, 4>();
    e.lds_bytes = 0;
    e.tune_only = 1;
    e.gen_tw = 1;
    e.wave = 1;
    e.fn = &wave_rows1024_kernel<NT>;
    return e;
}

template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_pipe_entry()
{
    KernelEntry e = pipe_shape<T, L, M, NT, LAY, INP, OUTP, RS...>();
    e.fn = &tile_fft_pipe_kernel<T, L, M, NT, LAY, INP, OUTP, RS...>;
    return e;
}

template <typename T, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_pipe_variant()
{
    KernelEntry e = make_pipe_entry<T, L, M, NT, LAY, INP, OUTP, RS...>();
    e.tune_only = 1;
    return e;
}

// Shape of a tile held in registers, without its kernel.
template <typename T, int L, int M, int NT, int INP, int OUTP, int... RS>
constexpr KernelEntry reg_shape()
{
    static_assert(((RS * ...) == L), "radices must multiply to L");
    static_assert(NT % 64 == 0 && NT <= 1024, "whole wavefronts, at most 1024 threads");
    using G = PlaneGeom<T, L, M, first_radix<RS...>(), INP == PAT_ROW>;
    static_assert(G::ELEMS * sizeof(T) <= 160 * 1024, "exchange plane exceeds gfx950 LDS");
    KernelEntry e{};
    e.prec = sizeof(T) == 8 ? 1 : 0;
    e.L = L;
    e.M = M;
    e.NT = NT;
    e.layout = INP == PAT_ROW ? LAY_SEQ : LAY_ELEM;
    e.inp = INP;
    e.outp = OUTP;
    e.nrad = sizeof...(RS);
    const int r[] = {RS...};
    for (int i = 0; i < (int)sizeof...(RS); i++) e.rad[i] = r[i];
    e.lds_bytes = (int)(G::ELEMS * sizeof(T));
    e.gen_tw = sizeof(T) == 4;
    e.reg = 1;
    return e;
}

template <typename T, int L, int M, int NT, int INP, int OUTP, int HINT, int... RS>
constexpr KernelEntry reg_entry()
{
    KernelEntry e = reg_shape<T, L, M, NT, INP, OUTP, RS...>();
    e.fn = &reg_tile_kernel<T, L, M, NT, INP, OUTP, HINT, RS...>;
    return e;
}

// reg_tile_kernel with its stores streamed or plain (KernelEntry::fn_plain).
template <typename T, int L, int M, int NT, int INP, int OUTP, int... RS>
constexpr KernelEntry make_reg_entry()
{
    KernelEntry e = reg_entry<T, L, M, NT, INP, OUTP, HINT_ST, RS...>();
    e.fn_plain = &reg_tile_kernel<T, L, M, NT, INP, OUTP, HINT_NONE, RS...>;
    return e;
}

// The row tile with streaming loads as well, which the planner takes for
// batches past the Infinity Cache (KernelEntry::wide).
template <typename T, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_wide()
{
    KernelEntry e = reg_entry<T, L, M, NT, PAT_ROW, PAT_ROW, HINT_LD | HINT_ST, RS...>();
    e.tune_only = 1;
    e.wide = 1;
    return e;
}

// Taken from `many` tiles per CU on.
template <typename T, int L, int M, int NT, int INP, int OUTP, int... RS>
constexpr KernelEntry make_reg_many(int many)
{
    KernelEntry e = make_reg_entry<T, L, M, NT, INP, OUTP, RS...>();
    e.many = many;
    return e;
}

// A column tile of a whole column transform (not of a four-step pass), which
// the planner picks by width (Builder::col_variant).
template <typename T, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_cols(int64_t most = 0, int64_t most_odd = 0)
{
    KernelEntry e = make_reg_entry<T, L, M, NT, PAT_COL, PAT_COL, RS...>();
    e.most = most;
    e.most_odd = most_odd;
    e.tune_only = 1;
    e.cols = 1;
    return e;
}

template <typename T, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_cols_big(int64_t least)
{
    KernelEntry e = make_reg_cols<T, L, M, NT, RS...>();
    e.least = least;
    e.one_round = least > 0;
    e.cols = 2;
    return e;
}

// A narrow row tile for batches that would leave CUs idle (the planner's
// narrow_row_variant).
template <typename T, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_narrow()
{
    KernelEntry e = make_reg_entry<T, L, M, NT, PAT_ROW, PAT_ROW, RS...>();
    e.tune_only = 1;
    return e;
}

// A row tile for batches that stay within the Infinity Cache.
template <typename T, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_cached(int64_t most = 0)
{
    KernelEntry e = make_reg_narrow<T, L, M, NT, RS...>();
    e.most = most;
    e.cached = 1;
    return e;
}

// A row longer than the LDS row tiles.
template <typename T, int L, int NT, int HINT, int... RS>
constexpr KernelEntry make_reg_long()
{
    KernelEntry e = reg_entry<T, L, 1, NT, PAT_ROW, PAT_ROW, HINT, RS...>();
    e.tune_only = 1;
    e.long_row = 1;
    e.wide = (HINT & HINT_LD) ? 1 : 0;
    return e;
}

// 16-bit storage form of a complex64 shape (tile_fft_kernel_h).
template <class S, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_entry_h()
{
    KernelEntry e = entry_shape<float, L, M, NT, LAY, INP, OUTP, RS...>();
    e.lds_bytes += M * (int)sizeof(float);
    e.store = std::is_same<S, st_f16>::value ? 1 : 2;
    e.fn = &tile_fft_kernel_h<S, L, M, NT, LAY, INP, OUTP, RS...>;
    return e;
}

// A row tile kept for layouts the register-held one cannot address.
template <class S, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_variant_h()
{
    KernelEntry e = make_entry_h<S, L, M, NT, LAY, INP, OUTP, RS...>();
    e.tune_only = 1;
    return e;
}

// 16-bit rows held in registers (reg_rows_kernel_h).
template <class S, int HINT, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_rows_h()
{
    KernelEntry e = reg_shape<float, L, M, NT, PAT_ROW, PAT_ROW, RS...>();
    e.lds_bytes += (NT / M > 64 ? NT / M / 64 : 1) * (int)sizeof(float);
    e.store = std::is_same<S, st_f16>::value ? 1 : 2;
    e.fn = &reg_rows_kernel_h<S, L, M, NT, HINT, RS...>;
    return e;
}

// The same for batches within the Infinity Cache only.
template <class S, int HINT, int L, int M, int NT, int... RS>
constexpr KernelEntry make_reg_cached_h()
{
    KernelEntry e = make_reg_rows_h<S, HINT, L, M, NT, RS...>();
    e.tune_only = 1;
    e.cached = 1;
    return e;
}

// Pipelined 16-bit storage form (tile_fft_pipe_kernel_h).
template <class S, int L, int M, int NT, int LAY, int INP, int OUTP, int... RS>
constexpr KernelEntry make_pipe_entry_h()
{
    KernelEntry e = pipe_shape<float, L, M, NT, LAY, INP, OUTP, RS...>();
    // its own LDS: the tile, the pass tables when they fit beside the tile
    // and the scales (else they are read from global memory), the scales
    using G = TileGeom<L, M, LAY, INP, OUTP>;
    constexpr int twn = pass_tw_count<1, RS...>();
    constexpr bool twl = pass_tw_in_lds<float, G::ELEMS + M / 2, twn>();
    e.lds_bytes = (int)((G::ELEMS + (twl && twn > 0 ? twn : 1)) * sizeof(cx<float>)) + M * (int)sizeof(float);
    e.gen_tw = 0;
    e.store = std::is_same<S, st_f16>::value ? 1 : 2;
    e.fn = &tile_fft_pipe_kernel_h<S, L, M, NT, LAY, INP, OUTP, RS...>;
    return e;
}

// A dual_pipe_kernel pairing two pipelined tile passes: role A (the four-step
// column pass of one chunk) and role B (the transposing row pass of the
// chunk before), identified by the single-pass kernels they replace.
struct DualEntry {
    int prec;
    int NT;
    int lds_bytes;
    void (*a_fn)(TileArgs);  // the tile_fft_pipe_kernel whose tiles role A runs
    void (*b_fn)(TileArgs);  // the same for role B
    void (*fn)(TileArgs, TileArgs, int);
};

template <class A, class B>
constexpr DualEntry make_dual(void (*a_fn)(TileArgs), void (*b_fn)(TileArgs))
{
    static_assert(A::NT == B::NT, "one thread count");
    constexpr int e = A::ELEMS > B::ELEMS ? A::ELEMS : B::ELEMS;
    static_assert(e * sizeof(cx<typename A::T>) <= 160 * 1024, "both roles fit gfx950 LDS");
    DualEntry d{};
    d.prec = sizeof(typename A::T) == 8 ? 1 : 0;
    d.NT = A::NT;
    d.lds_bytes = (int)(e * sizeof(cx<typename A::T>));
    d.a_fn = a_fn;
    d.b_fn = b_fn;
    d.fn = &dual_pipe_kernel<A, B>;
    return d;
}

// Defined in kern_tile_f32.hip / kern_tile_f64.hip / kern_tile_h.hip.
const KernelEntry *tile_kernels_f32(int *count);
const KernelEntry *tile_kernels_f64(int *count);
const DualEntry *dual_kernels_f32(int *count);
const DualEntry *dual_kernels_f64(int *count);
const KernelEntry *tile_kernels_f16(int *count);
const KernelEntry *tile_kernels_bf16(int *count);

}  // namespace gfft
