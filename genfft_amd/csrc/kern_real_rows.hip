// kern_real_rows.hip -- real transforms of n = 2L points with L up to the
// single-pass row length, in one HBM round trip.
//
//   r2c: the L-point FFT of the (even, odd) pairs of each row, then the
//        unpack of adjust_DIT_impl (generic/fft_dit_impl_generic.inl:27-61)
//        from LDS as the epilogue: bins k and L-k of pair p = k, bin 0 and
//        n/2 from Z_0, bin n/4 = conj Z_{L/2}; with a full spectrum also
//        F_{n-k} = conj F_k (FFTReal.h:204-213 with half = false).
//   c2r: the pack Z_k = (F_k + conj F_{L-k}) + i W_n^-k (F_k - conj F_{L-k})
//        as the prologue (both bins of a pair loaded by one thread, all
//        loads issued before the first LDS write), written re/im-swapped,
//        then the row FFT and the swapped store: the unscaled inverse.
//        The imaginary parts of bins 0 and n/2 are ignored, as in any c2r.
// A row tile holds M rows; the shapes are those of the c2c row tiles.  Long
// rows are held in registers instead of LDS (gfft_regtile.h), the unpack and
// the pack on the registers of one thread.
#include "gfft_r2c.h"

namespace gfft {
namespace {

template <typename T, int L, int M, int NT, int MODE, int... RS>
__global__ void __launch_bounds__(NT) real_rows_kernel(RealRowsArgs a)
{
    using G = TileGeom<L, M, LAY_SEQ, PAT_ROW, PAT_ROW>;
    constexpr int PP = L / 2 + 1;  // pairs per row, p = 0 .. L/2
    constexpr int IT = (M * PP + NT - 1) / NT;
    __shared__ cx<T> lds[G::ELEMS];
    const int tid = threadIdx.x;
    const int tile = a.t.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int s0 = tile * M;
    const int nvalid = min(M, a.t.n_inner - s0);
    const cx<T> *ptw = reinterpret_cast<const cx<T> *>(a.t.pass_tw);

    if constexpr (MODE == RR_R2C) {
        load_tile<T, L, M, NT, G, PAT_ROW>(lds, a.t, 0, 0, s0, nvalid, tid);
        __syncthreads();
        stockham_passes<T, L, M, NT, G, true, false, 1, RS...>(lds, ptw, tid, a.t, s0, 0, Tw4Pre{});
        cx<T> *out = reinterpret_cast<cx<T> *>(a.t.out);
#pragma unroll 2
        for (int it = 0; it < IT; it++) {
            const int q = tid + it * NT;
            const int s = q / PP, p = q - s * PP;
            if (q >= M * PP || s >= nvalid) continue;
            cx<T> *f = out + (int64_t)(s0 + s) * a.t.out_inner;
            if (p == 0) {
                const cx<T> z0 = lds[G::off(s, 0)];
                f[0] = {z0.re + z0.im, (T)0};
                f[L] = {z0.re - z0.im, (T)0};
            } else if (p == L / 2) {
                const cx<T> zq = lds[G::off(s, L / 2)];
                f[L / 2] = cj(zq);
                if (!a.half) f[2 * L - L / 2] = zq;
            } else {
                cx<T> fk, fj;
                unpack_pair(lds[G::off(s, p)], lds[G::off(s, L - p)], tw_w(a.tw, (uint64_t)p), fk, fj);
                f[p] = fk;
                f[L - p] = fj;
                if (!a.half) {
                    f[2 * L - p] = cj(fk);
                    f[L + p] = cj(fj);
                }
            }
        }
    } else {
        const cx<T> *in = reinterpret_cast<const cx<T> *>(a.t.in);
        cx<T> fa[IT], fb[IT];
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const int q = tid + it * NT;
            const int s = q / PP, p = q - s * PP;
            if (q < M * PP && s < nvalid) {
                const cx<T> *f = in + (int64_t)(s0 + s) * a.t.in_inner;
                fa[it] = f[p];
                fb[it] = f[L - p];
            }
        }
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const int q = tid + it * NT;
            const int s = q / PP, p = q - s * PP;
            if (q >= M * PP || s >= nvalid) continue;
            cx<T> f = fa[it], g = fb[it];
            if (p == 0) {
                f.im = (T)0;
                g.im = (T)0;
                lds[G::off(s, 0)] = swap_ri(packz(f, g, cx<double>{1.0, 0.0}));
            } else if (p == L / 2) {
                lds[G::off(s, p)] = swap_ri(packz(f, f, tw_w(a.tw, (uint64_t)p)));
            } else {
                const cx<double> w = tw_w(a.tw, (uint64_t)p);
                lds[G::off(s, p)] = swap_ri(packz(f, g, w));
                lds[G::off(s, L - p)] = swap_ri(packz(g, f, cx<double>{-w.re, w.im}));
            }
        }
        __syncthreads();
        stockham_passes<T, L, M, NT, G, true, false, 1, RS...>(lds, ptw, tid, a.t, s0, 0, Tw4Pre{});
        store_tile<T, L, M, NT, G, PAT_ROW>(lds, a.t, 0, 0, s0, nvalid, tid);
    }
}

// W_n^(t + r*LR), r = 0, 1, ... in turn: FP64 powers of W_n^LR for complex64,
// products of two table entries for complex128.
template <typename T>
struct RowTw {
    const TwTable &tab;
    int t, lr;
    cx<double> first;
    TwWalk walk;
    __device__ __forceinline__ RowTw(const TwTable &tab_, int t_, int lr_)
        : tab(tab_), t(t_), lr(lr_), first(tw_w(tab_, (uint64_t)t_)),
          walk(sizeof(T) == 4 ? TwWalk(first, tw_w(tab_, (uint64_t)lr_)) : TwWalk(first))
    {
    }
    __device__ __forceinline__ cx<double> at(int r)
    {
        if (r == 0) return first;
        if constexpr (sizeof(T) == 4) return walk.next();
        else return tw_w(tab, (uint64_t)(t + r * lr));
    }
};

// The same over rows held in registers (gfft_regtile.h).  The unpack and the
// pack work on pairs of elements k and L - k, which the last (r2c) or first
// (c2r) pass leaves in or takes from one thread's registers (MAP_M), so they
// need no exchange.  HINT: cache hints of the loads and stores.
template <typename T, int L, int M, int NT, int MODE, int HINT, int... RS>
__global__ void __launch_bounds__(NT, 4) real_rows_reg_kernel(RealRowsArgs a)
{
    constexpr int E = M * L / NT;
    constexpr int R1 = first_radix<RS...>(), RL = last_radix<RS...>();
    constexpr int R = MODE == RR_R2C ? RL : R1;  // the pass at the spectrum's side
    constexpr int LR = L / R;
    using G = PlaneGeom<T, L, M, R1, true>;
    using P = Bfly<L, M, NT, MAP_M, R>;
    __shared__ __align__(16) T plane[G::ELEMS];
    const int tid = threadIdx.x;
    const int tile = a.t.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int s0 = tile * M;
    const int nvalid = min(M, a.t.n_inner - s0);
    const cx<T> *ptw = reinterpret_cast<const cx<T> *>(a.t.pass_tw);
    // this thread's row and first butterfly at the spectrum's side
    const int ps = P::s(tid, 0), t = P::j(tid, 0);
    // HBM accesses: a uniform 64-bit base plus a 32-bit per-thread byte offset
    // (the host admits only layouts it fits).  Of bin t + r*LR and its mirror
    // L - t - r*LR the parts in r are uniform.
    const int64_t spitch = MODE == RR_R2C ? a.t.out_inner : a.t.in_inner;
    const uint32_t row = (uint32_t)ps * (uint32_t)spitch;
    constexpr uint32_t CS = sizeof(cx<T>);
    cx<T> v[E];
    if constexpr (MODE == RR_R2C) {
        using A = Bfly<L, M, NT, MAP_J, R1>;
        const char *ib = reinterpret_cast<const char *>(reinterpret_cast<const cx<T> *>(a.t.in) + (int64_t)s0 * a.t.in_inner);
#pragma unroll
        for (int q = 0; q < A::N; q++) {
            const int s = A::s(tid, q);
            const uint32_t to = ((uint32_t)s * (uint32_t)a.t.in_inner + (uint32_t)A::j(tid, q)) * CS;
#pragma unroll
            for (int r = 0; r < R1; r++) {
                v[q * R1 + r] = {(T)0, (T)0};
                if (M == 1 || s < nvalid)
                    reg_load<HINT, 1>(reinterpret_cast<const cx<T> *>(ib + r * A::LR * (int)CS + to), &v[q * R1 + r], 0);
            }
        }
        reg_passes<T, L, M, NT, G, MAP_J, MAP_J, MAP_M, 1, RS...>(plane, v, ptw, tid, a.t, RegTw<T, L, M, NT, 1, R1, MAP_J>{});
        if (M > 1 && ps >= nvalid) return;
        char *ob = reinterpret_cast<char *>(reinterpret_cast<cx<T> *>(a.t.out) + (int64_t)s0 * a.t.out_inner);
        auto put = [&](int64_t uniform, uint32_t own, cx<T> x) {
            reg_store<HINT, 1>(reinterpret_cast<cx<T> *>(ob + uniform * CS + (row + own) * CS), &x, 0);
        };
        cx<T> fk, fj;
        if (t != 0) {
            RowTw<T> w(a.tw, t, LR);
#pragma unroll
            for (int r = 0; r < R; r++) {
                unpack_pair(v[r], v[R + R - 1 - r], w.at(r), fk, fj);
                put(r * LR, t, fk);
                put(-r * LR, L - t, fj);
                if (!a.half) {  // bins n - k and n - (L - k)
                    put(-r * LR, 2 * L - t, cj(fk));
                    put(r * LR, L + t, cj(fj));
                }
            }
        } else {
            auto put2 = [&](int k, cx<T> x) {
                put(k, 0, x);
                if (!a.half) put(2 * L - k, 0, cj(x));
            };
            put(0, 0, {v[0].re + v[0].im, (T)0});
            put(L, 0, {v[0].re - v[0].im, (T)0});
            put2(L / 2, cj(v[R / 2]));
#pragma unroll
            for (int r = 1; r < R / 2; r++) {
                unpack_pair(v[r], v[R - r], tw_w(a.tw, (uint64_t)(r * LR)), fk, fj);
                put2(r * LR, fk);
                put2(L - r * LR, fj);
            }
#pragma unroll
            for (int r = 0; r < R / 2; r++) {
                unpack_pair(v[R + r], v[R + R - 1 - r], tw_w(a.tw, (uint64_t)(LR / 2 + r * LR)), fk, fj);
                put2(LR / 2 + r * LR, fk);
                put2(L - LR / 2 - r * LR, fj);
            }
        }
    } else {
        const char *ib = reinterpret_cast<const char *>(reinterpret_cast<const cx<T> *>(a.t.in) + (int64_t)s0 * a.t.in_inner);
        auto get = [&](int64_t uniform, uint32_t own) {
            cx<T> x = {(T)0, (T)0};
            if (M == 1 || ps < nvalid)
                reg_load<HINT, 1>(reinterpret_cast<const cx<T> *>(ib + uniform * CS + (row + own) * CS), &x, 0);
            return x;
        };
        // Z_k and Z_(L-k) of the pair, re/im swapped for the inverse
        auto pack2 = [&](cx<T> fk, cx<T> fj, cx<double> w, cx<T> &zk, cx<T> &zj) {
            zk = swap_ri(packz(fk, fj, w));
            zj = swap_ri(packz(fj, fk, cx<double>{-w.re, w.im}));
        };
        if (t != 0) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                v[r] = get(r * LR, t);
                v[R + R - 1 - r] = get(-r * LR, L - t);
            }
            RowTw<T> w(a.tw, t, LR);
#pragma unroll
            for (int r = 0; r < R; r++) pack2(v[r], v[R + R - 1 - r], w.at(r), v[r], v[R + R - 1 - r]);
        } else {
            // the imaginary parts of bins 0 and n/2 are ignored
            const cx<T> f0 = {get(0, 0).re, (T)0}, fl = {get(L, 0).re, (T)0}, fh = get(L / 2, 0);
            v[0] = swap_ri(packz(f0, fl, cx<double>{1.0, 0.0}));
            v[R / 2] = swap_ri(packz(fh, fh, tw_w(a.tw, (uint64_t)(L / 2))));
#pragma unroll
            for (int r = 1; r < R / 2; r++)
                pack2(get(r * LR, 0), get(L - r * LR, 0), tw_w(a.tw, (uint64_t)(r * LR)), v[r], v[R - r]);
#pragma unroll
            for (int r = 0; r < R / 2; r++)
                pack2(get(LR / 2 + r * LR, 0), get(L - LR / 2 - r * LR, 0), tw_w(a.tw, (uint64_t)(LR / 2 + r * LR)),
                      v[R + r], v[R + R - 1 - r]);
        }
        reg_passes<T, L, M, NT, G, MAP_M, MAP_J, MAP_J, 1, RS...>(plane, v, ptw, tid, a.t, RegTw<T, L, M, NT, 1, R1, MAP_M>{});
        using A = Bfly<L, M, NT, MAP_J, RL>;
        char *ob = reinterpret_cast<char *>(reinterpret_cast<cx<T> *>(a.t.out) + (int64_t)s0 * a.t.out_inner);
#pragma unroll
        for (int q = 0; q < A::N; q++) {
            const int s = A::s(tid, q);
            const uint32_t to = ((uint32_t)s * (uint32_t)a.t.out_inner + (uint32_t)A::j(tid, q)) * CS;
#pragma unroll
            for (int r = 0; r < RL; r++) {
                const cx<T> x = swap_ri(v[q * RL + r]);
                if (M == 1 || s < nvalid)
                    reg_store<HINT, 1>(reinterpret_cast<cx<T> *>(ob + r * A::LR * (int)CS + to), &x, 0);
            }
        }
    }
}

template <typename T, int MODE, int L, int M, int NT, int... RS>
constexpr RowsEntry lds_rows()
{
    return {entry_shape<T, L, M, NT, LAY_SEQ, PAT_ROW, PAT_ROW, RS...>(), MODE, 0, 0, &real_rows_kernel<T, L, M, NT, MODE, RS...>};
}

template <typename T, int MODE, int HINT, int L, int M, int NT, int... RS>
constexpr RowsEntry reg_rows(int64_t most = 0, int64_t most_full = 0)
{
    return {reg_shape<T, L, M, NT, PAT_ROW, PAT_ROW, RS...>(), MODE, most, most_full ? most_full : most, &real_rows_reg_kernel<T, L, M, NT, MODE, HINT, RS...>};
}

template <typename T, int MODE, int HINT, int L, int NT, int... RS>
constexpr RowsEntry long_rows()
{
    RowsEntry r = reg_rows<T, MODE, HINT, L, 1, NT, RS...>();
    r.entry.long_row = 1;
    return r;
}

// Register-held tiles first (MI355X, device time per call against the LDS
// tiles or, for the longest rows, the two-launch fused forms, r2c / c2r):
//   f32 n = 128, 4096 rows       8.6 -> 4.4 us / 8.0 -> 3.7 us
//   f32 n = 1024, 512 rows       8.8 -> 4.2 / 8.1 -> 4.8
//   f32 n = 4096, 16384 rows     124 -> 110 / 128 -> 102
//   f32 n = 16384, 16384 rows    496 -> 399 / 505 -> 382
//   f32 n = 32768, 2048 rows     175 -> 122 / 176 -> 114
//   f32 n = 65536, 1024 rows     241 -> 157 / 242 -> 141
//   f64 n = 1024, 256 rows       7.0 -> 4.5 / 6.7 -> 4.5
//   f64 n = 32768, 1024 rows     266 -> 137 / 219 -> 136
// The spectrum side of a short r2c writes two runs of bins per row in opposite
// directions, which past the caches merge into whole lines less well than the
// LDS tile's one run: f32 n = 512 lost from 32 MiB on (131072 rows 119 -> 169
// us), f64 n = 1024 at 1 GiB (406 -> 425 us), hence kSmall and kCached.  A full
// spectrum's four runs lose earlier, at an output past the Infinity Cache (LDS
// / registers: f64 n = 1024 x 24000 114 / 129 us, 2048 x 16000 147 / 161, 4096 x
// 8000 147 / 154; x a third of them 22-40% faster in registers), hence kFull.
// Eight elements per thread were faster than sixteen up to n = 2048, and for f64
// r2c n = 8192 (62 rows 10.5 -> 9.4 us, the LDS tile 10.1).
// The LDS tiles follow the c2c row-tile shapes; from L = 2 (n = 4) on, so
// short real transforms are one launch as well (n = 2 runs as a copy and the
// unpack).  Lengths whose register-held tiles hold several rows keep an LDS
// one for layouts past 32-bit offsets, those with a limit one beyond it.
constexpr int F = RR_R2C, B = RR_C2R;
constexpr int64_t kSmall = (int64_t)16 << 20, kCached = (int64_t)512 << 20;
constexpr int64_t kFull = (int64_t)96 << 20;
const RowsEntry kRowsF32[] = {
    reg_rows<float, F, HINT_LD, 64, 8, 64, 4, 4, 4>(kSmall),
    reg_rows<float, F, HINT_LD, 128, 4, 64, 8, 4, 4>(kSmall),
    reg_rows<float, F, HINT_LD, 256, 2, 64, 8, 8, 4>(kSmall),
    reg_rows<float, F, HINT_LD, 512, 1, 64, 8, 4, 4, 4>(0, (int64_t)160 << 20),
    reg_rows<float, F, HINT_LD, 1024, 1, 128, 8, 8, 4, 4>(),
    reg_rows<float, F, HINT_LD, 2048, 1, 128, 16, 16, 8>(0, kFull),
    reg_rows<float, F, HINT_LD, 4096, 1, 256, 8, 8, 8, 8>(),
    reg_rows<float, F, HINT_LD, 8192, 1, 512, 16, 8, 8, 8>(),
    reg_rows<float, F, HINT_LD, 16384, 1, 512, 32, 32, 16>(),
    long_rows<float, F, HINT_LD, 32768, 1024, 16, 16, 8, 16>(),
    reg_rows<float, B, HINT_ST, 64, 8, 64, 4, 4, 4>(kSmall),
    reg_rows<float, B, HINT_ST, 128, 4, 64, 4, 4, 8>(kSmall),
    reg_rows<float, B, HINT_ST, 256, 4, 64, 8, 4, 8>(),
    reg_rows<float, B, HINT_ST, 512, 2, 64, 8, 8, 8>(),
    reg_rows<float, B, HINT_ST, 1024, 1, 64, 8, 8, 16>(),
    reg_rows<float, B, HINT_ST, 2048, 1, 128, 8, 16, 16>(),
    reg_rows<float, B, HINT_ST, 4096, 1, 256, 8, 8, 8, 8>(),
    reg_rows<float, B, HINT_ST, 8192, 1, 512, 8, 16, 8, 8>(),
    reg_rows<float, B, HINT_ST, 16384, 1, 512, 16, 32, 32>(),
    long_rows<float, B, HINT_ST, 32768, 1024, 16, 8, 16, 16>(),
#define BOTH(...) lds_rows<float, F, __VA_ARGS__>(), lds_rows<float, B, __VA_ARGS__>()
    BOTH(2, 1024, 128, 2), BOTH(4, 1024, 256, 4), BOTH(8, 512, 256, 8), BOTH(16, 256, 256, 16), BOTH(32, 128, 256, 8, 4),
    BOTH(64, 64, 256, 8, 8), BOTH(128, 32, 256, 16, 8), BOTH(256, 16, 256, 16, 16), BOTH(512, 8, 256, 8, 8, 8),
    lds_rows<float, F, 2048, 2, 256, 16, 16, 8>(),
#undef BOTH
};
const RowsEntry kRowsF64[] = {
    reg_rows<double, F, HINT_LD, 128, 4, 64, 8, 4, 4>(kSmall),
    reg_rows<double, F, HINT_LD, 256, 2, 64, 8, 8, 4>(kSmall),
    reg_rows<double, F, HINT_LD, 512, 1, 64, 8, 4, 4, 4>(kCached, kFull),
    reg_rows<double, F, HINT_LD, 1024, 1, 128, 8, 8, 4, 4>(kCached, kFull),
    reg_rows<double, F, HINT_LD, 2048, 1, 256, 8, 8, 8, 4>(0, kFull),
    reg_rows<double, F, HINT_LD, 4096, 1, 512, 8, 8, 4, 4, 4>(),
    reg_rows<double, F, HINT_LD, 8192, 1, 512, 16, 8, 8, 8>(),
    long_rows<double, F, HINT_LD, 16384, 1024, 16, 16, 8, 8>(),
    reg_rows<double, B, HINT_ST, 128, 4, 64, 4, 4, 8>(kSmall),
    reg_rows<double, B, HINT_ST, 256, 2, 64, 4, 8, 8>((int64_t)192 << 20),
    reg_rows<double, B, HINT_ST, 512, 1, 64, 4, 4, 4, 8>(),
    reg_rows<double, B, HINT_ST, 1024, 1, 128, 4, 4, 8, 8>(),
    reg_rows<double, B, HINT_ST, 2048, 1, 256, 4, 8, 8, 8>(),
    reg_rows<double, B, HINT_ST, 4096, 1, 256, 8, 8, 4, 16>(),
    reg_rows<double, B, HINT_ST, 8192, 1, 512, 8, 8, 8, 16>(),
    long_rows<double, B, HINT_ST, 16384, 1024, 8, 8, 16, 16>(),
#define BOTH(...) lds_rows<double, F, __VA_ARGS__>(), lds_rows<double, B, __VA_ARGS__>()
    BOTH(2, 512, 64, 2), BOTH(4, 512, 128, 4), BOTH(8, 256, 128, 8), BOTH(16, 128, 128, 16), BOTH(32, 64, 128, 8, 4),
    BOTH(64, 32, 128, 8, 8), BOTH(128, 16, 128, 16, 8), BOTH(256, 8, 256, 8, 8, 4),
    lds_rows<double, F, 512, 4, 256, 8, 8, 8>(), lds_rows<double, F, 1024, 2, 256, 8, 4, 8, 4>(),
    lds_rows<double, F, 2048, 1, 256, 8, 8, 8, 4>(),
#undef BOTH
};

template <size_t K>
const RowsEntry *rows_find(const RowsEntry (&tab)[K], int L, int mode, int64_t bytes, bool full, bool lds, bool long_row)
{
    for (size_t i = 0; i < K; i++) {
        const KernelEntry &e = tab[i].entry;
        const int64_t most = full ? tab[i].most_full : tab[i].most;
        if (e.L == L && tab[i].mode == mode && !(lds && e.reg) && (e.long_row != 0) == long_row && (!most || bytes <= most))
            return &tab[i];
    }
    return nullptr;
}

}  // namespace

const RowsEntry *real_rows_entry(int prec, int L, int mode, int64_t bytes, bool full, bool lds, bool long_row)
{
    return prec ? rows_find(kRowsF64, L, mode, bytes, full, lds, long_row)
                : rows_find(kRowsF32, L, mode, bytes, full, lds, long_row);
}

hipError_t launch_real_rows(const RowsEntry *e, const RealRowsArgs &a, int64_t grid, hipStream_t s, hipEvent_t stop)
{
    return launch_stop(e->fn, dim3((unsigned)grid), dim3(e->entry.NT), s, a, stop);
}

}  // namespace gfft
