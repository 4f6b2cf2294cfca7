// gfft_regtile.h -- tiles held in registers, exchanged through LDS one
// component at a time.
//
// tile_fft_kernel keeps its tile in LDS as complex numbers, so a tile is at
// most 160 KB: 16384 complex64 or 8192 complex128 elements.  Here a workgroup
// of NT threads holds E = M*L/NT elements per thread in VGPRs (a CU has
// 512 KB of them), and between two Stockham passes the real parts go through
// an LDS plane of M*L scalars, then the imaginary parts through the same
// plane: twice the elements for the same LDS.  The first pass reads its
// butterfly inputs straight from HBM into registers and the last one stores
// straight from them, so a transform of P passes makes P - 1 exchanges and no
// other LDS sweep.
//
// What bounds it: HBM, with the pass twiddles next.  On c64 rows of 32768
// points (1 GiB batch, MI355X) reading the twiddles from a table in L2 took
// 0.594 ms per call, against 0.440 ms with none at all; built as FP64 powers
// of one base per butterfly, rounded once, 0.46-0.49 ms (the four-step of two
// passes: 0.73-0.78 ms; a 1 GiB copy: 0.39 ms).  complex128 keeps the tables,
// since powers would add rounding errors there (0.43 ms for rows of 16384;
// four-step 0.77 ms).  Up to 32 complex64 or 16 complex128 elements per thread
// fit 128 VGPRs without spills, the budget of 16 waves per CU.
#pragma once
#include "gfft_device.h"

namespace gfft {

// Plane address of element n of sequence s, in scalars of T.
//   Element-major (columns in and out): the M sequences of one element index
//   adjacent, one pad row after every R1 (the first radix), so the stride-R1
//   writes of the first pass fall on alternating halves of the banks.
//   Sequence-major (rows in): one pad scalar per 32 (float) or 16 (double)
//   breaks the same stride along a row, and the sequence pitch is B/M modulo
//   the B scalars of a bank row, so that M sequences times B/M consecutive
//   elements (a COL-side walk) hit distinct banks.
// Both are sums of a term in s and a term in n, and the term in n is additive
// over numbers with no common bits: an access is one thread base plus a
// compile-time offset.
template <typename T, int L, int M, int R1, bool SEQ_>
struct PlaneGeom {
    static constexpr bool SEQ = SEQ_;
    static constexpr int B = 128 / (int)sizeof(T);  // scalars per bank row
    static constexpr int PB = SEQ ? ilog2c(B) : ilog2c(R1);
    static constexpr int LP = L + (L >> PB);
    static constexpr int SS0 = (LP + B - 1) / B * B;
    static constexpr int SS = !SEQ ? 1 : M == 1 ? LP : SS0 + (M < B ? B / M : 1);
    static constexpr int ELEMS = SEQ ? M * SS : LP * M;
    static __host__ __device__ constexpr int seq(int s) { return s * SS; }
    static __host__ __device__ constexpr int elem(int n) { return SEQ ? n + (n >> PB) : (n + (n >> PB)) * M; }
};

// How a pass of radix R deals its butterflies (s, j) to the threads: along
// the sequence first (MAP_J), across the sequences first (MAP_S), or across
// pairs of adjacent sequences (MAP_P: butterflies 2q and 2q + 1 of a thread
// are the same j of sequences s and s + 1, so their HBM accesses join into
// 16 bytes and they share their twiddles), or along the sequence in mirror
// pairs (MAP_M, two butterflies per thread: thread t of a sequence has j = t
// and L/R - t, whose elements are k and L - k; t = 0 has 0 and L/2R, which
// mirror themselves), or in pairs of neighbours (MAP_N: thread t of a sequence
// has j = 2t and 2t + 1, whose HBM accesses join).
enum : int { MAP_J = 0, MAP_S = 1, MAP_P = 2, MAP_M = 3, MAP_N = 4 };
template <int L, int M, int NT, int MAP, int R>
struct Bfly {
    static constexpr int LR = L / R;
    static constexpr int W = MAP == MAP_P ? 2 : 1;  // butterflies that share j
    static constexpr int N = M * L / NT / R / W;    // groups of them per thread
    static_assert(N >= 1 && N * W * R * NT == M * L, "whole butterflies per thread");
    static_assert((MAP != MAP_M && MAP != MAP_N) || N == 2, "pairs of butterflies");
    static __device__ __forceinline__ int s(int tid, int q)
    {
        const int b = tid + q * NT;
        if constexpr (M == 1) return 0;
        else if constexpr (MAP == MAP_M || MAP == MAP_N) return tid / (LR / 2);
        else return MAP == MAP_J ? b / LR : MAP == MAP_S ? b % M : b % (M / 2) * 2;
    }
    static __device__ __forceinline__ int j(int tid, int q)
    {
        const int b = tid + q * NT;
        if constexpr (MAP == MAP_M) {
            const int t = tid % (LR / 2);
            return q == 0 ? t : t ? LR - t : LR / 2;
        } else if constexpr (MAP == MAP_N) {
            return tid % (LR / 2) * 2 + q;
        } else if constexpr (M == 1) return b;
        else return MAP == MAP_J ? b % LR : MAP == MAP_S ? b / M : b / (M / 2);
    }
};

template <typename T>
struct alignas(2 * sizeof(T)) scalar2 {
    T a, b;
};

// One exchange between the pass of radix R (NS = product of the radices
// before it, mapping MP) and the next one of radix R2 (mapping MP2).  FIRST:
// no earlier exchange has to be waited for.
template <typename T, int L, int M, int NT, class G, int NS, int R, int MP, int R2, int MP2, bool FIRST>
__device__ __forceinline__ void reg_exchange(T *plane, cx<T> (&v)[M * L / NT], int tid)
{
    using A = Bfly<L, M, NT, MP, R>;
    using D = Bfly<L, M, NT, MP2, R2>;
    auto at = [&](int k, int c) -> T & { return c ? v[k].im : v[k].re; };
    auto put = [&](int c) {
#pragma unroll
        for (int q = 0; q < A::N; q++) {
            const int j = A::j(tid, q), m = j & (NS - 1), s = A::s(tid, q);
            T *p = plane + G::seq(s) + G::elem((j - m) * R + m);
#pragma unroll
            for (int r = 0; r < R; r++) {
                T *d = p + G::elem(r * NS);
                if constexpr (A::W == 1) *d = at(q * R + r, c);
                else if constexpr (!G::SEQ) *reinterpret_cast<scalar2<T> *>(d) = {at(2 * q * R + r, c), at((2 * q + 1) * R + r, c)};
                else {
                    d[0] = at(2 * q * R + r, c);
                    d[G::SS] = at((2 * q + 1) * R + r, c);
                }
            }
        }
    };
    auto get = [&](int c) {
#pragma unroll
        for (int q = 0; q < D::N; q++) {
            const T *p = plane + G::seq(D::s(tid, q)) + G::elem(D::j(tid, q));
#pragma unroll
            for (int r = 0; r < R2; r++) {
                const T *d = p + G::elem(r * D::LR);
                if constexpr (D::W == 1) at(q * R2 + r, c) = *d;
                else if constexpr (!G::SEQ) {
                    const scalar2<T> x = *reinterpret_cast<const scalar2<T> *>(d);
                    at(2 * q * R2 + r, c) = x.a;
                    at((2 * q + 1) * R2 + r, c) = x.b;
                } else {
                    at(2 * q * R2 + r, c) = d[0];
                    at((2 * q + 1) * R2 + r, c) = d[G::SS];
                }
            }
        }
    };
    if constexpr (!FIRST) __syncthreads();
    put(0);
    __syncthreads();
    get(0);
    __syncthreads();
    put(1);
    __syncthreads();
    get(1);
}

// Twiddle bases of a pass (complex64): W_{NS*R}^m of each butterfly group, an
// FP64 product from the two-level table of W_L (TileArgs::gen_lo / gen_hi).
template <typename T, int L, int M, int NT, int NS, int R, int MP>
struct RegTw {
    using A = Bfly<L, M, NT, MP, R>;
    static constexpr bool GEN = sizeof(T) == 4 && NS > 1;
    cx<double> base[GEN ? A::N : 1];
    __device__ __forceinline__ void load(const TileArgs &a, int tid)
    {
        if constexpr (GEN) {
            constexpr int LB = (ilog2c(L) + 1) / 2;
            const cx<double> *lo = reinterpret_cast<const cx<double> *>(a.gen_lo);
            const cx<double> *hi = reinterpret_cast<const cx<double> *>(a.gen_hi);
#pragma unroll
            for (int q = 0; q < A::N; q++) {
                const uint32_t x = (uint32_t)(A::j(tid, q) & (NS - 1)) * (uint32_t)(L / (NS * R));
                base[q] = cmul(hi[x >> LB], lo[x & ((1u << LB) - 1u)]);
            }
        }
    }
};

// Powers of a unit complex number by the three-term recurrence
// w_(r+1) = 2 cos(theta) w_r - w_(r-1): two FP64 FMAs a step where a product
// takes four.  Its rounding errors grow as r^2 at most: below 2e-13 after 32
// steps, far under the 6e-8 of the FP32 rounding that follows.
struct TwWalk {
    cx<double> w0, w1;
    double k;
    __device__ __forceinline__ TwWalk(cx<double> b) : w0{1.0, 0.0}, w1(b), k(2.0 * b.re) {}
    // start w, ratio b
    __device__ __forceinline__ TwWalk(cx<double> w, cx<double> b) : w0(w), w1(cmul(w, b)), k(2.0 * b.re) {}
    __device__ __forceinline__ cx<double> next()
    {
        const cx<double> w = w1;
        w1 = {__builtin_fma(k, w.re, -w0.re), __builtin_fma(k, w.im, -w0.im)};
        w0 = w;
        return w;
    }
};

// The passes from (NS, R) on: mapping MP for this one, MPL for the last one
// and MPM for those between.  complex64 builds a butterfly's twiddles as FP64 powers of its base,
// rounded once; complex128 reads them from `tw`, W_{NS*R}^(r*m) at
// [(r - 1) * NS + m] for each pass with NS > 1.
template <typename T, int L, int M, int NT, class G, int MP, int MPM, int MPL, int NS, int R, int... RS>
__device__ __forceinline__ void reg_passes(T *plane, cx<T> (&v)[M * L / NT], const cx<T> *__restrict__ tw, int tid,
                                           const TileArgs &a, const RegTw<T, L, M, NT, NS, R, MP> &w)
{
    using A = Bfly<L, M, NT, MP, R>;
#pragma unroll
    for (int q = 0; q < A::N; q++) {
        cx<T> *x = &v[q * A::W * R];
        if constexpr (NS > 1 && sizeof(T) == 4) {
            TwWalk wk(w.base[q]);
#pragma unroll
            for (int r = 1; r < R; r++) {
                const cx<double> wr = wk.next();
                const cx<T> t = {(T)wr.re, (T)wr.im};
#pragma unroll
                for (int e = 0; e < A::W; e++) x[e * R + r] = cmul(x[e * R + r], t);
            }
        } else if constexpr (NS > 1) {
            const int m = A::j(tid, q) & (NS - 1);
#pragma unroll
            for (int r = 1; r < R; r++) {
                const cx<T> t = tw[(r - 1) * NS + m];
#pragma unroll
                for (int e = 0; e < A::W; e++) x[e * R + r] = cmul(x[e * R + r], t);
            }
        }
#pragma unroll
        for (int e = 0; e < A::W; e++) dft<R, (M * L / NT < 32)>(x + e * R);
    }
    if constexpr (sizeof...(RS) > 0) {
        constexpr int R2 = first_radix<RS...>();
        constexpr int MP2 = sizeof...(RS) == 1 ? MPL : MPM;
        RegTw<T, L, M, NT, NS * R, R2, MP2> w2;
        w2.load(a, tid);
        reg_exchange<T, L, M, NT, G, NS, R, MP, R2, MP2, NS == 1>(plane, v, tid);
        reg_passes<T, L, M, NT, G, MP2, MPM, MPL, NS * R, RS...>(plane, v, tw + (NS > 1 ? NS * (R - 1) : 0), tid, a, w2);
    }
}

// Mapping of the passes on a COL side: pairs of sequences where every radix
// leaves a thread two butterflies.
template <typename T, int L, int M, int NT, int... RS>
constexpr int col_map()
{
    constexpr int E = M * L / NT;
    return M % 2 == 0 && M <= 8 && ((E / RS >= 2) && ...) ? MAP_P : MAP_S;
}

// Cache hints of a launch's HBM accesses: HINT_LD / HINT_ST mark its loads /
// stores nontemporal (streaming); HINT_AGENT its loads as of agent scope, for
// what another CU wrote earlier in the same launch (whole tiles of rows only).
enum : int { HINT_NONE = 0, HINT_LD = 1, HINT_ST = 2, HINT_AGENT = 4 };

// W adjacent elements, read or written together (complex64 pairs as 16 bytes
// at the 8-byte alignment of an element, which global accesses allow).
template <int HINT, int W, typename T>
__device__ __forceinline__ void reg_load(const cx<T> *p, cx<T> *x, int stride)
{
    typedef T vec __attribute__((ext_vector_type(2)));
    typedef T vec4 __attribute__((ext_vector_type(4), aligned(2 * sizeof(T))));
    if constexpr (W == 2 && sizeof(T) == 4) {
        const vec4 q = (HINT & HINT_LD) ? __builtin_nontemporal_load(reinterpret_cast<const vec4 *>(p))
                                        : *reinterpret_cast<const vec4 *>(p);
        x[0] = {q.x, q.y};
        x[stride] = {q.z, q.w};
    } else {
#pragma unroll
        for (int e = 0; e < W; e++) {
            const vec q = (HINT & HINT_LD) ? __builtin_nontemporal_load(reinterpret_cast<const vec *>(p + e))
                                           : *reinterpret_cast<const vec *>(p + e);
            x[e * stride] = {q.x, q.y};
        }
    }
}

template <int HINT, int W, typename T>
__device__ __forceinline__ void reg_store(cx<T> *p, const cx<T> *x, int stride)
{
    typedef T vec __attribute__((ext_vector_type(2)));
    typedef T vec4 __attribute__((ext_vector_type(4), aligned(2 * sizeof(T))));
    if constexpr (W == 2 && sizeof(T) == 4) {
        const vec4 q = {x[0].re, x[0].im, x[stride].re, x[stride].im};
        if constexpr (HINT & HINT_ST) __builtin_nontemporal_store(q, reinterpret_cast<vec4 *>(p));
        else *reinterpret_cast<vec4 *>(p) = q;
    } else {
#pragma unroll
        for (int e = 0; e < W; e++) {
            const vec q = {x[e * stride].re, x[e * stride].im};
            if constexpr (HINT & HINT_ST) __builtin_nontemporal_store(q, reinterpret_cast<vec *>(p + e));
            else *reinterpret_cast<vec *>(p + e) = q;
        }
    }
}

// One element, `own` + `step` bytes from a uniform base, read at agent scope
// (sc1): past the CU's own cache.  `buffer` ends with the tile.
template <typename T>
__device__ __forceinline__ cx<T> agent_load(__amdgpu_buffer_rsrc_t buffer, uint32_t own, int step)
{
    constexpr int SC1 = 16;
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(cx<T>, __builtin_amdgcn_raw_buffer_load_b64(buffer, (int)own, step, SC1));
    else
        return __builtin_bit_cast(cx<T>, __builtin_amdgcn_raw_buffer_load_b128(buffer, (int)own, step, SC1));
}

// One tile: sequences s0 .. s0 + nvalid - 1 of transform o, read from `in` and
// written to `out` (the transform's first elements).  INP / OUTP as in
// tile_fft_kernel.  The first pass walks along the rows when they are read
// (INP = ROW), the later ones when they are written.
template <typename T, int L, int M, int NT, int INP, int OUTP, int HINT, int... RS>
__device__ __forceinline__ void reg_tile(T *plane, const TileArgs &a, const cx<T> *in, cx<T> *out, int s0, int o,
                                         int nvalid, int tid)
{
    constexpr int E = M * L / NT;
    constexpr int R1 = first_radix<RS...>(), RL = last_radix<RS...>();
    constexpr int CM = col_map<T, L, M, NT, RS...>();
    constexpr int MP = INP == PAT_ROW ? MAP_J : CM, MPL = OUTP == PAT_ROW ? MAP_J : CM;
    using G = PlaneGeom<T, L, M, R1, INP == PAT_ROW>;
    // Columns of 4096 rows: a wave has three loads on their way, not all of them;
    // the tiles that share their lines stay closer together (c64 us all / three:
    // 4096 x 3000 77 / 72, 4096 x 1024 24.4 / 22.3, 4096 x 8 9.8 / 9.9; 2048 x 5000
    // 48.0 / 49.3, 1024 x 8192 24.1 / 25.6, c128 1024 x 4096 28.7 / 31.7)
    constexpr bool kFewLoads = INP == PAT_COL && sizeof(T) == 4 && L >= 4096;
    cx<T> v[E];
    // HBM accesses: a uniform 64-bit base for each r plus one 32-bit
    // per-thread byte offset (the host admits only layouts it fits)
    {
        using A = Bfly<L, M, NT, MP, R1>;
        in += INP == PAT_ROW ? (int64_t)s0 * a.in_inner : (int64_t)s0;
        const int64_t step = (INP == PAT_ROW ? (int64_t)A::LR : (int64_t)A::LR * a.in_elem) * (int64_t)sizeof(cx<T>);
        const char *ib = reinterpret_cast<const char *>(in);
#pragma unroll
        for (int q = 0; q < A::N; q++) {
            // a sequence past the last one is computed on that one's elements
            // and not stored (a branch around each load instead made the one
            // partly filled tile the slowest: c64 4096 x 107 columns 20.4 us, 17.8 so);
            // pairs stay one access, of the last two sequences
            const int s = min(A::s(tid, q), max(nvalid - A::W, 0)), j = A::j(tid, q);
            const uint32_t to = (INP == PAT_ROW ? (uint32_t)s * (uint32_t)a.in_inner + (uint32_t)j
                                                : (uint32_t)j * (uint32_t)a.in_elem + (uint32_t)s) * (uint32_t)sizeof(cx<T>);
            cx<T> *x = &v[q * A::W * R1];
            if constexpr ((HINT & HINT_AGENT) != 0) {
                static_assert(INP == PAT_ROW && A::W == 1, "tiles of rows");
                const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<char *>(ib), 0, (int)(M * a.in_inner * (int64_t)sizeof(cx<T>)), 0x00027000);
#pragma unroll
                for (int r = 0; r < R1; r++) x[r] = agent_load<T>(buffer, to, (int)(r * step));
                continue;
            }
            if (A::W == 1 || nvalid > 1) {
#pragma unroll
                for (int r = 0; r < R1; r++) {
                    reg_load<HINT, A::W>(reinterpret_cast<const cx<T> *>(ib + r * step + to), x + r, R1);
                    if constexpr (kFewLoads) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
                }
            } else {
#pragma unroll
                for (int r = 0; r < R1; r++) {
                    reg_load<HINT, 1>(reinterpret_cast<const cx<T> *>(ib + r * step + to), x + r, R1);
                    x[(A::W - 1) * R1 + r] = x[r];
                }
            }
        }
        // read once the loads are on their way: the wait for it would hold them up
        // (c128 64 x 64 images 6.9 us, 6.7 so)
        asm volatile("" ::: "memory");
        if (swap_in_of(a, o)) {
#pragma unroll
            for (int k = 0; k < E; k++) v[k] = swap_ri(v[k]);
        }
        if (A::W == 2 && (nvalid & 1)) {
            // the last sequence is the second of the two its thread has read
            // (the other result of that thread is not stored)
#pragma unroll
            for (int q = 0; q < A::N; q++)
#pragma unroll
                for (int r = 0; r < R1; r++)
                    if (A::s(tid, q) >= nvalid - 1) v[q * A::W * R1 + r] = v[(q + 1) * A::W * R1 - R1 + r];
        }
    }
    reg_passes<T, L, M, NT, G, MP, MPL, MPL, 1, RS...>(plane, v, reinterpret_cast<const cx<T> *>(a.pass_tw), tid, a,
                                                  RegTw<T, L, M, NT, 1, R1, MP>{});
    {
        using A = Bfly<L, M, NT, MPL, RL>;
        const bool sw = swap_out_of(a, o);
        out += OUTP == PAT_ROW ? (int64_t)s0 * a.out_inner : (int64_t)s0;
        const int64_t step = (OUTP == PAT_ROW ? (int64_t)A::LR : (int64_t)A::LR * a.out_elem) * (int64_t)sizeof(cx<T>);
        char *ob = reinterpret_cast<char *>(out);
#pragma unroll
        for (int q = 0; q < A::N; q++) {
            const int s = A::s(tid, q), j = A::j(tid, q);
            cx<T> *x = &v[q * A::W * RL];
            if (a.tw_mode != TW_NONE) {
                // four-step twiddle W_Ntw^(c*k), k = j + r*L/RL
#pragma unroll
                for (int e = 0; e < A::W; e++) {
                    const uint32_t c = a.tw_mode == TW_INNER ? (uint32_t)(s0 + s + e) : (uint32_t)o;
                    if constexpr (sizeof(T) == 4) {
                        // FP64 geometric progression, rounded once per element
                        const cx<double> wj = tw_fp64(a, c * (uint32_t)j);
                        TwWalk wk(wj, tw_fp64(a, c * (uint32_t)A::LR));
                        x[e * RL] = apply_tw(x[e * RL], wj);
#pragma unroll
                        for (int r = 1; r < RL; r++) x[e * RL + r] = apply_tw(x[e * RL + r], wk.next());
                    } else {
#pragma unroll
                        for (int r = 0; r < RL; r++)
                            x[e * RL + r] = apply_tw(x[e * RL + r], tw_fp64(a, c * (uint32_t)(j + r * A::LR)));
                    }
                }
            }
            if (sw) {
#pragma unroll
                for (int k = 0; k < A::W * RL; k++) x[k] = swap_ri(x[k]);
            }
            const uint32_t to = (OUTP == PAT_ROW ? (uint32_t)s * (uint32_t)a.out_inner + (uint32_t)j
                                                 : (uint32_t)j * (uint32_t)a.out_elem + (uint32_t)s) * (uint32_t)sizeof(cx<T>);
#pragma unroll
            for (int r = 0; r < RL; r++) {
                cx<T> *p = reinterpret_cast<cx<T> *>(ob + r * step + to);
                if (M == 1 || nvalid == M) {
                    reg_store<HINT, A::W>(p, x + r, RL);
                } else if (A::W == 2 && s + 1 < nvalid) {
                    reg_store<HINT_NONE, A::W>(p, x + r, RL);
                } else if (s < nvalid) {
                    *p = x[r];
                }
            }
        }
    }
}

template <typename T, int L, int M, int NT, int INP, int OUTP, int HINT, int... RS>
__global__ void __launch_bounds__(NT, 4) reg_tile_kernel(TileArgs a)
{
    using G = PlaneGeom<T, L, M, first_radix<RS...>(), INP == PAT_ROW>;
    __shared__ __align__(16) T plane[G::ELEMS];
    const int tile = a.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int t2 = tile / a.tiles_inner;
    const int ti = tile - t2 * a.tiles_inner;
    const int o2 = t2 / a.n_outer1;
    const int o = t2 - o2 * a.n_outer1;
    const int s0 = ti * M;
    reg_tile<T, L, M, NT, INP, OUTP, HINT, RS...>(
        plane, a, reinterpret_cast<const cx<T> *>(a.in) + in_base(a, o2, o),
        reinterpret_cast<cx<T> *>(a.out) + out_base(a, o2, o), s0, o, min(M, a.n_inner - s0), threadIdx.x);
}

// scale of a 16-bit transform from the largest |re| + |im| of its input: the
// largest power of two up to 1 with m * gain * scale <= limit
__device__ __forceinline__ float scale_from_max(float m, float gain, float limit)
{
    const float q = m * gain / limit;  // limit is a power of two: exact division
    if (!(q > 1.0f) || !(q <= 3.0e38f)) return 1.0f;  // fits already, or not finite
    const uint32_t u = __float_as_uint(q);
    const int k = (int)((u >> 23) & 255u) - 127 + ((u & 0x7fffffu) ? 1 : 0);  // ceil(log2 q), q normal
    return __uint_as_float((uint32_t)(127 - k) << 23);
}

// Rows of 16-bit storage (FP16 / BF16 pairs, FP32 arithmetic), a whole row per
// workgroup, so the automatic scale (TileArgs::auto_scale) needs no pass of its
// own: each thread takes the largest |re| + |im| of the elements it loads, the
// row's threads reduce it, and the store multiplies by the scale.
template <class S, int L, int M, int NT, int HINT, int... RS>
__global__ void __launch_bounds__(NT, 4) reg_rows_kernel_h(TileArgs a)
{
    using T = float;
    constexpr int E = M * L / NT;
    constexpr int R1 = first_radix<RS...>(), RL = last_radix<RS...>();
    static_assert(E == 2 * R1 && E == 2 * RL, "one pair of butterflies per thread at both ends");
    using G = PlaneGeom<T, L, M, R1, true>;
    using A = Bfly<L, M, NT, MAP_N, R1>;
    using B = Bfly<L, M, NT, MAP_N, RL>;
    constexpr int TPS = NT / M;  // threads of a row
    typedef uint32_t word2 __attribute__((ext_vector_type(2), aligned(4)));
    __shared__ __align__(16) T plane[G::ELEMS];
    __shared__ float red[TPS > 64 ? TPS / 64 : 1];
    const int tid = threadIdx.x;
    const int tile = a.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int t2 = tile / a.tiles_inner;
    const int ti = tile - t2 * a.tiles_inner;
    const int o2 = t2 / a.n_outer1;
    const int o = t2 - o2 * a.n_outer1;
    const int s0 = ti * M;
    const int nvalid = min(M, a.n_inner - s0);
    const int s = A::s(tid, 0), j = A::j(tid, 0);
    const int64_t ibase = in_base(a, o2, o) + (int64_t)s0 * a.in_inner;
    cx<T> v[E];
    float m = 0.0f;
    {
        const bool sw = swap_in_of(a, o);
        const char *ib = reinterpret_cast<const char *>(reinterpret_cast<const uint32_t *>(a.in) + ibase);
        const uint32_t to = ((uint32_t)s * (uint32_t)a.in_inner + (uint32_t)j) * 4u;
#pragma unroll
        for (int r = 0; r < R1; r++) {
            word2 w = {0u, 0u};
            if (M == 1 || s < nvalid) {
                const word2 *p = reinterpret_cast<const word2 *>(ib + r * A::LR * 4 + to);
                w = (HINT & HINT_LD) ? __builtin_nontemporal_load(p) : *p;
            }
            const cx<T> x0 = hdec<S>(w.x), x1 = hdec<S>(w.y);
            m = fmaxf(m, fmaxf(fabsf(x0.re) + fabsf(x0.im), fabsf(x1.re) + fabsf(x1.im)));
            v[r] = sw ? swap_ri(x0) : x0;
            v[R1 + r] = sw ? swap_ri(x1) : x1;
        }
    }
    if (a.auto_scale) {
#pragma unroll
        for (int off = (TPS < 64 ? TPS : 64) / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
        if (TPS > 64 && (tid & 63) == 0) red[tid >> 6] = m;  // read after the passes' barriers
    }
    reg_passes<T, L, M, NT, G, MAP_N, MAP_J, MAP_N, 1, RS...>(plane, v, nullptr, tid, a, RegTw<T, L, M, NT, 1, R1, MAP_N>{});
    float scl = 1.0f;
    if (a.auto_scale) {
        if constexpr (TPS > 64) {
            static_assert(M == 1 && sizeof...(RS) > 1, "the row's waves are the workgroup's, with barriers between the passes");
#pragma unroll
            for (int i = 0; i < TPS / 64; i++) m = fmaxf(m, red[i]);
        }
        scl = scale_from_max(m, a.bound.gain, a.bound.limit);
        if (tid % TPS == 0 && s < nvalid) a.auto_scale[s0 + s] = scl;
    } else if (a.scale && s < nvalid) {
        scl = a.scale[(a.scale_off + ibase + (int64_t)s * a.in_inner) / a.scale_div];
    }
    {
        const bool sw = swap_out_of(a, o);
        char *ob = reinterpret_cast<char *>(reinterpret_cast<uint32_t *>(a.out) + out_base(a, o2, o) +
                                            (int64_t)s0 * a.out_inner);
        const uint32_t to = ((uint32_t)s * (uint32_t)a.out_inner + (uint32_t)B::j(tid, 0)) * 4u;
        if (M == 1 || s < nvalid) {
#pragma unroll
            for (int r = 0; r < RL; r++) {
                const cx<T> x0 = {v[r].re * scl, v[r].im * scl}, x1 = {v[RL + r].re * scl, v[RL + r].im * scl};
                const word2 w = {henc<S>(sw ? swap_ri(x0) : x0), henc<S>(sw ? swap_ri(x1) : x1)};
                word2 *p = reinterpret_cast<word2 *>(ob + r * B::LR * 4 + to);
                if constexpr (HINT & HINT_ST) __builtin_nontemporal_store(w, p);
                else *p = w;
            }
        }
    }
}

}  // namespace gfft
