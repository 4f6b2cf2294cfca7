// kern_xcd.hip -- both passes of a four-step in one persistent launch, each
// transform on one XCD (see gfft_xcd.h).
//
// What bounds it: the traffic past the L2, which is that of two launches (2.0 GiB
// read and 2.0 written for 1 GiB of c64 2^20 or 2^16: 6.7 TB/s, where copies that
// stay in the Infinity Cache reach 7), and for the shortest lengths the turns of
// an XCD's counters.  Four workgroups of 256 threads (or two of 512) hold 4 MB of
// tiles per XCD, as much as its L2, so the ring's traffic goes on to the Infinity
// Cache, and a row tile must come that many tasks after its column tiles not to
// wait: with `lag` 2 instead of 10, c64 2^16 x 2048 takes 0.83-2.1 ms instead of
// 0.62.  MI355X against two launches, ms at 1 GiB / us at an eighth to a half of it:
// c64 2^16 0.75 -> 0.62 / 118 -> 103 (x 260), 2^17 0.79 -> 0.64 / 146 -> 122 (x 164),
// 2^18 0.77 -> 0.65 / 264 -> 233 (x 164), 2^19 0.85 -> 0.65 / 429 -> 348 (x 130), 2^20
// 0.82 -> 0.64 / 441 -> 335 (x 64); c128 2^15 0.76 -> 0.63 / 131 -> 113 (x 290), 2^16
// 0.81 -> 0.63 / 157 -> 119 (x 162), 2^17 0.85 -> 0.70 / 300 -> 250 (x 171), 2^18 0.83
// -> 0.68 / 290 -> 248 (x 84); a 1 GiB copy takes 0.39.  Near the smallest batches:
// c64 2^16 x 146 73.6 -> 69.9 us, x 190 85.1 -> 84.7, 2^17 x 82 80.5 -> 73.3, 2^20 x 26
// 191 -> 182, c128 2^15 x 112 59.4 -> 59.8, 2^18 x 42 158 -> 142: it is taken wherever
// its ring fits the workspace the two launches would have (but for layouts
// whose runs share lines, see the table).  Longer transforms' rings leave the
// Infinity Cache; c128 2^19 gained 4% at 1 GiB and nothing at 238 MiB and stays
// on two launches.
#include "gfft_regtile.h"
#include "gfft_xcd.h"

namespace gfft {
namespace {

__device__ __forceinline__ uint32_t xcc_id()
{
    // s_getreg_b32 HW_REG_XCC_ID (20), 4 bits from bit 0
    return (uint32_t)__builtin_amdgcn_s_getreg(20 | (3 << 11)) & (kXcds - 1);
}

__device__ __forceinline__ uint32_t bump(uint32_t *p, uint32_t by = 1u)
{
    return __hip_atomic_fetch_add(p, by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until *p >= v, by adding nothing to it.  With atomic loads instead (and
// the row tiles' stores waited for) c64 2^16 x 256 took 196 us, with these 127.
__device__ __forceinline__ uint32_t await(uint32_t *p, uint32_t v)
{
    uint32_t zero = 0, x;
    asm volatile("" : "+v"(zero));
    while ((x = bump(p, zero)) < v) __builtin_amdgcn_s_sleep(1);
    return x;
}

// Takes the next task of an XCD's queue.  Whoever takes a block's first task
// claims the next transform of the batch for the block at once, after the block
// before has its own, so an XCD's blocks run out of transforms in order.
__device__ __forceinline__ uint32_t take(uint32_t *pop, uint32_t *blk, uint32_t *state, uint32_t per_block,
                                         uint32_t blocks)
{
    const uint32_t j = bump(pop), b = j / per_block;
    if (j % per_block == 0 && b < blocks) {
        uint32_t *const w = blk + (int64_t)b * 4;
        if (b) await(w - 4, 1u);
        bump(w, bump(state) + 1u);
    }
    return j;
}

template <int... RS>
struct Radices {};

// Scalars of the exchange plane, for either pass.
template <typename T, int N1, int N2, int M, int... RA, int... RB>
constexpr int plane_of(Radices<RA...>, Radices<RB...>)
{
    constexpr int a = PlaneGeom<T, N1, M, first_radix<RA...>(), false>::ELEMS;
    constexpr int b = PlaneGeom<T, N2, M, first_radix<RB...>(), true>::ELEMS;
    return a > b ? a : b;
}

template <typename T, int L, int M, int NT, int INP, int... RS>
constexpr KernelEntry shape_of(Radices<RS...>)
{
    return reg_shape<T, L, M, NT, INP, PAT_COL, RS...>();
}

template <typename T, int L, int M, int NT, int INP, int HINT, int... RS>
__device__ __forceinline__ void tile_of(T *plane, const TileArgs &a, const cx<T> *in, cx<T> *out, int s0, int o,
                                        int tid, Radices<RS...>)
{
    reg_tile<T, L, M, NT, INP, PAT_COL, HINT, RS...>(plane, a, in, out, s0, o, M, tid);
}

// Transform length N1 * N2: T1 column tiles (N1 points, M of the N2 columns),
// then T2 row tiles (N2 points, M of the N1 rows, stored transposed).
//
// Each XCD has a queue: task j of block b = j / (T1 + T2) is a column tile of
// its b-th transform or a row tile of its (b - lag)-th, handed out by one
// counter.  The blocks claim transforms from the whole batch (take), so any
// spread of workgroups over XCDs finishes it.  A task waits only for tasks
// handed out before it (a row tile for its transform's column tiles, a column
// tile for the row tiles that read the ring slot before), which their workgroups
// run in order, and a claim only for the claim before it, so the earliest
// unfinished task never waits and the grid always drains; a workgroup ends at
// the first row task of a block past the batch, which no later task can be
// inside, and holds no other task then.
//
// What one CU hands to another stays on one XCD, so no cache is written back:
// stores are in the L2 once vmcnt is 0.  The readers are on other CUs, whose own
// caches may hold lines of the ring from the slot's last transform, so they load
// it at agent scope (HINT_AGENT), from the L2.  MI355X, us, start of a batch's
// range / 1 GiB: c64 2^16 69.9 / 617, 2^20 182 / 642, c128 2^16 98.9 / 634 so;
// 73.2 / 632, 186 / 644, 105 / 667 with an agent-scope invalidate (buffer_inv sc1)
// by the thread that saw the count instead, and c64 2^20 794 with one by every
// wave.  A workgroup-scope invalidate (sc0) need not drop those lines.
template <typename T, int N1, int N2, int M, int NT, int WPE, int PLAIN, class RA, class RB>
__global__ void __launch_bounds__(NT, WPE) xcd_fft_kernel(XcdArgs x)
{
    constexpr int T1 = N2 / M, T2 = N1 / M;
    constexpr int64_t N = (int64_t)N1 * N2;
    __shared__ __align__(16) T plane[plane_of<T, N1, N2, M>(RA{}, RB{})];
    __shared__ int task[4];
    const int tid = threadIdx.x;
    const uint32_t q = xcc_id();
    uint32_t *const pop = x.state + 32 * (1 + q);
    uint32_t *const blk = x.state + 32 * (1 + kXcds) + (int64_t)q * x.blocks * 4;  // {claim, columns done, rows done, -}
    cx<T> *const ring = reinterpret_cast<cx<T> *>(x.col.out) + (int64_t)q * x.ring * N;
    uint32_t next = 0;  // thread 0: taken one task ahead
    if (tid == 0) next = take(pop, blk, x.state, T1 + T2, x.blocks);
    for (;;) {
        if (tid == 0) {
            const int b = (int)(next / (T1 + T2)), r = (int)(next % (T1 + T2));
            const bool rows = r >= T1;
            const int c = rows ? b - x.lag : b;
            int g = -1;  // nothing to do
            if (b >= x.blocks) {
                g = -2;  // end
            } else if (c >= 0) {
                uint32_t *const w = blk + (int64_t)c * 4;
                g = (int)await(w, 1u) - 1;
                if (g >= x.batch) g = rows ? -2 : -1;
                else if (rows) await(w + 1, T1);
                else if (c >= x.ring) await(w - (int64_t)x.ring * 4 + 2, T2);
            }
            task[0] = g;
            task[1] = r;
            task[2] = c;
            if (g != -2) next = take(pop, blk, x.state, T1 + T2, x.blocks);
        }
        __syncthreads();
        // uniform, so that the tiles' bases stay in scalar registers
        const int g = __builtin_amdgcn_readfirstlane(task[0]), r = __builtin_amdgcn_readfirstlane(task[1]),
                  c = __builtin_amdgcn_readfirstlane(task[2]);
        if (g == -2) break;
        if (g >= 0) {
            cx<T> *const slot = ring + (int64_t)(c % x.ring) * N;
            if (r < T1) {
                tile_of<T, N1, M, NT, PAT_COL, (PLAIN & XCD_PLAIN_LD) ? HINT_NONE : HINT_LD>(
                    plane, x.col, reinterpret_cast<const cx<T> *>(x.col.in) + in_base(x.col, 0, g), slot, r * M, g, tid,
                    RA{});
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else {
                tile_of<T, N2, M, NT, PAT_ROW, HINT_AGENT | ((PLAIN & XCD_PLAIN_ST) ? HINT_NONE : HINT_ST)>(
                    plane, x.row, slot, reinterpret_cast<cx<T> *>(x.row.out) + out_base(x.row, 0, g), (r - T1) * M, g,
                    tid, RB{});
            }
        }
        __syncthreads();
        if (tid == 0 && g >= 0) bump(blk + (int64_t)c * 4 + (r < T1 ? 1 : 2));
    }
}

__global__ void __launch_bounds__(256) xcd_reset_kernel(uint32_t *state, int64_t words)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < words) state[i] = 0u;
}

// WPE: waves per SIMD the registers are budgeted for
template <typename T, int N1, int N2, int M, int NT, int WPE, int PLAIN, class RA, class RB>
constexpr XcdEntry make_xcd(int lag, int ring, int per_cu, RA ra, RB rb, int64_t out_least = 0, int64_t both_least = 0)
{
    XcdEntry e{};
    e.prec = sizeof(T) == 8 ? 1 : 0;
    for (int n = N1 * N2; n > 1; n >>= 1) e.lg++;
    e.col = shape_of<T, N1, M, NT, PAT_COL>(ra);
    e.row = shape_of<T, N2, M, NT, PAT_ROW>(rb);
    e.NT = NT;
    e.lds_bytes = plane_of<T, N1, N2, M>(ra, rb) * (int)sizeof(T);
    e.lag = lag;
    e.ring = ring;
    e.per_cu = per_cu;
    e.plain = PLAIN;
    e.out_least = out_least;
    e.both_least = both_least;
    e.fn[0] = &xcd_fft_kernel<T, N1, N2, M, NT, WPE, 0, RA, RB>;
    e.fn[XCD_PLAIN_ST] = &xcd_fft_kernel<T, N1, N2, M, NT, WPE, XCD_PLAIN_ST, RA, RB>;  // Builder's kXcdKeptBytes too
    if constexpr ((PLAIN & XCD_PLAIN_LD) != 0) {
        e.fn[XCD_PLAIN_LD] = &xcd_fft_kernel<T, N1, N2, M, NT, WPE, XCD_PLAIN_LD, RA, RB>;
        e.fn[XCD_PLAIN_LD | XCD_PLAIN_ST] = &xcd_fft_kernel<T, N1, N2, M, NT, WPE, XCD_PLAIN_LD | XCD_PLAIN_ST, RA, RB>;
    }
    return e;
}

// Where a length is listed twice, the first whose ring fits the workspace.
// Radix 32 * 16 and 32 * 32 with 16 or 32 elements per thread against more
// threads of fewer, ms at 1 GiB: 2^17 0.63 / 0.73, 2^18 0.64 / 0.67, 2^19 0.66 /
// 0.91, 2^20 0.64 / 0.84 (16 * 4 * 16).  c128 2^15 with 16 sequences a tile
// instead of 8: half the turns of the XCD's counters, which bound its 16 KB
// tiles (x 105 61.3 -> 56.0 us, where two launches take 56.2; x 2000 684 -> 627).
//
// Layouts whose runs share lines (xcd_hints): two launches / streamed / plain
// loads / plain stores / both plain, us, for 1 element between the inputs, the
// outputs, or 3 and 5 (the sides' alignment decides, not the numbers):
//   c64 2^16 x 300   130 / 129 / 121 / 129 / 122   147 / 144 / 154 / 134 / 131   148 / 158 / 154 / 152 / 134
//   c64 2^18 x 200   318 / 335 / 308 / 332 / 323   396 / 439 / 425 / 381 / 426   400 / 487 / 441 / 442 / 443
//   c64 2^19 x 120   408 / 386 / 376 / 404 / 395   487 / 472 / 512 / 500 / 523   494 / 535 / 548 / 578 / 539
//   c64 2^20 x 60    447 / 373 / 397 / 443 / 407   518 / 478 / 598 / 542 / 540   547 / 538 / 611 / 614 / 552
//   c128 2^16 x 140  135 / 123 / 117 / 128 / 127   148 / 158 / 160 / 144 / 141   150 / 172 / 162 / 162 / 147
//   c128 2^18 x 100  342 / 337 / 327 / 331 / 342   410 / 362 / 348 / 333 / 385   413 / 400 / 364 / 387 / 405
// 2^18 and 2^19 write an odd output side in two launches below 400 / 480 MiB and
// where the input's is odd as well; c128 2^18 x 44 (176 MiB) 184 / 198 with both
// odd.  Outputs in whole 32-byte sectors want streamed stores whatever else
// (c64 2^17 x 300, 4 elements apart: 332 / 224).
constexpr int LD = XCD_PLAIN_LD, ST = XCD_PLAIN_ST;
constexpr int64_t MiB = 1 << 20;
const XcdEntry kXcd[] = {
    make_xcd<float, 256, 256, 16, 256, 4, LD | ST>(10, 18, 4, Radices<16, 16>{}, Radices<16, 16>{}),
    make_xcd<float, 256, 512, 16, 256, 4, LD | ST>(5, 10, 4, Radices<16, 16>{}, Radices<32, 16>{}),
    make_xcd<float, 512, 512, 16, 256, 4, LD | ST>(6, 10, 4, Radices<32, 16>{}, Radices<32, 16>{}, 400 * MiB, -1),
    make_xcd<float, 1024, 512, 16, 512, 4, LD>(3, 6, 2, Radices<32, 32>{}, Radices<16, 2, 16>{}, 480 * MiB, -1),
    make_xcd<float, 1024, 1024, 16, 512, 4, 0>(2, 4, 2, Radices<32, 32>{}, Radices<32, 32>{}),
    make_xcd<float, 1024, 1024, 16, 512, 4, LD | ST>(1, 3, 2, Radices<32, 32>{}, Radices<32, 32>{}),
    make_xcd<double, 128, 256, 16, 256, 3, 0>(7, 12, 3, Radices<8, 2, 8>{}, Radices<16, 16>{}),
    make_xcd<double, 256, 256, 8, 128, 3, LD | ST>(10, 16, 4, Radices<16, 16>{}, Radices<16, 16>{}),
    make_xcd<double, 256, 512, 8, 256, 2, LD | ST>(4, 8, 2, Radices<8, 4, 8>{}, Radices<16, 2, 16>{}),
    make_xcd<double, 512, 512, 8, 256, 2, LD | ST>(2, 5, 2, Radices<16, 2, 16>{}, Radices<16, 2, 16>{}, 0, 256 * MiB),
};

}  // namespace

const XcdEntry *xcd_entries(int *count)
{
    *count = (int)(sizeof(kXcd) / sizeof(kXcd[0]));
    return kXcd;
}

hipError_t launch_xcd_reset(uint32_t *state, int64_t words, hipStream_t s)
{
    hipLaunchKernelGGL(xcd_reset_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, state, words);
    return hipGetLastError();
}

}  // namespace gfft
