// gfft_xcd.h -- four-steps with both passes in one persistent launch.
//
// Two launches write the whole intermediate to HBM and read it back.  Here each
// XCD takes whole transforms, its workgroups running the column tiles of one
// and, a few transforms later, its transposing row tiles; the intermediate in
// between passes through a ring of 48-256 MiB (3-18 transforms per XCD) that is
// reused before the Infinity Cache has to write all of it out: the traffic past
// the L2 is that of two launches, at 6.7 TB/s where those reach 5.3.  Tiles hand
// over within one XCD, whose L2 is common to them, which needs no cache
// write-back.
#pragma once
#include "gfft_registry.h"

namespace gfft {

constexpr int kXcds = 8;  // of an MI355X; XCC_ID is 0 .. 7

struct XcdArgs {
    TileArgs col, row;   // col.in / row.out: the caller's buffers; the other sides: scratch
    uint32_t *state;     // xcd_state_words(), zeroed before each launch
    int32_t batch;
    int32_t lag, ring;   // row tiles run `lag` transforms behind; ring slots per XCD
    int32_t blocks;      // transforms an XCD may count (xcd_blocks)
};

struct XcdEntry {
    int prec, lg;
    KernelEntry col, row;  // shapes (for their twiddle tables and the bounds proof)
    int NT, lds_bytes;
    int lag, ring, per_cu;  // chosen per length, see kern_xcd.hip
    // The kernel by its cache hints: XCD_PLAIN_LD / XCD_PLAIN_ST are the column
    // tiles' loads / the row tiles' stores not streamed (null: not compiled).
    void (*fn[4])(XcdArgs);
    int plain;               // the hints taken where a side's runs share lines (xcd_hints)
    int64_t out_least, both_least;  // bytes a side from which it is taken there (-1: never)
};

enum : int { XCD_PLAIN_LD = 1, XCD_PLAIN_ST = 2 };

// The hints of a launch of `bytes` a side whose runs start at multiples of `in`
// and `out` bytes (or any addresses with their low bits), or -1: two launches.
// Streamed loads want whole 128-byte lines, streamed stores whole 32-byte
// sectors; see kern_xcd.hip for the figures.
inline int xcd_hints(const XcdEntry &e, int64_t bytes, uint64_t in, uint64_t out)
{
    const bool in_parts = in % 128 != 0, out_parts = out % 32 != 0;
    const int64_t least = out_parts ? (in_parts ? e.both_least : e.out_least) : 0;
    if (least < 0 || bytes < least) return -1;
    return e.plain & ((in_parts ? XCD_PLAIN_LD : 0) | (out_parts ? XCD_PLAIN_ST : 0));
}

const XcdEntry *xcd_entries(int *count);
hipError_t launch_xcd_reset(uint32_t *state, int64_t words, hipStream_t s);

// Transforms one XCD may count: all of them, the lag, and what every workgroup
// of the launch may take past the last one before it finds out.
inline int64_t xcd_blocks(int64_t batch, int64_t lag, int64_t grid) { return batch + lag + grid + 8; }
inline int64_t xcd_state_words(int64_t blocks) { return 32 * (1 + kXcds) + (int64_t)kXcds * blocks * 4; }

}  // namespace gfft
