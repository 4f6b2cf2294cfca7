// gfft_xcd.h -- four-steps with both passes in one persistent launch.
//
// Two launches write the whole intermediate to HBM and read it back.  Here each
// XCD takes whole transforms, its workgroups running the column tiles of one
// and, a few transforms later, its transposing row tiles; the intermediate in
// between lives in a ring of 48-160 MB (8-16 transforms per XCD) that the 256 MB
// Infinity Cache holds, so HBM moves the input and the output only.  Tiles hand
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
    void (*fn)(XcdArgs);
};

const XcdEntry *xcd_entries(int *count);
hipError_t launch_xcd_reset(uint32_t *state, int64_t words, hipStream_t s);

// Transforms one XCD may count: all of them, the lag, and what every workgroup
// of the launch may take past the last one before it finds out.
inline int64_t xcd_blocks(int64_t batch, int64_t lag, int64_t grid) { return batch + lag + grid + 8; }
inline int64_t xcd_state_words(int64_t blocks) { return 32 * (1 + kXcds) + (int64_t)kXcds * blocks * 4; }

}  // namespace gfft
