// What conv_dw_pw.hip and conv_blocks.hip share: a pair's arguments and the block that keeps them.
#pragma once
#include "common.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"

namespace mg {

struct DwPwArgs {
    const uint32_t* src;
    const uint32_t* dflt;    // [C/4][3][3] dwords of 4 channel bytes
    const int32_t* dbias;    // or NULL
    const int8_t* wp;        // packed pointwise filter [C/32][OCP][32], halves swapped when (oc >> 3) & 1
    const int32_t* pbias;    // or NULL
    uint32_t* dst;
    int src_bytes, dst_bytes;
    int ih, iw, oh, ow, OC, OCP;
    int plane;               // bytes of an input plane set
    int xg, groups;          // groups of 4 pixels per row, in all (a tile: 16 SUB groups)
    int slices;              // workgroups that share a tile's output channels
    // tiles of an XCD and how many XCDs have one more, runs of an XCD; tiles of a run and how many runs of an XCD with
    // the fewer tiles have one more (a single "XCD" where the runs are no multiple of eight); workgroups of an XCD where
    // those are one, else 0
    int xcds, xcd_q, xcd_r, xcd_runs, run_q, run_r, per_xcd;
    FastDiv d_xg, d_oh, d_slices;
    RequantPack dq, pq;
};
// What a workgroup reads at its start, in whole 64-byte lines. The kernel gets its address: 8 bytes of
// arguments, which the launch costs the host 2.5 us, where the 256 themselves cost 3.3 (up to 104 bytes 2.6, 2 KB 3.9),
// and an argument that short is in registers when a wave starts (the build asks for it), so that the first round trip goes
// to these lines instead of the argument segment. Launched again and again, 32 channels N=1 4.5 -> 4.0 us, 512 6.8 -> 6.2.
struct DwPwParams {
    union {
        DwPwArgs a;
        unsigned words[64];
    };
};
static_assert(sizeof(DwPwArgs) <= 256 && sizeof(DwPwParams) % 64 == 0, "four lines");

// What is kept of a pair from one launch to the next: how it is launched, and its arguments on the device - both forms that the
// requantisation's switch chooses between, written once and never again: whatever is launched, captured or replayed
// later, on whichever stream, finds them as they were.
typedef void (*DwPwKernel)(const DwPwParams*);
struct DpLaunch {
    DwPwKernel kern;
    size_t lds;
    unsigned workgroups;
};
struct DwPwBlock {
    DwPwParams* dev = nullptr;  // [2]: by the proven multiply-adds where there are any, by the reference's sequence (mode 3)
    DwPwParams host[2];
    DpLaunch launch;
    int act = 0;  // of the pointwise layer
};
}  // namespace mg
