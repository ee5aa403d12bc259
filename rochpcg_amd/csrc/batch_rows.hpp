// batch_rows.hpp -- the batched kernels over the rows of the ELL (SpMV, sweeps,
// restriction) and their launcher; the bodies are the row_* functions of
// kernels.hpp.  batch_rows_pat.hip and batch_rows_col.hip instantiate the
// launcher for the two column sources.
#pragma once
#include "batch.hpp"
#include "kernels.hpp"

namespace hpcgx
{

// the segment of logical block b: the block map's words by scalar loads
__device__ __forceinline__ int seg_of(const BSeg* segs, int nseg, int64_t b)
{
    typedef const __attribute__((address_space(4))) uint32_t ConstWord;
    return (int)((((ConstWord*)seg_map(segs, nseg))[b >> 1] >> (16 * (int)(b & 1))) & 0xffffu);
}

// A block's way to its rows: map -> segment -> flag -> pattern, each a load that
// waits for the one before.  All are scalar loads, and the fields every kernel needs
// come together (the asm has them in registers before the flag is looked at); with
// vector loads of the map and the flag and the fields behind the flag, 64 problems of
// 16^3 to 96^3 took 131.7 and 72.9 ms to 1e-9 (FP64, mixed) where they take 128.4 and
// 68.6.
#define BSEG()                                                                                              \
    const int64_t b_ = xcd_block(blockIdx.x, gridDim.x);                                                    \
    const BSeg& S = segs[seg_of(segs, nseg, b_)];                                                           \
    asm volatile("" ::"s"(S.off), "s"(S.size), "s"(S.blk0), "s"(S.cols.pat), "s"(S.cols.tab),               \
                 "s"(S.cols.npat), "s"(S.val), "s"(S.dg), "s"(S.r), "s"(S.x), "s"(S.gate));                 \
    if(gated(S.gate)) return;                                                                               \
    const int64_t lb = b_ - S.blk0;

// launches a BLaunch of a kind up to BK_RESTRICT; PAT: every segment has row patterns
template <bool PAT>
int launch_batch_rows(const BLaunch& L, hipStream_t s);

}  // namespace hpcgx
