// batch_rows.hpp -- the batched kernels over the rows of the ELL (SpMV, sweeps,
// restriction) and their launcher; the bodies are the row_* functions of
// kernels.hpp.  batch_rows_pat.hip and batch_rows_col.hip instantiate the
// launcher for the two column sources.
#pragma once
#include "batch.hpp"
#include "kernels.hpp"

namespace hpcgx
{

#define BSEG()                                                \
    const int64_t b_ = xcd_block(blockIdx.x, gridDim.x);      \
    const BSeg& S = segs[seg_map(segs, nseg)[b_]];            \
    if(gated(S.gate)) return;                                 \
    const int64_t lb = b_ - S.blk0;

// launches a BLaunch of a kind up to BK_RESTRICT; PAT: every segment has row patterns
template <bool PAT>
int launch_batch_rows(const BLaunch& L, hipStream_t s);

}  // namespace hpcgx
