// batch_rows_impl.hpp -- kernels and launcher declared in batch_rows.hpp.
#pragma once
#include "batch_rows.hpp"

namespace hpcgx
{

// LDS of the row patterns a block stages, and its rows' column source; threads
// past the end of the segment work on its last rows and store nothing
#define BCOLS(R)                                                                    \
    __shared__ int4 pat_lds[PAT ? PAT_MAX * PAT_QUADS : 1];                          \
    const int64_t i = (lb * BS + threadIdx.x) * (R);                                \
    const bool live = i < S.size;                                                   \
    const int64_t row = S.off + (live ? i : S.size - (R));                          \
    Cols<PAT, (R), BS> cols(S.cols, pat_lds, row, true);

// the whole level, block by block of one colour (one segment per colour)
template <bool PAT, typename VT, typename XT, typename YT, bool DOT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_spmv(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    double acc = 0.0;
    XT s[R];
    row_spmv<VT, XT, R>(row, cols, (const VT*)S.val, (const XT*)S.r, s);
    if(live)
    {
        st_cvt<R>((YT*)S.x + row, s);
        if(DOT)
        {
            XT xr[R];
            ld<R>((const XT*)S.r + row, xr);
#pragma unroll
            for(int k = 0; k < R; ++k) acc = fmaT((double)xr[k], (double)s[k], acc);
        }
    }
    if(DOT) block_partial<BS>(acc, S.ra.partial, S.part0 + lb);
}

// The sweeps are compiled for the widest window of the launch's segments
// (BLaunch::win), like the single-problem kernels, and for R rows per thread
// (BLaunch::rows; 2 only when every segment's offset and size are even).
template <bool PAT, int NS, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_fwd_zero(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    row_fwd_zero<NS, VT, XT, RT, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (const RT*)S.r, (XT*)S.x);
}

template <bool PAT, int NS, typename VT, typename XT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_bwd_zero(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    if(S.t)
        row_bwd_zero<NS, VT, XT, true, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (XT*)S.x, (XT*)S.t);
    else
        row_bwd_zero<NS, VT, XT, false, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (XT*)S.x, nullptr);
}

// every segment reuses its pre-smoother's upper sums (BLaunch::all_u)
template <bool PAT, int NA, int NB, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_fwd_full_u(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    row_fwd_full_u<NA, NB, VT, XT, RT, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (const RT*)S.r,
                                          (XT*)S.x, (XT*)S.t);
}

template <bool PAT, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_fwd_full(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    if(S.use_u)
        row_fwd_full_u<W - 1, W - 1, VT, XT, RT, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg,
                                                    (const RT*)S.r, (XT*)S.x, (XT*)S.t);
    else if(S.t)
        row_fwd_full<VT, XT, RT, R>(row, live, cols, (const VT*)S.val, (const RT*)S.r, (XT*)S.x, (XT*)S.t);
    else   // a last colour: no upper entries, and no backward visit that needs t
        row_fwd_zero<W - 1, VT, XT, RT, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (const RT*)S.r,
                                           (XT*)S.x);
}

template <bool PAT, int NS, typename VT, typename XT, int R, int BS>
__global__ __launch_bounds__(BS) void kb_bwd_full(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCOLS(R);
    row_bwd_full<NS, VT, XT, R>(row, live, cols, (const VT*)S.val, (const VT*)S.dg, (const XT*)S.t, (XT*)S.x);
}

template <bool PAT, typename VT, typename XT, typename RT, int BS>
__global__ __launch_bounds__(BS) void kb_restrict(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    __shared__ int4 pat_lds[PAT ? PAT_MAX * PAT_QUADS : 1];
    const int64_t k = lb * BS + threadIdx.x;
    const int64_t row = S.f2c_fine[k < S.size ? k : S.size - 1];
    Cols<PAT, 1, BS> cols(S.cols, pat_lds, row, true);
    const XT s = row_restrict<VT, XT, RT>(row, cols, (const VT*)S.val, (const RT*)S.r, (const XT*)S.x);
    if(k < S.size) ((XT*)S.rc)[S.f2c_coarse[k]] = s;
}

template <typename F>
static void with_rows(int rows, F&& f)
{
    if(rows == 2)
        f(std::integral_constant<int, 2>{});
    else
        f(std::integral_constant<int, 1>{});
}

template <bool PAT, int BS>
static void launch_rows_bs(const BLaunch& L, hipStream_t s)
{
    const dim3 g((unsigned)L.nblocks), b(BS);
    const BSeg* T = L.segs;
    const int n = L.nseg;
    const bool f64 = L.prec == PREC_F64;
    switch(L.kind)
    {
    case BK_SPMV:
        // outer SpMV: f64 vectors over either store; MG-internal SpMV is not batched
        with_rows(L.rows, [&](auto RR) {
            constexpr int R = decltype(RR)::value;
            if(f64)
            {
                if(L.dot)
                    hipLaunchKernelGGL((kb_spmv<PAT, double, double, double, true, R, BS>), g, b, 0, s, T, n);
                else
                    hipLaunchKernelGGL((kb_spmv<PAT, double, double, double, false, R, BS>), g, b, 0, s, T, n);
            }
            else
            {
                if(L.dot)
                    hipLaunchKernelGGL((kb_spmv<PAT, __half, double, double, true, R, BS>), g, b, 0, s, T, n);
                else
                    hipLaunchKernelGGL((kb_spmv<PAT, __half, double, double, false, R, BS>), g, b, 0, s, T, n);
            }
        });
        break;
    case BK_FWD_ZERO:
        with_rows(L.rows, [&](auto RR) {
            constexpr int R = decltype(RR)::value;
            with_window(L.win, [&](auto NN) {
                constexpr int NS = decltype(NN)::value;
                if(f64)
                    hipLaunchKernelGGL((kb_fwd_zero<PAT, NS, double, double, double, R, BS>), g, b, 0, s, T, n);
                else if(L.r_f64)
                    hipLaunchKernelGGL((kb_fwd_zero<PAT, NS, __half, float, double, R, BS>), g, b, 0, s, T, n);
                else
                    hipLaunchKernelGGL((kb_fwd_zero<PAT, NS, __half, float, float, R, BS>), g, b, 0, s, T, n);
            });
        });
        break;
    case BK_BWD_ZERO:
        with_rows(L.rows, [&](auto RR) {
            constexpr int R = decltype(RR)::value;
            with_window(L.win, [&](auto NN) {
                constexpr int NS = decltype(NN)::value;
                if(f64)
                    hipLaunchKernelGGL((kb_bwd_zero<PAT, NS, double, double, R, BS>), g, b, 0, s, T, n);
                else
                    hipLaunchKernelGGL((kb_bwd_zero<PAT, NS, __half, float, R, BS>), g, b, 0, s, T, n);
            });
        });
        break;
    case BK_FWD_FULL:
        with_rows(L.rows, [&](auto RR) {
            constexpr int R = decltype(RR)::value;
            if(L.all_u)
                with_window_pair(L.win, L.win_tail, [&](auto NA_, auto NB_) {
                    constexpr int NA = decltype(NA_)::value, NB = decltype(NB_)::value;
                    if(f64)
                        hipLaunchKernelGGL((kb_fwd_full_u<PAT, NA, NB, double, double, double, R, BS>), g, b, 0, s, T,
                                           n);
                    else if(L.r_f64)
                        hipLaunchKernelGGL((kb_fwd_full_u<PAT, NA, NB, __half, float, double, R, BS>), g, b, 0, s, T,
                                           n);
                    else
                        hipLaunchKernelGGL((kb_fwd_full_u<PAT, NA, NB, __half, float, float, R, BS>), g, b, 0, s, T,
                                           n);
                });
            else if(f64)
                hipLaunchKernelGGL((kb_fwd_full<PAT, double, double, double, R, BS>), g, b, 0, s, T, n);
            else if(L.r_f64)
                hipLaunchKernelGGL((kb_fwd_full<PAT, __half, float, double, R, BS>), g, b, 0, s, T, n);
            else
                hipLaunchKernelGGL((kb_fwd_full<PAT, __half, float, float, R, BS>), g, b, 0, s, T, n);
        });
        break;
    case BK_BWD_FULL:
        with_rows(L.rows, [&](auto RR) {
            constexpr int R = decltype(RR)::value;
            with_window(L.win, [&](auto NN) {
                constexpr int NS = decltype(NN)::value;
                if(f64)
                    hipLaunchKernelGGL((kb_bwd_full<PAT, NS, double, double, R, BS>), g, b, 0, s, T, n);
                else
                    hipLaunchKernelGGL((kb_bwd_full<PAT, NS, __half, float, R, BS>), g, b, 0, s, T, n);
            });
        });
        break;
    case BK_RESTRICT:
        if(f64)
            hipLaunchKernelGGL((kb_restrict<PAT, double, double, double, BS>), g, b, 0, s, T, n);
        else if(L.r_f64)
            hipLaunchKernelGGL((kb_restrict<PAT, __half, float, double, BS>), g, b, 0, s, T, n);
        else
            hipLaunchKernelGGL((kb_restrict<PAT, __half, float, float, BS>), g, b, 0, s, T, n);
        break;
    default: break;
    }
}

template <bool PAT>
int launch_batch_rows(const BLaunch& L, hipStream_t s)
{
    switch(L.block)
    {
    case 64: launch_rows_bs<PAT, 64>(L, s); break;
    case 128: launch_rows_bs<PAT, 128>(L, s); break;
    default: launch_rows_bs<PAT, 256>(L, s); break;
    }
    HPCGX_HIP(hipGetLastError());
    return 0;
}

}  // namespace hpcgx
