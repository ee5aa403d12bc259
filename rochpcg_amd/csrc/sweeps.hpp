// sweeps.hpp -- the per-colour SymGS sweep kernels and their launcher for one
// (value, vector, rhs) type triple and column source; instantiated by
// sweeps_f64.hip and sweeps_mixed.hip.  The bodies are the row_* functions of
// kernels.hpp.
//
// Reference kernels whose results these reproduce:
//   SymGS sweep         kernel_symgs_sweep        ComputeSYMGS.cpp:113-151, :369-404
//   zero-guess SymGS    kernel_pointwise_mult / kernel_forward_sweep_0 /
//                       kernel_backward_sweep_0   ComputeSYMGS.cpp:238-341, :406-454
#pragma once
#include "launch.hpp"
#include "ops.hpp"

namespace hpcgx
{

// Per-colour sweeps: block b covers rows off + T*BS*R + [0, BS*R), where T is
// L = xcd_block(b), mapped through the colour's column order (ZMap) on large
// planes.  Consecutive colour launches alternate direction (size < 0 marks a
// reversed launch): each XCD then starts a launch on the slab it finished the
// previous one on, whose neighbours' x is still in its caches.  Threads past
// the end work on the last rows and store nothing.
// The flag that stops converged solves is looked at behind the row's arithmetic
// and its pattern's load (cheap, and in range whatever the flag), ahead of its
// values: an iteration of 104^3 takes 553 in place of 569 us in FP64 and 397 in
// place of 412 mixed, one that is stopped the same 0.17 ms.  The kernels take the
// flag and what the row's arithmetic needs first, where arguments are preloaded.
#define SWEEP_ROW()                                                                   \
    const bool stop_ = gated(gate);                                                   \
    PAT_LDS();                                                                        \
    int64_t Lb_ = xcd_block(blockIdx.x, gridDim.x);                                   \
    if(size < 0)                                                                      \
    {                                                                                 \
        size = -size;                                                                 \
        Lb_ = (int64_t)gridDim.x - 1 - Lb_;                                           \
    }                                                                                 \
    if(zm.k > 1)                                                                      \
    {                                                                                 \
        const unsigned per_ = (unsigned)zm.planes * (unsigned)zm.tpc;                 \
        const unsigned lb_ = (unsigned)Lb_, col_ = lb_ / per_, rem_ = lb_ - col_ * per_; \
        const unsigned pl_ = rem_ / (unsigned)zm.tpc;                                 \
        Lb_ = ((int64_t)pl_ * zm.k + col_) * zm.tpc + (rem_ - pl_ * (unsigned)zm.tpc); \
    }                                                                                 \
    const int64_t i = Lb_ * (BS * R) + (int64_t)threadIdx.x * R;                      \
    const bool live = i < size;                                                       \
    const int64_t row = off + (live ? i : size - R);                                  \
    Cols<PAT, R, BS> cols(ca, pat_lds, row, true);                                    \
    if(stop_) return;

template <bool PAT, int NS, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void k_fwd_zero(const int* gate, int64_t off, int64_t size, const VT* __restrict__ val,
                                                 const VT* __restrict__ dg, const RT* __restrict__ r,
                                                 XT* __restrict__ x, ZMap zm, ColArgs ca)
{
    SWEEP_ROW();
    row_fwd_zero<NS, VT, XT, RT, R>(row, live, cols, val, dg, r, x);
}

template <bool PAT, int NS, typename VT, typename XT, bool STORE_U, int R, int BS>
__global__ __launch_bounds__(BS) void k_bwd_zero(const int* gate, int64_t off, int64_t size, const VT* __restrict__ val,
                                                 const VT* __restrict__ dg, XT* __restrict__ x, XT* __restrict__ u,
                                                 ZMap zm, ColArgs ca)
{
    SWEEP_ROW();
    row_bwd_zero<NS, VT, XT, STORE_U, R>(row, live, cols, val, dg, x, u);
}

template <bool PAT, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void k_fwd_full(int64_t off, int64_t size, ZMap zm, ColArgs ca,
                                                 const VT* __restrict__ val, const RT* __restrict__ r,
                                                 XT* __restrict__ x, XT* __restrict__ t, const int* gate)
{
    SWEEP_ROW();
    row_fwd_full<VT, XT, RT, R>(row, live, cols, val, r, x, t);
}

template <bool PAT, int NA, int NB, typename VT, typename XT, typename RT, int R, int BS>
__global__ __launch_bounds__(BS) void k_fwd_full_u(const int* gate, int64_t off, int64_t size,
                                                   const VT* __restrict__ val, const VT* __restrict__ dg,
                                                   const RT* __restrict__ r, XT* __restrict__ x, XT* __restrict__ t,
                                                   ZMap zm, ColArgs ca)
{
    SWEEP_ROW();
    row_fwd_full_u<NA, NB, VT, XT, RT, R>(row, live, cols, val, dg, r, x, t);
}

template <bool PAT, int NS, typename VT, typename XT, int R, int BS>
__global__ __launch_bounds__(BS) void k_bwd_full(const int* gate, int64_t off, int64_t size, const VT* __restrict__ val,
                                                 const VT* __restrict__ dg, const XT* __restrict__ t,
                                                 XT* __restrict__ x, ZMap zm, ColArgs ca)
{
    SWEEP_ROW();
    row_bwd_full<NS, VT, XT, R>(row, live, cols, val, dg, t, x);
}
#undef SWEEP_ROW

// The sweeps' block order for a colour of `size` rows in tiles of `tile` rows
// (grid = its tile count).  Planes of the half-resolution colour grid whose x
// gathers (7 other colours, 3 planes, 8 B) outgrow an XCD's 4 MB L2 are cut
// into columns of >= min_rows rows (measured best: 8192 for the f64 sweeps,
// 4096 for the f16/f32 ones), so that the blocks in flight on an XCD march
// through one column's planes; Level::zcols > 0 forces a column count.
static ZMap zmap_for(const Level& L, int64_t size, int tile, unsigned grid, int64_t min_rows)
{
    ZMap z;
    if(L.zcols == 1 || L.ncolors != 8 || ((L.nx | L.ny | L.nz) & 1) != 0) return z;
    const int64_t plane = (int64_t)(L.nx / 2) * (L.ny / 2), planes = L.nz / 2;
    if(size != plane * planes || plane % tile) return z;
    const int64_t tpp = plane / tile;
    int64_t k = L.zcols;
    if(k == 0)
    {
        if(plane * 8 * 21 <= ((int64_t)6 << 20)) return z;
        k = 1;
        while(tpp % (2 * k) == 0 && (tpp / (2 * k)) * tile >= min_rows) k *= 2;
    }
    if(k <= 1 || tpp % k || (int64_t)grid != planes * tpp) return z;
    z.k = (int)k;
    z.tpc = (int)(tpp / k);
    z.planes = (int)planes;
    return z;
}

// one launch per colour c in [c0, c1) (step +1) or (c0, c1] (step -1); a
// colour whose slot window (kind `wk`, one row per thread) exceeds 16 slots
// runs with the op's wide shape, the others with its narrow shape
template <typename Launch>
static int per_color(const Level& L, int prec, int which, int wk, int c_first, int c_last, int step,
                     Launch&& launch)
{
    for(int c = c_first; step > 0 ? c <= c_last : c >= c_last; c += step)
    {
        if(L.sizes[c] == 0) continue;
        const bool wide = (wk < 0) || L.win[wk][c] > 16;
        const Shape sh = fit(L, L.shp[prec][wide ? which : which + SH_NARROW]);
        HPCGX_TRY(with_shape(sh, [&](auto RR, auto BB) -> int {
            constexpr int R = decltype(RR)::value, BS = decltype(BB)::value;
            const dim3 grid(nblk(ceil_div(L.sizes[c], R), BS));
            // odd colours walk their blocks backwards (in both sweeps: forward
            // ends on colour 7 reversed, backward starts on colour 6 forwards,
            // so every launch starts on the slab the previous one ended on)
            const int64_t size = (c & 1) ? -(int64_t)L.sizes[c] : (int64_t)L.sizes[c];
            launch(RR, BB, grid, c, size, zmap_for(L, L.sizes[c], BS * R, grid.x, prec == PREC_F64 ? 8192 : 4096));
            HPCGX_KCHECK();
            return 0;
        }));
    }
    return 0;
}

// The sweep kernels of a level: part 0 = zero-guess forward (colours 0..n-1),
// 1 = zero-guess backward (n-2..0), 2 = forward keeping t (0..n-1), 3 =
// backward from t (n-2..0), 4 = part 1 also keeping the upper sums outside
// the last colour in t, 5 = part 2 reusing them (valid after part 4 when
// only last-colour rows changed in between).
template <bool PAT, typename VT, typename XT, typename RT>
static int sweep_t(const Level& L, int part, const void* rv, void* xv, void* tv, hipStream_t s, const int* gate)
{
    const RT* r = (const RT*)rv;
    XT* x = (XT*)xv;
    XT* t = (XT*)tv;
    const VT* val = vals_of<VT>(L);
    const VT* dg = diag_of<VT>(L);
    const int last = L.ncolors - 1;
    const int pr = std::is_same<VT, double>::value ? PREC_F64 : PREC_MIXED;
    auto fwd_zero = [&](auto RR, auto BB, dim3 grid, int c, int64_t sz, ZMap zm) {
        constexpr int R = decltype(RR)::value, BS = decltype(BB)::value;
        with_window(L.win[WIN_LOWER][c], [&](auto NN) {
            constexpr int NS = decltype(NN)::value;
            hipLaunchKernelGGL((k_fwd_zero<PAT, NS, VT, XT, RT, R, BS>), grid, dim3(BS), 0, s, gate,
                               (int64_t)L.offsets[c], sz, val, dg, r, x, zm, L.cols(c));
        });
    };
    switch(part)
    {
    case 0: return per_color(L, pr, SH_FWD_ZERO, WIN_LOWER, 0, last, 1, fwd_zero);
    case 1:
    case 4:
        if(last < 1) return 0;
        return per_color(L, pr, SH_BWD_ZERO, WIN_UPPER, last - 1, 0, -1, [&](auto RR, auto BB, dim3 grid, int c, int64_t sz, ZMap zm) {
            constexpr int R = decltype(RR)::value, BS = decltype(BB)::value;
            with_window(L.win[WIN_UPPER][c], [&](auto NN) {
                constexpr int NS = decltype(NN)::value;
                if(part == 4)
                    hipLaunchKernelGGL((k_bwd_zero<PAT, NS, VT, XT, true, R, BS>), grid, dim3(BS), 0, s,
                                       gate, (int64_t)L.offsets[c], sz, val, dg, x, t, zm, L.cols(c));
                else
                    hipLaunchKernelGGL((k_bwd_zero<PAT, NS, VT, XT, false, R, BS>), grid, dim3(BS), 0, s,
                                       gate, (int64_t)L.offsets[c], sz, val, dg, x, t, zm, L.cols(c));
            });
        });
    case 2:
    case 5:
        return per_color(L, pr, SH_FWD_FULL, part == 5 ? WIN_LOWER : -1, 0, last, 1, [&](auto RR, auto BB, dim3 grid, int c, int64_t sz, ZMap zm) {
            constexpr int R = decltype(RR)::value, BS = decltype(BB)::value;
            if(c == last)
                fwd_zero(RR, BB, grid, c, sz, zm);   // no upper entries, and no backward visit that needs t
            else if(part == 5)
                with_window_pair(L.win[WIN_LOWER][c], L.win[WIN_TAIL][c], [&](auto NA_, auto NB_) {
                    constexpr int NA = decltype(NA_)::value, NB = decltype(NB_)::value;
                    hipLaunchKernelGGL((k_fwd_full_u<PAT, NA, NB, VT, XT, RT, R, BS>), grid, dim3(BS), 0, s,
                                       gate, (int64_t)L.offsets[c], sz, val, dg, r, x, t, zm, L.cols(c));
                });
            else
                hipLaunchKernelGGL((k_fwd_full<PAT, VT, XT, RT, R, BS>), grid, dim3(BS), 0, s,
                                   (int64_t)L.offsets[c], sz, zm, L.cols(c), val, r, x, t, gate);
        });
    case 3:
        if(last < 1) return 0;
        return per_color(L, pr, SH_BWD_FULL, WIN_UPPER, last - 1, 0, -1, [&](auto RR, auto BB, dim3 grid, int c, int64_t sz, ZMap zm) {
            constexpr int R = decltype(RR)::value, BS = decltype(BB)::value;
            with_window(L.win[WIN_UPPER][c], [&](auto NN) {
                constexpr int NS = decltype(NN)::value;
                hipLaunchKernelGGL((k_bwd_full<PAT, NS, VT, XT, R, BS>), grid, dim3(BS), 0, s,
                                   gate, (int64_t)L.offsets[c], sz, val, dg, (const XT*)t, x, zm, L.cols(c));
            });
        });
    }
    set_error("invalid sweep part");
    return -2;
}

}  // namespace hpcgx
