// launch.hpp -- host helpers shared by the launchers of the ELL kernels
// (ops.hip, sweeps_*.hip).  Include from .hip files only.
#pragma once
#include "common.hpp"
#include "kernels.hpp"

#include <string>
#include <type_traits>

namespace hpcgx
{

// LDS of the row patterns a block stages (Cols<true>)
#define PAT_LDS() __shared__ int4 pat_lds[PAT ? PAT_MAX * PAT_QUADS : 1]

static inline unsigned nblk(int64_t n, int bs) { return (unsigned)ceil_div(n, bs); }

#define HPCGX_KCHECK() HPCGX_HIP(hipGetLastError())

// Launch shapes compiled in: rows per thread {1,2} x block {64,128,256}.
template <typename F>
static int with_shape(const Shape& sh, F&& f)
{
    using std::integral_constant;
    switch(sh.rows * 1000 + sh.block)
    {
    case 1064: return f(integral_constant<int, 1>{}, integral_constant<int, 64>{});
    case 1128: return f(integral_constant<int, 1>{}, integral_constant<int, 128>{});
    case 1256: return f(integral_constant<int, 1>{}, integral_constant<int, 256>{});
    case 2064: return f(integral_constant<int, 2>{}, integral_constant<int, 64>{});
    case 2128: return f(integral_constant<int, 2>{}, integral_constant<int, 128>{});
    case 2256: return f(integral_constant<int, 2>{}, integral_constant<int, 256>{});
    default: break;
    }
    set_error("unsupported launch shape (rows " + std::to_string(sh.rows) + ", block " + std::to_string(sh.block) + ")");
    return -2;
}

// R rows per thread need every colour block to be R-aligned (a thread's R
// rows then share their ELL slice).
static Shape fit(const Level& L, Shape sh)
{
    bool ok = true;
    for(int c = 0; c < L.ncolors && ok; ++c) ok = (L.offsets[c] % sh.rows) == 0 && (L.sizes[c] % sh.rows) == 0;
    if(!ok) sh.rows = 1;
    return sh;
}

// Launches read the row patterns where the level has them (Level::pat), the
// column array elsewhere.
template <typename F>
static auto with_pat(const Level& L, F&& f)
{
    if(L.use_pat()) return f(std::integral_constant<bool, true>{});
    return f(std::integral_constant<bool, false>{});
}

// element-type views of a level's arrays
template <typename VT>
inline const VT* vals_of(const Level& L);
template <>
inline const double* vals_of<double>(const Level& L) { return L.ell_val; }
template <>
inline const __half* vals_of<__half>(const Level& L) { return L.ell_h; }

template <typename VT>
inline const VT* diag_of(const Level& L);
template <>
inline const double* diag_of<double>(const Level& L) { return L.diag64; }
template <>
inline const __half* diag_of<__half>(const Level& L) { return L.diag_h; }

}  // namespace hpcgx
