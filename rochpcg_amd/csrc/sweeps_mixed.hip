// sweeps_mixed.hip -- the SymGS sweeps with f16 values and f32 vectors (f64
// right-hand side on level 0 of the mixed CG, f32 below).
#include "sweeps.hpp"

namespace hpcgx
{

int sweep_mixed(const Level& L, int part, const void* r, bool r_f64, void* x, void* t, hipStream_t s, const int* gate)
{
    return with_pat(L, [&](auto PP) -> int {
        constexpr bool PAT = decltype(PP)::value;
        if(r_f64) return sweep_t<PAT, __half, float, double>(L, part, r, x, t, s, gate);
        return sweep_t<PAT, __half, float, float>(L, part, r, x, t, s, gate);
    });
}

}  // namespace hpcgx
