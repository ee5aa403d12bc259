// sweeps_f64.hip -- the SymGS sweeps with f64 values and vectors.
#include "sweeps.hpp"

namespace hpcgx
{

int sweep_f64(const Level& L, int part, const void* r, void* x, void* t, hipStream_t s, const int* gate)
{
    return with_pat(L, [&](auto PP) -> int {
        return sweep_t<decltype(PP)::value, double, double, double>(L, part, r, x, t, s, gate);
    });
}

}  // namespace hpcgx
