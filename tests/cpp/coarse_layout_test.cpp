// coarse_layout_test.cpp -- host-only check of the layout of a coarse plan's
// allocation (rochpcg_amd/csrc/coarse.hpp).  For every line "rows steps levels"
// of stdin: the steps and the level descriptions start at addresses their types
// may have (the allocation itself at a multiple of 256), nothing overlaps, and
// the descriptions end the allocation.  Prints "ok <lines>" or the first failure.
#include <cstdio>

#include "../../rochpcg_amd/csrc/coarse.hpp"

using namespace hpcgx;

int main()
{
    unsigned long long rows, steps, levels, n = 0;
    while(scanf("%llu %llu %llu", &rows, &steps, &levels) == 3)
    {
        const size_t columns = (size_t)SEC_COUNT * ((W + 3) / 4) * 4 * rows;
        const CoarseLayout o = coarse_layout(columns, steps, levels);
        if(o.steps % alignof(CoarseStep) || o.levels % alignof(CoarseLevel) || o.steps < 2 * columns ||
           o.levels < o.steps + steps * sizeof(CoarseStep) || o.bytes != o.levels + levels * sizeof(CoarseLevel))
        {
            printf("FAIL rows %llu steps %llu levels %llu: steps at %zu, levels at %zu\n", rows, steps, levels, o.steps,
                   o.levels);
            return 1;
        }
        ++n;
    }
    printf("ok %llu\n", n);
    return 0;
}
