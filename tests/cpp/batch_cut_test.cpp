// batch_cut_test.cpp -- host-only check of how a batched launch of many segments is
// cut into launches (launch_end in rochpcg_amd/csrc/batch.hpp).  For every line
// "problems segments" of stdin: the launches follow each other, hold every segment
// once, at most MAX_SEGS each, no problem in two of them, and no two neighbours that
// would fit one launch.  Prints "ok <launches>..." or the first failure.
#include <cstdio>

#include "../../rochpcg_amd/csrc/batch.hpp"

using namespace hpcgx;

int main()
{
    unsigned long long problems, subs;
    std::string counts;
    while(scanf("%llu %llu", &problems, &subs) == 2)
    {
        std::vector<size_t> prob;
        for(size_t k = 0; k < problems; ++k)
            for(size_t c = 0; c < subs; ++c) prob.push_back(k);
        size_t launches = 0;
        for(size_t j0 = 0, e; j0 < prob.size(); j0 = e, ++launches)
        {
            e = launch_end(prob, j0);
            const bool whole = e == prob.size() || (prob[e] != prob[e - 1] && e + subs - j0 > MAX_SEGS);
            if(e <= j0 || e > prob.size() || e - j0 > MAX_SEGS || !whole)
            {
                printf("FAIL %llu problems of %llu segments: launch [%zu, %zu)\n", problems, subs, j0, e);
                return 1;
            }
        }
        counts += " " + std::to_string(launches);
    }
    printf("ok%s\n", counts.c_str());
    return 0;
}
