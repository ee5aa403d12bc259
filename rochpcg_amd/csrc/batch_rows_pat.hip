// batch_rows_pat.hip -- the batched row kernels, columns from the row patterns.
#include "batch_rows_impl.hpp"

namespace hpcgx
{

template int launch_batch_rows<true>(const BLaunch& L, hipStream_t s);

}  // namespace hpcgx
