// batch_rows_col.hip -- the batched row kernels, columns from the column array.
#include "batch_rows_impl.hpp"

namespace hpcgx
{

template int launch_batch_rows<false>(const BLaunch& L, hipStream_t s);

}  // namespace hpcgx
