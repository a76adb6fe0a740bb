// Instantiates the sixteen-lane lookup kernels for int64_t ids, kUnweighted (see tbe_group_impl.h).
#include "tbe_group_impl.h"

namespace tra {
TRA_DEFINE_GROUP(int64_t, kUnweighted)
}  // namespace tra
