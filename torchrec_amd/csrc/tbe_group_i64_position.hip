// Instantiates the sixteen-lane lookup kernels for int64_t ids, kByPosition (see tbe_group_impl.h).
#include "tbe_group_impl.h"

namespace tra {
TRA_DEFINE_GROUP(int64_t, kByPosition)
}  // namespace tra
