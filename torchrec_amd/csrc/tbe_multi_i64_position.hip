// Instantiates the several-class window kernels for int64_t ids, kByPosition (see tbe_multi_impl.h).
#include "tbe_multi_impl.h"

namespace tra {
TRA_DEFINE_MULTI(int64_t, kByPosition)
}  // namespace tra
