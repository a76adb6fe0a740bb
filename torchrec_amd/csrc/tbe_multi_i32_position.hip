// Instantiates the several-class window kernels for int32_t ids, kByPosition (see tbe_multi_impl.h).
#include "tbe_multi_impl.h"

namespace tra {
TRA_DEFINE_MULTI(int32_t, kByPosition)
}  // namespace tra
