// Row kernels of class group D, FP64 evaluation.
#include <mutex>

#include "eri_row_impl.hpp"

namespace cqx {
CQX_ROW_GROUP(3, CQX_ROW_CLASSES_D)
}  // namespace cqx
