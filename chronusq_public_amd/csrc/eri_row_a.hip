// Row kernels of class group A, FP64 and FP32 evaluation.
#include <mutex>

#include "eri_row_impl.hpp"

namespace cqx {
CQX_ROW_GROUP(0, CQX_ROW_CLASSES_A)
}  // namespace cqx
