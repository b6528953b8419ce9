// Row kernels of class group C, FP64 and FP32 evaluation.
#include <mutex>

#include "eri_row_impl.hpp"

namespace cqx {
CQX_ROW_GROUP(2, CQX_ROW_CLASSES_C)
}  // namespace cqx
