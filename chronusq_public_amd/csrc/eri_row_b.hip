// Row kernels of class group B, FP64 and FP32 evaluation.
#include <mutex>

#include "eri_row_impl.hpp"

namespace cqx {
CQX_ROW_GROUP(1, CQX_ROW_CLASSES_B)
}  // namespace cqx
