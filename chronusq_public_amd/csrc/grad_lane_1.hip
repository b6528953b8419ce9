// Templated gradient kernels, class group 1 (eri_grad_impl.hpp).
#include "eri_grad_impl.hpp"

namespace cqx {
CQX_GRAD_GROUP(1)
}  // namespace cqx
