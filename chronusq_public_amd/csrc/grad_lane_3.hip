// Templated gradient kernels, class group 3 (eri_grad_impl.hpp).
#include "eri_grad_impl.hpp"

namespace cqx {
CQX_GRAD_GROUP(3)
}  // namespace cqx
