// Templated gradient kernels, class group 2 (eri_grad_impl.hpp).
#include "eri_grad_impl.hpp"

namespace cqx {
CQX_GRAD_GROUP(2)
}  // namespace cqx
