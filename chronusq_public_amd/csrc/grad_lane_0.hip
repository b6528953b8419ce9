// Templated gradient kernels, class group 0 (eri_grad_impl.hpp).
#include "eri_grad_impl.hpp"

namespace cqx {
CQX_GRAD_GROUP(0)
}  // namespace cqx
