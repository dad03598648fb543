// layer norm kernels with weight and bias for float elements (see layernorm_kernels.hpp).
#include "layernorm_kernels.hpp"

namespace plh {
PLH_LN_INSTANTIATE_AFFINE(float)
}  // namespace plh
