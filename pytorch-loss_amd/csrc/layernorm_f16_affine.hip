// layer norm kernels with weight and bias for f16 elements (see layernorm_kernels.hpp).
#include "layernorm_kernels.hpp"

namespace plh {
PLH_LN_INSTANTIATE_AFFINE(f16)
}  // namespace plh
