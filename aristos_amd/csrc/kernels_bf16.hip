// The kernels of the MoE layer forward for Element = bf16_t (see kernels_impl.hpp); the persistent kernels of more than 32
// experts are in kernels_bf16_64.hip and kernels_bf16_512.hip.
#include "kernels_impl.hpp"

namespace kleos_amd {
KLEOS_EXTERN_PLANS(bf16_t, 4, 8)
KLEOS_EXTERN_PLANS(bf16_t, 16, 0)
KLEOS_INSTANTIATE_ELEMENT(bf16_t)
}  // namespace kleos_amd
