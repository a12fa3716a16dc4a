// The persistent kernels of more than 128 experts for Element = bf16_t (see kernels_impl.hpp).
#include "kernels_impl.hpp"

namespace kleos_amd {
KLEOS_INSTANTIATE_PLANS(bf16_t, 16, 0)
}  // namespace kleos_amd
