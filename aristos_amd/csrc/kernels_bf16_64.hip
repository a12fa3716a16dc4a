// The persistent kernels of 33 to 128 experts for Element = bf16_t (see kernels_impl.hpp).
#include "kernels_impl.hpp"

namespace kleos_amd {
KLEOS_INSTANTIATE_PLANS(bf16_t, 4, 8)
}  // namespace kleos_amd
