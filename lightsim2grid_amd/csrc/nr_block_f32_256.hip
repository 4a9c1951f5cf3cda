#include "nr_block_kernel.hpp"

namespace pfgpu_block {
const void* kernel_f32_256(int G, bool lean) { return lean ? variant<float, 256, true>(G) : variant<float, 256, false>(G); }
}  // namespace pfgpu_block
