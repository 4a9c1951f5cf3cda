#include "nr_block_kernel.hpp"

namespace pfgpu_block {
const void* kernel_f32_1024(int G, bool lean) { return lean ? variant<float, 1024, true>(G) : variant<float, 1024, false>(G); }
}  // namespace pfgpu_block
