#include "nr_block_kernel.hpp"

namespace pfgpu_block {
const void* kernel_f64_256(int G, bool lean) { return lean ? variant<double, 256, true>(G) : variant<double, 256, false>(G); }
}  // namespace pfgpu_block
