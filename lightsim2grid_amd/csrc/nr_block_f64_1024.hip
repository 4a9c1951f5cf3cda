#include "nr_block_kernel.hpp"

namespace pfgpu_block {
const void* kernel_f64_1024(int G, bool lean) { return lean ? variant<double, 1024, true>(G) : variant<double, 1024, false>(G); }
}  // namespace pfgpu_block
