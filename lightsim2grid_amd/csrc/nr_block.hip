// Launches of the block-plan kernel: its variants are compiled in nr_block_*.hip.
#include "nr_block.hpp"

#include "engine.hpp"

namespace pfgpu_block {

const void* kernel_f32_1024(int G, bool lean);
const void* kernel_f32_256(int G, bool lean);
const void* kernel_f64_1024(int G, bool lean);
const void* kernel_f64_256(int G, bool lean);

const void* kernel(int fsize, int G, int NT, bool lean) {
    if (fsize == 4) return NT == 1024 ? kernel_f32_1024(G, lean) : kernel_f32_256(G, lean);
    return NT == 1024 ? kernel_f64_1024(G, lean) : kernel_f64_256(G, lean);
}

void launch(const BArgs& a, int fsize, int G, int NT, bool lean, int nblocks, size_t lds, hipStream_t stream) {
    void* args[] = {const_cast<BArgs*>(&a)};
    HIP_OK(hipLaunchKernel(kernel(fsize, G, NT, lean), dim3(nblocks), dim3(NT), args, lds, stream));
}

}  // namespace pfgpu_block
