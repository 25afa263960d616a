// Split implicit-GEMM conv kernel instance (bf16 matrix cores, each f32
// operand as three bf16 terms); the kernel is in conv_mfma_tile.hpp.
#include "conv_mfma_tile.hpp"

namespace pdefa {
namespace k {

bool launch_conv_tiles_split(int tile, const ConvArgs& a, bool vec, dim3 grid, hipStream_t s) {
    if (!is_split_tile(tile)) return false;
    if (!vec || a.groups != 1) fail("split tiles take ungrouped convs with vector loads");
    launch_split_tile<128, 128, 64, 32>(a, grid, s);
    return true;
}

}  // namespace k
}  // namespace pdefa
