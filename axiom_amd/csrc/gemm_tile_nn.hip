// matmul(a, b) of plain row-major matrices: see gemm_tile_kernel.hpp.
#include "gemm_tile_kernel.hpp"

namespace axhip {
template <bool BF16> static int launch_nn(const TileArgs &g, int shape, bool aligned, hipStream_t s) {
    if (!aligned) return launch_tile_kernel<BF16, true, false, 4, 2, 2, 2, 64, 2>(g, s);
    switch (shape) {
    case TILE_256x128: return launch_tile_kernel<BF16, true, true, 8, 2, 2, 2, 64, 3>(g, s);
    case TILE_192x128: return launch_tile_kernel<BF16, true, true, 6, 2, 2, 2, 64, 3>(g, s);
    case TILE_128x128: return launch_tile_kernel<BF16, true, true, 4, 2, 2, 2, 64, 4>(g, s);
    default: return launch_tile_kernel<BF16, true, true, 4, 1, 2, 4, 128, 3>(g, s);
    }
}
int launch_tile_nn(const TileArgs &g, bool bf16, int shape, bool aligned, hipStream_t s) {
    return bf16 ? launch_nn<true>(g, shape, aligned, s) : launch_nn<false>(g, shape, aligned, s);
}
} // namespace axhip
