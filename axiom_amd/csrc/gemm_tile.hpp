// Shared by gemm.hip and the gemm_tile_*.hip translation units: the 16-bit matrix-core kernel of middle-sized products.
#pragma once
#include "gemm_skinny.hpp"

#include <algorithm>

namespace axhip {

// Kernel arguments of the tile and small-product kernels.  Kept within 96 bytes: a launch whose arguments are longer
// takes the host 3.3 us instead of 2.7 us, which is what a chain of short kernels is bound by.
struct TileArgs {
    const void *a, *b;
    void *c;
    const void *bias, *residual;
    int64_t sa, sb, sc;              // batch strides, elements
    int M, N, K, lda, ldb, ldc;      // b: [N, K] rows of ldb elements, or [K, N] (NN)
    int epilogue;
    int batch;                       // products of this launch
};
static_assert(sizeof(TileArgs) <= 96, "kernel arguments");

// Work-group -> (product, tile of C), -1 past the last: XCD x (work-groups x, x + 8, ...) owns a contiguous range of all the
// launch's tiles, product by product, so that a product's operands stay in one L2 and every XCD has the same number of tiles
// (dealt product by product, 12 tiles each went to 6 of the 8: 32 x (192 x 1536 x 2112) 75 us instead of 48).
// (An eighth of the grid is formed from the tiles, as tile_grid() does: gridDim would come with the runtime's own arguments, 256
// bytes behind the kernel's on each launch -- 64 x 1024 x 512 4.1 us a call instead of 3.8, fp32 48 x 384 x 384 4.0 instead of 3.6.)
__device__ __forceinline__ int tile_of_work_group(int tiles, int batch, int &product) {
    const int per_xcd = (tiles * batch + 7) / 8;
    const int t = (static_cast<int>(blockIdx.x) % 8) * per_xcd + static_cast<int>(blockIdx.x) / 8;
    product = 0;
    if (batch == 1) return t < tiles ? t : -1;
    if (t >= tiles * batch) return -1;
    product = t / tiles;
    return t - product * tiles;
}
// The grid for `products` of `tiles` each, and how many of them a launch of `threads` a work-group can hold (at least one: the
// caller has seen that one fits).
inline unsigned tile_grid(int64_t tiles, int64_t products) { return static_cast<unsigned>(8 * ((tiles * products + 7) / 8)); }
inline int64_t products_per_launch(int64_t tiles, int threads) {
    const int64_t blocks = std::min<int64_t>((int64_t(1) << 31) - 1, ((int64_t(1) << 32) - 1) / threads) - 7;
    return std::max<int64_t>(1, blocks / tiles);
}
// `launch(args, grid)` for the products of g, `es` bytes an element
template <class Args, class Launch> void launch_products(const Args &g, int64_t tiles, int threads, int es, Launch launch) {
    if (launch_fits(tiles * g.batch + 7, threads)) return launch(g, tile_grid(tiles, g.batch));
    const int64_t most = products_per_launch(tiles, threads);
    for (int64_t b0 = 0; b0 < g.batch; b0 += most) {
        Args part = g;
        part.a = static_cast<const char *>(g.a) + b0 * g.sa * es;
        part.b = static_cast<const char *>(g.b) + b0 * g.sb * es;
        part.c = static_cast<char *>(g.c) + b0 * g.sc * es;
        if (g.residual) part.residual = static_cast<const char *>(g.residual) + b0 * g.sc * es;
        part.batch = static_cast<int>(std::min<int64_t>(most, g.batch - b0));
        launch(part, tile_grid(tiles, part.batch));
    }
}

// The work-group tiles (M x N): every wavefront owns 16 MI x 64 of C for a share of each k-tile.
enum TileShape { TILE_256x128, TILE_192x128, TILE_128x128, TILE_64x128, TILE_SHAPES };
struct TileGeometry { int tm, tn, tk; };
constexpr TileGeometry TILE_GEOMETRY[TILE_SHAPES] = {{256, 128, 64}, {192, 128, 64}, {128, 128, 64}, {64, 128, 128}};

// Launches the kernel of `shape`; `aligned`: every row of a and b starts on a 16-byte boundary and K (and N where b is
// [K, N]) is a multiple of 8.  Defined in gemm_tile_nt.hip (b is [N, K]) and gemm_tile_nn.hip (b is [K, N]).
int launch_tile_nt(const TileArgs &g, bool bf16, int shape, bool aligned, hipStream_t s);
int launch_tile_nn(const TileArgs &g, bool bf16, int shape, bool aligned, hipStream_t s);

} // namespace axhip
