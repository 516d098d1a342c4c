// Shared by gemm.hip and the gemm_tile_*.hip translation units: the 16-bit matrix-core kernel of middle-sized products.
#pragma once
#include "gemm_skinny.hpp"

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
};
static_assert(sizeof(TileArgs) <= 96, "kernel arguments");

// The work-group tiles (M x N): every wavefront owns 16 MI x 64 of C for a share of each k-tile.
enum TileShape { TILE_256x128, TILE_192x128, TILE_128x128, TILE_64x128, TILE_SHAPES };
struct TileGeometry { int tm, tn, tk; };
constexpr TileGeometry TILE_GEOMETRY[TILE_SHAPES] = {{256, 128, 64}, {192, 128, 64}, {128, 128, 64}, {64, 128, 128}};

// Launches the kernel of `shape`; `aligned`: every row of a and b starts on a 16-byte boundary and K (and N where b is
// [K, N]) is a multiple of 8.  Defined in gemm_tile_nt.hip (b is [N, K]) and gemm_tile_nn.hip (b is [K, N]).
int launch_tile_nt(const TileArgs &g, bool bf16, int shape, bool aligned, int batch, hipStream_t s);
int launch_tile_nn(const TileArgs &g, bool bf16, int shape, bool aligned, int batch, hipStream_t s);

} // namespace axhip
