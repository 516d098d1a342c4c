// Shared by gemm.hip and gemm_small.hip: products with few rows or few output tiles, 16-bit.
#pragma once
#include "gemm_tile.hpp"

namespace axhip {

// work-group tiles (M x N); NN products (b is [K, N]) take the 64 columns wide ones, the others all but 16 x 64
enum SmallShape { SMALL_16x16, SMALL_32x16, SMALL_32x32, SMALL_16x64, SMALL_32x64, SMALL_64x64, SMALL_SHAPES };
struct SmallGeometry { int tm, tn; };
constexpr SmallGeometry SMALL_GEOMETRY[SMALL_SHAPES] = {{16, 16}, {32, 16}, {32, 32}, {16, 64}, {32, 64}, {64, 64}};

// `waves`: 4 or 8 wavefronts share k.  K >= 8 and, NN, N >= 8; no alignment beyond the elements'.
int launch_small(const TileArgs &g, bool bf16, bool nn, int shape, int waves, hipStream_t s);

} // namespace axhip
