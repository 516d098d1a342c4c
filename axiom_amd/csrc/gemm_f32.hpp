// Shared by gemm.hip and gemm_f32.hip: fp32 products without shared LDS tiles.
#pragma once
#include "gemm_tile.hpp"

namespace axhip {

// work-group tiles (M x N) and the k each of its eight wavefronts takes at a time
enum F32Shape { F32_16x16, F32_16x32, F32_16x64, F32_32x32, F32_32x64, F32_64x64, F32_32x64_PARTS, F32_SHAPES };
struct F32Geometry { int tm, tn, tk; };
constexpr F32Geometry F32_GEOMETRY[F32_SHAPES] = {{16, 16, 64}, {16, 32, 64}, {16, 64, 32}, {32, 32, 32}, {32, 64, 32}, {64, 64, 32}, {32, 64, 32}};

// a [M, K]; b [N, K], or [K, N] (nn).  K >= 1, N >= 4; no alignment beyond the elements'.
int launch_f32_direct(const TileArgs &g, bool nn, int shape, hipStream_t s);

} // namespace axhip
