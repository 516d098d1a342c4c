// fp32 products on the bf16 matrix instruction, shared by gemm.hip and gemm_f32.hip.
//
// An fp32 number is the sum of three bf16 ones: the nearest, the nearest to what is left, and the rest, which has at most
// eight significant bits and is one exactly.  Of the nine products of two such sums, six carry all that fp32 holds; the three
// left out are below 2^-26 of a b (each part is at most 2^-9 of the one before).  v_mfma_f32_16x16x32_bf16 multiplies bf16
// exactly and sums in fp32, at 16 times the rate of the fp32 matrix instruction, so six of them do in 96 cycles what that
// does in 256.  A chain of six starts at zero for every 32 k and is added to the sum behind it: K / 32 fp32 additions in
// place of the K / 4 of v_mfma_f32_16x16x4_f32, which is why the results come out closer to the exact ones than with fp32
// products: 2048^3 1.6e-7 off against 1.8e-7, 333 x 1280 x 1280 0.9e-7 against 2.3e-7 (one sum through all MFMAs instead: 2.4 to 4.5 times
// as far as these).
//
// Range: operands are multiplied by 2^16 before they are split.  Without that the last part of a number below 2^-110 would
// lie among bf16's denormals, which are kept but coarser; with it every fp32 number down to the smallest denormal has its
// three parts.  What is too large then (operands from 2^111, sums from 2^96 in size), infinities and NaN make the
// result an infinity or a NaN, never a finite number: the tile is computed again with fp32 products.
#pragma once
#include "common.hpp"

namespace axhip {
namespace {

constexpr float SPLIT_SCALE = 65536.0f;                                   // of each operand
constexpr float SPLIT_UNSCALE = 1.0f / (SPLIT_SCALE * SPLIT_SCALE);       // of the sums

// Two numbers -> their parts, packed.  (The first part is cut off rather than rounded, a perm and two ANDs for a conversion at
// half rate and two unpackings: what is left then has the number's sign, and the last part, which meets it in the products
// that are left out, both signs, so those still add up to nothing.)
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&part)[3]) {
    a *= SPLIT_SCALE;
    b *= SPLIT_SCALE;
    const uint32_t wa = __builtin_bit_cast(uint32_t, a), wb = __builtin_bit_cast(uint32_t, b);
    part[0] = __builtin_amdgcn_perm(wb, wa, 0x07060302u);
    a -= __builtin_bit_cast(float, wa & 0xFFFF0000u);
    b -= __builtin_bit_cast(float, wb & 0xFFFF0000u);
    part[1] = pack_bf16x2(a, b);
    a -= __builtin_bit_cast(float, part[1] << 16);
    b -= __builtin_bit_cast(float, part[1] & 0xFFFF0000u);
    part[2] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}

struct SplitFragment { uint4_t part[3]; };
__device__ __forceinline__ SplitFragment split_fragment(const float (&x)[8]) { // eight k of one row
    SplitFragment f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t w[3];
        split_pair(x[2 * e], x[2 * e + 1], w);
#pragma unroll
        for (int q = 0; q < 3; ++q) f.part[q][e] = w[q];
    }
    return f;
}

typedef float split_acc_t __attribute__((ext_vector_type(4)));
// sum + b-part x (a-part)^T
__device__ __forceinline__ split_acc_t split_mfma(const uint4_t &b, const uint4_t &a, const split_acc_t &sum) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), sum, 0, 0, 0);
}
// The products that count, smallest first: part SPLIT_A[n] of a with part SPLIT_B[n] of b
constexpr int SPLIT_PRODUCTS = 6;
constexpr int SPLIT_A[SPLIT_PRODUCTS] = {0, 1, 2, 0, 1, 0}, SPLIT_B[SPLIT_PRODUCTS] = {2, 1, 0, 1, 0, 0};

// Whether any of the work-group's lanes says so; `flags`: a word of LDS for each of its W wavefronts, used for nothing else.
// (__syncthreads_or() asks the runtime for the work-group's size, 256 bytes of arguments behind the kernel's own.)
template <int W> __device__ __forceinline__ bool work_group_any(bool mine, uint32_t *flags) {
    const bool wave_any = __builtin_amdgcn_ballot_w64(mine) != 0;
    if (threadIdx.x % WAVE == 0) flags[threadIdx.x / WAVE] = wave_any;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) any |= flags[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

__device__ __forceinline__ bool split_failed(float sum) { return !(__builtin_fabsf(sum) < __builtin_inff()); }

} // namespace
} // namespace axhip
