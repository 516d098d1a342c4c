// fp32 products on the bf16 matrix instruction, shared by gemm.hip and gemm_f32.hip.
//
// An fp32 number is the sum of three bf16 ones: its first eight bits, the nearest to what is left, and the rest, which has at
// most eight significant bits and is one exactly (splitting a factor into parts whose products are exact: Dekker 1971).  Of a in
// [1, 2) the second part is at most 2^-7, the third 2^-16, so of the nine products of two such sums all but the last, which is
// at most 2^-32 of a b, are taken.  (Six of them, without the second by the third parts, which reach 2^-22 of a b, left a single
// product up to 2.9 ulp off.)
// v_mfma_f32_16x16x32_bf16 multiplies bf16 exactly and sums in fp32, at 16 times the rate of the fp32 matrix instruction, so
// eight of them do in 128 cycles what that does in 256.  But it cuts off what it adds at 2^-24 of its largest term before it rounds (a
// product of 1 .. 2 and a sum 2^-7 as large: up to 1 ulp off, a quarter of them not the nearest).  So the products of first parts,
// of 16 bits each, whose sums of like size are exact, have a chain of their own; a second chain takes the other seven, at most 2^-6 as
// large, and the two are added as fp32 numbers.  A single product comes out within 0.5 + 7 / 128 ulp (0.514 measured, 0.4 %
// of them not the nearest).  Both chains start at zero for every 32 k and are added to the sum behind them: K / 32 fp32 additions in
// place of the K / 4 of v_mfma_f32_16x16x4_f32, for which long sums are closer to the exact ones than with fp32 products: 1024^3 0.9e-7 off against
// 1.5e-7, 2048^3 1.5e-7 against 1.8e-7, 333 x 1280 x 1280 0.8e-7 against 2.3e-7.
//
// Range: operands are multiplied by 2^16 before they are split.  Without that the last part of a number below 2^-110 would
// lie among bf16's denormals, which are kept but coarser; with it every fp32 number down to the smallest denormal has its
// three parts (those of the smallest are denormals, the matrix instruction takes them as they are).  What is too large then
// (operands from 2^112, sums from 2^96 in size), infinities and NaN make the result an infinity or a NaN, never a finite
// number: the tile is computed again with fp32 products.
#pragma once
#include "common.hpp"

namespace axhip {
namespace {

constexpr float SPLIT_SCALE = 65536.0f;                                   // of each operand
constexpr float SPLIT_UNSCALE = 1.0f / (SPLIT_SCALE * SPLIT_SCALE);       // of the sums

// Two numbers -> their parts, packed.  (The first part is cut off rather than rounded: a perm and two ANDs for a conversion at
// half rate and two unpackings.)
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
// The products that count: that of the first parts, which is summed by itself, then the others, smallest first (and those of last
// parts before the rest, so that their registers are free early): part SPLIT_A[n] of a with part SPLIT_B[n] of b
constexpr int SPLIT_PRODUCTS = 8;
constexpr int SPLIT_A[SPLIT_PRODUCTS] = {0, 1, 2, 0, 2, 1, 0, 1}, SPLIT_B[SPLIT_PRODUCTS] = {0, 2, 1, 2, 0, 1, 1, 0};

// The lane's number, made anew: where the k loop leaves no register for what is needed behind it.  (mbcnt as a builtin, or what is made of
// threadIdx, would be computed once and kept.)
__device__ __forceinline__ int lane_again() {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}

// Whether any of the work-group's lanes says so; `flags`: a word of LDS for each of its W wavefronts, used for nothing else.
// (__syncthreads_or() asks the runtime for the work-group's size, 256 bytes of arguments behind the kernel's own.)
template <int W> __device__ __forceinline__ bool work_group_any(bool mine, uint32_t *flags, int wavefront, int lane) {
    const bool wave_any = __builtin_amdgcn_ballot_w64(mine) != 0;
    if (lane == 0) flags[wavefront] = wave_any;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) any |= flags[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

__device__ __forceinline__ bool split_failed(float sum) { return !(__builtin_fabsf(sum) < __builtin_inff()); }

} // namespace
} // namespace axhip
