// Loads and LDS reads shared by the 16-bit product kernels (gemm_tile_kernel.hpp, gemm_small.hip).
#pragma once
#include "common.hpp"

namespace axhip {
namespace {

typedef int int4_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane from a buffer straight into LDS: lane i's data lands at lds_base + 16 i; lanes whose voffset lies
// beyond the descriptor's extent write zeros.
__device__ __forceinline__ void tile_load_to_lds(const int4_t &rsrc, uint32_t lds_base_uniform, int voffset, int soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_base_uniform), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}
__device__ __forceinline__ int4_t tile_rsrc(const void *base, int bytes) {
    const uint64_t pa = reinterpret_cast<uint64_t>(base);
    return int4_t{static_cast<int>(static_cast<uint32_t>(pa)), static_cast<int>(static_cast<uint32_t>(pa >> 32) & 0xFFFFu), bytes, 0x00020000};
}
// 4 consecutive k of one column out of [k][n] rows in LDS: within a group of 16 lanes, lane i receives element i & 3 of
// the 8-byte pieces addressed by lanes (i >> 2) + 4 j, j = 0..3
__device__ __forceinline__ uint2_t tile_read_tr(const unsigned char *p) {
    typedef short short4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4_t lds_short4_t;
    return __builtin_bit_cast(uint2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)(p)));
}

// v: the 16 bytes of a row of n >= 8 16-bit elements at element min(at, n - 8).  What is left of [at, at + 8), in place,
// zeros behind it.
__device__ __forceinline__ uint4_t tile_row_chunk_in_place(uint4_t v, int at, int n) {
    const int drop = at - min(at, n - 8); // elements in front of the chunk
    if (drop == 0) return v;
    if (drop >= 8) return uint4_t{0, 0, 0, 0};
    return __builtin_bit_cast(uint4_t, __builtin_bit_cast(unsigned __int128, v) >> (16 * drop));
}

// LDS that the lanes of ONE wavefront exchange: what was written before is what is read behind (the hardware keeps the
// order, the compiler has to be told: it sees one lane's addresses only).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

} // namespace
} // namespace axhip
