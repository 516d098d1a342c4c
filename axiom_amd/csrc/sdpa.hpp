// What the attention kernels share: their arguments, the arithmetic of the softmax, the launches of sdpa_direct.hip.
#pragma once

#include "common.hpp"

namespace axhip {

struct SdpaArgs {
    const void *q, *k, *v;
    void *o;
    const uint8_t *mask;
    int B, H, Sq, Skv, D;
    float scale;       // softmax scale
    float scale_log2e; // scale * log2(e)
    int causal;
    int nqb; // query blocks per (batch, head)
    int dtype;
    int64_t qs[3], ks[3], vs[3], os[3], ms[2];
    // key split of sdpa_direct16_kernel and sdpa_mfma_kernel (decoding: few query rows, few heads, a long key sequence): `ksplit` work-groups
    // per (batch, head) take `kchunk` keys each and leave normalised fp32 partial outputs and the base-2 logarithm of
    // their softmax denominators (reference maximum included) for sdpa_merge_kernel
    int ksplit, kchunk;
    float *opart, *lse;
    int pairs; // sdpa_mfma_pingpong_kernel, causal: query blocks i and n - 1 - i go to one work-group
    // an explicit mask as sdpa_pack_mask_kernel left it: the plane of (b, h) is b * mask_plane[0] + h * mask_plane[1]
    const uint32_t *mask_bits;
    const int2_t *mask_range;
    int mask_tiles, mask_plane[2];
};

constexpr float NEG_INF_F = -__builtin_huge_valf();

// Growth of the running row maximum (log2 domain) that is tolerated before the
// accumulators are rescaled: exponentials stay below 2^8, far inside fp32/bf16/f16 range.
constexpr float RESCALE_THRESHOLD = 8.0f;

template <bool BF16> __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    if constexpr (BF16) {
        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
        typedef float float2_t __attribute__((ext_vector_type(2)));
        float2_t f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t)); // v_cvt_pk_bf16_f32, RNE
    } else {
        return pack_f16x2(lo, hi); // v_cvt_pk_f16_f32, RNE
    }
}

// acc + lo + hi of a packed pair, one v_dot2c instruction
template <bool BF16> __device__ __forceinline__ float add_pair(uint32_t packed, float acc) {
    if constexpr (BF16) {
        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, packed), __builtin_bit_cast(bf16x2_t, 0x3F803F80u), acc, false);
    } else {
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, packed), __builtin_bit_cast(half2_t, 0x3C003C00u), acc, false);
    }
}

// sdpa_direct.hip: a few query rows against many keys, short fp32 sequences
constexpr int DIRECT_WAVES = 8;      // per work-group
constexpr int DIRECT_ROWS = 8;       // query rows of the 16-bit kernel, at most
constexpr int DIRECT_KEYS = 32;      // keys of one step of a wave; a.kchunk is a multiple of it
int launch_sdpa_direct16(const SdpaArgs &a, bool bf16, hipStream_t s);
int launch_sdpa_direct_f32(const SdpaArgs &a, hipStream_t s);
// out = the `a.ksplit` partial results in a.opart / a.lse of every query row, weighed together; `D` columns a partial row
void launch_sdpa_merge(const SdpaArgs &a, bool bf16, int D, hipStream_t s);

} // namespace axhip
