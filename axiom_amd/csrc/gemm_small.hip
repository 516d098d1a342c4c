// Products with few rows or few output tiles, 16-bit: see the kernel's comment.
#include "gemm_small.hpp"
#include "gemm_tile_device.hpp"

namespace axhip {
namespace {

// The piece of k in a wavefront's stage (rows of 128 bytes: 16 MI of A, then of B) -> MFMA fragments.
__device__ __forceinline__ int small_nn_xor(int k) { return 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1)); }
template <bool NN, int MI, int NJ>
__device__ __forceinline__ void small_read_fragments(uint4_t (&fa)[2][MI], uint4_t (&fb)[2][NJ], const unsigned char *st, int l16, int g4) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[h][i] = *reinterpret_cast<const uint4_t *>(st + (16 * i + l16) * 128 + (((4 * h + g4) ^ ((l16 >> 1) & 7)) * 16));
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (NN) {
                uint2_t part[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int k = 32 * h + 8 * g4 + 4 * q + (l16 >> 2);
                    part[q] = tile_read_tr(st + MI * 2048 + k * 128 + (((2 * j + ((l16 & 3) >> 1)) ^ small_nn_xor(k)) * 16) + (l16 & 1) * 8);
                }
                fb[h][j] = uint4_t{part[0].x, part[0].y, part[1].x, part[1].y};
            } else {
                fb[h][j] = *reinterpret_cast<const uint4_t *>(st + MI * 2048 + (16 * j + l16) * 128 + (((4 * h + g4) ^ ((l16 >> 1) & 7)) * 16));
            }
        }
    }
}
// (B fragment) x (A fragment)^T: a lane holds four consecutive columns of one row of C
template <bool BF16> __device__ __forceinline__ float4_t small_mfma(const uint4_t &fb, const uint4_t &fa, const float4_t &acc) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fb), __builtin_bit_cast(bf16x8_t, fa), acc, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, fb), __builtin_bit_cast(half8_t, fa), acc, 0, 0, 0);
}

// The W wavefronts' sums meet in LDS; bias, residual, activation, store.  Columns below n_low are another work-group's.
template <bool BF16, int MI, int NJ, int W>
__device__ __forceinline__ void small_finish(const TileArgs &g, const float4_t (&acc)[MI][NJ], int m0, int n0, int n_low, int64_t coff, unsigned char *small_lds) {
    constexpr int F = MI * NJ;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<float4_t *>(small_lds + ((wave * F + i * NJ + j) * 64 + lane) * 16) = acc[i][j];
    __syncthreads();
    for (int x = tid; x < F * 64; x += 64 * W) {
        const int f = x / 64, row = m0 + 16 * (f / NJ) + (x % 16), col = n0 + 16 * (f % NJ) + 4 * ((x % 64) / 16);
        float4_t v = *reinterpret_cast<const float4_t *>(small_lds + x * 16);
#pragma unroll
        for (int w = 1; w < W; ++w) v += *reinterpret_cast<const float4_t *>(small_lds + (w * F * 64 + x) * 16);
        const int first = max(0, n_low - col), valid = min(4, g.N - col); // the columns col + [first, valid) of C
        if (row >= g.M || first >= valid) continue;
        const int64_t at = coff + static_cast<int64_t>(row) * g.ldc + col;
        uint16_t *c = static_cast<uint16_t *>(g.c) + at;
        const uint16_t *bias = static_cast<const uint16_t *>(g.bias) + col, *res = static_cast<const uint16_t *>(g.residual) + at;
        float y[4] = {v[0], v[1], v[2], v[3]};
        auto widen = [](uint32_t h) { return BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h); };
        auto add4 = [&](const uint16_t *p) {
            if (valid - first == 4) {
                const uint2_t q = reinterpret_cast<const uint2_unaligned_t *>(p)->v;
                y[0] += widen(q.x & 0xFFFFu); y[1] += widen(q.x >> 16); y[2] += widen(q.y & 0xFFFFu); y[3] += widen(q.y >> 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e >= first && e < valid) y[e] += widen(p[e]);
            }
        };
        if (g.bias) add4(bias);
        if (g.residual) add4(res);
        gemm_epilogue16_all(g.epilogue, y);
        const uint32_t w0 = BF16 ? pack_bf16x2(y[0], y[1]) : pack_f16x2(y[0], y[1]), w1 = BF16 ? pack_bf16x2(y[2], y[3]) : pack_f16x2(y[2], y[3]);
        if (valid - first == 4) { // (any alignment)
            reinterpret_cast<uint2_unaligned_t *>(c)->v = uint2_t{w0, w1};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e >= first && e < valid) c[e] = static_cast<uint16_t>((e < 2 ? w0 : w1) >> (16 * (e % 2)));
        }
    }
}

// C = A B (b [N, K], or [K, N]: NN), bf16 / f16, any alignment: work-group tile 16 MI x 16 NJ, W wavefronts that split k
// between them (wavefront w takes the 64-element pieces w, w + W, ...) and meet in LDS once, at the end.
// What bounds products of this size is latency, of memory and of the instructions themselves.
//   * A ring of k-tiles shared by the work-group costs a barrier and an LDS round trip per k-tile (64 x 4096 x 4096 took
//     24 us on 64 x 128 tiles: 32 work-groups of 64 steps, whatever the caches held).  Here every wavefront has a stage of
//     LDS of its own and waits for nobody until the sums are added, and the tile is as narrow as it takes to give every
//     CU work: 9 us.  The price is that nothing is shared but through the caches.
//   * A piece travels through registers, the next one's loads in flight while one is multiplied, rather than through a
//     deeper ring filled by buffer_load ... lds (equal or slower at every size measured); the loads need no alignment
//     then.  Fragments loaded straight into registers, 64 bytes of each of 16 rows per instruction, came at a quarter of
//     the rate that whole 128-byte lines do.
//   * Nothing is unrolled over the pieces: what is not in a loop is fetched from memory once, and a product of this size
//     is over before a long kernel's instructions have arrived (four pieces in flight in an unrolled loop: 10 us for
//     50 x 9 x 17, against 3 us).
// The last chunk of a row is fetched as the 16 bytes that end with it and shifted into place.  Needs K >= 8 (NN: and
// N >= 8).
template <bool BF16, bool NN, int MI, int NJ, int W>
__global__ __launch_bounds__(64 * W) void gemm_small_kernel(const TileArgs g) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char small_lds[];
    constexpr int NL = 2 * (MI + NJ), NA = 2 * MI, STAGEB = NL * 1024;
    static_assert(!NN || NJ == 4, "NN pieces are 64 columns wide");
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int l16 = lane % 16, g4 = lane / 16;
    const int tiles_m = (g.M + 16 * MI - 1) / (16 * MI);
    int product;
    const int t = tile_of_work_group(tiles_m * ((g.N + 16 * NJ - 1) / (16 * NJ)), g.batch, product);
    if (t < 0) return;
    const int m0 = (t % tiles_m) * 16 * MI, n_low = (t / tiles_m) * 16 * NJ;
    // (NN: the last column tile is moved left to end with the rows; the columns it shares are its neighbour's to store)
    const int n0 = NN ? max(0, min(n_low, g.N - 16 * NJ)) : n_low;
    const int64_t bz = product;
    const char *A = reinterpret_cast<const char *>(static_cast<const uint16_t *>(g.a) + bz * g.sa + static_cast<int64_t>(m0) * g.lda);
    const char *B = reinterpret_cast<const char *>(static_cast<const uint16_t *>(g.b) + bz * g.sb + (NN ? static_cast<int64_t>(n0) : static_cast<int64_t>(n0) * g.ldb));
    const int rows_a = min(16 * MI, g.M - m0), rows_b = min(16 * NJ, g.N - n0);
    const int ld_r = lane >> 3;
    unsigned char *st = small_lds + wave * STAGEB;

    int src[NL];       // the chunk of its row that a lane's load n fetches: the one that belongs at position lane & 7
    uint32_t off[NL];  // and where the row starts (NN, b: where the chunk lies in its row)
#pragma unroll
    for (int n = 0; n < NL; ++n) {
        const int row = 8 * (n < NA ? n : n - NA) + ld_r;
        src[n] = (lane & 7) ^ (NN && n >= NA ? small_nn_xor(row) : ((row >> 1) & 7));
        if (n < NA) off[n] = static_cast<uint32_t>(min(row, rows_a - 1)) * g.lda * 2; // (rows past the end repeat the last one: they are not stored)
        else if (NN) off[n] = static_cast<uint32_t>(min(8 * src[n], g.N - n0 - 8)) * 2;
        else off[n] = static_cast<uint32_t>(min(row, rows_b - 1)) * g.ldb * 2;
    }
    uint4_t regs[NL];
    auto load = [&](int piece) { // (past the end of k: the row's end, or the last row, again)
#pragma unroll
        for (int n = 0; n < NL; ++n) {
            const uint32_t at = NN && n >= NA ? static_cast<uint32_t>(min(64 * piece + 8 * (n - NA) + ld_r, g.K - 1)) * g.ldb * 2
                                              : static_cast<uint32_t>(min(64 * piece + 8 * src[n], g.K - 8)) * 2;
            regs[n] = reinterpret_cast<const uint4_unaligned_t *>((n < NA ? A : B) + (off[n] + at))->v;
        }
    };
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int pieces = (g.K + 63) / 64;
    load(wave);
#pragma unroll 1
    for (int p = wave; p < pieces; p += W) {
        if (64 * (p + 1) > g.K || (NN && g.N < 16 * NJ)) {
#pragma unroll
            for (int n = 0; n < NL; ++n) {
                if (NN && n >= NA) {
                    regs[n] = tile_row_chunk_in_place(regs[n], 8 * src[n], g.N - n0);
                    if (64 * p + 8 * (n - NA) + ld_r >= g.K) regs[n] = uint4_t{0, 0, 0, 0};
                } else {
                    regs[n] = tile_row_chunk_in_place(regs[n], 64 * p + 8 * src[n], g.K);
                }
            }
        }
#pragma unroll
        for (int n = 0; n < NL; ++n) *reinterpret_cast<uint4_t *>(st + n * 1024 + lane * 16) = regs[n];
        if (p + W < pieces) load(p + W);
        wave_lds_fence();
        uint4_t fa[2][MI], fb[2][NJ];
        small_read_fragments<NN, MI, NJ>(fa, fb, st, l16, g4);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = small_mfma<BF16>(fb[h][j], fa[h][i], acc[i][j]);
        wave_lds_fence();
    }
    __syncthreads();
    small_finish<BF16, MI, NJ, W>(g, acc, m0, n0, n_low, bz * g.sc, small_lds);
}

template <bool BF16, bool NN, int MI, int NJ, int W> int launch_kernel(const TileArgs &g, hipStream_t s) {
    constexpr int stages = W * (MI + NJ) * 2048, sums = W * MI * NJ * 1024, lds = stages > sums ? stages : sums;
    const auto kernel = gemm_small_kernel<BF16, NN, MI, NJ, W>;
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    AXHIP_CHECK_HIP(configured);
    const int64_t tiles = static_cast<int64_t>((g.M + 16 * MI - 1) / (16 * MI)) * ((g.N + 16 * NJ - 1) / (16 * NJ));
    AXHIP_REQUIRE(launch_fits(tiles + 7, 64 * W), AXHIP_ERR_UNSUPPORTED, "axhip_gemm: too many tiles");
    launch_products(g, tiles, 64 * W, 2, [&](const TileArgs &part, unsigned grid) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * W), lds, s, part); });
    return AXHIP_OK;
}
template <bool BF16, bool NN, int MI, int NJ> int launch_waves(const TileArgs &g, int waves, hipStream_t s) {
    return waves == 8 ? launch_kernel<BF16, NN, MI, NJ, 8>(g, s) : launch_kernel<BF16, NN, MI, NJ, 4>(g, s);
}
template <bool BF16> int launch_shape(const TileArgs &g, bool nn, int shape, int waves, hipStream_t s) {
    if (nn) switch (shape) {
        case SMALL_16x64: return launch_waves<BF16, true, 1, 4>(g, waves, s);
        case SMALL_32x64: return launch_waves<BF16, true, 2, 4>(g, waves, s);
        default: return launch_waves<BF16, true, 4, 4>(g, waves, s);
        }
    switch (shape) {
    case SMALL_16x16: return launch_waves<BF16, false, 1, 1>(g, waves, s);
    case SMALL_32x16: return launch_waves<BF16, false, 2, 1>(g, waves, s);
    case SMALL_32x32: return launch_waves<BF16, false, 2, 2>(g, waves, s);
    case SMALL_32x64: return launch_waves<BF16, false, 2, 4>(g, waves, s);
    default: return launch_waves<BF16, false, 4, 4>(g, waves, s);
    }
}
} // namespace

int launch_small(const TileArgs &g, bool bf16, bool nn, int shape, int waves, hipStream_t s) {
    return bf16 ? launch_shape<true>(g, nn, shape, waves, s) : launch_shape<false>(g, nn, shape, waves, s);
}
} // namespace axhip
