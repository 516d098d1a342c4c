// fp32 products without shared LDS tiles: see the kernel's comment.
#include "common.hpp"
#include "gemm_f32.hpp"
#include "gemm_f32_split.hpp"
#include "gemm_tile_device.hpp"

namespace axhip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int N> struct __attribute__((packed, aligned(4))) Floats { float v[N]; };

constexpr int F32_WAVES = 8;

template <bool NN, bool SPLIT, int MI, int NJ, int P> constexpr int direct_lds_bytes() { // the stages or the sums (SPLIT: and a flag of each wavefront)
    const int stages = F32_WAVES * P * 2 * (MI + (NN ? 0 : NJ)) * 1024, sum = F32_WAVES * MI * NJ * 1024;
    return (stages > sum ? stages : sum) + (SPLIT ? 64 : 0);
}

// C = A B (b [N, K], or [K, N]: NN) on v_mfma_f32_16x16x4_f32: fp32 products and sums.  Work-group tile 16 MI x 16 NJ;
// eight wavefronts take pieces of 32 P elements of k in turn and add their sums through LDS at the end; until then no
// wavefront waits for another.
// The fp32 matrix rate is a sixteenth of the 16-bit one, so an operand that comes from the caches for every tile costs
// little next to the MFMAs it feeds.  Rows along k (a, and b as [N, K]) pass through a stage of LDS that is the
// wavefront's own, so that they are loaded in whole 128-byte lines (as fragments, 16 bytes of each of 16 rows side by
// side, they took four times the address cycles: 1024^3 28.5 us); b as [K, N] needs no stage and no transpose: which
// column a lane contributes to which MFMA is free, so lane (l16, g) loads the NJ columns NJ l16 .. of rows 4 g .. 4 g + 3.
// Bound by the matrix pipe at 64 x 64 and by latency below, where narrower tiles put more CUs to work.
// SPLIT: by products of bf16 parts (gemm_f32_split.hpp), each wavefront splitting what it multiplies.  That pays at 32 x 64, where
// eight fragments' splitting, 1250 cycles, and 1024 of MFMAs stand for 2048 of fp32 MFMAs (333 x 1280 x 1280 18.1 -> 15.2 us), once there
// is k enough for its longer end (32 x (64 x 240 x 145) 6.5 us with fp32 products, 6.95 with parts); 32 x 32 and below have no more
// MFMAs than splitting to do (64 x 1280 x 5120 28.2 and 28.1, 512^3 6.0 and 6.6, with six products), and the fragments of
// 64 x 64 do not fit the registers.
template <bool NN, bool SPLIT, int MI, int NJ, int P>
__global__ __launch_bounds__(64 * F32_WAVES, 2) void gemm_f32_direct_kernel(const TileArgs g) {
    extern __shared__ __attribute__((aligned(1024))) float sums[];
    constexpr int W = F32_WAVES, TM = 16 * MI, TN = 16 * NJ, KP = 32 * P, U = 2 * P;
    constexpr int NA = 2 * MI, NS = NA + (NN ? 0 : 2 * NJ); // staged loads of 8 rows x 128 bytes per 32 k
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, l16 = lane % 16, g4 = lane / 16;
    const int tiles_m = (g.M + TM - 1) / TM;
    int product;
    const int t = tile_of_work_group(tiles_m * ((g.N + TN - 1) / TN), g.batch, product);
    if (t < 0) return;
    const int m0 = (t % tiles_m) * TM, n0 = (t / tiles_m) * TN;
    const int64_t bz = product;
    const float *A = static_cast<const float *>(g.a) + bz * g.sa, *B = static_cast<const float *>(g.b) + bz * g.sb;

    // rows and columns past the end repeat the last ones: they are not stored
    const float *row[NS], *cols = nullptr; // this lane's four k of a staged row; its columns of b
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        const int r = 8 * (n < NA ? n : n - NA) + lane / 8, chunk = (lane & 7) ^ ((r >> 1) & 7); // (the chunk that belongs at position lane & 7)
        row[n] = (n < NA ? A + static_cast<int64_t>(min(m0 + r, g.M - 1)) * g.lda : B + static_cast<int64_t>(min(n0 + r, g.N - 1)) * g.ldb) + 4 * chunk;
    }
    if constexpr (NN) cols = B + static_cast<int64_t>(4 * g4) * g.ldb + min(n0 + NJ * l16, g.N - NJ);

    unsigned char *stage = reinterpret_cast<unsigned char *>(sums) + wave * P * NS * 1024;
    f32x4_t regs[P][NS];
    float fb[NN ? U : 1][NJ][4];
    auto load = [&](int k0) { // a whole piece
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                const Floats<4> v = *reinterpret_cast<const Floats<4> *>(row[n] + k0 + 32 * p);
                regs[p][n] = f32x4_t{v.v[0], v.v[1], v.v[2], v.v[3]};
            }
        if constexpr (NN) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const Floats<NJ> v = *reinterpret_cast<const Floats<NJ> *>(cols + static_cast<int64_t>(k0 + 16 * u + c) * g.ldb);
#pragma unroll
                    for (int j = 0; j < NJ; ++j) fb[u][j][c] = v.v[j];
                }
        }
    };
    auto load_last = [&](int k0) { // what is left of k, zeros behind it
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                const int r = 8 * (n < NA ? n : n - NA) + lane / 8, at = k0 + 32 * p + 4 * ((lane & 7) ^ ((r >> 1) & 7));
#pragma unroll
                for (int c = 0; c < 4; ++c) regs[p][n][c] = at + c < g.K ? row[n][k0 + 32 * p + c] : 0.0f;
            }
        if constexpr (NN) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int at = k0 + 16 * u + c;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) fb[u][j][c] = at + 4 * g4 < g.K ? cols[static_cast<int64_t>(at) * g.ldb + j] : 0.0f;
                }
        }
    };

    f32x4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto to_stage = [&] {
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int n = 0; n < NS; ++n) *reinterpret_cast<f32x4_t *>(stage + (p * NS + n) * 1024 + lane * 16) = regs[p][n];
    };
    // (b fragment) x (a fragment)^T: a lane holds row l16 of tile i, and of the columns what the epilogue says
    auto multiply = [&](const float (&xb)[NN ? U : 1][NJ][4]) {
        wave_lds_fence();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            auto fragment = [&](int first, int tile) { // k = 16 u + 4 g4 .. + 3 of row l16 of the tile
                return *reinterpret_cast<const f32x4_t *>(stage + ((u / 2) * NS + first) * 1024 + (16 * tile + l16) * 128 + (((4 * (u % 2) + g4) ^ ((l16 >> 1) & 7)) * 16));
            };
            f32x4_t fa[MI], fn[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[i] = fragment(0, i);
            if constexpr (!NN) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) fn[j] = fragment(NA, j);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(NN ? xb[NN ? u : 0][j][c] : fn[j][c], fa[i][c], acc[i][j], 0, 0, 0);
        }
        wave_lds_fence();
    };

    auto multiply_parts = [&](const float (&xb)[NN ? U : 1][NJ][4]) {
        wave_lds_fence();
#pragma unroll
        for (int p = 0; p < P; ++p) {
            auto whole_fragment = [&](int first, int tile) __attribute__((always_inline)) { // k = 32 p + 4 g4 .. + 3 and, 16 on, four more
                float x[8];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const f32x4_t v = *reinterpret_cast<const f32x4_t *>(stage + (p * NS + first) * 1024 + (16 * tile + l16) * 128 + (((4 * u + g4) ^ ((l16 >> 1) & 7)) * 16));
#pragma unroll
                    for (int c = 0; c < 4; ++c) x[4 * u + c] = v[c];
                }
                return split_fragment(x);
            };
            SplitFragment sb[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if constexpr (NN) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = xb[2 * p + e / 4][j][e % 4];
                    sb[j] = split_fragment(x);
                } else {
                    sb[j] = whole_fragment(NA, j);
                }
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const SplitFragment sa = whole_fragment(0, i);
                const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                f32x4_t first[NJ], rest[NJ];
#pragma unroll
                for (int n = 0; n < SPLIT_PRODUCTS; ++n)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        if (n == 0) first[j] = split_mfma(sb[j].part[SPLIT_B[n]], sa.part[SPLIT_A[n]], zero);
                        else rest[j] = split_mfma(sb[j].part[SPLIT_B[n]], sa.part[SPLIT_A[n]], n == 1 ? zero : rest[j]);
                    }
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] += first[j] + rest[j];
            }
        }
        wave_lds_fence();
    };

    const int whole = g.K / KP * KP;
    int k = wave * KP;
    if (k < whole) load(k);
#pragma unroll 1
    while (k < whole) {
        float xb[NN ? U : 1][NJ][4];
        if constexpr (NN) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int c = 0; c < 4; ++c) xb[u][j][c] = fb[u][j][c];
        }
        to_stage();
        k += W * KP;
        if (k < whole) load(k);
        if constexpr (SPLIT) multiply_parts(xb);
        else multiply(xb);
    }
    if (whole < g.K && k == whole) { // this wavefront's turn
        load_last(k);
        to_stage();
        if constexpr (SPLIT) multiply_parts(fb);
        else multiply(fb);
    }
    constexpr int F = MI * NJ;
    auto total = [&](int x) { // this lane's four columns
        f32x4_t v = *reinterpret_cast<const f32x4_t *>(&sums[x * 4]);
#pragma unroll
        for (int w = 1; w < W; ++w) v += *reinterpret_cast<const f32x4_t *>(&sums[(w * F * 64 + x) * 4]);
        return v;
    };
    float scale = SPLIT_UNSCALE;
    for (;;) {
        __syncthreads(); // the stages become the sums

        // sums[wave][f][lane], four columns each: NN f = (i, e) columns NJ (4 g4 + e) + 0 .. (fewer than four tiles: the
        // columns of several e side by side); else f = (i, j) columns 16 j + 4 g4 + 0 .. 3
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int f = 0; f < NJ; ++f) {
                f32x4_t v;
                if constexpr (NN) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = acc[i][(4 * f + x) % NJ][(4 * f + x) / NJ];
                } else {
                    v = acc[i][f];
                }
                *reinterpret_cast<f32x4_t *>(&sums[((wave * F + i * NJ + f) * 64 + lane) * 4]) = v;
            }
        __syncthreads();
        if (!SPLIT || scale == 1.0f) break;
        bool failed = false;
        for (int x = tid; x < F * 64; x += 64 * W) {
            const f32x4_t v = total(x);
#pragma unroll
            for (int e = 0; e < 4; ++e) failed = failed || split_failed(v[e]);
        }
        if (!work_group_any<W>(failed, reinterpret_cast<uint32_t *>(sums) + direct_lds_bytes<NN, SPLIT, MI, NJ, P>() / 4 - 16, wave, lane)) break;
        scale = 1.0f; // again, with fp32 products
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int again = wave * KP; again < g.K; again += W * KP) {
            load_last(again);
            to_stage();
            multiply(fb);
        }
    }
    float *C = static_cast<float *>(g.c) + bz * g.sc;
    const float *bias = static_cast<const float *>(g.bias), *res = g.residual ? static_cast<const float *>(g.residual) + bz * g.sc : nullptr;
    for (int x = tid; x < F * 64; x += 64 * W) {
        const int f = x / 64 % NJ, m = m0 + 16 * (x / 64 / NJ) + x % 16, xg = x % 64 / 16;
        if (m >= g.M) continue;
        f32x4_t v = total(x);
        if constexpr (SPLIT) v *= scale;
        // columns col .. col + 3.  (NN: a lane whose columns were moved left to end with the rows owns those at and
        // behind the place it was moved from)
        const int col = n0 + (NN ? 4 * NJ * xg + 4 * f : 16 * f + 4 * xg);
        const bool whole = col + 4 <= g.N; // all four, and none of them moved (col and n0 are multiples of four, and NJ divides four)
        int at[4];                         // (-1: not this lane's)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            at[e] = col + e;
            if constexpr (NN) {
                const int first = at[e] / NJ * NJ;
                at[e] = min(first, g.N - NJ) + (at[e] - first);
                if (at[e] < first) at[e] = -1;
            }
            if (at[e] >= g.N) at[e] = -1;
        }
        // one epilogue for both kinds of lanes: with one each, which a wavefront at the end of the rows goes through both of,
        // a b 2496 x 128 x 64 took 5.1 us instead of 4.5
        float y[4] = {v[0], v[1], v[2], v[3]};
        auto add4 = [&](const float *row) {
            if (whole) {
                const Floats<4> t = *reinterpret_cast<const Floats<4> *>(row + col);
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += t.v[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (at[e] >= 0) y[e] += row[at[e]];
            }
        };
        const int64_t row0 = static_cast<int64_t>(m) * g.ldc;
        if (bias) add4(bias);
        if (res) add4(res + row0);
        gemm_epilogue_all(g.epilogue, y);
        if (whole) {
            *reinterpret_cast<Floats<4> *>(C + row0 + col) = Floats<4>{{y[0], y[1], y[2], y[3]}};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (at[e] >= 0) C[row0 + at[e]] = y[e];
        }
    }
}

template <bool NN, bool SPLIT, int MI, int NJ, int P> int launch_kernel(const TileArgs &g, hipStream_t s) {
    constexpr int lds = direct_lds_bytes<NN, SPLIT, MI, NJ, P>();
    const auto kernel = gemm_f32_direct_kernel<NN, SPLIT, MI, NJ, P>;
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    AXHIP_CHECK_HIP(configured);
    const int64_t tiles = static_cast<int64_t>((g.M + 16 * MI - 1) / (16 * MI)) * ((g.N + 16 * NJ - 1) / (16 * NJ));
    AXHIP_REQUIRE(launch_fits(tiles + 7, 64 * F32_WAVES), AXHIP_ERR_UNSUPPORTED, "axhip_gemm: too many tiles");
    launch_products(g, tiles, 64 * F32_WAVES, 4, [&](const TileArgs &part, unsigned grid) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * F32_WAVES), lds, s, part); });
    return AXHIP_OK;
}
template <bool NN> int launch_shape(const TileArgs &g, int shape, hipStream_t s) {
    switch (shape) {
    case F32_16x16: return launch_kernel<NN, false, 1, 1, 2>(g, s);
    case F32_16x32: return launch_kernel<NN, false, 1, 2, 2>(g, s);
    case F32_16x64: return launch_kernel<NN, false, 1, 4, 1>(g, s);
    case F32_32x32: return launch_kernel<NN, false, 2, 2, 1>(g, s);
    case F32_32x64: return launch_kernel<NN, false, 2, 4, 1>(g, s);
    case F32_32x64_PARTS: return launch_kernel<NN, true, 2, 4, 1>(g, s);
    default: return launch_kernel<NN, false, 4, 4, 1>(g, s);
    }
}
} // namespace

int launch_f32_direct(const TileArgs &g, bool nn, int shape, hipStream_t s) {
    return nn ? launch_shape<true>(g, shape, s) : launch_shape<false>(g, shape, s);
}
} // namespace axhip
