// C = op(A) op(B) (+ bias) (+ residual), activation epilogue: the dispatch, and
//
//   gemm_mfma_nt_256_kernel    large bf16 / f16 x W^T: 256 x 256 tiles
//   gemm_mfma_f32_ring_kernel  large fp32 products, b along k or [k, n], by products of bf16 parts or on the fp32 matrix instruction
//   gemm_generic_kernel        any dtype / any transpose combination, 16x16 LDS tiles, fp32 FMA
//
// The other 16-bit kernels are in gemm_tile_*.hip (middle-sized products), gemm_small.hip (few rows or few output
// tiles) and gemm_skinny.hip (at most eight rows), the smaller fp32 products in gemm_f32.hip.
#include "common.hpp"
#include "gemm_f32.hpp"
#include "gemm_f32_split.hpp"
#include "gemm_small.hpp"
#include "gemm_skinny.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <set>
#include <utility>
#include <type_traits>

namespace axhip {

struct GemmArgs {
    const void *a, *b;
    void *c;
    const void *bias, *residual;
    int dtype, epilogue;
    int64_t M, N, K;
    int64_t a_rs, a_cs, b_rs, b_cs, ldc; // element strides of op(A)[m][k], op(B)[k][n]
    int64_t sa, sb, sc;                   // batch strides
    int batch;                            // products of this launch
};

// ------------------------------------------------------------------- generic
__global__ __launch_bounds__(256) void gemm_generic_kernel(const GemmArgs g) {
    __shared__ float As[16][17], Bs[16][17];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int64_t bz = blockIdx.z;
    const int64_t m = static_cast<int64_t>(blockIdx.y) * 16 + ty, n = static_cast<int64_t>(blockIdx.x) * 16 + tx;
    const int64_t aoff = bz * g.sa, boff = bz * g.sb, coff = bz * g.sc;
    float acc = 0.0f;
    for (int64_t k0 = 0; k0 < g.K; k0 += 16) {
        const int64_t ka = k0 + tx, kb = k0 + ty;
        As[ty][tx] = (m < g.M && ka < g.K) ? load_any(g.a, g.dtype, aoff + m * g.a_rs + ka * g.a_cs) : 0.0f;
        Bs[ty][tx] = (kb < g.K && n < g.N) ? load_any(g.b, g.dtype, boff + kb * g.b_rs + n * g.b_cs) : 0.0f;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(As[ty][k], Bs[k][tx], acc);
        __syncthreads();
    }
    if (m < g.M && n < g.N) {
        if (g.bias) acc += load_any(g.bias, g.dtype, n);
        if (g.residual) acc += load_any(g.residual, g.dtype, coff + m * g.ldc + n);
        store_any(g.c, g.dtype, coff + m * g.ldc + n, gemm_epilogue(g.epilogue, acc));
    }
}

template <bool BF16>
__device__ __forceinline__ float load16(const void *p, int64_t i) {
    const uint16_t b = static_cast<const uint16_t *>(p)[i];
    return BF16 ? bf16_bits_to_f32(b) : f16_bits_to_f32(b);
}
template <bool BF16>
__device__ __forceinline__ void store16(void *p, int64_t i, float x) {
    static_cast<uint16_t *>(p)[i] = BF16 ? f32_to_bf16_bits(x) : f32_to_f16_bits(x);
}

constexpr int TK = 64; // k-tile of the 256 x 256 kernel

// ----------------------------------------------------------- MFMA NT, 256x256
// Large products: work-group tile 256 x 256 x 64, 8 waves in a 2 x 4 layout, each owning 128 x 64 of C as 8 x 4
// tiles of v_mfma_f32_16x16x32 (128 accumulator registers).  The kernel runs on the chip's power limit, where time
// follows the energy a launch spends rather than its cycle count, and on operands that change every k-step the
// 16x16x32 form does the same flops for about 15 % less than 32x32x16 (a bare loop of either: 1.9 - 2.0 against
// 1.67 - 1.75 PFLOP/s).  A and B k-tiles go L2 -> LDS directly (buffer_load ... lds: no staging registers, no
// ds_write; staging through registers spends as many cycles and more power) into two 64 KiB buffers, one barrier per
// k-tile.  LDS rows are the 128 bytes of one k-tile row with the 16-byte chunk index XOR-ed by (row >> 1) & 7, which
// spreads the 16 rows of a fragment read over all banks.
// A k-tile is two k-steps of 32 MFMAs.  The A fragments are single-buffered: the registers of fragment row i are
// refilled for the next k-step right behind the row's fourth MFMA, 28 MFMAs before they are needed; the B fragments
// are double-buffered.  Every LDS read and every global load sits between two MFMAs (scheduling fences pin the
// order): a wave that meets a batch of reads, or several loads in a row -- a direct-to-LDS load holds the wave's
// issue for about 60 cycles --, starves the matrix pipe of its SIMD.  The barrier comes after the first fragment row
// of the second k-step: by then every wave has read the whole tile, so the buffer takes the tile after next (the
// loads are dealt out one per three MFMAs from there) and the reads turn to the next tile.
// Work-groups are dealt to the 8 XCDs so that each XCD owns a compact block of C tiles and its L2 sees every A / B
// panel few times.
typedef int int4_t __attribute__((ext_vector_type(4)));
constexpr int BIG = 256;              // tile rows (M) and columns (N)
constexpr int BIG_ROWB = TK * 2;      // bytes per LDS row
constexpr int BIG_TILEB = BIG * BIG_ROWB; // 32 KiB per A or B k-tile

// 16 bytes per lane from a buffer straight into LDS: lane i's data lands at lds_base + 16 i.
// Lanes whose voffset lies beyond the descriptor's extent write zeros.
__device__ __forceinline__ void gemm_load_to_lds(const int4_t &rsrc, uint32_t lds_base_uniform, int voffset, int soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_base_uniform), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}

__device__ __forceinline__ int4_t gemm_rsrc(const void *base, int bytes) {
    const uint64_t pa = reinterpret_cast<uint64_t>(base);
    // (the same in every lane: kept in scalar registers)
    return int4_t{__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(pa))),
                  __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(pa >> 32) & 0xFFFFu)), __builtin_amdgcn_readfirstlane(bytes), 0x00020000};
}

// The epilogue for 16x16 accumulator tiles computed as B-fragment x A-fragment^T: lane (l16, g4) holds, of tile
// (i, j), row 16 i + l16 and the four consecutive columns 16 j + 4 g4 .. + 3.
typedef float float4_t __attribute__((ext_vector_type(4)));
template <bool BF16, int RESIDUAL_T, int OP> // RESIDUAL_T: 0 no, 1 yes, 2 decided at run time
__device__ __forceinline__ void gemm_store_tiles16_as(const GemmArgs &g, const float4_t (&acc)[8][4], int64_t m_base, int64_t n_base, int64_t coff, int l16, int g4, unsigned char *stage) {
    const bool RESIDUAL = RESIDUAL_T == 1 || (RESIDUAL_T == 2 && g.residual != nullptr);
    const int cols_valid = static_cast<int>(min<int64_t>(64, g.N - n_base));
    const int rows_valid = static_cast<int>(min<int64_t>(128, g.M - m_base));
    const int64_t origin = coff + m_base * g.ldc + n_base;
    uint16_t *cbase = static_cast<uint16_t *>(g.c) + origin;
    const uint16_t *rbase = static_cast<const uint16_t *>(RESIDUAL ? g.residual : g.c) + origin;
    float bias[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int col = 16 * j + 4 * g4 + e;
            bias[j][e] = g.bias && col < cols_valid ? load16<BF16>(g.bias, n_base + col) : 0.0f;
        }
    // The block goes through the wave's 16 KiB of LDS (free once the k loop has ended): the finished 16-bit values are
    // written in accumulator layout and read back row by row, so that every global store carries 16 bytes per lane and a
    // store instruction fills eight whole 128-byte lines -- of rows that may start anywhere.  While C is
    // written no MFMA runs anywhere on the chip (all work-groups end their k loops together), so the write phase is
    // pure HBM time: 8-byte stores, 32 bytes of a row per instruction, take 9.3 us for the 32 MiB of 4096^2 values.
    const int lane = 16 * g4 + l16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = 16 * i + l16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = 16 * j + 4 * g4;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = acc[i][j][e] + bias[j][e];
            if (RESIDUAL && row < rows_valid) {
                const uint16_t *r = rbase + static_cast<int64_t>(row) * g.ldc + col;
                if (col + 4 <= cols_valid) {
                    const uint2_t t = reinterpret_cast<const uint2_unaligned_t *>(r)->v;
                    const uint32_t rw[2] = {t.x, t.y};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint16_t h = static_cast<uint16_t>(rw[e / 2] >> (16 * (e % 2)));
                        x[e] += BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < cols_valid) x[e] += BF16 ? bf16_bits_to_f32(r[e]) : f16_bits_to_f32(r[e]);
                }
            }
            uint32_t w[2];
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const float y0 = gemm_epilogue16(OP, x[e]), y1 = gemm_epilogue16(OP, x[e + 1]);
                w[e / 2] = BF16 ? pack_bf16x2(y0, y1) : pack_f16x2(y0, y1);
            }
            // 128-byte rows; the 16-byte chunk index is XOR-ed with the row so that neither pass meets bank conflicts
            *reinterpret_cast<uint2_t *>(stage + row * 128 + (((2 * j + (g4 >> 1)) ^ (row & 7)) * 16) + (g4 & 1) * 8) = uint2_t{w[0], w[1]};
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (other lanes' values: the hardware keeps the order, the compiler is told to)
    __builtin_amdgcn_wave_barrier();
    const int q = lane & 7, left = cols_valid - 8 * q; // columns of this lane's chunk and behind
#pragma unroll
    for (int n = 0; n < 16; ++n) {
        const int r = 8 * n + (lane >> 3);
        const uint4_t v = *reinterpret_cast<const uint4_t *>(stage + r * 128 + ((q ^ (r & 7)) * 16));
        if (r >= rows_valid) continue;
        uint16_t *c = cbase + static_cast<int64_t>(r) * g.ldc + 8 * q;
        if (left >= 8) {
            reinterpret_cast<uint4_unaligned_t *>(c)->v = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (e < left) c[e] = static_cast<uint16_t>(v[e / 2] >> (16 * (e % 2)));
        }
    }
}

template <bool BF16>
__device__ __forceinline__ void gemm_store_tiles16(const GemmArgs &g, const float4_t (&acc)[8][4], int64_t m_base, int64_t n_base, int64_t coff, int l16, int g4, unsigned char *stage) {
    if (m_base >= g.M || n_base >= g.N) return;
    // the cheap epilogues get a specialisation with and without residual; the transcendental ones are large when
    // unrolled 128 times, and one general instance each is enough
    switch (g.epilogue) {
    case AXHIP_OP_RELU:
        if (g.residual) gemm_store_tiles16_as<BF16, 1, AXHIP_OP_RELU>(g, acc, m_base, n_base, coff, l16, g4, stage);
        else gemm_store_tiles16_as<BF16, 0, AXHIP_OP_RELU>(g, acc, m_base, n_base, coff, l16, g4, stage);
        break;
    case AXHIP_OP_GELU: gemm_store_tiles16_as<BF16, 2, AXHIP_OP_GELU>(g, acc, m_base, n_base, coff, l16, g4, stage); break;
    case AXHIP_OP_SILU: gemm_store_tiles16_as<BF16, 2, AXHIP_OP_SILU>(g, acc, m_base, n_base, coff, l16, g4, stage); break;
    case AXHIP_OP_SIGMOID: gemm_store_tiles16_as<BF16, 2, AXHIP_OP_SIGMOID>(g, acc, m_base, n_base, coff, l16, g4, stage); break;
    case AXHIP_OP_TANH: gemm_store_tiles16_as<BF16, 2, AXHIP_OP_TANH>(g, acc, m_base, n_base, coff, l16, g4, stage); break;
    default:
        if (g.residual) gemm_store_tiles16_as<BF16, 1, 0>(g, acc, m_base, n_base, coff, l16, g4, stage);
        else gemm_store_tiles16_as<BF16, 0, 0>(g, acc, m_base, n_base, coff, l16, g4, stage);
        break;
    }
}

// Requires K % 64 == 0 and 256 * max(lda, ldb) * 2 < 2^31 (checked by the launcher).
template <bool BF16>
__global__ __launch_bounds__(512, 1) void gemm_mfma_nt_256_kernel(const GemmArgs g, const int tiles_m, const int tiles_n) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char big_lds[]; // A0 B0 A1 B1
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int l16 = lane % 16, g4 = lane / 16;

    // the tiles of a product run down groups of 4 tile rows
    int product;
    const int t = tile_of_work_group(tiles_m * tiles_n, g.batch, product);
    if (t < 0) return;
    constexpr int GR = 4;
    const int group = t / (GR * tiles_n), first_m = group * GR;
    const int gsz = min(GR, tiles_m - first_m);
    const int rem = t - group * GR * tiles_n;
    const int tm = first_m + rem % gsz, tn = rem / gsz;
    const int64_t m0 = static_cast<int64_t>(tm) * BIG, n0 = static_cast<int64_t>(tn) * BIG;
    const int64_t bz = product;
    const uint16_t *A = static_cast<const uint16_t *>(g.a) + bz * g.sa + m0 * g.a_rs;
    const uint16_t *B = static_cast<const uint16_t *>(g.b) + bz * g.sb + n0 * g.b_cs;
    const int arow_bytes = static_cast<int>(g.a_rs) * 2, brow_bytes = static_cast<int>(g.b_cs) * 2;
    const int rows_a = static_cast<int>(min<int64_t>(BIG, g.M - m0)), rows_b = static_cast<int>(min<int64_t>(BIG, g.N - n0));
    const int4_t arsrc = gemm_rsrc(A, (rows_a - 1) * arow_bytes + static_cast<int>(g.K) * 2);
    const int4_t brsrc = gemm_rsrc(B, (rows_b - 1) * brow_bytes + static_cast<int>(g.K) * 2);

    // ---- L2 -> LDS mapping: one wave-wide load moves 8 rows of 128 bytes; load n of wave w
    // covers tile rows 64 n + 8 w + (lane >> 3); the lane fetches the chunk that belongs at
    // position lane & 7 of the swizzled row
    const int ld_r = 8 * wave + (lane >> 3);
    const int ld_c = (lane & 7) ^ ((ld_r >> 1) & 7);
    int a_voff[4], b_voff[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        a_voff[n] = (64 * n + ld_r) * arow_bytes + ld_c * 16;
        b_voff[n] = (64 * n + ld_r) * brow_bytes + ld_c * 16;
    }
    const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(big_lds));
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(lds_base + 8 * wave * BIG_ROWB);
    auto load_one = [&](const int4_t &ar, const int4_t &br, int kt, int buf, int n) __attribute__((always_inline)) { // n: 0..3 of A, 4..7 of B
        const int soff = kt * BIG_ROWB;
        if (n < 4) gemm_load_to_lds(ar, lds_wave + buf * 2 * BIG_TILEB + n * 64 * BIG_ROWB, a_voff[n % 4], soff);
        else gemm_load_to_lds(br, lds_wave + buf * 2 * BIG_TILEB + BIG_TILEB + (n - 4) * 64 * BIG_ROWB, b_voff[n % 4], soff);
    };

    // ---- fragment reads: row l16 of a 16-row block, 16-byte chunk 4 s + g4 of the row's eight (s: k-step of the tile)
    const int wm = (wave / 4) * 128, wn = (wave % 4) * 64;
    int f_off[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) f_off[s] = l16 * BIG_ROWB + (((4 * s + g4) ^ ((l16 >> 1) & 7)) * 16);

    float4_t acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    uint4_t fa[8], fb[2][4];
    auto read_a = [&](int buf, int s, int i) __attribute__((always_inline)) {
        fa[i] = *reinterpret_cast<const uint4_t *>(big_lds + buf * 2 * BIG_TILEB + (wm + 16 * i) * BIG_ROWB + f_off[s]);
    };
    auto read_b = [&](int slot, int buf, int s, int j) __attribute__((always_inline)) {
        fb[slot][j] = *reinterpret_cast<const uint4_t *>(big_lds + buf * 2 * BIG_TILEB + BIG_TILEB + (wn + 16 * j) * BIG_ROWB + f_off[s]);
    };
    // D = (B fragment) x (A fragment)^T: the lane holds four consecutive columns of one row of C
    auto mfma = [&](int slot, int i, int j) __attribute__((always_inline)) {
        if constexpr (BF16)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fb[slot][j]), __builtin_bit_cast(bf16x8_t, fa[i]), acc[i][j], 0, 0, 0);
        else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, fb[slot][j]), __builtin_bit_cast(half8_t, fa[i]), acc[i][j], 0, 0, 0);
    };
#define AXHIP_FENCE() __builtin_amdgcn_sched_barrier(0)

    const int nk = static_cast<int>(g.K / TK);
#pragma unroll
    for (int n = 0; n < 8; ++n) load_one(arsrc, brsrc, 0, 0, n);
    if (nk > 1) {
#pragma unroll
        for (int n = 0; n < 8; ++n) load_one(arsrc, brsrc, 1, 1, n);
        __builtin_amdgcn_s_waitcnt(0x0F78); // vmcnt(8): tile 0 has landed
    } else {
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) read_a(0, 0, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) read_b(0, 0, 0, j);
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        // past the last tile the loads run on empty descriptors (every lane out of range: zeros into a buffer nobody
        // reads, no memory traffic) rather than behind eight branches
        const bool more = kt + 2 < nk;
        const int4_t ar = int4_t{arsrc.x, arsrc.y, more ? arsrc.z : 0, arsrc.w}, br = int4_t{brsrc.x, brsrc.y, more ? brsrc.z : 0, brsrc.w};
        AXHIP_FENCE();
        // k-step 0: B slot 0; the refills fetch k-step 1 of this tile
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                mfma(0, i, j);
                AXHIP_FENCE();
                if (j == 2 && i < 4) {
                    read_b(1, buf, 1, i);
                    AXHIP_FENCE();
                }
                if (j == 3) {
                    read_a(buf, 1, i);
                    AXHIP_FENCE();
                }
            }
        // k-step 1: B slot 1; behind the barrier the refills fetch k-step 0 of the next tile (after the last tile: a
        // harmless read of stale LDS) and this tile's buffer takes the tile after next
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i == 1) {
                __builtin_amdgcn_s_waitcnt(0x0F70); // this wave's share of tile kt+1 has landed
                __syncthreads();                    // ... everyone's has, and tile kt is no longer read
                AXHIP_FENCE();
                read_a(buf ^ 1, 0, 0);
                AXHIP_FENCE();
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                mfma(1, i, j);
                AXHIP_FENCE();
                if (i >= 1) {
                    const int q = (i - 1) * 4 + j; // MFMAs since the barrier
                    if (q % 3 == 1 && q / 3 < 8) {
                        load_one(ar, br, kt + 2, buf, q / 3);
                        AXHIP_FENCE();
                    }
                    if (q % 2 == 0 && q >= 2 && q <= 8) {
                        read_b(0, buf ^ 1, 0, q / 2 - 1);
                        AXHIP_FENCE();
                    }
                    if (j == 3) {
                        read_a(buf ^ 1, 0, i);
                        AXHIP_FENCE();
                    }
                }
            }
        }
    }
#undef AXHIP_FENCE

    // the tile buffers become the staging area of the epilogue: no load of this work-group is still on its way into them
    // (past the last tile they write zeros), and every wave has its last fragments
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    gemm_store_tiles16<BF16>(g, acc, m0 + wm, n0 + wn, bz * g.sc, l16, g4, big_lds + wave * 16384);
}

// ------------------------------------------------------------------ fp32, MFMA
// C = A B^T (B [N,K]) or A B (NN: B [K,N]) in fp32 on v_mfma_f32_32x32x2_f32: fp32 products, fp32 accumulation, so no
// precision is given up against the FMA kernel.  Work-group tile TM x TNR, four wavefronts with a quarter of it each; a
// ring of S k-tiles of 32 floats, i.e. the 128-byte LDS rows, XOR swizzle and direct-to-LDS loads of the 256 x 256 kernel.
// A lane's 16-byte fragment read holds four k values that feed four successive MFMAs (which k a lane contributes to which
// MFMA is free as long as A and B agree).  NN: a k-tile of B is 32 rows of TNR floats, and a lane's four k values of its
// column are four 4-byte reads -- as many LDS cycles as the one of 16 bytes, and no pass that transposes B first.
// At 1/16 of the 16-bit rate the matrix pipe is the bound, so nothing but the barrier may stand between two MFMAs of a
// wavefront, of which a SIMD has one: four more wavefronts, one per SIMD, issue the loads (a direct-to-LDS load holds the
// issue of its wavefront for longer than an MFMA takes, wherever it stands: 64 x 1536 x 4096 on 64 x 64 tiles 84 us, with
// loaders 76), the fragments of the next eight k are read under the MFMAs of these, the barrier of a k-tile comes before its
// last steps (by then every wavefront has read the whole tile), and behind it the reads turn to the next tile.  One k-tile of
// 64 x 64, one work-group a CU: 1024 cycles of MFMAs in 1310.  The values of a finished block then take bias, residual and
// activation together: with a branch on the activation for each, 60 KB of code that every CU read anew, 4096 x 4096 x 512 + GELU
// took 228 us instead of 176.
// Products of parts (SplitRing) take its place where their time is less, which takes k enough: of this form's tiles of 64 x 64 three
// work-groups share a CU (8 x (2939 x 704 x 66) 41 us against 54 on parts, when those were six products).  Tiles whose parts have no finite sums run it, too.
// Rows may start anywhere: the loads need 4-byte alignment.  The chunk that K ends in is fetched as the four floats that
// end with the row and shifted into place in LDS by the lane that loaded it; chunks behind it, and k-tiles past the last,
// are sent out of the descriptor's range and arrive as zeros.  NN rows that are no whole chunks: the last column tile is
// moved left to end with them (N >= TNR); the columns it shares with its neighbour are the neighbour's to store.

// The same tiles by products of bf16 parts (gemm_f32_split.hpp).  Splitting an element takes seven VALU operations, of which about
// five fit beside a 32-cycle MFMA of another wavefront, so each is split once for the whole work-group: the loading wavefronts keep
// DEPTH k-tiles on their way in registers, split one and write its parts to LDS, in the order in which fragments are read: a block of
// 32 rows, 8 k at a time, is 512 bytes, 16 a row (the row XOR-ed so that what 32 lanes write at a time meets all banks).
// The multiplying ones, one per SIMD, hold all fragments of 32 k and refill them under the MFMAs of blocks that need them no
// more.  Barrier kt: k-tile kt is in LDS and k-tile kt - 1 has been read.
// What bounds it: VALU issue where CUs have one tile (1024^3: 30.6 k of 49.5 k cycles, beside 16.4 k of MFMAs, under each of which about five
// of eight VALU slots are free), the matrix pipe under the power limit on a full chip (4096^3: 74 % busy).  So 64 x 64 has two loading
// wavefronts per SIMD (1024^3 22.5 us with one, 19.4 with two, of six products) and 64 k at a time for half the barriers.
// v_mfma_f32_16x16x32, which leaves less room beside it, took 3 % less on full chips and 10 % more on others.
// With fp32 products and with these, us: 1024^3 21.6 and 21.0 (b as [k, n] 22.1 and 22.4), 2048^3 133 and 114, 4096 x 2000 x 1000 134 and
// 118, 4096^3 1014 and 832.  (Six of the products, to fewer bits: 18.9, 95, 101, 697.)
template <int TM, int TNR, int KF, int LW, bool NN> struct SplitRing { // KF: floats per k-tile; LW: loading wavefronts
    static constexpr int MI = TM / 64, NJ = TNR / 64, DEPTH = KF == 32 || LW == 8 ? 3 : 2;
    static constexpr int CHUNKS = KF / 4, ROWS = WAVE / CHUNKS * LW;      // 16-byte chunks of a row along k, rows that the loading wavefronts fetch at a time
    static constexpr int NLA = TM / ROWS, NLB = TNR / ROWS;               // loads of a lane per k-tile
    static constexpr int PLANE_A = TM * KF * 2, PLANE_B = TNR * KF * 2, STAGEB = 3 * (PLANE_A + PLANE_B);

    // where the 8 k of chunk pair kc of row r of an operand's plane lie
    static __device__ __forceinline__ int at(int r, int kc) { return (r / 32) * (KF * 64) + kc * 512 + (((r % 32) ^ (((r / 16) & 3) | ((kc & 3) << 2)) ^ (kc / 4 * 2)) * 16); }

    static __device__ __forceinline__ void load(const GemmArgs &g, const float *A, const float *B, int rows_a, int rows_b, unsigned char *lds, int wave, int lane) {
        const int arow = static_cast<int>(g.a_rs) * 4, brow = static_cast<int>(NN ? g.b_rs : g.b_cs) * 4;
        const int K = static_cast<int>(g.K), nk = (K + KF - 1) / KF;
        const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, (rows_a - 1) * arow + K * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, NN ? (K - 1) * brow + rows_b * 4 : (rows_b - 1) * brow + K * 4, 0x00020000);
        constexpr uint32_t OUT_OF_RANGE = 0x7FFFFFF0u;
        // rows along k: load n is row ROWS n + r0, floats k0 .. + 3 of the k-tile
        const int r0 = WAVE / CHUNKS * wave + lane / CHUNKS, k0 = 4 * (lane % CHUNKS);
        // b as [k, n]: load n is row bk + n, columns bn .. + 3 (of every 32 lanes 16 lie side by side and 16 on the next rows: what
        // they write then meets all banks)
        constexpr int WIDE = TNR / 64; // runs of 16 lanes to a row
        const int run = wave * 4 + lane / 16, bk = (run / (2 * WIDE) * 2 + run % 2) * NLB, bn = (run / 2 % WIDE * 16 + lane % 16) * 4;
        uint4_t regs[DEPTH][NLA + NLB];
        auto fetch = [&](int set, int kt, int n) __attribute__((always_inline)) { // n: of a, then of b
            const int k = kt * KF + k0;
            const uint32_t along = k < K ? static_cast<uint32_t>(min(k, K - 4)) * 4u : OUT_OF_RANGE;
            if (n < NLA) {
                regs[set][n] = __builtin_amdgcn_raw_buffer_load_b128(ar, static_cast<uint32_t>((ROWS * n + r0) * arow) + along, 0, 0);
            } else if constexpr (NN) {
                const int row = kt * KF + bk + n - NLA;
                regs[set][n] = __builtin_amdgcn_raw_buffer_load_b128(br, row < K && bn < rows_b ? static_cast<uint32_t>(row * brow + bn * 4) : OUT_OF_RANGE, 0, 0);
            } else {
                regs[set][n] = __builtin_amdgcn_raw_buffer_load_b128(br, static_cast<uint32_t>((ROWS * (n - NLA) + r0) * brow) + along, 0, 0);
            }
        };
        // k-tile kt -> LDS; `behind(n)` once the registers of load n are free: the loads of a later k-tile stand between the splits of
        // this one (side by side they wait for each other, 16 cycles of the CU's address path each)
        auto write = [&](int set, int kt, auto behind) __attribute__((always_inline)) {
            if (K % 4 != 0 && kt == nk - 1) {
                const int drop = kt * KF + k0 + 4 - K; // floats in front of the chunk that K ends in
                if (drop > 0 && drop < 4) {
#pragma unroll
                    for (int n = 0; n < NLA + (NN ? 0 : NLB); ++n) regs[set][n] = __builtin_bit_cast(uint4_t, __builtin_bit_cast(unsigned __int128, regs[set][n]) >> (32 * drop));
                }
            }
            unsigned char *stage = lds + (kt & 1) * STAGEB;
            if constexpr (NN) {
                float4_t v[NLB];
#pragma unroll
                for (int n = 0; n < NLB; ++n) v[n] = __builtin_bit_cast(float4_t, regs[set][NLA + n]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t w[NLB / 2][3];
#pragma unroll
                    for (int n = 0; n < NLB / 2; ++n) split_pair(v[2 * n][j], v[2 * n + 1][j], w[n]);
                    unsigned char *to = stage + 3 * PLANE_A + at(bn + j, bk / 8) + (bk % 8) * 2;
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        if constexpr (NLB == 8) *reinterpret_cast<uint4_t *>(to + q * PLANE_B) = uint4_t{w[0][q], w[1][q], w[NLB / 2 - 2][q], w[NLB / 2 - 1][q]};
                        else if constexpr (NLB == 4) *reinterpret_cast<uint2_t *>(to + q * PLANE_B) = uint2_t{w[0][q], w[NLB / 2 - 1][q]};
                        else *reinterpret_cast<uint32_t *>(to + q * PLANE_B) = w[0][q];
                    }
                }
            }
#pragma unroll
            for (int n = 0; n < NLA + (NN ? 0 : NLB); ++n) {
                const bool a = n < NLA;
                const float4_t v = __builtin_bit_cast(float4_t, regs[set][n]);
                uint32_t lo[3], hi[3];
                split_pair(v[0], v[1], lo);
                split_pair(v[2], v[3], hi);
                unsigned char *to = stage + (a ? 0 : 3 * PLANE_A) + at(ROWS * (a ? n : n - NLA) + r0, k0 / 8) + (k0 / 4 & 1) * 8;
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2_t *>(to + q * (a ? PLANE_A : PLANE_B)) = uint2_t{lo[q], hi[q]};
                __builtin_amdgcn_sched_barrier(0);
                behind(n);
                if constexpr (NN) {
#pragma unroll
                    for (int x = n * NLB / NLA; x < (n + 1) * NLB / NLA; ++x) behind(NLA + x);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int n = 0; n < NLA + NLB; ++n) fetch(d, d, n);
        int kt = 0;
        for (; kt + DEPTH <= nk; kt += DEPTH) { // (no branch inside: the compiler would wait for every load in flight where the paths meet)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                write(d, kt + d, [&](int n) __attribute__((always_inline)) { fetch(d, kt + d + DEPTH, n); });
                __syncthreads();
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d) {
            if (kt + d < nk) {
                write(d, kt + d, [](int) {});
                __syncthreads();
            }
        }
        __syncthreads(); // barrier nk
    }

    static __device__ __forceinline__ float16_t mfma(const uint4_t &a, const uint4_t &b, const float16_t &sum) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), sum, 0, 0, 0);
    }

    // -> sum[i][j]: as the fp32 MFMAs leave them, times SPLIT_SCALE^2
    static __device__ __forceinline__ void multiply(int K, const unsigned char *lds, int wm, int wn, int lane, float16_t (&sum)[MI][NJ]) {
        const int nk = (K + KF - 1) / KF, l32 = lane % 32, g2 = lane / 32;
        // KF = 32, four blocks: the fragments of one are dead long before the next k-tile needs them.  KF = 64: the halves of a k-tile in turn
        constexpr int SLOTS = KF / 32, BLOCKS = MI * NJ;
        static_assert(SLOTS == 1 ? MI == 2 && NJ == 2 : MI == 1, "blocks");
        uint4_t fa[SLOTS][MI][2][2], fb[SLOTS][NJ][2][2], fa_last[MI][2], fb_last[NJ][2]; // (the last parts are used first: one set of registers for both halves)
        auto frag_a = [&](int h, int i, int ks, int part) __attribute__((always_inline)) -> uint4_t & { return part == 2 ? fa_last[i][ks] : fa[h][i][ks][part & 1]; };
        auto frag_b = [&](int h, int j, int ks, int part) __attribute__((always_inline)) -> uint4_t & { return part == 2 ? fb_last[j][ks] : fb[h][j][ks][part & 1]; };
        // One offset for a block of 32 rows, from which those of the other k of a k-tile are made: at(r, kc + 4) = (at(r, kc) ^ 32) + 2048, at(r, kc + 2) =
        // (at(r, kc) ^ 128) + 1024.  (The stage is in it before the XOR, so that all of them are not kept, in registers that the fragments need.)
        int a_off[MI], b_off[NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i) a_off[i] = at(wm + 32 * i + l32, g2);
#pragma unroll
        for (int j = 0; j < NJ; ++j) b_off[j] = 3 * PLANE_A + at(wn + 32 * j + l32, g2);
        static_assert(STAGEB % 512 == 0 && PLANE_A % 512 == 0, "the XOR is of the bits below 512");
        auto read_a = [&](int h, int stage, int i, int n) __attribute__((always_inline)) { // n: 3 ks + part
            frag_a(h, i, n / 3, n % 3) = *reinterpret_cast<const uint4_t *>(lds + (((stage + a_off[i]) ^ (h * 32 + n / 3 * 128)) + h * 2048 + n / 3 * 1024 + n % 3 * PLANE_A));
        };
        auto read_b = [&](int h, int stage, int j, int n) __attribute__((always_inline)) {
            frag_b(h, j, n / 3, n % 3) = *reinterpret_cast<const uint4_t *>(lds + (((stage + b_off[j]) ^ (h * 32 + n / 3 * 128)) + h * 2048 + n / 3 * 1024 + n % 3 * PLANE_B));
        };
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) sum[i][j] = float16_t{};
        float16_t first[2] = {float16_t{}, float16_t{}}, rest{};
        // block (i, j) of 32 k: sixteen MFMAs, behind MFMA x what `between` does.  The products of first parts, then, in a chain of their own, the rest;
        // under the next block's MFMAs the two are added up, and to the sum of their block (`before`)
        auto block = [&](int h, int i, int j, float16_t &before, auto between) __attribute__((always_inline)) {
            const int turn = BLOCKS > 1 ? (i * NJ + j) & 1 : h;
#pragma unroll
            for (int x = 0; x < 2 * SPLIT_PRODUCTS; ++x) {
                const int n = x / 2, ks = x % 2;
                if (x < 2) first[turn] = mfma(frag_a(h, i, ks, SPLIT_A[n]), frag_b(h, j, ks, SPLIT_B[n]), x == 0 ? float16_t{} : first[turn]);
                else rest = mfma(frag_a(h, i, ks, SPLIT_A[n]), frag_b(h, j, ks, SPLIT_B[n]), x == 2 ? float16_t{} : rest);
                __builtin_amdgcn_sched_barrier(0);
                if (x < 2) {
#pragma unroll
                    for (int e = 8 * x; e < 8 * x + 8; ++e) first[turn ^ 1][e] += rest[e];
                } else if (x >= 3 && x < 11) {
#pragma unroll
                    for (int e = 2 * (x - 3); e < 2 * (x - 3) + 2; ++e) before[e] += first[turn ^ 1][e];
                }
                between(x);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        __syncthreads(); // barrier 0
        if constexpr (SLOTS == 1) {
#pragma unroll
            for (int n = 0; n < 6; ++n) {
                read_a(0, 0, 0, n);
                read_b(0, 0, 0, n);
            }
            for (int kt = 0; kt < nk; ++kt) {
                const int cur = (kt & 1) * STAGEB, next = STAGEB - cur;
                block(0, 0, 0, sum[1][1], [&](int x) __attribute__((always_inline)) {
                    if (x < 6) read_b(0, cur, 1, x);
                    else read_a(0, cur, 1, x - 6);
                });
                block(0, 0, 1, sum[0][0], [](int) {});
                __syncthreads(); // barrier kt + 1 (behind the last k-tile: what is read below is not used)
                block(0, 1, 0, sum[0][1], [&](int x) __attribute__((always_inline)) {
                    if (x < 6) read_a(0, next, 0, x);
                });
                block(0, 1, 1, sum[1][0], [&](int x) __attribute__((always_inline)) {
                    if (x < 6) read_b(0, next, 0, x);
                });
            }
            sum[1][1] += first[1] + rest;
        } else {
            float16_t odd[NJ]; // the second halves' sums: two chains of K / 64 additions
#pragma unroll
            for (int j = 0; j < NJ; ++j) odd[j] = float16_t{};
            auto half = [&](int h, int stage) __attribute__((always_inline)) { // multiplies half h and reads the other one from `stage`
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    block(h, 0, j, j == 0 ? (h == 0 ? odd[NJ - 1] : sum[0][NJ - 1]) : (h == 0 ? sum[0][j - 1] : odd[j - 1]), [&](int x) __attribute__((always_inline)) {
                        if (j == 0 && x < 4) read_a(h ^ 1, stage, 0, x / 2 * 3 + x % 2);
                        if (j == 0 && x < 4 * NJ) read_b(h ^ 1, stage, x / 4, x % 4 / 2 * 3 + x % 2);
                        // (behind their last use, of SPLIT_B by MFMA 7 and of SPLIT_A by MFMA 9)
                        if (x == 8 || x == 9) read_b(h ^ 1, stage, j, (x - 8) * 3 + 2);
                        if (j == NJ - 1 && (x == 10 || x == 11)) read_a(h ^ 1, stage, 0, (x - 10) * 3 + 2);
                    });
            };
#pragma unroll
            for (int n = 0; n < 6; ++n) {
                read_a(0, 0, 0, n);
#pragma unroll
                for (int j = 0; j < NJ; ++j) read_b(0, 0, j, n);
            }
            for (int kt = 0; kt < nk; ++kt) {
                half(0, (kt & 1) * STAGEB);
                __syncthreads(); // barrier kt + 1
                half(1, ((kt & 1) ^ 1) * STAGEB);
            }
            odd[NJ - 1] += first[1] + rest;
#pragma unroll
            for (int j = 0; j < NJ; ++j) sum[0][j] += odd[j];
        }
    }
};

constexpr int RING_STAGES = 3;
template <int TM, int TNR> constexpr int ring_lds_bytes() { return RING_STAGES * (TM + TNR) * BIG_ROWB; }
template <int TM, int TNR, int KF, int LW> constexpr int split_lds_bytes() { // the ring or both stages of parts, and a flag of each wavefront
    const int ring = ring_lds_bytes<TM, TNR>(), split = 2 * SplitRing<TM, TNR, KF, LW, false>::STAGEB;
    return (ring > split ? ring : split) + 64;
}

template <int TM, int TNR, int KF, int LW, bool NN> // KF: 0 fp32 products, else products of parts
__global__ __launch_bounds__(64 * (4 + LW), 1) void gemm_mfma_f32_ring_kernel(const GemmArgs g, const int tiles_m, const int tiles_n) {
    constexpr int MI = TM / 64, NJ = TNR / 64;
    constexpr int NLA = TM / 32, NLB = TNR / 32, NL = NLA + NLB; // loads of 1 KiB per wavefront and k-tile
    constexpr int RK = 32, S = RING_STAGES, STAGEB = (TM + TNR) * BIG_ROWB; // (fp32 products: floats per k-tile, stages)
    extern __shared__ __attribute__((aligned(1024))) unsigned char big_lds[];
    const int wavefront = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), wave = wavefront % 4;
    const bool loader = wavefront >= 4;

    int product;
    const int t = tile_of_work_group(tiles_m * tiles_n, g.batch, product);
    if (t < 0) return;
    constexpr int GR = 4;
    const int group = t / (GR * tiles_n), first_m = group * GR;
    const int gsz = min(GR, tiles_m - first_m);
    const int rem = t - group * GR * tiles_n;
    const int tm = first_m + rem % gsz, tn = rem / gsz;
    const int64_t m0 = static_cast<int64_t>(tm) * TM, n_low = static_cast<int64_t>(tn) * TNR;
    const int64_t n0 = NN && g.N % 4 != 0 ? min<int64_t>(n_low, g.N - TNR) : n_low;
    const int64_t bz = product;
    const float *A = static_cast<const float *>(g.a) + bz * g.sa + m0 * g.a_rs;
    const float *B = static_cast<const float *>(g.b) + bz * g.sb + n0 * (NN ? 1 : g.b_cs);
    const int arow_bytes = static_cast<int>(g.a_rs) * 4, brow_bytes = static_cast<int>(NN ? g.b_rs : g.b_cs) * 4;
    const int rows_a = static_cast<int>(min<int64_t>(TM, g.M - m0)), rows_b = static_cast<int>(min<int64_t>(TNR, g.N - n0));
    const int K = static_cast<int>(g.K), nk = (K + RK - 1) / RK;
    const int4_t arsrc = gemm_rsrc(A, (rows_a - 1) * arow_bytes + K * 4);
    const int4_t brsrc = gemm_rsrc(B, NN ? (K - 1) * brow_bytes + rows_b * 4 : (rows_b - 1) * brow_bytes + K * 4);

    const int wm = (wave / 2) * (TM / 2), wn = (wave % 2) * (TNR / 2);

    float16_t sum[MI][NJ];
    bool fp32_products = true;
    if constexpr (KF != 0) {
        using Split = SplitRing<TM, TNR, KF, LW, NN>;
        bool failed = false;
        if (loader) {
            Split::load(g, A, B, rows_a, rows_b, big_lds, wavefront - 4, lane_again());
        } else {
            Split::multiply(K, big_lds, wm, wn, lane_again(), sum);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        failed = failed || split_failed(sum[i][j][e]);
                        sum[i][j][e] *= SPLIT_UNSCALE;
                    }
        }
        fp32_products = work_group_any<4 + LW>(failed, reinterpret_cast<uint32_t *>(big_lds + split_lds_bytes<TM, TNR, KF, LW>() - 64), wavefront, lane_again());
    }
    const int lane = KF == 0 ? static_cast<int>(threadIdx.x % WAVE) : lane_again(), l32 = lane % 32, g2 = lane / 32;
    if (fp32_products) {
    const int ld_r = 8 * wave + (lane >> 3);
    const int ld_k = 4 * ((lane & 7) ^ ((ld_r >> 1) & 7)); // this lane's chunk of a row along k: floats ld_k .. ld_k + 3 of the k-tile
    constexpr int OUT_OF_RANGE = 0x7FFFFFF0;
    int a_row[NLA], b_row[NLB]; // where the rows of this lane's chunks start (NN, b: where the chunks of k-tile 0 do)
#pragma unroll
    for (int n = 0; n < NLA; ++n) a_row[n] = (32 * n + ld_r) * arow_bytes;
#pragma unroll
    for (int n = 0; n < NLB; ++n) {
        const int at = (4 * n + wave) * 1024 + lane * 16; // of the tile
        if (NN) b_row[n] = at % (TNR * 4) < rows_b * 4 ? at / (TNR * 4) * brow_bytes + at % (TNR * 4) : OUT_OF_RANGE;
        else b_row[n] = (32 * n + ld_r) * brow_bytes;
    }
    const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(big_lds));
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(lds_base + 8 * wave * BIG_ROWB);
    auto load = [&](int kt, int stage_off, int n) __attribute__((always_inline)) { // n: of A, then of B
        const int k0 = kt * RK;
        const int along = k0 + ld_k < K ? min(k0 + ld_k, K - 4) * 4 : OUT_OF_RANGE; // of a row along k
        if (n < NLA) {
            gemm_load_to_lds(arsrc, lds_wave + stage_off + n * 32 * BIG_ROWB, along == OUT_OF_RANGE ? OUT_OF_RANGE : a_row[n < NLA ? n : 0] + along, 0);
        } else {
            const int nb = n < NLA ? 0 : n - NLA;
            const uint32_t to = lds_wave + stage_off + TM * BIG_ROWB + nb * 32 * BIG_ROWB;
            if (NN) gemm_load_to_lds(brsrc, to, k0 + ((4 * nb + wave) * 1024 + lane * 16) / (TNR * 4) < K ? b_row[nb] : OUT_OF_RANGE, kt < nk ? k0 * brow_bytes : 0);
            else gemm_load_to_lds(brsrc, to, along == OUT_OF_RANGE ? OUT_OF_RANGE : b_row[nb] + along, 0);
        }
    };
    // the last k-tile, where K is no multiple of 4: this lane's chunks that K ends in, already in LDS, are put in place
    auto mend = [&](int stage_off) __attribute__((always_inline)) {
        const int drop = (nk - 1) * RK + ld_k + 4 - K; // floats in front of the chunk
        if (drop <= 0 || drop >= 4) return;
#pragma unroll
        for (int n = 0; n < (NN ? NLA : NL); ++n) {
            float4_t *c = reinterpret_cast<float4_t *>(big_lds + stage_off + n * 32 * BIG_ROWB + wave * 1024 + lane * 16);
            *c = __builtin_bit_cast(float4_t, __builtin_bit_cast(unsigned __int128, *c) >> (32 * drop));
        }
    };

#define AXHIP_FENCE() __builtin_amdgcn_sched_barrier(0)
#define AXHIP_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | 0x0F70 | (((n) >> 4) << 14))
    static_assert(S >= 3 && NL * (S - 1) < 64, "vmcnt is a 6-bit counter");
    if (LW > 4 && wavefront >= 8) { // (four load)
        for (int kt = 0; kt <= nk; ++kt) __syncthreads();
    } else if (loader) {
#pragma unroll
        for (int st = 0; st < S - 1; ++st)
#pragma unroll
            for (int n = 0; n < NL; ++n) load(st, st * STAGEB, n);
        AXHIP_VMCNT(NL * (S - 2)); // tile 0 has landed
        __syncthreads();
        int next = STAGEB, to = (S - 1) * STAGEB; // stages of tile kt + 1, and of kt + S - 1 (that of kt - 1: everyone has read it)
        for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
            for (int n = 0; n < NL; ++n) load(kt + S - 1, to, n);
            AXHIP_VMCNT(NL * (S - 2)); // tile kt + 1 has landed
            if (K % 4 != 0 && kt + 2 == nk) mend(next);
            __syncthreads();
            next = next + STAGEB == S * STAGEB ? 0 : next + STAGEB;
            to = to + STAGEB == S * STAGEB ? 0 : to + STAGEB;
        }
        AXHIP_VMCNT(0); // no load is still on its way into LDS
    } else {

    int f_off[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) f_off[ks] = l32 * BIG_ROWB + (((2 * ks + g2) ^ ((l32 >> 1) & 7)) * 16);

    // The sums of a k-tile are added to those of all before: chains of 32 fp32 additions, then one of K / 32, in place of one
    // of K (2048^3, one chain: 8.1e-7 off the exact result, these 1.8e-7).
    float16_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) sum[i][j] = float16_t{};

    // fragments of LOOK steps of eight k are on their way while one is multiplied: with one block a wavefront has four MFMAs
    // for these, less than a read takes next to three other wavefronts'
    constexpr int LOOK = MI * NJ == 1 ? 2 : 1, SLOTS_F = 2 * LOOK;
    float4_t fa[SLOTS_F][MI], fb[SLOTS_F][NJ];
    auto read_a = [&](int slot, int stage_off, int step, int i) __attribute__((always_inline)) {
        fa[slot][i] = *reinterpret_cast<const float4_t *>(big_lds + stage_off + (wm + 32 * i) * BIG_ROWB + f_off[step]);
    };
    auto read_b = [&](int slot, int stage_off, int step, int j) __attribute__((always_inline)) {
        const unsigned char *Bs = big_lds + stage_off + (NN ? TM : TM + wn) * BIG_ROWB;
        if constexpr (NN) {
#pragma unroll
            for (int c = 0; c < 4; ++c) fb[slot][j][c] = reinterpret_cast<const float *>(Bs)[(8 * step + 4 * g2 + c) * TNR + wn + 32 * j + l32];
        } else {
            fb[slot][j] = *reinterpret_cast<const float4_t *>(Bs + 32 * j * BIG_ROWB + f_off[step]);
        }
    };
    // eight k: 4 MI NJ MFMAs; behind MFMA (c, i, j) what `between` does
    auto multiply = [&](int slot, bool first, auto between) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[slot][i][c], fb[slot][j][c], first && c == 0 ? float16_t{} : acc[i][j], 0, 0, 0);
                    AXHIP_FENCE();
                    between(c, i, j);
                    AXHIP_FENCE();
                }
    };

    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < LOOK; ++ks) {
#pragma unroll
        for (int i = 0; i < MI; ++i) read_a(ks, 0, ks, i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) read_b(ks, 0, ks, j);
    }
    int cur = 0; // offset of k-tile kt's stage
    for (int kt = 0; kt < nk; ++kt) {
        const int next = cur + STAGEB == S * STAGEB ? 0 : cur + STAGEB;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            constexpr int LAST = 4 - LOOK; // from here on the reads are the next tile's
            const int from = ks >= LAST ? next : cur;
            if (ks == LAST) {
                __syncthreads(); // tile kt + 1 has landed, and tile kt is no longer read
                AXHIP_FENCE();
            }
            multiply(ks % SLOTS_F, ks == 0, [&](int c, int i, int j) __attribute__((always_inline)) {
                const int x = (c * MI + i) * NJ + j;
                if (x < MI) read_a((ks + LOOK) % SLOTS_F, from, (ks + LOOK) % 4, x);
                if (x < NJ) read_b((ks + LOOK) % SLOTS_F, from, (ks + LOOK) % 4, x);
            });
        }
        cur = next;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) sum[i][j] += acc[i][j];
    }
    }
#undef AXHIP_VMCNT
#undef AXHIP_FENCE
    }
    if (loader) return;

    // epilogue: accumulator element e of tile (i, j) is C[m + 32 i + 8 (e / 4) + 4 g2 + e % 4][n + 32 j + l32].  The 16
    // values of a tile take each step together: one branch on the epilogue, one set of loads on their way.
    float *Cb = static_cast<float *>(g.c) + bz * g.sc;
    const float *Rb = g.residual ? static_cast<const float *>(g.residual) + bz * g.sc : nullptr;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int64_t col = n0 + wn + 32 * j + l32;
        if (col >= g.N || col < n_low) continue;
        const float bias = g.bias ? static_cast<const float *>(g.bias)[col] : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int64_t row0 = m0 + wm + 32 * i + 4 * g2, at0 = row0 * g.ldc + col;
            const int rows = static_cast<int>(min<int64_t>(32, g.M - row0)); // (row 8 (e / 4) + e % 4 of these)
            float x[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) x[e] = sum[i][j][e] + bias;
            if (Rb) {
#pragma unroll
                for (int e = 0; e < 16; ++e) x[e] += 8 * (e / 4) + e % 4 < rows ? Rb[at0 + (8 * (e / 4) + e % 4) * g.ldc] : 0.0f;
            }
            gemm_epilogue_all(g.epilogue, x);
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (8 * (e / 4) + e % 4 < rows) Cb[at0 + (8 * (e / 4) + e % 4) * g.ldc] = x[e];
        }
    }
}

} // namespace axhip

using namespace axhip;

// AXHIP_GEMM_F32_MFMA=0 routes fp32 products to the FMA kernel (for A/B timing)
static bool f32_mfma_enabled() {
    static const bool on = [] { const char *e = std::getenv("AXHIP_GEMM_F32_MFMA"); return !(e && e[0] == '0'); }();
    return on;
}

// AXHIP_GEMM_SKINNY=0: products with at most 8 rows on the tiled kernels (for A/B timing)
static bool skinny_enabled() {
    static const bool on = [] { const char *e = std::getenv("AXHIP_GEMM_SKINNY"); return !(e && e[0] == '0'); }();
    return on;
}

namespace {
// Whether a product is of a form that may have to be repacked (and into how many padded columns): large, with an operand
// stored the other way or a k off the vector grid.  axhip_gemm_workspace_bytes answers for the form; the kernels that read
// such operands as they lie (16-bit ones with A along k, most fp32 ones) leave the memory alone.
struct Repack { bool on, a, b; int64_t kp; };
Repack repack_plan(const AxhipGemmParams &p) {
    const int64_t kvec = p.dtype == AXHIP_DTYPE_F32 ? 4 : 8;
    const bool pad_k = p.k % kvec != 0;
    Repack r{false, false, false, p.k};
    if ((p.trans_a || !p.trans_b || pad_k) && p.k >= 32 &&
        2.0 * static_cast<double>(p.m) * static_cast<double>(p.n) * static_cast<double>(p.k) * static_cast<double>(p.batch) >= double(1 << 30)) { // (about 70 us on the FMA kernel)
        r.on = true;
        r.kp = pad_k ? (p.k + 63) / 64 * 64 : p.k;
        r.a = p.trans_a || pad_k;
        r.b = !p.trans_b || pad_k;
    }
    return r;
}
size_t repack_bytes(const AxhipGemmParams &p) {
    const Repack r = repack_plan(p);
    if (!r.on) return 0;
    const size_t es = p.dtype == AXHIP_DTYPE_F32 ? 4 : 2;
    size_t n = 0;
    if (r.a) n += CallScratch::rounded(static_cast<size_t>(p.stride_a == 0 ? 1 : p.batch) * p.m * r.kp * es);
    if (r.b) n += CallScratch::rounded(static_cast<size_t>(p.stride_b == 0 ? 1 : p.batch) * p.n * r.kp * es);
    return n;
}
thread_local const char *last_kernel = "none";

int gemm_impl(const void *a, const void *b, void *c, const AxhipGemmParams *params, CallScratch *scratch_in, void *workspace, size_t workspace_bytes, void *stream);
} // namespace

extern "C" size_t axhip_gemm_workspace_bytes(const AxhipGemmParams *params) {
    if (!params || !valid_dtype(params->dtype) || params->m <= 0 || params->n <= 0 || params->k < 0 || params->batch <= 0) return 0;
    AxhipGemmParams part = *params;
    part.batch = std::min<int64_t>(part.batch, 65535); // larger batches run as consecutive launches that share the workspace
    return repack_bytes(part);
}

extern "C" int axhip_gemm(const void *a, const void *b, void *c, const AxhipGemmParams *params, void *stream) {
    return gemm_impl(a, b, c, params, nullptr, nullptr, 0, stream);
}

extern "C" const char *axhip_gemm_last_kernel(void) { return last_kernel; }

extern "C" int axhip_gemm_ws(const void *a, const void *b, void *c, const AxhipGemmParams *params, void *workspace, size_t workspace_bytes, void *stream) {
    return gemm_impl(a, b, c, params, nullptr, workspace, workspace_bytes, stream);
}

namespace {
// ---- 16-bit products: which kernel
// A stored along k, and everything within the 32-bit offsets the kernels address with.
bool takes_half_kernels(const AxhipGemmParams &p) {
    constexpr int64_t LD = int64_t(1) << 21, SIDE = int64_t(1) << 30;
    return !p.trans_a && p.k >= 8 && (p.trans_b || p.n >= 8) && p.m < SIDE && p.n < SIDE && p.k < SIDE && p.lda < LD && p.ldb < LD &&
           p.ldc < (int64_t(1) << 31) && (p.trans_b || (p.k + 64) * p.ldb < SIDE);
}
// rows of both operands on 16-byte boundaries and in whole 16-byte vectors
bool half_aligned(const AxhipGemmParams &p, const void *a, const void *b) {
    return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0 && (p.k | p.lda | p.ldb | p.stride_a | p.stride_b | (p.trans_b ? 0 : p.n)) % 8 == 0;
}

// The candidates with the time each takes, in us: start + k (per_k + per_k_full u) r + per_round (r - 1), r being the
// rounds its work-groups take on the 256 CUs (whole rounds of the tile kernels, of which a CU holds one; the small ones
// share a CU, and a part of a round costs about half of what is missing from a whole one) and u how full the first is.
// The coefficients are fitted to 300 products of m 16 .. 3000, n 128 .. 5120, k 128 .. 4096, bf16, operands from the
// caches: mean error 3 - 9 %, and the kernel picked is on average 1 % slower than the fastest of all.
struct HalfKernel {
    enum Kind { BIG256, TILE, SMALL } kind;
    int shape, waves;
    float start, per_k, per_k_full, per_round;
    bool nt, nn, ragged;
};
constexpr HalfKernel HALF_KERNELS[] = {
    {HalfKernel::BIG256, 0, 8, 7.0f, 0.0160f, 0.0057f, 4.0f, true, false, false},
    {HalfKernel::TILE, TILE_256x128, 8, 6.5f, 0.0080f, 0.0034f, 6.4f, true, true, false},
    {HalfKernel::TILE, TILE_192x128, 8, 5.7f, 0.0063f, 0.0024f, 4.9f, true, true, false},
    {HalfKernel::TILE, TILE_128x128, 8, 4.9f, 0.0048f, 0.0014f, 4.1f, true, true, false},
    {HalfKernel::TILE, TILE_64x128, 8, 4.9f, 0.0032f, 0.0009f, 3.7f, true, true, false},
    {HalfKernel::TILE, TILE_128x128, 8, 6.5f, 0.0080f, 0.0f, 5.9f, true, true, true}, // (through registers)
    {HalfKernel::SMALL, SMALL_64x64, 8, 4.35f, 0.00245f, 0.00148f, 3.6f, true, true, false},
    {HalfKernel::SMALL, SMALL_64x64, 4, 4.15f, 0.00324f, 0.00047f, 1.65f, true, true, false},
    {HalfKernel::SMALL, SMALL_32x64, 8, 3.50f, 0.00170f, 0.00085f, 2.3f, true, true, false},
    {HalfKernel::SMALL, SMALL_32x64, 4, 3.30f, 0.00210f, 0.00030f, 0.6f, true, true, false},
    {HalfKernel::SMALL, SMALL_16x64, 8, 3.19f, 0.00150f, 0.00035f, 0.77f, false, true, false},
    {HalfKernel::SMALL, SMALL_16x64, 4, 3.04f, 0.00183f, 0.00008f, 0.27f, false, true, false},
    {HalfKernel::SMALL, SMALL_32x32, 8, 3.07f, 0.00105f, 0.00045f, 0.76f, true, false, false},
    {HalfKernel::SMALL, SMALL_32x32, 4, 2.95f, 0.00148f, 0.00005f, 0.26f, true, false, false},
    {HalfKernel::SMALL, SMALL_32x16, 8, 2.92f, 0.00074f, 0.00032f, 0.33f, true, false, false},
    {HalfKernel::SMALL, SMALL_32x16, 4, 2.91f, 0.00102f, 0.00004f, 0.10f, true, false, false},
    {HalfKernel::SMALL, SMALL_16x16, 8, 2.95f, 0.00045f, 0.00024f, 0.19f, true, false, false},
    {HalfKernel::SMALL, SMALL_16x16, 4, 2.94f, 0.00069f, 0.00004f, 0.02f, true, false, false},
};

// Unaligned rows: what an operand whose rows start on odd elements, on other even ones, or on other multiples of four
// adds to the small kernels' time per element of k, and a quarter of it to the tile kernel's (18 products of k 75 .. 3582,
// which the kernels picked run in 0.91 of the time that one factor for all alignments led to).
float half_misalignment(int64_t ld) { return ld % 2 != 0 ? 0.55f : ld % 4 != 0 ? 0.45f : ld % 8 != 0 ? 0.1f : 0.0f; }

struct HalfChoice { const HalfKernel *best; float cost; };
// One candidate.  (The candidates are a parameter of the template so that their tiles are constants here: divisions by what a
// table holds took 0.5 us of the 3.5 that a small product costs its caller.)
template <size_t I> void consider_half_kernel(const AxhipGemmParams &p, bool aligned, float misaligned, HalfChoice &c) {
    constexpr const HalfKernel &h = HALF_KERNELS[I];
    if (p.trans_b ? !h.nt : !h.nn) return;
    if (h.kind != HalfKernel::SMALL && h.ragged == aligned) return;
    if (h.kind == HalfKernel::BIG256 && (p.k % TK != 0 || p.m < BIG || p.n < BIG || p.ldc >= (1 << 21))) return;
    constexpr uint32_t tm = h.kind == HalfKernel::BIG256 ? BIG : h.kind == HalfKernel::TILE ? TILE_GEOMETRY[h.kind == HalfKernel::TILE ? h.shape : 0].tm : SMALL_GEOMETRY[h.kind == HalfKernel::SMALL ? h.shape : 0].tm;
    constexpr uint32_t tn = h.kind == HalfKernel::BIG256 ? BIG : h.kind == HalfKernel::TILE ? TILE_GEOMETRY[h.kind == HalfKernel::TILE ? h.shape : 0].tn : SMALL_GEOMETRY[h.kind == HalfKernel::SMALL ? h.shape : 0].tn;
    const uint32_t rows = (static_cast<uint32_t>(p.m) + tm - 1) / tm, cols = (static_cast<uint32_t>(p.n) + tn - 1) / tn;
    if (!launch_fits(static_cast<int64_t>(rows) * cols + 7, 64 * h.waves)) return;
    const float k = static_cast<float>((p.k + 63) / 64 * 64);
    const float full = static_cast<float>(p.batch) * static_cast<float>(rows) * static_cast<float>(cols) * (1.0f / 256.0f);
    float r = 1.0f;
    if (full > 1.0f) {
        float whole = full < 1e9f ? static_cast<float>(static_cast<int>(full)) : full;
        if (whole < full) whole += 1.0f;
        r = h.kind == HalfKernel::SMALL ? 0.5f * (whole + full) : whole;
    }
    const float slower = aligned ? 1.0f : h.kind == HalfKernel::SMALL ? 1.0f + misaligned : 1.0f + 0.25f * misaligned;
    const float cost = h.start + k * (h.per_k + h.per_k_full * std::min(full, 1.0f)) * slower * r + h.per_round * (r - 1.0f);
    if (!c.best || cost < c.cost) c = {&h, cost};
}
template <size_t... I> const HalfKernel *choose_half_kernel(const AxhipGemmParams &p, bool aligned, std::index_sequence<I...>) {
    HalfChoice c{nullptr, 0.0f};
    const float misaligned = aligned ? 0.0f : half_misalignment(p.lda) + half_misalignment(p.ldb);
    (consider_half_kernel<I>(p, aligned, misaligned, c), ...);
    return c.best;
}
// (NULL: no kernel whose work-groups, as many as the product has tiles, can be launched at once)
const HalfKernel *choose_half_kernel(const AxhipGemmParams &p, bool aligned) {
    return choose_half_kernel(p, aligned, std::make_index_sequence<sizeof(HALF_KERNELS) / sizeof(HALF_KERNELS[0])>{});
}

// ---- fp32 products: which kernel
// The ring kernel's tiles, by fp32 products and by products of parts, with the time each takes, in us: start + k (per_k +
// (per_k_full + per_k_odd odd) u) r + per_round (r - 1), r being the rounds its work-groups take on the 256 CUs, u how full the
// first is (all CUs at work lower the clock) and odd 1 for rows off the 16-byte grid.
enum RingTile { RING_64x64, RING_64x128, RING_128x128_PARTS, RING_64x128_PARTS, RING_64x64_PARTS, RING_TILES };
struct F32RingTile { int tm, tn, tk; float start, per_k, per_k_full, per_round, per_k_odd; };
constexpr F32RingTile F32_RING_TILES[RING_TILES] = {{64, 64, 32, 4.25f, 0.0166f, 0.0f, 0.78f, 0.0f},
                                                    {64, 128, 32, 5.20f, 0.0320f, 0.0f, 1.66f, 0.0015f},
                                                    {128, 128, 32, 9.22f, 0.0271f, 0.0202f, 6.69f, 0.0f},
                                                    {64, 128, 64, 6.93f, 0.0183f, 0.0100f, 5.17f, 0.0005f},
                                                    {64, 64, 64, 4.85f, 0.0119f, 0.0041f, 3.32f, 0.0012f}};
struct F32Ring { int tile; float cost; };
// (one candidate; the candidates are a parameter of the template, as those of the 16-bit kernels are)
template <size_t I> void consider_f32_ring_tile(const AxhipGemmParams &p, float odd, F32Ring &best) {
    constexpr F32RingTile t = F32_RING_TILES[I];
    const float k = static_cast<float>((p.k + t.tk - 1) / t.tk * t.tk);
    const uint64_t tiles = ((static_cast<uint64_t>(p.m) + t.tm - 1) / t.tm) * ((static_cast<uint64_t>(p.n) + t.tn - 1) / t.tn) * static_cast<uint64_t>(p.batch);
    const float r = static_cast<float>(static_cast<int64_t>((tiles + 255) / 256)), u = tiles < 256 ? static_cast<float>(static_cast<int>(tiles)) * (1.0f / 256.0f) : 1.0f;
    const float cost = t.start + k * (t.per_k + (t.per_k_full + t.per_k_odd * odd) * u) * r + t.per_round * (r - 1.0f);
    if (I == 0 || cost < best.cost) best = {static_cast<int>(I), cost};
}
template <size_t... I> F32Ring f32_ring_tile(const AxhipGemmParams &p, std::index_sequence<I...>) {
    F32Ring best{0, 0.0f};
    const float odd = p.k % 4 != 0 || (!p.trans_b && p.n % 4 != 0) ? 1.0f : 0.0f;
    (consider_f32_ring_tile<I>(p, odd, best), ...);
    return best;
}
F32Ring f32_ring_tile(const AxhipGemmParams &p) { return f32_ring_tile(p, std::make_index_sequence<RING_TILES>{}); }
// A along k, offsets of 32 bits, rows of b as [k, n] of whole chunks or at least a tile (128 columns at most)
bool takes_f32_ring(const AxhipGemmParams &p, const void *a, const void *b) {
    return !p.trans_a && (p.trans_b || ((p.n % 4 == 0 || p.n >= 128) && p.n < (1 << 24) && (p.k + 64) * p.ldb < (int64_t(1) << 29))) && p.k >= 32 &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 3u) == 0 && p.lda < (1 << 21) && p.ldb < (1 << 21) && p.k < (1 << 24) &&
           p.m * p.n * p.batch >= 64 * 64 * 16 && f32_mfma_enabled();
}
// The time of the kernels of gemm_f32.hip in us, as for the 16-bit ones above: start + k (per_k + (per_k_full +
// per_k_odd) u) r + per_round (r - 1), per_k_odd for rows off the 16-byte grid.  Fitted with the ring kernel's to 260
// products of m 9 .. 8192, n 64 .. 8192, k 64 .. 8192 (mean error 2 - 4 % of the ring's, 6 - 10 % of these), those of parts to
// 400 with k from 32 (2 - 3 %).  Of 1200 products the one picked is 1.3 % slower than the fastest on average; they take 0.976 of the time that
// they take without the tiles of parts, 19 of them 2 % more or longer and 11 of these 5 % (33 x 8192 x 8192, b along k, 79 -> 90 us, the worst;
// 3264 x 1280 x 1536 100 -> 104);
// 2.3 times as fast as the ring and FMA kernels, which had the small ones to themselves:
// 99 x 1024 x 5120 104 -> 18 us, 186 x 640 x 958 35 -> 8, 48 x 384 x 2048 77 -> 6.3.  Large products with both operands
// along k stay on the ring: 2048^3 115 us against 188.
struct F32Kernel { float start, per_k, per_k_full, per_round, per_k_odd; };
constexpr F32Kernel F32_KERNELS[F32_SHAPES] = {
    {3.28f, 0.00144f, 0.00039f, 0.43f, 0.00063f}, {3.59f, 0.00249f, 0.00096f, 1.11f, 0.00074f}, {3.84f, 0.00524f, 0.00076f, 1.69f, 0.00091f}, {3.76f, 0.00472f, 0.00079f, 1.11f, 0.00138f},
    {4.59f, 0.00939f, 0.00112f, 3.91f, 0.00138f}, {6.25f, 0.01761f, 0.00329f, 6.68f, 0.00394f}, {5.40f, 0.00618f, 0.00378f, 3.44f, 0.00093f}};

template <size_t I> void consider_f32_kernel(const AxhipGemmParams &p, float k, float u, bool ring, int &best, float &best_cost) {
    constexpr F32Kernel h = F32_KERNELS[I];
    constexpr uint32_t tm = F32_GEOMETRY[I].tm, tn = F32_GEOMETRY[I].tn;
    const uint32_t rows = (static_cast<uint32_t>(p.m) + tm - 1) / tm, cols = (static_cast<uint32_t>(p.n) + tn - 1) / tn; // (m, n < 2^30)
    if (!launch_fits(static_cast<int64_t>(rows) * cols + 7, 512)) return; // (eight wavefronts a tile)
    const float full = static_cast<float>(p.batch) * static_cast<float>(rows) * static_cast<float>(cols) * (1.0f / 256.0f);
    const float r = full <= 1.0f ? 1.0f : 0.5f * (std::ceil(full) + full);
    // (b as [k, n]: the small tiles of fp32 products are slower, 78 x 4096 x 2048 27.3 us on 16 x 16 against 18.7 with b along k)
    const float per_k = I <= F32_32x32 && !p.trans_b ? 1.05f * h.per_k : h.per_k;
    const float cost = h.start + k * (per_k + (h.per_k_full + h.per_k_odd * u) * std::min(full, 1.0f)) * r + h.per_round * (r - 1.0f);
    if ((best < 0 && !ring) || cost < best_cost) { best_cost = cost; best = static_cast<int>(I); }
}
template <size_t... I> void consider_f32_kernels(const AxhipGemmParams &p, float k, float u, bool ring, int &best, float &best_cost, std::index_sequence<I...>) {
    (consider_f32_kernel<I>(p, k, u, ring, best, best_cost), ...);
}

// An F32Shape, or -1: the kernel that this product had otherwise (`ring`: the ring kernel, after `repacked` bytes were
// written and read if there are any; else the FMA kernel).
int choose_f32_kernel(const AxhipGemmParams &p, bool ring, double repacked) {
    constexpr int64_t SIDE = int64_t(1) << 30, LD = int64_t(1) << 31;
    // (below 64 K multiplications the FMA kernel is as fast: 17 x 70 x 33 3.5 us on either)
    if (p.trans_a || p.k < 32 || p.n < 4 || p.m >= SIDE || p.n >= SIDE || p.k >= SIDE || p.lda >= LD || p.ldb >= LD || p.ldc >= LD ||
        p.m * p.n * p.batch < 65536 / p.k || !f32_mfma_enabled())
        return -1;
    const float k = static_cast<float>(p.k), u = p.k % 4 != 0 || (!p.trans_b && p.n % 4 != 0) ? 1.0f : 0.0f;
    int best = -1;
    float best_cost = 0.0f;
    if (ring) best_cost = f32_ring_tile(p).cost + (repacked > 0.0 ? 4.7f + 2.1e-7f * static_cast<float>(repacked) : 0.0f);
    consider_f32_kernels(p, k, u, ring, best, best_cost, std::make_index_sequence<F32_SHAPES>{});
    return best;
}

int launch_big(const GemmArgs &g, bool bf, hipStream_t s) {
    const int tiles_m = static_cast<int>((g.M + BIG - 1) / BIG), tiles_n = static_cast<int>((g.N + BIG - 1) / BIG);
    constexpr size_t lds_bytes = 4 * BIG_TILEB;
    static const bool configured = [] {
        bool ok = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_mfma_nt_256_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) == hipSuccess;
        ok = ok && hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_mfma_nt_256_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) == hipSuccess;
        return ok;
    }();
    AXHIP_REQUIRE(configured, AXHIP_ERR_UNSUPPORTED, "axhip_gemm: cannot reserve %zu bytes of LDS", lds_bytes);
    launch_products(g, static_cast<int64_t>(tiles_m) * tiles_n, 512, 2, [&](const GemmArgs &part, unsigned grid) {
        if (bf) hipLaunchKernelGGL((gemm_mfma_nt_256_kernel<true>), dim3(grid), dim3(512), lds_bytes, s, part, tiles_m, tiles_n);
        else hipLaunchKernelGGL((gemm_mfma_nt_256_kernel<false>), dim3(grid), dim3(512), lds_bytes, s, part, tiles_m, tiles_n);
    });
    return AXHIP_OK;
}

TileArgs tile_args(const AxhipGemmParams &p, const void *a, const void *b, void *c) {
    TileArgs t{};
    t.a = a; t.b = b; t.c = c; t.bias = p.bias; t.residual = p.residual;
    t.sa = p.stride_a; t.sb = p.stride_b; t.sc = p.stride_c;
    t.M = static_cast<int>(p.m); t.N = static_cast<int>(p.n); t.K = static_cast<int>(p.k);
    t.lda = static_cast<int>(p.lda); t.ldb = static_cast<int>(p.ldb); t.ldc = static_cast<int>(p.ldc);
    t.epilogue = p.epilogue_op;
    t.batch = static_cast<int>(p.batch);
    return t;
}

int launch_half(const AxhipGemmParams &p, const void *a, const void *b, void *c, const HalfKernel &k, bool aligned, bool bf, hipStream_t s) {
    const TileArgs t = tile_args(p, a, b, c);
    if (k.kind == HalfKernel::SMALL) return launch_small(t, bf, !p.trans_b, k.shape, k.waves, s);
    return p.trans_b ? launch_tile_nt(t, bf, k.shape, aligned, s) : launch_tile_nn(t, bf, k.shape, aligned, s);
}

int gemm_impl(const void *a, const void *b, void *c, const AxhipGemmParams *params, CallScratch *scratch_in, void *workspace, size_t workspace_bytes, void *stream) {
    AXHIP_REQUIRE(params != nullptr, AXHIP_ERR_INVALID_ARG, "axhip_gemm: params is NULL");
    const AxhipGemmParams &p = *params;
    AXHIP_REQUIRE(valid_dtype(p.dtype), AXHIP_ERR_INVALID_ARG, "axhip_gemm: bad dtype %d", p.dtype);
    AXHIP_REQUIRE(p.m >= 0 && p.n >= 0 && p.k >= 0 && p.batch >= 0, AXHIP_ERR_INVALID_ARG, "axhip_gemm: negative extent");
    AXHIP_REQUIRE(p.lda >= 0 && p.ldb >= 0 && p.ldc >= p.n, AXHIP_ERR_INVALID_ARG, "axhip_gemm: bad leading dimension");
    AXHIP_REQUIRE(p.epilogue_op == 0 || p.epilogue_op == AXHIP_OP_RELU || p.epilogue_op == AXHIP_OP_GELU || p.epilogue_op == AXHIP_OP_SILU ||
                      p.epilogue_op == AXHIP_OP_SIGMOID || p.epilogue_op == AXHIP_OP_TANH,
                  AXHIP_ERR_INVALID_ARG, "axhip_gemm: unsupported epilogue op %d", p.epilogue_op);
    last_kernel = "empty";
    if (p.m == 0 || p.n == 0 || p.batch == 0) return AXHIP_OK;
    AXHIP_REQUIRE(a && b && c, AXHIP_ERR_INVALID_ARG, "axhip_gemm: NULL matrix");
    if (p.batch >= 65536) {
        // larger batches run as consecutive calls: the batch is a grid dimension of the FMA kernel (at most 65 535), and a
        // workspace has to hold the repacked operands of one call only
        const int64_t es = p.dtype == AXHIP_DTYPE_F32 ? 4 : 2;
        for (int64_t b0 = 0; b0 < p.batch; b0 += 65535) {
            AxhipGemmParams part = p;
            part.batch = std::min<int64_t>(65535, p.batch - b0);
            if (p.residual) part.residual = static_cast<const char *>(p.residual) + b0 * p.stride_c * es;
            const int rc_part = gemm_impl(static_cast<const char *>(a) + b0 * p.stride_a * es, static_cast<const char *>(b) + b0 * p.stride_b * es,
                                          static_cast<char *>(c) + b0 * p.stride_c * es, &part, nullptr, workspace, workspace_bytes, stream);
            if (rc_part) return rc_part;
        }
        return AXHIP_OK;
    }
    int rc = ensure_init();
    if (rc) return rc;
    hipStream_t s = resolve_stream(stream);

    // The matrix kernels read A along k, rows that start anywhere, and B either way (takes_half_kernels and takes_f32_ring say
    // where they do not).  An operand they do not take, A as [k, m] above all, leaves only the FMA kernel below, a hundred
    // times slower on a large product.  Such a product
    // is repacked first, into stream-ordered temporary memory (freed in stream order behind the product): the operand
    // that lies the other way is transposed; an unaligned k is zero-padded to the next multiple of 64 in both operands.
    const Repack rp = repack_plan(p);
    if (workspace) {
        const size_t need = repack_bytes(p);
        AXHIP_REQUIRE(workspace_bytes >= need, AXHIP_ERR_WORKSPACE, "axhip_gemm: the workspace holds %zu bytes, the call needs %zu (ask axhip_gemm_workspace_bytes)", workspace_bytes, need);
    }
    const bool f32 = p.dtype == AXHIP_DTYPE_F32;
    auto half_kernel = [&] { return !f32 && takes_half_kernels(p) ? choose_half_kernel(p, half_aligned(p, a, b)) : nullptr; };
    const bool repack = rp.on && !scratch_in && !(f32 ? takes_f32_ring(p, a, b) : half_kernel() != nullptr);
    const double repacked = repack ? 8.0 * static_cast<double>(p.batch) * static_cast<double>((rp.a ? p.m : 0) + (rp.b ? p.n : 0)) * static_cast<double>(p.k) : 0.0;
    const int f32_shape = f32 ? choose_f32_kernel(p, repack || takes_f32_ring(p, a, b), repacked) : -1;
    if (repack && f32_shape < 0) {
        const bool pad_k = rp.kp != p.k;
        const int64_t es = p.dtype == AXHIP_DTYPE_F32 ? 4 : 2, kp = rp.kp;
        AxhipGemmParams q = p;
        q.k = kp;
        CallScratch scratch(workspace, workspace_bytes, s);
        void *ta = nullptr, *tb = nullptr;
        // a contiguous [copies, rows, kp] image of an operand whose element (row, kk) lies at row * rs + kk * cs
        auto repacked = [&](const void *src, int64_t rows, int64_t rs, int64_t cs, int64_t batch_stride, void **out) -> int {
            const int64_t copies = batch_stride == 0 ? 1 : p.batch;
            const int rc_take = scratch.take(out, static_cast<size_t>(copies * rows * kp * es), "axhip_gemm");
            if (rc_take) return rc_take;
            const int64_t shape[3] = {copies, rows, p.k}, strides[3] = {batch_stride, rs, cs}, before[3] = {0, 0, 0}, after[3] = {0, 0, kp - p.k};
            if (pad_k) return axhip_pad(src, *out, p.dtype, 3, shape, strides, before, after, 0.0, stream);
            return axhip_strided_copy(src, p.dtype, *out, p.dtype, 3, shape, strides, stream);
        };
        if (rp.a) {
            rc = repacked(a, p.m, p.trans_a ? 1 : p.lda, p.trans_a ? p.lda : 1, p.stride_a, &ta);
            q.trans_a = 0; q.lda = kp; q.stride_a = p.stride_a == 0 ? 0 : p.m * kp;
        }
        if (!rc && rp.b) {
            rc = repacked(b, p.n, p.trans_b ? p.ldb : 1, p.trans_b ? 1 : p.ldb, p.stride_b, &tb);
            q.trans_b = 1; q.ldb = kp; q.stride_b = p.stride_b == 0 ? 0 : p.n * kp;
        }
        if (!rc) rc = gemm_impl(ta ? ta : a, tb ? tb : b, c, &q, &scratch, nullptr, 0, stream); // (q is not repacked again)
        const int freed = scratch.release();
        return rc ? rc : freed;
    }

    GemmArgs g{};
    g.a = a; g.b = b; g.c = c; g.bias = p.bias; g.residual = p.residual;
    g.dtype = p.dtype; g.epilogue = p.epilogue_op;
    g.M = p.m; g.N = p.n; g.K = p.k;
    g.a_rs = p.trans_a ? 1 : p.lda; g.a_cs = p.trans_a ? p.lda : 1;
    g.b_rs = p.trans_b ? 1 : p.ldb; g.b_cs = p.trans_b ? p.ldb : 1;
    g.ldc = p.ldc; g.sa = p.stride_a; g.sb = p.stride_b; g.sc = p.stride_c; g.batch = static_cast<int>(p.batch);

    const bool half = p.dtype != AXHIP_DTYPE_F32;
    auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
    const bool nt = !p.trans_a && p.trans_b && p.k % 8 == 0 && p.lda % 8 == 0 && p.ldb % 8 == 0 && p.stride_a % 8 == 0 &&
                    p.stride_b % 8 == 0 && al16(a) && al16(b) && p.ldc < (1 << 21);
    // fp32: always.  A lane adds up every 64th product; the kernels with shared tiles add up an eighth of k, or k-tile after
    // k-tile, and come out 1.5 to 2.9 times as far from the exact sums, although most products are faster there (W from HBM,
    // here and there: 8 x 4096 x 4096 26.3 us, error 1.6e-7, and 14.9, 4.1e-7; 8 x 1280 x 1280 6.1, 1.1e-7 and 5.3, 2.4e-7;
    // 6 x 2048 x 2048 8.3, 1.2e-7 and 7.0, 2.9e-7; 4 x 20096 x 560 15.8, 0.9e-7 and 18.3, 1.7e-7).
    // 16 bits: its wavefronts, one per row of W, each read all of x.  With the outputs, m n, grow the reads from L1, and the other
    // kernels share them (W from HBM, us here and there: 4 x 2048 x 4096 7.8 and 8.6, 6 x 2048 x 4096 9.2 and 8.4, 8 x 768 x
    // 3072 5.5 and 5.6, 3 x 4096 x 4096 10.8 and 9.8).  With one or two rows W alone counts (1 x 51865 x 4096 70 and 84), unless
    // rows of W so short that a wavefront has hardly anything to wait for meet so many of them (1 x 51865 x 512 16.6 and 12.3,
    // 2 x 51865 x 1280 29.9 and 26.0, 1 x 51865 x 1280 25.0 and 26.2).
    const int64_t w_elems = p.n * p.k;
    const bool alone = !takes_half_kernels(p); // (else the FMA kernel)
    const bool skinny_pays = p.m <= 8 && (f32 || p.m * p.n <= 8192 || (p.m <= 2 && p.m * p.n <= 64 * p.k) || alone);
    const bool f32_nt = p.dtype == AXHIP_DTYPE_F32 && !p.trans_a && p.trans_b && p.k % 4 == 0 && p.lda % 4 == 0 && p.ldb % 4 == 0 && al16(a) && al16(b);
    // (the kernel carries leading dimensions as 32-bit element counts)
    const bool ld32 = p.lda < (int64_t(1) << 31) && p.ldb < (int64_t(1) << 31) && p.ldc < (int64_t(1) << 31);
    if (((half && nt) || f32_nt) && p.batch == 1 && skinny_pays && p.k >= 256 && launch_fits(p.n / 4 + 1, 256) && p.k < (1 << 30) && ld32 && skinny_enabled()) {
        // a decoding step: bound by one read of W
        SkinnyArgs k{};
        k.x = a; k.w = b; k.c = c; k.bias = p.bias; k.residual = p.residual;
        k.dtype = p.dtype; k.epilogue = p.epilogue_op;
        k.N = static_cast<int>(p.n); k.K = static_cast<int>(p.k);
        k.ldx = static_cast<int>(p.lda); k.ldw = static_cast<int>(p.ldb); k.ldc = static_cast<int>(p.ldc);
        // A wavefront per row of W, each lane with four 16-byte pieces of it requested at a time: the fewest rows are
        // streamed at once, each in the longest runs (1 x 16384 x 16384: 88.8 us = 76 % of the HBM peak against
        // 95.2 / 101.2 us with two / four rows per wavefront; 1 x 50304 x 4096: 64.2 against 68.4 / 71.8 us; 1 x 4096 x
        // 4096 from the caches: 4.3 against 6.6 / 7.1 us).  Two rows per wavefront share the reads of x where two or
        // more rows of x meet a large W (2 x 16384 x 16384: 97.4 against 102.7 us).
        // AXHIP_GEMM_SKINNY_ROWS=1|2|4 (read once) forces the count.
        static const int forced_rows = [] { const char *e = std::getenv("AXHIP_GEMM_SKINNY_ROWS"); return e ? std::atoi(e) : 0; }();
        const int rows_per_wave = forced_rows == 1 || forced_rows == 2 || forced_rows == 4 ? forced_rows : (p.m >= 2 && w_elems >= (int64_t(64) << 20)) ? 2 : 1;
        const unsigned blocks = static_cast<unsigned>((p.n + 4 * rows_per_wave - 1) / (4 * rows_per_wave));
        launch_skinny(k, static_cast<int>(p.m), rows_per_wave, blocks, s);
        last_kernel = "skinny";
    } else if (const HalfKernel *k = half_kernel()) {
        const bool aligned = half_aligned(p, a, b), bf = p.dtype == AXHIP_DTYPE_BF16;
        last_kernel = k->kind == HalfKernel::BIG256 ? "big" : k->kind == HalfKernel::TILE ? "tile" : "small";
        rc = k->kind == HalfKernel::BIG256 ? launch_big(g, bf, s) : launch_half(p, a, b, c, *k, aligned, bf, s);
        if (rc) return rc;
    } else if (f32_shape >= 0) {
        static constexpr const char *names[F32_SHAPES] = {"f32_16x16", "f32_16x32", "f32_16x64", "f32_32x32", "f32_32x64", "f32_64x64", "f32_32x64_parts"};
        last_kernel = names[f32_shape];
        rc = launch_f32_direct(tile_args(p, a, b, c), !p.trans_b, f32_shape, s);
        if (rc) return rc;
    } else if (f32 && takes_f32_ring(p, a, b)) {
        // the fp32 MFMA, b along k or [k, n]
        auto launch = [&](auto kernel, int tm_rows, int tn_cols, int threads, size_t lds_bytes) -> int {
            static std::mutex mu;
            static std::set<const void *> configured;
            {
                std::lock_guard<std::mutex> lk(mu);
                if (!configured.count(reinterpret_cast<const void *>(kernel))) {
                    AXHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
                    configured.insert(reinterpret_cast<const void *>(kernel));
                }
            }
            // (more tiles than a launch may have: a strip of the longer side at a time; rows where b is [k, n], of which n < 2^24)
            const int64_t tiles_m = (p.m + tm_rows - 1) / tm_rows, tiles_n = (p.n + tn_cols - 1) / tn_cols;
            const bool by_rows = !p.trans_b || tiles_m >= tiles_n;
            const int64_t across = by_rows ? tiles_n : tiles_m, size = by_rows ? p.m : p.n;
            AXHIP_REQUIRE(launch_fits(across + 7, threads), AXHIP_ERR_UNSUPPORTED, "axhip_gemm: too many tiles");
            const int64_t strip = products_per_launch(across, threads) * (by_rows ? tm_rows : tn_cols);
            for (int64_t at = 0; at < size; at += strip) {
                GemmArgs part = g;
                (by_rows ? part.M : part.N) = std::min(strip, size - at);
                const int64_t in_c = 4 * at * (by_rows ? g.ldc : 1);
                if (by_rows) part.a = static_cast<const char *>(g.a) + 4 * at * g.a_rs;
                else part.b = static_cast<const char *>(g.b) + 4 * at * g.b_cs;
                part.c = static_cast<char *>(g.c) + in_c;
                if (g.residual) part.residual = static_cast<const char *>(g.residual) + in_c;
                if (g.bias && !by_rows) part.bias = static_cast<const char *>(g.bias) + 4 * at;
                const int rows = static_cast<int>((part.M + tm_rows - 1) / tm_rows), cols = static_cast<int>((part.N + tn_cols - 1) / tn_cols);
                launch_products(part, static_cast<int64_t>(rows) * cols, threads, 4, [&](const GemmArgs &some, unsigned grid) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds_bytes, s, some, rows, cols); });
            }
            return AXHIP_OK;
        };
        int rc2;
        static constexpr const char *names[RING_TILES] = {"ring_64x64", "ring_64x128", "ring_128x128_parts", "ring_64x128_parts", "ring_64x64_parts"};
        const int tile = f32_ring_tile(p).tile;
        last_kernel = names[tile];
        switch (tile) {
#define AXHIP_RING(TM, TN, KF, LW, LDS) \
    rc2 = p.trans_b ? launch(gemm_mfma_f32_ring_kernel<TM, TN, KF, LW, false>, TM, TN, 64 * (4 + LW), LDS) : launch(gemm_mfma_f32_ring_kernel<TM, TN, KF, LW, true>, TM, TN, 64 * (4 + LW), LDS)
        case RING_64x64: AXHIP_RING(64, 64, 0, 4, (ring_lds_bytes<64, 64>())); break;
        case RING_64x128: AXHIP_RING(64, 128, 0, 4, (ring_lds_bytes<64, 128>())); break;
        case RING_128x128_PARTS: AXHIP_RING(128, 128, 32, 4, (split_lds_bytes<128, 128, 32, 4>())); break;
        case RING_64x128_PARTS: AXHIP_RING(64, 128, 64, 4, (split_lds_bytes<64, 128, 64, 4>())); break;
        default: AXHIP_RING(64, 64, 64, 8, (split_lds_bytes<64, 64, 64, 8>())); break;
#undef AXHIP_RING
        }
        if (rc2) return rc2;
    } else {
        last_kernel = "fma";
        dim3 grid(static_cast<unsigned>((p.n + 15) / 16), static_cast<unsigned>((p.m + 15) / 16), static_cast<unsigned>(p.batch));
        AXHIP_REQUIRE(grid.y < 65536, AXHIP_ERR_UNSUPPORTED, "axhip_gemm: m too large for the generic kernel");
        AXHIP_REQUIRE(launch_fits((p.n + 15) / 16, 16 * 16), AXHIP_ERR_UNSUPPORTED, "axhip_gemm: n too large for the generic kernel");
        hipLaunchKernelGGL(gemm_generic_kernel, grid, dim3(256), 0, s, g);
    }
    AXHIP_CHECK_HIP(hipGetLastError());
    return AXHIP_OK;
}
} // namespace
