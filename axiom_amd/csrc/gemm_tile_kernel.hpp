// ------------------------------------------------------- middle-sized products
// C = A B (+ bias) (+ residual), activation: bf16 / f16, A [M, K] along k, B [N, K] along k (NT) or [K, N] as matmul(a, b)
// has it (NN).  Work-group tile TM x TN, k-tiles of TK in an S-stage ring in LDS.
//
// What bounds such a product is not the memory system (with every operand byte in the caches the kernel this one
// replaces took the same time) but what one wavefront per SIMD serialises: a burst of tile loads, each held for the
// 16 bytes x 64 lanes / 64 bytes per clock the CU's load path takes, then LDS reads, then MFMAs.  So:
//   * two wavefronts per SIMD, and they do not split the tile further but the k-tile: WK groups of wavefronts each own
//     whole 16 MI x 64 blocks for a part of every k-tile.  A wavefront's block sets what it reads from LDS per MFMA,
//     and LDS reads (128 bytes per clock) are the second bound: 256 x 128 tiles read 96 KiB per 64 of k against 128 KiB
//     with eight disjoint 64 x 64 blocks.  The groups' sums meet in LDS once, at the end.
//   * every LDS read and every tile load sits between two MFMAs (scheduling fences pin the order); A fragments are
//     refilled behind their row's last MFMA, B fragments are double-buffered.  The barrier sits after the first
//     fragment row of a k-tile's last k-step: by then every wavefront has read the whole tile, so its stage takes the
//     tile S ahead, and the reads turn to the next tile.
//   * LDS rows of A (and of B, NT) are the TK elements of a k-tile row with the 16-byte chunk index XOR-ed by the row;
//     rows of B (NN) are TN elements of one k, fragments read through ds_read_b64_tr_b16, the chunk index XOR-ed so
//     that the sixteen rows of such a read meet all banks.
// DMA: tiles go L2 -> LDS directly (buffer_load ... lds).  Otherwise (rows off the 16-byte grid, K or N not whole
// vectors) through registers: unaligned 16-byte loads of one tile in flight while the previous is multiplied; the last
// chunk of a row is fetched as the 16 bytes that end with the row and shifted into place.
#pragma once
#include "gemm_tile.hpp"
#include "gemm_tile_device.hpp"

#include <type_traits>

namespace axhip {
namespace {

template <bool BF16> __device__ __forceinline__ float tile_widen(uint32_t h) { return BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h); }

// The wavefront's MB blocks of 16 x 64 sums -> C.  They pass through the wavefront's own LDS (`stage`, 4 KiB per block)
// so that a lane holds eight consecutive columns of a row: whole 128-byte lines per store, 16-byte reads of bias and
// residual -- and so that the code is one short loop: these kernels run for a few microseconds, in which every
// instruction that is not in a loop is fetched from memory once, and the fully unrolled form (a copy per block and
// activation) took longer than the products it belonged to.  Columns below n_low are another work-group's.
template <bool BF16, int MB>
__device__ __forceinline__ void tile_store_blocks(const TileArgs &g, const float4_t (&own)[MB][4], int m_base, int n_base, int n_low, int64_t coff, int lane, unsigned char *stage) {
    const int l16 = lane % 16, g4 = lane / 16;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<float4_t *>(stage + (16 * i + l16) * 256 + (((4 * j + g4) ^ l16) * 16)) = own[i][j];
    wave_lds_fence();
    const int q = lane & 7, col = n_base + 8 * q;
    const int first = max(0, n_low - col), last = min(8, g.N - col); // this lane's columns of C: col + [first, last)
    if (first >= last) return;
    const bool whole = first == 0 && last == 8;
    uint16_t *c = static_cast<uint16_t *>(g.c) + coff + col;
    const uint16_t *res = static_cast<const uint16_t *>(g.residual) + coff + col, *bias = static_cast<const uint16_t *>(g.bias) + col;
    float b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = 0.0f;
    if (g.bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (whole || (e >= first && e < last)) b[e] = tile_widen<BF16>(bias[e]);
    }
#pragma unroll 1
    for (int r = lane >> 3; r < 16 * MB; r += 8) {
        const int row = m_base + r;
        if (row >= g.M) break;
        float x[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4_t v = *reinterpret_cast<const float4_t *>(stage + r * 256 + (((2 * q + h) ^ (r & 15)) * 16));
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * h + e] = v[e] + b[4 * h + e];
        }
        const int64_t at = static_cast<int64_t>(row) * g.ldc;
        if (g.residual) {
            if (whole) {
                const uint4_t t = reinterpret_cast<const uint4_unaligned_t *>(res + at)->v;
                const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] += tile_widen<BF16>((w[e / 2] >> (16 * (e % 2))) & 0xFFFFu);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (e >= first && e < last) x[e] += tile_widen<BF16>(res[at + e]);
            }
        }
        gemm_epilogue16_all(g.epilogue, x);
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) w[e / 2] = BF16 ? pack_bf16x2(x[e], x[e + 1]) : pack_f16x2(x[e], x[e + 1]);
        if (whole) { // (any alignment: element by element, 975 x 51865 x 384 took 1.4 times as long on these kernels, 140 us instead of 65 on the 256 x 256 one)
            reinterpret_cast<uint4_unaligned_t *>(c + at)->v = uint4_t{w[0], w[1], w[2], w[3]};
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (e >= first && e < last) c[at + e] = static_cast<uint16_t>(w[e / 2] >> (16 * (e % 2)));
        }
    }
}

template <bool BF16, bool NN, bool DMA, int MI, int WM, int WN, int WK, int TK, int S>
__global__ __launch_bounds__(64 * WM * WN * WK, 1) void gemm_tile_kernel(const TileArgs g) {
    constexpr int NW = WM * WN * WK, TM = 16 * MI * WM, TN = 64 * WN;
    constexpr int KS = TK / 32 / WK;                      // k-steps of 32 per k-tile and wavefront
    constexpr int AROWB = TK * 2, ACH = TK / 8;           // bytes / 16-byte chunks per LDS row of A
    constexpr int BROWB = NN ? TN * 2 : TK * 2, BCH = BROWB / 16;
    constexpr int STAGEB = (TM + TN) * TK * 2, ABYTES = TM * TK * 2;
    constexpr int NLA = TM * TK * 2 / 1024 / NW, NLB = TN * TK * 2 / 1024 / NW, NL = NLA + NLB; // 1 KiB loads per wavefront and k-tile
    static_assert(KS >= 1 && NLA >= 1 && NLB >= 1 && MI >= 4 && MI % WK == 0, "tile");
    static_assert((NW * 64 / ACH) % 16 == 0 && (NN ? (NW * 64 / BCH) % 16 == 0 : true), "the XOR of a lane's row must not depend on the load");
    extern __shared__ __attribute__((aligned(1024))) unsigned char tile_lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int l16 = lane % 16, g4 = lane / 16;
    const int wk = wave / (WM * WN), wt = wave % (WM * WN), wm = (wt / WN) * 16 * MI, wn = (wt % WN) * 64;

    // the tiles of a product run down groups of GR tile rows, so that an XCD's L2 sees a compact block of C and each panel of
    // A and B few times
    const int tiles_m = (g.M + TM - 1) / TM, tiles_n = (g.N + TN - 1) / TN;
    int product;
    const int t = tile_of_work_group(tiles_m * tiles_n, g.batch, product);
    if (t < 0) return;
    constexpr int GR = TM >= 128 ? 4 : 8;
    const int group = t / (GR * tiles_n), first_m = group * GR;
    const int gsz = min(GR, tiles_m - first_m);
    const int rem = t - group * GR * tiles_n;
    const int m0 = (first_m + rem % gsz) * TM, n_low = (rem / gsz) * TN;
    // (through registers, NN: the last column tile is moved left to end with the rows, so that no chunk of B reaches past
    // one; the columns it shares with its neighbour are the neighbour's to store)
    const int n0 = NN && !DMA ? max(0, min(n_low, g.N - TN)) : n_low;
    const int64_t bz = product;
    const uint16_t *A = static_cast<const uint16_t *>(g.a) + bz * g.sa + static_cast<int64_t>(m0) * g.lda;
    const uint16_t *B = static_cast<const uint16_t *>(g.b) + bz * g.sb + (NN ? static_cast<int64_t>(n0) : static_cast<int64_t>(n0) * g.ldb);
    const int rows_a = min(TM, g.M - m0), cols_b = min(TN, g.N - n0);

    // ---- tile loads: load n of a wavefront moves chunks 64 (n NW + wave) + lane of the tile's LDS image
    const int a_row = (wave * 64 + lane) / ACH, a_pos = lane % ACH;
    const int a_src = a_pos ^ (TK == 64 ? (a_row >> 1) & 7 : a_row & 15); // the chunk that belongs at this position
    const int b_row = (wave * 64 + lane) / BCH, b_pos = lane % BCH;       // (NN: row = k, chunks along n)
    auto b_xor = [](int row) -> int {
        if constexpr (!NN) return TK == 64 ? (row >> 1) & 7 : row & 15;
        else if constexpr (TN == 128) return 2 * ((row & 3) | (((row >> 3) & 1) << 2));
        else return 2 * (((row >> 1) & 1) | (((row >> 3) & 1) << 1));
    };
    const int b_src = b_pos ^ b_xor(b_row);
    constexpr int A_STEP = NW * 64 / ACH, B_STEP = NW * 64 / BCH; // rows between a wavefront's consecutive loads
    constexpr int OUT_OF_RANGE = 0x7FFFFFF0;
    const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(tile_lds));
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(lds_base + wave * 1024);

    // DMA: offsets of this lane's chunks; a row past the tile's valid ones lies past the descriptor's extent
    const int4_t arsrc = tile_rsrc(A, ((rows_a - 1) * g.lda + g.K) * 2);
    const int4_t brsrc = tile_rsrc(B, NN ? 0x7FFFFFE0 : ((cols_b - 1) * g.ldb + g.K) * 2);
    int a_voff[NLA], b_voff[NLB];
    if constexpr (DMA) {
#pragma unroll
        for (int n = 0; n < NLA; ++n) a_voff[n] = (a_row + n * A_STEP) * g.lda * 2 + a_src * 16;
#pragma unroll
        for (int n = 0; n < NLB; ++n) {
            b_voff[n] = (b_row + n * B_STEP) * g.ldb * 2 + b_src * 16;
            if (NN && n0 + 8 * b_src >= g.N) b_voff[n] = OUT_OF_RANGE;
        }
    }
    auto dma_load = [&](int kt, int stage_off, int n) { // n: 0 .. NLA - 1 of A, then of B; past the last k-tile every lane is out of range
        const int k_left = g.K - kt * TK, k_at = k_left > 0 ? kt * TK * 2 : 0;
        if (n < NLA) {
            const int v = 8 * a_src < k_left ? a_voff[n < NLA ? n : 0] : OUT_OF_RANGE;
            tile_load_to_lds(arsrc, lds_wave + stage_off + n * NW * 1024, v, k_at);
        } else {
            const int nb = n - NLA < NLB ? n - NLA < 0 ? 0 : n - NLA : 0;
            const bool ok = NN ? b_row + nb * B_STEP < k_left : 8 * b_src < k_left;
            tile_load_to_lds(brsrc, lds_wave + stage_off + ABYTES + nb * NW * 1024, ok ? b_voff[nb] : OUT_OF_RANGE, NN ? k_at * g.ldb : k_at);
        }
    };
    // through registers (rows past the tile's end repeat its last one: they are not stored)
    constexpr int R = DMA ? 1 : 4; // k-tiles in flight in registers
    uint4_t regs[R][NL];
    uint32_t r_off[NL];
    if constexpr (!DMA) {
#pragma unroll
        for (int n = 0; n < NLA; ++n) r_off[n] = static_cast<uint32_t>(min(a_row + n * A_STEP, rows_a - 1)) * g.lda * 2;
#pragma unroll
        for (int n = 0; n < NLB; ++n)
            r_off[NLA + n] = NN ? static_cast<uint32_t>(min(8 * b_src, g.N - n0 - 8)) * 2 : static_cast<uint32_t>(min(b_row + n * B_STEP, cols_b - 1)) * g.ldb * 2;
    }
    auto reg_load = [&](int set, int kt, int n) { // (past the last k-tile: the row's end, or the last row, again)
        const char *base = reinterpret_cast<const char *>(n < NLA ? A : B);
        uint32_t off = r_off[n];
        if (NN && n >= NLA) off += static_cast<uint32_t>(min(kt * TK + b_row + (n - NLA) * B_STEP, g.K - 1)) * g.ldb * 2;
        else off += static_cast<uint32_t>(min(kt * TK + 8 * (n < NLA ? a_src : b_src), g.K - 8)) * 2;
        regs[set][n] = reinterpret_cast<const uint4_unaligned_t *>(base + off)->v;
    };
    auto chunk_at = [&](int stage_off, int n) { return reinterpret_cast<uint4_t *>(tile_lds + stage_off + (n < NLA ? n : n - NLA) * NW * 1024 + (n < NLA ? 0 : ABYTES) + wave * 1024 + lane * 16); };
    const int nk = (g.K + TK - 1) / TK;
    // (k-tiles past the last one, which the unrolled loop multiplies too, are zeros)
    auto reg_write = [&](int set, int kt, int stage_off, int n) { *chunk_at(stage_off, n) = kt < nk ? regs[set][n] : uint4_t{0, 0, 0, 0}; };
    // the last k-tile, where it reaches past the end of k (and every one of NN rows shorter than the tile): this lane's
    // chunks, already in LDS, are put in place
    auto mend = [&](int kt, int stage_off) {
        if (!(kt == nk - 1 && nk * TK > g.K) && !(NN && g.N < TN && kt < nk)) return;
#pragma unroll
        for (int n = 0; n < NL; ++n) {
            uint4_t v = *chunk_at(stage_off, n);
            if (NN && n >= NLA) {
                v = tile_row_chunk_in_place(v, 8 * b_src, g.N - n0);
                if (kt * TK + b_row + (n - NLA) * B_STEP >= g.K) v = uint4_t{0, 0, 0, 0};
            } else {
                v = tile_row_chunk_in_place(v, kt * TK + 8 * (n < NLA ? a_src : b_src), g.K);
            }
            *chunk_at(stage_off, n) = v;
        }
    };

    // ---- fragment reads
    int fa_off[KS], fb_off[KS][NN ? 2 : 1][NN ? 4 : 1];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int ks = wk * KS + s;
        fa_off[s] = (wm + l16) * AROWB + (((4 * ks + g4) ^ (TK == 64 ? (l16 >> 1) & 7 : l16 & 15)) * 16);
        if constexpr (!NN) {
            fb_off[s][0][0] = ABYTES + (wn + l16) * BROWB + (((4 * ks + g4) ^ b_xor(l16)) * 16);
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = 32 * ks + 8 * g4 + 4 * h + (l16 >> 2);
#pragma unroll
                for (int j = 0; j < 4; ++j) // 8-byte piece l16 & 3 of the 32 bytes of columns wn + 16 j ..
                    fb_off[s][h][j] = ABYTES + k * BROWB + (((wn / 8 + 2 * j + ((l16 & 3) >> 1)) ^ b_xor(k)) * 16) + (l16 & 1) * 8;
            }
        }
    }
    float4_t acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    uint4_t fa[MI], fb[2][4];
    auto read_a = [&](int stage_off, int s, int i) { fa[i] = *reinterpret_cast<const uint4_t *>(tile_lds + stage_off + fa_off[s] + 16 * i * AROWB); };
    auto read_b = [&](int slot, int stage_off, int s, int j) {
        if constexpr (!NN) {
            fb[slot][j] = *reinterpret_cast<const uint4_t *>(tile_lds + stage_off + fb_off[s][0][0] + 16 * j * BROWB);
        } else {
            const uint2_t lo = tile_read_tr(tile_lds + stage_off + fb_off[s][0][j]), hi = tile_read_tr(tile_lds + stage_off + fb_off[s][1][j]);
            fb[slot][j] = uint4_t{lo.x, lo.y, hi.x, hi.y};
        }
    };
    auto mfma = [&](int slot, int i, int j) { // (B fragment) x (A fragment)^T: the lane holds four consecutive columns of one row of C
        if constexpr (BF16)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fb[slot][j]), __builtin_bit_cast(bf16x8_t, fa[i]), acc[i][j], 0, 0, 0);
        else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, fb[slot][j]), __builtin_bit_cast(half8_t, fa[i]), acc[i][j], 0, 0, 0);
    };
#define AXHIP_FENCE() __builtin_amdgcn_sched_barrier(0)
    // s_waitcnt vmcnt(n) with the other counters left alone
#define AXHIP_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | 0x0F70 | (((n) >> 4) << 14))
    static_assert(NL * (S - 1) < 64, "vmcnt is a 6-bit counter");
    if constexpr (DMA) {
#pragma unroll
        for (int st = 0; st < S; ++st)
#pragma unroll
            for (int n = 0; n < NL; ++n) dma_load(st, st * STAGEB, n);
        AXHIP_VMCNT(NL * (S - 1)); // tile 0 has landed
    } else {
        static_assert(DMA || (S == 2 && KS == 1 && R == 4), "through registers: two stages in LDS, four k-tiles in registers");
        // k-tile t travels in register set (t - 2) & 3; the first two go to LDS at once
#pragma unroll
        for (int t0 = 0; t0 < 4; ++t0)
            if (t0 < 2 || t0 < nk) {
#pragma unroll
                for (int n = 0; n < NL; ++n) reg_load((t0 + 2) & 3, t0, n);
            }
#pragma unroll
        for (int t0 = 0; t0 < 2; ++t0) {
#pragma unroll
            for (int n = 0; n < NL; ++n) reg_write(t0 + 2, t0, t0 * STAGEB, n);
            mend(t0, t0 * STAGEB);
            if (t0 + 4 < nk) {
#pragma unroll
                for (int n = 0; n < NL; ++n) reg_load(t0 + 2, t0 + 4, n);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MI; ++i) read_a(0, 0, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) read_b(0, 0, 0, j);

    int cur = 0; // offset of k-tile kt's stage
    auto tile = [&](auto phase_tag, auto last_tag, int kt) { // phase: kt modulo the unrolling; last (through registers): nothing left to load
        constexpr bool LAST = decltype(last_tag)::value;
        constexpr int P = decltype(phase_tag)::value & 1, SET = DMA ? 0 : decltype(phase_tag)::value % R; // set SET holds k-tile kt + 2
        const int next = cur + STAGEB == S * STAGEB ? 0 : cur + STAGEB;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            constexpr int SLOTS = (MI - 1) * 4; // MFMAs behind the barrier of the last k-step
            const int slot = (P + s) & 1;
            const bool last = s == KS - 1;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                if (last && i == 1) {
                    if constexpr (DMA) AXHIP_VMCNT(NL * (S - 2)); // this wavefront's share of tile kt + 1 has landed
                    __syncthreads();                              // ... everyone's has, and tile kt is no longer read
                    AXHIP_FENCE();
                    read_a(next, 0, 0);
                    AXHIP_FENCE();
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    mfma(slot, i, j);
                    AXHIP_FENCE();
                    if (!last) {
                        if (j == 2 && i < 4) {
                            read_b(slot ^ 1, cur, s + 1, i);
                            AXHIP_FENCE();
                        }
                        if (j == 3) {
                            read_a(cur, s + 1, i);
                            AXHIP_FENCE();
                        }
                    } else if (i >= 1) {
                        const int q = (i - 1) * 4 + j;
                        constexpr int PERIOD = SLOTS / NL > 0 ? SLOTS / NL : 1;
                        if (q % 2 == 0 && q <= 6) {
                            read_b(slot ^ 1, next, 0, q / 2);
                            AXHIP_FENCE();
                        }
                        if (DMA && q % PERIOD == PERIOD - 1 && q / PERIOD < NL) {
                            dma_load(kt + S, cur, q / PERIOD);
                            AXHIP_FENCE();
                        }
                        if (!DMA && q % PERIOD == PERIOD - 1 && q / PERIOD < NL) {
                            reg_write(SET, kt + 2, cur, q / PERIOD);
                            AXHIP_FENCE();
                        }
                        if (j == 3) {
                            read_a(next, 0, i);
                            AXHIP_FENCE();
                        }
                    }
                }
            }
        }
        if constexpr (!DMA) {
            mend(kt + 2, cur);
            if constexpr (!LAST) {
#pragma unroll
                for (int n = 0; n < NL; ++n) reg_load(SET, kt + 2 + R, n);
            }
            AXHIP_FENCE();
        }
        cur = next;
    };
    if constexpr (!DMA) {
        // (No branch inside: the compiler would wait for every load in flight where the paths meet.  The tiles that are
        // already in registers when nothing is left to load go through a loop of their own: unaligned loads are half
        // as fast as aligned ones, and those past the end made 10 of the 13 that a product of three k-tiles took.)
        auto four = [&](auto last_tag, int kt) {
            tile(std::integral_constant<int, 0>{}, last_tag, kt);
            tile(std::integral_constant<int, 1>{}, last_tag, kt + 1);
            tile(std::integral_constant<int, 2>{}, last_tag, kt + 2);
            tile(std::integral_constant<int, 3>{}, last_tag, kt + 3);
        };
        int kt = 0;
        for (; kt + 2 + R < nk; kt += 4) four(std::false_type{}, kt);
        for (; kt < nk; kt += 4) four(std::true_type{}, kt);
    } else if constexpr (KS % 2 == 0) {
        for (int kt = 0; kt < nk; ++kt) tile(std::integral_constant<int, 0>{}, std::false_type{}, kt);
    } else {
        for (int kt = 0; kt < nk; kt += 2) {
            tile(std::integral_constant<int, 0>{}, std::false_type{}, kt);
            if (kt + 1 < nk) tile(std::integral_constant<int, 1>{}, std::false_type{}, kt + 1);
        }
    }
#undef AXHIP_FENCE

    // ---- the WK groups' sums meet in LDS: group w finishes row blocks [w MB, (w + 1) MB) of its wavefront tile
    AXHIP_VMCNT(0); // no load of this wavefront is still on its way into the ring
#undef AXHIP_VMCNT
    __syncthreads();
    constexpr int MB = MI / WK;
    float4_t own[MB][4];
    auto part = [&](int owner, int source, int i) -> unsigned char * { // 4 KiB: block i of `owner`, from `source` (!= owner)
        const int src = source - (source > owner ? 1 : 0);
        return tile_lds + ((((wt * WK + owner) * (WK - 1) + src) * MB + i) * 4096);
    };
    if constexpr (WK > 1) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int owner = i / MB;
            if (owner != wk) {
                unsigned char *p = part(owner, wk, i % MB);
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<float4_t *>(p + j * 1024 + lane * 16) = acc[i][j];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int w = 0; w < WK; ++w)
        if (wk == w) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) own[i][j] = acc[w * MB + i][j];
        }
    if constexpr (WK > 1) {
#pragma unroll
        for (int src = 0; src < WK - 1; ++src)
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const unsigned char *p = tile_lds + ((((wt * WK + wk) * (WK - 1) + src) * MB + i) * 4096);
#pragma unroll
                for (int j = 0; j < 4; ++j) own[i][j] += *reinterpret_cast<const float4_t *>(p + j * 1024 + lane * 16);
            }
    }
    // (the blocks that a wavefront has just read are its staging area)
    unsigned char *stage = tile_lds + (WK > 1 ? (wt * WK + wk) * (WK - 1) * MB * 4096 : wave * MB * 4096);
    tile_store_blocks<BF16, MB>(g, own, m0 + wm + wk * MB * 16, n0 + wn, n_low, bz * g.sc, lane, stage);
}

// bytes of LDS: the ring, or what the groups exchange at the end where that is more
template <int MI, int WM, int WN, int WK, int TK, int S> constexpr size_t tile_lds_bytes() {
    const size_t ring = size_t(S) * (16 * MI * WM + 64 * WN) * TK * 2;
    const size_t parts = WK > 1 ? size_t(WM * WN) * WK * (WK - 1) * (MI / WK) * 4096 : size_t(WM * WN) * MI * 4096;
    return ring > parts ? ring : parts;
}

template <bool BF16, bool NN, bool DMA, int MI, int WM, int WN, int WK, int TK, int S>
int launch_tile_kernel(const TileArgs &g, hipStream_t s) {
    constexpr size_t lds = tile_lds_bytes<MI, WM, WN, WK, TK, S>();
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    const auto kernel = gemm_tile_kernel<BF16, NN, DMA, MI, WM, WN, WK, TK, S>;
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    AXHIP_CHECK_HIP(configured);
    constexpr int TM = 16 * MI * WM, TN = 64 * WN;
    const int64_t tiles = static_cast<int64_t>((g.M + TM - 1) / TM) * ((g.N + TN - 1) / TN);
    AXHIP_REQUIRE(launch_fits(tiles + 7, 64 * WM * WN * WK), AXHIP_ERR_UNSUPPORTED, "axhip_gemm: too many tiles");
    launch_products(g, tiles, 64 * WM * WN * WK, 2, [&](const TileArgs &part, unsigned grid) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * WM * WN * WK), lds, s, part); });
    return AXHIP_OK;
}

} // namespace
} // namespace axhip
