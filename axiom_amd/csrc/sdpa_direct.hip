// Attention without shared LDS tiles, for few query rows and short sequences.
//
// A work-group owns one block of query rows; its eight waves take 32-key steps of the keys in turn and meet once, at
// the end, through LDS.  V goes from memory straight into the operands of the matrix instructions.  What makes a detour
// through LDS unnecessary is that the order in which keys and head dimensions run through an MFMA is free as long as
// both operands agree on it:
//   S^T = K Q^T    leaves lane (l16, g) with query l16 and keys 4 g + i of a 16-key sub-tile;
//   O^T = V^T P^T  then takes these keys as k-slots (the probabilities are the B operand as they stand), and lane
//                  (l16, g) needs, of V, the rows of ITS keys and, for output tile t, dimension l16 * (D / 16) + t --
//                  so its whole share of V is a few rows of 16-byte runs that it loads itself, and the transpose is
//                  byte permutes between its own registers.
#include "sdpa.hpp"
#include "gemm_tile_device.hpp" // wave_lds_fence

namespace axhip {

namespace {

// K can be loaded as fragments -- 16 bytes of each of 16 rows side by side, four times the lines of an instruction that
// loads whole rows -- or as rows, through 8 KiB of LDS that are the wave's own.  The rows are the faster ones where a
// work-group's latency counts (fp32 B1 H8 S512 10.3 -> 9.5 us, 96 slices of 700 keys 7.1 -> 6.2, 12 of 300 of 128 dims 6.4 ->
// 5.5), the fragments by 1 - 4 % where the chip streams (128 slices of 16384 keys of 128 178 against 180 us, 256 of 4096
// 89.7 against 93.0).
// 16-byte chunk c of row r of a stage, CH chunks a row, spread so that neither the rows written nor the 16 rows of a
// fragment read meet on a bank:
constexpr int DIRECT_STAGE = 8192;
template <int CH> __device__ __forceinline__ int stage_at(int r, int c) { return (r * CH + (c ^ (CH == 8 ? (r >> 1) & 7 : r & 15))) * 16; }

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <bool BF16> __device__ __forceinline__ f32x4_t mfma_16x16x32(uint4_t a, uint4_t b, f32x4_t c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}

// maximum / sum over the four lane groups that share a query (lanes l16, l16 + 16, + 32, + 48)
__device__ __forceinline__ float group_max(float x) {
    return across32(across16(x, lanes_max), lanes_max);
}
__device__ __forceinline__ float group_sum(float x) {
    return across32(across16(x, lanes_add), lanes_add);
}

// The waves' states of a block of `rows` query rows: [wave][row][D + 4] accumulators, then [wave][row] reference maxima
// and denominators.
template <int D> constexpr int direct_lds_bytes(int rows) { return DIRECT_WAVES * rows * (D + 4 + 2) * 4; }

// The merged state of four columns of one query row.
struct Merged { f32x4_t o; float top, den; };
template <int D> __device__ __forceinline__ Merged direct_merge(const float *lds, int rows, int q, int d) {
    const float *m = lds + DIRECT_WAVES * rows * (D + 4), *l = m + DIRECT_WAVES * rows;
    Merged r{{0.0f, 0.0f, 0.0f, 0.0f}, NEG_INF_F, 0.0f};
#pragma unroll
    for (int w = 0; w < DIRECT_WAVES; ++w) r.top = fmaxf(r.top, m[w * rows + q]);
    if (r.top == NEG_INF_F) return r; // no key of this row is left
#pragma unroll
    for (int w = 0; w < DIRECT_WAVES; ++w) {
        const float scale = __builtin_amdgcn_exp2f(m[w * rows + q] - r.top);
        r.o += scale * *reinterpret_cast<const f32x4_t *>(&lds[(w * rows + q) * (D + 4) + d]);
        r.den += scale * l[w * rows + q];
    }
    return r;
}

} // namespace

// ------------------------------------------------------------- 16-bit, decoding
// Up to DIRECT_ROWS query rows against a long run of keys: bound by one read of K and V.  A step of a wave is 32 keys,
// 16 loads of 16 bytes (D = 64: 4, and 8 of 8), requested one step ahead, so a work-group has 128 KiB on the way or in use
// (D = 128) and needs no barrier to keep it so.  Of the 16 query columns of the MFMAs most are empty; they cost nothing
// that the loads would not cost anyway (16 MFMAs of 16 cycles for 16 KiB).
template <bool BF16, int D, bool SPLIT, bool STAGED>
__global__ __launch_bounds__(64 * DIRECT_WAVES, 2) void sdpa_direct16_kernel(const SdpaArgs a) {
    constexpr int KJ = D / 32; // 32-dim fragments of a K row
    constexpr int NT = D / 16; // output tiles; elements of V a lane holds per key
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, l16 = lane % 16, g = lane / 16;
    const int bh = SPLIT ? blockIdx.x / a.ksplit : blockIdx.x, split = SPLIT ? blockIdx.x % a.ksplit : 0;
    const int b = bh / a.H, h = bh % a.H;
    const uint16_t *Q = static_cast<const uint16_t *>(a.q) + b * a.qs[0] + h * a.qs[1];
    const uint16_t *K = static_cast<const uint16_t *>(a.k) + b * a.ks[0] + h * a.ks[1];
    const uint16_t *V = static_cast<const uint16_t *>(a.v) + b * a.vs[0] + h * a.vs[1];
    const int dv = a.D, rows = a.Sq;

    // keys past the end of the sequence and dims past the head size read as zero (the lanes that would fetch such dims
    // aim past the descriptors)
    const int krow = static_cast<int>(a.ks[2]) * 2, vrow = static_cast<int>(a.vs[2]) * 2;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(K), 0, (a.Skv - 1) * krow + dv * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(V), 0, (a.Skv - 1) * vrow + dv * 2, 0x00020000);
    constexpr int OUTSIDE = static_cast<int>(0x80000000u);
    constexpr int CH = D / 8, RL = WAVE / CH, KL = DIRECT_KEYS / RL; // chunks of a row, rows of a load, loads of a step
    const int k_row = lane / CH, k_ch = lane % CH;
    static_assert(KL == 2 * KJ, "the fragments of a step");
    int koff[STAGED ? 1 : KJ]; // of the row; of the fragments of a row
#pragma unroll
    for (int j = 0; j < (STAGED ? 1 : KJ); ++j) {
        const int d = STAGED ? k_ch * 8 : 32 * j + 8 * g;
        koff[j] = d < dv ? (STAGED ? k_row : l16) * krow + d * 2 : OUTSIDE;
    }
    unsigned char *stage = reinterpret_cast<unsigned char *>(lds) + wave * DIRECT_STAGE;
    const int voff = l16 * NT < dv ? 4 * g * vrow + l16 * NT * 2 : OUTSIDE;

    uint4_t qf[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j)
        qf[j] = l16 < rows && 32 * j + 8 * g < dv ? *reinterpret_cast<const uint4_t *>(Q + l16 * a.qs[2] + 32 * j + 8 * g) : uint4_t{0, 0, 0, 0};

    const int k_first = SPLIT ? split * a.kchunk : 0, k_end = SPLIT ? min(a.Skv, k_first + a.kchunk) : a.Skv;
    uint4_t kf[KL];
    uint32_t vf[8][NT / 2];
    auto load = [&](int at) {
#pragma unroll
        for (int n = 0; n < KL; ++n)
            kf[n] = __builtin_amdgcn_raw_buffer_load_b128(kr, koff[STAGED ? 0 : n % KJ] + (at + (STAGED ? RL * n : 16 * (n / KJ))) * krow, 0, 0);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int off = voff + (at + 16 * (e / 4) + e % 4) * vrow;
            if constexpr (D == 128) {
                const uint4_t t = __builtin_amdgcn_raw_buffer_load_b128(vr, off, 0, 0);
                vf[e][0] = t.x; vf[e][1] = t.y; vf[e][2] = t.z; vf[e][3] = t.w;
            } else {
                const uint2_t t = __builtin_amdgcn_raw_buffer_load_b64(vr, off, 0, 0);
                vf[e][0] = t.x; vf[e][1] = t.y;
            }
        }
    };

    f32x4_t oacc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) oacc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = NEG_INF_F, l_run = 0.0f;
    constexpr int STRIDE = DIRECT_KEYS * DIRECT_WAVES;
    int at = k_first + DIRECT_KEYS * wave;
    if (at < k_end) load(at);
    while (at < k_end) {
        uint4_t kc[STAGED ? 1 : KL];
        uint32_t vc[8][NT / 2];
#pragma unroll
        for (int n = 0; n < KL; ++n) {
            if constexpr (STAGED) *reinterpret_cast<uint4_t *>(stage + stage_at<CH>(RL * n + k_row, k_ch)) = kf[n];
            else kc[n] = kf[n];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int w = 0; w < NT / 2; ++w) vc[e][w] = vf[e][w];
        const int now = at;
        at += STRIDE;
        if (at < k_end) load(at);

        f32x4_t s[2];
        if constexpr (STAGED) wave_lds_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            s[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < KJ; ++j) {
                uint4_t k;
                if constexpr (STAGED) k = *reinterpret_cast<const uint4_t *>(stage + stage_at<CH>(16 * u + l16, 4 * j + g));
                else k = kc[u * KJ + j];
                s[u] = mfma_16x16x32<BF16>(k, qf[j], s[u]);
            }
        }
        if constexpr (STAGED) wave_lds_fence();
        if (now + DIRECT_KEYS > a.Skv) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (now + 16 * u + 4 * g + i >= a.Skv) s[u][i] = NEG_INF_F;
        }
        float top = NEG_INF_F;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) top = fmaxf(top, s[u][i]);
        const float m_new = fmaxf(m_run, group_max(top) * a.scale_log2e);
        if (__builtin_amdgcn_ballot_w64(m_new - m_run > RESCALE_THRESHOLD) != 0) {
            const float alpha = m_new == NEG_INF_F ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < NT; ++t) oacc[t] *= alpha;
        }
        const float m_use = m_run == NEG_INF_F ? 0.0f : m_run;
        uint4_t p;
#pragma unroll
        for (int w = 0; w < 4; ++w) { // slot 8 g + e of the second product is key 4 g + e % 4 of sub-tile e / 4
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[w / 2][2 * (w % 2)], a.scale_log2e, -m_use));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[w / 2][2 * (w % 2) + 1], a.scale_log2e, -m_use));
            p[w] = pack2<BF16>(p0, p1);
            l_run = add_pair<BF16>(p[w], l_run); // the denominator sums exactly what the MFMA multiplies
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            uint4_t vt;
#pragma unroll
            for (int w = 0; w < 4; ++w) vt[w] = __builtin_amdgcn_perm(vc[2 * w + 1][t / 2], vc[2 * w][t / 2], t % 2 ? 0x07060302u : 0x05040100u);
            oacc[t] = mfma_16x16x32<BF16>(vt, p, oacc[t]);
        }
    }

    // tile t, element i of lane (l16, g): query l16, dim (4 g + i) * NT + t
    const float l_tot = group_sum(l_run);
    if constexpr (STAGED) __syncthreads(); // the stages become the states
    if (l16 < rows) {
        float *row = &lds[(wave * rows + l16) * (D + 4)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t4 = 0; t4 < NT / 4; ++t4)
                *reinterpret_cast<f32x4_t *>(&row[(4 * g + i) * NT + 4 * t4]) = f32x4_t{oacc[4 * t4][i], oacc[4 * t4 + 1][i], oacc[4 * t4 + 2][i], oacc[4 * t4 + 3][i]};
        if (g == 0) {
            lds[DIRECT_WAVES * rows * (D + 4) + wave * rows + l16] = m_run;
            lds[DIRECT_WAVES * rows * (D + 5) + wave * rows + l16] = l_tot;
        }
    }
    __syncthreads();
    for (int item = tid; item < rows * (D / 4); item += 64 * DIRECT_WAVES) {
        const int q = item / (D / 4), d = item % (D / 4) * 4;
        const Merged r = direct_merge<D>(lds, rows, q, d);
        const f32x4_t o = r.o * (r.den > 0.0f ? 1.0f / r.den : 0.0f);
        if constexpr (SPLIT) {
            const int64_t slot = (static_cast<int64_t>(bh) * a.ksplit + split) * rows + q;
            *reinterpret_cast<f32x4_t *>(a.opart + slot * D + d) = o;
            if (d == 0) a.lse[slot] = r.den > 0.0f ? r.top + __builtin_amdgcn_logf(r.den) : NEG_INF_F; // (v_log_f32: base 2)
        } else if (d < dv) {
            uint16_t *O = static_cast<uint16_t *>(a.o) + b * a.os[0] + h * a.os[1] + q * a.os[2];
            *reinterpret_cast<uint2_t *>(O + d) = uint2_t{pack2<BF16>(o[0], o[1]), pack2<BF16>(o[2], o[3])};
        }
    }
}

int launch_sdpa_direct16(const SdpaArgs &a, bool bf16, hipStream_t s) {
    const bool split = a.ksplit > 0;
    const unsigned grid = static_cast<unsigned>(a.B * a.H * (split ? a.ksplit : 1));
    const bool narrow = a.D <= 64;
    // (from 200 slices on the chip streams: 240 slices of 1102 keys of 64 14.6 us by fragments, 14.8 by rows; 4096 of 16 keys
    // 20.6 and 22.2)
    const bool staged = !split && a.B * a.H < 200;
    constexpr int stages = DIRECT_WAVES * DIRECT_STAGE;
    static_assert(direct_lds_bytes<128>(DIRECT_ROWS) <= stages && stages <= 65536, "the states take the place of the stages");
    const int lds = staged ? stages : narrow ? direct_lds_bytes<64>(a.Sq) : direct_lds_bytes<128>(a.Sq);
#define AXHIP_DIRECT(BF, DD)                                                                                              \
    do {                                                                                                                  \
        const dim3 threads(64 * DIRECT_WAVES);                                                                            \
        if (split) hipLaunchKernelGGL((sdpa_direct16_kernel<BF, DD, true, false>), dim3(grid), threads, lds, s, a);       \
        else if (staged) hipLaunchKernelGGL((sdpa_direct16_kernel<BF, DD, false, true>), dim3(grid), threads, lds, s, a); \
        else hipLaunchKernelGGL((sdpa_direct16_kernel<BF, DD, false, false>), dim3(grid), threads, lds, s, a);            \
    } while (0)
    if (bf16 && narrow) AXHIP_DIRECT(true, 64);
    else if (bf16) AXHIP_DIRECT(true, 128);
    else if (narrow) AXHIP_DIRECT(false, 64);
    else AXHIP_DIRECT(false, 128);
#undef AXHIP_DIRECT
    AXHIP_CHECK_HIP(hipGetLastError());
    return AXHIP_OK;
}

// out = sum_s 2^(lse_s - max lse) O_s / sum_s 2^(lse_s - max lse) over the `ksplit` (at most 64) partial results of a
// (batch, head, query row).  A wave per row: lane s weighs partial s, then groups of D / 4 lanes take the partials in
// turn, four columns a lane, eight loads in flight.
template <bool BF16, int D>
__global__ __launch_bounds__(64) void sdpa_merge_kernel(const SdpaArgs a) {
    constexpr int LANES = D / 4, TAKE = WAVE / LANES, AHEAD = 8;
    const int lane = threadIdx.x, d = lane % LANES * 4, first = lane / LANES;
    const int64_t row = blockIdx.x, bh = row / a.Sq; // (batch, head, query row)
    const int q = static_cast<int>(row - bh * a.Sq);
    const float lse = lane < a.ksplit ? a.lse[(bh * a.ksplit + lane) * a.Sq + q] : NEG_INF_F;
    // (requested before the weights are known: one trip to memory for both; with the exchanges between lanes kept out of LDS,
    // 20 heads of 1152 x 128 8.0 -> 7.7 us, 8 of 16384 x 128 16.4 -> 15.8)
    f32x4_t o[AHEAD];
    auto fetch = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int s = min(s0 + TAKE * i + first, a.ksplit - 1);
            o[i] = *reinterpret_cast<const f32x4_t *>(a.opart + ((bh * a.ksplit + s) * a.Sq + q) * D + d);
        }
    };
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);
    const float top = wave_max(lse), weight = top == NEG_INF_F ? 0.0f : __builtin_amdgcn_exp2f(lse - top), den = wave_sum(weight);
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0;;) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int s = s0 + TAKE * i + first;
            const float w = __shfl(weight, min(s, WAVE - 1), WAVE); // (0 past the last partial, except that 63 may be one)
            acc += (s < a.ksplit ? w : 0.0f) * o[i];
        }
        s0 += TAKE * AHEAD;
        if (s0 >= a.ksplit) break;
        fetch(s0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (LANES <= 16) acc[c] = across16(acc[c], lanes_add);
        acc[c] = across32(acc[c], lanes_add);
    }
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    if (first == 0 && d < a.D) {
        uint16_t *orow = static_cast<uint16_t *>(a.o) + (bh / a.H) * a.os[0] + (bh % a.H) * a.os[1] + static_cast<int64_t>(q) * a.os[2];
        *reinterpret_cast<uint2_t *>(orow + d) = uint2_t{pack2<BF16>(acc[0] * inv, acc[1] * inv), pack2<BF16>(acc[2] * inv, acc[3] * inv)};
    }
}

void launch_sdpa_merge(const SdpaArgs &a, bool bf16, int D, hipStream_t s) {
    const unsigned grid = static_cast<unsigned>(a.B * a.H * a.Sq);
    if (D == 64) {
        if (bf16) hipLaunchKernelGGL((sdpa_merge_kernel<true, 64>), dim3(grid), dim3(64), 0, s, a);
        else hipLaunchKernelGGL((sdpa_merge_kernel<false, 64>), dim3(grid), dim3(64), 0, s, a);
    } else {
        if (bf16) hipLaunchKernelGGL((sdpa_merge_kernel<true, 128>), dim3(grid), dim3(64), 0, s, a);
        else hipLaunchKernelGGL((sdpa_merge_kernel<false, 128>), dim3(grid), dim3(64), 0, s, a);
    }
}

// ------------------------------------------------------------- fp32, short sequences
// The same on v_mfma_f32_16x16x4_f32 for fp32 inputs: fp32 products and fp32 accumulation.  Problems of few 32-row
// blocks leave most CUs without work on sdpa_mfma_f32_kernel; this one has twice the blocks (16 rows) and eight waves on
// each, and nothing between a wave and its keys but one load latency.
template <int D, bool HAS_MASK>
__global__ __launch_bounds__(64 * DIRECT_WAVES, 2) void sdpa_direct_f32_kernel(const SdpaArgs a) {
    constexpr int SUB = D == 64 ? 2 : 1;  // 16-key sub-tiles of a step (what two steps' registers allow)
    constexpr int KJ = D / 16, VH = D / 64;
    constexpr int ROWS = 16, KEYS = 16 * SUB, STRIDE = KEYS * DIRECT_WAVES;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, l16 = lane % 16, g = lane / 16;
    const int BH = a.B * a.H;
    int bh, qb;
    if (BH % 8 == 0) { // one (batch, head) stays on one XCD, whose L2 then holds its K / V
        bh = (blockIdx.x / 8 / a.nqb) * 8 + blockIdx.x % 8;
        qb = blockIdx.x / 8 % a.nqb;
    } else {
        bh = blockIdx.x / a.nqb;
        qb = blockIdx.x % a.nqb;
    }
    if (a.causal) qb = a.nqb - 1 - qb; // heaviest blocks first
    const int b = bh / a.H, h = bh % a.H;
    const float *Q = static_cast<const float *>(a.q) + b * a.qs[0] + h * a.qs[1];
    const float *K = static_cast<const float *>(a.k) + b * a.ks[0] + h * a.ks[1];
    const float *V = static_cast<const float *>(a.v) + b * a.vs[0] + h * a.vs[1];
    const uint8_t *M = HAS_MASK ? a.mask + b * a.ms[0] + h * a.ms[1] : nullptr;
    const int dv = a.D, q0 = qb * ROWS, q = q0 + l16;
    const bool q_ok = q < a.Sq;

    const int krow = static_cast<int>(a.ks[2]) * 4, vrow = static_cast<int>(a.vs[2]) * 4;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(K), 0, (a.Skv - 1) * krow + dv * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(V), 0, (a.Skv - 1) * vrow + dv * 4, 0x00020000);
    constexpr int OUTSIDE = static_cast<int>(0x80000000u);
    constexpr int CH = D / 4, RL = WAVE / CH, KL = KEYS / RL; // chunks of a row, rows of a load, loads of a step
    static_assert(KEYS * CH * 16 == DIRECT_STAGE, "a step of K");
    const int k_row = lane / CH, k_ch = lane % CH;
    const int koff = k_ch * 4 < dv ? k_row * krow + k_ch * 16 : OUTSIDE;
    unsigned char *stage = reinterpret_cast<unsigned char *>(lds) + wave * DIRECT_STAGE;
    int voff[VH];
#pragma unroll
    for (int v = 0; v < VH; ++v) voff[v] = 64 * v + 4 * l16 < dv ? 4 * g * vrow + (64 * v + 4 * l16) * 4 : OUTSIDE;

    f32x4_t qf[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j)
        qf[j] = q_ok && 16 * j + 4 * g < dv ? *reinterpret_cast<const f32x4_t *>(Q + q * a.qs[2] + 16 * j + 4 * g) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int k_end = a.causal ? min(a.Skv, q0 + ROWS) : a.Skv;
    uint4_t kf[KL];
    f32x4_t vf[SUB][4][VH];
    uint32_t mf[SUB]; // the mask bytes of this lane's four keys
    auto load = [&](int at) {
#pragma unroll
        for (int n = 0; n < KL; ++n) kf[n] = __builtin_amdgcn_raw_buffer_load_b128(kr, koff + (at + RL * n) * krow, 0, 0);
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int v = 0; v < VH; ++v)
                    vf[u][i][v] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(vr, voff[v] + (at + 16 * u + i) * vrow, 0, 0));
            if constexpr (HAS_MASK) {
                mf[u] = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) { // (rows and keys that do not exist read a byte that does)
                    const int key = min(at + 16 * u + 4 * g + i, a.Skv - 1);
                    mf[u] |= static_cast<uint32_t>(M[static_cast<int64_t>(min(q, a.Sq - 1)) * a.Skv + key]) << (8 * i);
                }
            }
        }
    };

    f32x4_t oacc[VH][4];
#pragma unroll
    for (int v = 0; v < VH; ++v)
#pragma unroll
        for (int c = 0; c < 4; ++c) oacc[v][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = NEG_INF_F, l_run = 0.0f;
    int at = KEYS * wave;
    if (at < k_end) load(at);
    while (at < k_end) {
        f32x4_t vc[SUB][4][VH];
        uint32_t mc[SUB];
#pragma unroll
        for (int n = 0; n < KL; ++n) *reinterpret_cast<uint4_t *>(stage + stage_at<CH>(RL * n + k_row, k_ch)) = kf[n];
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int v = 0; v < VH; ++v) vc[u][i][v] = vf[u][i][v];
            mc[u] = HAS_MASK ? mf[u] : 0;
        }
        const int now = at;
        at += STRIDE;
        if (at < k_end) load(at);

        f32x4_t s[SUB];
#pragma unroll
        for (int u = 0; u < SUB; ++u) s[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
            f32x4_t kc[SUB];
#pragma unroll
            for (int u = 0; u < SUB; ++u) kc[u] = *reinterpret_cast<const f32x4_t *>(stage + stage_at<CH>(16 * u + l16, 4 * j + g));
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int u = 0; u < SUB; ++u) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[u][c], qf[j][c], s[u], 0, 0, 0);
        }
        wave_lds_fence();
        if (HAS_MASK || now + KEYS > a.Skv || (a.causal && now + KEYS - 1 > q0)) {
            const int last = a.causal ? min(a.Skv - 1, q) : a.Skv - 1;
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool masked = now + 16 * u + 4 * g + i > last || ((mc[u] >> (8 * i)) & 0xFFu) != 0;
                    s[u][i] = masked ? NEG_INF_F : s[u][i];
                }
        }
        float top = NEG_INF_F;
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) top = fmaxf(top, s[u][i]);
        const float m_new = fmaxf(m_run, group_max(top) * a.scale_log2e);
        if (__builtin_amdgcn_ballot_w64(m_new - m_run > RESCALE_THRESHOLD) != 0) {
            const float alpha = m_new == NEG_INF_F ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int v = 0; v < VH; ++v)
#pragma unroll
                for (int c = 0; c < 4; ++c) oacc[v][c] *= alpha;
        }
        const float m_use = m_run == NEG_INF_F ? 0.0f : m_run;
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][i], a.scale_log2e, -m_use));
                l_run += p;
#pragma unroll
                for (int v = 0; v < VH; ++v)
#pragma unroll
                    for (int c = 0; c < 4; ++c) oacc[v][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vc[u][i][v][c], p, oacc[v][c], 0, 0, 0);
            }
    }

    // tile (v, c), element i of lane (l16, g): query l16, dim 64 v + 4 (4 g + i) + c
    const float l_tot = group_sum(l_run);
    __syncthreads(); // the stages become the states
    float *row = &lds[(wave * ROWS + l16) * (D + 4)];
#pragma unroll
    for (int v = 0; v < VH; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4_t *>(&row[64 * v + 16 * g + 4 * i]) = f32x4_t{oacc[v][0][i], oacc[v][1][i], oacc[v][2][i], oacc[v][3][i]};
    if (g == 0) {
        lds[DIRECT_WAVES * ROWS * (D + 4) + wave * ROWS + l16] = m_run;
        lds[DIRECT_WAVES * ROWS * (D + 5) + wave * ROWS + l16] = l_tot;
    }
    __syncthreads();
    for (int item = tid; item < ROWS * (D / 4); item += 64 * DIRECT_WAVES) {
        const int r = item / (D / 4), d = item % (D / 4) * 4;
        if (q0 + r >= a.Sq || d >= dv) continue;
        const Merged m = direct_merge<D>(lds, ROWS, r, d);
        float *O = static_cast<float *>(a.o) + b * a.os[0] + h * a.os[1] + static_cast<int64_t>(q0 + r) * a.os[2];
        *reinterpret_cast<f32x4_t *>(O + d) = m.o * (m.den > 0.0f ? 1.0f / m.den : 0.0f);
    }
}

template <int D> static int launch_direct_f32(const SdpaArgs &a, hipStream_t s) {
    constexpr int stages = DIRECT_WAVES * DIRECT_STAGE, states = direct_lds_bytes<D>(16), lds = stages > states ? stages : states;
    static const hipError_t attr = [] {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&sdpa_direct_f32_kernel<D, false>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        return e != hipSuccess ? e : hipFuncSetAttribute(reinterpret_cast<const void *>(&sdpa_direct_f32_kernel<D, true>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    }();
    AXHIP_CHECK_HIP(attr);
    const unsigned grid = static_cast<unsigned>(a.nqb) * static_cast<unsigned>(a.B * a.H);
    if (a.mask) hipLaunchKernelGGL((sdpa_direct_f32_kernel<D, true>), dim3(grid), dim3(64 * DIRECT_WAVES), lds, s, a);
    else hipLaunchKernelGGL((sdpa_direct_f32_kernel<D, false>), dim3(grid), dim3(64 * DIRECT_WAVES), lds, s, a);
    AXHIP_CHECK_HIP(hipGetLastError());
    return AXHIP_OK;
}

int launch_sdpa_direct_f32(const SdpaArgs &a, hipStream_t s) { return a.D <= 64 ? launch_direct_f32<64>(a, s) : launch_direct_f32<128>(a, s); }

} // namespace axhip
