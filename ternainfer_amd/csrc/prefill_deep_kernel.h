// The MFMA-tiled kernel for grids that leave a CU with few workgroups (prefill_packed_kernel.h has the one for full chips).
//
// What bounds such a launch: what one wave does in a row.  A step's matrix instructions take 256 - 512 clocks of a wave; in the
// kernel for full chips, which counts on three more waves on the SIMD, the step of a lone wave takes 800 - 1000 clocks, because an
// operand read waits an LDS trip for every group of matrix instructions (64 clocks of work).  Here
//   * a step's operands are read from LDS while the step before multiplies;
//   * the wait + barrier for the next stage stands in the middle of a step: half its matrix instructions are under way when a wave waits
//     for the others, and the operands read behind it have the other half to arrive;
//   * a stage is 128 columns of the tile's activations (direct loads, 16-byte pieces XOR-swizzled) AND of its weights (2-bit words,
//     1 KB per 32 features, wave-private, one direct load; one LDS read per step and operand): half as many steps and barriers
//     for bf16, and no register ring;
//   * with at most one workgroup per CU it has two sets of four waves (KS = 2): each takes half of K with stages of its own, and in
//     the end each finishes one of the two row tiles -- two waves per SIMD and half the steps in a row;
//   * one wait + barrier per step; D - 1 stages in flight (more than three bought nothing).  The steps whose third next stage does
//     not exist are another loop: the same conditions in the main one cost 3 - 5 %;
//   * with two halves of K, what the epilogue reads is requested behind the first stages, and the sums and result rows go to stages that
//     nobody reads any more: one barrier behind the loop instead of three.
// Measured, us, kernel for full chips / this one, 64 x 128 tiles: QKV M = 512 bf16 17.9 / 13.1, int8 11.2 / 9.5; gate+up M = 256
// bf16 20.2 / 19.4, int8 12.9 / 12.2; O M = 1024 bf16 19.5 / 18.1, int8 12.6 / 11.7; at 640 tiles (O M = 2048) 26.6 / 29.9.
// Halves of K: gate+up M = 100 int8 9.8 -> 9.0, QKV M = 400 int8 9.5 -> 8.7, bf16 12.6 -> 12.0, O M = 600 int8 9.5 -> 8.4 (at 257 - 512
// tiles they lose 3 - 5 us).
// Barrier in the middle, nothing loaded past the end, epilogue requested ahead, us before -> after: int8 QKV M = 300 8.6 -> 8.0, O M = 500
// 8.4 -> 7.9, gate+up M = 128 9.1 -> 8.6, down M = 500 15.8 -> 14.7, M = 1200 N = 1024 K = 448 4.7 -> 4.5; bf16 QKV M = 300 11.8 -> 11.1,
// O M = 500 11.6 -> 11.1, M = 1200 N = 1024 K = 448 5.3 -> 4.8; at two workgroups a CU QKV M = 1000 int8 15.1 -> 14.6, bf16 23.7 -> 23.2.
// Of a step's 945 clocks (two halves of K, int8) 534 are matrix instructions; without direct loads it takes 700, without the barrier 800,
// without operand reads 730, without either of the first two 560.
// Tried: four parts of K in a workgroup, a wave on 64 x 64 (half the operand reads, the same 57 clocks a matrix instruction; 0.5 us more
// for the sums: level for int8, 0 - 3 % ahead for bf16) or, one wave a SIMD, on 64 x 128 (1 us slower: bound by what one wave issues).
// Tried: matrix, LDS and vector instructions interleaved by hand (2 - 8 % slower), four more waves that only issue the loads
// (level), 32-, 128-row and 256-feature tiles (slower in all but a few cells).
#pragma once

#include "prefill_packed_kernel.h"

namespace terna {

constexpr int kDeepStages = 4;

template <typename Act, int MB, int NA, int D = kDeepStages>
struct DeepShape {
    static constexpr int kRow = 128 * static_cast<int>(sizeof(Act));     // a stage's piece of an activation row
    static constexpr int kX = 32 * MB * kRow;
    static constexpr int kStage = kX + 4 * NA * 1024;
    static constexpr int kBytes = D * kStage;
};

template <typename Act, int MB, int NA, int KS = 1, int EPI = PACKED_STORE, int D = kDeepStages>
__global__ __launch_bounds__(256 * KS) void terna_prefill_deep_kernel(
    const Act* __restrict__ x, const uint32_t* __restrict__ packed, uint16_t* __restrict__ out,
    Epilogue ep, int M, int N, int K, int xcd_map, int /*splits: 1*/, void* /*partial*/, int guard_on, PackedExtra<EPI> guard)
{
    const int tile_rows = static_cast<int>(gridDim.y) - (guard_on ? 1 : 0);
    if constexpr (EPI == PACKED_STORE) {
        if (guard_on && static_cast<int>(blockIdx.y) == tile_rows) {     // the check of a cached copy (see the other kernel)
            if (blockIdx.x == 0 && threadIdx.x < 64) repack_guard_role(guard, threadIdx.x);
            return;
        }
    }
    using S = DeepShape<Act, MB, NA, D>;
    constexpr bool I8 = sizeof(Act) == 1;
    constexpr int SZ = static_cast<int>(sizeof(Act));
    using AccV = typename std::conditional<I8, i32x16, f32x16>::type;
    constexpr int BN = 128 * NA, BM = 32 * MB;
    constexpr int PIECES = 8 * SZ, ROWS = 64 / PIECES;                   // 16-byte pieces of a stage row, rows per direct load
    constexpr int XI = BM / ROWS / 4;                                     // direct loads of activations per wave and stage
    constexpr int PER = XI + NA;
    constexpr int GROUPS = 4 * SZ, HALF = GROUPS / 2;                                        // matrix instructions per accumulator and stage
    constexpr int TW = I8 ? 1 : 2;                                        // weight reads per 32 features and stage
    static_assert(D == 4 && PER < 64, "three stages requested, vmcnt is a six-bit count");

    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int part = __builtin_amdgcn_readfirstlane(tid >> 8);            // of K
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    int n_tile = blockIdx.x, m_tile = blockIdx.y;
    if (xcd_map) {                                                        // as in the other kernel
        const int linear = blockIdx.y * gridDim.x + blockIdx.x;
        const int per_xcd = tile_rows >> 3;
        const int xcd = linear & 7, idx = linear >> 3;
        m_tile = xcd * per_xcd + idx % per_xcd;
        n_tile = idx / per_xcd;
    }
    const int n0 = n_tile * BN, m0 = m_tile * BM;
    const int ktiles = K >> 6, steps = (ktiles + 1) >> 1;
    const bool half_tail = ktiles & 1;                                    // the last stage has one 64-column tile only
    // steps of a part; of an odd number the first part's last does not exist, so that the last step of all is a part's last
    const int turns = (steps + KS - 1) / KS;
    const int k_begin = part == 0 ? 0 : steps - turns;
    const int k_end = part == KS - 1 ? steps : steps - turns;
    const int last_band = (N >> 4) - 1;
    const int kb = lane >> 5, l32 = lane & 31;

    // ---- this lane's place in the direct loads
    auto swizzle = [](int row) { return I8 ? (row >> 1) & 7 : row & 15; };
    uint32_t x_off[XI], x_back[XI], w_off[NA];
#pragma unroll
    for (int j = 0; j < XI; ++j) {
        const int row = ROWS * (wave + 4 * j) + lane / PIECES;
        const int piece = (lane % PIECES) ^ swizzle(row);
        const int m = m0 + row < M ? m0 + row : M - 1;
        x_off[j] = static_cast<uint32_t>(m) * static_cast<uint32_t>(K * SZ) + piece * 16;
        x_back[j] = piece >= 4 * SZ ? 64 * SZ : 0;                        // a tile that does not exist: the one before it
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        int band = (n0 >> 4) + 2 * NA * wave + 2 * a + (lane >> 5);
        band = band < last_band ? band : last_band;
        w_off[a] = static_cast<uint32_t>(band) * static_cast<uint32_t>(ktiles) * 256u + (lane & 31) * 16;
    }
    const uint32_t w_back = (lane & 31) >= 16 ? 256 : 0;
    const uint8_t* x_base = reinterpret_cast<const uint8_t*>(x);
    const uint8_t* w_base = reinterpret_cast<const uint8_t*>(packed);
    uint8_t* const stages = smem + part * S::kBytes;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(stages));
    auto issue = [&](int k, int st) __attribute__((always_inline)) {
        const bool back = half_tail && k == steps - 1;
        const uint8_t* xs = x_base + static_cast<size_t>(k) * S::kRow;
        const uint8_t* ws = w_base + static_cast<size_t>(k) * 512;
#pragma unroll
        for (int j = 0; j < XI; ++j) lds_dma_b128(xs, back ? x_off[j] - x_back[j] : x_off[j], lds0 + st + (wave + 4 * j) * 1024);
#pragma unroll
        for (int a = 0; a < NA; ++a) lds_dma_b128(ws, back ? w_off[a] - w_back : w_off[a], lds0 + st + S::kX + (wave * NA + a) * 1024);
    };

    AccV acc[NA][MB];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0;

    // B operand of group q, row tile b: int8 columns 64 kb + 16 q .. +15, bf16 columns 16 q + 8 kb .. +7
    // ... and the weight words of the wave's features: everything one step multiplies, in registers
    struct Ops { u32x4 b[GROUPS][MB], w[NA][TW]; };
    const int b_row = l32 * S::kRow;
    const int w_lane = S::kX + wave * NA * 1024 + (l32 >> 4) * 512 + (I8 ? kb * 256 : 0) + (l32 & 15) * 16;
    auto load = [&](int st, auto qc, Ops& r) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
        const int piece = (I8 ? 4 * kb + q : 2 * q + kb) ^ swizzle(l32);
#pragma unroll
        for (int b = 0; b < MB; ++b) r.b[q][b] = *reinterpret_cast<const u32x4*>(stages + st + b_row + b * 32 * S::kRow + piece * 16);
        if constexpr (q % 4 == 0 && q / 4 < TW) {
#pragma unroll
            for (int a = 0; a < NA; ++a) r.w[a][q / 4] = *reinterpret_cast<const u32x4*>(stages + st + w_lane + a * 1024 + q / 4 * 256);
        }
    };
    const int wshift = 4 - 4 * kb;
    auto mma = [&](const Ops& v, auto qc, uint32_t wmask = kTopFieldMask) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            if constexpr (I8) {
                const i32x4 af = expand_word_i8(v.w[a][0][q], wmask);
#pragma unroll
                for (int b = 0; b < MB; ++b) acc[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, __builtin_bit_cast(i32x4, v.b[q][b]), acc[a][b], 0, 0, 0);
            } else {
                const bf16x8 af = __builtin_bit_cast(bf16x8, expand_chunk_bf16(v.w[a][q >> 2][q & 3] << wshift));
#pragma unroll
                for (int b = 0; b < MB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, __builtin_bit_cast(bf16x8, v.b[q][b]), acc[a][b], 0, 0, 0);
            }
        }
    };

    auto next = [](int st) { return st == (D - 1) * S::kStage ? 0 : st + S::kStage; };
    // everybody's part of stage k has landed (one stage behind it is under way, if there is one), and all operand reads so far are done
    auto await = [&](int k) __attribute__((always_inline)) {
        if (k + 1 < k_end) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PER) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
    };
    if (k_begin < k_end) issue(k_begin, 0);                               // (uniform over the part)
    if (k_begin + 1 < k_end) issue(k_begin + 1, S::kStage);
    await(k_begin);
    int st_next = S::kStage, st_dma = (D - 1) * S::kStage;
    Ops even, odd;
    static_for<0, GROUPS>([&](auto qc) { load(0, qc, even); });
    using Ahead = typename std::conditional<KS == 2, RequestedEpilogue, NothingRequested>::type;
    Ahead ahead;
    if constexpr (KS == 2) {
        static_assert(NA == 1, "a tile of 32 features");
        ahead = request_epilogue<EPI>(out, ep, guard, M, N, n0 + 32 * wave, m0 + 32 * part, lane);
        asm volatile("" ::: "memory");
    }
    if (k_begin + 2 < k_end) issue(k_begin + 2, 2 * S::kStage);
    // INSIDE: step k + 3 exists, here and in the other part
    auto step = [&](int k, auto inside, const Ops& cur, Ops& nxt) __attribute__((always_inline)) {
        constexpr bool INSIDE = decltype(inside)::value;
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, HALF>([&](auto qc) { mma(cur, qc); });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (INSIDE) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER) : "memory");
        else await(k + 1);
        static_for<HALF, GROUPS>([&](auto qc) {
            constexpr int q = decltype(qc)::value, r = 2 * (q - HALF);
            __builtin_amdgcn_sched_barrier(0);                            // keeps the reads between the groups
            load(st_next, std::integral_constant<int, r>{}, nxt);
            load(st_next, std::integral_constant<int, r + 1>{}, nxt);
            mma(cur, qc);
            if constexpr (q == HALF) {
                if (INSIDE || k + D - 1 < k_end) issue(k + D - 1, st_dma);         // into the stage of step k - 1
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        st_next = next(st_next);
        st_dma = next(st_dma);
    };
    // The last turn multiplies what is in registers.  A last stage with one tile: int8 multiplies both by weights that are 0 where the
    // lane's tile does not exist; bf16 leaves the groups of the other one out (its activations are the first tile's, which may be
    // infinite: 0 times that is NaN).
    auto last_step = [&](int k, const Ops& cur) __attribute__((always_inline)) {
        if (k >= k_end) return;                                           // uniform over the part
        const bool half = half_tail && k == steps - 1;
        constexpr int LOWER = I8 ? GROUPS : GROUPS / 2;                   // groups of the first tile (int8: of both)
        static_for<0, LOWER>([&](auto qc) { mma(cur, qc, half && kb ? 0u : kTopFieldMask); });
        if (!half) static_for<LOWER, GROUPS>([&](auto qc) { mma(cur, qc); });
    };
    int t = 0;
    using Inside = std::true_type;
    using Edge = std::false_type;
    for (; t + D < steps - (KS - 1) * turns; t += 2) {
        step(k_begin + t, Inside{}, even, odd);
        step(k_begin + t + 1, Inside{}, odd, even);
    }
    for (; t + 2 < turns; t += 2) {
        step(k_begin + t, Edge{}, even, odd);
        step(k_begin + t + 1, Edge{}, odd, even);
    }
    if (t + 1 < turns) {
        step(k_begin + t, Edge{}, even, odd);
        last_step(k_begin + t + 1, odd);
    } else {
        last_step(k_begin + t, even);
    }
    // ---- results as whole rows through LDS (prefill_packed_kernel.h), in place of two stages that nobody reads any more: the last one's
    // operands were read behind the last barrier
    const int last_stage = st_next == 0 ? (D - 1) * S::kStage : st_next - S::kStage;
    uint8_t* const free_stages = stages + (last_stage >= 2 * S::kStage ? 0 : 2 * S::kStage);
    static_assert(4 * OutTile<NA>::kBytes <= 2 * S::kStage, "output tiles fit in two stages");
    const bool rows_ok = ((reinterpret_cast<uintptr_t>(out) | (static_cast<uintptr_t>(N) * 2)) & 15) == 0;
    if constexpr (KS == 2) {
        // each part leaves the row tile that the other one finishes
        static_assert(KS == 1 || (MB == 2 && 4 * NA * 4096 <= 2 * S::kStage), "two row tiles, one per part");
        float* mine = reinterpret_cast<float*>(free_stages) + wave * NA * 1024 + lane;
        const float* other = reinterpret_cast<const float*>(free_stages + (part == 0 ? S::kBytes : -S::kBytes)) + wave * NA * 1024 + lane;
        AccV sum[NA][1];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const auto give = part == 0 ? acc[a][1][v] : acc[a][0][v];
                mine[(16 * a + v) * 64] = __builtin_bit_cast(float, give);
                sum[a][0][v] = part == 0 ? acc[a][0][v] : acc[a][1][v];
            }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int v = 0; v < 16; ++v) sum[a][0][v] += __builtin_bit_cast(typename std::conditional<I8, int, float>::type, other[(16 * a + v) * 64]);
        uint8_t* const tile = stages + (free_stages == stages ? 2 * S::kStage : 0) + wave * OutTile<NA>::kBytes;
        if constexpr (EPI == PACKED_GATE) {
            packed_prefill_gate_epilogue<1, NA>(sum, out, ep, M, N, n0 + 32 * NA * wave, m0 + 32 * part, lane, tile, ahead);
            return;
        }
        if constexpr (EPI == PACKED_ROPE) {
            packed_prefill_rope_epilogue<1, NA>(sum, out, ep, guard, M, N, n0 + 32 * NA * wave, m0 + 32 * part, lane, tile, ahead);
            return;
        }
        if constexpr (EPI == PACKED_RESIDUAL) {
            packed_prefill_epilogue<1, NA, AccV, false, true>(sum, out, ep, M, N, n0 + 32 * NA * wave, m0 + 32 * part, lane,
                                                              tile, guard, ahead);
            return;
        }
        packed_prefill_epilogue<1, NA, AccV, true>(sum, out, ep, M, N, n0 + 32 * NA * wave, m0 + 32 * part, lane,
                                                   rows_ok ? tile : nullptr,
                                                   ResidualRows{nullptr}, ahead);
        return;
    }
    if constexpr (EPI == PACKED_GATE) {
        packed_prefill_gate_epilogue<MB, NA>(acc, out, ep, M, N, n0 + 32 * NA * wave, m0, lane, free_stages + wave * OutTile<NA>::kBytes);
        return;
    }
    if constexpr (EPI == PACKED_ROPE) {
        packed_prefill_rope_epilogue<MB, NA>(acc, out, ep, guard, M, N, n0 + 32 * NA * wave, m0, lane, free_stages + wave * OutTile<NA>::kBytes);
        return;
    }
    if constexpr (EPI == PACKED_RESIDUAL) {
        packed_prefill_epilogue<MB, NA, AccV, false, true>(acc, out, ep, M, N, n0 + 32 * NA * wave, m0, lane, free_stages + wave * OutTile<NA>::kBytes, guard);
        return;
    }
    packed_prefill_epilogue<MB, NA, AccV, MB * NA <= 2>(acc, out, ep, M, N, n0 + 32 * NA * wave, m0, lane,
                                                        rows_ok ? free_stages + wave * OutTile<NA>::kBytes : nullptr);
}

}  // namespace terna
