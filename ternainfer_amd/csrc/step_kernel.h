// A decode step of a few sequences -- the five linears-and-attention phases of every block -- in ONE launch.
//
// As launches of their own (chain_chunk_kernel.h, attention_kernel.h) the phases of a block are bound by the boundary between
// them: 1.55 us for a graph node and 1.2 us for the first cold round trip behind it, five times a block.  Here 256
// workgroups, one a CU, stay for the whole step.  A phase hands its output over in device memory, and the words are their own
// flags: the buffers (a part for every phase of every block, no word is written twice) are cleared to 0xffffffff by the
// launch in front, a producer stores with device scope, a consumer loads the words it needs with device scope until none
// of them reads 0xffffffff any more.  That word is a pair of NaNs no producer writes (step_word).  There is no counter, no fence
// and no second trip for the data.  A handover alone: 1.44 us from one poll to the next (160 workgroups, 32-byte slices, 5 KB;
// 256 writers of 20 bytes each, which share lines, 1.95).
// Measured, us a step of 30 blocks of the 2B shape with the LM head, launches -> this: one sequence, 384 slots 813 -> 640, 4096 slots
// filled to 50 % 920 -> 766, to 90 % 1132 -> 867; two, 384 slots 895 -> 732; three, 101 slots 885 -> 798; four, 384 slots 939 -> 856.
//
// Bound: what is left of the handovers (0.7 - 1.3 us each, five or six a block), and behind each wait the instructions of one wave per
// SIMD, 4 - 8 cycles apiece: 1.6 - 2.7 us a phase.  Hence, in the order of what they gave:
//   * nothing may load behind a prefetch: loads return in order, so a spilled register, a scale or a pointer read there waits for
//     device memory.  What all blocks need lies in LDS from the start, the registers never spill (-disable-machine-licm), and
//     no branch leaves a poll's loads open (step_largest).
//   * four waves of 128 registers instead of eight of 64: no phase spills, and what every wave repeats is done by half as many;
//   * the weights come into the XCD's L2 two phases ahead (step_prefetch) and into registers, partly expanded, during the wait;
//   * an element takes four instructions to its int8 byte (quant_rounded4).
//
// Waiting is safe.  All workgroups are resident together as a rule: a workgroup takes a quarter of a CU at most (four waves of
// up to 128 registers, 40 KB of LDS), the launcher checks that the device holds four grids at once, and the runtime runs
// kernels of at most four queues of a process side by side.  Where they are not -- more steps at once, of several processes or
// on streams of several priorities; a captured step replayed on a stream with few CUs -- the waits end: after kStepPatience
// polls a wave gives up, says so to all others (StepControl::alive), and the rest of the launch runs through without
// waiting, on what it finds.  The launch behind it (ORDERED) then does the step again, from the same inputs and over everything the
// first wrote, in a way that needs no workgroups side by side: a few of them take the units of work one by one in the order
// in which they depend on each other (step_ticket), so that whatever one waits for is held by a workgroup that runs (30 blocks of
// the 2B shape, 384 slots: 3 ms with one sequence, 4 with four).  Where nobody gave up it ends at once, 2 - 4 us.
//
// Every result has the bits of the launches this replaces: integer sums, and for all that is rounded the same operations in
// the same order (the partial statistics of 16 columns are formed by the consumer instead of the producer).
//
// Workgroup -> work, the same in every block: band w of QKV, of O and of the down projection, bands 4w .. 4w+3 of the
// interleaved gate+up matrix; attention units from the last workgroup downwards, so that they mostly sit where no band
// of O is.  The residual stream of a band's 16 columns stays in its LDS.
// K is shared by the four waves in whole tiles of 64 columns: a run of 4 CH + SG tiles per wave -- ten for K <= 2560 -- four as
// one 16-byte load per lane, single ones as a word per lane.
#pragma once

#include "attention_kernel.h"
#include "chain_chunk_kernel.h"
#include "step_layout.h"

namespace terna {

constexpr int kStepMaxBlocks = 32;               // blocks per launch: their pointers travel as arguments (4 KB)
constexpr int kStepMaxSplits = 8;                // splits of the cache, one sequence; four at a time are merged
constexpr int kStepRecord = (kStepHeadDim + 4) * 4;      // bytes a (head, split) hands over: 128 sums, maximum, sum of numerators
// Slots of a cache that is not split; of a split.  Every (sequence, head, half) walks its whole prefix, so the lines lie where that takes as
// long as the launches with the attention split over the chip (us a step, caches filled to 90 %, those -> this: two sequences, 1280 slots
// 1027 -> 945; three, 1024 1052 -> 985; four, 700 1054 -> 939, 1024 1064 -> 1012, filled to half 1045 -> 910.  With 1528 slots two 1033 -> 1052,
// three 1066 -> 1145, four 1078 -> 1174, taken before each XCD fetched what its own workgroups read, which gave 30 - 40 at the lines; they are where they were).
constexpr int step_max_slots(int M) { return M == 2 ? 1280 : 1024; }
constexpr int kStepMaxSplitSlots = 1024;
constexpr uint32_t kStepEmpty = 0xffffffffu;
// Polls of one wait before a wave gives up: 20 ms where they take 0.15 us (an idle chip), more on a busy one -- longer than the kernels
// of other streams hold a part of the grid back.  Polls and not wall clock: a process that was suspended has not waited.
constexpr int kStepPatience = 1 << 17;
constexpr int kStepOrderedGroups = 64;           // workgroups that do a step in order
constexpr int kStepOrderedPolls = 1 << 26;       // ... whose waits end too (10 s and more, for work of microseconds)
constexpr int kStepControlBytes = 512;           // scratch in front of the exchange: word 0 StepArgs::alive, 1 + 2 i and 2 + 2 i the tickets of launch i
constexpr int kDeviceScope = 16;                 // cache policy of a raw buffer access: sc1

struct StepBlock {
    const uint32_t *wqkv, *wo, *w13, *w2;        // P2; w13 with its bands interleaved
    const uint16_t *ws_qkv, *ws_o, *ws_13, *ws_2;
    const uint16_t *attention_norm, *attn_sub_norm, *ffn_norm, *ffn_sub_norm;
    uint16_t *cache_k, *cache_v;
};

// Where the phases of a block leave their outputs: byte offsets within the block's part of the exchange buffer.
struct StepExchange {
    uint32_t qkv, attention, mid, inner, quantised, scales, out, bytes;
};

struct StepArgs {
    char* exchange;                              // [blocks][StepExchange::bytes]
    uint32_t* alive;                             // polls a wait may take, 0 once a wave has given up
    const uint16_t* x;                           // the stream in front of the first block, no word 0xffffffff
    const float2* stats;                         // its partials under the first block's norm, [M][stats_count]; nullptr: formed here
    uint16_t* x_out;                             // the stream behind the last block
    const long long* pos;
    const float *cosv, *sinv;
    int blocks, M, dim, ffn, H, KV, S, SP, per_seq, stats_count, quant_mode, ws_qkv, ws_o, ws_2;
    float eps, scale;
    StepExchange at;
    StepBlock block[kStepMaxBlocks];
    uint32_t* tickets;                           // ORDERED: [0] taken, [1] done, both from 0xffffffff
};
static_assert(sizeof(StepArgs) <= 4096, "kernel arguments");

void launch_step_ordered(const StepArgs& a, hipStream_t st);      // launch_step_ordered.hip: the ORDERED kernel

// What a producer stores: never the word that stands for "not there yet" (a pair of bf16 NaNs, or an fp32 one: the last
// bit of a NaN goes).
__device__ __forceinline__ uint32_t step_word(uint32_t v) { return v < kStepEmpty ? v : kStepEmpty - 1; }

struct StepControl {
    uint32_t* alive;
    bool gave_up;

    // every 256 polls of a wave
    __device__ void check(int polls)
    {
        gave_up = polls > __builtin_amdgcn_readfirstlane(static_cast<int>(__hip_atomic_load(alive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
        if (gave_up) __hip_atomic_store(alive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // load(): requests what the lane needs; there(): all of it has come.  meanwhile(): once, while the first requests are on their way.
    template <typename Load, typename There, typename Meanwhile>
    __device__ __forceinline__ void await(Load load, There there, Meanwhile meanwhile)
    {
        load();
        asm volatile("" ::: "memory");
        meanwhile();
        bool all = __all(there());
        for (int n = 1; !all && !gave_up; ++n) {
            asm volatile("" ::: "memory");       // the loads are made again
            load();
            all = __all(there());
            if ((n & 255) == 0) check(n);
        }
        asm volatile("" ::: "memory");
    }
    template <typename Load, typename There>
    __device__ __forceinline__ void await(Load load, There there) { await(load, there, [] {}); }
};

__device__ __forceinline__ u32x4 step_load16(__amdgpu_buffer_rsrc_t r, int offset) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, kDeviceScope)); }
__device__ __forceinline__ u32x2 step_load8(__amdgpu_buffer_rsrc_t r, int offset) { return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, offset, 0, kDeviceScope)); }
// The largest word: kStepEmpty where one has not come yet.  (No && over the words: a branch past some of them would leave their
// loads open behind the wait, and whoever uses them would wait for the prefetches issued meanwhile.)
__device__ __forceinline__ uint32_t step_max(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t step_largest(const u32x4& v) { return step_max(step_max(v.x, v.y), step_max(v.z, v.w)); }
__device__ __forceinline__ uint32_t step_largest(const u32x2& v) { return step_max(v.x, v.y); }

// LDS of the linear phases: a slab per wave -- its int8 rows, then in the same place its accumulators -- and the partial
// statistics of the rows.
template <int MR>
struct StepLds {
    static constexpr int kPitch = kStepWideTiles / kStepWaves * 64 + 16;       // a wave's tiles of a row + 16 bytes (conflict-free operand reads)
    static constexpr int kSlab = MR * kPitch;
    static constexpr int kPartials = MR == 1 ? kStepWideTiles * 4 : kStepTiles * 4;        // of a row
    static constexpr int kPartialBytes = (MR * kPartials > kStepWideTiles * 4 ? MR * kPartials : kStepWideTiles * 4) * 8;
    static constexpr int kLinear = kStepWaves * kSlab + kPartialBytes;
    // attention: slices and groups of output dimensions, scores
    static constexpr int kScores = (MR == 1 ? kStepMaxSplitSlots : step_max_slots(MR)) + 32;
    static constexpr int kAttention = ((16 + 2) * kStepHeadDim + kScores) * 4;             // (slices and groups: the same number of floats split or not)
    static constexpr int kBytes = kLinear > kAttention ? kLinear : kAttention;
    static_assert(4 * MR * 64 <= kSlab, "the accumulators of four bands fit a wave's slab");
};

// How the consumer of a row forms its partial statistics, each in the order of the launch it stands for.
enum StepStats {
    STEP_GROUPS,      // 16 columns, pairwise                       (producing epilogues of the chained linears)
    STEP_HEADS,       // 128 columns, pairwise                      (the unsplit attention as a producer)
    STEP_CHUNKS       // 4 columns in order, then 256 pairwise      (terna_chain_norm_kernel)
};

// Weights and norm weights of one phase, requested ahead of the wait for its input; the first EX (tile, band) pairs are also
// expanded to operands there.  Behind the wait a wave has its SIMD to itself and issues an instruction in 4 - 8 cycles: the
// seven of an expansion, forty times in gate+up, are 0.5 us and more.
template <int MR, int NB, int CH, int SG, int EX, bool NORM = true>
struct StepOperands {
    static constexpr int TPW = 4 * CH + SG;                       // tiles of a wave
    static constexpr int TPR = 4 / MR;                            // tiles of a round: 16 lanes x 4 columns of one row each
    static constexpr int ROUNDS = (TPW + TPR - 1) / TPR;
    u32x4 wc[NB][CH];
    uint32_t wt[NB][SG > 0 ? SG : 1];
    i32x4 ex[EX];
    u32x2 nw[NORM ? ROUNDS : 1];

    // word of pair (tile t of the run, band b): in chunks a lane holds component t & 3 of one load
    __device__ __forceinline__ uint32_t word(int t, int b) const { return t < 4 * CH ? wc[b][t >> 2][t & 3] : wt[b][t - 4 * CH]; }

    // (Tiles past K: words of the next band or nothing, times activations that are zero.  All of the offset is the lane's, which is what
    // the buffer's range is held against: a run of the last band may begin past the matrix.)
    __device__ __forceinline__ void request(const uint32_t* packed, int bands, int band0, int K, const uint16_t* norm_w, int lane, int wave)
    {
        const int ktiles = K >> 6, first = wave * TPW, i = lane & 15, g = lane >> 4;
        const __amdgpu_buffer_rsrc_t rw = make_raw_buffer(packed, static_cast<uint32_t>(bands) * ktiles * 256u);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int chunk = step_weight_offset(band0 + b, ktiles, first, lane * 16), single = step_weight_offset(band0 + b, ktiles, first, (4 * i + g) * 4);
#pragma unroll
            for (int c = 0; c < CH; ++c) wc[b][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, chunk + 1024 * c, 0, 0));
#pragma unroll
            for (int s = 0; s < SG; ++s) wt[b][s] = __builtin_amdgcn_raw_buffer_load_b32(rw, single + 256 * (4 * CH + s), 0, 0);
        }
        if constexpr (NORM) {
            const __amdgpu_buffer_rsrc_t rn = make_raw_buffer(norm_w, static_cast<uint32_t>(K) * 2u);
            const int at = ((first + g / MR) * 64 + 4 * i) * 2;
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) nw[r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rn, at + r * TPR * 128, 0, 0));
        }
        asm volatile("" ::: "memory");           // requested here
    }
    __device__ __forceinline__ void expand()
    {
#pragma unroll
        for (int e = 0; e < EX; ++e) {
            ex[e] = expand_word_i8(word(e / NB, e % NB));
            asm volatile("" : "+v"(ex[e]));      // expanded here
        }
    }
    // acc[b] of the wave's K run; the slab holds its int8 rows
    __device__ __forceinline__ void multiply(const uint8_t* slab, i32x4 (&acc)[NB], int lane) const
    {
        const int i = lane & 15, g = lane >> 4;
        const uint8_t* row = slab + (i & (MR - 1)) * StepLds<MR>::kPitch;         // columns past the rows are not read again
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            // a chunk's k index runs over (tile, column): operand p of it is piece p of tile g
            const u32x4 x = *reinterpret_cast<const u32x4*>(t < 4 * CH ? row + ((t & ~3) + g) * 64 + 16 * (t & 3) : row + t * 64 + 16 * g);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const i32x4 w = t * NB + b < EX ? ex[t * NB + b < EX ? t * NB + b : 0] : expand_word_i8(word(t, b));
                acc[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, __builtin_bit_cast(i32x4, x), acc[b], 0, 0, 0);
            }
        }
    }
};

// The same value, computed anew from here on: what depends on it is not hoisted out of the loop over the blocks (which kept
// three hundred registers of offsets alive across all phases).
__device__ __forceinline__ int step_lane()
{
    int v = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int step_uniform(int v)
{
    asm volatile("" : "+s"(v));
    return v;
}

// What a phase computes with, anew in every one (step_lane); the shape comes out of LDS, where it takes no register meanwhile.
struct StepShape {
    int M, dim, ffn, H, KV, SP, quant_mode;
    float eps;
};
struct StepPhase : StepShape {
    int lane, wave, w, wide, qkv_n;
};

struct StepScale {
    float rstd, mul, s;       // 1 / rms, what multiplies, its bf16 value
};
__device__ __forceinline__ StepScale step_scale(float sum, float pmax, int K, float eps, int quant_mode)
{
    StepScale r;
    r.rstd = rsqrtf(sum / static_cast<float>(K) + eps);
    uint16_t sb;
    r.mul = quant_scale(fabsf(round_bf16(__fmul_rn(pmax, r.rstd))), quant_mode, &sb);       // = of max |y|, exactly
    r.s = bf16_bits_to_float(sb);
    return r;
}

// A row's statistics from its partials: all lanes of a wave, the same value in all.  TILES: what K can be at most.
template <int KIND, int TILES>
__device__ __forceinline__ StepScale step_row_scale(const float2* part, int K, float eps, int quant_mode, int lane)
{
    float sum = 0.0f, pmax = 0.0f;
    if constexpr (KIND == STEP_GROUPS) {
        constexpr int PT = (4 * TILES + 63) / 64;
        const int count = K >> 4;
        float2 v[PT];
#pragma unroll
        for (int t = 0; t < PT; ++t) v[t] = part[lane + 64 * t < count ? lane + 64 * t : 0];
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            sum += lane + 64 * t < count ? v[t].x : 0.0f;
            pmax = max_keep_nan(pmax, v[t].y);                     // (the first one again does not change it)
        }
        sum = wave_sum(sum);
        pmax = wave_amax(pmax);
    } else if constexpr (KIND == STEP_HEADS) {
        if (lane < K / kStepHeadDim) {
            sum = part[2 * lane].x + part[2 * lane + 1].x;
            pmax = max_keep_nan(part[2 * lane].y, part[2 * lane + 1].y);
        }
        sum = wave_sum(sum);
        pmax = wave_amax(pmax);
    } else {
        const int c = 4 * (lane & 15), tiles = K >> 6;
        float2 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = part[c + e < tiles ? c + e : 0];
#pragma unroll
        for (int e = 0; e < 4; ++e) pmax = max_keep_nan(pmax, v[e].y);
        auto x = [&](int e) { return c + e < tiles ? v[e].x : 0.0f; };
        sum = group_reduce<16, false>((x(0) + x(1)) + (x(2) + x(3)));
        pmax = group_amax<16>(pmax);
    }
    return step_scale(sum, pmax, K, eps, quant_mode);
}

// The lane's columns -- four of one tile in every round -> their partial statistics, in LDS.  Several rounds in one region of
// code, so that their chains of dependent operations run side by side.
constexpr int kStepBatch = 4;
template <int KIND, typename Op>
__device__ __forceinline__ void step_partials(const u32x2 (&h)[Op::ROUNDS], const u32x2 (&w)[Op::ROUNDS], float2* part, float2* nowhere, int first, int t0, int ktiles,
                                              int lane)
{
    static_for<0, (Op::ROUNDS + kStepBatch - 1) / kStepBatch>([&](auto batch) {
        constexpr int FROM = decltype(batch)::value * kStepBatch, COUNT = Op::ROUNDS - FROM < kStepBatch ? Op::ROUNDS - FROM : kStepBatch;
        float2 out[COUNT];
#pragma unroll
        for (int q = 0; q < COUNT; ++q) {
            const uint32_t hd[2] = {h[FROM + q].x, h[FROM + q].y}, wd[2] = {w[FROM + q].x, w[FROM + q].y};
            float f[4], m[4];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                f[2 * j] = __uint_as_float(hd[j] << 16);
                f[2 * j + 1] = __uint_as_float(hd[j] & 0xffff0000u);
                m[2 * j] = fabsf(__fmul_rn(f[2 * j], __uint_as_float(wd[j] << 16)));
                m[2 * j + 1] = fabsf(__fmul_rn(f[2 * j + 1], __uint_as_float(wd[j] & 0xffff0000u)));
            }
            float ssq;                           // (squares of bf16 values are exact: contracted or not, the same sums)
            if constexpr (KIND == STEP_CHUNKS) {
                ssq = fmaf(f[0], f[0], 0.0f);
#pragma unroll
                for (int e = 1; e < 4; ++e) ssq = fmaf(f[e], f[e], ssq);
            } else {
                ssq = (f[0] * f[0] + f[1] * f[1]) + (f[2] * f[2] + f[3] * f[3]);
            }
            const float pmax = max_keep_nan(max_keep_nan(m[0], m[1]), max_keep_nan(m[2], m[3]));
            constexpr int LANES = KIND == STEP_GROUPS ? 4 : 16;
            out[q] = float2{group_reduce<LANES, false>(ssq), group_amax<LANES>(pmax)};
        }
        constexpr int PER = KIND == STEP_GROUPS ? 4 : 1;          // partials of a tile
        if ((lane & (16 / PER - 1)) == 0) {
#pragma unroll
            for (int q = 0; q < COUNT; ++q) {
                const int t = (FROM + q) * Op::TPR + t0;
                float2* to = t < Op::TPW && first + t < ktiles ? part + PER * (first + t) + (lane & 15) * PER / 16 : nowhere;
                *to = out[q];
            }
        }
    });
}

// One normed and quantised linear: the lane's columns (round r: tile r TPR + (lane >> 4) / MR of the wave's run, row
// (lane >> 4) % MR) are in xr.  Leaves the accumulators of all waves in their slabs behind a barrier; returns the scale of
// the row this lane finishes.
template <int MR, int KIND, int TILES, int NB, typename Op>
__device__ __forceinline__ float step_norm_linear(const Op& op, const u32x2 (&xr)[Op::ROUNDS], const StepPhase& p, int K, const float2* given, int given_count,
                                                  uint8_t* lds, float2* nowhere, StepScale* scale_s)
{
    using Lds = StepLds<MR>;
    const int lane = p.lane, wave = p.wave;
    uint8_t* slab = lds + wave * Lds::kSlab;
    float2* partials = reinterpret_cast<float2*>(lds + kStepWaves * Lds::kSlab);
    const int first = wave * Op::TPW, ktiles = K >> 6;
    const int row = (lane >> 4) % MR, t0 = (lane >> 4) / MR;
    step_partials<KIND, Op>(xr, op.nw, partials + row * Lds::kPartials, nowhere, first, t0, ktiles, lane);
    __syncthreads();
    auto row_scale = [&](int m) {
        if (given != nullptr) {                  // uniform: the partials of another launch, few
            float sum = 0.0f, pmax = 0.0f;
            if (lane < given_count) {
                const float2 v = given[m * given_count + lane];
                sum = v.x;
                pmax = v.y;
            }
            sum = wave_sum(sum);
            pmax = wave_amax(pmax);
            return step_scale(sum, pmax, K, p.eps, p.quant_mode);
        }
        return step_row_scale<KIND, TILES>(partials + m * Lds::kPartials, K, p.eps, p.quant_mode, lane);
    };
    StepScale mine;
    float finish;
    if constexpr (MR == 1) {                     // every wave for itself
        mine = row_scale(0);
        finish = mine.s;
    } else {
        if (wave < p.M) {
            const StepScale sc = row_scale(wave);
            if (lane == 0) scale_s[wave] = sc;
        }
        __syncthreads();
        mine = scale_s[row < p.M ? row : 0];
        const int f = lane >> 4;
        finish = scale_s[f < p.M ? f : 0].s;
    }
    static_for<0, (Op::ROUNDS + kStepBatch - 1) / kStepBatch>([&](auto batch) {
        constexpr int FROM = decltype(batch)::value * kStepBatch, COUNT = Op::ROUNDS - FROM < kStepBatch ? Op::ROUNDS - FROM : kStepBatch;
        uint32_t hd[2 * COUNT], wd[2 * COUNT], d[COUNT];
#pragma unroll
        for (int q = 0; q < COUNT; ++q) {
            hd[2 * q] = xr[FROM + q].x, hd[2 * q + 1] = xr[FROM + q].y;
            wd[2 * q] = op.nw[FROM + q].x, wd[2 * q + 1] = op.nw[FROM + q].y;
        }
        chain_quantise<4 * COUNT>(hd, wd, mine.rstd, mine.mul, p.quant_mode, d);
#pragma unroll
        for (int q = 0; q < COUNT; ++q) {
            const int t = (FROM + q) * Op::TPR + t0;
            // (tiles past the run, in the last round: into the padding of the row)
            *reinterpret_cast<uint32_t*>(slab + row * Lds::kPitch + (t < Op::TPW ? t * 64 + 4 * (lane & 15) : Lds::kPitch - 16 + 4 * (lane & 3))) = d[q];
        }
    });
    i32x4 acc[NB];
    op.multiply(slab, acc, lane);
    const int i = lane & 15, g = lane >> 4;
    if (i < MR) {
#pragma unroll
        for (int b = 0; b < NB; ++b) *reinterpret_cast<i32x4*>(slab + (b * MR + i) * 64 + 16 * g) = acc[b];
    }
    __syncthreads();
    return finish;
}

// Sum of a band over the waves, for lane (row lane >> 4, column lane & 15).
template <int MR>
__device__ __forceinline__ int step_band_sum(const uint8_t* lds, int band, int lane)
{
    const int* p = reinterpret_cast<const int*>(lds + (band * MR + ((lane >> 4) & (MR - 1))) * 64) + (lane & 15);
    int sum = p[0];
#pragma unroll
    for (int w = 1; w < kStepWaves; ++w) sum += p[w * (StepLds<MR>::kSlab / 4)];
    return sum >> kI8WeightShift;
}

// bf16 value of the lane's column, two columns a word, to [row][cols]: what a consumer waits for.
__device__ __forceinline__ void step_store_pair(__amdgpu_buffer_rsrc_t to, uint16_t bits, int cols, int n, bool row_ok, int lane)
{
    const uint32_t v = bits;
    const uint32_t pair = step_word(v | (dpp_permute_u32<kDppSwapPairs>(v) << 16));
    const int row = lane >> 4;
    __builtin_amdgcn_raw_buffer_store_b32(pair, to, row_ok && (lane & 1) == 0 ? (row * cols + n) * 2 : kBufferOutOfRange, 0, kDeviceScope);
}

// Rows of bf16 that another phase hands over: the lane's columns of every round.  Past K or the rows: zeros.
template <int MR, typename Op, typename Meanwhile>
__device__ __forceinline__ void step_fetch_rows(StepControl& ctl, const void* from, int M, int K, u32x2 (&xr)[Op::ROUNDS], int lane, int wave, Meanwhile meanwhile)
{
    const __amdgpu_buffer_rsrc_t rx = make_raw_buffer(from, static_cast<uint32_t>(M) * K * 2u);
    const int first = wave * Op::TPW, left = (K >> 6) - first, tiles = left < Op::TPW ? left : Op::TPW;
    const int row = (lane >> 4) % MR, t0 = row < M ? (lane >> 4) / MR : 1 << 20;
    const int at = (row * K + (first + t0) * 64 + 4 * (lane & 15)) * 2;
    ctl.await([&]() {
#pragma unroll
        for (int r = 0; r < Op::ROUNDS; ++r) xr[r] = step_load8(rx, r * Op::TPR + t0 < tiles ? at + r * Op::TPR * 128 : kBufferOutOfRange);
    }, [&]() {
        uint32_t top = 0u;
#pragma unroll
        for (int r = 0; r < Op::ROUNDS; ++r) top = step_max(top, step_largest(xr[r]));
        return top != kStepEmpty;
    }, meanwhile);
}

// One sequence: the merged attention output's columns from the splits' partial results (attention_merge's arithmetic).  The
// weights of a wave's heads -- ten tiles lie in six heads at most -- are formed by a lane per (head, split) and pass
// through LDS: in registers of every column they cost sixteen more.
struct StepMerge {
    float w[kStepMaxSplits], sum[kStepMaxSplits];
};
template <typename Op, bool ORDERED, typename Meanwhile>
__device__ __forceinline__ void step_fetch_merged(StepControl& ctl, const void* from, int H, int SP, u32x2 (&xr)[Op::ROUNDS], StepMerge (&merge)[8], int lane, int wave, Meanwhile meanwhile)
{
    const int K = H * kStepHeadDim, first = wave * Op::TPW, ktiles = K >> 6, head0 = first >> 1;
    const __amdgpu_buffer_rsrc_t rp = make_raw_buffer(from, static_cast<uint32_t>(H) * SP * kStepRecord);
    const int own_head = head0 + (lane >> 3), own_split = lane & 7;
    u32x2 ml;
    // The last words of a record first, on their own: polling all 42 KB in 160 workgroups would fill the memory system while the
    // attention works.
    ctl.await([&]() {
        ml = step_load8(rp, own_head < H && own_split < SP ? (own_head * SP + own_split) * kStepRecord + kStepHeadDim * 4 : kBufferOutOfRange);
    }, [&]() { return step_largest(ml) != kStepEmpty; }, meanwhile);
    // ... then the rest, which by now is mostly there, through the L2 that twenty workgroups share; a line that came too early
    // shows its empty words and is loaded again past it.  (ORDERED: past it at once, the words were not cleared.)
    using First = std::integral_constant<int, ORDERED ? kDeviceScope : 0>;
    u32x4 o[Op::ROUNDS][4];
    auto load = [&](int j0, auto scope) {
#pragma unroll
        for (int r = 0; r < Op::ROUNDS; ++r) {
            const int t = r * 4 + (lane >> 4), tile = first + t;
            const int at = t < Op::TPW && tile < ktiles ? ((tile >> 1) * SP + j0) * kStepRecord + ((tile & 1) * 64 + 4 * (lane & 15)) * 4 : kBufferOutOfRange;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[r][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, j0 + j < SP ? at + j * kStepRecord : kBufferOutOfRange, 0, decltype(scope)::value));
        }
    };
    auto there = [&]() {
        uint32_t top = 0u;
#pragma unroll
        for (int r = 0; r < Op::ROUNDS; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) top = step_max(top, step_largest(o[r][j]));
        return top != kStepEmpty;
    };
    load(0, First{});
    {
        const float m = own_split < SP ? __uint_as_float(ml.x) : -INFINITY;
        const float w = __expf(m - group_reduce<8, true>(m));          // a split that is empty or not there: exp(-inf) = 0
        merge[lane >> 3].w[own_split] = w;
        merge[lane >> 3].sum[own_split] = __uint_as_float(ml.y);
    }
    if (!__all(there())) ctl.await([&]() { load(0, std::integral_constant<int, kDeviceScope>{}); }, there);
    float num[Op::ROUNDS][4], den[Op::ROUNDS];
    auto add = [&](int j0) {
#pragma unroll
        for (int r = 0; r < Op::ROUNDS; ++r) {
            const int t = r * 4 + (lane >> 4), tile = first + t;
            const StepMerge& mg = merge[t < Op::TPW && tile < ktiles ? (tile >> 1) - head0 : 0];
#pragma unroll
            for (int j = 0; j < 4; ++j) {        // in split order
                const float w = mg.w[j0 + j];
                den[r] = fmaf(w, mg.sum[j0 + j], j0 + j == 0 ? 0.0f : den[r]);
#pragma unroll
                for (int e = 0; e < 4; ++e) num[r][e] = fmaf(w, __uint_as_float(o[r][j][e]), j0 + j == 0 ? 0.0f : num[r][e]);
            }
        }
    };
    add(0);
    if (SP > 4) {
        load(4, First{});
        if (!__all(there())) ctl.await([&]() { load(4, std::integral_constant<int, kDeviceScope>{}); }, there);
        add(4);
    }
#pragma unroll
    for (int r = 0; r < Op::ROUNDS; ++r) {
        const int t = r * 4 + (lane >> 4);
        float merged[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) merged[e] = t < Op::TPW && first + t < ktiles ? num[r][e] / den[r] : 0.0f;
        xr[r] = u32x2{pack_bf16x2(merged[0], merged[1]), pack_bf16x2(merged[2], merged[3])};
    }
}

// RoPE, cache write and attention of one unit: terna_decode_attention_kernel's arithmetic -- unsplit with eight waves (several
// sequences: a unit is a (sequence, head, half of its dimensions); both halves form all scores), or split with four (one
// sequence: a (head, split), whose unnormalised result is handed over).  Keys up to 128 slots and a round of values are
// requested before the wait for the new token's rows, later ones as their registers come free.
// Bound: issue, as everything behind a wait -- so four MFMAs' scores are picked out of their accumulators together (q's pieces
// stand in all sixteen columns of the operand: column 4 j' + c is taken from MFMA j'), and masks and the new token's rows
// are looked at in the last tile and the last round only.
template <int MR>
__device__ __forceinline__ void step_attention(StepControl& ctl, const StepArgs& a, const StepPhase& p, uint16_t* cache_k, uint16_t* cache_v, const char* qkv, char* to,
                                               StepUnit unit, int n, bool pos_ok, uint8_t* lds, float* red)
{
    constexpr bool SPLIT = MR == 1;
    // NT: threads of the launch this stands for, whose sums run in their order; DW: dimensions of the output here
    constexpr int D = kStepHeadDim, NT = SPLIT ? 256 : 512, DW = SPLIT ? D : D / 2, DT = 8, CH = DW / DT, SLICES = kStepThreads / CH, GROUPS = kStepThreads / DW;
    static_assert(SLICES == NT / (D / DT) && GROUPS == NT / D, "the slices and groups of that launch");
    constexpr int VU = 4, KT = 2, ROUND = VU * SLICES;
    constexpr int NJ = D / 32, R = D / 32, SPM = 16 / R;
    static_assert(R == 4 && NJ == 4, "four pieces, four MFMAs a tile");
    float* part = reinterpret_cast<float*>(lds);
    float* part2 = part + SLICES * DW;
    float* score = part2 + GROUPS * DW;
    const int lane = p.lane, wave = p.wave, tid = 64 * wave + lane, H = p.H, KV = p.KV, S = a.S, SP = SPLIT ? p.SP : 1;
    const int per = H / KV, member = SPLIT ? unit.head : unit.head >> 1, dim0 = SPLIT ? 0 : DW * (unit.head & 1);
    const int b = SPLIT ? 0 : unit.group / KV, sp = SPLIT ? unit.group % SP : 0, kvh = SPLIT ? unit.group / SP : unit.group - b * KV;
    const int h = kvh * per + member, pb = a.per_seq ? b : 0;
    auto cache_slot = [&](int l) { return (((l >> 4) * SP + sp) << 4) + (l & 15); };
    uint16_t* kbase = cache_k + (static_cast<size_t>(b) * KV + kvh) * S * D;
    uint16_t* vbase = cache_v + (static_cast<size_t>(b) * KV + kvh) * S * D + dim0;
    const int tiles = (n + 15) >> 4, ltiles = tiles > sp ? (tiles - sp + SP - 1) / SP : 0, nl = 16 * ltiles;
    const int last_tile = (n - 1) >> 4;
    const uint32_t seen = static_cast<uint32_t>(n) * D * 2u;      // requests are bounded by the prefix
    const __amdgpu_buffer_rsrc_t rk = make_raw_buffer(kbase, seen), rv = make_raw_buffer(vbase, seen - 2 * dim0);
    const int r16 = lane & 15, kblk = lane >> 4, piece = (r16 & 3) + R * kblk, sl = r16 >> 2;
    const int chunk = tid % CH, slice = tid / CH;

    u32x4 kr[KT][NJ], vr[VU];
    auto load_keys = [&](int ltile, u32x4 (&dst)[NJ]) {         // (tiles past the last one too: the lane's offset says so)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            dst[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, (16 * (ltile * SP + sp) + SPM * j + sl) * D * 2 + 16 * piece, 0, 0));
    };
    auto load_value = [&](int l) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, (cache_slot(l) * D + chunk * DT) * 2, 0, 0)); };
#pragma unroll
    for (int t = 0; t < KT; ++t)
        if (wave + kStepWaves * t < ltiles) load_keys(wave + kStepWaves * t, kr[t]);
#pragma unroll
    for (int u = 0; u < VU; ++u) vr[u] = load_value(slice + u * SLICES);
    const f32x4 cs = *reinterpret_cast<const f32x4*>(a.cosv + pb * (D / 2) + 4 * piece);
    const f32x4 sn = *reinterpret_cast<const f32x4*>(a.sinv + pb * (D / 2) + 4 * piece);
    asm volatile("" ::: "memory");
    __syncthreads();                             // the last phase's finishing waves have read its accumulators

    u32x4 q_own, k_own, vnew;
    const int rows = H + 2 * KV;
    const __amdgpu_buffer_rsrc_t rq = make_raw_buffer(qkv, static_cast<uint32_t>(p.M) * rows * D * 2u);
    ctl.await([&]() {
        q_own = step_load16(rq, ((b * rows + h) * D + 8 * piece) * 2);
        k_own = step_load16(rq, ((b * rows + H + kvh) * D + 8 * piece) * 2);
        vnew = step_load16(rq, ((b * rows + H + KV + kvh) * D + dim0 + chunk * DT) * 2);
    }, [&]() { return step_max(step_max(step_largest(q_own), step_largest(k_own)), step_largest(vnew)) != kStepEmpty; });
    auto rotate = [&](const u32x4& own) {
        float x[8], y[8];
        unpack_bf16x8(own, x);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma clang fp contract(off)                   // as terna_rope_kv_store_kernel: every product and sum rounded once
            y[2 * m] = x[2 * m] * cs[m] - x[2 * m + 1] * sn[m];
            y[2 * m + 1] = x[2 * m + 1] * cs[m] + x[2 * m] * sn[m];
        }
        return pack_bf16x8(y);
    };
    const u32x4 qb = rotate(q_own), knew = rotate(k_own);
    if (member == 0 && sp == 0 && pos_ok) {      // this kv group's writer: slot pos of both caches
        if (dim0 == 0 && wave == 0 && r16 < R) *reinterpret_cast<u32x4*>(kbase + static_cast<size_t>(n - 1) * D + 8 * piece) = knew;
        if (slice == 0) *reinterpret_cast<u32x4*>(vbase + static_cast<size_t>(n - 1) * D + chunk * DT) = vnew;
    }

    // ---- scores
    float mx = -INFINITY;
    auto score_tile = [&](int ltile, const u32x4 (&kin)[NJ]) {
        const int tile = ltile * SP + sp;
        const bool last = tile == last_tile;     // uniform
        f32x4 acc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            u32x4 k = kin[j];
            if (last) k = 16 * tile + SPM * j + sl == n - 1 ? knew : k;
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k), __builtin_bit_cast(bf16x8, qb), zero, 0, 0, 0);
        }
        // column 4 j + c: component c of MFMA j, the partial score of slot 4 j + kblk; c runs over a quad
        float y[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const float lo = r16 & 1 ? acc[j][1] : acc[j][0], hi = r16 & 1 ? acc[j][3] : acc[j][2];
            y[j] = r16 & 2 ? hi : lo;
        }
        const float lo = sl & 1 ? y[1] : y[0], hi = sl & 1 ? y[3] : y[2];
        float x = sl & 2 ? hi : lo;
        x += dpp_permute<kDppSwapPairs>(x);
        x += dpp_permute<kDppSwapHalfQuads>(x);
        const int ls = SPM * sl + kblk;
        const float d = x * a.scale;
        if (!last || 16 * tile + ls < n) {
            if ((r16 & 3) == 0) score[16 * ltile + ls] = d;
            mx = fmaxf(mx, d);
        }
    };
    key_rounds<KT, kStepWaves>(wave, ltiles, kr, load_keys, score_tile);
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < kStepWaves; ++w) mx = fmaxf(mx, red[w]);

    // ---- softmax numerators and their sum
    float sums[NT / kStepThreads];
#pragma unroll
    for (int v = 0; v < NT / kStepThreads; ++v) {
        sums[v] = 0.0f;
        for (int l = tid + kStepThreads * v; l < nl; l += NT) {
            const float e = cache_slot(l) < n ? __expf(score[l] - mx) : 0.0f;
            score[l] = e;
            sums[v] += e;
        }
        sums[v] = wave_sum(sums[v]);
        if (lane == 0) red[8 + kStepWaves * v + wave] = sums[v];
    }
    __syncthreads();
    float sum = red[8];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) sum += red[8 + w];

    // ---- weighted sum of the value rows
    const int tid2 = 64 * wave + step_lane(), chunk2 = tid2 % CH, slice2 = tid2 / CH;
    float acc[DT];
#pragma unroll
    for (int e = 0; e < DT; ++e) acc[e] = 0.0f;
    for (int l0 = 0; l0 < nl; l0 += ROUND) {
        auto weigh = [&](float w, const u32x4& row) {
            float vf[8];
            unpack_bf16x8(row, vf);
#pragma unroll
            for (int e = 0; e < DT; ++e) acc[e] = fmaf(w, vf[e], acc[e]);
        };
        if (l0 + ROUND < nl) {                   // uniform: every row of the round stands in front of the last tile
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int l = l0 + slice2 + u * SLICES;
                weigh(score[l], vr[u]);
                vr[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, (cache_slot(l + ROUND) * D + chunk2 * DT) * 2, 0, 0));   // the next round's row in its place
            }
        } else {
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                if (l0 + u * SLICES >= nl) break;                  // uniform
                const int l = l0 + slice2 + u * SLICES, s = cache_slot(l);
                const bool ok = l < nl && s < n;
                u32x4 row = s == n - 1 ? vnew : vr[u];
                row = ok ? row : u32x4{0u, 0u, 0u, 0u};            // never multiply stale cache contents
                weigh(ok ? score[ok ? l : 0] : 0.0f, row);
            }
        }
    }
    *reinterpret_cast<f32x4*>(part + slice2 * DW + chunk2 * DT) = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *reinterpret_cast<f32x4*>(part + slice2 * DW + chunk2 * DT + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
    __syncthreads();
    {
        const int d = tid2 % DW, grp = tid2 / DW;
        float v[SLICES / GROUPS];
#pragma unroll
        for (int s8 = 0; s8 < SLICES / GROUPS; ++s8) v[s8] = part[(grp * (SLICES / GROUPS) + s8) * DW + d];
        float o = 0.0f;
#pragma unroll
        for (int s8 = 0; s8 < SLICES / GROUPS; ++s8) o += v[s8];
        part2[grp * DW + d] = o;
    }
    __syncthreads();
    if (tid2 < DW) {
        float o = 0.0f;
#pragma unroll
        for (int grp = 0; grp < GROUPS; ++grp) o += part2[grp * DW + tid2];
        if constexpr (SPLIT) {
            const __amdgpu_buffer_rsrc_t ro = make_raw_buffer(to + static_cast<size_t>(h * SP + sp) * kStepRecord, kStepRecord);
            __builtin_amdgcn_raw_buffer_store_b32(step_word(__float_as_uint(o)), ro, tid2 * 4, 0, kDeviceScope);
            if (tid2 < 2) __builtin_amdgcn_raw_buffer_store_b32(step_word(__float_as_uint(tid2 == 0 ? mx : sum)), ro, (D + tid2) * 4, 0, kDeviceScope);
        } else {
            const uint32_t v = float_to_bf16_bits(o / sum);
            const uint32_t pair = step_word(v | (dpp_permute_u32<kDppSwapPairs>(v) << 16));
            const __amdgpu_buffer_rsrc_t ro = make_raw_buffer(to + ((static_cast<size_t>(b) * H + h) * D + dim0) * 2, DW * 2);
            __builtin_amdgcn_raw_buffer_store_b32(pair, ro, (tid2 & 1) == 0 ? tid2 * 2 : kBufferOutOfRange, 0, kDeviceScope);
        }
    }
    __syncthreads();                             // the LDS goes to the next phase
}

// Norm + quantisation of a quarter of a row's columns (several sequences, in front of the down projection: repeating it
// for 6912 columns of every row in each of its 160 workgroups costs more than a hand-over).  unit = 4 row + quarter; every
// unit forms the row's statistics, then quantises every fourth of the waves' rounds.
template <int MR>
__device__ __forceinline__ void step_quantise(StepControl& ctl, const StepPhase& p, const uint16_t* norm_w, const char* from, char* to, char* scales, int unit,
                                              uint8_t* lds, float2* nowhere)
{
    using Op = StepOperands<1, 1, 7, 0, 1>;      // the lanes' columns: one row
    const int lane = p.lane, wave = p.wave, m = unit >> 2, quarter = unit & 3, K = p.ffn;
    const int first = wave * Op::TPW, ktiles = K >> 6, t0 = lane >> 4;
    float2* partials = reinterpret_cast<float2*>(lds + kStepWaves * StepLds<MR>::kSlab);
    u32x2 nw[Op::ROUNDS], xr[Op::ROUNDS];
    const __amdgpu_buffer_rsrc_t rn = make_raw_buffer(norm_w, static_cast<uint32_t>(K) * 2u);
#pragma unroll
    for (int r = 0; r < Op::ROUNDS; ++r) {
        const int t = r * 4 + t0;
        nw[r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(
                                              rn, t < Op::TPW && first + t < ktiles ? ((first + t) * 64 + 4 * (lane & 15)) * 2 : kBufferOutOfRange, 0, 0));
    }
    asm volatile("" ::: "memory");
    step_fetch_rows<1, Op>(ctl, from + static_cast<size_t>(m) * K * 2, 1, K, xr, lane, wave, [] {});
    step_partials<STEP_GROUPS, Op>(xr, nw, partials, nowhere, first, t0, ktiles, lane);
    __syncthreads();
    const StepScale sc = step_row_scale<STEP_GROUPS, kStepWideTiles>(partials, K, p.eps, p.quant_mode, lane);
    const __amdgpu_buffer_rsrc_t rq = make_raw_buffer(to + static_cast<size_t>(m) * K, static_cast<uint32_t>(K));
#pragma unroll
    for (int r = 0; r < Op::ROUNDS; ++r) {
        if ((r & 3) != quarter) continue;        // uniform
        const uint32_t hd[2] = {xr[r].x, xr[r].y}, wd[2] = {nw[r].x, nw[r].y};
        uint32_t d[1];
        chain_quantise<4>(hd, wd, sc.rstd, sc.mul, p.quant_mode, d);
        const int t = r * 4 + t0;
        // the integers lie in [-127, 127] (QUANT_EAGER is refused): flipped, no word of them is the empty one
        __builtin_amdgcn_raw_buffer_store_b32(d[0] ^ 0x7f7f7f7fu, rq, t < Op::TPW && first + t < ktiles ? (first + t) * 64 + 4 * (lane & 15) : kBufferOutOfRange, 0,
                                              kDeviceScope);
    }
    if (quarter == 0 && wave == 0) {
        const __amdgpu_buffer_rsrc_t rs = make_raw_buffer(scales + m * 64, 4);
        __builtin_amdgcn_raw_buffer_store_b32(step_word(__float_as_uint(sc.s)), rs, lane == 0 ? 0 : kBufferOutOfRange, 0, kDeviceScope);
    }
    __syncthreads();                             // the partials are read before the next phase writes its own
}

// Lines of device memory on their way into the L2 of this XCD, without a register: a word of each goes to a place in LDS nobody
// reads.  The lane's line begins at byte `at`; past the range nothing is read.  (asm: the compiler would wait for the builtin's LDS
// writes in front of the next LDS access of any kind.)
__device__ __forceinline__ void step_prefetch(const void* base, int bytes, int at, uint32_t lds_words)
{
    const uint64_t from = reinterpret_cast<uint64_t>(base);
    const i32x4 range = {static_cast<int>(from), static_cast<int>(from >> 32), bytes, kBufferRsrcFlags};
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_words), "v"(at), "s"(range) : "memory");
}

// Slots of a sequence's prefix; negative: its position lies outside the cache (clamped).
__device__ __forceinline__ int step_seen(const StepArgs& a, int sequence)
{
    const long long p = a.pos[a.per_seq ? sequence : 0];
    return __builtin_amdgcn_readfirstlane(p < 0 ? -1 : p >= a.S ? -a.S : static_cast<int>(p) + 1);
}

// ORDERED: the next unit, once it may start, for the whole workgroup; a block past the last where there is none.
__device__ __forceinline__ StepTicket step_take(const StepArgs& a, StepTicket* shared, bool first)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // this wave's outputs have arrived
    __syncthreads();
    if (threadIdx.x == 0) {
        if (!first) __hip_atomic_fetch_add(a.tickets + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int mine = static_cast<int>(__hip_atomic_fetch_add(a.tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1);
        StepTicket t = step_ticket(mine, a.M, a.dim, a.ffn, a.H, a.KV, a.SP);
        bool ready = t.block >= a.blocks;
        for (int polls = 0; !ready && polls < kStepOrderedPolls; ++polls)
            ready = static_cast<int>(__hip_atomic_load(a.tickets + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1) >= t.before;
        if (!ready) t.block = a.blocks;
        *shared = t;
    }
    __syncthreads();
    asm volatile("" ::: "memory");
    return {__builtin_amdgcn_readfirstlane(shared->block), __builtin_amdgcn_readfirstlane(shared->kind), __builtin_amdgcn_readfirstlane(shared->w), 0};
}

template <int MR, bool ORDERED>
__global__ __launch_bounds__(kStepThreads, ORDERED ? 2 : 4) void terna_decode_step_kernel(const StepArgs a)
{
    if constexpr (ORDERED) {
        if (__hip_atomic_load(a.alive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return;     // the step is done
    }
    using Lds = StepLds<MR>;
    constexpr bool QUANT = MR >= 2;              // the down projection's rows quantised by a phase of its own
    __shared__ __align__(16) uint8_t lds[Lds::kBytes];
    __shared__ StepScale scale_s[4];
    __shared__ float red[8 + 8];
    __shared__ StepMerge merge_s[MR == 1 ? kStepWaves : 1][8];
    // pointers and weight scales of all blocks: a first touch of either costs a microsecond, and a phase would wait for it
    __shared__ __align__(16) StepBlock block_s[kStepMaxBlocks];
    __shared__ uint16_t weight_s[kStepMaxBlocks][16];             // QKV, O, gate+up, down: four each
    __shared__ uint32_t dummy_s[64];
    __shared__ float2 nowhere_s;
    __shared__ StepTicket ticket_s;              // (ORDERED)
    __shared__ int sharing_s;                    // prefetch_cache: how many share a unit's keys and values << 16 | which of them this is
    // What the lanes of wave 0 keep for the columns they finish -- row lane >> 4, column lane & 15 of band w: the residual stream, and the
    // weight-scale groups of QKV, O and down.  (In registers they would be spilled, and a load of a spilled register waits behind
    // the prefetches like any other.)
    __shared__ float stream_s[64];
    __shared__ uint8_t group_s[3][64];
    __shared__ __align__(16) StepShape shape_s;
    static_assert(sizeof(lds) + sizeof(scale_s) + sizeof(red) + sizeof(merge_s) + sizeof(block_s) + sizeof(weight_s) + sizeof(dummy_s) + sizeof(stream_s) + sizeof(group_s) + 96 <= 40 * 1024, "a quarter of a CU");
    const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int w0 = ORDERED ? -1 : blockIdx.x;          // (ORDERED: of the unit that is being done)
    if (threadIdx.x == 0) shape_s = StepShape{a.M, a.dim, a.ffn, a.H, a.KV, a.SP, a.quant_mode, a.eps};
    __syncthreads();
    auto uniform = [](int v) { return ORDERED ? __builtin_amdgcn_readfirstlane(v) : v; };      // (what another unit changes)
    auto phase = [&]() {
        StepPhase p;
        p.M = __builtin_amdgcn_readfirstlane(shape_s.M);
        p.dim = __builtin_amdgcn_readfirstlane(shape_s.dim);
        p.ffn = __builtin_amdgcn_readfirstlane(shape_s.ffn);
        p.H = __builtin_amdgcn_readfirstlane(shape_s.H);
        p.KV = __builtin_amdgcn_readfirstlane(shape_s.KV);
        p.SP = __builtin_amdgcn_readfirstlane(shape_s.SP);
        p.quant_mode = __builtin_amdgcn_readfirstlane(shape_s.quant_mode);
        p.eps = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(shape_s.eps)));
        p.lane = step_lane();
        p.wave = step_uniform(wave0);
        p.w = step_uniform(uniform(w0));
        p.wide = p.H * kStepHeadDim;
        p.qkv_n = (p.H + 2 * p.KV) * kStepHeadDim;
        return p;
    };
    bool has_qkv, has_out, has_gate, has_unit, has_quant;
    bool out_now, down_now;                      // ORDERED: which of has_out's two phases
    StepUnit unit;
    int seen = 0;                                // slots of the unit's prefix; negative: the position lies outside the cache (clamped)
    auto find_groups = [&](const StepPhase& p) {
        const int fin_n = 16 * p.w + (p.lane & 15);
        group_s[0][p.lane] = has_qkv && a.ws_qkv != 1 ? ws_group_decode(fin_n, p.qkv_n, a.ws_qkv) : 0;
        group_s[1][p.lane] = has_out && a.ws_o != 1 ? ws_group_decode(fin_n, p.dim, a.ws_o) : 0;
        group_s[2][p.lane] = has_out && a.ws_2 != 1 ? ws_group_decode(fin_n, p.dim, a.ws_2) : 0;
    };
    {
        const StepPhase p = phase();
        if constexpr (!ORDERED) {
            unit = step_unit(p.w, MR == 1 ? p.KV * p.SP : p.M * p.KV, p.H / p.KV * (MR == 1 ? 1 : 2));
            has_qkv = p.w < p.qkv_n >> 4;
            has_out = p.w < p.dim >> 4;
            has_gate = 4 * p.w < p.ffn >> 3;
            has_unit = unit.group >= 0;
            if (has_unit) seen = step_seen(a, MR == 1 ? 0 : unit.group / p.KV);        // (once: a load behind the prefetches would wait for them)
            has_quant = QUANT && kStepGroups - 1 - p.w < 4 * p.M;
            if (has_unit) {
                const int per = p.H / p.KV * (MR == 1 ? 1 : 2), past = MR == 1 ? 0 : step_unit_past(unit, per, p.qkv_n >> 4);
                sharing_s = (per - past) << 16 | (unit.head - past);      // (of those past the bands, with several sequences: not read)
            }
            if (p.wave == 0) {
                find_groups(p);
                stream_s[p.lane] = has_out && (p.lane >> 4) < p.M ? bf16_bits_to_float(a.x[(p.lane >> 4) * p.dim + 16 * p.w + (p.lane & 15)]) : 0.0f;
            }
        }
        const int tid = 64 * p.wave + p.lane;
        const uint32_t* from = reinterpret_cast<const uint32_t*>(a.block);
        uint32_t* to = reinterpret_cast<uint32_t*>(block_s);
        for (int i = tid; i < static_cast<int>(sizeof(block_s) / 4); i += kStepThreads) to[i] = from[i];
        __syncthreads();
        for (int i = tid; i < 16 * a.blocks; i += kStepThreads) {
            const int n = i >> 4, which = (i >> 2) & 3, g = i & 3;
            const StepBlock& blk = block_s[n];
            const uint16_t* ws = which == 0 ? blk.ws_qkv : which == 1 ? blk.ws_o : which == 2 ? blk.ws_13 : blk.ws_2;
            const int held = which == 0 ? a.ws_qkv : which == 1 ? a.ws_o : which == 2 ? 2 : a.ws_2, cols = which == 0 ? p.qkv_n : p.dim;
            // (columns that the groups do not divide: ws_group_decode's last group is one more)
            weight_s[n][4 * which + g] = ws[g < held || (which != 2 && g == held && cols % held != 0) ? g : 0];
        }
        __syncthreads();
    }
    StepControl ctl{a.alive, false}; // (ORDERED: step_take has waited, every poll finds its words)
    const uint32_t dummy = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint32_t*)dummy_s));

    // (operands expanded ahead of the wait: as many as the registers of the phase hold)
    using Narrow = StepOperands<MR, 1, 2, 2, MR == 4 ? 8 : 10>;
    using Out = StepOperands<MR, 1, 2, 2, MR == 1 ? 3 : MR == 2 ? 10 : 8>;
    using Gate = StepOperands<MR, 4, 2, 2, MR == 1 ? 16 : MR == 2 ? 12 : 5>;
    using Down = StepOperands<MR, 1, 7, 0, MR == 4 ? 14 : 16, !QUANT>;
    auto pointer = [](auto* held) {              // a pointer out of LDS, in scalar registers
        const uint64_t v = reinterpret_cast<uint64_t>(held);
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
        return reinterpret_cast<decltype(held)>(static_cast<uint64_t>(hi) << 32 | lo);
    };
    auto outputs = [](int sum, float s, uint32_t ws) {
        EpilogueRegs e;
        e.s = s;
        e.w[0] = __uint_as_float(ws << 16);
        return apply_epilogue<int>(EP_I8_DECODE, e, 0, sum);
    };
    // The next block's matrix of this phase (this workgroup's bands of it) and its norm weights (a few lines by every workgroup of
    // the XCD), right behind a wait: in front of one its polls would return behind the lines.
    auto prefetch = [&](const StepPhase& p, const uint32_t* packed, int band0, int bands, const uint16_t* norm_w, int K) {
        if constexpr (ORDERED) return;
        const int bytes = bands * (K >> 6) * 256;
        for (int l = p.wave; 8192 * l < bytes; l += kStepWaves) step_prefetch(packed + static_cast<size_t>(band0) * K, bytes, (64 * l + p.lane) * 128, dummy);
        if (p.wave == kStepWaves - 1) step_prefetch(norm_w, 2 * K, (p.lane < 4 ? 4 * (p.w >> 3) + p.lane : 1 << 20) * 128, dummy);
    };
    // A block's keys and values, what the unit's group reads of them shared out over its workgroups, right behind the wait for the
    // stream.  Those past the bands of QKV, which do not wait there: one sequence, at any time before their attention (4096 slots, filled to 90 %, 901 -> 867 us
    // a step, 8192 1130 -> 1048; left to the others 879 and 1102); several, nothing, the others take their shares (two, 1280 slots 986 -> 944, four,
    // 1024 1046 -> 1016; by themselves 934 and 1021, but for the registers of a second copy of this code 5 - 9 more in short caches).
    auto prefetch_cache = [&](const StepPhase& p, int n) {
        if constexpr (!ORDERED) {
            const int b = MR == 1 ? 0 : unit.group / p.KV, kvh = MR == 1 ? unit.group / p.SP : unit.group - b * p.KV;
            const int split = MR == 1 ? unit.group % p.SP : 0, splits = MR == 1 ? p.SP : 1;
            const int sharing = __builtin_amdgcn_readfirstlane(sharing_s), members = sharing >> 16;
            const int bytes = 2 * kStepHeadDim * (seen < 0 ? -seen : seen);
            const size_t at = (static_cast<size_t>(b) * p.KV + kvh) * a.S * kStepHeadDim;
            const uint16_t *k = pointer(block_s[n].cache_k) + at, *v = pointer(block_s[n].cache_v) + at;
#pragma unroll 1
            for (int share = (sharing & 0xffff) + members * p.wave; step_cache_share(share, split, splits, bytes); share += members * kStepWaves) {
                const int line = step_cache_line(share, p.lane, split, splits);
                step_prefetch(k, bytes, line, dummy);
                step_prefetch(v, bytes, line, dummy);
            }
        }
    };
    for (int n = 0; ORDERED || n < a.blocks; ++n) {
        if constexpr (ORDERED) {                 // the next unit: of the phases below, its one alone is this workgroup's
            const StepTicket t = step_take(a, &ticket_s, w0 < 0);
            if (t.block >= a.blocks) break;
            n = t.block;
            w0 = t.w;
            has_qkv = t.kind == STEP_QKV, out_now = t.kind == STEP_OUT, has_gate = t.kind == STEP_GATE, has_quant = t.kind == STEP_QUANT, down_now = t.kind == STEP_DOWN;
            has_out = out_now || down_now, has_unit = t.kind == STEP_ATTENTION;
            const StepPhase p = phase();
            if (has_unit) {
                unit = step_unit(p.w, MR == 1 ? p.KV * p.SP : p.M * p.KV, p.H / p.KV * (MR == 1 ? 1 : 2));
                has_unit = unit.group >= 0;
                seen = has_unit ? step_seen(a, MR == 1 ? 0 : unit.group / p.KV) : 0;
            }
            if (p.wave == 0) {
                find_groups(p);
                // the stream of the columns: what their last phase handed over
                const char* from = a.exchange + static_cast<size_t>(n) * a.at.bytes;
                from = down_now ? from + a.at.mid : n == 0 ? reinterpret_cast<const char*>(a.x) : from - a.at.bytes + a.at.out;
                const __amdgpu_buffer_rsrc_t rx = make_raw_buffer(from, static_cast<uint32_t>(p.M) * p.dim * 2u);
                const bool mine = has_out && (p.lane >> 4) < p.M;
                const uint16_t bits = __builtin_amdgcn_raw_buffer_load_b16(rx, mine ? ((p.lane >> 4) * p.dim + 16 * p.w + (p.lane & 15)) * 2 : kBufferOutOfRange, 0, kDeviceScope);
                stream_s[p.lane] = bf16_bits_to_float(bits);
            }
            __syncthreads();
        }
        char* ex = a.exchange + static_cast<size_t>(n) * a.at.bytes;
        const int ahead = n + 1 < a.blocks ? n + 1 : n;
        // ---- QKV
        if (has_qkv) {
            const StepPhase p = phase();
            Narrow op;
            op.request(pointer(block_s[n].wqkv), p.qkv_n >> 4, p.w, p.dim, pointer(block_s[n].attention_norm), p.lane, p.wave);
            u32x2 xr[Narrow::ROUNDS];
            step_fetch_rows<MR, Narrow>(ctl, n == 0 ? reinterpret_cast<const char*>(a.x) : ex - a.at.bytes + a.at.out, p.M, p.dim, xr, p.lane, p.wave, [&] { op.expand(); });
            if (has_out) prefetch(p, pointer(block_s[n].wo), p.w, 1, pointer(block_s[n].attn_sub_norm), p.wide);
            if (has_gate) prefetch(p, pointer(block_s[n].w13), 4 * p.w, 4, pointer(block_s[n].ffn_norm), p.dim);
            if (!has_gate) prefetch(p, pointer(block_s[ahead].wqkv), p.w, 1, pointer(block_s[ahead].attention_norm), p.dim);
            if (has_unit) prefetch_cache(p, n);
            const float s = step_norm_linear<MR, STEP_GROUPS, kStepTiles, 1>(op, xr, p, p.dim, n == 0 ? a.stats : nullptr, a.stats_count, lds, &nowhere_s, scale_s);
            if (p.wave == 0) {
                const uint16_t o = outputs(step_band_sum<MR>(lds, 0, p.lane), s, weight_s[n][group_s[0][p.lane]]);
                step_store_pair(make_raw_buffer(ex + a.at.qkv, static_cast<uint32_t>(p.M) * p.qkv_n * 2u), o, p.qkv_n, 16 * p.w + (p.lane & 15), (p.lane >> 4) < p.M, p.lane);
            }
        }
        // ---- attention
        if (has_unit) {
            if (MR == 1 && !has_qkv) prefetch_cache(phase(), n);
            const StepPhase p = phase();
            step_attention<MR>(ctl, a, p, pointer(block_s[n].cache_k), pointer(block_s[n].cache_v), ex + a.at.qkv, ex + a.at.attention, StepUnit{step_uniform(uniform(unit.group)), step_uniform(uniform(unit.head))},
                               seen < 0 ? -seen : seen, seen > 0, lds, red);
        }
        // ---- O projection, added to the stream
        if (ORDERED ? out_now : has_out) {
            const StepPhase p = phase();
            Out op;
            op.request(pointer(block_s[n].wo), p.dim >> 4, p.w, p.wide, pointer(block_s[n].attn_sub_norm), p.lane, p.wave);
            u32x2 xr[Out::ROUNDS];
            if constexpr (MR == 1) step_fetch_merged<Out, ORDERED>(ctl, ex + a.at.attention, p.H, p.SP, xr, merge_s[p.wave], p.lane, p.wave, [&] { op.expand(); });
            else step_fetch_rows<MR, Out>(ctl, ex + a.at.attention, p.M, p.wide, xr, p.lane, p.wave, [&] { op.expand(); });
            prefetch(p, pointer(block_s[n].w2), p.w, 1, pointer(block_s[n].ffn_sub_norm), p.ffn);
            const float s = step_norm_linear<MR, MR == 1 ? STEP_CHUNKS : STEP_HEADS, kStepTiles, 1>(op, xr, p, p.wide, nullptr, 0, lds, &nowhere_s, scale_s);
            if (p.wave == 0) {
                const bool row_ok = (p.lane >> 4) < p.M;
                const uint16_t o = outputs(step_band_sum<MR>(lds, 0, p.lane), s, weight_s[n][4 + group_s[1][p.lane]]);
                const float stream = row_ok ? round_bf16(stream_s[p.lane] + bf16_bits_to_float(o)) : 0.0f;
                stream_s[p.lane] = stream;
                step_store_pair(make_raw_buffer(ex + a.at.mid, static_cast<uint32_t>(p.M) * p.dim * 2u), float_to_bf16_bits(stream), p.dim, 16 * p.w + (p.lane & 15), row_ok, p.lane);
            }
        }
        // ---- gate+up
        if (has_gate) {
            const StepPhase p = phase();
            Gate op;
            op.request(pointer(block_s[n].w13), p.ffn >> 3, 4 * p.w, p.dim, pointer(block_s[n].ffn_norm), p.lane, p.wave);
            u32x2 xr[Gate::ROUNDS];
            step_fetch_rows<MR, Gate>(ctl, ex + a.at.mid, p.M, p.dim, xr, p.lane, p.wave, [&] { op.expand(); });
            if (has_qkv) prefetch(p, pointer(block_s[ahead].wqkv), p.w, 1, pointer(block_s[ahead].attention_norm), p.dim);
            const float s = step_norm_linear<MR, STEP_GROUPS, kStepTiles, 4>(op, xr, p, p.dim, nullptr, 0, lds, &nowhere_s, scale_s);
            if (p.wave < 2) {                    // a gate / up pair each
                const float x1 = bf16_bits_to_float(outputs(step_band_sum<MR>(lds, 2 * p.wave, p.lane), s, weight_s[n][8]));
                const float x3 = bf16_bits_to_float(outputs(step_band_sum<MR>(lds, 2 * p.wave + 1, p.lane), s, weight_s[n][9]));
                const float r = max_keep_nan(x1, 0.0f);
                step_store_pair(make_raw_buffer(ex + a.at.inner, static_cast<uint32_t>(p.M) * p.ffn * 2u), float_to_bf16_bits(round_bf16(r * r) * x3), p.ffn,
                                (2 * p.w + p.wave) * 16 + (p.lane & 15), (p.lane >> 4) < p.M, p.lane);
            }
        }
        // ---- down projection, added to the stream
        if constexpr (QUANT) {
            if (has_quant) {
                const StepPhase p = phase();
                step_quantise<MR>(ctl, p, pointer(block_s[n].ffn_sub_norm), ex + a.at.inner, ex + a.at.quantised, ex + a.at.scales, kStepGroups - 1 - p.w, lds, &nowhere_s);
            }
        }
        if (ORDERED ? down_now : has_out) {
            const StepPhase p = phase();
            Down op;
            op.request(pointer(block_s[n].w2), p.dim >> 4, p.w, p.ffn, pointer(block_s[n].ffn_sub_norm), p.lane, p.wave);
            float s;
            if constexpr (QUANT) {
                constexpr int PIECES = Down::TPW * 4, VEC = (MR * PIECES + 63) / 64;         // 16-byte pieces of a wave's rows
                const __amdgpu_buffer_rsrc_t rx = make_raw_buffer(ex + a.at.quantised, static_cast<uint32_t>(p.M) * p.ffn);
                const __amdgpu_buffer_rsrc_t rs = make_raw_buffer(ex + a.at.scales, static_cast<uint32_t>(p.M) * 64u);
                uint8_t* slab = lds + p.wave * Lds::kSlab;
                __syncthreads();                 // the last phase's finishing waves have read its accumulators (a wave past K waits for nothing)
                u32x4 v[VEC];
                uint32_t sc;
                ctl.await([&]() {
#pragma unroll
                    for (int j = 0; j < VEC; ++j) {
                        const int at = p.lane + 64 * j, row = at / PIECES, col = p.wave * Down::TPW * 64 + 16 * (at % PIECES);
                        v[j] = step_load16(rx, row < p.M && col < p.ffn ? row * p.ffn + col : kBufferOutOfRange);
                    }
                    sc = __builtin_amdgcn_raw_buffer_load_b32(rs, (p.lane >> 4) < p.M ? (p.lane >> 4) * 64 : kBufferOutOfRange, 0, kDeviceScope);
                }, [&]() {
                    uint32_t top = sc;
#pragma unroll
                    for (int j = 0; j < VEC; ++j) top = step_max(top, step_largest(v[j]));
                    return top != kStepEmpty;
                }, [&] { op.expand(); });
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    const int at = p.lane + 64 * j, row = at / PIECES, col = p.wave * Down::TPW * 64 + 16 * (at % PIECES);
                    if (row < MR) *reinterpret_cast<u32x4*>(slab + row * Lds::kPitch + 16 * (at % PIECES)) = v[j] ^ (row < p.M && col < p.ffn ? 0x7f7f7f7fu : 0u);
                }
                i32x4 acc[1];
                op.multiply(slab, acc, p.lane);
                if ((p.lane & 15) < MR) *reinterpret_cast<i32x4*>(slab + (p.lane & 15) * 64 + 16 * (p.lane >> 4)) = acc[0];
                __syncthreads();
                s = __uint_as_float(sc);
            } else {
                u32x2 xr[Down::ROUNDS];
                step_fetch_rows<MR, Down>(ctl, ex + a.at.inner, p.M, p.ffn, xr, p.lane, p.wave, [&] { op.expand(); });
                s = step_norm_linear<MR, STEP_GROUPS, kStepWideTiles, 1>(op, xr, p, p.ffn, nullptr, 0, lds, &nowhere_s, scale_s);
            }
            if (p.wave == 0) {
                const bool row_ok = (p.lane >> 4) < p.M;
                const uint16_t o = outputs(step_band_sum<MR>(lds, 0, p.lane), s, weight_s[n][12 + group_s[2][p.lane]]);
                const float stream = row_ok ? round_bf16(stream_s[p.lane] + bf16_bits_to_float(o)) : 0.0f;
                stream_s[p.lane] = stream;
                char* to = n + 1 == a.blocks ? reinterpret_cast<char*>(a.x_out) : ex + a.at.out;
                step_store_pair(make_raw_buffer(to, static_cast<uint32_t>(p.M) * p.dim * 2u), float_to_bf16_bits(stream), p.dim, 16 * p.w + (p.lane & 15), row_ok, p.lane);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // the last prefetches have written their words: the LDS may go
}

}  // namespace terna
