// TernaSpMM kernel on the P2 layout for the row counts between a decode step and a long prompt (17 rows .. a few hundred).
//
// What bounds it: neither bytes nor MFMA but what ONE CU has to pull through its 64 bytes a clock and the round trips it
// waits for one after the other.  A workgroup owns 16 RT rows x 16 FB features over all of K, so it reads
// 16 RT * K activations and 16 FB * K / 4 bytes of weights, whatever the chip is doing; the MFMA-tiled kernel of the long
// prompts walks K in dependent steps of half a microsecond (20 steps for K = 2560), and the ring kernel of the small
// batches stages every activation through registers.  So here
//   * K is split over the workgroup's waves: a wave takes chunks of 256 columns (w, w + W, ...) and requests everything a
//     chunk needs before it waits for anything; the other waves and workgroups of the CU fill the wait (two chunks in
//     flight per wave bought nothing: the second slot halves the workgroups that fit);
//   * weights: one 16-byte load per lane and band fetches four band-tiles; MFMA number c of the chunk takes component c of
//     every lane (the operand order of decode_chunk_kernel.h: the k index runs over (tile, column));
//   * activations: global -> LDS directly (16 bytes per lane, whole 256 / 512-byte row pieces), wave-private slots, so no
//     barrier before the sum; 16-byte piece p of row r sits at p ^ (r & 15), which spreads the operand reads over all banks;
//   * a weight is expanded once for all RT row tiles, an activation operand read once for all FB bands;
//   * the waves' partial sums meet in LDS (each wave's in place of its activations, 16-byte units XOR-swizzled by the row)
//     behind the only barrier, are added in wave order (bit-reproducible; integer sums exact) and leave as whole rows.
// Every load of the main part is issued and awaited by hand (see prefill_packed_kernel.h).
// Measured, us per launch, weights rotating over 20 copies, ring / MFMA-tiled kernel before -> this kernel (tile choice:
// launch_mid.hip):             QKV 2560->3840   O 2560->2560   gate+up 2560->13824   down 6912->2560
//   bf16 M = 37                6.9 -> 5.0       6.8 -> 4.1     16.5 -> 8.6            13.3 -> 6.4
//   bf16 M = 100               12.1 -> 6.3      11.5 -> 6.1    16.7 -> 14.3           15.3 -> 10.5
//   int8 M = 37                5.5 -> 4.5       5.4 -> 3.9     11.4 -> 6.8            9.4 -> 5.2
//   int8 M = 100               7.7 -> 5.3       7.5 -> 5.2     11.4 -> 10.0           12.9 -> 7.8
//   int8 M = 300               10.9 -> 8.8      11.1 -> 6.7    16.4 (stays)           16.3 -> 11.1
#pragma once

#include "prefill_packed_kernel.h"

namespace terna {

constexpr int kMidMaxWaves = 12;

template <typename Act, int RT, int FB>
struct MidShape {
    static constexpr int kRowBytes = 256 * static_cast<int>(sizeof(Act));    // a chunk's piece of one activation row
    static constexpr int kWaveBytes = 16 * RT * kRowBytes;                     // a wave's LDS: activations, then partial sums
    static_assert(FB == 2 || FB == 4, "result rows of 8 or 16 units: see the swizzle of the partial sums");
    static_assert(RT * FB * 1024 <= kWaveBytes, "partial sums (1 KB per 16 x 16 tile) take the place of the activations");
};

// EPI: plain outputs, the sum with the stream, the feed-forward gate or the rotary embedding and cache write (see the epilogues of prefill_packed_kernel.h)
template <typename Act, int RT, int FB, bool GUARD, int EPI = PACKED_STORE>
__global__ __launch_bounds__(kMidMaxWaves * 64) void terna_mid_kernel(
    const Act* __restrict__ x, const uint32_t* __restrict__ packed, uint16_t* __restrict__ out,
    int M, int N, int K, int row_tiles, int waves, Epilogue ep, PackedExtra<EPI> guard)
{
    if constexpr (GUARD) {
        if (blockIdx.x == 0) {
            if (threadIdx.x < 64) repack_guard_role(guard, threadIdx.x);
            return;
        }
    }
    using T = ActTraits<Act>;
    using Acc = typename T::Acc;
    using AccScalar = typename T::AccScalar;
    using S = MidShape<Act, RT, FB>;
    constexpr bool BF16 = sizeof(Act) == 2;
    constexpr int SZ = static_cast<int>(sizeof(Act));
    constexpr int PIECES = 16 * SZ;                      // 16-byte pieces of a chunk row
    constexpr int ROWS_PER_LOAD = 64 / PIECES;           // rows one direct load fills
    constexpr int XI = 16 * RT / ROWS_PER_LOAD;          // direct loads per chunk
    extern __shared__ __align__(16) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroups go to the XCDs round robin: the row tiles of a feature tile follow each other on one XCD, so its weights
    // cross the fabric once.  The grid is padded to whole rounds of 8 feature tiles.
    const int index = static_cast<int>(blockIdx.x) - (GUARD ? 1 : 0);
    const int slot_of_xcd = index >> 3;
    const int round = __builtin_amdgcn_readfirstlane(slot_of_xcd / row_tiles);
    const int ftile = (index & 7) + 8 * round;
    const int m0 = (slot_of_xcd - round * row_tiles) * (16 * RT);
    if (ftile * (16 * FB) >= N) return;
    const int ktiles = K >> 6, chunks = (ktiles + 3) >> 2;
    const int band0 = ftile * FB;
    const int i = lane & 15, g = lane >> 4;
    const int rowbytes = K * SZ;

    // ---- this lane's place in the loads
    const uint8_t* wbase = reinterpret_cast<const uint8_t*>(packed) + static_cast<size_t>(band0) * ktiles * 256;
    const uint8_t* xbase = reinterpret_cast<const uint8_t*>(x);
    const int r0 = lane / PIECES, piece0 = (lane % PIECES) ^ r0;
    uint32_t xrow[XI];                                   // rows past M read the last one: never stored
#pragma unroll
    for (int j = 0; j < XI; ++j) {
        const int m = m0 + r0 + ROWS_PER_LOAD * j;
        xrow[j] = static_cast<uint32_t>(m < M ? m : M - 1) * static_cast<uint32_t>(rowbytes);
    }
    uint8_t* mine = smem + wave * S::kWaveBytes;
    const uint32_t lds_mine = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(mine));

    struct RawW { u32x4 w[FB]; };
    RawW rw;
    auto issue = [&](int at_chunk) __attribute__((always_inline)) {
        const int chunk = __builtin_amdgcn_readfirstlane(at_chunk);
        // columns past K (a partial last chunk): loads pulled back into the row, zeros in place of their activations before these are used
        const int tile0 = chunk * 4;
        const int left = ktiles - 1 - tile0;
        const uint32_t woff = static_cast<uint32_t>(tile0 * 256 + (g < left ? g : left) * 256 + i * 16);
#pragma unroll
        for (int b = 0; b < FB; ++b) global_load_b128_nowait(rw.w[b], wbase + static_cast<size_t>(b) * ktiles * 256, woff);
        const int col = chunk * S::kRowBytes;
        const int last = left < 3 ? rowbytes - 16 - col : S::kRowBytes;
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            const int at = (piece0 ^ ((ROWS_PER_LOAD * j) & 15)) * 16;
            lds_dma_b128(xbase + col, xrow[j] + (at < last ? at : last), lds_mine + j * 1024);
        }
    };

    Acc acc[RT][FB];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int b = 0; b < FB; ++b) acc[r][b] = Acc{0, 0, 0, 0};

    // Tiles that do not exist: what was loaded in their place are other activations of the row, which may be infinite, and zero weights
    // would make NaN of them.  Each lane clears what it is going to read.
    auto clear_past_end = [&](int chunk) __attribute__((always_inline)) {
        if (chunk * 4 + 4 <= ktiles) return;             // uniform
        if (chunk * 4 + g < ktiles) return;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int p = 0; p < 4 * SZ; ++p)
                *reinterpret_cast<u32x4*>(mine + (16 * r + i) * S::kRowBytes + (((4 * SZ * g + p) ^ i) * 16)) = u32x4{0u, 0u, 0u, 0u};
    };
    // the activations that MFMA number c of a chunk (bf16: numbers 2 c and 2 c + 1) takes, read one c ahead of their use
    constexpr int HALVES = BF16 ? 2 : 1;
    struct Ops { u32x4 v[RT][HALVES]; };
    auto read = [&](int c, Ops& o) __attribute__((always_inline)) {
        const uint8_t* src = mine + i * S::kRowBytes;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int h = 0; h < HALVES; ++h)
                o.v[r][h] = *reinterpret_cast<const u32x4*>(src + 16 * r * S::kRowBytes + (((4 * HALVES * g + HALVES * c + h) ^ i) * 16));
    };
    auto multiply = [&] __attribute__((always_inline)) {
        Ops ops[2];
        read(0, ops[0]);
#pragma unroll
        for (int b = 0; b < FB; ++b) landed(rw.w[b]);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            __builtin_amdgcn_sched_barrier(0);                           // keeps the reads ahead
            if (c < 3) read(c + 1, ops[(c + 1) & 1]);
            const Ops& now = ops[c & 1];
            if constexpr (BF16) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    bf16x8 a[FB];
#pragma unroll
                    for (int b = 0; b < FB; ++b) a[b] = __builtin_bit_cast(bf16x8, expand_chunk_bf16(h ? rw.w[b][c] : rw.w[b][c] << 4));
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int b = 0; b < FB; ++b)
                            acc[r][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[b], __builtin_bit_cast(bf16x8, now.v[r][h]), acc[r][b], 0, 0, 0);
                }
            } else {
                i32x4 a[FB];
#pragma unroll
                for (int b = 0; b < FB; ++b) a[b] = expand_word_i8(rw.w[b][c]);
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int b = 0; b < FB; ++b)
                        acc[r][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[b], __builtin_bit_cast(i32x4, now.v[r][0]), acc[r][b], 0, 0, 0);
            }
        }
    };

    // ---- the wave's chunks (at least one: waves <= chunks)
    issue(wave);
    // what the first of this thread's results needs at the end
    constexpr int UNITS = 4 * FB;                        // 16-byte units (four features) of a result row
    constexpr int SWZ = FB == 4 ? 0 : 1;
    constexpr int RESULTS = 16 * RT * UNITS;
    const int fin_m = m0 + tid / UNITS;
    const bool fin = tid < RESULTS && fin_m < M;
    EpilogueRaw raw = load_epilogue_raw_flat<BF16>(ep, fin ? fin_m : 0, band0 * 16 + 4 * (tid % UNITS), N);
    float2 turn_c = {1.0f, 1.0f}, turn_s = {0.0f, 0.0f};
    uint16_t* turn_to = nullptr;
    auto load_turn = [&](int m, int n0) __attribute__((always_inline)) {
        if constexpr (EPI == PACKED_ROPE) {
            const int table_row = guard.table_row(m);
            turn_c = guard.angles2(guard.cos, table_row, n0);
            turn_s = guard.angles2(guard.sin, table_row, n0);
            turn_to = guard.place(out, m, n0, N);
        }
    };
    if (fin) load_turn(fin_m, band0 * 16 + 4 * (tid % UNITS));
    u32x2 stream = {0u, 0u};
    if constexpr (EPI == PACKED_RESIDUAL) {
        const int n0 = band0 * 16 + 4 * (tid % UNITS);
        stream = *reinterpret_cast<const u32x2*>(guard.rows + static_cast<size_t>(fin ? fin_m : 0) * N + (n0 < N ? n0 : 0));
    }
    for (int chunk = wave;;) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        clear_past_end(chunk);
        multiply();
        __builtin_amdgcn_sched_barrier(0);
        chunk += waves;
        if (chunk >= chunks) break;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");               // the slot has been read
        issue(chunk);
    }

    // ---- partial sums in place of the wave's activations: unit q = 4 b + g of row 16 r + i
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int b = 0; b < FB; ++b)
            *reinterpret_cast<Acc*>(mine + ((16 * r + i) * UNITS + ((4 * b + g) ^ ((i >> SWZ) & (UNITS - 1)))) * 16) = acc[r][b];
    asm volatile("" : "+v"(raw.s), "+v"(raw.w[0]), "+v"(raw.w[1]), "+v"(raw.w[2]), "+v"(raw.w[3]));
    __syncthreads();
    if constexpr (EPI == PACKED_GATE) {
        for (int idx = tid; idx < RESULTS / 2; idx += waves * 64) {
            const int row = idx / (UNITS / 2), u = idx % (UNITS / 2), m = m0 + row, q = 8 * (u >> 2) + (u & 3);
            if (m >= M) break;
            const int swz = ((row & 15) >> SWZ) & (UNITS - 1);
            const uint8_t *from1 = smem + (row * UNITS + (q ^ swz)) * 16, *from3 = smem + (row * UNITS + ((q + 4) ^ swz)) * 16;
            Acc x1 = *reinterpret_cast<const Acc*>(from1), x3 = *reinterpret_cast<const Acc*>(from3);
            for (int v = 1; v < waves; ++v) {
                x1 += *reinterpret_cast<const Acc*>(from1 + v * S::kWaveBytes);
                x3 += *reinterpret_cast<const Acc*>(from3 + v * S::kWaveBytes);
            }
            EpilogueRegs e1, e3;
            e1.s = e3.s = bf16_bits_to_float(ep.s[m]);
            uint16_t o[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                e1.w[v] = bf16_bits_to_float(ep.ws[0]);
                e3.w[v] = bf16_bits_to_float(ep.ws[ep.ws_num - 1]);
                const float r = max_keep_nan(bf16_bits_to_float(apply_epilogue<int>(ep.kind, e1, v, x1[v] >> kI8WeightShift)), 0.0f);
                o[v] = float_to_bf16_bits(bf16_bits_to_float(float_to_bf16_bits(r * r)) *
                                          bf16_bits_to_float(apply_epilogue<int>(ep.kind, e3, v, x3[v] >> kI8WeightShift)));
            }
            *reinterpret_cast<u32x2*>(out + static_cast<size_t>(m) * (N >> 1) + band0 * 8 + 4 * u) =
                u32x2{o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16)};
        }
        return;
    }
    for (int idx = tid; idx < RESULTS; idx += waves * 64) {
        const int row = idx / UNITS, q = idx % UNITS, m = m0 + row, n0 = band0 * 16 + 4 * q;
        if (m >= M) break;
        const uint8_t* from = smem + (row * UNITS + (q ^ (((row & 15) >> SWZ) & (UNITS - 1)))) * 16;
        Acc sum = *reinterpret_cast<const Acc*>(from);
        for (int v = 1; v < waves; ++v) sum += *reinterpret_cast<const Acc*>(from + v * S::kWaveBytes);
        if (idx != tid) raw = load_epilogue_raw_flat<BF16>(ep, m, n0, N);
        const EpilogueRegs e = finish_epilogue(ep, raw);
        uint16_t o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if constexpr (BF16) o[v] = apply_epilogue<float>(EP_BF16, e, v, static_cast<AccScalar>(sum[v] * kBf16WeightUndo));
            else o[v] = apply_epilogue<int>(ep.kind, e, v, sum[v] >> kI8WeightShift);
        }
        if constexpr (EPI == PACKED_ROPE) {
            if (idx != tid) load_turn(m, n0);
            u32x2 turned = {o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16)};
            if (guard.part(n0) < 2) turned = u32x2{RopeStore::rotate(turned.x, turn_c.x, turn_s.x), RopeStore::rotate(turned.y, turn_c.y, turn_s.y)};
            if (turn_to != nullptr) *reinterpret_cast<u32x2*>(turn_to) = turned;
            continue;
        }
        u32x2 v = {o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16)};
        if constexpr (EPI == PACKED_RESIDUAL) {
            if (idx != tid) stream = *reinterpret_cast<const u32x2*>(guard.rows + static_cast<size_t>(m) * N + n0);
            v = ResidualRows::add(v, stream);
        }
        *reinterpret_cast<u32x2*>(out + static_cast<size_t>(m) * N + n0) = v;
    }
}

}  // namespace terna
