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
//     behind the only barrier, are added in wave order (bit-reproducible; integer sums exact) and leave as whole rows; every thread finishes
//     one to four features at a time, all waves' sums of them read at once.  In one to two threads per wave and one sum after the other that
//     was 2000 - 3500 of a workgroup's 6000 - 12000 clocks, now 850 - 1700: decode step of 32 sequences x 512 slots 1461 -> 1355 us, prompt of
//     100 tokens 1580 -> 1541.
// Every load of the main part is issued and awaited by hand (see prefill_packed_kernel.h).
// Measured, us per launch, weights rotating over 8 copies, the ring / MFMA-tiled kernel that such calls had before -> this kernel (tile choice
// and what is left to the MFMA-tiled one, "-": launch_mid.hip):
//                              QKV 2560->3840   O 2560->2560   gate+up 2560->13824   down 6912->2560
//   bf16 M = 37                6.9 -> 4.8       6.8 -> 3.9     16.5 -> 9.0            13.3 -> 6.2
//   bf16 M = 100               12.1 -> 6.2      11.5 -> 5.8    -                      15.3 -> 11.0
//   int8 M = 37                5.5 -> 3.8       5.4 -> 3.3     11.4 -> 6.3            9.4 -> 4.6
//   int8 M = 100               7.7 -> 4.6       7.5 -> 4.4     -                      12.9 -> 7.2
//   int8 M = 300               -                11.1 -> 5.7    -                      16.3 -> 11.1
#pragma once

#include "chain_chunk_kernel.h"
#include "prefill_packed_kernel.h"

namespace terna {

constexpr int kMidMaxWaves = 16;

// f(std::integral_constant<int, n>{}) for n = 1 .. MOST: a uniform branch to code that knows the number.
template <int MOST, typename Function>
__device__ __forceinline__ void with_constant(int n, Function&& f)
{
    static_assert(MOST >= 1 && MOST <= 16, "cases below");
    switch (n) {
#define TERNA_CASE(V) \
    case V: \
        if constexpr (V <= MOST) f(std::integral_constant<int, V>{}); \
        break
        TERNA_CASE(1); TERNA_CASE(2); TERNA_CASE(3); TERNA_CASE(4); TERNA_CASE(5); TERNA_CASE(6); TERNA_CASE(7); TERNA_CASE(8);
        TERNA_CASE(9); TERNA_CASE(10); TERNA_CASE(11); TERNA_CASE(12); TERNA_CASE(13); TERNA_CASE(14); TERNA_CASE(15); TERNA_CASE(16);
#undef TERNA_CASE
    default: __builtin_unreachable();
    }
}

template <typename Act, int RT, int FB>
struct MidShape {
    static constexpr int kRowBytes = 256 * static_cast<int>(sizeof(Act));    // a chunk's piece of one activation row
    static constexpr int kWaveBytes = 16 * RT * kRowBytes;                     // a wave's LDS: activations, then partial sums
    static_assert(FB == 2 || FB == 4, "result rows of 8 or 16 units: see the swizzle of the partial sums");
    static_assert(RT * FB * 1024 <= kWaveBytes, "partial sums (1 KB per 16 x 16 tile) take the place of the activations");
};
// A wave's LDS where the rows are quantised inside (a chunk of 16 int8 rows), and what follows all waves': every wave's row maxima, its
// copy of the multipliers, the scales.
struct MidQuantShape {
    static constexpr int kWaveBytes = 16 * kChainSlabPitch;
    static constexpr int bytes(int waves) { return waves * kWaveBytes + (16 + 16) * kMidMaxWaves * 4 + 16 * 4; }
};

// QUANT (RT = 1, Act = int8_t, a wave for every chunk): x is bf16 and quantised inside -- quant_input and the linear of a module call in
// one launch, for the host's sake: a call of two launches takes it 10.6 us, one 6.9.  A wave holds its chunk of 16 rows in registers; their
// maxima meet in LDS, every wave forms the 16 scales for itself and writes int8 rows where the other form has them by direct loads.  Two
// chunks a wave (K = 6912) were 10 us of the device, where the two launches are 7.
// EPI: plain outputs, the sum with the stream, the feed-forward gate or the rotary embedding and cache write (see the epilogues of prefill_packed_kernel.h)
template <typename Act, int RT, int FB, bool GUARD, int EPI = PACKED_STORE, bool QUANT = false>
__global__ __launch_bounds__(kMidMaxWaves * 64) void terna_mid_kernel(
    const Act* __restrict__ x, const uint32_t* __restrict__ packed, uint16_t* __restrict__ out,
    int M, int N, int K, int row_tiles, int waves, Epilogue ep, PackedExtra<EPI> guard, int quant_mode)
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
    static_assert(!QUANT || (RT == 1 && !BF16 && EPI == PACKED_STORE && FB * 1024 <= MidQuantShape::kWaveBytes), "see above");
    constexpr int WAVE_BYTES = QUANT ? MidQuantShape::kWaveBytes : S::kWaveBytes;
    constexpr int MOST_WAVES = 160 * 1024 / WAVE_BYTES < kMidMaxWaves ? 160 * 1024 / WAVE_BYTES : kMidMaxWaves;
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
    uint8_t* mine = smem + wave * WAVE_BYTES;
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
    u32x4 xr[8];                                         // QUANT: rows 2 q + (lane >> 5), columns 8 (lane & 31) .. +7
    const int l32 = lane & 31, odd = lane >> 5;
    if constexpr (QUANT) {
        // what is in the caches first: requested behind the weights it would arrive with them
        const __amdgpu_buffer_rsrc_t rx = make_raw_buffer(x, static_cast<uint32_t>(M) * K * 2u);
        const int col = wave * 256 + 8 * l32;
        int at = ((m0 + odd) * K + col) * 2;                             // (a row past M is past the buffer)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            xr[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, col < K ? at : kBufferOutOfRange, 0, 0));
            at += 4 * K;
        }
        __builtin_amdgcn_s_barrier();
        const __amdgpu_buffer_rsrc_t rb = make_raw_buffer(packed, static_cast<uint32_t>(N >> 4) * static_cast<uint32_t>(ktiles) * 256u);
#pragma unroll
        for (int b = 0; b < FB; ++b)
            rw.w[b] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                rb, wave * 4 + g < ktiles ? ((band0 + b) * ktiles + wave * 4) * 256 + lane * 16 : kBufferOutOfRange, 0, 0));
    } else {
        issue(wave);
    }
    // ---- a thread's results: 2^f neighbouring features of one row, as few as give every thread of the workgroup some (four are a unit of sums)
    constexpr bool GATE = EPI == PACKED_GATE;
    constexpr int X = GATE ? 2 : 1;
    constexpr int UNITS = 4 * FB;                        // 16-byte units (four features) of a row of sums
    constexpr int OUT_UNITS = UNITS / X;                 // ... of a row of results
    constexpr int RESULTS = 16 * RT * OUT_UNITS * 4;
    constexpr auto log_features = [](int of_waves) {
        const int few = EPI == PACKED_ROPE ? 2 : 1, f = RESULTS / (64 * (of_waves >= 8 ? 8 : of_waves >= 4 ? 4 : 1)), n = f < few ? few : f;
        return n >= 4 ? 2 : n == 2 ? 1 : 0;
    };
    constexpr int MANY = 1 << log_features(8);           // of eight waves or more
    // (One wave of K <= 256 with a feature a thread went eight times through its results, each time waiting for their scales: 17 x 704 x 192 4.6 us int8,
    // 4.1 bf16; four features a thread 3.6, 3.0.)
    // What they need at the end, the first of them requested here.  Values on the way must not be moved, not even to where two branches meet: that
    // waits for every load before them (two ways of requesting them, by the number of waves, cost every launch 0.3 us).  So there is
    // one way, and the scales that only threads with more features have are in branches that nothing else ends in.
    struct Finish {
        uint32_t s, w[4];
        u32x2 stream;                                    // the unit of four
        float2 turn_c, turn_s;                           // "
        uint16_t* to;
    };
    const int out_n0 = band0 * (GATE ? 8 : 16);
    auto request_finish = [&](int idx, auto log_f) __attribute__((always_inline)) {
        Finish f;
        constexpr int LOG_ROW = __builtin_ctz(OUT_UNITS * 4);
        const int shift = LOG_ROW - log_f, row = idx >> shift, m = m0 + row < M ? m0 + row : M - 1;
        const int n0 = out_n0 + ((idx & ((1 << shift) - 1)) << log_f);
        if constexpr (!BF16 && !QUANT) f.s = ep.s[m];
        if constexpr (GATE) {
            f.w[0] = ep.ws[0];
            f.w[1] = ep.ws[ep.ws_num - 1];
        } else {
            int group[4] = {0, 0, 0, 0};
            if (ep.ws_num != 1) {
                ws_group_decode4(n0, N, ep.ws_num, group);
                if (ep.kind == EP_I8_PREFILL) group[0] = group[1] = group[2] = group[3] = ws_group_prefill(n0, N, ep.ws_num);
            }
            auto scale_of = [&](int v) -> uint32_t { return BF16 ? __float_as_uint(ep.scale[group[v]]) : ep.ws[group[v]]; };
#pragma unroll
            for (int v = 0; v < MANY; ++v) f.w[v] = scale_of(v);
#pragma unroll
            for (int v = MANY; v < 4; ++v)
                if (v < 1 << log_f) f.w[v] = scale_of(v);                // uniform
        }
        if constexpr (EPI == PACKED_RESIDUAL) f.stream = *reinterpret_cast<const u32x2*>(guard.rows + static_cast<size_t>(m) * N + (n0 & ~3));
        if constexpr (EPI == PACKED_ROPE) {
            const int at = guard.table_row(m);
            f.turn_c = guard.angles2(guard.cos, at, n0 & ~3);
            f.turn_s = guard.angles2(guard.sin, at, n0 & ~3);
            f.to = guard.place(out, m, n0, N);
        }
        return f;
    };
    const int log_first = waves >= 8 ? log_features(8) : waves >= 4 ? log_features(4) : log_features(1);
    Finish first = request_finish(tid < (RESULTS >> log_first) ? tid : 0, log_first);
    float* const maxima = reinterpret_cast<float*>(smem + waves * WAVE_BYTES);          // [row][wave]
    float* const multiplier = maxima + 16 * kMidMaxWaves + 16 * wave;                    // of row r: at 8 (r & 1) + r / 2
    float* const scale = maxima + 32 * kMidMaxWaves;
    if constexpr (QUANT) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            float most = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                most = max_keep_nan(max_keep_nan(most, fabsf(__uint_as_float(xr[q][j] << 16))), fabsf(__uint_as_float(xr[q][j] & 0xffff0000u)));
            most = group_amax<32>(most);
            if (l32 == 0) maxima[(2 * q + odd) * kMidMaxWaves + wave] = most;
        }
        __syncthreads();
        {
            const int row = lane >> 2;
            float most = 0.0f;
            for (int w = lane & 3; w < waves; w += 4) most = max_keep_nan(most, maxima[row * kMidMaxWaves + w]);
            most = group_amax<4>(most);
            uint16_t bits;
            const float mul = quant_scale(most, quant_mode, &bits);
            if ((lane & 3) == 0) {
                multiplier[8 * (row & 1) + (row >> 1)] = mul;
                if (wave == 0) scale[row] = bf16_bits_to_float(bits);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const f32x4 mul_lo = *reinterpret_cast<const f32x4*>(multiplier + 8 * odd), mul_hi = *reinterpret_cast<const f32x4*>(multiplier + 8 * odd + 4);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            landed(xr[q]);                                               // (unpacked again, not kept unpacked: twice the registers)
            const uint32_t pairs[4] = {xr[q].x, xr[q].y, xr[q].z, xr[q].w}, none[4] = {};
            uint32_t d[2];
            chain_quantise<8, false>(pairs, none, 0.0f, q < 4 ? mul_lo[q & 3] : mul_hi[q & 3], quant_mode, d);
            *reinterpret_cast<u32x2*>(mine + (2 * q + odd) * kChainSlabPitch + 8 * l32) = u32x2{d[0], d[1]};
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const i32x4 v = *reinterpret_cast<const i32x4*>(mine + i * kChainSlabPitch + 64 * g + 16 * c);
#pragma unroll
            for (int b = 0; b < FB; ++b) acc[0][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(expand_word_i8(rw.w[b][c]), v, acc[0][b], 0, 0, 0);
        }
    }
    for (int chunk = wave; !QUANT;) {
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
    constexpr int SWZ = FB == 4 ? 0 : 1;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int b = 0; b < FB; ++b)
            *reinterpret_cast<Acc*>(mine + ((16 * r + i) * UNITS + ((4 * b + g) ^ ((i >> SWZ) & (UNITS - 1)))) * 16) = acc[r][b];
    asm volatile("" : "+v"(first.w[0]));
    if constexpr (!BF16 && !QUANT) asm volatile("" : "+v"(first.s));
    if constexpr (EPI == PACKED_RESIDUAL) asm volatile("" : "+v"(first.stream));
    __syncthreads();
    // All waves' sums of a result are read before the first is added (one after the other they took 2000 - 3500 of a launch's 6000 - 12000
    // clocks), by code of its own for every number of waves.  Read as up to eight or sixteen, the ones that are not there cost, us a launch, int8; bf16:
    // 32 rows of N = 2560 K = 4096 3.9 (sixteen by number) / 4.3; 300 rows of N = 704 K = 320 (two) 3.5 / 3.9; 4.0 / 4.6.
    with_constant<MOST_WAVES>(waves, [&](auto count) __attribute__((always_inline)) {
        constexpr int W = decltype(count)::value, LOG_F = log_features(W), F = 1 << LOG_F, PER_ROW = OUT_UNITS * 4 / F;
        typedef AccScalar Sums __attribute__((ext_vector_type(F)));
        for (int idx = tid; idx < RESULTS / F; idx += W * 64) {
            const int row = idx / PER_ROW, n = F * (idx % PER_ROW), m = m0 + row, u = n >> 2, sub = n & 3;
            if (m >= M) break;
            const int q = GATE ? 8 * (u >> 2) + (u & 3) : u;
            Sums part[X][W], sum[X];
#pragma unroll
            for (int x = 0; x < X; ++x) {
                const uint8_t* from = smem + (row * UNITS + ((q + 4 * x) ^ (((row & 15) >> SWZ) & (UNITS - 1)))) * 16 + sub * 4;
#pragma unroll
                for (int v = 0; v < W; ++v) part[x][v] = *reinterpret_cast<const Sums*>(from + v * WAVE_BYTES);
            }
            const Finish f = idx == tid ? first : request_finish(idx, std::integral_constant<int, LOG_F>{});
#pragma unroll
            for (int x = 0; x < X; ++x) {
                sum[x] = part[x][0];
#pragma unroll
                for (int v = 1; v < W; ++v) sum[x] += part[x][v];
            }
            // sums -> outputs rounded to bf16, as apply_epilogue has them; under the prefill rule F features of a 128-column tile share a scale
            const float s = BF16 ? 1.0f : QUANT ? scale[row] : __uint_as_float(f.s << 16);
            float r[X][F];
#pragma unroll
            for (int x = 0; x < X; ++x)
#pragma unroll
                for (int v = 0; v < F; ++v) {
                    if constexpr (BF16) r[x][v] = sum[x][v] * kBf16WeightUndo;
                    else r[x][v] = static_cast<float>(sum[x][v] >> kI8WeightShift);
                }
            auto weight = [&](int x, int v) { return __uint_as_float(BF16 ? f.w[v] : f.w[GATE ? x : v] << 16); };
            if constexpr (BF16) {
#pragma unroll
                for (int v = 0; v < F; ++v) r[0][v] *= weight(0, v);
            } else if (ep.kind == EP_I8_DECODE) {
                const RowQuotient by(s);
#pragma unroll
                for (int x = 0; x < X; ++x) {
                    by.of(r[x]);
#pragma unroll
                    for (int v = 0; v < F; ++v) r[x][v] = __fmul_rn(r[x][v], weight(x, v));
                }
            } else {
#pragma unroll
                for (int x = 0; x < X; ++x) {
                    const float coeff = s != 0.0f ? __fdiv_rn(weight(x, 0), s) : 0.0f;
#pragma unroll
                    for (int v = 0; v < F; ++v) r[x][v] = __fmul_rn(r[x][v], coeff);
                }
            }
            uint16_t o[F];
#pragma unroll
            for (int v = 0; v < F; ++v) {
                o[v] = float_to_bf16_bits(r[0][v]);
                if constexpr (GATE) {
                    const float x1 = max_keep_nan(bf16_bits_to_float(o[v]), 0.0f);
                    o[v] = float_to_bf16_bits(bf16_bits_to_float(float_to_bf16_bits(x1 * x1)) * bf16_bits_to_float(float_to_bf16_bits(r[GATE][v])));
                }
            }
            uint32_t pair[(F + 1) / 2];
#pragma unroll
            for (int v = 0; v < (F + 1) / 2; ++v) {
                pair[v] = F == 1 ? o[0] : o[2 * v] | (static_cast<uint32_t>(o[F == 1 ? 0 : 2 * v + 1]) << 16);
                // (of a unit's two pairs, or of a pair's two features, this thread's first)
                if constexpr (EPI == PACKED_RESIDUAL) {
                    const uint32_t word = F == 4 ? f.stream[v] : sub < 2 ? f.stream[0] : f.stream[1];
                    pair[v] = ResidualRows::pair(pair[v], F == 1 && (sub & 1) ? word >> 16 : word);
                }
                if constexpr (EPI == PACKED_ROPE) {
                    const bool second = F == 4 ? v == 1 : sub >= 2;
                    if (guard.part(out_n0 + n) < 2) pair[v] = RopeStore::rotate(pair[v], second ? f.turn_c.y : f.turn_c.x, second ? f.turn_s.y : f.turn_s.x);
                }
            }
            uint16_t* to = EPI == PACKED_ROPE ? f.to : out + static_cast<size_t>(m) * (GATE ? N >> 1 : N) + out_n0 + n;
            if (EPI == PACKED_ROPE && to == nullptr) continue;
            if constexpr (F == 1) *to = static_cast<uint16_t>(pair[0]);
            else if constexpr (F == 2) *reinterpret_cast<uint32_t*>(to) = pair[0];
            else *reinterpret_cast<u32x2*>(to) = u32x2{pair[0], pair[1]};
        }
    });
}

}  // namespace terna
