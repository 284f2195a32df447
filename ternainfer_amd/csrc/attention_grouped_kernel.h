// Decode attention of several sequences with the heads of a kv group in one workgroup: (sequence, KV HEAD, split).  The GQ = H / KV
// heads of a group read the same keys and values, so a cache line is requested once on the whole chip.
//
//   requests  keys and values go global -> LDS directly (16-byte pieces of the keys XOR-swizzled on the way), 4 KB at a time, each wave its
//             own: its keys, then its share of the values.  Two such units of a wave are under way while there are keys: eight waves'
//             64 KB are what a CU has outstanding at most, a further load holds up the wave that issues it.  Before the position is known a
//             wave requests one unit of keys, the rest is bounded by the prefix.  One wave rotates the group's queries and
//             one the new key, through LDS, for all.
//   pass 1    scores: v_mfma_f32_16x16x32_bf16 with 16 slots as rows and the group's heads as columns; MFMA number j takes the pieces j, j + R,
//             j + 2 R, j + 3 R (R = D / 32) of the rows, and the R partial scores are added pairwise
//   pass 2    softmax numerators [slot][head], all waves' slots together
//   pass 3    weighted sums of the value rows: a thread holds 8 dimensions of one row in SLICES, and v_mfma_f32_4x4x1_16b_f32 -- sixteen blocks
//             of four lanes, one product a block: exactly one fused multiply-add per sum -- weights a dimension of four lanes with
//             the four heads' numerators: 256 of them in 8 clocks, half of what they take as vector instructions
//
// Every head's arithmetic is that of the per-head kernel (attention_kernel.h) in the same order, so the results are the same bits.  RoPE and
// the cache write of the new token are folded in as there (split 0 writes the kv head's new rows).
//
// Bound: what one CU has outstanding against device memory (64 KB: 40 clocks for a 1 KB load, 16 from L2), in front of it 0.4 us and the first
// trip, behind it the third pass and the sums.  Measured, the launch alone in a graph, us, keys and values in registers with vector multiply-adds ->
// this: 32 sequences x 512 slots of different lengths filled to 60 % 10.6 -> 9.3, of one length 11.1 -> 9.8, 8 x 1528 to 90 % over six splits 10.5 -> 8.8,
// 16 x 512 over three 8.6 -> 7.1, 48 x 400 10.5 -> 9.1, 64 x 1000 21.6 -> 20.9; a decode step of 8 x 1528 1200 -> 1157, of 32 x 512 1500 -> 1461.
// The last batch of values apart from the others, its rows behind the prefix not weighed, the slices' sums read ahead, us before -> after (in registers):
// 6 sequences x 64 slots, D = 64, 8 heads on 4 6.0 -> 4.9 (4.7), 8 x 200 to 10 % 6.0 -> 5.4 (5.8); 32 x 512 9.0 -> 8.4 (9.5), 64 x 2048 to 95 % 54.5 -> 51.5 (50.9).
// Tried: four units of a wave under way, from the start or once the keys are in (level to 7 % slower).
#pragma once

#include "attention_kernel.h"

namespace terna {

template <int D, int NW, int GQ>
struct GroupedShape {
    static constexpr int kRow = 2 * D;                       // bytes of a cache row
    static constexpr int kUnit = 4096, kLoads = 4;           // bytes and direct loads of a unit
    static constexpr int kKeyRows = kUnit / kRow;            // slots of a unit of keys; one of values is four rows per thread
    static constexpr int kFixed = (GQ + 2) * kRow + 2 * NW * GQ * 4;          // the group's queries, the new rows, the waves' maxima and sums
    static constexpr int score_bytes(int S) { return ((S + 15) & ~15) * GQ * 4; }
    static constexpr int kWave = 2 * kUnit;                  // two buffers; in the end a wave's sums, [slice][head][D]
    static constexpr int bytes(int S) { return NW * kWave + kFixed + score_bytes(S); }
    static_assert(64 / (D / 8) * GQ * D * 4 <= kWave, "sums");
};

// The first sixteen dwords of arguments arrive with the wave: what a workgroup needs ahead of its first request.  shape: KV | splits << 16 |
// per_seq << 24 | prefetching workgroups behind the others << 25; inv_kv, inv_splits: 2^32 over them, rounded up -- the upper half
// of a product with it is the quotient, for numbers whose product with the divisor is below 2^32.
// WHOLE: one split, and the output rows themselves instead of partial results.  ROPE = false: `q` is rotated queries [B][H][D], and the
// caches hold the new token already (WHOLE only).
template <int D, bool ROPE, bool ADJACENT, int NW, int GQ, bool WHOLE>
__global__ __launch_bounds__(64 * NW) void terna_decode_attention_grouped_kernel(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ cache_k, uint16_t* __restrict__ cache_v, const long long* __restrict__ pos,
    uint32_t shape, int S, uint32_t inv_kv, uint32_t inv_splits, const float* __restrict__ cosv_all, const float* __restrict__ sinv_all, float scale,
    int slots, float* __restrict__ partial, uint16_t* __restrict__ out, AttentionPrefetch pf)
{
    static_assert(D == 64 || D == 128, "head dimension");
    static_assert(ROPE || (WHOLE && !ADJACENT), "the split launch rotates and writes the new token itself");
    static_assert(GQ == 2 || GQ == 4, "the heads of a group are rows of a 4 x 4 block");
    using Shape = GroupedShape<D, NW, GQ>;
    constexpr int NT = 64 * NW;
    constexpr int ROW = Shape::kRow, PIECES = D / 8;         // 16-byte pieces of a row
    constexpr int RPL = 64 / PIECES;                         // rows of a direct load, and slices of a wave
    constexpr int LOADS = Shape::kLoads, KROWS = Shape::kKeyRows;
    constexpr int STEP = NW * RPL;                           // slots of one value row per thread: SLICES
    constexpr int R = D / 32;
    constexpr int GROUP = 8;                                 // slices added up before the groups of them are
    static_assert(GQ * PIECES <= 64, "a wave rotates the group's queries");
    extern __shared__ __align__(16) uint8_t smem[];
    if (shape >> 25) {                                       // prefetch-only workgroups
        asm volatile("s_nop 0");                             // (an argument that is not there yet is read in here only)
        if (static_cast<int>(blockIdx.x) >= slots) {
            attention_prefetch_role(pf, slots, NT);
            return;
        }
    }
    const int KV = shape & 0xffff, SP = WHOLE ? 1 : (shape >> 16) & 0xff;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto quotient = [](uint32_t v, uint32_t inv, int by) { return by == 1 ? static_cast<int>(v) : static_cast<int>(__umulhi(v, inv)); };
    const int grp_id = WHOLE ? blockIdx.x : quotient(blockIdx.x, inv_splits, SP);          // (sequence, kv head)
    const int sp = WHOLE ? 0 : blockIdx.x - grp_id * SP;
    const int b = quotient(grp_id, inv_kv, KV), kvh = grp_id - b * KV;
    const int H = KV * GQ;
    auto cache_slot = [&](int l) { return (((l >> 4) * SP + sp) << 4) + (l & 15); };
    const int pb = (shape >> 24) & 1 ? b : 0;
    const long long p0 = pos[pb];
    uint16_t* const krows = cache_k + (static_cast<size_t>(b) * KV + kvh) * S * D;
    uint16_t* const vrows = cache_v + (static_cast<size_t>(b) * KV + kvh) * S * D;
    const int c = lane & 15, g = lane >> 4;                  // column and row group of a matrix product
    const int lrow = lane / PIECES, piece = lane % PIECES;   // row of a direct load, its 16 bytes

    uint8_t* const mine = smem + wave * Shape::kWave;
    const uint32_t lds_mine = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(mine));
    uint8_t* const qrows = smem + NW * Shape::kWave;             // queries [GQ][D], new key, new value
    float* const red_m = reinterpret_cast<float*>(qrows + (GQ + 2) * ROW);     // [NW][GQ]
    float* const red_s = red_m + NW * GQ;
    float* const score = red_s + NW * GQ;                    // [slot][GQ]

    // A wave's units in order: `keys` of keys -- unit l of the workgroup is wave l mod NW's --, then those of values.  Rows past the prefix: its
    // last one, with a weight of zero.
    auto key_swizzle = [](int row) { return D == 128 ? row & 15 : (row >> 1) & 7; };
    auto buffer_of = [&](int unit) { return (unit & 1) * Shape::kUnit; };
    auto load_keys = [&](int unit, int last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int row = RPL * i + lrow;
            lds_dma_b128(krows, min(cache_slot((wave + NW * unit) * KROWS + row), last) * ROW + ((piece ^ key_swizzle(row)) << 4), lds_mine + buffer_of(unit) + i * 1024);
        }
    };
    auto load_values = [&](int unit, int k, int last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            lds_dma_b128(vrows, min(cache_slot((k * LOADS + i) * STEP + wave * RPL + lrow), last) * ROW + (piece << 4), lds_mine + buffer_of(unit) + i * 1024);
    };
    auto prefix = [&] {
        long long p = p0;
        asm volatile("" : "+s"(p));                          // looked at here, not ahead of the first requests
        return __builtin_amdgcn_readfirstlane(p < 0 ? 1 : (p >= S ? S : static_cast<int>(p) + 1));
    };
    auto tiles_of = [&](int n) {                             // of 16 slots, of this workgroup; local tile l is tile l SP + sp
        const int tiles = (n + 15) >> 4;
        return tiles > sp ? quotient(tiles - sp + SP - 1, inv_splits, SP) : 0;
    };
    auto keys_of = [&](int ltiles) { return max(1, ((16 * ltiles + KROWS - 1) / KROWS - wave + NW - 1) / NW); };      // (a wave without keys: what it requests ahead)
    auto values_of = [&](int ltiles) { return (16 * ltiles + LOADS * STEP - 1) / (LOADS * STEP); };
    auto request = [&](int unit, int keys, int last) __attribute__((always_inline)) {
        if (unit < keys) load_keys(unit, last);
        else load_values(unit, unit - keys, last);
    };
    // the first two units (the second where there is one)
    auto request_first = [&]() __attribute__((always_inline)) {
        load_keys(0, S - 1);
        const int n = prefix(), ltiles = tiles_of(n), keys = keys_of(ltiles);
        const bool second = keys + values_of(ltiles) > 1;
        if (second) request(1, keys, n - 1);
        return second;
    };
    // waits for everything but the unit requested last
    auto await_all_but = [](bool one) __attribute__((always_inline)) {
        if (one) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    if (wave < 2) {
        // the new token: wave 0 the group's query heads, wave 1 its key row and (not rotated) its value row
        constexpr int TABLES = ADJACENT ? 1 : 2;             // 16-byte pieces of cosines and of sines
        const int head_of = lane / PIECES;
        u32x4 own, other, cs[TABLES], sn[TABLES];
        if constexpr (!ROPE) {
            global_load_b128_nowait(own, q + (static_cast<size_t>(b) * H + kvh * GQ) * D, (head_of < GQ ? head_of : 0) * ROW + piece * 16);
        } else {
            const uint16_t* row = q + static_cast<size_t>(b) * (H + 2 * KV) * D;
            const int head = wave == 0 ? kvh * GQ + (head_of < GQ ? head_of : 0) : H + kvh + (head_of == 1 ? KV : 0);
            const float *cosv = cosv_all + pb * (D / 2), *sinv = sinv_all + pb * (D / 2);
            global_load_b128_nowait(own, row, head * ROW + piece * 16);
            if constexpr (!ADJACENT) global_load_b128_nowait(other, row, head * ROW + ((piece + PIECES / 2) % PIECES) * 16);
#pragma unroll
            for (int t = 0; t < TABLES; ++t) {
                const uint32_t at = (ADJACENT ? piece : 2 * (piece % (PIECES / 2)) + t) * 16;
                global_load_b128_nowait(cs[t], cosv, at);
                global_load_b128_nowait(sn[t], sinv, at);
            }
        }
        if (request_first()) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        landed(own);
        if constexpr (ROPE) {
            if constexpr (!ADJACENT) landed(other);
#pragma unroll
            for (int t = 0; t < TABLES; ++t) {
                landed(cs[t]);
                landed(sn[t]);
            }
            float a[8], o[8];
            unpack_bf16x8(own, a);
            if constexpr (ADJACENT) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
#pragma clang fp contract(off)
                    const float cc = __uint_as_float(cs[0][m]), sv = __uint_as_float(sn[0][m]);
                    o[2 * m] = a[2 * m] * cc - a[2 * m + 1] * sv;
                    o[2 * m + 1] = a[2 * m + 1] * cc + a[2 * m] * sv;
                }
            } else {
                float p[8];
                unpack_bf16x8(other, p);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
                    const float cc = __uint_as_float(cs[e >> 2][e & 3]), sv = __uint_as_float(sn[e >> 2][e & 3]);
                    const float lo = a[e] * cc - p[e] * sv;
                    const float hi = a[e] * cc + p[e] * sv;
                    o[e] = piece < PIECES / 2 ? lo : hi;
                }
            }
            const bool value = wave == 1 && head_of == 1;
            const u32x4 turned = pack_bf16x8(o);
            own = value ? own : turned;
            if (wave == 1 && head_of < 2) {
                *reinterpret_cast<u32x4*>(qrows + (GQ + head_of) * ROW + piece * 16) = own;
                if (sp == 0 && p0 >= 0 && p0 < S) *reinterpret_cast<u32x4*>((value ? vrows : krows) + static_cast<size_t>(p0) * D + 8 * piece) = own;
            }
        }
        if (wave == 0 && head_of < GQ) *reinterpret_cast<u32x4*>(qrows + head_of * ROW + piece * 16) = own;
    } else {
        request_first();
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int n = prefix(), ltiles = tiles_of(n);
    const int nl = 16 * ltiles, keys = keys_of(ltiles), batches = values_of(ltiles), units = keys + batches;

    // ---- pass 1
    bf16x8 bq[R];
#pragma unroll
    for (int j = 0; j < R; ++j) bq[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qrows + (c % GQ) * ROW + 16 * (j + R * g)));
    float mx = -INFINITY;                                    // of the column's head
    for (int unit = 0; unit < keys; ++unit) {
        await_all_but(unit + 1 < units);
        uint8_t* const rows = mine + buffer_of(unit);
#pragma unroll
        for (int t = 0; t < KROWS / 16; ++t) {
            const int ltile = (wave + NW * unit) * (KROWS / 16) + t;
            if (ltile >= ltiles) break;                      // uniform
            uint8_t* const tile = rows + t * 16 * ROW;
            const int from = 16 * (ltile * SP + sp);
            const bool last = from + 16 >= n;                // uniform: the tile of the new token, and the only one with slots past it
            if (ROPE && last && lane < PIECES) {             // its key row is in LDS
                const int row = n - 1 - from;
                *reinterpret_cast<u32x4*>(tile + row * ROW + ((piece ^ key_swizzle(row)) << 4)) = *reinterpret_cast<const u32x4*>(qrows + GQ * ROW + piece * 16);
            }
            f32x4 of[R];
#pragma unroll
            for (int j = 0; j < R; ++j)
                of[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(tile + c * ROW + (((j + R * g) ^ key_swizzle(c)) << 4))), bq[j], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {                    // slot 4 g + v of the tile
                const float x = R == 4 ? (of[0][v] + of[1][v]) + (of[R - 2][v] + of[R - 1][v]) : of[0][v] + of[1][v];
                const float d = x * scale;
                if (!last || from + 4 * g + v < n) {
                    if (c < GQ) score[(16 * ltile + 4 * g + v) * GQ + c] = d;
                    mx = fmaxf(mx, d);
                }
            }
        }
        if (unit + 2 < units) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // the unit's buffer has been read
            request(unit + 2, keys, n - 1);
        }
    }
    mx = cross_row_reduce<true>(mx);
    if (g == 0 && c < GQ) red_m[wave * GQ + c] = mx;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- pass 2: softmax numerators and their sums
    typedef float Heads __attribute__((ext_vector_type(GQ)));
    Heads mxh = *reinterpret_cast<const Heads*>(red_m), sum = 0.0f;
#pragma unroll
    for (int w = 1; w < NW; ++w) {
        const Heads other = *reinterpret_cast<const Heads*>(red_m + w * GQ);
#pragma unroll
        for (int h = 0; h < GQ; ++h) mxh[h] = fmaxf(mxh[h], other[h]);
    }
    for (int l = tid; l < nl; l += NT) {
        Heads* const at = reinterpret_cast<Heads*>(score + l * GQ);
        const Heads d = *at;
        const bool ok = cache_slot(l) < n;
        Heads p;
#pragma unroll
        for (int h = 0; h < GQ; ++h) {
            p[h] = ok ? __expf(d[h] - mxh[h]) : 0.0f;
            sum[h] += p[h];
        }
        *at = p;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int h = 0; h < GQ; ++h) {                           // (needed at the end)
        sum[h] = wave_sum(sum[h]);
        if (lane == 0) red_s[wave * GQ + h] = sum[h];
    }

    // ---- pass 3: value rows of slice wave RPL + lrow, dimensions 8 piece .. +7, times the heads' numerators (lane i of a block of four: head i's)
    f32x4 acc[8];                                            // [dimension][head]
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto weigh = [&](float p, const u32x4& row) __attribute__((always_inline)) {
        float v[8];
        unpack_bf16x8(row, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, v[e], acc[e], 0, 0, 0);
    };
    const int lslot = wave * RPL + lrow;
    float p[LOADS];
    u32x4 row[LOADS];
    auto read_batch = [&](int k, int most) __attribute__((always_inline)) {                // (numerators past local slot `most`: slot 0's)
        const uint8_t* const from = mine + buffer_of(keys + k) + lane * 16;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int l = (k * LOADS + i) * STEP + lslot;
            row[i] = *reinterpret_cast<const u32x4*>(from + i * 1024);
            p[i] = score[(l >= most ? 0 : l) * GQ + (lane & (GQ - 1))];
        }
    };
    int k = 0;
    for (; k + 1 < batches; ++k) {                           // every row stands in front of the last tile
        await_all_but(true);
        read_batch(k, 1 << 30);
        if (k + 2 < batches) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            load_values(keys + k + 2, k + 2, n - 1);
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) weigh(p[i], row[i]);
    }
    if (k < batches) {
        await_all_but(false);
        read_batch(k, nl);
        // slots past the prefix hold anything, also what times 0 is no number; the new token's value row is in LDS
        const u32x4 vnew = *reinterpret_cast<const u32x4*>(qrows + (GQ + 1) * ROW + piece * 16);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            // (uniform; weighing rows that are not there, with zeros, made launches of 20 - 60 slots 0.3 - 0.4 us longer)
            if ((k * LOADS + i) * STEP >= nl) break;
            const int l = (k * LOADS + i) * STEP + lslot, s = cache_slot(l);
            const bool ok = l < nl && s < n;
            if (ROPE) row[i] = s == n - 1 ? vnew : row[i];
            row[i] = ok ? row[i] : u32x4{0u, 0u, 0u, 0u};
            weigh(ok ? p[i] : 0.0f, row[i]);
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");            // (a wave without keys: what it requested ahead)

    // ---- sums of the slices, eight at a time, then of those
    auto sum_at = [](int dim4) { return D == 128 ? dim4 ^ ((dim4 >> 4) & 1) : dim4; };    // of four dimensions: the writes of 16 lanes cover all banks
#pragma unroll
    for (int h = 0; h < GQ; ++h)
#pragma unroll
        for (int e = 0; e < 8; e += 4)
            *reinterpret_cast<f32x4*>(mine + ((lrow * GQ + h) * D + 4 * sum_at(2 * piece + (e >> 2))) * 4) = f32x4{acc[e][h], acc[e + 1][h], acc[e + 2][h], acc[e + 3][h]};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const size_t heads_total = static_cast<size_t>(slots / SP) * GQ;      // B * H
    for (int idx = tid; idx < GQ * D; idx += NT) {
        const int h = idx / D, d = idx - h * D;
        const uint8_t* const from = smem + (h * D + 4 * sum_at(d >> 2) + (d & 3)) * 4;
        // (all read ahead of the first addition: a pair at a time as they were added, the launch was 0.1 us longer, 0.2 with the 64 slices of D = 64)
        float of[STEP], o = 0.0f;
#pragma unroll
        for (int slice = 0; slice < STEP; ++slice) of[slice] = *reinterpret_cast<const float*>(from + (slice / RPL) * Shape::kWave + (slice % RPL) * GQ * D * 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int grp = 0; grp < STEP / GROUP; ++grp) {
            float part = 0.0f;
#pragma unroll
            for (int i = 0; i < GROUP; ++i) part += of[grp * GROUP + i];
            o += part;
        }
        float all = red_s[h];
#pragma unroll
        for (int w = 1; w < NW; ++w) all += red_s[w * GQ + h];
        const size_t bh = static_cast<size_t>(b) * H + kvh * GQ + h;
        if constexpr (WHOLE) {
            out[bh * D + d] = float_to_bf16_bits(o / all);
        } else {
            partial[attention_stat_floats(heads_total) + (bh * SP + sp) * D + d] = o;
            if (d == 0) {
                float m = red_m[h];
#pragma unroll
                for (int w = 1; w < NW; ++w) m = fmaxf(m, red_m[w * GQ + h]);
                float* const stat = partial + bh * kAttentionStatFloats;
                stat[sp] = m;
                stat[kAttentionMaxSplits + sp] = all;
            }
        }
    }
}

}  // namespace terna
