// Multi-token attention of four query heads per kv head, 128 dimensions: what terna_prefill_attention_group_kernel does, bit for bit
// (a step = 32 slots, the same two products, the same order of every sum), at less than its time.
//
// What bounded that kernel: the chain of one wave.  A step was scores -> maximum -> exponentials -> outputs one after the other, each
// waiting for the last and for LDS: about 2500 clocks for 384 of matrix work, and a causal triangle's longest query block (60 steps
// at 1920 tokens) is what a launch waits for.  Here a step works on three of them at once, none of which waits for another: the values
// of step i times its probabilities, the probabilities of step i + 1, the scores of step i + 2.  They are woven in slices of two
// matrix instructions, about ten vector ones, one or two operand reads and a tile load (the order is held by scheduling
// barriers: left to the compiler, a step is 8 % slower).  Also
//   * key and value tiles go global -> LDS directly, three steps ahead (four buffers; 64 KB, two workgroups per CU), one barrier per
//     step; 16-byte pieces are XOR-swizzled on the way -- keys by row % 16 for the 16-byte operand reads of 16 rows, values by
//     2 (row % 8) for the transposing reads of 8 rows -- so that neither conflicts, and a buffer's address is a constant;
//   * rows past the prefix are read from its last row: finite values times a probability of zero;
//   * a workgroup is the four heads over 16 queries; its mapping to the XCDs is below.
// What bounds it now: instruction issue of a wave (about 200 instructions, 1280 clocks a step) in a launch of few workgroups, LDS reads
// (640 of 870 clocks per step and workgroup) in a full one.  Measured, 20 / 5 heads, us, group kernel / this one: 1 x 100 6.0 / 5.3,
// 1 x 512 17.2 / 12.8, 1 x 1920 69 / 46, 8 x 256 24.3 / 14.3, 4 x 512 37 / 19, 2 x 2048 152 / 99.  Tried, same bits: two heads per
// wave (half the LDS reads, twice the chain: 75 us at 1920), three buffers and three workgroups per CU (2 x 2048: 93, but
// 1 x 1920: 49), skipping the rescale where no maximum moved (level: twice the code).
#pragma once

#include "prefill_attention_kernel.h"

namespace terna {

constexpr int kWideRing = 4;                                           // tiles of 32 slots in LDS, keys and values
constexpr int kWideTile = kPrefillAttnKeys * 256;                      // bytes of one
constexpr int kWideLds = 2 * kWideRing * kWideTile;

// key_groups_reduce as statements that may be scheduled among others (all lanes are active wherever it stands)
template <bool IS_MAX>
__device__ __forceinline__ float wide_groups_reduce(float v)
{
    auto op = [](float a, float b) { return IS_MAX ? fmaxf(a, b) : a + b; };
    float a = v, b = v;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    v = op(a, b);
    a = v;
    b = v;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return op(a, b);
}

__global__ __launch_bounds__(256, 2) void terna_prefill_attention_wide_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ cache_k, const uint16_t* __restrict__ cache_v,
    const long long* __restrict__ pos, uint16_t* __restrict__ out, int B, int T, int H, int KV, int S, float scale, int per_seq, int q_row)
{
// as in the other kernels: the bits have to be theirs
#pragma clang fp contract(off)
    constexpr int D = 128, G = 4, DS = D / 32, DT = D / 16, KB = kPrefillAttnKeys;
    constexpr int ROWS = KB / G, LOADS = ROWS / 4;                    // a wave's rows of a tile, four to a load
    __shared__ __align__(16) uint8_t smem[kWideLds];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = lane & 15, g = lane >> 4;
    // Workgroups go to the XCDs round robin.  An XCD takes a run of the (sequence, kv head) pairs' eighths -- eighth c of a pair:
    // the query blocks c, c + 8, ... from the last one down -- so that the keys and values its workgroups read are those of
    // a few pairs (they stay in its L2: with every pair on every XCD the launch ran at the memory-side cache's rate), and
    // walks them longest prefixes first.
    const int pairs = B * KV, blocks = (T + 15) / 16;
    const int slot = blockIdx.x >> 3, round8 = slot / pairs;
    const int eighth = pairs * (blockIdx.x & 7) + slot - round8 * pairs;
    const int from_last = 8 * round8 + (eighth & 7);
    if (from_last >= blocks) return;
    const int t0 = (blocks - 1 - from_last) * 16, kvh = (eighth >> 3) % KV, b = (eighth >> 3) / KV;
    const int h = kvh * G + wave;
    const int t = t0 + qi < T ? t0 + qi : T - 1;
    long long p64 = pos[(per_seq ? b * T : 0) + t];
    p64 = p64 < 0 ? 0 : (p64 >= S ? S - 1 : p64);
    const int my_last = static_cast<int>(p64);
    int n_keys = my_last + 1, n_full = my_last + 1;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        n_keys = max(n_keys, __shfl_xor(n_keys, off));
        n_full = min(n_full, __shfl_xor(n_full, off));
    }
    n_keys = __builtin_amdgcn_readfirstlane(n_keys);
    n_full = __builtin_amdgcn_readfirstlane(n_full);
    const int steps = (n_keys + KB - 1) / KB;

    // q [B][H][T][D], or rows of q_row elements (q_row != 0)
    const uint16_t* qrow = q + (q_row ? (static_cast<size_t>(b) * T + t) * q_row + static_cast<size_t>(h) * D
                                      : ((static_cast<size_t>(b) * H + h) * T + t) * D);
    bf16x8 bq[DS];
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
        bq[ds] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qrow + 32 * ds + 8 * g));
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(bq[ds]));   // landed before the first hand-issued request

    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(cache_k + (static_cast<size_t>(b) * KV + kvh) * S * D);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(cache_v + (static_cast<size_t>(b) * KV + kvh) * S * D);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + wave * (ROWS * 256);
    const int r4 = lane >> 4, at = lane & 15;
    uint32_t k_piece[LOADS], v_piece[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = ROWS * wave + 4 * i + r4;
        k_piece[i] = (at ^ (row & 15)) << 4;
        v_piece[i] = (at ^ ((row & 7) << 1)) << 4;
    }
    // rows past the prefix are read from its last row
    auto load_rows = [&](const uint8_t* base, uint32_t piece, int step, int i, uint32_t lds) __attribute__((always_inline)) {
        const int k0 = step * KB < n_keys ? step * KB : n_keys - 1;    // uniform
        const int row = min(ROWS * wave + 4 * i + r4, n_keys - 1 - k0);
        lds_dma_b128(base + static_cast<size_t>(k0) * 256, row * 256 + piece, lds + i * 1024);
    };
    auto load_keys_at = [&](int step, int slot4, int i) __attribute__((always_inline)) { load_rows(kbase, k_piece[i], step, i, lds0 + slot4 * kWideTile); };
    auto load_values_at = [&](int step, int slot4, int i) __attribute__((always_inline)) {
        load_rows(vbase, v_piece[i], step, i, lds0 + (kWideRing + slot4) * kWideTile);
    };
    auto load_keys = [&](int step, int slot4) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_keys_at(step, slot4, i);
    };
    auto load_values = [&](int step, int slot4) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_values_at(step, slot4, i);
    };

    // operand addresses inside a tile: keys row 16 j + qi, piece 4 ds + g; values row 16 j + 4 g + qi / 4, dims 16 dt + 4 (qi % 4) .. +3
    int ka[DS], va[DT];
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) ka[ds] = qi * 256 + (((4 * ds + g) ^ qi) << 4);
    const int vrow = 4 * g + (qi >> 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) va[dt] = vrow * 256 + (((2 * dt + ((qi & 3) >> 1)) ^ ((vrow & 7) << 1)) << 4) + 8 * (qi & 1);
    auto key_operand = [&](const uint8_t* tile, int n) __attribute__((always_inline)) {          // n = 2 ds + j
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(tile + ka[n >> 1] + (n & 1) * 4096));
    };
    auto value_operand = [&](const uint8_t* tile, int dt) __attribute__((always_inline)) {
        using Tr = s16x4 __attribute__((address_space(3)))*;
        const u32x2 a0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Tr)(tile + va[dt])));
        const u32x2 a1 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Tr)(tile + va[dt] + 4096)));
        return __builtin_bit_cast(bf16x8, u32x4{a0.x, a0.y, a1.x, a1.y});
    };

    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -1e30f, l_run = 0.0f, alpha = 1.0f;
    struct Scores { f32x4 s[2]; };                                     // [16-key tile]
    bf16x8 p_hi, p_lo;
    bf16x8 kop[8];                                                     // the key operands of the next scores

    // Step i: its values times its probabilities, the next step's probabilities, the scores of the one after -- three strands that
    // do not depend on each other, woven by hand: 12 slices of two matrix instructions and about ten vector ones.
    auto step = [&](int i, int c, Scores& next, Scores& then, auto masked) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * LOADS) : "memory");
        const uint8_t* kt_next = smem + ((c + 3) & 3) * kWideTile;
        const uint8_t* vt = smem + (kWideRing + c) * kWideTile;
        const int left = my_last - (i + 1) * KB - 4 * g;               // key 16 j + v of the next step's tiles is visible: <= left
        bf16x8 vop[DT];
        float top = -1e30f, m_new = 0.0f, alpha_next = 1.0f, psum = 0.0f, p[8];
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            // ---- memory: operands of four slices ahead, tiles of steps ahead, spread so that the waves' bursts do not queue
            if (k < 8) vop[k] = value_operand(vt, k);
            if (k >= 4) kop[k - 4] = key_operand(kt_next, k - 4);
            if (k >= 1 && (k - 1) % 3 == 0) {
                const int l = (k - 1) / 3;
                if (l < LOADS) load_keys_at(i + 5, (c + 1) & 3, l);
                else if (l < 2 * LOADS) load_values_at(i + 3, (c + 3) & 3, l - LOADS);
            }
            // ---- matrix: 4 slices of scores, 8 of outputs
            if (k < 4) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    next.s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[2 * k + j], bq[k], k == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : next.s[j], 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 8; ++v) o[2 * k + (v >> 2)][v & 3] *= alpha;
            } else {
                const int d = ((k - 4) >> 1) * 2;
#pragma unroll
                for (int dt = d; dt < d + 2; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vop[dt], k % 2 == 0 ? p_hi : p_lo, o[dt], 0, 0, 0);
            }
            // ---- vector
            if (k < 2) {                                               // scaled, masked, maximum
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    then.s[k][v] = (!MASKED || 16 * k + v <= left) ? then.s[k][v] * scale : -1e30f;
                    top = fmaxf(top, then.s[k][v]);
                }
                asm volatile("" : "+v"(top));
            } else if (k == 2) {
                top = wide_groups_reduce<true>(top);
                asm volatile("" : "+v"(top));
            } else if (k == 3) {
                m_new = fmaxf(m_run, top);
                alpha_next = __expf(m_run - m_new);
                m_run = m_new;
                asm volatile("" : "+v"(alpha_next));
            } else if (k < 8) {                                        // a masked key's term is exp(-1e30 - maximum) = 0
#pragma unroll
                for (int e = 2 * (k - 4); e < 2 * (k - 4) + 2; ++e) {
                    p[e] = __expf(then.s[e >> 2][e & 3] - m_new);
                    psum += p[e];
                }
                asm volatile("" : "+v"(psum));
            } else {
                const int w = k - 8;
                hi[w] = pack_bf16x2(p[2 * w], p[2 * w + 1]);
                lo[w] = pack_bf16x2(p[2 * w] - __uint_as_float(hi[w] << 16), p[2 * w + 1] - __uint_as_float(hi[w] & 0xffff0000u));
                asm volatile("" : "+v"(hi[w]), "+v"(lo[w]));
            }
            __builtin_amdgcn_sched_barrier(0x4);               // scalar instructions may pass
        }
        l_run = __fmaf_rn(l_run, alpha_next, psum);
        p_hi = __builtin_bit_cast(bf16x8, u32x4{hi[0], hi[1], hi[2], hi[3]});
        p_lo = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], lo[2], lo[3]});
        alpha = alpha_next;
    };

    Scores s0, s1;
    auto scores = [&](const uint8_t* tile, Scores& to) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 8; ++n)
            to.s[n & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(key_operand(tile, n), bq[n >> 1], n < 2 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : to.s[n & 1], 0, 0, 0);
    };
    load_keys(0, 0);
    if (steps == 1) {
        load_values(0, 0);
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        scores(smem, s0);
    } else {
        load_keys(1, 1);
        load_keys(2, 2);
        load_values(0, 0);
        load_keys(3, 3);
        load_values(1, 1);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * LOADS) : "memory");          // keys of the steps 0, 1
        scores(smem, s0);
        scores(smem + kWideTile, s1);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * LOADS) : "memory");
        load_keys(4, 0);
        load_values(2, 2);
#pragma unroll
        for (int n = 0; n < 8; ++n) kop[n] = key_operand(smem + 2 * kWideTile, n);
    }
    {   // the first step's probabilities
        float p[8], hi_f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = 16 * (e >> 2) + 4 * g + (e & 3) <= my_last ? s0.s[e >> 2][e & 3] * scale : -1e30f;
            m_run = fmaxf(m_run, p[e]);
        }
        m_run = wide_groups_reduce<true>(m_run);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = __expf(p[e] - m_run);
            l_run += p[e];
        }
        const u32x4 hi = pack_bf16x8(p);
        unpack_bf16x8(hi, hi_f);
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] -= hi_f[e];
        p_hi = __builtin_bit_cast(bf16x8, hi);
        p_lo = __builtin_bit_cast(bf16x8, pack_bf16x8(p));
    }
    int i = 0;
    for (; KB * (i + 5) <= n_full; i += 4) {
        step(i, 0, s0, s1, std::false_type{});
        step(i + 1, 1, s1, s0, std::false_type{});
        step(i + 2, 2, s0, s1, std::false_type{});
        step(i + 3, 3, s1, s0, std::false_type{});
    }
    for (; i + 1 < steps; ++i) {
        step(i, i & 3, s0, s1, std::true_type{});
        s1 = s0;
    }
    {
        const uint8_t* vt = smem + (kWideRing + (i & 3)) * kWideTile;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const bf16x8 a = value_operand(vt, dt);
            o[dt] *= alpha;
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p_hi, o[dt], 0, 0, 0);
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p_lo, o[dt], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    uint8_t* rows = smem + wave * (16 * 272);                          // bf16 [16 queries][128], rows 16 bytes apart in the banks
    const float inv = 1.0f / wide_groups_reduce<false>(l_run);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<u32x2*>(rows + qi * 272 + (16 * dt + 4 * g) * 2) =
            u32x2{pack_bf16x2(o[dt][0] * inv, o[dt][1] * inv), pack_bf16x2(o[dt][2] * inv, o[dt][3] * inv)};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int row = 4 * n + r4;
        if (t0 + row < T)
            *reinterpret_cast<u32x4*>(out + (static_cast<size_t>(b) * T + t0 + row) * (static_cast<size_t>(H) * D) + static_cast<size_t>(h) * D + 8 * at) =
                *reinterpret_cast<const u32x4*>(rows + row * 272 + at * 16);
    }
}

}  // namespace terna
