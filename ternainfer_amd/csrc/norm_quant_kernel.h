// Fused prologue of a ternary linear: [residual add | relu(x1)^2 * x3] -> RMSNorm -> per-row
// absmax int8 quantisation, one workgroup per activation row.
//
// This is the glue the reference runs as separate PyTorch / xformers / Inductor kernels between two
// bitlinear calls (model.py:120-123 quant_input; model.py:236 attn_sub_norm; :280 ffn_sub_norm over
// squared_relu(x1) * x3; :330, :334 the residual adds and the two block norms).  Per row:
//
//   h  = x                                   (plain)
//      = bf16(x + residual)                  (residual add; h is also written back as the new stream)
//      = bf16(bf16(relu(x1)^2) * x3)         (gated FFN; x1 = row[0:F], x3 = row[F:2F])
//   y  = bf16(h * rsqrt(mean(h^2) + eps) * weight)          fp32 inside, one rounding at the end
//   s  = bf16(127 / max(max|y|, 1e-5));  q = clamp(rint(y * s), -128, 127)   (fp32 inside; `quant_mode` selects
//        which of the reference's ways of evaluating these two lines is reproduced: QuantMode in terna_common.h)
//
// The row stays in registers between the three passes; HBM sees each input element once and each
// output element once.  Rows are independent, so the grid is M workgroups of 256 threads, or of one for every
// eight elements (terna_norm_quant_wide_kernel: few rows), and those of fetch_next_weights.
#pragma once

#include "terna_common.h"

namespace terna {

constexpr int kNormThreads = 256;
constexpr int kNormMaxVecs = 4;                       // 8-element vectors per thread: K <= 8192

// Reductions over groups of LANES consecutive lanes (LANES = 2 .. 64, a power of two) with the data
// parallel primitives of the VALU instead of LDS-crossbar shuffles: a ds_bpermute round trip costs
// on the order of a hundred cycles and a 64-lane butterfly needs six of them in sequence; the
// quad / half-row / row permutations below are ordinary VALU operands.  Every lane of the wave must
// be active.  The result is the same in every lane of a group; the order of the additions is
// fixed (pairs, quads, eights, sixteens, then rows 0+1 and 2+3, then the halves).
template <int CTRL>
__device__ __forceinline__ float dpp_permute(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_permute_u32(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true));
}
constexpr int kDppRowShl4 = 0x104;        // lane i <- lane i + 4 within 16 lanes (0 past the row)
constexpr int kDppRowShl8 = 0x108;
constexpr int kDppRowShl12 = 0x10C;
constexpr int kDppSwapPairs = 0xB1;       // quad_perm [1, 0, 3, 2]: lane ^ 1
constexpr int kDppSwapHalfQuads = 0x4E;   // quad_perm [2, 3, 0, 1]: lane ^ 2
constexpr int kDppHalfRowMirror = 0x141;  // lane i <-> 7 - i within 8 lanes
constexpr int kDppRowMirror = 0x140;      // lane i <-> 15 - i within 16 lanes

template <int LANES, typename Op>
__device__ __forceinline__ uint32_t group_fold(uint32_t v, Op op)
{
    static_assert(LANES >= 1 && LANES <= 64 && (LANES & (LANES - 1)) == 0, "group size");
    if constexpr (LANES >= 2) v = op(v, dpp_permute_u32<kDppSwapPairs>(v));
    if constexpr (LANES >= 4) v = op(v, dpp_permute_u32<kDppSwapHalfQuads>(v));
    if constexpr (LANES >= 8) v = op(v, dpp_permute_u32<kDppHalfRowMirror>(v));     // quads are uniform by now
    if constexpr (LANES >= 16) v = op(v, dpp_permute_u32<kDppRowMirror>(v));        // ... and so are the halves of a row
    if constexpr (LANES >= 32) {
        const uint32_t r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
        const uint32_t r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
        // 32 lanes: rows 0|1 and 2|3, lane ^ 16 through the row's uniform value of the neighbouring row
        if constexpr (LANES == 32) v = (threadIdx.x & 32) ? op(r2, r3) : op(r0, r1);
        else v = op(op(r0, r1), op(r2, r3));
    }
    return v;
}
template <int LANES, bool IS_MAX>
__device__ __forceinline__ float group_reduce(float v)
{
    return __uint_as_float(group_fold<LANES>(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        const float x = __uint_as_float(a), y = __uint_as_float(b);
        return __float_as_uint(IS_MAX ? fmaxf(x, y) : x + y);
    }));
}
// Maximum of magnitudes that keeps a NaN (max_keep_nan): as bits, without their sign, numbers, infinity and NaN are in order,
// and an integer maximum takes its operand through the permutation where a float one needs three instructions.
template <int LANES>
__device__ __forceinline__ float group_amax(float v)
{
    return __uint_as_float(group_fold<LANES>(__float_as_uint(v) & 0x7fffffffu, [](uint32_t a, uint32_t b) { return a > b ? a : b; }));
}

__device__ __forceinline__ float wave_sum(float v) { return group_reduce<64, false>(v); }
__device__ __forceinline__ float wave_max(float v) { return group_reduce<64, true>(v); }
__device__ __forceinline__ float wave_amax(float v) { return group_amax<64>(v); }

__device__ __forceinline__ void unpack_bf16x8(const u32x4& v, float f[8])
{
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = __uint_as_float(d[j] << 16);
        f[2 * j + 1] = __uint_as_float(d[j] & 0xffff0000u);
    }
}
__device__ __forceinline__ u32x4 pack_bf16x8(const float f[8])
{
    uint32_t d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) d[j] = pack_bf16x2(f[2 * j], f[2 * j + 1]);
    return u32x4{d[0], d[1], d[2], d[3]};
}
__device__ __forceinline__ float round_bf16(float v) { return bf16_bits_to_float(float_to_bf16_bits(v)); }

// The last two passes: the row's maximum from the threads' own (`amax`), then the scale and the int8 values.
template <int NV>
__device__ __forceinline__ void quant_pass(const float (&h)[NV][8], float amax, int K, size_t row, int8_t* __restrict__ xq_out,
                                           uint16_t* __restrict__ s_out, int quant_mode)
{
    __shared__ float red[kNormThreads / 64];
    const int tid = threadIdx.x;
    const int nvec = K >> 3;
    amax = wave_amax(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = max_keep_nan(max_keep_nan(red[0], red[1]), max_keep_nan(red[2], red[3]));
    uint16_t s_bits;
    const float s = quant_scale(amax, quant_mode, &s_bits);
    if (tid == 0) s_out[row] = s_bits;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kNormThreads;
        if (v < nvec) {
            uint32_t q[2] = {0u, 0u};
            if (quant_mode == QUANT_ROUNDED) {
#pragma unroll
                for (int j = 0; j < 2; ++j) q[j] = quant_rounded4(h[i][4 * j], h[i][4 * j + 1], h[i][4 * j + 2], h[i][4 * j + 3], s);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float r = quant_value(h[i][j], s, quant_mode);
                    q[j >> 2] |= (static_cast<uint32_t>(static_cast<int>(r)) & 0xffu) << (8 * (j & 3));
                }
            }
            *reinterpret_cast<u32x2*>(xq_out + row * K + 8 * v) = u32x2{q[0], q[1]};
        }
    }
}

// The passes behind the formation of a row in registers (h[i][j] = element
// 8 (tid + kNormThreads i) + j, vectors past K / 8 unused; raw_w the norm weights of the same elements): sum of squares
// -- per thread in element order, the lanes of a wave by group_reduce, the four waves pairwise -- then the norm, the row
// maximum, the scale and the int8 values.  y_out / xq_out + s_out: optional outputs.
template <int NV>
__device__ __forceinline__ void norm_quant_passes(float (&h)[NV][8], const u32x4 (&raw_w)[NV], int K, float eps, size_t row,
                                                  uint16_t* __restrict__ y_out, int8_t* __restrict__ xq_out,
                                                  uint16_t* __restrict__ s_out, int quant_mode)
{
    __shared__ float red[kNormThreads / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int nvec = K >> 3;
    float ssq = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (tid + i * kNormThreads < nvec) {
#pragma unroll
            for (int j = 0; j < 8; ++j) ssq = fmaf(h[i][j], h[i][j], ssq);
        }
    }
    ssq = wave_sum(ssq);
    if (lane == 0) red[wave] = ssq;
    __syncthreads();
    const float total = (red[0] + red[1]) + (red[2] + red[3]);
    const float rstd = rsqrtf(total / static_cast<float>(K) + eps);

    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kNormThreads;
        if (v < nvec) {
            float w[8];
            unpack_bf16x8(raw_w[i], w);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                h[i][j] = round_bf16(h[i][j] * rstd * w[j]);
                amax = max_keep_nan(amax, fabsf(h[i][j]));
            }
            if (y_out != nullptr) *reinterpret_cast<u32x4*>(y_out + row * K + 8 * v) = pack_bf16x8(h[i]);
        }
    }
    if (xq_out == nullptr) return;

    quant_pass<NV>(h, amax, K, row, xq_out, s_out, quant_mode);
}

// Spare workgroups of a launch that norms and quantises rows bring the packed weights of the linear behind it into the L2s while its few
// workgroups wait for memory and each other: the linear then starts on data that is one L2 trip away instead of one to HBM (a model's
// weights are read once per pass and twice the size of the last cache).  A load of four bytes fetches a line; nobody waits for it but
// the end of the launch.  Measured in turn, us, without -> with: decode step of 32 sequences x 512 slots of different lengths 1567 -> 1501, of one length
// 1588 -> 1519, 64 x 512 1905 -> 1817, 64 x 1000 2159 -> 2073; prompts of 100 and 1920 tokens 1614 -> 1581 and 6576 -> 6444; in the launch that also
// merges the attention's splits 8 x 1528 slots 1214 -> 1199, 16 x 1528 1361 -> 1354.  (Cards differ: the first of these with 1500 - 1540, the 1920 tokens with 6440 - 7050.)
// Tried: weights of the launch after next as well, or instead (32 sequences 1505 - 1531), 64 workgroups
// (1525) and 384 (1508); in the shorter launch that quantises from a producer's statistics (up to 16 rows) it costs 5 - 20 us
// a step, in the quantisation in front of a linear module's call it is level.
__device__ __forceinline__ void fetch_next_weights(const NextWeights& next, int first)
{
    const uint32_t xcd = blockIdx.x & 7, per_xcd = next.workgroups >> 3;
    const uint32_t rank = (blockIdx.x - first - ((xcd - (first & 7) + 8) & 7)) >> 3;    // among the fetching workgroups of this XCD
    const uint32_t step = per_xcd * blockDim.x;
    const __amdgpu_buffer_rsrc_t lines = make_raw_buffer(next.base, next.lines << 7);      // a load past them fetches nothing
    auto line_of = [&](uint32_t g) {                     // of this XCD's lines, tile by tile: ascending
        const uint32_t tile = g / next.tile_lines;
        return (8 * tile + xcd) * next.tile_lines + (g - tile * next.tile_lines);
    };
    for (uint32_t g = rank * blockDim.x + threadIdx.x; line_of(g) < next.lines; g += 4 * step) {
        uint32_t d[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = __builtin_amdgcn_raw_buffer_load_b32(lines, line_of(g + j * step) << 7, 0, 0);
        asm volatile("" ::"v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]));
    }
}

// GLU = false: x [M][K], optional residual [M][K] and sum_out [M][K].
// GLU = true : x [M][2K] holding x1 | x3; residual / sum_out unused.
// NV = 8-element vectors per thread (K <= 2048 NV); SECOND = there is a second operand (the residual, or x3).
template <bool GLU, int NV = kNormMaxVecs, bool SECOND = true>
__global__ __launch_bounds__(kNormThreads) void terna_norm_quant_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight, int K,
    float eps, uint16_t* __restrict__ sum_out, uint16_t* __restrict__ y_out, int8_t* __restrict__ xq_out,
    uint16_t* __restrict__ s_out, int quant_mode, int rows, NextWeights next)
{
    static_assert(!GLU || SECOND, "the gate has two operands");
    if (static_cast<int>(blockIdx.x) >= rows) {
        fetch_next_weights(next, rows);
        return;
    }
    const int tid = threadIdx.x;
    const size_t row = blockIdx.x;
    const int nvec = K >> 3;
    const uint16_t* xr = x + row * static_cast<size_t>(GLU ? 2 * K : K);

    // Every global load of the row -- input, second operand, norm weight -- is issued before the
    // first use: with one row per workgroup the kernel's time is its chain of memory round trips, and the address
    // unit takes a wave's load in a dozen cycles whatever it fetches: no more loads than the row needs.
    // The loads are unconditional on clamped addresses (a load inside a branch is waited for at
    // the join, which would serialise them).
    u32x4 raw_x[NV], raw_b[NV], raw_w[NV];
    const uint16_t* br = GLU ? xr + K : (SECOND ? residual + row * K : xr);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kNormThreads;
        const int vc = v < nvec ? v : nvec - 1;
        raw_x[i] = *reinterpret_cast<const u32x4*>(xr + 8 * vc);
        if constexpr (SECOND) raw_b[i] = *reinterpret_cast<const u32x4*>(br + 8 * vc);
        raw_w[i] = *reinterpret_cast<const u32x4*>(weight + 8 * vc);
    }
    // pin the loads here: otherwise they are sunk into the branches below, next to their uses
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        pin_registers(raw_x[i]);
        if constexpr (SECOND) pin_registers(raw_b[i]);
        pin_registers(raw_w[i]);
    }

    float h[NV][8];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kNormThreads;
        if (v < nvec) {
            unpack_bf16x8(raw_x[i], h[i]);
            if constexpr (GLU) {
                float g[8];
                unpack_bf16x8(raw_b[i], g);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float r = max_keep_nan(h[i][j], 0.0f);
                    h[i][j] = round_bf16(round_bf16(r * r) * g[j]);
                }
            } else if constexpr (SECOND) {
                float r[8];
                unpack_bf16x8(raw_b[i], r);
#pragma unroll
                for (int j = 0; j < 8; ++j) h[i][j] = round_bf16(h[i][j] + r[j]);
                if (sum_out != nullptr) *reinterpret_cast<u32x4*>(sum_out + row * K + 8 * v) = pack_bf16x8(h[i]);
            }
        }
    }
    norm_quant_passes<NV>(h, raw_w, K, eps, row, y_out, xq_out, s_out, quant_mode);
}

// The plain form for few rows: a thread for every eight-element vector (up to sixteen waves).  The sum of squares is defined by 256
// threads that take the vectors t, t + 256, ... in turn: the first four waves read those as well and add them up so; everything behind
// the sum is one vector a thread.  A row's launch is what one wave does in a row: of 4000 clocks (K = 2560; 5900 for K = 6912) the request took 900,
// the data 600, the sum 550, norm and maximum 1100, quantisation 700, and the first wave had two vectors in each (four).  Blocks of a pass
// in a graph, us, the form above -> this: 32 sequences 41.4 -> 40.9, a prompt of 100 tokens 47.5 -> 46.9; of 256 65.5 -> 65.5, 600 102.6 -> 104.3, 1920 216 ->
// 224: many rows fill the chip either way, and the sums read twice.
constexpr int kNormWideRows = 128;
template <int NV>
__global__ __launch_bounds__(1024) void terna_norm_quant_wide_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ weight, int K, float eps, int rows, int quant_mode,
    int8_t* __restrict__ xq_out, uint16_t* __restrict__ s_out, uint16_t* __restrict__ y_out, NextWeights next)
{
    if (static_cast<int>(blockIdx.x) >= rows) {
        fetch_next_weights(next, rows);
        return;
    }
    __shared__ float sums[kNormThreads / 64];
    __shared__ __align__(16) float maxima[16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t row = blockIdx.x;
    const int nvec = K >> 3, vc = tid < nvec ? tid : nvec - 1;
    const uint16_t* xr = x + row * static_cast<size_t>(K);
    u32x4 raw = *reinterpret_cast<const u32x4*>(xr + 8 * vc);
    u32x4 raw_w;
    if (wave < kNormThreads / 64) {
        u32x4 more[NV];
#pragma unroll
        for (int i = 1; i < NV; ++i) {
            const int v = tid + i * kNormThreads;
            more[i] = *reinterpret_cast<const u32x4*>(xr + 8 * (v < nvec ? v : nvec - 1));
        }
        raw_w = *reinterpret_cast<const u32x4*>(weight + 8 * vc);
        if (tid < 16) maxima[tid] = 0.0f;
        more[0] = raw;
        float ssq = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            float f[8];
            unpack_bf16x8(more[i], f);
            if (tid + i * kNormThreads < nvec) {
#pragma unroll
                for (int j = 0; j < 8; ++j) ssq = fmaf(f[j], f[j], ssq);
            }
        }
        ssq = wave_sum(ssq);
        if (lane == 0) sums[wave] = ssq;
    } else {
        raw_w = *reinterpret_cast<const u32x4*>(weight + 8 * vc);
    }
    __syncthreads();
    const float total = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    const float rstd = rsqrtf(total / static_cast<float>(K) + eps);
    float h[8], w[8], amax = 0.0f;
    unpack_bf16x8(raw, h);
    unpack_bf16x8(raw_w, w);
#pragma unroll
    for (int j = 0; j < 8; ++j) {                                    // (a clamped vector is one of the row's: the maximum may see it twice)
        h[j] = round_bf16(h[j] * rstd * w[j]);
        amax = max_keep_nan(amax, fabsf(h[j]));
    }
    amax = wave_amax(amax);
    if (lane == 0) maxima[wave] = amax;
    if (y_out != nullptr && tid < nvec) *reinterpret_cast<u32x4*>(y_out + row * K + 8 * tid) = pack_bf16x8(h);
    __syncthreads();
    amax = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const f32x4 m = *reinterpret_cast<const f32x4*>(&maxima[4 * q]);
        amax = max_keep_nan(max_keep_nan(amax, max_keep_nan(m[0], m[1])), max_keep_nan(m[2], m[3]));
    }
    uint16_t s_bits;
    const float s = quant_scale(amax, quant_mode, &s_bits);
    if (tid == 0) s_out[row] = s_bits;
    if (tid >= nvec) return;
    uint32_t q[2] = {0u, 0u};
    if (quant_mode == QUANT_ROUNDED) {
#pragma unroll
        for (int j = 0; j < 2; ++j) q[j] = quant_rounded4(h[4 * j], h[4 * j + 1], h[4 * j + 2], h[4 * j + 3], s);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j >> 2] |= (static_cast<uint32_t>(static_cast<int>(quant_value(h[j], s, quant_mode))) & 0xffu) << (8 * (j & 3));
    }
    *reinterpret_cast<u32x2*>(xq_out + row * K + 8 * tid) = u32x2{q[0], q[1]};
}

// quant_input of rows that no norm precedes (SpBitLinear on its own): x [M][K] -> (xq, s), one workgroup per row.
// Bound: HBM on many rows, the launch on few.  It stands for the eleven elementwise and reduction launches of the same
// lines in PyTorch (5000 x 6912: 350 us there, 21 us here; one row: 75 us of host time there, 2 us).
template <int NV>
__global__ __launch_bounds__(kNormThreads) void terna_quant_input_kernel(const uint16_t* __restrict__ x, int K, int8_t* __restrict__ xq_out,
                                                                         uint16_t* __restrict__ s_out, int quant_mode)
{
    const int tid = threadIdx.x;
    const size_t row = blockIdx.x;
    const int nvec = K >> 3;
    u32x4 raw[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {              // all requests first, on clamped addresses
        const int v = tid + i * kNormThreads;
        raw[i] = *reinterpret_cast<const u32x4*>(x + row * K + 8 * (v < nvec ? v : nvec - 1));
    }
    float h[NV][8], amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {              // (a clamped vector is one of the row's: the maximum may see it twice)
        unpack_bf16x8(raw[i], h[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = max_keep_nan(amax, fabsf(h[i][j]));
    }
    quant_pass<NV>(h, amax, K, row, xq_out, s_out, quant_mode);
}

}  // namespace terna
