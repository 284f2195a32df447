// The inputs of a single-token step, by one workgroup of 256 threads per sequence: x_out[b] = embedding[tokens[b]] with its
// partials under norm_w (per 512 columns the sum of h^2 and the maximum of |h * norm_w|, as terna_row_stats_kernel leaves
// them), and the rows of the RoPE table at the sequences' positions, cos rows then sin rows (rope_out [2][B][half]; table
// [S][2][half]).  A token or position outside its table is clamped (device memory the host cannot check).
#pragma once

#include "norm_quant_kernel.h"

namespace terna {

struct StepInputs {
    const long long *tokens, *pos;
    int per_seq;
    const uint16_t* embedding;
    int V, K;
    const float* rope_table;
    int S, half;
    const uint16_t* norm_w;
    uint16_t* x_out;
    float2* stats_out;
    float* rope_out;
    int count;                                   // partials of a row
};

// HANDOVER: x_out is read where the words are their own flags (step_kernel.h): 0xffffffff is not one of them.
template <bool HANDOVER>
__device__ __forceinline__ void step_inputs_row(const StepInputs& in, int b, int B)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int V = in.V, K = in.K, S = in.S, half = in.half;
    long long t = in.tokens[b], p = in.pos[in.per_seq ? b : 0];
    t = t < 0 ? 0 : (t >= V ? V - 1 : t);
    p = p < 0 ? 0 : (p >= S ? S - 1 : p);
    const uint16_t* row = in.embedding + static_cast<size_t>(t) * K;
    if (tid < 2 * half / 4) {                           // half is a multiple of 4: 16-byte pieces, cos row then sin row
        const int which = tid / (half / 4), piece = tid - which * (half / 4);
        const f32x4 v = *reinterpret_cast<const f32x4*>(in.rope_table + (static_cast<size_t>(p) * 2 + which) * half + 4 * piece);
        *reinterpret_cast<f32x4*>(in.rope_out + (static_cast<size_t>(which) * B + b) * half + 4 * piece) = v;
    }
    for (int part = wave; part < in.count; part += 4) {
        const int c = part * 512 + lane * 8;
        float ssq = 0.0f, pmax = 0.0f;
        if (c < K) {                                    // K is a multiple of 8
            u32x4 hv = *reinterpret_cast<const u32x4*>(row + c);
            if constexpr (HANDOVER) {
#pragma unroll
                for (int e = 0; e < 4; ++e) hv[e] = hv[e] < 0xffffffffu ? hv[e] : 0xfffffffeu;
            }
            *reinterpret_cast<u32x4*>(in.x_out + static_cast<size_t>(b) * K + c) = hv;
            float f[8], w[8];
            unpack_bf16x8(hv, f);
            unpack_bf16x8(*reinterpret_cast<const u32x4*>(in.norm_w + c), w);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                ssq = fmaf(f[e], f[e], ssq);
                pmax = max_keep_nan(pmax, fabsf(__fmul_rn(f[e], w[e])));
            }
        }
        ssq = wave_sum(ssq);
        pmax = wave_amax(pmax);
        if (lane == 0) in.stats_out[static_cast<size_t>(b) * in.count + part] = float2{ssq, pmax};
    }
}

}  // namespace terna
