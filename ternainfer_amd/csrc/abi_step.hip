// C ABI of the decode step in one launch (step_kernel.h).  Declarations: include/ternaspmm.h.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "../../include/ternaspmm.h"
#include "host_util.h"
#include "step_inputs.h"
#include "step_kernel.h"

using namespace terna;

namespace {

constexpr int kClearGroups = 512;

// In front of the step: its inputs (the first B workgroups), and the exchange buffer cleared to "not there yet"; its first word
// (StepArgs::alive) is what a wait may take.
__global__ __launch_bounds__(256) void terna_step_begin_kernel(const StepInputs in, int B, u32x4* clear, long long vecs, uint32_t patience)
{
    const int b = blockIdx.x;
    if (b < B) {
        step_inputs_row<true>(in, b, B);
        return;
    }
    for (long long v = static_cast<long long>(b - B) * 256 + threadIdx.x; v < vecs; v += static_cast<long long>(gridDim.x - B) * 256)
        clear[v] = u32x4{v == 0 ? patience : kStepEmpty, kStepEmpty, kStepEmpty, kStepEmpty};
}

uint32_t up(long long bytes) { return static_cast<uint32_t>((bytes + 255) & ~255ll); }

StepExchange exchange_of(const ternaspmm_step_desc& d)
{
    const long long M = d.M, wide = static_cast<long long>(d.heads) * d.head_dim, qkv_n = wide + 2ll * d.kv_heads * d.head_dim;
    StepExchange e{};
    uint32_t at = 0;
    auto part = [&](long long bytes) {
        const uint32_t here = at;
        at += up(bytes);
        return here;
    };
    e.qkv = part(M * qkv_n * 2);
    e.attention = part(M == 1 ? static_cast<long long>(d.heads) * d.splits * kStepRecord : M * wide * 2);
    e.mid = part(M * d.dim * 2);
    e.inner = part(M * d.ffn * 2);
    e.quantised = part(M > 1 ? M * d.ffn : 0);
    e.scales = part(M > 1 ? M * 64 : 0);
    e.out = part(M * d.dim * 2);
    e.bytes = at;
    return e;
}

const void* step_kernel_of(int M)
{
    return M == 1 ? reinterpret_cast<const void*>(terna_decode_step_kernel<1, false>)
                  : M == 2 ? reinterpret_cast<const void*>(terna_decode_step_kernel<2, false>) : reinterpret_cast<const void*>(terna_decode_step_kernel<4, false>);
}

// Whether as many grids as the runtime runs side by side for a process are resident together, whatever their order: the workgroups
// of a step wait for each other, and one whose do not come loses the time of the waits and of doing it in order.  A
// queue with a mask of CUs has to hold them with those.
bool grids_fit(int M, hipStream_t st)
{
    static const int queues = [] {               // hardware queues per process (HIP's default: 4)
        const char* v = std::getenv("GPU_MAX_HW_QUEUES");
        const int n = v ? std::atoi(v) : 4;
        return n < 4 ? 4 : n;
    }();
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
    static std::mutex mutex;
    static int resident[64][3] = {};             // workgroups of the kernel on the device; 0: not asked yet
    static int device_cus[64] = {};
    const int which = M == 1 ? 0 : M == 2 ? 1 : 2;
    {
        std::lock_guard<std::mutex> lock(mutex);
        if (resident[dev][which] == 0) {
            int per_cu = 0;
            if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, step_kernel_of(M), kStepThreads, 0) != hipSuccess || per_cu < 1) {
                (void)hipGetLastError();
                return false;
            }
            resident[dev][which] = per_cu;
            device_cus[dev] = cus;
        }
        cus = device_cus[dev];
    }
    uint32_t mask[16] = {};
    if (hipExtStreamGetCUMask(st, 16, mask) == hipSuccess) {
        int allowed = 0;
        for (uint32_t m : mask) allowed += __builtin_popcount(m);
        if (allowed > 0 && allowed < cus) cus = allowed;
    } else {
        (void)hipGetLastError();
    }
    return static_cast<long>(resident[dev][which]) * cus >= static_cast<long>(queues) * kStepGroups;
}

bool step_shape_ok(const ternaspmm_step_desc& d)
{
    const long wide = static_cast<long>(d.heads) * d.head_dim, qkv_n = wide + 2l * d.kv_heads * d.head_dim;
    if (d.M < 1 || d.M > 4 || d.layers < 1 || d.layers > 1024 || d.heads < 1 || d.kv_heads < 1 || d.heads % d.kv_heads != 0 || d.head_dim != kStepHeadDim ||
        d.dim < 64 || d.dim % 64 != 0 || d.dim > 64 * kStepTiles || wide > 64 * kStepTiles || d.ffn < 64 || d.ffn % 64 != 0 || d.ffn > 64 * kStepWideTiles ||
        qkv_n / 16 > kStepGroups || d.slots < 1 || d.vocab < 1 || !groups_ok(d.ws_num_qkv) || !groups_ok(d.ws_num_o) || !groups_ok(d.ws_num_down) ||
        ternaspmm_row_stats_count(d.dim) < 1 || ternaspmm_row_stats_count(d.dim) > 64)
        return false;
    const int per = d.heads / d.kv_heads;
    if (step_unit_groups((d.M == 1 ? d.splits : d.M) * d.kv_heads, d.M == 1 ? per : 2 * per) > kStepGroups) return false;
    if (d.M == 1) {
        if ((d.splits != 2 && d.splits != 4 && d.splits != 8) || d.slots > d.splits * kStepMaxSplitSlots) return false;
    } else {
        if (d.splits != 1 || d.slots > step_max_slots(d.M)) return false;
    }
    return d.M == 1 || quant_mode() != QUANT_EAGER;          // (the int8 words that are handed over need one value no integer takes)
}

// groups, patience: of the resident launches.
int enqueue_step(const ternaspmm_step_desc* d, const ternaspmm_step_block* blocks, const long long* tokens, const long long* pos, const terna_bf16* embedding,
                 const float* rope_table, void* scratch, terna_bf16* x_out, int groups, uint32_t patience, terna_stream stream)
{
    const long long bytes = ternaspmm_decode_step_bytes(d);
    if (bytes < 0 || blocks == nullptr || tokens == nullptr || pos == nullptr || embedding == nullptr || rope_table == nullptr || scratch == nullptr ||
        x_out == nullptr)
        return -1;
    auto misaligned = [](const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
    if (misaligned(embedding) || misaligned(rope_table) || misaligned(x_out) || (reinterpret_cast<uintptr_t>(scratch) & 255) != 0) return -1;
    for (int n = 0; n < d->layers; ++n) {
        const ternaspmm_step_block& b = blocks[n];
        if (misaligned(b.wqkv) || misaligned(b.wo) || misaligned(b.w13) || misaligned(b.w2) || misaligned(b.attention_norm) || misaligned(b.attn_sub_norm) ||
            misaligned(b.ffn_norm) || misaligned(b.ffn_sub_norm) || misaligned(b.cache_k) || misaligned(b.cache_v) || b.ws_qkv == nullptr || b.ws_o == nullptr ||
            b.ws_13 == nullptr || b.ws_down == nullptr)
            return -1;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!grids_fit(d->M, st)) return -1;

    const int count = ternaspmm_row_stats_count(d->dim), half = d->head_dim / 2;
    StepArgs a{};
    a.at = exchange_of(*d);
    char* base = static_cast<char*>(scratch);
    const long long cleared = kStepControlBytes + static_cast<long long>(d->layers) * a.at.bytes;
    uint16_t* x = reinterpret_cast<uint16_t*>(base + cleared);
    float2* stats = reinterpret_cast<float2*>(base + cleared + up(2ll * d->M * d->dim));
    float* rope = reinterpret_cast<float*>(base + cleared + up(2ll * d->M * d->dim) + up(8ll * d->M * count));
    const StepInputs in{tokens, pos, d->per_sequence != 0, embedding, d->vocab, d->dim, rope_table, d->slots, half, blocks[0].attention_norm, x, stats, rope, count};
    terna_step_begin_kernel<<<dim3(d->M + kClearGroups), dim3(256), 0, st>>>(in, d->M, reinterpret_cast<u32x4*>(base), cleared / 16, patience);

    a.alive = reinterpret_cast<uint32_t*>(base);
    a.pos = pos;
    a.cosv = rope;
    a.sinv = rope + static_cast<size_t>(d->M) * half;
    a.M = d->M, a.dim = d->dim, a.ffn = d->ffn, a.H = d->heads, a.KV = d->kv_heads, a.S = d->slots, a.SP = d->splits, a.per_seq = d->per_sequence != 0;
    a.stats_count = count, a.quant_mode = quant_mode(), a.ws_qkv = d->ws_num_qkv, a.ws_o = d->ws_num_o, a.ws_2 = d->ws_num_down;
    a.eps = d->eps, a.scale = d->scale;
    auto launches = [&](auto ordered) {
        constexpr bool ORDERED = decltype(ordered)::value;
        for (int first = 0; first < d->layers; first += kStepMaxBlocks) {
            a.blocks = d->layers - first < kStepMaxBlocks ? d->layers - first : kStepMaxBlocks;
            a.tickets = a.alive + 1 + 2 * (first / kStepMaxBlocks);
            a.exchange = base + kStepControlBytes + static_cast<size_t>(first) * a.at.bytes;
            a.x = first == 0 ? x : reinterpret_cast<const uint16_t*>(a.exchange - a.at.bytes + a.at.out);
            a.stats = first == 0 ? stats : nullptr;
            // (behind the last block of a launch that is not the last: where that block's consumers look for it)
            a.x_out = first + a.blocks == d->layers ? x_out : reinterpret_cast<uint16_t*>(a.exchange + static_cast<size_t>(a.blocks - 1) * a.at.bytes + a.at.out);
            for (int n = 0; n < a.blocks; ++n) {
                const ternaspmm_step_block& b = blocks[first + n];
                a.block[n] = StepBlock{static_cast<const uint32_t*>(b.wqkv), static_cast<const uint32_t*>(b.wo), static_cast<const uint32_t*>(b.w13),
                                       static_cast<const uint32_t*>(b.w2), b.ws_qkv, b.ws_o, b.ws_13, b.ws_down, b.attention_norm, b.attn_sub_norm, b.ffn_norm,
                                       b.ffn_sub_norm, b.cache_k, b.cache_v};
            }
            if constexpr (ORDERED) launch_step_ordered(a, st);
            else if (d->M == 1) terna_decode_step_kernel<1, false><<<dim3(groups), dim3(kStepThreads), 0, st>>>(a);
            else if (d->M == 2) terna_decode_step_kernel<2, false><<<dim3(groups), dim3(kStepThreads), 0, st>>>(a);
            else terna_decode_step_kernel<4, false><<<dim3(groups), dim3(kStepThreads), 0, st>>>(a);
        }
    };
    launches(std::false_type{});
    launches(std::true_type{});                  // (behind all of them: one that gave up left nothing for the next)
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) die("ternaspmm_decode_step", e, __LINE__);
    return 0;
}

}  // namespace

extern "C" {

long long ternaspmm_decode_step_bytes(const ternaspmm_step_desc* d)
{
    if (d == nullptr || !step_shape_ok(*d)) return -1;
    const long long count = ternaspmm_row_stats_count(d->dim);
    return kStepControlBytes + static_cast<long long>(d->layers) * exchange_of(*d).bytes + up(2ll * d->M * d->dim) + up(8ll * d->M * count) + up(4ll * d->M * d->head_dim);
}

int ternaspmm_decode_step(const ternaspmm_step_desc* d, const ternaspmm_step_block* blocks, const long long* tokens, const long long* pos,
                          const terna_bf16* embedding, const float* rope_table, void* scratch, terna_bf16* x_out, terna_stream stream)
{
    return enqueue_step(d, blocks, tokens, pos, embedding, rope_table, scratch, x_out, kStepGroups, kStepPatience, stream);
}

int ternaspmm_probe_decode_step(const ternaspmm_step_desc* d, const ternaspmm_step_block* blocks, const long long* tokens, const long long* pos,
                                const terna_bf16* embedding, const float* rope_table, void* scratch, terna_bf16* x_out, int workgroups, int polls, terna_stream stream)
{
    if (workgroups < 1 || workgroups > kStepGroups || polls < 1 || polls > kStepPatience) return -1;
    return enqueue_step(d, blocks, tokens, pos, embedding, rope_table, scratch, x_out, workgroups, polls, stream);
}

}  // extern "C"
