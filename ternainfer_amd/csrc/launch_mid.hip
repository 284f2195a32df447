// Launcher of the kernel for 17 rows .. a few hundred on the P2 layout (mid_kernel.h): which calls it takes, which tile.
#include "launchers.h"
#include "host_util.h"
#include "mid_kernel.h"

namespace terna {
namespace {

struct MidTile {
    int rt, fb;                  // 16-row tiles, 16-feature bands of a workgroup
    int waves;
};

// A CU's load time is what a launch takes beyond its fixed part, so the tile is the one with the least of
// (workgroups per CU, rounded up) x (bytes of one workgroup per 4 columns of K: 64 rt sz activations + 16 fb weights).
// One workgroup per CU: as many waves as K has chunks for, evenly (K = 6912, 27 chunks: fourteen waves take them in two rounds, twelve in three: 32 rows
// 5.6 -> 5.0 us a launch); more of them: four waves each, whose small LDS shares
// let four or five workgroups overlap on a CU.  How many a CU has is counted with feature tiles in eights, as they lie on the XCDs (N = 128: a workgroup per
// CU by their number, four on the CUs that have any; sixteen waves' LDS each then run one after the other: 1500 rows, K = 6912, int8 15.7 -> 12.2 us,
// bf16 26.1 -> 21.2; 1000 rows, N = 256, K = 4096, bf16 12.4 -> 11.2; 1224 launches of N = 64 - 1536, geometric mean 0.978).  The tile is chosen by their number: counted
// in eights for that too, the mean is 0.94, but 32-row tiles of short K come out up to 1.3 times as slow (850 rows, N = 704, K = 64: 4.6 -> 5.7 us).
MidTile choose_tile(int M, int N, int K, int sz)
{
    const int chunks = (K / 64 + 3) / 4;
    constexpr int kTiles[3][2] = {{1, 2}, {1, 4}, {2, 4}};
    MidTile best{};
    long best_cost = 0;
    for (const auto& t : kTiles) {
        const long tiles = static_cast<long>((M + 16 * t[0] - 1) / (16 * t[0])) * ((N / 16 + t[1] - 1) / t[1]);
        const long cost = (tiles + 255) / 256 * (64 * t[0] * sz + 16 * t[1]);
        if (best.rt == 0 || cost < best_cost) {
            best = MidTile{t[0], t[1], 0};
            best_cost = cost;
        }
    }
    const bool shared = static_cast<long>((M + 16 * best.rt - 1) / (16 * best.rt)) * ((N / 16 + 8 * best.fb - 1) / (8 * best.fb) * 8) > 256;
    const int fit = 160 * 1024 / (16 * best.rt * 256 * sz);                // LDS of a workgroup
    const int most = shared ? 4 : (fit < kMidMaxWaves ? fit : kMidMaxWaves);
    const int rounds = (chunks + most - 1) / most;
    best.waves = shared ? (chunks < most ? chunks : most) : (chunks + rounds - 1) / rounds;
    return best;
}

template <typename Act, int RT, int FB, int EPI = PACKED_STORE>
void launch_mid_as(const Act* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, int waves,
                   const PackedExtra<EPI>* extra, hipStream_t st)
{
    using S = MidShape<Act, RT, FB>;
    const int row_tiles = (M + 16 * RT - 1) / (16 * RT), feature_tiles = (N / 16 + FB - 1) / FB;
    const unsigned grid = static_cast<unsigned>((feature_tiles + 7) / 8 * 8 * row_tiles);
    const dim3 block(waves * 64);
    const int lds = waves * S::kWaveBytes;
    if constexpr (EPI == PACKED_STORE) {
        if (extra != nullptr) {
            auto kernel = terna_mid_kernel<Act, RT, FB, true>;
            if (lds > kPlainLds) allow_dynamic_lds(kernel, 160 * 1024, "hipFuncSetAttribute(mid)", __LINE__);
            launch(kernel, dim3(grid + 1), block, lds, st, x, packed, out, M, N, K, row_tiles, waves, ep, *extra, 0);
            return;
        }
    }
    auto kernel = terna_mid_kernel<Act, RT, FB, false, EPI>;
    if (lds > kPlainLds) allow_dynamic_lds(kernel, 160 * 1024, "hipFuncSetAttribute(mid)", __LINE__);
    launch(kernel, dim3(grid), block, lds, st, x, packed, out, M, N, K, row_tiles, waves, ep, extra != nullptr ? *extra : PackedExtra<EPI>{}, 0);
}

template <typename Act, int EPI>
void launch_mid_tile(const Act* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, hipStream_t st,
                     const PackedExtra<EPI>* extra)
{
    const MidTile t = choose_tile(M, N, K, sizeof(Act));
    if (t.rt == 2) launch_mid_as<Act, 2, 4, EPI>(x, packed, out, ep, M, N, K, t.waves, extra, st);
    else if (t.fb == 4) launch_mid_as<Act, 1, 4, EPI>(x, packed, out, ep, M, N, K, t.waves, extra, st);
    else launch_mid_as<Act, 1, 2, EPI>(x, packed, out, ep, M, N, K, t.waves, extra, st);
}

// The quantising form: 16 rows a workgroup; the bands of a workgroup, 0 where it does not pay: up to one workgroup a CU, two where K is short,
// feature tiles counted in eights as they lie on the XCDs.  us of the device, two launches / one: K = 2560, 64 x 2560 6.3 / 6.4, 64 x 3840
// 6.4 / 6.6, 16 x 2560 5.2 / 5.8, 16 x 13824 7.1 / 6.7, two workgroups a CU 128 x 2560 7.1 / 9.2; 32 rows of K = 4096, N = 4096 6.6 / 7.4; two
// workgroups a CU, K = 1024, 512 x 1024 6.9 / 6.0, K = 2048 8.0 / 8.0.  The host's share of a module call is 10.6 / 6.9.
int quant_tile_bands(int M, int N, int K)
{
    const long row_tiles = (M + 15) / 16, bands = N / 16;
    const int chunks = (K / 64 + 3) / 4;
    if (chunks > kMidMaxWaves) return 0;
    return row_tiles * ((bands + 15) / 16 * 8) <= 256 ? 2 : row_tiles * ((bands + 31) / 32 * 8) <= (chunks <= 8 ? 512 : 256) ? 4 : 0;
}

template <int FB, bool GUARD>
void launch_mid_quant_as(const uint16_t* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, hipStream_t st,
                         const RepackGuard& guard)
{
    const int feature_tiles = (N / 16 + FB - 1) / FB, row_tiles = (M + 15) / 16, waves = (K / 64 + 3) / 4;
    auto kernel = terna_mid_kernel<int8_t, 1, FB, GUARD, PACKED_STORE, true>;
    const int lds = MidQuantShape::bytes(waves);
    if (lds > kPlainLds) allow_dynamic_lds(kernel, 160 * 1024, "hipFuncSetAttribute(mid quant)", __LINE__);
    launch(kernel, dim3((feature_tiles + 7) / 8 * 8 * row_tiles + (GUARD ? 1 : 0)), dim3(waves * 64), lds, st,
           reinterpret_cast<const int8_t*>(x), packed, out, M, N, K, row_tiles, waves, ep, guard, quant_mode());
}

}  // namespace

bool mid_quant_takes(const uint16_t* x, const uint16_t* out, int M, int N, int K)
{
    return (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0 &&
           (static_cast<uint64_t>(M) + 16) * K * 2 < (1ull << 31) && static_cast<uint64_t>(N) * K / 4 < (1ull << 31) && quant_tile_bands(M, N, K) != 0;
}
void launch_mid_quant(const uint16_t* x, const uint32_t* packed, uint16_t* out, const uint16_t* ws, int ws_num, int M, int N, int K, hipStream_t st,
                      const RepackGuard* guard)
{
    const Epilogue ep{nullptr, ws, nullptr, ws_num, M <= 64 ? EP_I8_DECODE : EP_I8_PREFILL};
    if (quant_tile_bands(M, N, K) == 2) {
        if (guard != nullptr) launch_mid_quant_as<2, true>(x, packed, out, ep, M, N, K, st, *guard);
        else launch_mid_quant_as<2, false>(x, packed, out, ep, M, N, K, st, RepackGuard{});
    } else {
        if (guard != nullptr) launch_mid_quant_as<4, true>(x, packed, out, ep, M, N, K, st, *guard);
        else launch_mid_quant_as<4, false>(x, packed, out, ep, M, N, K, st, RepackGuard{});
    }
}

// Up to 16 rows the small-M kernels are faster (16 rows, us, small-M / this kernel, int8; bf16: O 2.9 / 3.3; 3.3 / 3.7, QKV 3.1 / 3.3; 3.5 / 3.8, down
// 4.1 / 4.7; 5.5 / 6.1; wide and shallow matrices are level or the other way round: gate+up 4.7 / 4.5; 5.7 / 5.4).  Upwards the MFMA-tiled kernel, whose activations are shared by 128
// features, is ahead where the tiles of 32 x 64 are more than two a CU -- counted as they lie on the XCDs, in eights of feature
// tiles (N = 256 leaves half of the XCDs without one).  Measured, us, MFMA-tiled / this kernel, int8; bf16: QKV M = 250 (480 tiles) 7.7 / 7.0;
// 10.9 / 9.7, M = 280 (576) 7.7 / 8.2; 10.9 / 12.0; gate+up M = 64 (432) 8.1 / 7.2; 10.9 / 9.8, M = 70 (648) 7.8 / 8.4; 11.2 / 12.1; down M = 350
// (440) 13.0 / 11.4; 22.0 / 18.2, M = 430 (560) 13.5 / 14.3; 22.1 / 27.2; N = 1024 = K, M = 1000 (512) 5.2 / 4.7; 6.4 / 5.8, M = 1200 (608) 5.4 / 5.6;
// 6.6 / 6.9; N = 256, M = 1000 (256) 6.9 / 4.8; 11.3 / 8.2, M = 4000 (1000) 7.6 / 13.8; 11.8 / 24.0; N = 704, K = 320, M = 1500 (752) 4.4 / 5.3; 4.6 / 6.7.
// Few rows of a wide matrix stay here up to four tiles a CU: a tile of the MFMA-tiled kernel has 64 rows, half of them and more for nothing, and up to 32 rows the
// small-M kernel takes what this one leaves.  The other kernel / this one: 17 rows, N = 65536 (1024 tiles) K = 1024 9.1 / 7.7; 11.5 / 11.1, K = 4096 20.7 / 15.4; 30.5 / 23.9;
// 32 rows, N = 40960 K = 4096 15.8 / 12.7; 22.9 / 17.6; 33 - 48 rows, N = 20480 (640) K = 1024 6.4 / 5.0; 7.0 / 6.1, K = 4096 10.5 / 9.2; 15.1 / 14.1, N = 32768 (1024)
// 11.9 / 12.2; 16.3 / 19.3; 64 rows, N = 20480 10.8 / 11.5; 15.4 / 16.9.  Where K is short the others are ahead: 32 rows, N = 49152 K = 64 4.4 / 6.7;
// 5.4 / 6.1, K = 320 5.4 / 6.4; 6.8 / 6.8, K = 512 6.2 / 6.5; 7.1 / 6.9; 40 rows, N = 20480, K = 320 5.4 / 4.7; 4.9 / 5.3.
bool mid_kernel_takes(const void* x, int M, int N, int K, size_t act_bytes)
{
    const long tiles = static_cast<long>((M + 31) / 32) * ((N / 16 + 31) / 32 * 8);
    const long most = M > 48 ? 512 : M > 32 ? (K >= 512 ? 640 : 512) : K * act_bytes >= 1024 ? 1024 : 512;
    return M > 16 && tiles <= most && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
           static_cast<uint64_t>(M) * K * act_bytes < (1ull << 31) && static_cast<uint64_t>(N) * K / 4 < (1ull << 31);
}

template <typename Act>
void launch_mid(const Act* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, hipStream_t st,
                const RepackGuard* guard)
{
    launch_mid_tile<Act, PACKED_STORE>(x, packed, out, ep, M, N, K, st, guard);
}

void launch_mid_gate(const int8_t* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, hipStream_t st)
{
    launch_mid_tile<int8_t, PACKED_GATE>(x, packed, out, ep, M, N, K, st, nullptr);
}
void launch_mid_rope(const int8_t* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, const RopeStore& rope, hipStream_t st)
{
    launch_mid_tile<int8_t, PACKED_ROPE>(x, packed, out, ep, M, N, K, st, &rope);
}
void launch_mid_residual(const int8_t* x, const uint32_t* packed, uint16_t* out, const Epilogue& ep, int M, int N, int K, const ResidualRows& stream,
                         hipStream_t st)
{
    launch_mid_tile<int8_t, PACKED_RESIDUAL>(x, packed, out, ep, M, N, K, st, &stream);
}

// Up to 2048 rows (a launch of 4000 has no spare moments: 11361 against 11380 us a prompt), and up to half of every L2 (4 MiB an XCD).
NextWeights next_weights(const void* packed, int N, int K, bool gate, int M)
{
    NextWeights next{};
    const long bytes = static_cast<long>(N) * K / 4;
    if (packed == nullptr || N < 64 || K < 64 || (N & 63) || (K & 63) || M > 2048 || bytes > (16l << 20)) return next;
    int bands;                                           // of one workgroup of the launch that will run
    if (M <= 16) bands = gate || N / 16 > 256 ? 4 : 1;
    else if (mid_kernel_takes(nullptr, M, N, K, 1)) bands = choose_tile(M, N, K, 1).fb;
    else bands = plan_prefill_packed<int8_t>(nullptr, M, N, K, nullptr, 0).bn / 16;
    next.base = static_cast<const uint8_t*>(packed);
    next.lines = static_cast<uint32_t>(bytes / 128);
    next.tile_lines = static_cast<uint32_t>(bands * K / 32);
    next.workgroups = static_cast<int>(next.lines / 256 + 7) / 8 * 8;
    if (next.workgroups > 192) next.workgroups = 192;
    return next;
}

template void launch_mid<int8_t>(const int8_t*, const uint32_t*, uint16_t*, const Epilogue&, int, int, int, hipStream_t, const RepackGuard*);
template void launch_mid<uint16_t>(const uint16_t*, const uint32_t*, uint16_t*, const Epilogue&, int, int, int, hipStream_t, const RepackGuard*);

}  // namespace terna
