// The rules of ternainfer_amd/csrc/step_layout.h, over small and large shapes: built with g++ and run by test_step_layout.py.
#include <cstdio>
#include <set>
#include <tuple>
#include <vector>

#include "../ternainfer_amd/csrc/step_layout.h"

using namespace terna;

static int failures = 0;
#define CHECK(cond, ...)                                   \
    do {                                                   \
        if (!(cond) && ++failures < 20) {                  \
            std::printf("%s:%d: %s: ", __FILE__, __LINE__, #cond); \
            std::printf(__VA_ARGS__);                      \
            std::printf("\n");                             \
        }                                                  \
    } while (0)

struct Shape {
    int M, dim, ffn, H, KV, SP;
};

// What a workgroup of the resident launch does (the conditions in its prologue).
static bool resident_does(const Shape& s, int kind, int w)
{
    switch (kind) {
        case STEP_QKV: return w < (s.H + 2 * s.KV) * kStepHeadDim / 16;
        case STEP_ATTENTION: return step_unit(w, s.M == 1 ? s.KV * s.SP : s.M * s.KV, s.H / s.KV * (s.M == 1 ? 1 : 2)).group >= 0;
        case STEP_GATE: return 4 * w < s.ffn >> 3;
        case STEP_QUANT: return s.M > 1 && kStepGroups - 1 - w < 4 * s.M;
        default: return w < s.dim >> 4;
    }
}

// Every unit of the resident launch is a ticket, once; the tickets of a phase stand together, behind all it depends on.
static void check_tickets(const Shape& s)
{
    std::set<std::tuple<int, int, int>> seen;
    int previous = -1, start = 0, t = 0;
    for (;; ++t) {
        const StepTicket k = step_ticket(t, s.M, s.dim, s.ffn, s.H, s.KV, s.SP);
        if (k.block >= 2) break;
        const int phase = k.block * STEP_KINDS + k.kind;
        CHECK(phase >= previous, "ticket %d: phase %d behind %d", t, phase, previous);
        if (phase != previous) start = t;
        previous = phase;
        CHECK(k.before == start, "ticket %d waits for %d, its phase starts at %d", t, k.before, start);
        CHECK(k.w >= 0 && k.w < kStepGroups, "ticket %d: workgroup %d", t, k.w);
        CHECK(seen.insert({k.block, k.kind, k.w}).second, "ticket %d: done twice", t);
        // (units that only fill a round of eight groups are tickets too, with nothing to do)
        CHECK(k.kind == STEP_ATTENTION || resident_does(s, k.kind, k.w), "ticket %d: kind %d workgroup %d has none", t, k.kind, k.w);
    }
    for (int block = 0; block < 2; ++block)
        for (int kind = 0; kind < STEP_KINDS; ++kind)
            for (int w = 0; w < kStepGroups; ++w)
                CHECK(!resident_does(s, kind, w) || seen.count({block, kind, w}), "block %d kind %d workgroup %d is no ticket", block, kind, w);
}

// What a wave requests of a matrix lies in it, or wholly past its last byte, where the buffer's range check -- an unsigned
// comparison with the lane's offset -- returns zeros; and every tile of a band is requested by the wave whose run it is in.
static void check_weight_requests(int bands, int K, int per_workgroup, int chunks, int singles)
{
    const int ktiles = K / 64, run = 4 * chunks + singles, range = bands * ktiles * 256;
    for (int band = 0; band < (bands + per_workgroup - 1) / per_workgroup * per_workgroup; ++band) {
        std::vector<bool> read(static_cast<size_t>(ktiles) * 256);
        auto request = [&](long long at, int size) {
            CHECK(at >= 0 && at < 0x7fffffff && (at + size <= range || at >= range), "band %d of %d, K %d: %d bytes at %lld of %d", band, bands, K, size, at, range);
            for (long long b = at; b < at + size; ++b)
                if (b >= static_cast<long long>(band) * ktiles * 256 && b < static_cast<long long>(band + 1) * ktiles * 256) read[b - static_cast<long long>(band) * ktiles * 256] = true;
        };
        for (int wave = 0; wave < kStepWaves; ++wave)
            for (int lane = 0; lane < 64; ++lane) {
                for (int c = 0; c < chunks; ++c) request(step_weight_offset(band, ktiles, wave * run, lane * 16) + 1024 * c, 16);
                for (int s = 0; s < singles; ++s) request(step_weight_offset(band, ktiles, wave * run, lane * 4) + 256 * (4 * chunks + s), 4);
            }
        for (size_t b = 0; b < read.size(); ++b) CHECK(band >= bands || read[b], "band %d, K %d: byte %zu is requested by no wave", band, K, b);
    }
}

// The lines of the keys that the workgroups of a unit's group bring into the L2 of their XCD: those the group reads, each once --
// with several sequences by those of its workgroups that have a band of QKV, if any has.
static void check_cache_lines(const Shape& s, int slots_seen)
{
    const int groups = s.M == 1 ? s.KV * s.SP : s.M * s.KV, per = s.H / s.KV * (s.M == 1 ? 1 : 2), splits = s.M == 1 ? s.SP : 1;
    const int bytes = 2 * kStepHeadDim * slots_seen, lines = bytes / 128;
    std::vector<std::vector<int>> fetched(groups, std::vector<int>(lines));
    std::vector<int> xcd(groups, -1), fetching(groups);
    const int bands = (s.H + 2 * s.KV) * kStepHeadDim / 16;
    for (int w = 0; w < kStepGroups; ++w) {
        const StepUnit u = step_unit(w, groups, per);
        if (u.group < 0) continue;
        CHECK(xcd[u.group] < 0 || xcd[u.group] == w % 8, "group %d sits on two XCDs", u.group);
        xcd[u.group] = w % 8;
        const int split = s.M == 1 ? u.group % s.SP : 0, past = s.M == 1 ? 0 : step_unit_past(u, per, bands);
        CHECK(s.M == 1 || (u.head >= past) == resident_does(s, STEP_QKV, w), "workgroup %d, %d of its group past %d bands", w, past, bands);
        if (u.head < past) continue;
        ++fetching[u.group];
        for (int wave = 0; wave < kStepWaves; ++wave)
            for (int share = u.head - past + (per - past) * wave; step_cache_share(share, split, splits, bytes); share += (per - past) * kStepWaves)
                for (int lane = 0; lane < 64; ++lane) {
                    const int at = step_cache_line(share, lane, split, splits);
                    CHECK(at >= 0 && at % 128 == 0, "byte %d", at);
                    if (at >= bytes) continue;                    // (nothing is read)
                    CHECK(at / (16 * 2 * kStepHeadDim) % splits == split, "split %d of %d fetches byte %d of another", split, splits, at);
                    ++fetched[u.group][at / 128];
                }
    }
    for (int g = 0; g < groups; ++g)
        for (int l = 0; l < lines; ++l) {
            const int split = s.M == 1 ? g % s.SP : 0, own = fetching[g] > 0 && l * 128 / (16 * 2 * kStepHeadDim) % splits == split;
            CHECK(fetched[g][l] == own, "group %d, %d slots: line %d is fetched %d times", g, slots_seen, l, fetched[g][l]);
        }
}

int main()
{
    std::vector<Shape> shapes;
    for (int M = 1; M <= 4; ++M)
        for (int SP : {1, 2, 4, 8})
            for (const auto& [H, KV, dim, ffn] : std::vector<std::tuple<int, int, int, int>>{
                     {20, 5, 2560, 6912}, {20, 5, 2560, 7168}, {2, 1, 256, 192}, {9, 3, 1152, 1088}, {5, 5, 640, 64}, {1, 1, 64, 64}, {16, 4, 2048, 5632}, {20, 1, 192, 6976}}) {
                const Shape s{M, dim, ffn, H, KV, SP};
                if ((M == 1) == (SP > 1) && step_unit_groups(M == 1 ? KV * SP : M * KV, H / KV * (M == 1 ? 1 : 2)) <= kStepGroups) shapes.push_back(s);
            }
    for (const Shape& s : shapes) {
        check_tickets(s);
        for (int slots_seen : {1, 15, 16, 17, 100, 254, 1024}) check_cache_lines(s, slots_seen);
    }
    for (int ktiles : {1, 2, 3, 9, 10, 11, 30, 39, kStepTiles})
        for (int bands : {4, 12, 160}) {
            check_weight_requests(bands, 64 * ktiles, 1, 2, 2);
            check_weight_requests(bands, 64 * ktiles, 4, 2, 2);
        }
    for (int ktiles : {1, 27, 28, 29, 85, 108, kStepWideTiles})
        for (int bands : {4, 160}) check_weight_requests(bands, 64 * ktiles, 1, 7, 0);
    if (failures == 0) std::printf("step layout ok: %zu shapes\n", shapes.size());
    return failures != 0;
}
