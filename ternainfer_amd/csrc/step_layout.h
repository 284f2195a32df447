// Who does what in a decode step in one launch (step_kernel.h): integer rules alone, so that they can be checked without a GPU.
#pragma once

#if defined(__HIP__)
#define TERNA_STEP_FUNCTION __host__ __device__ inline
#else
#define TERNA_STEP_FUNCTION inline
#endif

namespace terna {

constexpr int kStepWaves = 4, kStepThreads = 64 * kStepWaves, kStepGroups = 256;
constexpr int kStepHeadDim = 128;
constexpr int kStepWideTiles = 112;              // tiles of the down projection's K: ffn <= 7168
constexpr int kStepTiles = 40;                   // tiles of the other linears' K: <= 2560

// Byte of a P2 matrix where a lane's part of a wave's run begins: tile `first` and on of a band, 256 bytes a tile.
TERNA_STEP_FUNCTION int step_weight_offset(int band, int ktiles, int first, int lane_bytes) { return (band * ktiles + first) * 256 + lane_bytes; }

// Attention units over the workgroups, from the last one downwards: the H / KV heads of a kv group read the same keys and values
// and sit on one XCD (workgroups go to the eight of them round robin).  A group is a (sequence, kv head), or (one sequence) a
// (kv head, split); per: its workgroups.  group < 0: no unit.
struct StepUnit {
    int group, head;                             // head within the group (several sequences: 2 head + half)
};
TERNA_STEP_FUNCTION int step_unit_groups(int groups, int per) { return 8 * per * ((groups + 7) / 8); }      // workgroups they take
TERNA_STEP_FUNCTION StepUnit step_unit(int w, int groups, int per)
{
    const int u = kStepGroups - 1 - w;
    const int q = u >> 3, group = 8 * (q / per) + (u & 7);
    return {u < step_unit_groups(groups, per) && group < groups ? group : -1, q % per};
}

// Workgroups of a group that stand past the bands of QKV: its first ones.
TERNA_STEP_FUNCTION int step_unit_past(const StepUnit& unit, int per, int bands)
{
    const int q = (kStepGroups - bands - (unit.group & 7) + 7) >> 3;      // those with u = 8 q' + (group & 7) < kStepGroups - bands
    const int past = q - per * (unit.group >> 3);
    return past < 0 ? 0 : past > per ? per : past;
}

// Byte of a kv head's keys (or values) whose line of 128 a lane brings into the L2 of its XCD: of the split it reads itself -- tiles of 16
// slots, split, split + splits, ... -- two tiles a share, shares dealt out over the workgroups of the group, which sit on one XCD.
// step_cache_share: whether a share has a line within the prefix.
TERNA_STEP_FUNCTION int step_cache_line(int share, int lane, int split, int splits)
{
    return (((2 * share + (lane >> 5)) * splits + split) * 16 + (lane & 31) / 2) * kStepHeadDim * 2 + (lane & 1) * 128;
}
TERNA_STEP_FUNCTION bool step_cache_share(int share, int split, int splits, int bytes) { return step_cache_line(share, 0, split, splits) < bytes; }

// The step's units of work in the order of their dependences: those of a phase, then those of the next, block by block.  A
// workgroup of the ORDERED launch takes one after the other from a counter; a unit may start once as many are done as stand in front of
// its phase (a later one cannot be among them).
enum StepKind { STEP_QKV, STEP_ATTENTION, STEP_OUT, STEP_GATE, STEP_QUANT, STEP_DOWN, STEP_KINDS };
struct StepTicket {
    int block, kind, w, before;                  // w: the workgroup of the other launch that does this unit; before: units in front of the phase
};
TERNA_STEP_FUNCTION StepTicket step_ticket(int ticket, int M, int dim, int ffn, int H, int KV, int SP)
{
    const int bands = (H + 2 * KV) * kStepHeadDim / 16, units = step_unit_groups(M == 1 ? KV * SP : M * KV, H / KV * (M == 1 ? 1 : 2));
    const int count[STEP_KINDS] = {bands, units, dim >> 4, ((ffn >> 3) + 3) / 4, M == 1 ? 0 : 4 * M, dim >> 4};
    int all = 0;
    for (int k = 0; k < STEP_KINDS; ++k) all += count[k];
    StepTicket t{ticket / all, 0, ticket % all, ticket / all * all};
    while (t.w >= count[t.kind]) t.w -= count[t.kind], t.before += count[t.kind], ++t.kind;
    if (t.kind == STEP_ATTENTION || t.kind == STEP_QUANT) t.w = kStepGroups - 1 - t.w;       // these go from the last workgroup downwards
    return t;
}

}  // namespace terna
