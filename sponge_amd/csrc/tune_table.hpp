// Default launch shapes of the fused step, by system size, from the shape
// sweep of sponge_amd/autotune.py (times per MD step of plain water boxes
// beside each row): the fastest candidate, or one within the ~1 % that two
// sweeps of the same shape differ by. A row applies to systems of up to
// max_atoms atoms; the last row to all larger ones. Regenerate with
// `python -m sponge_amd.autotune --table` (which takes the fastest).
// Soft-core handles take the rows of their size, and prune only with a radius
// below cutoff + skin.
//
// Columns: pair_waves (i-clusters per block of the force-only pair kernel),
// conv_split (-1: by plane size, one workgroup per plane up to 64 x 64; 0 /
// 1 / 2 forced: plane, lines, slab), conv_threads (per-plane workgroup),
// step_form (0 two streams,
// 1 serial), prune_div (inner list pruned every max(1, refresh / prune_div)
// fused steps; 0: no inner list), prune_margin (prune radius = cutoff +
// prune_margin * skin).
#pragma once

namespace snb {

struct TuneRow {
    int max_atoms;
    int pair_waves;
    int conv_split;
    int conv_threads;
    int step_form;
    int prune_div;
    float prune_margin;
};

// clang-format off
constexpr TuneRow kTuneTable[] = {
    {      3908, 2, -1, 256, 0, 1, 1.0f},  // 648 atoms, PME 20x20x20: 39.20 us/step
    {     47597, 8,  1, 256, 0, 1, 1.0f},  // 23570 atoms, PME 64x64x64: 63.70 us/step (kept: 5th, 1st 63.11)
    {0x7fffffff, 4, -1, 256, 0, 1, 1.0f},  // 96120 atoms, PME 108x108x108: 159.69 us/step
};
// clang-format on

inline const TuneRow& tune_row(int atoms) {
    constexpr int nrows = (int)(sizeof(kTuneTable) / sizeof(kTuneTable[0]));
    for (int r = 0; r < nrows; r++)
        if (atoms <= kTuneTable[r].max_atoms) return kTuneTable[r];
    return kTuneTable[nrows - 1];
}

}  // namespace snb
