// svmi_tuning.hpp -- planning of batched circuits per qubit count.
// By svmi/autotune.py (AMD Radeon Graphics (gfx950), n = 4..22, 2026-12-02).
// From 13 on the tiles were set by hand for the sweeps that hold their tile in
// registers, on batches of mixed sizes: what the tuner finds
// for batches of one size (its candidates differ by less than its runs there)
// runs 96 circuits of 10-20 qubits in 12.9 ms instead of 12.2, 32 of 12-18 in
// 5.3 instead of 5.0.  So compare its output on mixed batches before it takes
// this file's place.  From kBatchLargeAdj qubits on adj_tile is not read.
#pragma once

#include <stdint.h>

namespace svmi {

struct BatchTuning {
    uint8_t n;          // qubits
    uint8_t fwd_tile;   // forward sweep tile qubits
    uint8_t adj_tile;   // backward sweep tile qubits
    uint8_t op_cost;    // fusion op cost
};

constexpr const char* kBatchTuningSource = "AMD Radeon Graphics (gfx950), n = 4..22 2026-12-02; tiles by hand from 13";
constexpr BatchTuning kBatchTuning[] = {
    {4, 12, 11, 1}, {5, 12, 11, 0}, {6, 12, 11, 0}, {7, 12, 11, 1}, {8, 12, 11, 0}, {9, 9, 11, 0},
    {10, 12, 10, 0}, {11, 12, 11, 0}, {12, 12, 11, 0}, {13, 13, 11, 0}, {14, 13, 11, 1}, {15, 13, 11, 1},
    {16, 13, 11, 0}, {17, 13, 11, 0}, {18, 13, 11, 0}, {19, 13, 11, 2}, {20, 13, 11, 2}, {21, 13, 11, 2},
    {22, 13, 11, 2}, {23, 13, 11, 2}, {24, 13, 11, 2}, {25, 13, 11, 2}, {26, 13, 11, 2}, {27, 13, 11, 2},
    {28, 13, 11, 2}, {29, 13, 11, 2}, {30, 13, 11, 2},
};

// Entry for an n-qubit circuit (the nearest size in the table).
inline const BatchTuning& batch_tuning(int n)
{
    constexpr int count = int(sizeof(kBatchTuning) / sizeof(kBatchTuning[0]));
    int best = 0;
    for (int i = 1; i < count; i++) {
        const int d = n - int(kBatchTuning[i].n), db = n - int(kBatchTuning[best].n);
        if ((d < 0 ? -d : d) < (db < 0 ? -db : db)) best = i;
    }
    return kBatchTuning[best];
}

}  // namespace svmi
