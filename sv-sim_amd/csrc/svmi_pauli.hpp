// svmi_pauli.hpp -- grouping and tiling of Pauli sums (host only).
#pragma once

#include <vector>

#include "../../include/svmi.h"
#include "svmi_kernels.hpp"

namespace svmi {

struct PauliPlan {
    std::vector<PauliGroup> groups;   // in pass order
    std::vector<PauliTerm> terms;
    std::vector<PauliPass> passes;    // the first covers every amplitude of lam; at least one
};

// Plan for a state of n qubits with tiles of up to tile_qubits (<= kPauliTileQubits)
// and up to max_passes passes, the first one's tiles the lowest qubits; lam:
// H psi is written, not only summed.
void plan_pauli(const svmi_pauli_term* terms, size_t n_terms, int n, int tile_qubits, bool lam, int max_passes,
                PauliPlan& plan);

// The same with the tiles and passes that run a state of n qubits fastest.
void plan_pauli_state(const svmi_pauli_term* terms, size_t n_terms, int n, bool lam, PauliPlan& plan);

}  // namespace svmi
