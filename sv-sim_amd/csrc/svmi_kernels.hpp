// svmi_kernels.hpp -- host-side launchers of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "svmi_internal.hpp"

namespace svmi {

// Pauli sums (planned by plan_pauli, svmi_pauli.cpp).  A group holds the terms
// of one X mask: (H psi)[y] = sum_groups f(y) psi[y ^ xmask] with
// f(y) = sum_terms (-1)^{|y & zmask|} (cre + i cim).
struct PauliGroup {
    uint64_t xmask;      // physical, or tile-local for a pass's tile groups
    uint32_t begin, end; // terms
    uint32_t imag;       // some term has cim != 0
    uint32_t flat;       // one term with zmask 0: f is a constant
};
struct PauliTerm {
    uint64_t zmask;
    double cre, cim;     // coeff * i^{|x & z|} * (-1)^{|x & z|}
    uint32_t jsign;      // bit j: parity of zmask on register j's offset (PauliPass::col[j])
    uint32_t last;       // the last of the group's terms with this jsign (they are neighbours)
};
constexpr int kPauliTileQubits = 12;   // 2^12 amplitudes: 64 KiB of LDS, two workgroups per CU
constexpr int kPauliThreadBits = 9;    // tile-local bits of the 512 threads, the rest are registers
constexpr int kPauliThreads = 1 << kPauliThreadBits;
constexpr int kPauliRegs = 1 << (kPauliTileQubits - kPauliThreadBits);
constexpr int kPauliLow = 4;           // low qubits every tile keeps: 256-byte segments
constexpr int kMaxPauliPasses = 6;
// One pass over the state in tiles of the qubits pos[0..k): its groups
// [begin, tile_end) flip tile qubits only and read the tile in LDS -- those of
// [begin, flat_end) are flat and have consecutive terms -- and its groups
// [tile_end, end) read psi[y ^ xmask] from memory.
struct PauliPass {
    uint64_t extmask;    // qubits outside the tile
    uint64_t col[kPauliRegs];   // physical offset of register j
    uint32_t pos[kPauliTileQubits];
    uint32_t k;
    uint32_t begin, flat_end, tile_end, end;
};

// ---- batched execution (one launch per dependency level) ----
struct BatchStep {
    uint32_t kind;        // BSTEP_*
    uint32_t circuit;
    int32_t dep;          // previous step of the same circuit (an earlier level), -1 = none
    uint32_t sweep;       // FWD/ADJ: index into the sweep array
    uint64_t task_begin;  // first queue task of this step
    uint64_t n_tasks;
    uint64_t partial;     // PAULI: first E partial; ADJ: first gradient partial
    uint32_t init_zero;   // FWD: generate |0..0> instead of loading
    uint32_t pad;
};
enum : uint32_t { BSTEP_FWD = 0, BSTEP_PAULI = 1, BSTEP_ADJ = 2 };

struct BatchCircuit {
    c64* phi;             // state (forward result, then adjoint phi)
    c64* lam;             // H psi, then adjoint lambda
    uint32_t n;           // qubits of the device state
    uint32_t group_begin, flat_end, tile_end, group_end;   // Pauli groups, as a PauliPass has them
    uint32_t e_partial, n_e_partials;  // PAULI partials
    uint32_t slot_begin, n_slots;      // gradient accumulators (global numbering)
};

// Device tables of a program's sweeps.
struct SweepTables {
    const LayoutPhase* lphases;
    const uint64_t* lane_tab;
    const uint64_t* wave_tab;
    const DOp* ops;
    const c64* coef;
};

struct BatchArgs {
    const BatchStep* steps;
    const BatchCircuit* circuits;
    const SweepInfo* sweeps;
    const SweepIO* io;
    SweepTables t;
    const PauliGroup* groups;
    const PauliTerm* terms;
    double* e_partials;
    double* grad_partials;
};

constexpr uint32_t kPauliChunk = 1u << kPauliTileQubits;   // amplitudes per Pauli task of a batch

// One launch of a batch: the steps [step_begin, step_end) of one level,
// all of one kind and (sweeps) one tile size k; their tasks are
// [task_begin, task_begin + n_tasks).
struct BatchLaunch {
    uint32_t step_begin, step_end;
    uint32_t kind, k;
    uint32_t max_grad;      // ADJ: largest n_grad of the group's sweeps
    uint32_t init;          // FWD: first sweeps (tiles start as |0..0>)
    uint32_t max_xf;        // largest n_xf of the group's sweeps
    uint32_t max_dense;     // widest dense block of the group's sweeps
    uint32_t max_stage;     // largest SweepInfo::stage of the group's sweeps
    uint64_t task_begin, n_tasks;
};
// The lane and wave tables of a batch's n phases from their columns.
hipError_t launch_thread_tables(hipStream_t st, const ThreadCols* cols, uint64_t n, uint64_t* lane_tab,
                                uint64_t* wave_tab);
size_t batch_launch_smem(const BatchLaunch& L);   // without what the latency builds add
hipError_t launch_batch(hipStream_t st, const BatchArgs& a, const BatchLaunch& L);

hipError_t init_sweep_kernels();
hipError_t init_sample_kernels();   // after init_sweep_kernels
size_t sweep_smem_limit();
size_t sweep_smem_bytes(const SweepInfo& sw, int ns);
hipError_t launch_sweep(hipStream_t st, int ns, c64* s0, c64* s1, const SweepInfo& sw, const SweepIO* io /* device */,
                        const SweepTables& t, double* grad_partials);
hipError_t launch_standalone(hipStream_t st, c64* s, int n, const StandaloneOp& so, const c64* coef);
hipError_t launch_fill_basis(hipStream_t st, c64* s, uint64_t dim);
hipError_t launch_gather(hipStream_t st, const c64* s, uint64_t dim, const uint64_t* idx, uint64_t cnt, c64* out);
uint32_t random_state_grid(uint64_t dim);
hipError_t launch_random_state(hipStream_t st, c64* s, uint64_t dim, uint64_t seed, double* partials);
hipError_t launch_scale(hipStream_t st, c64* s, uint64_t dim, double f);
hipError_t launch_copy(hipStream_t st, c64* d, const c64* s, uint64_t dim);
hipError_t launch_block_totals(hipStream_t st, const c64* s, uint64_t nblocks, uint32_t nthr,
                               uint32_t chunk, double* totals);
hipError_t launch_sample(hipStream_t st, const c64* s, uint32_t nthr, uint32_t chunk,
                         const uint64_t* jobs, uint32_t njobs, const double* offsets,
                         const double* draws, uint64_t* out);
// One pass of a Pauli sum: lam (optional) = or, with `accumulate`, += the pass's
// groups applied to psi; copy (optional) = psi; pauli_grid partials of
// Re <psi | the pass's part of H psi>.
uint32_t pauli_grid(uint64_t dim, const PauliPass& pass);
hipError_t launch_pauli(hipStream_t st, const c64* psi, c64* lam, uint64_t dim, const PauliPass& pass,
                        bool accumulate, const PauliGroup* groups, const PauliTerm* terms, double* partials,
                        c64* copy = nullptr);
// dst[seg.dst] = sum of src[seg.src, seg.src + seg.len), per segment, in a
// fixed order (one workgroup per segment).
struct SumSegment {
    uint64_t src, len, dst;
};
hipError_t launch_sum_segments(hipStream_t st, const double* src, const SumSegment* segs, uint64_t nseg,
                               double* dst);
// dst[r] = sum of src[r * len, (r + 1) * len), r < rows, same order.
hipError_t launch_sum_rows(hipStream_t st, const double* src, uint32_t rows, uint64_t len, double* dst);

// One mid-circuit measurement on the device.
struct MeasureResult {
    double prob;         // P(1)
    int32_t outcome;     // draw < P(1)
    int32_t pad;
};
// P(1) of qubit q over the 2^n-amplitude state s, the outcome for `draw`,
// and the collapse factors written into collapse[0] (bit 0) and collapse[1]
// (bit 1): (0, 1/sqrt(P)) for outcome 1, (1/sqrt(1-P), 0) for outcome 0.
// dm_n > 0: s is a density matrix of dm_n qubits (n = 2 dm_n, index row |
// col << dm_n), P(1) sums |Re rho[i, i]| over the rows with bit q set and the
// factors are 1/P and 1/(1-P).  partials: measure_partials(n) doubles of
// scratch.
uint32_t measure_partials(int n);
hipError_t launch_measure(hipStream_t st, const c64* s, int n, uint32_t q, double draw, double* partials,
                          c64* collapse, MeasureResult* res, int dm_n = 0);

}  // namespace svmi
