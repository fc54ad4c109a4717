// svmi_kernels.hip -- CDNA4 (gfx950) kernels of the state-vector engine.
//
// k_sweep1 / k_sweep2: one tiled sweep (the hot kernels).  One workgroup per
//   tile of 2^k amplitudes (per state), 16 amplitudes per thread in registers;
//   each phase runs its ops on them and the tile changes hands through LDS in
//   between.  Loads and stores are 16 bytes per lane and the low c physical
//   qubits of every tile are contiguous, so each group of 2^c lanes reads one
//   2^c*16-byte segment.  k_sweep2 runs the adjoint sweep over (phi, lambda)
//   and accumulates gradient partial sums per tile.
// Standalone ops (5-qubit dense, per-op mode), sampling, Pauli sums and
//   state fills are simple grid-stride kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "svmi_exec.hpp"
#include "svmi_kernels.hpp"

namespace svmi {

// ------------------------------------------------------------------ sweeps

// v of a lane moved by one DPP pattern (both halves of the double from the
// same source lane); lanes without a source, or outside row_mask, get 0.
template <int kCtrl, int kRowMask>
__device__ __attribute__((always_inline)) inline double dpp_move(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), kCtrl, kRowMask, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), kCtrl, kRowMask, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Sum of v over the 64 lanes of a wave, left in lane 63: an inclusive scan
// inside each 16-lane row (row_shr 1, 2, 4, 8), then row 0's total into row 1
// and row 2's into row 3 (row_bcast:15), then rows 0+1 into rows 2-3
// (row_bcast:31).  A fixed order, so the sum is the same on every run.
__device__ __attribute__((always_inline)) inline double wave_sum_lane63(double v)
{
    v += dpp_move<0x111, 0xf>(v);
    v += dpp_move<0x112, 0xf>(v);
    v += dpp_move<0x114, 0xf>(v);
    v += dpp_move<0x118, 0xf>(v);
    v += dpp_move<0x142, 0xa>(v);
    v += dpp_move<0x143, 0xc>(v);
    return v;
}

// The tile's phase factors (one per factor slot of the sweep) into LDS; the
// caller's next barrier publishes them.
__device__ __attribute__((always_inline)) inline void
tile_factors(c64* xf, const SweepInfo& sw, const DOp* __restrict__ ops, const c64* __restrict__ coef,
             uint64_t base, uint32_t tid)
{
    if (sw.n_xf == 0) return;
    // the sweep's lane tables, then the tile's factors
    const uint32_t nlt = 16u * sw.n_lt, lt0 = sw.n_xf - nlt;
    for (uint32_t i = tid; i < nlt; i += blockDim.x) xf[lt0 + i] = coef[sw.lt_coef + i];
    const uint64_t x = ext_index(sw, base);
    for (uint32_t o = sw.op_begin + tid; o < sw.op_end; o += blockDim.x) {
        const DOpHdr h = ops[o].h;
        if (has_tile_factor(h)) xf[h.grad] = tile_factor(h, coef, base, x);
    }
}

// LDS of a tile: exchange area (8 bytes per amplitude of every state; SweepInfo::whole
// adds as much) | phase factors | gradient accumulators.
size_t sweep_smem_bytes(const SweepInfo& sw, int ns)
{
    const size_t nwaves = (size_t(sweep_threads(sw.k, ns)) + 63) / 64;
    return (size_t(8) << sw.k) * ns + size_t(16) * sw.n_xf + size_t(8) * sw.n_grad * nwaves;
}

// The program's read-only tables, as restrict arguments of the kernels: from a
// struct of pointers the op records and coefficients would be read with
// vector loads instead of through the scalar cache.
#define SVMI_TABLES                                                                                 \
    const LayoutPhase *__restrict__ lph, const uint64_t *__restrict__ ltab,                         \
        const uint64_t *__restrict__ wtab, const DOp *__restrict__ ops, const c64 *__restrict__ coef
#define SVMI_TABLE_ARGS lph, ltab, wtab, ops, coef
#define SVMI_TABLES_OF(t) (t).lphases, (t).lane_tab, (t).wave_tab, (t).ops, (t).coef

__device__ __attribute__((always_inline)) inline double& lds_at(unsigned char* smem, uint32_t byte)
{
    return *reinterpret_cast<double*>(smem + byte);
}

// One tile of one sweep: load, phases, store (and for NS = 2 the tile's
// gradient partials).  init_zero: the tile is generated as |0..0>.
//
// The tile stays in registers: a[0..15] per thread (NS = 2: phi's 8
// amplitudes, then lambda's), 64 VGPRs, which with the op templates fit the
// 128 that leave four waves per SIMD.  Between two phases the amplitudes
// change threads through LDS, real parts first: 8 bytes per amplitude, so two
// 13-qubit tiles share a CU (tiles held in LDS: one, or two of 12 qubits at
// two waves per SIMD).  u3 brick wall at 30 qubits, 23 sweeps of 9.18 ms ->
// 19 of 8.65 ms (12-qubit tiles: 23 of 7.83); a two-state sweep at 25 qubits
// 641 -> 490 us.
//
// What bounds it: HBM (6.4 ms of the 8.65 at the copy rate), then the issue
// slots of a SIMD, which scalar instructions and branches share with the
// FMAs; hence the tables of ready offsets (LayoutPhase, SweepIO), 32-bit
// coefficient offsets and no loads ahead: 4070 -> 3490 instructions per wave,
// 1600 of them FMAs, u3 176 -> 167 ms.
//
// kLat: the build for sweeps of few tiles, which leave the chip idle and are
// bound by latency: a cold scalar load takes a microsecond, a register table
// four of them in a row.  Every phase's coefficients are staged in LDS during
// the phase before it and the next op's header is loaded during an op.  Where
// LDS allows (sw.whole), exchanges move whole amplitudes: one round trip and
// one barrier instead of two and three (ansatz of 20 u3 layers at 13 qubits
// 83.9 -> 82.2 us, random layers at 17 qubits 156.7 -> 151.9).
template <int NS, int kMaxQ, bool kLat = false>
__device__ __attribute__((always_inline)) inline void
sweep_tile(c64* __restrict__ s0, c64* __restrict__ s1, const SweepInfo& sw, const SweepIO* __restrict__ io, SVMI_TABLES,
           double* __restrict__ grad_partials, uint64_t tile, unsigned char* smem, bool init_zero)
{
    // kLat: a tile of less than a wave's threads has a whole wave; the others
    // repeat its threads (same values to the same places) but for the tables,
    // which all of them load (stid of snt): one thread took 33 of the 67 us of
    // 10 random layers at 4 qubits to stage them
    const uint32_t stid = threadIdx.x, snt = blockDim.x;
    const uint32_t nt = kLat ? min(snt, sweep_threads(sw.k, NS)) : snt, tid = kLat ? stid & (nt - 1) : stid;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nwaves = (nt + 63) / 64;
    coef += sw.coef_base;
    const uint32_t plane = uint32_t(8 * NS) << sw.k;
    const bool whole = kLat && sw.whole;   // uniform
    c64* xf = reinterpret_cast<c64*>(smem + (size_t(plane) << (whole ? 1 : 0)));
    double* gacc = reinterpret_cast<double*>(xf + sw.n_xf);
    uint64_t base = 0;
    for (uint32_t i = 0; i < io->n_runs; i++) {
        const TileRun r = io->run[i];
        base |= ((tile << r.shl) >> r.shr) & r.mask;
    }
    // the thread's byte offset of a load (0) or store (1)
    const auto thread_off = [&](int side) {
        uint64_t u = (base << 4) ^ io->wave[side][wave];
#pragma unroll
        for (int i = 0; i < kLaneBits; i++) u ^= ((lane >> i) & 1u) ? io->lane[side][i] : uint64_t(0);
        return u;
    };
    const auto amp = [](c64* s, uint64_t off) { return reinterpret_cast<c64*>(reinterpret_cast<char*>(s) + off); };
    // the tile's factors before its loads: their tables take 64 registers
    tile_factors(xf, sw, ops, coef, base, stid);
    c64 a[kRegs];
    {
        // in batches of four, so that addresses do not hold registers long
        const uint64_t g = thread_off(0);
        if (init_zero) {
#pragma unroll
            for (int r = 0; r < kRegs; r++) a[r] = c64{(g ^ io->reg[0][r]) == 0 ? 1.0 : 0.0, 0.0};
        } else if (io->additive & kIoAdditive) {
#pragma unroll
            for (int r = 0; r < kRegs; r++) {
                const bool second = NS == 2 && r >= kRegsAdj;
                a[r] = *amp(amp(second ? s1 : s0, g), io->reg[0][second ? r - kRegsAdj : r]);
                if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int r = 0; r < kRegs; r++) {
                const bool second = NS == 2 && r >= kRegsAdj;
                a[r] = *amp(second ? s1 : s0, g ^ io->reg[0][second ? r - kRegsAdj : r]);
                if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const uint32_t vhi = uint32_t(tile >> io->vhi_shift);
    // a phase's thread entry is loaded during the phase before it
    const uint32_t ph_begin = io->ph_begin, ph_end = io->ph_end;
    c64* const stage = reinterpret_cast<c64*>(gacc + sw.n_grad * nwaves + (sw.n_grad * nwaves & 1u));
    if constexpr (kLat) {
        const uint32_t n = lph[ph_begin].coef_n, c0 = lph[ph_begin].coef_begin;
        for (uint32_t i = stid; i < n; i += snt) stage[i] = coef[c0 + i];
    }
    if (kLat || sw.n_xf) __syncthreads();
    uint64_t le = ltab[size_t(ph_begin) * kLaneEntries + lane];
    for (uint32_t p = ph_begin; p < ph_end; p++) {
        const LayoutPhase& L = lph[p];
        const uint64_t te = le ^ wtab[size_t(p) * kWaveEntries + wave];
        const uint32_t pn = p + 1 < ph_end ? p + 1 : p;
        le = ltab[size_t(pn) * kLaneEntries + lane];
        if (p != ph_begin) {
            uint32_t w = uint32_t(te) & 0xffffu, rd = uint32_t(te) >> 16;
            const uint32_t flags = L.flags;
            const bool cross = flags & LPH_CROSS;
            // a wave's LDS operations complete in order: inside the waves the
            // order of the instructions is enough
            const auto meet = [&]() {
                if (cross) __syncthreads();
                else asm volatile("" ::: "memory");
            };
            if (whole) {   // (kLat's barrier after a phase's ops is the guard)
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    const uint32_t at = w ^ L.w[r];
                    lds_at(smem, at) = a[r].re;
                    lds_at(smem, at + plane) = a[r].im;
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                meet();
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    const uint32_t at = rd ^ L.rd[r];
                    a[r].re = lds_at(smem, at);
                    a[r].im = lds_at(smem, at + plane);
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                if (!kLat && (flags & LPH_GUARD)) __syncthreads();
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    lds_at(smem, w ^ L.w[r]) = a[r].re;
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                meet();
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    a[r].re = lds_at(smem, rd ^ L.rd[r]);
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                // fresh copies, or 32 addresses would stay in registers from the first half
                asm volatile("" : "+v"(w), "+v"(rd));
                meet();
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    lds_at(smem, w ^ L.w[r]) = a[r].im;
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                meet();
#pragma unroll
                for (int r = 0; r < kRegs; r++) {
                    a[r].im = lds_at(smem, rd ^ L.rd[r]);
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        const uint32_t goff = uint32_t(te >> 32) & 0xffffu, grp = uint32_t(te >> 48);
        const RegOffsets off{L.rcol};
        const uint32_t op_end = L.op_end;
        const DOp* __restrict__ op = ops + L.op_begin;
        // kLat: this phase's coefficients in one half of the stage; the next
        // one's are on their way, up to kPre per thread in registers
        constexpr uint32_t kPre = 4;
        const c64* __restrict__ cf = coef;
        c64 pre[kLat ? kPre : 1];
        uint32_t pre_n = 0, pre_c = 0;
        DOpHdr nxt;
        if constexpr (kLat) {
            cf = stage + ((p - ph_begin) & 1u) * sw.stage;
            if (p + 1 < ph_end) {
                pre_n = lph[p + 1].coef_n;
                pre_c = lph[p + 1].coef_begin;
            }
#pragma unroll
            for (uint32_t i = 0; i < kPre; i++)
                pre[i] = coef[stid + snt * i < pre_n ? pre_c + stid + snt * i : 0u];
            nxt = op->h;
        }
        for (uint32_t o = L.op_begin; o < op_end; o++, op++) {
            DOpHdr h;
            if constexpr (kLat) {   // (op arrays end with an unused record)
                h = nxt;
                nxt = op[1].h;
                h.coef -= L.coef_begin;
            } else {
                h = op->h;
            }
            if constexpr (NS == 2) {
                if (h.type == DOP_GRAD_DENSE || h.type == DOP_GRAD_DIAG) {
                    // every gradient op of a sweep has its own slot and each
                    // wave runs it once: a plain store, no read
                    double v = exec_grad_op<kMaxDenseQubitsAdj, kRegsAdj>(h, op, a, cf, goff, off, base);
                    if (nt >= 64) {
                        v = wave_sum_lane63(v);
                        if (lane == 63u) gacc[h.grad * nwaves + wave] = v;
                    } else {
                        const int width = int(nt);
                        for (int d = width >> 1; d > 0; d >>= 1) v += __shfl_xor(v, d, width);
                        if (tid == 0) gacc[h.grad * nwaves] = v;
                    }
                    continue;
                }
            }
            exec_state_op<kMaxQ>(h, op, a, cf, goff, grp, off, base, xf, sw.exthi, vhi);
        }
        if constexpr (kLat) {
            c64* const to = stage + ((p + 1 - ph_begin) & 1u) * sw.stage;
#pragma unroll
            for (uint32_t i = 0; i < kPre; i++)
                if (stid + snt * i < pre_n) to[stid + snt * i] = c64{pre[i].re, pre[i].im};   // (copied whole, pre[] stays in scratch memory)
            for (uint32_t i = stid + snt * kPre; i < pre_n; i += snt) to[i] = coef[pre_c + i];
            __syncthreads();
        }
    }
    if (io->store_guard) {
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wave's loads are done
        __syncthreads();
    }
    {
        const uint64_t g = thread_off(1);
        if (io->additive & (kIoAdditive << 1)) {
#pragma unroll
            for (int r = 0; r < kRegs; r++) {
                const bool second = NS == 2 && r >= kRegsAdj;
                *amp(amp(second ? s1 : s0, g), io->reg[1][second ? r - kRegsAdj : r]) = a[r];
                if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int r = 0; r < kRegs; r++) {
                const bool second = NS == 2 && r >= kRegsAdj;
                *amp(second ? s1 : s0, g ^ io->reg[1][second ? r - kRegsAdj : r]) = a[r];
                if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // gradient partials are stored grad-major ([i][tile]) so the sum over
    // tiles of one gradient reads one contiguous segment
    if constexpr (NS == 2) {
        if (sw.n_grad) __syncthreads();
        for (uint32_t i = tid; i < sw.n_grad; i += nt) {
            double v = 0.0;
            for (uint32_t w = 0; w < nwaves; w++) v += gacc[i * nwaves + w];
            grad_partials[i * sw.n_tiles + tile] = v;
        }
    }
}

// Waves per SIMD of the sweep kernels: dense blocks of three and four register
// qubits need up to 64 registers for their results.
template <int kMaxQ>
constexpr int kSweepWaves = kMaxQ <= 2 ? 4 : 2;

// One state, one tile per workgroup.
// kMaxQ: widest dense block compiled in (sweeps with blocks of at most two
// register qubits run the kMaxQ = 2 build, which holds fewer registers).
// kLat: see sweep_tile.
template <int kMaxQ, bool kLat>
__global__ void __launch_bounds__(kMaxTileThreads, kLat ? 2 : kSweepWaves<kMaxQ>)
k_sweep1(c64* __restrict__ s0, const SweepInfo sw, const SweepIO* __restrict__ io, SVMI_TABLES, uint64_t tile_offset)
{
    extern __shared__ __align__(16) unsigned char smem[];
    sweep_tile<1, kMaxQ, kLat>(s0, nullptr, sw, io, SVMI_TABLE_ARGS, nullptr, tile_offset + blockIdx.x, smem, false);
}

// Two states (adjoint), dense ops of at most 2 qubits.
template <bool kLat>
__global__ void __launch_bounds__(kMaxTileThreads, kLat ? 2 : 4)
k_sweep2(c64* __restrict__ s0, c64* __restrict__ s1, const SweepInfo sw, const SweepIO* __restrict__ io, SVMI_TABLES,
         double* __restrict__ grad_partials, uint64_t tile_offset)
{
    extern __shared__ __align__(16) unsigned char smem[];
    sweep_tile<2, kMaxDenseQubitsAdj, kLat>(s0, s1, sw, io, SVMI_TABLE_ARGS, grad_partials, tile_offset + blockIdx.x,
                                            smem, false);
}

// Sweeps run the latency build where all their waves fit the chip at its two
// per SIMD (2^17 threads, a wave per tile at least); where a phase has at most
// 8 coefficients per thread to stage; and not in the 512-thread tiles of one
// state on up to 64 CUs, whose two waves per SIMD hide the scalar loads
// themselves.  Latency / ordinary build: gradient of a 20-qubit ansatz with
// 11-qubit tiles (2^17 threads) 583 / 695 us, random layers of 22 qubits (2^18)
// 697 / 516 us; QFT of 20 qubits in 10-qubit tiles (up to 25 coefficients per
// thread) 164 / 120 us; random layers in 13-qubit tiles at 16 qubits (8 tiles)
// 174 / 160 us, at 20 (128) 333 / 359 us.
constexpr uint64_t kLatThreads = 1u << 17;
constexpr uint32_t kLatStage = 8;
// LDS of a CU's tiles up to which they exchange whole amplitudes (QFT of 21
// qubits, one 13-qubit tile of 136 KiB on each CU: 101 us, 94 by halves).
constexpr size_t kWholeBytes = 96 * 1024;
static size_t g_max_smem = 64 * 1024;  // dynamic LDS the sweep kernels may use

// --------------------------------------------------------------- batching
//
// A batch is a list of steps (forward sweep, Pauli step, adjoint sweep,
// reduction) of many circuits; a task is one tile (or chunk) of one step.
// Level l holds step l of every circuit that has one, so the tasks of a
// level are independent; inside a level the steps are grouped by kind and
// tile size, and each group is one launch (blockIdx.x -> task, blockDim =
// the group's tile threads).  Stream order between the launches supplies
// every dependency, so no workgroup ever waits for another one.

// The step of task t among steps [s0, s1): the last one whose task_begin is
// not above t.
__device__ inline uint32_t batch_step_of(const BatchStep* __restrict__ steps, uint32_t s0, uint32_t s1, uint64_t t)
{
    uint32_t lo = s0, hi = s1;
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (steps[mid].task_begin <= t) lo = mid;
        else hi = mid;
    }
    return lo;
}

#define SVMI_BATCH_TABLES                                                                           \
    const BatchStep *__restrict__ steps, const BatchCircuit *__restrict__ circuits,                 \
        const SweepInfo *__restrict__ sweeps, const SweepIO *__restrict__ ios

// One wave per phase (a batch has thousands of short ones: their tables by
// copy were two thirds of what its calls upload).
__global__ void __launch_bounds__(kThreads)
k_thread_tables(const ThreadCols* __restrict__ cols, uint64_t n, uint64_t* __restrict__ lane_tab,
                uint64_t* __restrict__ wave_tab)
{
    const uint64_t p = blockIdx.x * uint64_t(kThreads / 64) + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    if (p >= n) return;
    lane_tab[p * kLaneEntries + lane] = lane_entry(cols[p], lane);
    if (lane < uint32_t(kWaveEntries)) wave_tab[p * kWaveEntries + lane] = wave_entry(cols[p], lane);
}

hipError_t launch_thread_tables(hipStream_t st, const ThreadCols* cols, uint64_t n, uint64_t* lane_tab,
                                uint64_t* wave_tab)
{
    constexpr uint64_t per = kThreads / 64, max_grid = 1ull << 30;
    for (uint64_t p0 = 0; p0 < n; p0 += max_grid * per) {
        const uint64_t cnt = n - p0 < max_grid * per ? n - p0 : max_grid * per;
        hipLaunchKernelGGL(k_thread_tables, dim3(uint32_t((cnt + per - 1) / per)), dim3(kThreads), 0, st, cols + p0, cnt,
                           lane_tab + p0 * kLaneEntries, wave_tab + p0 * kWaveEntries);
    }
    return hipGetLastError();
}

// kInit: the steps are first forward sweeps (tiles generated as |0..0>).
// kLat, whole: see sweep_tile.
template <bool kInit, int kMaxQ, bool kLat>
__global__ void __launch_bounds__(kMaxTileThreads, kLat ? 2 : kSweepWaves<kMaxQ>)
k_batch_fwd(SVMI_BATCH_TABLES, SVMI_TABLES, uint32_t s0, uint32_t s1, uint64_t task0, uint32_t whole)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const uint64_t t = task0 + blockIdx.x;
    const BatchStep st = steps[batch_step_of(steps, s0, s1, t)];
    SweepInfo sw = sweeps[st.sweep];
    sw.whole = whole;
    const SweepIO* __restrict__ io = ios + st.sweep;
    sweep_tile<1, kMaxQ, kLat>(circuits[st.circuit].phi, nullptr, sw, io, SVMI_TABLE_ARGS, nullptr, t - st.task_begin, smem,
                         kInit);
}

template <bool kLat>
__global__ void __launch_bounds__(kMaxTileThreads, kLat ? 2 : 4)
k_batch_adj(SVMI_BATCH_TABLES, SVMI_TABLES, double* __restrict__ grad_partials, uint32_t s0, uint32_t s1,
            uint64_t task0, uint32_t whole)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const uint64_t t = task0 + blockIdx.x;
    const BatchStep st = steps[batch_step_of(steps, s0, s1, t)];
    SweepInfo sw = sweeps[st.sweep];
    sw.whole = whole;
    const SweepIO* __restrict__ io = ios + st.sweep;
    const BatchCircuit& c = circuits[st.circuit];
    sweep_tile<2, kMaxDenseQubitsAdj, kLat>(c.phi, c.lam, sw, io, SVMI_TABLE_ARGS, grad_partials + st.partial,
                                      t - st.task_begin, smem, false);
}

// ------------------------------------------------------------- Pauli sums
//
// The thread's M amplitudes of H psi at y = yb | col[j] (j < M): tile groups
// read the tile in LDS (thread tid's register j is tile-local index
// tid + nt j), the others read psi from memory.  A term's sign is
// (-1)^{|yb & z|} per thread times a uniform sign per register (jsign), so a
// term costs a few integer operations per thread and one add per amplitude
// instead of a 64-bit population count per amplitude.  Terms with the same
// register signs are neighbours and are summed first: one add per term, M
// adds per pattern of signs (the first pass of an Ising sum at 28 qubits, 27
// ZZ terms and 12 X masks, all passes: 4.07 -> 3.71 ms).
//
// Loads go in batches of up to 4, all issued before the first is used (left
// to itself the compiler keeps two LDS reads in flight here, and a pass over
// 28 qubits with 8 masks takes 2.84 ms instead of 1.0; all 29 masks of an
// Ising sum there 16.5 -> 3.7 ms, in 3 passes that read 4.3 GB each).

// l[j] += (cre + i cim) v[j - j0], j0 <= j < j0 + B
template <int M, int B>
__device__ __attribute__((always_inline)) inline void
pauli_add(c64 (&l)[M], const c64 (&v)[B], int j0, double cre, double cim)
{
#pragma unroll
    for (int j = 0; j < B; j++) {
        l[j0 + j].re = SVMI_FMA(cre, v[j].re, l[j0 + j].re);
        l[j0 + j].im = SVMI_FMA(cre, v[j].im, l[j0 + j].im);
    }
    if (cim != 0.0)   // uniform
#pragma unroll
        for (int j = 0; j < B; j++) {
            l[j0 + j].re = SVMI_FMA(-cim, v[j].im, l[j0 + j].re);
            l[j0 + j].im = SVMI_FMA(cim, v[j].re, l[j0 + j].im);
        }
}

// the amplitudes of registers j0 .. j0 + B - 1 with the tile-local bits x flipped
template <int B>
__device__ __attribute__((always_inline)) inline void
pauli_tile_read(c64 (&v)[B], const c64* t, int j0, uint32_t tid, uint32_t nt, uint32_t x)
{
    const uint32_t at = tid ^ x;   // x's thread bits, and its register bits above them
    if (x < nt) {
#pragma unroll
        for (int j = 0; j < B; j++) v[j] = t[at + nt * (j0 + j)];
    } else {
#pragma unroll
        for (int j = 0; j < B; j++) v[j] = t[at ^ (nt * (j0 + j))];
    }
}

// kFull: the tile has all nt * M amplitudes (otherwise tsize, the rest unused).
template <int M, bool kFull>
__device__ __attribute__((always_inline)) inline void
pauli_groups(c64 (&l)[M], const c64* t, const c64* __restrict__ psi, uint64_t yb, const uint64_t (&col)[M], uint32_t tid,
             uint32_t nt, uint32_t tsize, const PauliGroup* __restrict__ groups,
             const PauliTerm* __restrict__ terms, uint32_t g0, uint32_t gf, uint32_t gt, uint32_t g1)
{
    constexpr int B = M < 4 ? M : 4;
#pragma unroll
    for (int j = 0; j < M; j++) l[j] = c64{0.0, 0.0};
    if (g0 < gf) {   // group records and terms are read one group ahead
        const PauliTerm* __restrict__ ft = terms + groups[g0].begin;
        uint32_t x = uint32_t(groups[g0].xmask);
        double cre = ft[0].cre, cim = ft[0].cim;
        for (uint32_t g = g0; g < gf; g++) {
            const uint32_t nxt = g + 1 < gf ? g + 1 : g;
            const uint32_t xn = uint32_t(groups[nxt].xmask);
            const double cren = ft[nxt - g0].cre, cimn = ft[nxt - g0].cim;
#pragma unroll
            for (int j0 = 0; j0 < M; j0 += B) {
                c64 v[B];
                pauli_tile_read<B>(v, t, j0, tid, nt, x);
                __builtin_amdgcn_sched_barrier(0);
                pauli_add<M, B>(l, v, j0, cre, cim);
                __builtin_amdgcn_sched_barrier(0);
            }
            x = xn, cre = cren, cim = cimn;
        }
    }
    for (uint32_t g = gf; g < g1; g++) {
        const PauliGroup G = groups[g];
        const bool tile = g < gt;
        for (uint32_t part = 0; part <= G.imag; part++) {   // real coefficients, then imaginary ones
            double f[M];
#pragma unroll
            for (int j = 0; j < M; j++) f[j] = 0.0;
            double c = 0.0;
            for (uint32_t e = G.begin; e < G.end; e++) {
                const PauliTerm T = terms[e];
                const double c0 = part ? T.cim : T.cre;
                c += __hiloint2double(__double2hiint(c0) ^ int(uint32_t(__popcll(yb & T.zmask)) << 31),
                                      __double2loint(c0));
                if (T.last) {   // uniform
#pragma unroll
                    for (int j = 0; j < M; j++)   // +-c as a scalar +-1.0 in one FMA
                        f[j] = SVMI_FMA(__hiloint2double(int(0x3ff00000u | (T.jsign >> j) << 31), 0), c, f[j]);
                    c = 0.0;
                }
            }
#pragma unroll
            for (int j0 = 0; j0 < M; j0 += B) {
                c64 v[B];
                if (tile) {
                    pauli_tile_read<B>(v, t, j0, tid, nt, uint32_t(G.xmask));
                } else {
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        if (kFull || tid + nt * (j0 + j) < tsize) v[j] = psi[(yb | col[j0 + j]) ^ G.xmask];
                        else v[j] = c64{0.0, 0.0};
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                if (part) {
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        l[j0 + j].re = SVMI_FMA(-f[j0 + j], v[j].im, l[j0 + j].re);
                        l[j0 + j].im = SVMI_FMA(f[j0 + j], v[j].re, l[j0 + j].im);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        l[j0 + j].re = SVMI_FMA(f[j0 + j], v[j].re, l[j0 + j].re);
                        l[j0 + j].im = SVMI_FMA(f[j0 + j], v[j].im, l[j0 + j].im);
                    }
                }
            }
        }
    }
}

// <H> step: lam = H phi on a tile of the low qubits (kPauliChunk amplitudes,
// or the whole state where it is smaller) and the tile's partial sum of
// Re <phi|lam>.  The tile is staged in LDS, so only X masks above it read
// memory (from L2 mostly): 96 circuits of 10-20 qubits 2.09 -> 0.68 ms.
__global__ void __launch_bounds__(kPauliThreads, 4)
k_batch_pauli(BatchArgs a, uint32_t s0, uint32_t s1, uint64_t task0)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int M = kPauliRegs;
    c64* tl = reinterpret_cast<c64*>(smem);
    const uint64_t t = task0 + blockIdx.x;
    const BatchStep st = a.steps[batch_step_of(a.steps, s0, s1, t)];
    const BatchCircuit& c = a.circuits[st.circuit];
    const uint64_t task = t - st.task_begin;
    const uint32_t tsize = c.n < uint32_t(kPauliTileQubits) ? 1u << c.n : kPauliChunk;
    const uint64_t y0 = task * kPauliChunk;
    const uint32_t tid = threadIdx.x;
    c64 l[M];
    uint64_t col[M];
#pragma unroll
    for (int j = 0; j < M; j++) col[j] = uint64_t(kPauliThreads) * j;
    const c64* phi = c.phi;
    for (uint32_t x = tid; x < tsize; x += kPauliThreads) tl[x] = phi[y0 + x];
    __syncthreads();
    if (tsize == kPauliChunk)
        pauli_groups<M, true>(l, tl, phi, y0 + tid, col, tid, kPauliThreads, tsize, a.groups, a.terms, c.group_begin,
                              c.flat_end, c.tile_end, c.group_end);
    else
        pauli_groups<M, false>(l, tl, phi, y0 + tid, col, tid, kPauliThreads, tsize, a.groups, a.terms, c.group_begin,
                               c.flat_end, c.tile_end, c.group_end);
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < M; j++) {
        const uint32_t x = tid + kPauliThreads * j;
        if (x < tsize) {
            c.lam[y0 + x] = l[j];
            const c64 p = tl[x];
            acc += p.re * l[j].re + p.im * l[j].im;
        }
    }
    __syncthreads();
    double* red = reinterpret_cast<double*>(smem);
    red[tid] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (tid < k) red[tid] += red[tid + k];
        __syncthreads();
    }
    if (tid == 0) a.e_partials[st.partial + task] = red[0];
}

// The largest of a launch's sweeps.
static SweepInfo batch_sweep(const BatchLaunch& L)
{
    SweepInfo sw;
    std::memset(&sw, 0, sizeof(sw));
    sw.k = L.k;
    sw.n_xf = L.max_xf;
    sw.n_grad = L.kind == BSTEP_ADJ ? L.max_grad : 0;
    sw.stage = L.max_stage;
    sw.max_dense = L.max_dense;
    sw.n_tiles = L.n_tasks;
    return sw;
}

// Whether a launch of sw.n_tiles tiles runs the latency build, its threads
// per tile and bytes of LDS.  (A batch's launch counts the tiles of all its
// circuits: 4 circuits of 12 qubits 2.33 -> 2.04 ms, 64 of 12 4.07 -> 3.95.)
struct SweepLaunch {
    bool lat;
    uint32_t whole, threads;
    size_t smem;
};
static SweepLaunch sweep_launch(const SweepInfo& sw, int ns)
{
    const uint32_t nt = sweep_threads(sw.k, ns), threads = std::max(nt, 64u);
    const size_t smem = sweep_smem_bytes(sw, ns), lat_smem = smem + 8 + 32 * sw.stage;
    const size_t whole = lat_smem + (size_t(8) << sw.k) * ns;
    SweepLaunch l;
    l.lat = sw.max_dense <= 2 && sw.n_tiles * threads <= kLatThreads && sw.stage <= kLatStage * threads &&
            !(ns == 1 && nt == 512 && sw.n_tiles <= 64) && lat_smem <= g_max_smem;
    l.whole = l.lat && whole * ((sw.n_tiles + 255) / 256) <= kWholeBytes ? 1u : 0u;
    l.threads = l.lat ? threads : nt;
    l.smem = l.whole ? whole : l.lat ? lat_smem : smem;
    return l;
}

size_t batch_launch_smem(const BatchLaunch& L)
{
    if (L.kind != BSTEP_FWD && L.kind != BSTEP_ADJ) return size_t(16) * kPauliChunk;
    return sweep_smem_bytes(batch_sweep(L), L.kind == BSTEP_ADJ ? 2 : 1);
}

// The k_batch_fwd build of a forward launch.
using BatchFwdFn = void (*)(SVMI_BATCH_TABLES, SVMI_TABLES, uint32_t, uint32_t, uint64_t, uint32_t);
BatchFwdFn batch_fwd_kernel(const BatchLaunch& L, bool lat)
{
    if (lat) return L.init ? &k_batch_fwd<true, 2, true> : &k_batch_fwd<false, 2, true>;
    if (L.init) return L.max_dense <= 2 ? &k_batch_fwd<true, 2, false> : &k_batch_fwd<true, kRegBits, false>;
    return L.max_dense <= 2 ? &k_batch_fwd<false, 2, false> : &k_batch_fwd<false, kRegBits, false>;
}

hipError_t launch_batch(hipStream_t st, const BatchArgs& a, const BatchLaunch& L)
{
    SweepLaunch l{false, 0, uint32_t(kPauliThreads), batch_launch_smem(L)};
    if (L.kind != BSTEP_PAULI) l = sweep_launch(batch_sweep(L), L.kind == BSTEP_ADJ ? 2 : 1);
    if (l.smem > g_max_smem) return hipErrorInvalidConfiguration;
    const dim3 threads(l.threads);
    const size_t smem = l.smem;
    const uint64_t max_grid = 1ull << 30;
    for (uint64_t t0 = 0; t0 < L.n_tasks; t0 += max_grid) {
        const uint32_t cnt = uint32_t(L.n_tasks - t0 < max_grid ? L.n_tasks - t0 : max_grid);
        const uint64_t first = L.task_begin + t0;
        switch (L.kind) {
        case BSTEP_FWD: {
            auto* fn = batch_fwd_kernel(L, l.lat);
            hipLaunchKernelGGL(fn, dim3(cnt), threads, smem, st, a.steps, a.circuits, a.sweeps, a.io,
                               SVMI_TABLES_OF(a.t), L.step_begin, L.step_end, first, l.whole);
            break;
        }
        case BSTEP_ADJ: {
            auto* fn = l.lat ? &k_batch_adj<true> : &k_batch_adj<false>;
            hipLaunchKernelGGL(fn, dim3(cnt), threads, smem, st, a.steps, a.circuits, a.sweeps, a.io,
                               SVMI_TABLES_OF(a.t), a.grad_partials, L.step_begin, L.step_end, first, l.whole);
            break;
        }
        case BSTEP_PAULI:
            hipLaunchKernelGGL(k_batch_pauli, dim3(cnt), threads, smem, st, a, L.step_begin, L.step_end, first);
            break;
        default:
            return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

hipError_t launch_sweep(hipStream_t st, int ns, c64* s0, c64* s1, const SweepInfo& info, const SweepIO* io,
                        const SweepTables& t, double* grad_partials)
{
    SweepInfo sw = info;
    const SweepLaunch l = sweep_launch(sw, ns);
    sw.whole = l.whole;
    if (l.smem > g_max_smem || l.threads > uint32_t(kMaxTileThreads)) return hipErrorInvalidConfiguration;
    const uint64_t max_grid = 1ull << 30;
    for (uint64_t t0 = 0; t0 < sw.n_tiles; t0 += max_grid) {
        const uint64_t cnt = sw.n_tiles - t0 < max_grid ? sw.n_tiles - t0 : max_grid;
        const dim3 grid{uint32_t(cnt)}, threads(l.threads);
        if (ns == 1) {
            auto* fn = l.lat               ? &k_sweep1<2, true>
                       : sw.max_dense <= 2 ? &k_sweep1<2, false>
                                           : &k_sweep1<kRegBits, false>;
            hipLaunchKernelGGL(fn, grid, threads, l.smem, st, s0, sw, io, SVMI_TABLES_OF(t), t0);
        } else {
            hipLaunchKernelGGL(l.lat ? &k_sweep2<true> : &k_sweep2<false>, grid, threads, l.smem, st, s0, s1, sw, io,
                               SVMI_TABLES_OF(t), grad_partials, t0);
        }
    }
    return hipGetLastError();
}

size_t sweep_smem_limit() { return g_max_smem; }

// Raise the dynamic-LDS limit of the sweep kernels to what the device allows
// per workgroup (gfx950: 160 KiB per CU); 64 KiB always works.
hipError_t init_sweep_kernels()
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    int optin = 0;
    if (hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, dev) != hipSuccess || optin <= 0)
        optin = 64 * 1024;
    size_t want = size_t(optin);
    if (want > 160 * 1024) want = 160 * 1024;
    const auto raise = [&](const void* fn) {
        return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(want)) == hipSuccess;
    };
    if (want > 64 * 1024 &&
        !(raise(reinterpret_cast<const void*>(&k_sweep1<2, false>)) &&
          raise(reinterpret_cast<const void*>(&k_sweep1<kRegBits, false>)) &&
          raise(reinterpret_cast<const void*>(&k_sweep1<2, true>)) &&
          raise(reinterpret_cast<const void*>(&k_sweep2<false>)) &&
          raise(reinterpret_cast<const void*>(&k_sweep2<true>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_adj<false>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_adj<true>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<true, 2, false>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<false, 2, false>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<true, 2, true>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<false, 2, true>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<true, kRegBits, false>)) &&
          raise(reinterpret_cast<const void*>(&k_batch_fwd<false, kRegBits, false>)))) {
        (void)hipGetLastError();
        want = 64 * 1024;
    }
    g_max_smem = want;
    return hipSuccess;
}

// -------------------------------------------------------- standalone ops

struct QArgs {
    int q;
    int qubits[5];      // op order
    int sorted[5];      // ascending
};

template <int K>
__global__ void __launch_bounds__(256)
k_dense_full(c64* __restrict__ s, uint64_t ngroups, QArgs qa, const c64* __restrict__ M)
{
    constexpr int D = 1 << K;
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < ngroups;
         g += uint64_t(gridDim.x) * blockDim.x) {
        uint64_t b = g;
#pragma unroll
        for (int i = 0; i < K; i++) {
            const int p = qa.sorted[i];
            b = ((b >> p) << (p + 1)) | (b & ((1ull << p) - 1ull));
        }
        uint64_t idx[D];
        c64 v[D];
#pragma unroll
        for (int j = 0; j < D; j++) {
            uint64_t o = b;
#pragma unroll
            for (int i = 0; i < K; i++)
                if ((j >> i) & 1) o |= 1ull << qa.qubits[i];
            idx[j] = o;
            v[j] = s[o];
        }
#pragma unroll
        for (int r = 0; r < D; r++) {
            c64 acc{0.0, 0.0};
#pragma unroll
            for (int j = 0; j < D; j++) acc = cmac(acc, M[r * D + j], v[j]);
            s[idx[r]] = acc;
        }
    }
}

__global__ void __launch_bounds__(256)
k_diag_full(c64* __restrict__ s, uint64_t dim, QArgs qa, const c64* __restrict__ tab)
{
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < dim;
         x += uint64_t(gridDim.x) * blockDim.x) {
        uint32_t idx = 0;
        for (int i = 0; i < qa.q; i++) idx |= uint32_t((x >> qa.qubits[i]) & 1u) << i;
        s[x] = cmul(s[x], tab[idx]);
    }
}

__global__ void __launch_bounds__(256) k_srn_full(c64* __restrict__ s, uint64_t half, int q)
{
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < half;
         i += uint64_t(gridDim.x) * blockDim.x) {
        const uint64_t p0 = ((i >> q) << (q + 1)) | (i & ((1ull << q) - 1ull));
        const uint64_t p1 = p0 | (1ull << q);
        const c64 a0 = s[p0], a1 = s[p1];
        s[p0] = c64{0.5 * (a0.re + a1.re), 0.5 * (a0.im - a1.im)};
        s[p1] = c64{0.5 * (a0.re + a1.re), 0.5 * (-a0.im + a1.im)};
    }
}

static unsigned grid_for(uint64_t work, unsigned block)
{
    const uint64_t g = (work + block - 1) / block;
    const uint64_t cap = 65536;
    return unsigned(g < 1 ? 1 : (g > cap ? cap : g));
}

hipError_t launch_standalone(hipStream_t st, c64* s, int n, const StandaloneOp& so, const c64* coef)
{
    QArgs qa;
    qa.q = so.q;
    for (int i = 0; i < 5; i++) qa.qubits[i] = i < so.q ? so.qubits[i] : 0;
    for (int i = 0; i < 5; i++) qa.sorted[i] = qa.qubits[i];
    for (int i = 0; i < so.q; i++)
        for (int j = i + 1; j < so.q; j++)
            if (qa.sorted[j] < qa.sorted[i]) {
                const int t = qa.sorted[i];
                qa.sorted[i] = qa.sorted[j];
                qa.sorted[j] = t;
            }
    const uint64_t dim = 1ull << n;
    if (so.kind == 2) {
        hipLaunchKernelGGL(k_srn_full, dim3(grid_for(dim / 2, 256)), dim3(256), 0, st, s, dim / 2, so.qubits[0]);
    } else if (so.kind == 1) {
        hipLaunchKernelGGL(k_diag_full, dim3(grid_for(dim, 256)), dim3(256), 0, st, s, dim, qa, coef + so.coef);
    } else {
        const uint64_t ng = dim >> so.q;
        const dim3 gr(grid_for(ng, 256)), bl(256);
        const c64* M = coef + so.coef;
        switch (so.q) {
        case 1: hipLaunchKernelGGL(k_dense_full<1>, gr, bl, 0, st, s, ng, qa, M); break;
        case 2: hipLaunchKernelGGL(k_dense_full<2>, gr, bl, 0, st, s, ng, qa, M); break;
        case 3: hipLaunchKernelGGL(k_dense_full<3>, gr, bl, 0, st, s, ng, qa, M); break;
        case 4: hipLaunchKernelGGL(k_dense_full<4>, gr, bl, 0, st, s, ng, qa, M); break;
        default: hipLaunchKernelGGL(k_dense_full<5>, gr, bl, 0, st, s, ng, qa, M); break;
        }
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ state utils

__global__ void __launch_bounds__(256) k_fill_basis(c64* __restrict__ s, uint64_t dim)
{
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < dim;
         x += uint64_t(gridDim.x) * blockDim.x)
        s[x] = c64{x == 0 ? 1.0 : 0.0, 0.0};
}

__global__ void __launch_bounds__(256) k_copy(c64* __restrict__ d, const c64* __restrict__ s, uint64_t dim)
{
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < dim;
         x += uint64_t(gridDim.x) * blockDim.x)
        d[x] = s[x];
}

// splitmix64 finaliser (Steele, Lea & Flood 2014)
__device__ inline uint64_t splitmix64(uint64_t z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__global__ void __launch_bounds__(256)
k_random_state(c64* __restrict__ s, uint64_t dim, uint64_t seed, double* __restrict__ partials)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < dim;
         x += uint64_t(gridDim.x) * blockDim.x) {
        const double u0 = double((splitmix64(seed + 2 * x + 1) >> 11) + 1) * 0x1p-53;
        const double u1 = double((splitmix64(seed + 2 * x + 2) >> 11) + 1) * 0x1p-53;
        const double r = sqrt(-2.0 * log(u0));
        double sn, cs;
        sincospi(2.0 * u1, &sn, &cs);
        const c64 v{r * cs, r * sn};
        s[x] = v;
        acc += v.re * v.re + v.im * v.im;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_scale(c64* __restrict__ s, uint64_t dim, double f)
{
    for (uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < dim;
         x += uint64_t(gridDim.x) * blockDim.x) {
        s[x].re *= f;
        s[x].im *= f;
    }
}

uint32_t random_state_grid(uint64_t dim) { return grid_for(dim, 256) > 4096 ? 4096 : grid_for(dim, 256); }

hipError_t launch_random_state(hipStream_t st, c64* s, uint64_t dim, uint64_t seed, double* partials)
{
    hipLaunchKernelGGL(k_random_state, dim3(random_state_grid(dim)), dim3(256), 0, st, s, dim, seed, partials);
    return hipGetLastError();
}

hipError_t launch_scale(hipStream_t st, c64* s, uint64_t dim, double f)
{
    hipLaunchKernelGGL(k_scale, dim3(grid_for(dim, 256)), dim3(256), 0, st, s, dim, f);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256)
k_gather(const c64* __restrict__ s, uint64_t dim, const uint64_t* __restrict__ idx, uint64_t cnt, c64* __restrict__ out)
{
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < cnt) out[i] = idx[i] < dim ? s[idx[i]] : c64{0.0, 0.0};
}

hipError_t launch_gather(hipStream_t st, const c64* s, uint64_t dim, const uint64_t* idx, uint64_t cnt, c64* out)
{
    if (cnt == 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather, dim3(unsigned((cnt + 255) / 256)), dim3(256), 0, st, s, dim, idx, cnt, out);
    return hipGetLastError();
}

hipError_t launch_fill_basis(hipStream_t st, c64* s, uint64_t dim)
{
    hipLaunchKernelGGL(k_fill_basis, dim3(grid_for(dim, 256)), dim3(256), 0, st, s, dim);
    return hipGetLastError();
}

hipError_t launch_copy(hipStream_t st, c64* d, const c64* s, uint64_t dim)
{
    hipLaunchKernelGGL(k_copy, dim3(grid_for(dim, 256)), dim3(256), 0, st, d, s, dim);
    return hipGetLastError();
}

// -------------------------------------------------------------- sampling
//
// Scan definition (identical in both kernels, fixed operation order):
//   p_x = (re*re) + (im*im) with unfused IEEE ops (the reference's
//   expression, svsim_cpu_omp.hpp:345);
//   block of B = nthr*chunk amplitudes; thread t owns a contiguous chunk;
//   T_t = sequential sum of its chunk; P_t = exclusive prefix of T over the
//   threads (wave64 shuffle scan, then waves in order);
//   L_j = P_t + p_(first) + ... + p_j accumulated sequentially;
//   block total = L of the block's last amplitude.
// Global scan S_j = O_b + L_j with O_b the host's sequential prefix of the
// block totals; a draw r selects the first j with S_j > r (0 if none), which
// is the reference's interval rule scan[j] <= r < scan[j+1].

__device__ inline double prob_rn(c64 a) { return __dadd_rn(__dmul_rn(a.re, a.re), __dmul_rn(a.im, a.im)); }

__device__ double thread_prefix(const c64* __restrict__ blk, uint32_t chunk, double* lds_w)
{
    const uint32_t t = threadIdx.x, nthr = blockDim.x;
    double T = 0.0;
    for (uint32_t i = 0; i < chunk; i++) T = __dadd_rn(T, prob_rn(blk[size_t(t) * chunk + i]));
    const int width = nthr < 64 ? int(nthr) : 64;
    const int lane = int(t & 63u);
    double inc = T;
    for (int d = 1; d < width; d <<= 1) {
        const double u = __shfl_up(inc, d, width);
        if (lane >= d) inc = __dadd_rn(inc, u);
    }
    double exc = __shfl_up(inc, 1, width);
    if (lane == 0) exc = 0.0;
    const uint32_t w = t >> 6, nw = (nthr + 63) / 64;
    if (lane == width - 1) lds_w[w] = inc;
    __syncthreads();
    double wpre = 0.0;
    for (uint32_t v = 0; v < w; v++) wpre = __dadd_rn(wpre, lds_w[v]);
    (void)nw;
    __syncthreads();
    return w == 0 ? exc : __dadd_rn(wpre, exc);
}

__global__ void __launch_bounds__(256)
k_block_totals(const c64* __restrict__ s, uint32_t chunk, double* __restrict__ totals)
{
    __shared__ double lds_w[4];
    const uint64_t b = blockIdx.x;
    const c64* blk = s + b * uint64_t(blockDim.x) * chunk;
    double acc = thread_prefix(blk, chunk, lds_w);
    for (uint32_t i = 0; i < chunk; i++) acc = __dadd_rn(acc, prob_rn(blk[size_t(threadIdx.x) * chunk + i]));
    if (threadIdx.x == blockDim.x - 1) totals[b] = acc;
}

// The same two passes with the block's probabilities staged in LDS first:
// loaded lane-consecutive (coalesced), stored so that thread t's chunk sits
// at t * (chunk + 1) (the pad spreads the per-thread runs over the banks).
// Every sum keeps the order of the direct kernels above, so the totals and
// samples are bit-identical to theirs.
__device__ inline uint32_t staged_index(uint32_t j, uint32_t lg) { return j + (j >> lg); }

__device__ void stage_probs(const c64* __restrict__ blk, uint32_t lg, double* lp)
{
    const uint32_t bs = blockDim.x << lg;
    for (uint32_t j = threadIdx.x; j < bs; j += blockDim.x) lp[staged_index(j, lg)] = prob_rn(blk[j]);
    __syncthreads();
}

__device__ double thread_prefix_staged(const double* lp, uint32_t lg, double* lds_w)
{
    const uint32_t t = threadIdx.x, nthr = blockDim.x, chunk = 1u << lg;
    const double* mine = lp + t * (chunk + 1);
    double T = 0.0;
    for (uint32_t i = 0; i < chunk; i++) T = __dadd_rn(T, mine[i]);
    const int width = nthr < 64 ? int(nthr) : 64;
    const int lane = int(t & 63u);
    double inc = T;
    for (int d = 1; d < width; d <<= 1) {
        const double u = __shfl_up(inc, d, width);
        if (lane >= d) inc = __dadd_rn(inc, u);
    }
    double exc = __shfl_up(inc, 1, width);
    if (lane == 0) exc = 0.0;
    const uint32_t w = t >> 6;
    if (lane == width - 1) lds_w[w] = inc;
    __syncthreads();
    double wpre = 0.0;
    for (uint32_t v = 0; v < w; v++) wpre = __dadd_rn(wpre, lds_w[v]);
    __syncthreads();
    return w == 0 ? exc : __dadd_rn(wpre, exc);
}

__global__ void __launch_bounds__(256)
k_block_totals_staged(const c64* __restrict__ s, uint32_t lg, double* __restrict__ totals)
{
    extern __shared__ double lp[];
    __shared__ double lds_w[4];
    const uint64_t b = blockIdx.x;
    const uint32_t chunk = 1u << lg;
    stage_probs(s + (b * blockDim.x << lg), lg, lp);
    double acc = thread_prefix_staged(lp, lg, lds_w);
    const double* mine = lp + threadIdx.x * (chunk + 1);
    for (uint32_t i = 0; i < chunk; i++) acc = __dadd_rn(acc, mine[i]);
    if (threadIdx.x == blockDim.x - 1) totals[b] = acc;
}

// One workgroup per (block, shot range).  job = {block, first shot, n shots}.
__global__ void __launch_bounds__(256)
k_sample(const c64* __restrict__ s, uint32_t chunk, const uint64_t* __restrict__ jobs,
         const double* __restrict__ offsets, const double* __restrict__ draws,
         uint64_t* __restrict__ out)
{
    __shared__ double lds_w[4];
    __shared__ unsigned long long best;
    const uint64_t b = jobs[3 * blockIdx.x + 0];
    const uint64_t first = jobs[3 * blockIdx.x + 1];
    const uint64_t cnt = jobs[3 * blockIdx.x + 2];
    const uint64_t bsize = uint64_t(blockDim.x) * chunk;
    const c64* blk = s + b * bsize;
    const double P = thread_prefix(blk, chunk, lds_w);
    const double O = offsets[blockIdx.x];
    for (uint64_t q = 0; q < cnt; q++) {
        const double r = draws[first + q];
        if (threadIdx.x == 0) best = ~0ull;
        __syncthreads();
        double acc = P;
        uint64_t found = ~0ull;
        for (uint32_t i = 0; i < chunk; i++) {
            acc = __dadd_rn(acc, prob_rn(blk[size_t(threadIdx.x) * chunk + i]));
            if (__dadd_rn(O, acc) > r) {
                found = uint64_t(threadIdx.x) * chunk + i;
                break;
            }
        }
        if (found != ~0ull) atomicMin(&best, (unsigned long long)found);
        __syncthreads();
        if (threadIdx.x == 0) out[first + q] = best == ~0ull ? 0 : b * bsize + best;
        __syncthreads();
    }
}

// The same search with the block staged in LDS and one thread per draw.  The
// staged probabilities are replaced by the scan L_j itself, so a draw takes
// two binary searches (8 steps over the threads' runs, lg inside one run)
// instead of a pass of the whole workgroup over the block with three
// barriers: 1024 draws in one 2^12-amplitude block 3365 -> 9.7 us, and the
// draws of a block run in as many workgroups as the host cuts them into.
// O + L_j grows along a run (p_j >= 0 and rounding is monotone), but the next
// run starts from its own prefix and may begin an ulp lower, so the first
// run with a match is searched in the running maximum of the runs' last
// values: it first exceeds r where a run's own last value does, which is the
// smallest j that the definition above asks for.
__global__ void __launch_bounds__(256)
k_sample_staged(const c64* __restrict__ s, uint32_t lg, const uint64_t* __restrict__ jobs,
                const double* __restrict__ offsets, const double* __restrict__ draws,
                uint64_t* __restrict__ out)
{
    extern __shared__ double lp[];
    __shared__ double lds_w[4];
    __shared__ double top[256];   // running maximum of O + L at the end of each thread's run
    const uint32_t chunk = 1u << lg, t = threadIdx.x, nthr = blockDim.x;
    const uint64_t b = jobs[3 * blockIdx.x + 0];
    const uint64_t first = jobs[3 * blockIdx.x + 1];
    const uint64_t cnt = jobs[3 * blockIdx.x + 2];
    const uint64_t bsize = uint64_t(nthr) << lg;
    stage_probs(s + b * bsize, lg, lp);
    double acc = thread_prefix_staged(lp, lg, lds_w);
    const double O = offsets[blockIdx.x];
    double* mine = lp + t * (chunk + 1);
    for (uint32_t i = 0; i < chunk; i++) {
        acc = __dadd_rn(acc, mine[i]);
        mine[i] = acc;
    }
    const int width = nthr < 64 ? int(nthr) : 64;
    const int lane = int(t & 63u);
    double m = __dadd_rn(O, acc);
    for (int d = 1; d < width; d <<= 1) {
        const double u = __shfl_up(m, d, width);
        if (lane >= d && u > m) m = u;
    }
    if (lane == width - 1) lds_w[t >> 6] = m;
    __syncthreads();
    for (uint32_t v = 0; v < (t >> 6); v++)
        if (lds_w[v] > m) m = lds_w[v];
    top[t] = m;
    __syncthreads();
    for (uint64_t q = t; q < cnt; q += nthr) {
        const double r = draws[first + q];
        uint32_t lo = 0, len = nthr;   // smallest run with top > r in [lo, lo + len]
        while (len > 0) {
            const uint32_t half = len >> 1;
            if (top[lo + half] > r) len = half;
            else lo += half + 1, len -= half + 1;
        }
        uint64_t res = 0;
        if (lo < nthr) {
            const double* run = lp + lo * (chunk + 1);
            uint32_t j = 0;
            for (len = chunk - 1; len > 0;) {   // the run's last value exceeds r
                const uint32_t half = len >> 1;
                if (__dadd_rn(O, run[j + half]) > r) len = half;
                else j += half + 1, len -= half + 1;
            }
            res = b * bsize + (uint64_t(lo) << lg) + j;
        }
        out[first + q] = res;
    }
}

static size_t staged_smem(uint32_t nthr, uint32_t chunk) { return (size_t(nthr) * chunk + nthr) * sizeof(double); }
static size_t g_staged_smem = 0;   // dynamic LDS the staged sampling kernels may use

hipError_t init_sample_kernels()
{
    // the largest staged block: 2^14 amplitudes over 256 threads (the kernels
    // also use a little static LDS, so ask for exactly this)
    const size_t want = staged_smem(256, 64);
    g_staged_smem = 0;
    if (want > sweep_smem_limit()) return hipSuccess;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_block_totals_staged),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(want)) == hipSuccess &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sample_staged),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(want)) == hipSuccess)
        g_staged_smem = want;
    (void)hipGetLastError();
    return hipSuccess;
}

static uint32_t log2_u32(uint32_t v)
{
    uint32_t l = 0;
    while ((1u << l) < v) l++;
    return l;
}

hipError_t launch_block_totals(hipStream_t st, const c64* s, uint64_t nblocks, uint32_t nthr,
                               uint32_t chunk, double* totals)
{
    const size_t smem = staged_smem(nthr, chunk);
    const bool staged = smem <= g_staged_smem;
    for (uint64_t b0 = 0; b0 < nblocks; b0 += (1ull << 30)) {
        const uint64_t cnt = nblocks - b0 < (1ull << 30) ? nblocks - b0 : (1ull << 30);
        if (staged)
            hipLaunchKernelGGL(k_block_totals_staged, dim3(uint32_t(cnt)), dim3(nthr), smem, st,
                               s + b0 * uint64_t(nthr) * chunk, log2_u32(chunk), totals + b0);
        else
            hipLaunchKernelGGL(k_block_totals, dim3(uint32_t(cnt)), dim3(nthr), 0, st,
                               s + b0 * uint64_t(nthr) * chunk, chunk, totals + b0);
    }
    return hipGetLastError();
}

hipError_t launch_sample(hipStream_t st, const c64* s, uint32_t nthr, uint32_t chunk,
                         const uint64_t* jobs, uint32_t njobs, const double* offsets,
                         const double* draws, uint64_t* out)
{
    if (njobs == 0) return hipSuccess;
    const size_t smem = staged_smem(nthr, chunk);
    if (smem <= g_staged_smem)
        hipLaunchKernelGGL(k_sample_staged, dim3(njobs), dim3(nthr), smem, st, s, log2_u32(chunk), jobs, offsets,
                           draws, out);
    else
        hipLaunchKernelGGL(k_sample, dim3(njobs), dim3(nthr), 0, st, s, chunk, jobs, offsets, draws, out);
    return hipGetLastError();
}

// ------------------------------------------------- Pauli sums of one state

template <int M>
__global__ void __launch_bounds__(kPauliThreads, 4)
k_pauli(const c64* __restrict__ psi, c64* __restrict__ lam, uint64_t n_tiles, const PauliPass P, int accumulate,
        const PauliGroup* __restrict__ groups, const PauliTerm* __restrict__ terms, double* __restrict__ partials,
        c64* __restrict__ copy)
{
    extern __shared__ __align__(16) unsigned char smem[];
    c64* tl = reinterpret_cast<c64*>(smem);
    const uint32_t tid = threadIdx.x, nt = blockDim.x;   // nt = 512, or 2^k < 512 with M = 1
    uint64_t toff = 0;
#pragma unroll
    for (int b = 0; b < kPauliThreadBits; b++) toff |= uint64_t((tid >> b) & 1u) << P.pos[b];   // bits >= k of tid are 0
    uint64_t col[M];
#pragma unroll
    for (int j = 0; j < M; j++) col[j] = P.col[j];
    double acc = 0.0;
    for (uint64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const uint64_t yb = deposit_bits(tile, P.extmask) | toff;
#pragma unroll
        for (int j = 0; j < M; j++) {
            const c64 v = psi[yb | col[j]];
            tl[tid + nt * j] = v;
            if (copy) copy[yb | col[j]] = v;
        }
        __syncthreads();
        c64 l[M];
        pauli_groups<M, true>(l, tl, psi, yb, col, tid, nt, nt * M, groups, terms, P.begin, P.flat_end, P.tile_end,
                              P.end);
#pragma unroll
        for (int j = 0; j < M; j++) {
            const c64 v = tl[tid + nt * j];
            acc += v.re * l[j].re + v.im * l[j].im;
        }
        if (lam) {
            if (accumulate)
#pragma unroll
                for (int j = 0; j < M; j++) l[j] = cadd(l[j], lam[yb | col[j]]);
#pragma unroll
            for (int j = 0; j < M; j++) lam[yb | col[j]] = l[j];
        }
        __syncthreads();
    }
    double* red = reinterpret_cast<double*>(smem);
    red[tid] = acc;
    __syncthreads();
    for (uint32_t s = nt / 2; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    if (tid == 0) partials[blockIdx.x] = red[0];
}

uint32_t pauli_grid(uint64_t dim, const PauliPass& pass)
{
    const uint64_t g = dim >> pass.k;
    return g > 2048 ? 2048 : uint32_t(g);
}

hipError_t launch_pauli(hipStream_t st, const c64* psi, c64* lam, uint64_t dim, const PauliPass& pass,
                        bool accumulate, const PauliGroup* groups, const PauliTerm* terms, double* partials,
                        c64* copy)
{
    auto* fn = pass.k == 12 ? &k_pauli<8> : pass.k == 10 ? &k_pauli<2> : pass.k <= 9 ? &k_pauli<1> : nullptr;
    if (!fn) return hipErrorInvalidValue;
    const uint32_t nt = pass.k < 9 ? 1u << pass.k : uint32_t(kPauliThreads);
    hipLaunchKernelGGL(fn, dim3(pauli_grid(dim, pass)), dim3(nt), size_t(16) << pass.k, st, psi, lam, dim >> pass.k,
                       pass, int(accumulate), groups, terms, partials, copy);
    return hipGetLastError();
}

// Sum of per-tile gradient partials, one thread per accumulator (fixed order).
// ------------------------------------------------------- segment sums
//
// dst[seg.dst] = sum of src[seg.src .. seg.src + seg.len): one workgroup per
// segment; thread t adds elements t, t + 256, ... in order, then a fixed
// tree over the threads -- the same order on every run.

__global__ void __launch_bounds__(kThreads)
k_sum_segments(const double* __restrict__ src, const SumSegment* __restrict__ segs, double* __restrict__ dst)
{
    __shared__ double red[kThreads];
    const SumSegment g = segs[blockIdx.x];
    double acc = 0.0;
    for (uint64_t i = threadIdx.x; i < g.len; i += blockDim.x) acc += src[g.src + i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) dst[g.dst] = red[0];
}

// Rows of a [rows][len] array: dst[r] = sum of row r (same order as above).
__global__ void __launch_bounds__(kThreads)
k_sum_rows(const double* __restrict__ src, uint64_t len, double* __restrict__ dst)
{
    __shared__ double red[kThreads];
    const double* row = src + uint64_t(blockIdx.x) * len;
    double acc = 0.0;
    for (uint64_t i = threadIdx.x; i < len; i += blockDim.x) acc += row[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) dst[blockIdx.x] = red[0];
}

// ------------------------------------------------------- measurement
//
// P(1) of qubit q: thread t of the grid reads the amplitudes with bit q set
// at pair indices i = t, t + G, ... (G = grid threads; pos1 = i with a 1
// inserted at bit q), four loads in flight, and sums |a|^2 in that order;
// then a fixed tree per workgroup, and one workgroup sums the partials in a
// fixed order.  The same order on every run.

__global__ void __launch_bounds__(kThreads)
k_prob_one(const c64* __restrict__ s, uint64_t half, uint32_t q, double* __restrict__ partials)
{
    __shared__ double red[kThreads];
    const uint64_t G = uint64_t(gridDim.x) * blockDim.x;
    const uint64_t lo = (1ull << q) - 1;
    double acc = 0.0;
    uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i + 3 * G < half; i += 4 * G) {
        c64 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint64_t j = i + u * G;
            v[u] = s[((j & ~lo) << 1) | (1ull << q) | (j & lo)];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) acc += v[u].re * v[u].re + v[u].im * v[u].im;
    }
    for (; i < half; i += G) {
        const c64 v = s[((i & ~lo) << 1) | (1ull << q) | (i & lo)];
        acc += v.re * v.re + v.im * v.im;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

// Density matrix of nh qubits (index row | col << nh): partial sums of
// |Re rho[i, i]| over the rows i with bit q set -- the diagonal entries only
// (2^(nh-1) strided reads), as Measure_GATE of the density-matrix engine
// sums them (svsim_qsharp_noise/svsim_cpu_omp.hpp:1737-1757).
__global__ void __launch_bounds__(kThreads)
k_prob_one_dm(const c64* __restrict__ s, uint32_t nh, uint32_t q, double* __restrict__ partials)
{
    __shared__ double red[kThreads];
    const uint64_t G = uint64_t(gridDim.x) * blockDim.x;
    const uint64_t half = 1ull << (nh - 1);
    const uint64_t lo = (1ull << q) - 1;
    double acc = 0.0;
    for (uint64_t j = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; j < half; j += G) {
        const uint64_t i = ((j & ~lo) << 1) | (1ull << q) | (j & lo);
        acc += fabs(s[(i << nh) | i].re);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

// dm: collapse factors 1/P(1) or 1/(1 - P(1)) (density matrix) instead of
// their square roots (state vector).
__global__ void __launch_bounds__(kThreads)
k_measure_decide(const double* __restrict__ partials, uint32_t nparts, double draw, c64* __restrict__ collapse,
                 MeasureResult* __restrict__ res, int dm)
{
    __shared__ double red[kThreads];
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < nparts; i += blockDim.x) acc += partials[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double p = red[0];
        const bool one = draw < p;
        const double w = one ? p : 1.0 - p;
        const double f = dm ? 1.0 / w : 1.0 / sqrt(w);
        collapse[0] = c64{one ? 0.0 : f, 0.0};
        collapse[1] = c64{one ? f : 0.0, 0.0};
        MeasureResult r;
        r.prob = p;
        r.outcome = one ? 1 : 0;
        r.pad = 0;
        *res = r;
    }
}

uint32_t measure_partials(int n)
{
    const uint64_t half = 1ull << (n - 1);
    const uint64_t g = (half + kThreads * 4 - 1) / (kThreads * 4);
    return uint32_t(g > 2048 ? 2048 : (g < 1 ? 1 : g));
}

hipError_t launch_measure(hipStream_t st, const c64* s, int n, uint32_t q, double draw, double* partials,
                          c64* collapse, MeasureResult* res, int dm_n)
{
    if (dm_n > 0) {
        const uint32_t g = measure_partials(dm_n);
        hipLaunchKernelGGL(k_prob_one_dm, dim3(g), dim3(kThreads), 0, st, s, uint32_t(dm_n), q, partials);
        hipLaunchKernelGGL(k_measure_decide, dim3(1), dim3(kThreads), 0, st, partials, g, draw, collapse, res, 1);
        return hipGetLastError();
    }
    const uint32_t g = measure_partials(n);
    hipLaunchKernelGGL(k_prob_one, dim3(g), dim3(kThreads), 0, st, s, 1ull << (n - 1), q, partials);
    hipLaunchKernelGGL(k_measure_decide, dim3(1), dim3(kThreads), 0, st, partials, g, draw, collapse, res, 0);
    return hipGetLastError();
}

hipError_t launch_sum_segments(hipStream_t st, const double* src, const SumSegment* segs, uint64_t nseg,
                               double* dst)
{
    const uint64_t max_grid = 1ull << 30;
    for (uint64_t s0 = 0; s0 < nseg; s0 += max_grid) {
        const uint32_t cnt = uint32_t(nseg - s0 < max_grid ? nseg - s0 : max_grid);
        hipLaunchKernelGGL(k_sum_segments, dim3(cnt), dim3(kThreads), 0, st, src, segs + s0, dst);
    }
    return hipGetLastError();
}

hipError_t launch_sum_rows(hipStream_t st, const double* src, uint32_t rows, uint64_t len, double* dst)
{
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_rows, dim3(rows), dim3(kThreads), 0, st, src, len, dst);
    return hipGetLastError();
}

}  // namespace svmi
