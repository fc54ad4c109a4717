// svmi_jit.cpp -- source generation, hipRTC compilation and launch of
// specialised sweep kernels (see svmi_jit.hpp).
#include "svmi_jit.hpp"

#include <hip/hiprtc.h>

#include <chrono>
#include <cstdio>
#include <sstream>
#include <stdexcept>

namespace svmi {

// The engine headers the generated source includes (embedded by build.py).
extern const char* const kJitHeaderNames[];
extern const char* const kJitHeaderText[];
extern const int kJitHeaderCount;

namespace {


// Registers r (0..15) whose register bits satisfy `rsel`, as a list.
std::vector<int> selected(uint32_t rsel)
{
    std::vector<int> v;
    for (int r = 0; r < kRegs; r++)
        if ((rsel >> r) & 1u) v.push_back(r);
    return v;
}

// Tile-local offset of register r in phase ph (the register bits' part).
uint32_t reg_offset(const LayoutPhase& ph, int r)
{
    uint32_t o = 0;
    for (int b = 0; b < kRegBits; b++)
        if ((r >> b) & 1) o |= ph.rcol[b];
    return o;
}

// The variant of a register table over the qubits `emask` outside the tile.
std::string variant(uint64_t emask, const SweepInfo& sw)
{
    if (!emask) return "0u";
    return emask == sw.exthi ? "vhi" : "rtab_variant(" + std::to_string(emask) + "ull, base)";
}

// One op as direct code: the templates of svmi_exec.hpp / svmi_internal.hpp
// with every slot, mask and offset a literal, so no dispatch is compiled.
// Coefficient offsets count from the program's first one.
void emit_state_op(std::ostringstream& o, DOp d, const LayoutPhase& ph, const SweepInfo& sw)
{
    d.h.coef += sw.coef_base;
    const DOpHdr& h = d.h;
    const std::string cond = "(base & " + std::to_string(h.emask) + "ull) == " + std::to_string(h.emask) +
                             "ull && (goff & " + std::to_string(h.gmask) + "u) == " + std::to_string(h.gmask) + "u";
    switch (h.type) {
    case DOP_DENSE: o << "        apply_dense<" << h.smask << ">(a, coef + " << h.coef << ");\n"; return;
    case DOP_X: o << "        apply_x<" << h.s0 << ">(a);\n"; return;
    case DOP_CX: o << "        apply_cx<" << h.s0 << ", " << h.s1 << ">(a);\n"; return;
    case DOP_SWAP: o << "        apply_swap<" << h.s0 << ", " << h.s1 << ">(a);\n"; return;
    case DOP_SRN: o << "        apply_srn<" << h.s0 << ">(a);\n"; return;
    case DOP_LIFT2:
    case DOP_LIFT3:
        o << "        apply_lift<" << h.s0 << ", " << (h.type == DOP_LIFT3 ? "true" : "false") << ">(a, coef["
          << h.coef << "].re, coef[" << h.coef << "].im);\n";
        return;
    case DOP_RTAB:
        o << "        apply_rtab(a, coef + " << h.coef << "u + 16u * " << variant(h.emask, sw) << ");\n";
        return;
    case DOP_ROT:
        if (h.s0)
            o << "        apply_rtab(a, coef + " << (h.coef + 4u) << "u + 16u * " << variant(h.emask, sw) << ");\n";
        for (int sl = 0; sl < kRegBits; sl++)
            if ((h.smask >> sl) & 1u)
                o << "        apply_lift<" << sl << ", " << (((h.s1 >> sl) & 1u) ? "true" : "false") << ">(a, coef["
                  << (h.coef + uint32_t(sl)) << "].re, coef[" << (h.coef + uint32_t(sl)) << "].im);\n";
        return;
    case DOP_CDENSE:
        o << "        if (" << cond << ") apply_cdense<" << h.s0 << ">(a, coef + " << h.coef << ", " << h.rsel
          << "u);\n";
        return;
    case DOP_CPHASE: {
        o << "        if (" << cond << ") {\n            const c64 ph = coef[" << h.coef << "];\n";
        for (int r : selected(h.rsel)) o << "            a[" << r << "] = cmul(a[" << r << "], ph);\n";
        o << "        }\n";
        return;
    }
    case DOP_DIAG: {
        // table index: bit i from qubit i -- outside the tile from the tile
        // base, on a register bit a constant per register, else from goff
        o << "        {\n            const uint32_t ix = 0u";
        for (uint32_t i = 0; i < d.nq; i++) {
            if (d.qloc[i] < 0) o << " | (uint32_t((base >> " << d.qphys[i] << ") & 1u) << " << i << ")";
            else {
                bool reg = false;
                for (int b = 0; b < kRegBits; b++) reg = reg || ph.rcol[b] == 1u << d.qloc[i];
                if (!reg) o << " | (((goff >> " << d.qloc[i] << ") & 1u) << " << i << ")";
            }
        }
        o << ";\n";
        for (int r = 0; r < kRegs; r++) {
            const uint32_t ro = reg_offset(ph, r);
            uint32_t cidx = 0;
            for (uint32_t i = 0; i < d.nq; i++)
                if (d.qloc[i] >= 0 && ((ro >> d.qloc[i]) & 1u)) cidx |= 1u << i;
            o << "            a[" << r << "] = cmul(a[" << r << "], coef[" << h.coef << "u + (ix | " << cidx
              << "u)]);\n";
        }
        o << "        }\n";
        return;
    }
    case DOP_PHASESET: {
        o << "        {\n            const PhaseEntry* pe = reinterpret_cast<const PhaseEntry*>(coef + " << h.coef
          << ");\n            double pr = " << (h.s1 ? "xf[" + std::to_string(h.grad) + "].re" : "1.0")
          << ", pi = " << (h.s1 ? "xf[" + std::to_string(h.grad) + "].im" : "0.0") << ";\n"
          << "#pragma unroll 4\n            for (uint32_t e = 0; e < " << h.s0 << "u; e++) {\n"
          << "                const PhaseEntry E = pe[e];\n"
          << "                if ((base & E.emask) != E.emask) continue;\n"
          << "                const bool on = (goff & E.gmask) == E.gmask;\n"
          << "                const double tr = SVMI_FMA(pr, E.ph_re, -(pi * E.ph_im));\n"
          << "                const double ti = SVMI_FMA(pr, E.ph_im, pi * E.ph_re);\n"
          << "                pr = on ? tr : pr;\n                pi = on ? ti : pi;\n            }\n"
          << "            const c64 ph{pr, pi};\n";
        for (int r : selected(h.rsel)) o << "            a[" << r << "] = cmul(a[" << r << "], ph);\n";
        o << "        }\n";
        return;
    }
    case DOP_PHASETAB: {
        o << "        {\n            c64 ph = " << (h.s1 ? "xf[" + std::to_string(h.grad) + "]" : "c64{1.0, 0.0}")
          << ";\n";
        const bool global = h.gmask == kLaneTabGlobal;   // the lane tables, else in xf
        for (uint32_t j = 0; j < h.s0; j++)
            o << "            ph = cmul(ph, " << (global ? "coef[" : "xf[") << ((global ? h.coef : h.gmask) + 16u * j)
              << "u + ((grp >> " << 4 * j << ") & 15u)]);\n";
        for (int r : selected(h.rsel)) o << "            a[" << r << "] = cmul(a[" << r << "], ph);\n";
        o << "        }\n";
        return;
    }
    default: o << "        #error unsupported op type " << h.type << "\n"; return;
    }
}

// `var` = thread address `thread` XOR the literal `reg`.  `span` holds every bit
// a thread address can have: what the literal shares with it is XORed (a value
// that many registers have in common), the rest added, so that it can become
// the instruction's immediate offset.
std::string address(const char* thread, uint64_t reg, uint64_t span, const char* suffix)
{
    std::string e = thread;
    if (reg & span) e = "(" + e + " ^ " + std::to_string(reg & span) + suffix + ")";
    if (reg & ~span) e += " + " + std::to_string(reg & ~span) + suffix;
    return e;
}

// The thread's byte offset of the sweep's loads (side 0) or stores (1), and
// one line per register.
void emit_io(std::ostringstream& o, const SweepIO& io, int side, uint32_t threads)
{
    uint64_t span = 0;
    const uint32_t lanes = threads < uint32_t(kLaneEntries) ? threads : uint32_t(kLaneEntries);
    o << "    {\n        uint64_t g = base << 4;\n";
    for (int i = 0; i < kLaneBits && (1u << i) < lanes; i++) {
        span |= io.lane[side][i];
        o << "        g ^= (lane & " << (1u << i) << "u) ? " << io.lane[side][i] << "ull : 0ull;\n";
    }
    span |= io.wave[side][0];
    if (io.wave[side][0]) o << "        g ^= " << io.wave[side][0] << "ull;\n";
    for (uint32_t v = 1; v < threads / lanes; v *= 2) {   // XOR-linear in the wave's bits
        const uint64_t col = io.wave[side][v] ^ io.wave[side][0];
        span |= col;
        o << "        g ^= (wave & " << v << "u) ? " << col << "ull : 0ull;\n";
    }
    for (int r = 0; r < kRegs; r++) {
        const std::string at = "AMP(" + address("g", io.reg[side][r], span, "ull") + ")";
        if (side) o << "        " << at << " = a[" << r << "];\n";
        else o << "        { const c64 v = " << at << "; a[" << r << "] = c64{v.re, v.im}; }\n";
        if (r % 4 == 3) o << "        SCHED();\n";
    }
    o << "    }\n";
}

// One phase: the exchange that leads into it (the real parts, then the
// imaginary parts), its ops.
void emit_phase(std::ostringstream& o, const Program& prog, const SweepInfo& sw, uint32_t p, bool first)
{
    const LayoutPhase& L = prog.lphases[p];
    const ThreadCols& tc = prog.cols[p];
    o << "    {\n        const uint64_t te = ltab[" << uint64_t(p) * kLaneEntries << "u + lane] ^ wtab["
      << uint64_t(p) * kWaveEntries << "u + wave];\n";
    if (!first) {
        uint64_t span = tc.zero;
        for (uint64_t c : tc.lane) span |= c;
        for (uint64_t c : tc.wave) span |= c;
        o << "        const uint32_t w = uint32_t(te) & 0xffffu, rd = uint32_t(te) >> 16;\n";
        const char* meet = (L.flags & LPH_CROSS) ? "        __syncthreads();\n" : "        ORDER();\n";
        if (L.flags & LPH_GUARD) o << "        __syncthreads();\n";
        for (const char* part : {"re", "im"}) {
            for (int r = 0; r < kRegs; r++)
                o << "        LDS(" << address("w", L.w[r], span & 0xffffu, "u") << ") = a[" << r << "]." << part
                  << ";\n";
            o << meet;
            for (int r = 0; r < kRegs; r++)
                o << "        a[" << r << "]." << part << " = LDS("
                  << address("rd", L.rd[r], (span >> 16) & 0xffffu, "u") << ");\n";
            if (part[0] == 'r') o << meet;
        }
    }
    o << "        const uint32_t goff = uint32_t(te >> 32) & 0xffffu, grp = uint32_t(te >> 48);\n"
      << "        (void)goff;\n        (void)grp;\n";
    for (uint32_t op = L.op_begin; op < L.op_end; op++) {
        emit_state_op(o, prog.ops[op], L, sw);
        o << "        SCHED();\n";
    }
    o << "    }\n";
}

// The steps of sweep_tile (svmi_kernels.hip) for one sweep, with every
// offset, flag and op a literal: the tile in registers, four waves per SIMD,
// no dispatch and no address arithmetic per register, so that a sweep of a
// QFT runs at the copy rate.  Compiled kernels with the tile in LDS before /
// now: QFT of 27 qubits 5.00 / 4.17 ms (5 sweeps of 4.3 GB: 5.1 TB/s),
// u3 brickwall of 27, 20 layers, 18.3 / 14.7 ms, 20 random layers of 27 35.7 /
// 27.4 ms (with tiles of 13 qubits), QFT of 16 23.9 / 21.4 us.  (Double-buffered persistent kernels that
// fetched the next tile by LDS DMA took 6.2, 22.2 and 39.8 ms.)
void emit_sweep(std::ostringstream& o, const Program& prog, uint32_t i)
{
    const SweepInfo& sw = prog.sweeps[i];
    const SweepIO& io = prog.io[i];
    const uint32_t nt = 1u << (sw.k - kRegBits);
    bool wide = false;   // dense blocks of 3 or 4 qubits need registers for their results
    for (uint32_t op = sw.op_begin; op < sw.op_end; op++)
        wide = wide || (prog.ops[op].h.type == DOP_DENSE && __builtin_popcount(prog.ops[op].h.smask) > 2);
    // second bound: waves per SIMD
    o << "extern \"C\" __global__ void __launch_bounds__(" << nt << ", " << (wide ? 2 : 4) << ")\n"
      << "svmi_jit_" << i << "(c64* __restrict__ s, const c64* __restrict__ coef, const DOp* __restrict__ ops, "
         "const uint64_t* __restrict__ ltab, const uint64_t* __restrict__ wtab, uint64_t tile0)\n{\n"
      << "    __shared__ __align__(16) unsigned char ex[" << (8u << sw.k) << "];\n"
      << "    __shared__ __align__(16) c64 xf[" << (sw.n_xf ? sw.n_xf : 1u) << "];\n"
      << "    const uint32_t tid = threadIdx.x, lane = tid & 63u;\n"
      << "    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);\n"
      << "    const uint64_t tile = tile0 + blockIdx.x;\n    uint64_t base = 0;\n";
    for (uint32_t r = 0; r < io.n_runs; r++)
        o << "    base |= ((tile << " << io.run[r].shl << ") >> " << io.run[r].shr << ") & " << io.run[r].mask
          << "ull;\n";
    o << "    const uint32_t vhi = uint32_t(tile >> " << io.vhi_shift << ");\n    (void)vhi;\n";
    if (sw.n_xf) {   // as tile_factors (svmi_kernels.hip)
        const uint32_t nlt = 16u * sw.n_lt;
        if (nlt)
            o << "    for (uint32_t i = tid; i < " << nlt << "u; i += " << nt << "u) xf[" << (sw.n_xf - nlt)
              << "u + i] = coef[" << (sw.coef_base + sw.lt_coef) << "u + i];\n";
        o << "    const uint64_t xbits = extract_bits(base, " << sw.extmask << "ull);\n"
          << "    for (uint32_t o = " << sw.op_begin << "u + tid; o < " << sw.op_end << "u; o += " << nt << "u) {\n"
          << "        const DOpHdr h = ops[o].h;\n"
          << "        if (has_tile_factor(h)) xf[h.grad] = tile_factor(h, coef + " << sw.coef_base << "u, base, xbits);\n    }\n";
    }
    o << "    c64 a[kRegs];\n";
    emit_io(o, io, 0, nt);
    if (sw.n_xf) o << "    __syncthreads();\n";
    for (uint32_t p = io.ph_begin; p < io.ph_end; p++) emit_phase(o, prog, sw, p, p == io.ph_begin);
    if (io.store_guard) o << "    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)\n    __syncthreads();\n";
    emit_io(o, io, 1, nt);
    o << "}\n\n";
}

struct Rtc {
    hiprtcProgram prog = nullptr;
    ~Rtc()
    {
        if (prog) hiprtcDestroyProgram(&prog);
    }
};

bool compile(const std::string& src, const char* arch, std::vector<char>& code, double* ms, std::string& err)
{
    Rtc r;
    if (hiprtcCreateProgram(&r.prog, src.c_str(), "svmi_jit.hip", kJitHeaderCount,
                            const_cast<const char**>(kJitHeaderText),
                            const_cast<const char**>(kJitHeaderNames)) != HIPRTC_SUCCESS) {
        err = "hiprtcCreateProgram failed";
        return false;
    }
    const std::string a = std::string("--offload-arch=") + arch;
    const char* opts[] = {a.c_str(), "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                          "-packed-fp32-ops", "-mllvm", "-structurizecfg-skip-uniform-regions=true"};
    const auto t0 = std::chrono::steady_clock::now();
    const hiprtcResult rc = hiprtcCompileProgram(r.prog, int(sizeof(opts) / sizeof(opts[0])), opts);
    if (ms) *ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (rc != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(r.prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(r.prog, &log[0]);
        err = std::string("hiprtc: ") + hiprtcGetErrorString(rc) + "\n" + log.substr(0, 2000);
        return false;
    }
    size_t n = 0;
    hiprtcGetCodeSize(r.prog, &n);
    code.resize(n);
    hiprtcGetCode(r.prog, code.data());
    return n > 0;
}

}  // namespace

void JitSweeps::release()
{
    if (module) hipModuleUnload(module);
    module = nullptr;
    fn.clear();
}

std::string jit_source(const Program& prog, std::vector<char>& covered)
{
    covered.assign(prog.sweeps.size(), 0);
    std::ostringstream o;
    o << "#include \"svmi_exec.hpp\"\nusing namespace svmi;\n"
      << "#define AMP(off) (*reinterpret_cast<c64*>(reinterpret_cast<char*>(s) + (off)))\n"
      << "#define LDS(off) (*reinterpret_cast<double*>(ex + (off)))\n"
      << "#define SCHED() __builtin_amdgcn_sched_barrier(0)\n"
      << "#define ORDER() asm volatile(\"\" ::: \"memory\")\n\n";
    if (prog.n_states != 1) return o.str();
    for (uint32_t i = 0; i < prog.sweeps.size(); i++) {
        const SweepInfo& sw = prog.sweeps[i];
        if (sw.k > (prog.n >= kJitLargeQubits ? 13u : 12u)) continue;
        emit_sweep(o, prog, i);
        covered[i] = 1;
    }
    return o.str();
}

size_t jit_compile_only(const Program& prog, const char* arch, double* ms, std::string& err)
{
    std::vector<char> covered, code;
    const std::string src = jit_source(prog, covered);
    if (!compile(src, arch, code, ms, err)) return 0;
    return code.size();
}

bool jit_build(const Program& prog, const char* arch, JitSweeps& out, std::string& err)
{
    out.release();
    std::vector<char> covered, code;
    const std::string src = jit_source(prog, covered);
    bool any = false;
    for (char c : covered) any = any || c;
    if (!any) return false;
    if (!compile(src, arch, code, &out.compile_ms, err)) return false;
    if (hipModuleLoadData(&out.module, code.data()) != hipSuccess) {
        err = "hipModuleLoadData failed";
        out.module = nullptr;
        return false;
    }
    out.fn.assign(prog.sweeps.size(), nullptr);
    for (uint32_t i = 0; i < prog.sweeps.size(); i++) {
        if (!covered[i]) continue;
        const std::string name = "svmi_jit_" + std::to_string(i);
        if (hipModuleGetFunction(&out.fn[i], out.module, name.c_str()) != hipSuccess) {
            err = "hipModuleGetFunction(" + name + ") failed";
            out.release();
            return false;
        }
    }
    return true;
}

hipError_t jit_launch(hipStream_t st, const JitSweeps& j, uint32_t i, const SweepInfo& sw, c64* s,
                      const SweepTables& t)
{
    const uint32_t nt = 1u << (sw.k - kRegBits);
    const uint64_t max_grid = 1ull << 30;
    const c64* coef = t.coef;
    const DOp* ops = t.ops;
    const uint64_t *ltab = t.lane_tab, *wtab = t.wave_tab;
    for (uint64_t t0 = 0; t0 < sw.n_tiles; t0 += max_grid) {
        const uint32_t cnt = uint32_t(sw.n_tiles - t0 < max_grid ? sw.n_tiles - t0 : max_grid);
        uint64_t tile0 = t0;
        void* args[] = {&s, &coef, &ops, &ltab, &wtab, &tile0};
        const hipError_t e = hipModuleLaunchKernel(j.fn[i], cnt, 1, 1, nt, 1, 1, 0, st, args, nullptr);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace svmi
