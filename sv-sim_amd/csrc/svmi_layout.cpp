// svmi_layout.cpp -- register layouts of planned sweeps (host only).
//
// A planned phase says which LDS index y each (group, register) pair is
// gathered from and scattered to, through the tile map (PhaseInfo); the LDS
// itself no longer holds the tile between phases.  Here every phase gets an
// assignment of its group bits to lane and wave bits, and every pair of
// neighbouring phases an exchange: the previous phase's (thread, register)
// writes its amplitude to a slot, the next one's reads the slot of the
// amplitude it wants.
//
// Waves.  An exchange in which every wave only reads what it wrote needs no
// workgroup barrier.  10 of the tile's bits (6 lane, 4 register) belong to a
// wave, so the lane bits of a phase are chosen as the group bits that the
// following phases take as register bits, and the next exchange stays inside
// the waves whenever its register bits are among them.
//
// Slots.  A slot is numbered by its writer's coordinates (lane, register,
// wave): the wave number is the top of the slot number, and the low five bits
// are linear functions chosen so that the first 32 lanes hit 32 different
// slots (of 8 bytes: all 64 banks) on the write and on the read.
//
// Memory.  Loads and stores want the low qubits on the first lanes (256-byte
// segments); where the first or last phase holds more than one of them in
// registers, a phase without ops is put before or after it.
#include "svmi_layout.hpp"

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <utility>

namespace svmi {

namespace {

inline int popc32(uint32_t x) { return __builtin_popcount(x); }
inline uint32_t parity(uint32_t x) { return uint32_t(__builtin_parity(x)); }

constexpr int kMaxBits = 14;       // tile bits, with the state bit of two-state sweeps
constexpr int kBankBits = 5;       // 32 slots of 8 bytes: the 64 LDS banks
constexpr int kLowOnRegs = 1;      // low qubits a load or store may have on register bits

// GF(2) basis by leading bit.
template <class T>
struct SpanOf {
    T b[8 * sizeof(T)] = {};
    static int top(T v) { return 63 - __builtin_clzll(uint64_t(v)); }
    T reduce(T v) const
    {
        while (v) {
            const int t = top(v);
            if (!b[t]) return v;
            v ^= b[t];
        }
        return 0;
    }
    bool has(T v) const { return reduce(v) == 0; }
    bool add(T v)
    {
        v = reduce(v);
        if (!v) return false;
        b[top(v)] = v;
        return true;
    }
};
using Span = SpanOf<uint32_t>;
using Span64 = SpanOf<uint64_t>;

// Columns of the inverse of a GF(2) matrix given by K independent columns.
void invert(const uint32_t* col, int K, uint32_t* inv)
{
    uint32_t v[kMaxBits], e[kMaxBits];   // v = combination e of the columns
    for (int i = 0; i < K; i++) v[i] = col[i], e[i] = 1u << i;
    for (int t = 0; t < K; t++) {
        int p = t;
        while (p < K && !((v[p] >> t) & 1u)) p++;
        if (p == K) throw std::logic_error("layout: columns are not independent");
        std::swap(v[t], v[p]);
        std::swap(e[t], e[p]);
        for (int i = 0; i < K; i++)
            if (i != t && ((v[i] >> t) & 1u)) v[i] ^= v[t], e[i] ^= e[t];
    }
    for (int t = 0; t < K; t++) inv[t] = e[t];
}

uint32_t apply(const uint32_t* col, uint32_t v)
{
    uint32_t o = 0;
    for (; v; v &= v - 1) o ^= col[__builtin_ctz(v)];
    return o;
}

struct Group {            // a group bit of a phase
    uint32_t y;           // its LDS index column
    uint32_t goff, grp;   // tile-local bit, bit of the group number
};

struct Phase {
    uint32_t op_begin = 0, op_end = 0, coef_begin = 0, coef_end = 0, r[4] = {0, 0, 0, 0};
    uint32_t greg[4], gx = 0;       // gather
    uint32_t sreg[4], sx = 0;       // scatter
    Group grp[kMaxBits];
    int order[kMaxBits] = {};       // thread bit i <-> group bit order[i]
    uint32_t inv[kMaxBits];         // y -> (group bits, registers), group bit i <-> bit i, register s <-> bit t + s
};

struct Rng {              // xorshift: the same slots on every run
    uint32_t s = 0x9e3779b9u;
    uint32_t next()
    {
        s ^= s << 13;
        s ^= s >> 17;
        s ^= s << 5;
        return s;
    }
};

struct Builder {
    Program& prog;
    const SweepInfo& sw;
    int K, t, tl, tw, k;
    bool two;
    std::vector<Phase> ph;
    uint32_t finv[kMaxBits];   // y -> tile-local index at the store
    int low;                   // low qubits a memory segment wants on lanes

    Builder(Program& p, const SweepInfo& s) : prog(p), sw(s)
    {
        two = prog.n_states == 2;
        k = int(sw.k);
        K = k + (two ? 1 : 0);
        t = K - kRegBits;
        tl = t < kLaneBits ? t : kLaneBits;
        tw = t - tl;
        low = int(sw.c) < 4 ? int(sw.c) : 4;
        if (tw > kMaxWaveBits || t < 0) throw std::logic_error("layout: tile size");
        for (int i = 0; i < K; i++) finv[i] = 1u << i;
        if (sw.mapped) {
            uint32_t f[kMaxBits];
            for (int i = 0; i < k; i++) f[i] = sw.fcol[i];
            if (two) f[k] = 1u << k;
            invert(f, K, finv);
        }
    }

    void columns(const Phase& p, uint32_t* col) const
    {
        for (int i = 0; i < t; i++) col[i] = p.grp[i].y;
        for (int s = 0; s < kRegBits; s++) col[t + s] = p.sreg[s];
    }

    void take(const PhaseInfo& pi)
    {
        Phase p;
        p.op_begin = pi.op_begin;
        p.op_end = pi.op_end;
        p.coef_begin = pi.coef_begin - sw.coef_base;
        p.coef_end = pi.coef_end - sw.coef_base;
        p.gx = pi.gxor;
        p.sx = pi.sxor;
        uint32_t R = 0;
        for (int s = 0; s < kRegBits; s++) {
            p.r[s] = pi.r[s];
            R |= 1u << pi.r[s];
            p.greg[s] = pi.gcol[s];
            p.sreg[s] = pi.scol[s];
        }
        int gi = 0;
        for (int l = 0; l < k; l++)
            if (!((R >> l) & 1u)) {
                p.grp[gi] = Group{pi.gm[gi], 1u << l, 1u << gi};
                gi++;
            }
        ph.push_back(p);
    }

    // a phase without ops on the columns col[0..K): lanes and waves first, then registers
    void idle(std::vector<Phase>::iterator at, const uint32_t* col)
    {
        Phase p;
        p.op_begin = p.op_end = 0;
        for (int i = 0; i < t; i++) p.grp[i] = Group{col[i], 0u, 0u};
        for (int s = 0; s < kRegBits; s++) p.greg[s] = p.sreg[s] = col[t + s];
        for (int i = 0; i < t; i++) p.order[i] = i;
        uint32_t c[kMaxBits];
        columns(p, c);
        invert(c, K, p.inv);
        ph.insert(at, p);
    }

    // group bits (as a mask) that the vector y uses in phase p
    uint32_t support(const Phase& p, uint32_t y) const { return apply(p.inv, y) & ((1u << t) - 1u); }

    // lanes of phase i from what comes after it: `lanes` already holds fixed ones
    void choose(size_t i, uint32_t lanes)
    {
        Phase& p = ph[i];
        for (size_t q = i + 1; q <= ph.size() && popc32(lanes) < tl; q++) {
            uint32_t want = lanes;
            if (q < ph.size())
                for (int s = 0; s < kRegBits; s++) want |= support(p, ph[q].greg[s]);
            else
                for (int b = 0; b < low; b++) want |= support(p, store_low(b));
            if (popc32(want) > tl) break;
            lanes = want;
        }
        for (int g = 0; g < t && popc32(lanes) < tl; g++) lanes |= 1u << g;
        int n = 0;
        for (int g = 0; g < t; g++)
            if ((lanes >> g) & 1u) p.order[n++] = g;
        for (int g = 0; g < t; g++)
            if (!((lanes >> g) & 1u)) p.order[n++] = g;
    }

    // the LDS index column of tile-local bit b at the store
    uint32_t store_low(int b) const { return sw.mapped ? uint32_t(sw.fcol[b]) : 1u << b; }

    // Puts the lanes whose image under f is in the low qubits first; how many
    // of the low qubits the lanes then hold.
    int low_first(Phase& p, const uint32_t* f) const
    {
        int n = 0;
        for (int i = 0; i < tl; i++)
            if (!(apply(f, p.grp[p.order[i]].y) >> low)) {
                const int v = p.order[i];
                for (int j = i; j > n; j--) p.order[j] = p.order[j - 1];
                p.order[n++] = v;
            }
        return n;
    }

    Span wave_span(const Phase& p, bool scatter) const
    {
        Span s;
        for (int i = 0; i < tl; i++) s.add(p.grp[p.order[i]].y);
        for (int r = 0; r < kRegBits; r++) s.add(scatter ? p.sreg[r] : p.greg[r]);
        return s;
    }

    // Columns of a phase without ops whose tile bits are the vectors f[0..k):
    // the low ones on the first lanes and, if the wave span v consists of such
    // vectors and has the low ones, the rest of it on the other lanes and on
    // the registers, so that the exchange with v's phase stays in the waves.
    void idle_columns(const uint32_t* f, const Span& v, uint32_t* col) const
    {
        const int nreg = kRegBits - (two ? 1 : 0);
        int count = 0;
        for (int b = 0; b < k; b++) count += v.has(f[b]) ? 1 : 0;
        bool inside = count == tl + nreg;
        for (int b = 0; b < low; b++) inside = inside && v.has(f[b]);
        uint32_t used = 0, regs[kRegBits];
        int n = 0, nr = 0;
        for (int b = 0; b < low && b < t; b++) col[n++] = f[b], used |= 1u << b;
        for (int b = k - 1; b >= 0 && nr < nreg; b--)   // registers: the highest bits
            if (!((used >> b) & 1u) && (!inside || v.has(f[b]))) regs[nr++] = f[b], used |= 1u << b;
        for (int pass = 0; pass < 2; pass++)            // lanes of the wave, then the others
            for (int b = 0; b < k; b++)
                if (!((used >> b) & 1u) && (pass == 1 || !inside || v.has(f[b]))) col[n++] = f[b], used |= 1u << b;
        for (int s = 0; s < nr; s++) col[n++] = regs[s];
        if (two) col[n++] = 1u << k;
        if (n != K) throw std::logic_error("layout: idle phase");
    }

    void orders()
    {
        uint32_t unit[kMaxBits], f[kMaxBits], col[kMaxBits];
        for (int i = 0; i < K; i++) unit[i] = 1u << i;
        for (int b = 0; b < k; b++) f[b] = store_low(b);
        const bool large = sw.n_tiles > 1;   // one tile: no memory traffic worth a phase
        size_t first = 0;
        if (ph.empty()) {   // load and store only
            idle_columns(unit, Span(), col);
            idle(ph.begin(), col);
        } else {
            for (Phase& p : ph) {
                uint32_t c[kMaxBits];
                columns(p, c);
                invert(c, K, p.inv);
            }
            // the first phase: lanes that loads want, then what later phases want
            uint32_t lows = 0, all = 0;
            for (int g = 0; g < t; g++)
                if (!(ph[0].grp[g].y >> low)) lows |= 1u << g;
            for (int b = 0; b < low; b++) all |= support(ph[0], 1u << b);
            const bool direct = !large || low - popc32(lows) <= kLowOnRegs;
            const uint32_t want = direct ? lows : all;
            choose(0, popc32(want) <= tl ? want : 0u);
            low_first(ph[0], unit);
            if (!direct) {
                idle_columns(unit, wave_span(ph[0], false), col);
                idle(ph.begin(), col);
                first = 1;
            }
        }
        for (size_t i = first + 1; i < ph.size(); i++) {
            const Span v = wave_span(ph[i - 1], true);
            bool in = true;
            for (int s = 0; s < kRegBits; s++) in = in && v.has(ph[i].greg[s]);
            uint32_t lanes = 0;
            for (int g = 0; in && g < t; g++)
                if (v.has(ph[i].grp[g].y)) lanes |= 1u << g;
            choose(i, popc32(lanes) == tl ? lanes : 0u);
        }
        // the store; a phase that also loads keeps its lanes
        Phase kept = ph.back();
        int held = low_first(ph.back(), finv);
        if (ph.size() == 1 && std::memcmp(kept.order, ph.back().order, sizeof(kept.order)) != 0) {
            ph.back() = kept;
            held = large ? 0 : low;
        }
        if (large && low - held > kLowOnRegs) {
            idle_columns(f, wave_span(ph.back(), true), col);
            idle(ph.end(), col);
        }
    }

    // LDS byte columns of the writer's coordinates (lanes, registers, waves;
    // in units of 8 bytes << 3) such that the first lanes of writer and
    // reader (whose columns in these coordinates are rl) spread over the banks
    void slots(const uint32_t* rl, uint32_t* slot, Rng& rng) const
    {
        const int own = tl + kRegBits;               // coordinates of one wave
        const int nb = own < kBankBits ? own : kBankBits;
        uint32_t fun[kBankBits];
        Span indep;                                   // of the functions, on one wave's coordinates
        // the functions' values on the first lanes, as vectors over those lanes
        Span wv, rv;
        for (int i = 0; i < nb; i++) {
            const int lanes = i < 4 ? (tl < 4 ? tl : 4) : (tl < 5 ? tl : 5);
            if (i == 4) {   // five lanes now: the first four functions again
                wv = Span();
                rv = Span();
                for (int j = 0; j < 4; j++) wv.add(on_lanes(fun[j], nullptr, lanes)), rv.add(on_lanes(fun[j], rl, lanes));
            }
            uint32_t best = 0;
            int best_score = -1;
            for (int tries = 0; tries < 40; tries++) {
                const uint32_t f = rng.next() & ((1u << K) - 1u);
                if (indep.has(f & ((1u << own) - 1u))) continue;
                const int need = i < lanes ? 1 : 0;
                const int w = need && !wv.has(on_lanes(f, nullptr, lanes)) ? 1 : 0;
                const int r = need && !rv.has(on_lanes(f, rl, lanes)) ? 1 : 0;
                if (w + r > best_score) best_score = w + r, best = f;
                if (best_score == 2 * need) break;
            }
            if (best_score < 0)   // no random function was independent: a unit one is
                for (int b = 0; b < own; b++)
                    if (!indep.has(1u << b)) best = 1u << b;
            fun[i] = best;
            indep.add(best & ((1u << own) - 1u));
            wv.add(on_lanes(best, nullptr, lanes));
            rv.add(on_lanes(best, rl, lanes));
        }
        for (int c = 0; c < K; c++) {
            slot[c] = 0;
            for (int i = 0; i < nb; i++) slot[c] |= ((fun[i] >> c) & 1u) << i;
        }
        int pos = nb;
        for (int c = 0; c < own; c++)
            if (indep.add(1u << c)) slot[c] |= 1u << pos++;
        for (int c = own; c < K; c++) slot[c] |= 1u << c;
        for (int c = 0; c < K; c++) slot[c] <<= 3;
    }

    // values of function f on the first lanes (columns rl, or the writer's own lanes)
    static uint32_t on_lanes(uint32_t f, const uint32_t* rl, int lanes)
    {
        if (!rl) return f & ((1u << lanes) - 1u);
        uint32_t v = 0;
        for (int i = 0; i < lanes; i++) v |= parity(f & rl[i]) << i;
        return v;
    }

    uint64_t phys(uint32_t x) const   // tile-local index -> amplitude offset (state bit dropped)
    {
        uint64_t o = 0, tile = ((uint64_t(1) << prog.n) - 1) & ~sw.extmask;
        for (int b = 0; b < k; b++) {
            if ((x >> b) & 1u) o |= tile & (~tile + 1);
            tile &= tile - 1;
        }
        return o;
    }

    void emit(SweepIO& io)
    {
        std::memset(&io, 0, sizeof(io));
        io.ph_begin = uint32_t(prog.lphases.size());
        const Phase &first = ph.front(), &last = ph.back();
        for (int side = 0; side < 2; side++) {
            const Phase& p = side ? last : first;
            const auto to = [&](uint32_t y) { return 16 * phys(side ? apply(finv, y) : y); };
            uint64_t threads = 0, regs = 0;
            for (int i = 0; i < tl; i++) threads |= io.lane[side][i] = to(p.grp[p.order[i]].y);
            io.wave[side][0] = to(side ? p.sx : p.gx);
            for (int v = 1; v < (1 << tw); v++) {
                const int b = __builtin_ctz(v);
                io.wave[side][v] = io.wave[side][v & (v - 1)] ^ to(p.grp[p.order[tl + b]].y);
            }
            for (int v = 0; v < (1 << tw); v++) threads |= io.wave[side][v];
            for (int r = 1; r < kRegs; r++) {
                const int b = __builtin_ctz(r);
                regs |= io.reg[side][r] = io.reg[side][r & (r - 1)] ^ to(side ? p.sreg[b] : p.greg[b]);
            }
            if (!(threads & regs)) io.additive |= kIoAdditive << side;
        }
        // the tile id: low bits on extmask & ~exthi, then exthi, ascending
        int bit = 0;
        for (uint64_t m : {sw.extmask & ~sw.exthi, sw.exthi}) {
            while (m) {
                const int q = __builtin_ctzll(m), len = __builtin_ctzll(~(m >> q));
                if (io.n_runs == uint32_t(kMaxTileRuns)) throw std::logic_error("layout: tile runs");
                TileRun& r = io.run[io.n_runs++];
                r.mask = ((uint64_t(1) << len) - 1) << q;
                r.shl = q > bit ? uint32_t(q - bit) : 0u;
                r.shr = bit > q ? uint32_t(bit - q) : 0u;
                bit += len;
                m &= ~r.mask;
            }
        }
        io.vhi_shift = uint32_t(bit - __builtin_popcountll(sw.exthi));
        Rng rng;
        bool after_cross = false, crossed = false;
        for (size_t i = 0; i < ph.size(); i++) {
            const Phase& p = ph[i];
            LayoutPhase L;
            std::memset(&L, 0, sizeof(L));
            L.op_begin = p.op_begin;
            L.op_end = p.op_end;
            L.coef_begin = p.coef_begin;
            L.coef_n = p.coef_end - p.coef_begin;
            for (int s = 0; s < kRegBits; s++) L.rcol[s] = 1u << p.r[s];
            uint32_t wt[kMaxBits] = {}, rt[kMaxBits] = {}, rc = 0;   // byte columns of the thread bits
            if (i) {
                const Phase& w = ph[i - 1];
                // the reader's columns in the writer's coordinates
                uint32_t pos[kMaxBits];   // the writer's (group, register) coordinates -> lanes | registers | waves
                for (int j = 0; j < t; j++) pos[w.order[j]] = 1u << (j < tl ? j : j + kRegBits);
                for (int s = 0; s < kRegBits; s++) pos[t + s] = 1u << (tl + s);
                const auto coord = [&](uint32_t y) { return apply(pos, apply(w.inv, y)); };
                uint32_t rl[kMaxBits], rr[kRegBits], slot[kMaxBits];
                for (int j = 0; j < t; j++) rl[j] = coord(p.grp[p.order[j]].y);
                for (int s = 0; s < kRegBits; s++) rr[s] = coord(p.greg[s]);
                const uint32_t r0 = coord(p.gx ^ w.sx);
                slots(rl, slot, rng);
                for (int r = 1; r < kRegs; r++) {
                    const int b = __builtin_ctz(r);
                    L.w[r] = L.w[r & (r - 1)] ^ slot[tl + b];
                    L.rd[r] = L.rd[r & (r - 1)] ^ apply(slot, rr[b]);
                }
                for (int j = 0; j < t; j++) {
                    wt[j] = slot[j < tl ? j : j + kRegBits];
                    rt[j] = apply(slot, rl[j]);
                }
                rc = apply(slot, r0);
                // inside the waves: no lane or register of the reader leaves its
                // wave, and wave bit j is the writer's wave bit j
                const uint32_t waves = ~((1u << (tl + kRegBits)) - 1u);
                bool in = (r0 & waves) == 0;
                for (int j = 0; j < t; j++) in = in && (rl[j] & waves) == (j < tl ? 0u : 1u << (j + kRegBits));
                for (int s = 0; s < kRegBits; s++) in = in && (rr[s] & waves) == 0;
                L.flags = (in ? 0u : uint32_t(LPH_CROSS)) | (after_cross ? uint32_t(LPH_GUARD) : 0u);
                after_cross = !in;
                crossed = crossed || !in;
            }
            ThreadCols tc;
            std::memset(&tc, 0, sizeof(tc));
            tc.zero = thread_entry(0, rc, 0, 0);
            for (int j = 0; j < t; j++)
                (j < tl ? tc.lane[j] : tc.wave[j - tl]) =
                    thread_entry(wt[j], rt[j], p.grp[p.order[j]].goff, p.grp[p.order[j]].grp);
            prog.cols.push_back(tc);
            prog.lphases.push_back(L);
        }
        io.ph_end = uint32_t(prog.lphases.size());
        // without an exchange between the waves, every wave must store where it loaded
        Span64 own;
        for (int i = 0; i < tl; i++) own.add(io.lane[0][i]);
        for (int s = 0; s < kRegBits; s++) own.add(io.reg[0][1 << s]);
        bool same = true;
        for (int i = 0; i < tl; i++) same = same && own.has(io.lane[1][i]);
        for (int s = 0; s < kRegBits; s++) same = same && own.has(io.reg[1][1 << s]);
        for (int v = 0; v < (1 << tw); v++) same = same && own.has(io.wave[0][v] ^ io.wave[1][v]);
        io.store_guard = !crossed && !same ? 1u : 0u;
    }
};

}  // namespace

void build_layouts(Program& prog)
{
    prog.io.resize(prog.sweeps.size());
    prog.lphases.clear();
    prog.cols.clear();
    const size_t most = prog.phases.size() + 2 * prog.sweeps.size();
    prog.lphases.reserve(most);
    prog.cols.reserve(most);
    for (size_t i = 0; i < prog.sweeps.size(); i++) {
        Builder b(prog, prog.sweeps[i]);
        b.ph.reserve(b.sw.phase_end - b.sw.phase_begin + 2);
        for (uint32_t p = b.sw.phase_begin; p < b.sw.phase_end; p++) b.take(prog.phases[p]);
        b.orders();
        b.emit(prog.io[i]);
        SweepInfo& sw = prog.sweeps[i];
        sw.stage = 0;
        for (const Phase& p : b.ph) sw.stage = std::max(sw.stage, p.coef_end - p.coef_begin);
    }
}

}  // namespace svmi
