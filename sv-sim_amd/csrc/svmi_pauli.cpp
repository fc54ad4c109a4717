// svmi_pauli.cpp -- grouping and tiling of Pauli sums (host only).
//
// (H psi)[y] needs psi at y ^ xmask for every distinct X mask.  Read straight
// from memory that is one pass over the state per mask.  Here a pass stages
// tiles of 12 qubits in LDS and serves every mask inside them from there: the
// first pass has the 12 lowest qubits, and masks of higher qubits get passes
// with the 4 lowest qubits (for 256-byte segments) and 8 others, if they
// share enough of them.  An Ising sum at 28 qubits takes 3 passes instead of
// 29 reads.
#include "svmi_pauli.hpp"

#include <algorithm>
#include <cstring>
#include <numeric>

namespace svmi {

namespace {

void set_tile(PauliPass& p, uint64_t tile, int n)
{
    std::memset(&p, 0, sizeof(p));
    for (int q = 0; q < n; q++)
        if ((tile >> q) & 1) p.pos[p.k++] = uint32_t(q);
    p.extmask = ((uint64_t(1) << n) - 1) & ~tile;
    const int jb = std::max(0, int(p.k) - kPauliThreadBits);
    for (int j = 0; j < (1 << jb); j++)
        for (int b = 0; b < jb; b++)
            if ((j >> b) & 1) p.col[j] |= uint64_t(1) << p.pos[kPauliThreadBits + b];
}

// Terms grouped by X mask (ascending, terms in input order).
void group_terms(const svmi_pauli_term* terms, size_t n_terms, std::vector<PauliGroup>& groups,
                 std::vector<PauliTerm>& out)
{
    std::vector<size_t> idx(n_terms);
    std::iota(idx.begin(), idx.end(), 0);
    std::stable_sort(idx.begin(), idx.end(), [&](size_t a, size_t b) { return terms[a].xmask < terms[b].xmask; });
    groups.clear();
    out.clear();
    for (size_t i : idx) {
        const svmi_pauli_term& t = terms[i];
        if (groups.empty() || groups.back().xmask != t.xmask)
            groups.push_back(PauliGroup{t.xmask, uint32_t(out.size()), uint32_t(out.size()), 0, 0});
        // i^ny, times (-1)^ny for the sign taken at y instead of y ^ xmask: (-i)^ny
        const int ny = __builtin_popcountll(t.xmask & t.zmask) & 3;
        const double re[4] = {1, 0, -1, 0}, im[4] = {0, -1, 0, 1};
        PauliTerm o;
        std::memset(&o, 0, sizeof(o));
        o.zmask = t.zmask;
        o.cre = t.coeff * re[ny];
        o.cim = t.coeff * im[ny];
        out.push_back(o);
        PauliGroup& g = groups.back();
        g.end = uint32_t(out.size());
        if (o.cim != 0.0) g.imag = 1;
        g.flat = g.end == g.begin + 1 && t.zmask == 0 ? 1u : 0u;
    }
}

// Every seed looks at all masks after it: the search stays linear in them.
constexpr int kMaxFailedSeeds = 256;

}  // namespace

void plan_pauli(const svmi_pauli_term* terms, size_t n_terms, int n, int tile_qubits, bool lam, int max_passes,
                PauliPlan& plan)
{
    std::vector<PauliGroup> g;
    std::vector<PauliTerm> t;
    group_terms(terms, n_terms, g, t);
    plan.groups.clear();
    plan.terms.clear();
    plan.passes.clear();
    const int k = std::min(tile_qubits, n);
    const uint64_t low = (uint64_t(1) << k) - 1, keep = (uint64_t(1) << std::min(kPauliLow, k)) - 1;
    // a further pass reads psi once (and reads and writes lam), a mask left to
    // the first pass reads psi once more
    const size_t worth = lam ? 4 : 2;
    std::vector<uint64_t> tiles{low};
    std::vector<int> pass_of(g.size(), -1);   // -1: read from memory in the first pass
    for (size_t i = 0; i < g.size(); i++)
        if (!(g[i].xmask & ~low)) pass_of[i] = 0;
    int failed = 0;   // seeds that found too few masks to share a tile with
    for (size_t s = 0; s < g.size() && tiles.size() < size_t(max_passes) && failed < kMaxFailedSeeds; s++) {
        if (pass_of[s] >= 0 || __builtin_popcountll(keep | g[s].xmask) > k) continue;
        uint64_t tile = keep;
        size_t covered = 0;
        for (size_t i = s; i < g.size(); i++)
            if (pass_of[i] < 0 && __builtin_popcountll(tile | g[i].xmask) <= k) {
                tile |= g[i].xmask;
                covered++;
            }
        if (covered < worth) {
            failed++;
            continue;
        }
        for (int q = 0; q < n && __builtin_popcountll(tile) < k; q++) tile |= uint64_t(1) << q;
        for (size_t i = 0; i < g.size(); i++)
            if (pass_of[i] < 0 && !(g[i].xmask & ~tile)) pass_of[i] = int(tiles.size());
        tiles.push_back(tile);
    }
    auto add_group = [&](size_t i, const PauliPass& p, bool local) {
        PauliGroup G = g[i];
        if (local) {
            G.xmask = 0;
            for (uint32_t b = 0; b < p.k; b++) G.xmask |= ((g[i].xmask >> p.pos[b]) & 1) << b;
        }
        G.begin = uint32_t(plan.terms.size());
        for (uint32_t e = g[i].begin; e < g[i].end; e++) {
            PauliTerm o = t[e];
            o.jsign = 0;
            for (uint32_t j = 0; j < uint32_t(kPauliRegs); j++)
                o.jsign |= uint32_t(__builtin_popcountll(p.col[j] & o.zmask) & 1) << j;
            plan.terms.push_back(o);
        }
        G.end = uint32_t(plan.terms.size());
        std::stable_sort(plan.terms.begin() + G.begin, plan.terms.end(),
                         [](const PauliTerm& a, const PauliTerm& b) { return a.jsign < b.jsign; });
        for (uint32_t e = G.begin; e < G.end; e++)
            plan.terms[e].last = e + 1 == G.end || plan.terms[e + 1].jsign != plan.terms[e].jsign ? 1u : 0u;
        plan.groups.push_back(G);
    };
    for (size_t ps = 0; ps < tiles.size(); ps++) {
        PauliPass p;
        set_tile(p, tiles[ps], n);
        p.begin = uint32_t(plan.groups.size());
        for (uint32_t flat : {1u, 0u}) {
            for (size_t i = 0; i < g.size(); i++)
                if (pass_of[i] == int(ps) && g[i].flat == flat) add_group(i, p, true);
            if (flat) p.flat_end = uint32_t(plan.groups.size());
        }
        p.tile_end = uint32_t(plan.groups.size());
        for (size_t i = 0; ps == 0 && i < g.size(); i++)
            if (pass_of[i] < 0) add_group(i, p, false);
        p.end = uint32_t(plan.groups.size());
        plan.passes.push_back(p);
    }
}

void plan_pauli_state(const svmi_pauli_term* terms, size_t n_terms, int n, bool lam, PauliPlan& plan)
{
    // 12-qubit tiles need 20 qubits for a workgroup on every CU; below, smaller
    // tiles (2 or 1 amplitudes per thread) keep the chip busy.  States of up to
    // 21 qubits (32 MiB) stay in the last-level cache, where reading psi once
    // more for a mask costs less than a pass: one pass / several, 50 random
    // masks at 14 qubits 61 / 100 us, Heisenberg chain of 18 qubits 47 / 54.
    const int k = n >= 20 ? kPauliTileQubits : n >= 18 ? 10 : std::min(n, 8);
    const int passes = n >= 22 ? kMaxPauliPasses : 1;
    plan_pauli(terms, n_terms, n, k, lam, passes, plan);
    if (k < kPauliTileQubits) return;
    // Where few masks lie in a tile, the reads from memory want more workgroups
    // on a CU than the LDS of 12-qubit tiles lets in.  12 / 10 qubits: 50 random
    // masks at 24 qubits (none in a tile) 2.07 / 1.82 ms, all masks of 23 of 24
    // qubits 829 / 601 us; 1191 masks of 4 random qubits at 20 (a fifth in a
    // tile) 1.88 / 2.05 ms.
    size_t in_tile = 0, read = 0;
    for (const PauliPass& p : plan.passes) in_tile += p.tile_end - p.begin, read += p.end - p.tile_end;
    if (read > 8 * in_tile) plan_pauli(terms, n_terms, n, 10, lam, passes, plan);
}

}  // namespace svmi
