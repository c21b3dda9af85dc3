// pauli_plan.cpp - cutting the terms of a Pauli sum into passes (host).
//
// A pass takes terms whose x masks lie in its tile, as many slots of them as
// it has. Terms are grouped by x mask once; tile qubits are chosen for the
// masks left and kept while the terms within them fill whole passes, so that a
// plan takes time in proportion to the terms, plus the masks times the choices
// (20 qubits, 30000 terms on 1888 masks: 10 ms; with the masks gathered anew
// from all terms for each pass 2.7 s).
#include "pauli_plan.h"

#include <algorithm>
#include <set>

namespace qcs {

static int popc(uint64_t x) { return __builtin_popcountll(x); }

// The qubits of the next tile: the lowest ones, for whole memory lines, then
// the x masks that need the fewest more, in order of first appearance.
static uint64_t pauli_tile_qubits(const std::vector<uint64_t>& xs, uint64_t low, uint32_t n, uint32_t t) {
    uint64_t S = low;
    for (;;) {
        uint64_t best = 0;
        int need = 64;
        for (const uint64_t x : xs) {
            const int more = popc(x & ~S);
            if (more && more < need && more + popc(S) <= int(t)) {
                need = more;
                best = x;
            }
        }
        if (!best) break;
        S |= best;
    }
    for (uint32_t q = 0; q < n && popc(S) < int(t); ++q) S |= 1ull << q;
    return S;
}

// bits of m at the set bits of S, packed
static uint32_t pack_bits(uint64_t m, uint64_t S) {
    uint32_t v = 0, i = 0;
    for (; S; S &= S - 1, ++i) v |= uint32_t(m >> __builtin_ctzll(S) & 1) << i;
    return v;
}

PauliPlanner::PauliPlanner(uint32_t n, size_t amp_bytes, uint32_t nterms, const uint64_t* x, const uint64_t* z)
    : t(std::max<uint32_t>(2, std::min<uint32_t>(n, kPtMax))),
      ntiles(n > t ? 1u << (n - t) : 1),
      blocks(std::min<uint32_t>(ntiles, kPtBlocks)),
      n_(n),
      full_((1ull << n) - 1),
      low_((1ull << std::min<uint32_t>(n, amp_bytes == 16 ? 3 : 4)) - 1),
      z_(z) {
    std::unordered_map<uint64_t, size_t> at;
    for (uint32_t i = 0; i < nterms; ++i) {
        if (!x[i]) {
            diag_.push_back(i);
            continue;
        }
        const auto p = at.emplace(x[i], groups_.size());
        if (p.second) groups_.push_back(Group{x[i], {}});
        groups_[p.first->second].terms.push_back(i);
    }
    std::reverse(diag_.begin(), diag_.end());
    const bool big = (amp_bytes << n) > size_t(256) << 20;
    for (size_t g = 0; g < groups_.size(); ++g) {
        if (popc(groups_[g].x | low_) <= int(t) && !(big && apart(groups_[g])))
            live_.push_back(g);
        else
            wide.push_back(std::move(groups_[g]));
    }
}

// In units of one read of the state, a slot of a tile pass costs a twelfth
// of the pass and 0.05 for its trips to LDS, and a pass of k_pauli 1.25 for
// 16 terms of one x mask. So an x mask whose terms share few slots (z masks
// all over the register) is faster apart, where reading counts (30 qubits,
// 32 random z masks with one x mask: 10.5 ms in tile passes, 5.9 apart).
bool PauliPlanner::apart(const Group& g) const {
    constexpr size_t kApart = 10;  // slots that cost more than a pass of k_pauli
    if (g.terms.size() < kApart) return false;
    const uint64_t S = pauli_tile_qubits({g.x}, low_, n_, t);
    std::set<std::pair<uint64_t, int>> slots;
    for (const uint32_t i : g.terms) slots.insert({z_[i] & full_ & ~S, popc(g.x & z_[i]) & 1});
    return (1.0 / kPtSlots + 0.05) * double(slots.size()) > 1.25 * double((g.terms.size() + 15) / 16);
}

// Whether what is left within the tile fills a pass, or nothing is left outside it.
bool PauliPlanner::full() const {
    return classes_.size() - class_ >= size_t(kPtSlots) || waiting_ >= size_t(kPtTerms) || !inner_.empty() ||
           !outer_.empty();
}

// The next tile's qubits, and the terms within them; without x masks left, the
// terms with x = 0.
void PauliPlanner::choose() {
    for (; class_ < classes_.size(); ++class_) {
        Class& c = classes_[class_];
        auto& g = groups_[c.group].terms;
        g.insert(g.end(), c.terms.begin() + c.used, c.terms.end());
    }
    classes_.clear();
    class_ = waiting_ = 0;
    live_.erase(std::remove_if(live_.begin(), live_.end(), [&](size_t g) { return groups_[g].terms.empty(); }),
                live_.end());
    constexpr size_t kLook = 256;  // masks that have a say
    std::vector<uint64_t> xs;
    for (size_t k = 0; k < live_.size() && k < kLook; ++k) xs.push_back(groups_[live_[k]].x);
    S_ = n_ < t ? 3 : pauli_tile_qubits(xs, low_, n_, t);
    if (live_.empty()) {
        // Passes of even size: a sum takes its time, of which the reads hide a part
        for (const uint32_t i : diag_) (z_[i] & full_ & ~S_ ? outer_ : inner_).push_back(i);
        diag_.clear();
        const size_t k = outer_.size(), all = k + inner_.size();
        const size_t passes = std::max((k + 2 * kPtSlots - 1) / (2 * kPtSlots), (all + kPtTerms - 1) / kPtTerms);
        sums_ = passes ? (k + passes - 1) / passes : 0;
        return;
    }
    std::unordered_map<uint64_t, size_t> slot;
    for (const size_t k : live_) {
        Group& g = groups_[k];
        if (g.x & ~S_) continue;
        slot.clear();
        for (const uint32_t i : g.terms) {
            const bool im = popc(g.x & z_[i]) & 1;
            const uint32_t zt = pack_bits(z_[i], full_ & ~S_);
            const auto p = slot.emplace(uint64_t(zt) << 1 | im, classes_.size());
            if (p.second) classes_.push_back(Class{g.x, im, zt, k, {}, 0});
            classes_[p.first->second].terms.push_back(i);
        }
        waiting_ += g.terms.size();
        g.terms.clear();
    }
}

void PauliPlanner::geometry(PauliTile& P) const {
    P = PauliTile{};
    P.t = t;
    P.tile_bits = S_;
    P.step = blocks;
    uint32_t i = 0;
    for (uint64_t m = S_; m; m &= m - 1) P.pos[i++] = uint32_t(__builtin_ctzll(m));
    for (i = 0; i < t; ++i) {
        const uint64_t below = (1ull << P.pos[i]) - 1;
        P.step = ((P.step & ~below) << 1) | (P.step & below);
    }
}

bool PauliPlanner::next(PauliTile& P, bool& pairs, std::vector<uint32_t>& terms) {
    if (!full()) choose();
    geometry(P);
    terms.clear();
    constexpr uint32_t most = kPtTerms;
    auto put = [&](uint32_t i, uint32_t z) {
        terms.push_back(i);
        P.z[P.nt++] = z;
    };
    pairs = class_ < classes_.size();
    if (pairs) {
        for (; class_ < classes_.size() && P.ns < uint32_t(kPtSlots) && P.nt < most; ++P.ns) {
            Class& c = classes_[class_];
            P.x[P.ns] = pack_bits(c.x, S_);
            P.zt[P.ns] = c.zt;
            P.im |= uint32_t(c.im) << P.ns;
            P.first[P.ns] = P.nt;
            for (; c.used < c.terms.size() && P.nt < most; --waiting_) {
                const uint32_t i = c.terms[c.used++];
                put(i, pack_bits(z_[i], S_));
            }
            if (c.used == c.terms.size()) ++class_;
        }
        P.first[P.ns] = P.nt;
        // terms with x = 0 and z in the tile cost such a pass nothing
        constexpr size_t kLook = 1024;
        const size_t from = diag_.size() - std::min(diag_.size(), kLook);
        std::vector<uint32_t> stay;
        for (size_t k = diag_.size(); k-- > from;) {
            const uint32_t i = diag_[k];
            if (P.nt < most && !(z_[i] & full_ & ~S_))
                put(i, pack_bits(z_[i], S_));
            else
                stay.push_back(i);
        }
        diag_.resize(from);
        diag_.insert(diag_.end(), stay.rbegin(), stay.rend());
    } else {
        const uint32_t top = t - 2;
        for (uint32_t h = 0; h < sums_ && !outer_.empty() && P.nt < most; ++h) {
            const uint32_t i = outer_.back(), zl = pack_bits(z_[i], S_);
            outer_.pop_back();
            if (!(h & 1)) P.first[P.ns++] = P.nt;
            P.zt[h] = pack_bits(z_[i], full_ & ~S_) | (zl >> top) << 30;
            put(i, zl | (h & 1) << 15);
        }
        P.first[P.ns] = P.nt;
        for (; !inner_.empty() && P.nt < most; inner_.pop_back()) put(inner_.back(), pack_bits(z_[inner_.back()], S_));
    }
    return P.nt > 0;
}

}  // namespace qcs
