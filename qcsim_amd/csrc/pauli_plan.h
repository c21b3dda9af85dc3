// pauli_plan.h - which terms of a Pauli sum share a read of the state
// (expect_kernels.hip).
#pragma once

#include <cstddef>
#include <cstdint>
#include <unordered_map>
#include <vector>

namespace qcs {

constexpr int kPtMax = 12;  // tile qubits
constexpr int kPtSlots = 12;
constexpr int kPtTerms = 64;  // terms of a pass
constexpr int kPtBlocks = 256;

struct PauliTile {  // words throughout: the scalar unit loads nothing smaller
    uint32_t t, ns, nt;
    uint32_t im;                   // slots of imaginary parts
    uint32_t pos[kPtMax];          // tile qubits, ascending
    uint64_t tile_bits, step;      // the tile qubits; the grid's size on the qubits outside
    uint32_t x[kPtSlots];          // x mask within the tile
    uint32_t zt[2 * kPtSlots];     // z bits on the tile index; without pairs: from bit 30 on those on the register
                                   // qubits. With pairs one word a slot
    uint32_t first[kPtSlots + 1];  // terms first[j]..first[j+1] are slot j's, from first[ns] on those of x = 0
    uint32_t z[kPtTerms];          // z mask within the tile; without pairs: bit 15 for the slot's second sum
};

// The tile passes of the terms with masks x and z (which stay the caller's) on
// n qubits of amp_bytes each, one after the other.
class PauliPlanner {
  public:
    PauliPlanner(uint32_t n, size_t amp_bytes, uint32_t nterms, const uint64_t* x, const uint64_t* z);
    // The next pass; `terms` are the numbers of its terms in the order of its
    // sums. False if none is left.
    bool next(PauliTile& tile, bool& pairs, std::vector<uint32_t>& terms);

    struct Group {
        uint64_t x;
        std::vector<uint32_t> terms;
    };
    std::vector<Group> wide;  // x masks with passes of their own
    uint32_t t, ntiles, blocks;

  private:
    struct Class {  // terms of one slot
        uint64_t x;
        bool im;
        uint32_t zt;
        size_t group;
        std::vector<uint32_t> terms;
        size_t used;
    };
    bool apart(const Group& g) const;
    bool full() const;
    void choose();
    void geometry(PauliTile& P) const;

    uint32_t n_;
    uint64_t full_, low_;
    const uint64_t* z_;
    std::vector<Group> groups_;      // by x mask, in order of first appearance
    std::vector<size_t> live_;       // those with x != 0 and terms left
    std::vector<uint32_t> diag_;     // terms with x = 0 left, from the last to the first
    uint64_t S_ = 0;                 // the tile's qubits
    std::vector<Class> classes_;     // the terms within S_
    size_t class_ = 0, waiting_ = 0;  // the first class with terms left; how many all have
    std::vector<uint32_t> inner_, outer_;  // without pairs: diag_ by z mask, likewise
    size_t sums_ = 0;                // of outer_ a pass
};

}  // namespace qcs
