// The planner of pauli_plan.cpp for tests/test_pauli_plan.py.
#include "../../qcsim_amd/csrc/pauli_plan.h"

using namespace qcs;

extern "C" {

void* pauli_new(uint32_t n, uint64_t amp_bytes, uint32_t nterms, const uint64_t* x, const uint64_t* z) {
    return new PauliPlanner(n, amp_bytes, nterms, x, z);
}

void pauli_free(void* p) { delete static_cast<PauliPlanner*>(p); }

// The next pass into `tile`, the numbers of its terms into `terms`: how many,
// plus 1000 if it has pairs; 0 at the end.
uint32_t pauli_step(void* p, PauliTile* tile, uint32_t* terms) {
    bool pairs = false;
    std::vector<uint32_t> t;
    if (!static_cast<PauliPlanner*>(p)->next(*tile, pairs, t)) return 0;
    for (size_t i = 0; i < t.size(); ++i) terms[i] = t[i];
    return uint32_t(t.size()) + (pairs ? 1000 : 0);
}

// Terms with x masks of their own passes, into `terms`.
uint32_t pauli_wide(void* p, uint32_t* terms) {
    uint32_t k = 0;
    for (const auto& g : static_cast<PauliPlanner*>(p)->wide)
        for (const uint32_t i : g.terms) terms[k++] = i;
    return k;
}
}
