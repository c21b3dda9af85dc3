// circuit_plan.h - how a gate list is cut into passes over tiles (circuit.hip).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

#include "qcsim_amd.h"

namespace qcs {

constexpr int kTileReg = 3;    // register qubits of a round
constexpr int kTileMax = 12;   // tile qubits: 4096 amplitudes, 64 KiB of LDS

struct TileGeo {
    uint32_t t;
    uint8_t pos[kTileMax + 4];  // tile qubits, ascending
};

// Operation codes of a pass's stream: base + register bit, pair or triple.
enum : uint32_t {
    kOpGen1 = 0,    // + J: 2x2 on register bit J (8 reals)
    kOpReal = 4,    // + J: real 2x2 (4 reals): H, Ry
    kOpImag = 8,    // + J: real diagonal, imaginary off-diagonal (r00, i01, i10, r11): Rx
    kOpX = 12,      // + J: exchange
    kOpAnti = 16,   // + J: (m01, m10)
    kOpDiagR = 20,  // + J: (m00, m11) by register bit J
    kOpScale = 24,  // times m0
    kOpNeg = 25,    // sign change
    kOpSwap = 28,   // + pair: exchange
    kOpSwapP = 32,  // + pair: exchange times m0
    kOpZ = 36,      // + set of register bits: times re - i im (even parity) or re + i im (odd)
    kOpGen2 = 44,   // + pair: 4x4 (from here on handled outside the inner loop)
    kOpGen3 = 48,   // 8x8
    kOpRound = 49,  // the thread mask holds the register positions, a byte each
    kOpEnd = 50,
};

// A stream is a list of records: code | words << 16, thread mask | thread
// value << 16, register mask | kPickBit with its tile-index bit, tile-index
// mask, then the matrix entries. An operation applies to the threads whose
// masked bits equal the value, where every masked tile-index bit is 1, and to
// the amplitudes (for exchanges and matrices: the orbits, by their first
// amplitude) in the register mask. With kPickBit the second complex entry
// takes the place of the first where that tile-index bit is 1.
//
// kOpZ applies to every amplitude, by the parity of its register bits, of the
// thread bits in bits 8.. of the register mask and of the tile-index bits in
// the low word of the third real; its factor is in the first two.
//
// The first round is there from the start; kOpRound begins the next one.
// After the end come kTail words that may be read ahead.
constexpr uint32_t kHead = 4;
constexpr uint32_t kTail = 20;
constexpr uint32_t kPickBit = 1u << 24;  // the bit's number at 16..20

// The passes of a gate list, in order. The gates stay the caller's until the
// last step is taken.
class TilePlanner {
  public:
    // nq qubits (at least kTileReg) of amp_bytes each; a pass's stream keeps
    // to stream_bytes
    TilePlanner(const qcs_gate* gates, uint32_t n, uint32_t nq, size_t amp_bytes, size_t stream_bytes);
    TilePlanner(const TilePlanner&) = delete;
    ~TilePlanner();
    // The next step: a pass, whose stream replaces `words`, or with *single
    // set that gate's own launch. False if there is none.
    bool next(TileGeo& geo, std::vector<uint32_t>& words, const qcs_gate** single);
    // Whether the register is one that HBM bounds, not launches.
    bool big() const;

    struct Plan;

  private:
    Plan* p_;
};

// The width, of those from lo to hi (2..5), at whose dense blocks a list that
// the fusion pass takes runs rather than in passes; 0 if passes.
uint32_t blocks_width(const qcs_gate* gates, uint32_t n, uint32_t nq, size_t amp_bytes, size_t stream_bytes, uint32_t lo,
                      uint32_t hi);

}  // namespace qcs
