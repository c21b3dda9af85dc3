// Runs the passes that circuit_plan.cpp makes on a state in host memory: what
// each operation of a pass's stream does, stated in C++ (on the device it is
// one statement of assembly). For tests/test_circuit_plan.py.
#include <complex>
#include <cstring>
#include <utility>
#include <vector>

#include "../../qcsim_amd/csrc/circuit_plan.h"

namespace qcs {
int set_error(int code, const char*, ...) { return code; }  // fusion.cpp's
}  // namespace qcs
using namespace qcs;
typedef std::complex<double> Amp;

static uint32_t zero_at(uint32_t x, uint32_t p) {
    const uint32_t low = (1u << p) - 1;
    return (x & ~low) << 1 | (x & low);
}

static bool odd(uint32_t x) { return __builtin_popcount(x) & 1; }

// One operation on the eight amplitudes of a thread.
static void apply(Amp (&a)[8], uint32_t code, uint32_t mask, uint32_t blk, const double* body, uint32_t tid, uint32_t tile) {
    double m[128];
    std::memcpy(m, body, sizeof m);
    auto at = [&](int i) { return Amp(m[2 * i], m[2 * i + 1]); };
    if (code >= kOpZ && code < kOpGen2) {
        uint64_t zt;
        std::memcpy(&zt, &m[2], sizeof zt);
        for (uint32_t i = 0; i < 8; ++i)
            a[i] *= Amp(m[0], odd(i & (code - kOpZ)) ^ odd(tid & mask >> 8) ^ odd(tile & uint32_t(zt)) ? m[1] : -m[1]);
        return;
    }
    if ((tile & blk) != blk) return;
    const Amp first = (mask & kPickBit) && (tile >> (mask >> 16 & 31) & 1) ? at(1) : at(0);
    if (code >= kOpGen2) {
        const int D = code < kOpGen3 ? 4 : 8, A = code == kOpGen2 + 2, B = code == kOpGen2 ? 1 : 2;
        for (int i = 0; i < (D == 4 ? 8 : 1); ++i) {
            if (D == 4 && ((i >> A & 1) || (i >> B & 1) || !(mask >> i & 1))) continue;
            Amp x[8], y[8];
            auto idx = [&](int r) { return D == 8 ? r : i | (r & 1) << A | (r >> 1) << B; };
            for (int c = 0; c < D; ++c) x[c] = a[idx(c)];
            for (int r = 0; r < D; ++r) {
                y[r] = 0;
                for (int c = 0; c < D; ++c) y[r] += at(r * D + c) * x[c];
            }
            for (int r = 0; r < D; ++r) a[idx(r)] = y[r];
        }
        return;
    }
    const uint32_t J = code & 3;  // register bit, or pair
    for (uint32_t i = 0; i < 8; ++i) {
        if (!(mask >> i & 1)) continue;
        if (code < kOpDiagR) {
            if (i >> J & 1) continue;
            Amp &x = a[i], &y = a[i | 1u << J];
            const Amp p = x, q = y;
            if (code < kOpReal) {
                x = at(0) * p + at(1) * q;
                y = at(2) * p + at(3) * q;
            } else if (code < kOpImag) {
                x = m[0] * p + m[1] * q;
                y = m[2] * p + m[3] * q;
            } else if (code < kOpX) {
                x = m[0] * p + Amp(0, m[1]) * q;
                y = Amp(0, m[2]) * p + m[3] * q;
            } else {
                x = code < kOpAnti ? q : at(0) * q;
                y = code < kOpAnti ? p : at(1) * p;
            }
        } else if (code < kOpScale) {
            a[i] *= i >> J & 1 ? at(1) : at(0);
        } else if (code == kOpScale) {
            a[i] *= first;
        } else if (code == kOpNeg) {
            a[i] = -a[i];
        } else {
            const uint32_t A = J == 2, B = J == 0 ? 1 : 2;
            if ((i >> A & 1) || (i >> B & 1)) continue;
            std::swap(a[i | 1u << A], a[i | 1u << B]);
            if (code >= kOpSwapP) {
                a[i | 1u << A] *= at(0);
                a[i | 1u << B] *= at(0);
            }
        }
    }
}

extern "C" {

void* plan_new(const qcs_gate* gates, uint32_t n, uint32_t nq, uint64_t amp_bytes, uint64_t stream_bytes) {
    return new TilePlanner(gates, n, nq, amp_bytes, stream_bytes);
}

uint32_t plan_width(const qcs_gate* gates, uint32_t n, uint32_t nq, uint64_t amp_bytes, uint64_t stream_bytes, uint32_t lo,
                    uint32_t hi) {
    return blocks_width(gates, n, nq, amp_bytes, stream_bytes, lo, hi);
}

void plan_free(void* p) { delete static_cast<TilePlanner*>(p); }

// The next step: -1 at the end, the number of a gate of `gates` launched by
// itself, or -2 and a pass, of whose stream `bytes` tells the length. With
// `psi` (interleaved, 2^nq amplitudes) the pass is applied to it.
int64_t plan_step(void* plan, const qcs_gate* gates, uint32_t nq, double* psi, uint64_t* bytes) {
    TileGeo geo;
    std::vector<uint32_t> words;
    const qcs_gate* single = nullptr;
    if (!static_cast<TilePlanner*>(plan)->next(geo, words, &single)) return -1;
    if (single) return single - gates;
    *bytes = words.size() * 4;
    if (!psi) return -2;
    Amp* state = reinterpret_cast<Amp*>(psi);
    const uint32_t t = geo.t, threads = 1u << (t - kTileReg);
    words.resize(words.size() + 256, 0);  // apply() takes the longest record's entries
    std::vector<Amp> s(size_t(1) << t);
    std::vector<uint64_t> off(s.size(), 0);
    for (uint32_t i = 0; i < s.size(); ++i)
        for (uint32_t b = 0; b < t; ++b) off[i] |= uint64_t(i >> b & 1) << geo.pos[b];
    for (uint32_t tile = 0; tile < uint32_t(uint64_t(1) << (nq - t)); ++tile) {
        uint64_t base = tile;
        for (uint32_t b = 0; b < t; ++b) {
            const uint64_t low = (uint64_t(1) << geo.pos[b]) - 1;
            base = (base & ~low) << 1 | (base & low);
        }
        for (uint32_t i = 0; i < s.size(); ++i) s[i] = state[base | off[i]];
        uint32_t regs = 0;
        for (uint32_t i = 0; i < uint32_t(kTileReg); ++i) regs |= (t - kTileReg + i) << (8 * i);
        for (const uint32_t* w = words.data(); (w[0] & 0xffff) != kOpEnd; w += w[0] >> 16) {
            const uint32_t code = w[0] & 0xffff;
            if (code == kOpRound) {
                regs = w[1];
                continue;
            }
            double body[128];
            std::memcpy(body, w + kHead, sizeof body);
            for (uint32_t tid = 0; tid < threads; ++tid) {
                if ((tid & (w[1] & 0xffff)) != w[1] >> 16) continue;
                uint32_t first = tid;
                for (int i = 0; i < kTileReg; ++i) first = zero_at(first, regs >> (8 * i) & 255);
                uint32_t idx[8];
                Amp a[8];
                for (uint32_t k = 0; k < 8; ++k) {
                    idx[k] = first;
                    for (int i = 0; i < kTileReg; ++i) idx[k] |= (k >> i & 1) << (regs >> (8 * i) & 255);
                    a[k] = s[idx[k]];
                }
                apply(a, code, w[2], w[3], body, tid, tile);
                for (uint32_t k = 0; k < 8; ++k) s[idx[k]] = a[k];
            }
        }
        for (uint32_t i = 0; i < s.size(); ++i) state[base | off[i]] = s[i];
    }
    return -2;
}
}
