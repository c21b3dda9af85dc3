// circuit_plan.cpp - cutting a gate list into tile passes (host).
//
// Gates commute when they act diagonally on every qubit they share, so a
// pass takes, in list order, each gate that fits it and commutes with all
// gates left out before it; what is left keeps its order. The gates
// themselves are those of the gate kernels (same traits, same matrix
// entries), applied one by one.
#include "circuit_plan.h"

#include <algorithm>
#include <cstring>
#include <iterator>

namespace qcs {

double fuse_estimate(const qcs_gate* gates, uint32_t n, uint32_t width);

struct hcplx {
    double re, im;
};

struct TileGate {
    uint32_t op;          // kOpGen1, kOpX, ... (base code); kNoTile: not for a tile
    uint32_t nt = 0;      // targets
    uint8_t tq[3];        // in matrix bit order
    uint64_t T = 0;       // qubits acted on other than diagonally
    uint64_t D = 0;       // qubits acted on diagonally
    uint64_t ctrl = 0;    // bits that must be 1
    uint8_t nm = 0;       // matrix entries (complex)
    double f = 1;         // fraction of the state's bytes its own launch moves
    const qcs_gate* src = nullptr;  // null: several gates in one
    const double* mat = nullptr;
    uint32_t dim = 0, b0 = 0;  // matrix dimension, first row and column of its block
};
constexpr uint32_t kNoTile = ~0u;

static hcplx entry(const TileGate& g, uint32_t r, uint32_t c) {
    const double* m = g.mat + 2 * ((g.b0 + r) * g.dim + g.b0 + c);
    return hcplx{m[0], m[1]};
}

static bool is(hcplx z, double re) { return z.re == re && z.im == 0.0; }

// The gate as qcs_apply_gate / qcs_apply_dense dispatches it.
static TileGate tile_gate(const qcs_gate& g) {
    TileGate o;
    const bool dense = (g.flags & QCS_GATE_DENSE) || g.k > 3;
    const uint32_t t = dense ? 0 : g.traits;
    for (uint32_t i = 0; i < g.k && i < 5; ++i) o.T |= 1ull << g.qubits[i];
    o.op = kNoTile;
    if (g.k > 3) return o;
    o.mat = g.mat;
    o.dim = 1u << g.k;
    for (uint32_t i = 0; i < g.k; ++i) o.tq[i] = uint8_t(g.qubits[i]);
    const bool swap = g.k >= 2 && (t & QCS_TRAIT_SWAP);
    if (swap || (g.k == 2 && (t & (QCS_TRAIT_ISWAP | QCS_TRAIT_ISWAPDAG)))) {
        o.op = swap ? kOpSwap : kOpSwapP;
        o.nt = 2;
        o.nm = swap ? 0 : 1;
        o.b0 = t & QCS_TRAIT_ISWAP ? 1 : 0;  // sign of the factor +-i
        o.T = 1ull << g.qubits[0] | 1ull << g.qubits[1];
        o.ctrl = g.k == 3 ? 1ull << g.qubits[2] : 0;
        o.D = o.ctrl;
        o.f = g.k == 3 ? 0.25 : 0.5;
        return o;
    }
    const bool two = g.k == 3 && (t & QCS_TRAIT_CONTROLLED) && (t & QCS_TRAIT_CTRL_Q1);
    const bool one = !two && g.k >= 2 && (t & QCS_TRAIT_CONTROLLED);
    const uint32_t nc = two ? 2 : one ? 1 : 0;
    o.nt = g.k - nc;
    o.b0 = o.dim - (1u << o.nt);
    for (uint32_t i = o.nt; i < g.k; ++i) o.ctrl |= 1ull << g.qubits[i];
    o.D = o.ctrl;
    o.T &= ~o.ctrl;
    o.f = nc == 2 ? 0.25 : nc == 1 ? 0.5 : 1;
    if (o.nt > 1) {
        o.op = o.nt == 2 ? kOpGen2 : kOpGen3;
        o.nm = o.nt == 2 ? 16 : 64;
    } else if (t & QCS_TRAIT_DIAGONAL) {
        const hcplx d0 = entry(o, 0, 0), d1 = entry(o, 1, 1);
        if (is(d0, 1)) {
            o.op = is(d1, -1) ? kOpNeg : kOpScale;
            o.nm = o.op == kOpScale ? 1 : 0;
            o.ctrl |= o.T;
            o.f *= 0.5;
        } else {
            o.op = !nc && d0.re == d1.re && d0.im == -d1.im ? kOpZ : kOpDiagR;
            o.nm = 2;
        }
        o.D |= o.T;
        o.T = 0;
    } else if (t & QCS_TRAIT_ANTIDIAGONAL) {
        o.op = is(entry(o, 0, 1), 1) && is(entry(o, 1, 0), 1) ? kOpX : kOpAnti;
        o.nm = o.op == kOpAnti ? 2 : 0;
    } else {
        const hcplx a = entry(o, 0, 0), b = entry(o, 0, 1), c = entry(o, 1, 0), d = entry(o, 1, 1);
        const bool real = a.im == 0 && b.im == 0 && c.im == 0 && d.im == 0;
        const bool imag = a.im == 0 && b.re == 0 && c.re == 0 && d.im == 0;
        o.op = real ? kOpReal : imag ? kOpImag : kOpGen1;
        o.nm = real || imag ? 2 : 4;
    }
    return o;
}

static int popc(uint64_t x) { return __builtin_popcountll(x); }

// Gates in order, doubly linked, those not placed yet. They are taken in as the
// passes need them: a pass looks no further ahead than its stream has room for
// plus what it may leave out, so that the first pass of a long list goes out as
// soon as that of a short one.
struct TilePlanner::Plan {
    const qcs_gate* gates = nullptr;
    uint32_t count = 0, at = 0;  // of the caller's list; the next one to take in
    std::vector<TileGate> g;
    std::vector<int> next, prev;
    std::vector<uint8_t> waits;         // not placed, and no part of another gate
    std::vector<std::vector<int>> on;   // per qubit, the gates that touch it
    int head = -1, tail = -1;
    uint32_t waiting = 0;
    uint32_t n = 0, t = 0;
    uint64_t all = 0, low = 0;
    bool big = false;
    size_t max_bytes = 0;  // of a pass's stream
    std::vector<int> take;
    std::vector<const TileGate*> local;

    size_t op_bytes(const TileGate& o) const {
        return (kHead * 4 + 16 * o.nm + 15) / 16 * 16 + (!o.T ? 64 : 0);
    }
    void remove(int i) {
        (prev[i] < 0 ? head : next[prev[i]]) = next[i];
        (next[i] < 0 ? tail : prev[next[i]]) = prev[i];
        waits[i] = 0;
        --waiting;
    }
    void add(const qcs_gate& gate);
};
typedef TilePlanner::Plan TilePlan;

// Gates that a pass can see: 48 B of stream each at least, and 6 n + 16 left out.
constexpr uint32_t kAhead = 2048;

// CNOT(c, t) Z CNOT(c, t), with Z = exp(i phi) or its conjugate by the parity
// of qubits that include t, is such a gate too, in the parity that c joins or
// leaves: the Rz between two CNOTs of an Ising step, and the ladders around
// the rotations of Pauli strings. Each such sandwich becomes one gate: the
// same factor on the same amplitude (CNOTs move amplitudes unchanged), and a
// gate that any round can take. The gates that are left stay in order.
void TilePlan::add(const qcs_gate& gate) {
    const TileGate o = tile_gate(gate);
    if (o.op == kOpX && popc(o.ctrl) == 1) {
        const uint32_t c = uint32_t(__builtin_ctzll(o.ctrl));
        auto& ot = on[o.tq[0]];
        auto& oc = on[c];
        const int d = ot.size() > 1 ? ot.back() : -1, x = d >= 0 ? ot[ot.size() - 2] : -1;
        if (d >= 0 && waits[d] && waits[x] && g[x].op == kOpX && g[x].T == o.T && g[x].ctrl == o.ctrl) {
            TileGate& D = g[d];
            const bool has = D.D >> c & 1;
            if (D.op == kOpZ && (has ? oc.size() > 1 && oc.back() == d && oc[oc.size() - 2] == x : oc.back() == x)) {
                // of the two qubits' lists these are the last two entries
                ot.erase(ot.end() - 2);
                oc.erase(oc.end() - (has ? 2 : 1));
                remove(x);
                D.src = nullptr;
                D.D ^= 1ull << c;
                if (has)
                    oc.pop_back();
                else
                    oc.push_back(d);
                return;
            }
        }
    }
    const int i = int(g.size());
    for (uint64_t m = o.T | o.D; m; m &= m - 1) on[__builtin_ctzll(m)].push_back(i);
    g.push_back(o);
    g.back().src = &gate;
    next.push_back(-1);
    prev.push_back(tail);
    (tail < 0 ? head : next[tail]) = i;
    tail = i;
    waits.push_back(1);
    ++waiting;
}

// Gates, in order, that can run inside S before every gate left out: a gate
// left out blocks the qubits it touches, for diagonal action only where it
// acts diagonally itself. Returns their summed worth.
static double tile_scan(const TilePlan& P, uint64_t S, std::vector<int>* take) {
    uint64_t bT = 0, bD = 0;
    double worth = 0;
    size_t bytes = 0;
    int left = 0;
    const int most = int(6 * P.n) + 16;
    for (int i = P.head; i >= 0; i = P.next[i]) {
        const TileGate& o = P.g[i];
        if (!(o.T & (bT | bD | ~S)) && !(o.D & bT) && o.op != kNoTile) {
            bytes += P.op_bytes(o) + 2 * kHead * 4;
            if (bytes > P.max_bytes) break;
            worth += o.f;
            if (take) take->push_back(i);
            continue;
        }
        bT |= o.T;
        bD |= o.D;
        if (!(P.all & ~bT) || ++left > most) break;
    }
    return worth;
}

// The tile qubits of the next pass: the lowest ones, for whole memory lines,
// and then, from several seeds, the qubit most tied to those already chosen
// by the next gates (a gate of two qubits ties them, the less the more gates
// of two qubits either has before it; a gate on one qubit counts for itself).
static uint64_t tile_choose(const TilePlan& P) {
    if (P.n <= P.t) return P.all;
    constexpr float kFade = 0.6f;
    const uint32_t n = P.n;
    std::vector<float> tie(size_t(n) * n, 0.f), self(n, 0.f), fade(n, 1.f);
    uint64_t seeds[6], seen = 0;
    int ns = 0, looked = 0;
    for (int i = P.head; i >= 0 && looked < int(8 * n); i = P.next[i], ++looked) {
        const TileGate& o = P.g[i];
        const uint64_t m = o.T | o.D;
        if (!o.T || o.op == kNoTile) continue;
        float w = 1.f;
        for (uint64_t x = m; x; x &= x - 1) w = std::min(w, fade[__builtin_ctzll(x)]);
        if (popc(m) == 1) {
            self[__builtin_ctzll(m)] += w;
            continue;
        }
        for (uint64_t x = m; x; x &= x - 1) {
            const int q = __builtin_ctzll(x);
            for (uint64_t y = m & ~(1ull << q); y; y &= y - 1) tie[size_t(q) * n + __builtin_ctzll(y)] += w;
            fade[q] = w * kFade;
        }
        if (ns < 6 && !(m & seen) && popc(m | P.low) <= int(P.t)) seeds[ns++] = m;
        seen |= m;
    }
    if (!ns) seeds[ns++] = 0;
    uint64_t best = 0;
    double best_worth = -1;
    std::vector<float> gain(n);
    for (int k = 0; k < ns; ++k) {
        uint64_t S = 0;
        std::copy(self.begin(), self.end(), gain.begin());
        auto add = [&](uint32_t q) {
            S |= 1ull << q;
            for (uint32_t p = 0; p < n; ++p) gain[p] += tie[size_t(q) * n + p];
        };
        for (uint64_t x = P.low | seeds[k]; x; x &= x - 1) add(__builtin_ctzll(x));
        while (popc(S) < int(P.t)) {
            int q = -1;
            for (uint32_t p = 0; p < n; ++p)
                if (!(S >> p & 1) && (q < 0 || gain[p] > gain[q])) q = int(p);
            add(uint32_t(q));
        }
        const double w = tile_scan(P, S, nullptr);
        if (w > best_worth) {
            best_worth = w;
            best = S;
        }
    }
    return best;
}

// Rounds of one pass: the same rule over the pass's gates, R register qubits
// at a time.
struct TileRound {
    uint64_t regs;
    std::vector<int> ops;  // indices into the pass's gates
};

static int round_scan(const std::vector<const TileGate*>& g, const std::vector<int>& rest, uint64_t S,
                      std::vector<int>* take) {
    uint64_t bT = 0, bD = 0, live = S;
    int worth = 0;
    for (const int i : rest) {
        const TileGate& o = *g[i];
        if (!(o.T & (bT | bD | ~S)) && !(o.D & bT)) {
            worth += o.op <= kOpImag ? 2 : o.nt > 1 ? 3 : 1;
            if (take) take->push_back(i);
            continue;
        }
        bT |= o.T;
        bD |= o.D;
        live &= ~(bT | bD);
        if (!take && !live) break;
    }
    return worth;
}

static std::vector<TileRound> tile_rounds(const std::vector<const TileGate*>& g, uint64_t tile, uint64_t top) {
    std::vector<TileRound> out;
    std::vector<int> rest(g.size()), take, keep;
    for (size_t i = 0; i < g.size(); ++i) rest[i] = int(i);
    auto place = [&](uint64_t regs) {
        take.clear();
        round_scan(g, rest, regs, &take);
        keep.clear();
        std::set_difference(rest.begin(), rest.end(), take.begin(), take.end(), std::back_inserter(keep));
        rest.swap(keep);
        out.push_back(TileRound{regs, take});
    };
    place(top);
    while (!rest.empty()) {
        take.clear();
        round_scan(g, rest, top, &take);
        if (take.size() == rest.size()) break;  // the last round takes them
        // seeds: the qubits of the first gates that could run, each completed
        // by the qubit that lets the most gates run
        uint64_t best = 0, bT = 0, bD = 0, tried[8];
        int best_worth = -1, nt = 0;
        for (size_t k = 0; k < rest.size() && nt < 8; ++k) {
            const TileGate& o = *g[rest[k]];
            const bool free = !(o.T & (bT | bD)) && !(o.D & bT);
            bT |= o.T;
            bD |= o.D;
            if (!o.T || !free) {
                if (!o.T && free && best_worth < 0) {  // only diagonal gates so far: any registers do
                    best = top;
                    best_worth = 0;
                }
                if (!(tile & ~bT)) break;
                continue;
            }
            uint64_t seed = o.T;
            for (uint64_t x = o.D & tile; x && popc(seed) < kTileReg; x &= x - 1) seed |= x & -x;
            bool again = false;
            for (int j = 0; j < nt; ++j) again = again || tried[j] == seed;
            if (again) continue;
            tried[nt++] = seed;
            while (popc(seed) < kTileReg) {
                // partners: qubits that the next gates tie to the seed, else any with a gate
                uint64_t cand = 0;
                int looked = 0;
                for (const int i : rest) {
                    const uint64_t m = g[i]->T | g[i]->D;
                    if ((m & seed) && (m & ~seed)) cand |= m;
                    if (++looked > 40) break;
                }
                cand &= tile & ~seed;
                if (!cand) {
                    for (const int i : rest) cand |= g[i]->T & ~seed;
                    cand &= tile;
                }
                if (!cand) cand = tile & ~seed;
                uint64_t grown = 0;
                int w = -1;
                for (uint64_t x = cand; x; x &= x - 1) {
                    const int c = round_scan(g, rest, seed | (x & -x), nullptr);
                    if (c > w) {
                        w = c;
                        grown = seed | (x & -x);
                    }
                }
                seed = grown;
            }
            const int w = round_scan(g, rest, seed, nullptr);
            if (w > best_worth) {
                best_worth = w;
                best = seed;
            }
        }
        place(best);
    }
    if (!rest.empty() || out.back().regs != top) place(top);
    return out;
}

// A pass's stream in words, appended to `out`.
static void tile_emit(const std::vector<const TileGate*>& g, const std::vector<TileRound>& rounds, uint64_t tile,
                      uint32_t n, std::vector<uint32_t>& out) {
    uint8_t local[64], blkbit[64];  // tile position of a qubit; tile-index bit of an outside one
    for (uint32_t q = 0, i = 0, b = 0; q < n; ++q) {
        if (tile >> q & 1)
            local[q] = uint8_t(i++);
        else
            blkbit[q] = uint8_t(b++);
    }
    for (const TileRound& rd : rounds) {
        uint8_t rq[kTileReg];
        uint32_t packed = 0;
        int nr = 0;
        for (uint64_t x = rd.regs; x; x &= x - 1) {
            rq[nr] = uint8_t(__builtin_ctzll(x));
            packed |= uint32_t(local[rq[nr]]) << (8 * nr);
            ++nr;
        }
        if (&rd != &rounds.front()) out.insert(out.end(), {kOpRound | kHead << 16, packed, 0, 0});
        auto regbit = [&](uint32_t q) {
            for (int i = 0; i < kTileReg; ++i)
                if (rq[i] == q) return i;
            return -1;
        };
        auto lanebit = [&](uint32_t q) {
            uint32_t b = local[q];
            for (int i = 0; i < kTileReg; ++i) b -= local[rq[i]] < local[q] ? 1 : 0;
            return b;
        };
        for (const int oi : rd.ops) {
            const TileGate& o = *g[oi];
            uint32_t lane = 0, blk = 0, rmask = 0, rc = 0, code = o.op;
            for (uint64_t x = o.ctrl; x; x &= x - 1) {
                const uint32_t q = uint32_t(__builtin_ctzll(x));
                if (!(tile >> q & 1))
                    blk |= 1u << blkbit[q];
                else if (regbit(q) >= 0)
                    rc |= 1u << regbit(q);
                else
                    lane |= 1u << lanebit(q);
            }
            for (uint32_t i = 0; i < 1u << kTileReg; ++i) rmask |= (i & rc) == rc ? 1u << i : 0;
            double v[128];
            int nv = 0;
            auto put = [&](hcplx z) {
                v[nv++] = z.re;
                v[nv++] = z.im;
            };
            auto record = [&](uint32_t lval) {
                const size_t body = (sizeof(double) * nv + 15) / 16 * 4, at = out.size();
                out.resize(at + kHead + body, 0);
                out[at] = code | uint32_t(kHead + body) << 16;
                out[at + 1] = lane | lval << 16;
                out[at + 2] = rmask;
                out[at + 3] = blk;
                if (nv) std::memcpy(&out[at + kHead], v, sizeof(double) * nv);
                nv = 0;
            };
            if (o.op == kOpGen1) {
                code += uint32_t(regbit(o.tq[0]));
                for (uint32_t r = 0; r < 2; ++r)
                    for (uint32_t c = 0; c < 2; ++c) put(entry(o, r, c));
            } else if (o.op == kOpReal || o.op == kOpImag) {
                code += uint32_t(regbit(o.tq[0]));
                const bool im = o.op == kOpImag;
                put(hcplx{entry(o, 0, 0).re, im ? entry(o, 0, 1).im : entry(o, 0, 1).re});
                put(hcplx{im ? entry(o, 1, 0).im : entry(o, 1, 0).re, entry(o, 1, 1).re});
            } else if (o.op == kOpX || o.op == kOpAnti) {
                code += uint32_t(regbit(o.tq[0]));
                if (o.op == kOpAnti) {
                    put(entry(o, 0, 1));
                    put(entry(o, 1, 0));
                }
            } else if (o.op == kOpZ) {
                uint32_t zr = 0, zl = 0, zt = 0;
                for (uint64_t x = o.D; x; x &= x - 1) {
                    const uint32_t q = uint32_t(__builtin_ctzll(x));
                    if (!(tile >> q & 1))
                        zt |= 1u << blkbit[q];
                    else if (regbit(q) >= 0)
                        zr |= 1u << regbit(q);
                    else
                        zl |= 1u << lanebit(q);
                }
                code += zr;
                rmask = zl << 8;
                put(entry(o, 1, 1));
                const uint64_t bits = zt;
                std::memcpy(&v[nv], &bits, sizeof bits);
                nv += 2;
                v[3] = 0;
            } else if (o.op == kOpDiagR) {
                const uint32_t q = o.tq[0];
                put(entry(o, 0, 0));
                if ((tile >> q & 1) && regbit(q) < 0) {  // a thread bit: one record per value
                    const uint32_t l0 = lane;
                    code = kOpScale;
                    lane |= 1u << lanebit(q);
                    record(l0);
                    put(entry(o, 1, 1));
                } else {
                    put(entry(o, 1, 1));
                    if (tile >> q & 1) {
                        code += uint32_t(regbit(q));
                    } else {
                        code = kOpScale;
                        rmask |= kPickBit | uint32_t(blkbit[q]) << 16;
                    }
                }
            } else if (o.op == kOpScale) {
                put(entry(o, 1, 1));
            } else if (o.op == kOpSwap || o.op == kOpSwapP || o.op == kOpGen2) {
                int a = regbit(o.tq[0]), b = regbit(o.tq[1]);
                const bool flip = a > b;  // matrix bit 0 on the higher register bit
                if (flip) std::swap(a, b);
                code += uint32_t(a == 0 ? b - 1 : 2);
                if (o.op == kOpSwapP) put(hcplx{0, o.b0 ? 1.0 : -1.0});
                if (o.op == kOpGen2)
                    for (uint32_t r = 0; r < 4; ++r)
                        for (uint32_t c = 0; c < 4; ++c) {
                            auto sw = [&](uint32_t x) { return flip ? (x >> 1 | (x & 1) << 1) : x; };
                            put(entry(o, sw(r), sw(c)));
                        }
            } else if (o.op == kOpGen3) {
                int at[3];  // register bit of matrix bit i
                for (int i = 0; i < 3; ++i) at[i] = regbit(o.tq[i]);
                auto perm = [&](uint32_t x) {
                    uint32_t y = 0;
                    for (int i = 0; i < 3; ++i) y |= (x >> at[i] & 1) << i;
                    return y;
                };
                for (uint32_t r = 0; r < 8; ++r)
                    for (uint32_t c = 0; c < 8; ++c) put(entry(o, perm(r), perm(c)));
            }
            record(lane);
        }
    }
    out.insert(out.end(), {kOpEnd, 0, 0, 0});
    out.resize(out.size() + kTail, 0);
}

// Tile width for an n-qubit register: the whole register while one tile
// holds it, then as wide as leaves 2^8 tiles (one per CU).
static uint32_t tile_width(uint32_t n) {
    return n <= 10 ? n : std::min<uint32_t>(kTileMax, std::max<uint32_t>(10, n - 8));
}

TilePlanner::TilePlanner(const qcs_gate* gates, uint32_t n, uint32_t nq, size_t amp_bytes, size_t stream_bytes)
    : p_(new Plan) {
    Plan& P = *p_;
    P.gates = gates;
    P.count = n;
    P.n = nq;
    P.t = tile_width(nq);
    P.all = nq >= 64 ? ~0ull : (1ull << nq) - 1;
    P.big = (amp_bytes << nq) > (size_t(64) << 20);
    const uint32_t line = amp_bytes == 16 ? 3 : 4;
    P.low = (1ull << std::min(nq, P.big ? line + 1 : line)) - 1;
    P.max_bytes = stream_bytes;
    P.on.resize(nq);
}

TilePlanner::~TilePlanner() { delete p_; }

bool TilePlanner::big() const { return p_->big; }

bool TilePlanner::next(TileGeo& geo, std::vector<uint32_t>& words, const qcs_gate** single) {
    Plan& P = *p_;
    while (P.waiting < kAhead && P.at < P.count) P.add(P.gates[P.at++]);
    *single = nullptr;
    if (P.head < 0) return false;
    const uint64_t S = tile_choose(P);
    P.take.clear();
    const double worth = tile_scan(P, S, &P.take);
    // A pass moves the whole state once: it has to replace launches that
    // move more. Where launches cost more than bytes it has to replace
    // three (us for 2 / 3 / 5 gates on 16 qubits, launches against passes:
    // 10 / 14 / 23 against 12 / 13 / 14; on 20 qubits 15 / 18 / 37 against
    // 18 / 18 / 23; on 25 qubits, by worth, 208 / 382 / 602 against
    // 177 / 211 / 225).
    const TileGate& first = P.g[P.head];
    if (first.op == kNoTile || (first.src && !(P.big ? worth > 1.2 : P.take.size() > 2))) {
        *single = first.src;
        P.remove(P.head);
        return true;
    }
    P.local.clear();
    for (const int i : P.take) {
        P.local.push_back(&P.g[i]);
        P.remove(i);
    }
    geo = TileGeo{};
    uint64_t top = S;
    for (uint64_t x = S; x; x &= x - 1) geo.pos[geo.t++] = uint8_t(__builtin_ctzll(x));
    while (popc(top) > kTileReg) top &= top - 1;
    words.clear();
    tile_emit(P.local, tile_rounds(P.local, S, top), S, P.n, words);
    return true;
}

// ---------------------------------------------------------------------------
// Passes or dense blocks.
//
// Times are in ps per amplitude of a state that HBM bounds. Those of the steps
// of a plan were fitted to 135 runs of 16 kinds of list on 25 to 30 qubits, which
// they give to 10 % each; a pass is not below the time of its bytes. A dense
// block's are its kernel's rate on 30 qubits, and ms for its matrix's way there.
struct BlockTime {
    double ps, ms;
};

static BlockTime block_time(uint32_t k, bool c64) {
    if (k == 5) return c64 ? BlockTime{3.42, 0.14} : BlockTime{6.4, 0.14};
    return c64 ? BlockTime{2.88, 0.045} : BlockTime{5.6, 0.04};
}

static double pass_time(const std::vector<uint32_t>& words, bool c64) {
    double ps = 2.5;
    for (size_t i = 0; (words[i] & 0xffff) != kOpEnd; i += words[i] >> 16) {
        const uint32_t code = words[i] & 0xffff;
        if (code == kOpRound) {
            ps += 0.29;
            continue;
        }
        if (code >= kOpZ && code < kOpGen2) {
            ps += 0.16;
            continue;
        }
        // of the amplitudes, or the tiles, those with every control set
        const double part = popc(words[i + 2] & 255) / 8.0 / double(1 << popc(words[i + 3]));
        ps += part * (code < kOpReal                       ? 0.26
                      : code < kOpX                        ? 0.18
                      : code < kOpDiagR                    ? 0.20
                      : code < kOpSwap                     ? 0.16
                      : code < kOpZ                        ? 0.20
                      : code < kOpGen3                     ? 0.97
                                                           : 1.5);
    }
    return std::max(ps, c64 ? 4.4 : 7.1);
}

// Mostly above the time a gate takes in a pass with its share of the rounds,
// and without a plan.
static double gate_time(const qcs_gate& g, bool c64) {
    if (g.k > 3) return block_time(g.k, c64).ps;
    const uint32_t t = (g.flags & QCS_GATE_DENSE) ? 0 : g.traits;
    if (g.k == 1) return 0.3;
    if (t & (QCS_TRAIT_SWAP | QCS_TRAIT_ISWAP | QCS_TRAIT_ISWAPDAG)) return 0.7;
    const uint32_t targets = !(t & QCS_TRAIT_CONTROLLED) ? g.k : g.k == 3 && !(t & QCS_TRAIT_CTRL_Q1) ? 2 : 1;
    return targets == 1 ? 0.6 : targets == 2 ? 1.5 : 2.7;
}

// Blocks multiply on the matrix cores, at nearly the rate of their bytes for
// as many gates as meet on four or five qubits; a pass computes each gate by
// itself, on any qubits, and a phase over many for the price of one. So lists
// that keep to neighbourhoods are faster in blocks, and others in passes (ms at
// width 5, blocks and passes; 28 qubits complex128: Heisenberg steps, 1377
// gates, 29.4 and 54.9; layers of U(2) and CNOT, 504 gates, 72.3 and 46.7; Ising
// steps, 654 gates, 47.2 and 23.0. Complex64: 17.2 and 55.6, 41.6 and 43.9, 26.8
// and 23.9. 26 qubits complex128: 8.7 and 12.8, 21.9 and 10.8, 14.3 and 5.4).
//
// complex128, from 25 qubits on (below, the host's fusion takes longer than the
// passes): blocks where they take less than 0.85 of the passes' time, and
// where a quarter of the gates or more join qubits, as for others the fusion
// itself takes longest. Both compute in FP64; of a normalised state of 13 qubits
// after 612 gates the passes err by 1.1e-15, the blocks by 1.5e-15. complex64, where blocks are in FP32 and passes in FP64:
// from 28 qubits on blocks, unless the passes take less than 0.9 of their time;
// below always passes, which are 20 times as exact (27 qubits, the lists above:
// 9.9 and 27.5, 22.9 and 20.5, 14.3 and 11.2 ms).
uint32_t blocks_width(const qcs_gate* gates, uint32_t n, uint32_t nq, size_t amp_bytes, size_t stream_bytes, uint32_t lo,
                      uint32_t hi) {
    constexpr uint32_t kSample = 4096;  // of a long list, its beginning tells
    const bool c64 = amp_bytes == 8;
    if (hi < 4 || nq < (c64 ? 28u : 25u)) return 0;
    n = std::min(n, kSample);
    uint32_t joined = 0;
    double quick = 0;
    for (uint32_t i = 0; i < n; ++i) {
        joined += gates[i].k > 1;
        quick += gate_time(gates[i], c64);
    }
    if (!c64 && 4 * joined < n) return 0;
    const double ms = double(1ull << nq) * 1e-9;  // a ps per amplitude
    double blocks = 0;
    uint32_t width = 0;
    for (uint32_t w = std::max(lo, 4u); w <= hi; ++w) {
        const BlockTime t = block_time(w, c64);
        const double b = fuse_estimate(gates, n, w) * (t.ps * ms + t.ms);
        if (!width || b < blocks) {
            blocks = b;
            width = w;
        }
    }
    // plainly the one or the other, by the gates alone
    quick *= ms;
    if (c64 ? quick < 0.9 * blocks : blocks > 0.85 * quick) return 0;
    if (blocks < 0.3 * quick) return width;
    TilePlanner plan(gates, n, nq, amp_bytes, stream_bytes);
    TileGeo geo;
    std::vector<uint32_t> words;
    const qcs_gate* single = nullptr;
    double passes = 0;
    while (plan.next(geo, words, &single))
        passes += !single ? pass_time(words, c64) : single->k > 3 ? block_time(single->k, c64).ps : c64 ? 3.8 : 5.2;
    passes *= ms;
    return (c64 ? passes < 0.9 * blocks : blocks > 0.85 * passes) ? 0 : width;
}

}  // namespace qcs
