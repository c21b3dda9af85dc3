// vqe.hip - batched VQE energies: many small registers of uneven size, each
// prepared by the reference's hardware-efficient ansatz and scored with the
// exact FP64 energy of a Pauli-string Hamiltonian, in one launch.
//
// Ansatz (VQE::PauliStringVQE::Ansatz, VQE.h:78-114), from |0...0>: with
// parameters p[0..P) (nothing at all when P < n), the first layer puts
// Ry(p[2q]) then Rz(p[2q+1]) on qubits q = 0, 1, ... while two parameters
// remain; then, while two parameters remain, an entangling ladder
// (alternately CNOT(target q+1, control q) for q = 0..n-2 plus, for n > 2,
// CNOT(target 0, control n-1); and CNOT(target q-1, control q) for
// q = n-1..1 plus, for n > 2, CNOT(target n-1, control 0)) followed by
// another Ry / Rz layer.
//
// Energy: sum_t c_t <psi|P_t|psi> with P_t = i^{|x_t & z_t|} X^{x_t} Z^{z_t},
// evaluated as in k_pauli (one pair sum per term); for a VQE term this is
// the exact value of the estimate that EstimateEnergy samples (VQE.h:116-142
// after the change of basis of :33-44).
//
// An instance lives in LDS (n <= 12: 64 KiB of complex128), from where its
// threads take 16 amplitudes of four qubits at a time into registers; the
// final state is written to the instance's slot of an arena in HBM. One of up
// to ten qubits belongs to one wave, four to a block, without barriers; a
// larger one to a block. What a batch costs is a chain of dependent steps, so
// there are few of them: the first layer is a product state, each ladder a
// permutation of the index that the next layer's first reads carry out, the
// sines of 64 rotations are computed at once, and the terms add up in each
// thread, with one sum over the threads at the end.
//
// 1024 instances of 4..12 qubits, 24 terms, 2 layers: 158 us with a step for
// each gate and a sum for each term, in three launches; now 28 us in one, of
// which each instance's own chain is 20 (three steps to LDS and back a layer,
// one a term).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.h"

namespace qcs {

constexpr uint32_t kVqeMaxQubits = 12;

struct VInst {
    uint64_t off;       // first amplitude of the instance in the arena
    uint32_t n;         // qubits
    uint32_t nterms;    // Hamiltonian terms
    uint32_t toff;      // first term
    uint32_t nparams;   // ansatz parameters (set per evaluation)
    uint32_t poff;      // first parameter
    uint32_t pad;
};

constexpr uint32_t kVqeReg = 4;       // register qubits
constexpr uint32_t kVqeWaveQubits = 10;  // the largest instance of a single wave

// A block's work: one instance (wide), or up to four, one for each wave.
struct VUnit {
    uint32_t inst[4], count, wide;
};

// LDS slot of amplitude i: orbits of four neighbouring qubits spread over the banks.
__device__ __forceinline__ uint32_t vqe_slot(uint32_t i) { return i ^ (i >> 4 & 15); }

// The index whose amplitude the CNOT ladder brings to index i: its gates
// undone from the last to the first, each of which flips a bit above (or
// below) the ones still to be read.
__device__ __forceinline__ uint32_t vqe_ladder(uint32_t i, uint32_t n, bool flip) {
    if (flip) {
        if (n > 2) i ^= (i & 1) << (n - 1);
        return i ^ i >> 1;
    }
    if (n > 2) i ^= i >> (n - 1) & 1;
    return i ^ (i << 1 & ((1u << n) - 1));
}

__device__ __forceinline__ double readlane(double v, uint32_t lane) {
    const long long b = __double_as_longlong(v);
    return __longlong_as_double((long long)(uint64_t(uint32_t(__builtin_amdgcn_readlane(int(b >> 32), int(lane)))) << 32 |
                                            uint32_t(__builtin_amdgcn_readlane(int(b), int(lane)))));
}

__device__ __forceinline__ double2 vqe_mul(double2 x, double2 y) {
    return double2{x.x * y.x - x.y * y.y, x.x * y.y + x.y * y.x};
}

// sum of v[k] (-1)^{parity of the bits of k in z}, z the same in the whole wave
template <int K>
__device__ __forceinline__ double vqe_signed_sum(double (&v)[K], uint32_t z) {
#pragma unroll
    for (int h = K / 2; h >= 1; h /= 2) {
        // the highest bit left pairs k with k + h
        const double sgn = z & uint32_t(h) ? -1.0 : 1.0;
#pragma unroll
        for (int k = 0; k < h; ++k) v[k] = fma(v[k + h], sgn, v[k]);
    }
    return v[0];
}

// k without its bit B
__host__ __device__ constexpr uint32_t vqe_drop(uint32_t k, uint32_t B) {
    return (k >> (B + 1)) << B | (k & ((1u << B) - 1));
}

// The eight pairs of a thread for a mask whose highest register bit is B: the
// register indices with that bit clear, their partners' amplitudes from LDS at
// `at` ^ c[k].
template <uint32_t B>
__device__ __forceinline__ double vqe_pairs(const char* s, const double2 (&a)[16], uint32_t at, const uint32_t (&c)[16],
                                            bool odd, uint32_t zr) {
    double2 w[8];
    double v[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t k = (j >> B) << (B + 1) | (j & ((1u << B) - 1));
        w[j] = *reinterpret_cast<const double2*>(s + (at ^ c[k]));
    }
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
        const double2 u = a[(j >> B) << (B + 1) | (j & ((1u << B) - 1))];
        v[j] = odd ? u.x * w[j].y - u.y * w[j].x : u.x * w[j].x + u.y * w[j].y;
    }
    return vqe_signed_sum(v, vqe_drop(zr, B));
}

// One instance, by the whole block or by one wave: s its amplitudes, tab room
// for the factors of 64 rotations (of this wave).
template <bool WIDE>
__device__ void vqe_run(const VInst I, uint32_t id, double2* s, double (*tab)[4], double* red,
                        const double* __restrict__ params, const uint64_t* __restrict__ xm,
                        const uint64_t* __restrict__ zm, const double* __restrict__ coef, double2* __restrict__ arena,
                        double* __restrict__ energy) {
    const uint32_t lane = threadIdx.x & 63, tid = WIDE ? threadIdx.x : lane, nthr = WIDE ? 256 : 64;
    auto sync = [] {
        if constexpr (WIDE) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };
    const uint32_t n = I.n, m = n < kVqeReg ? kVqeReg : n, A = 1u << n;
    const uint32_t rots = I.nparams >= n ? I.nparams / 2 : 0;
    const double* p = params + I.poff;
    const bool active = tid < 1u << (m - kVqeReg);
    double2 a[16];
    // Rz = e^{-i phi/2} diag(1, e^{i phi}): the first factor is the whole
    // state's, and waits for the end, as the sum of the angles with what
    // rounding took from it; a rotation's table entry is cos and sin of theta/2
    // and of phi. (The product of the factors, and cos and sin of phi from those
    // of phi/2, took the same time and erred more: 160 instances of 4 to 11
    // qubits, states by 4.8e-16 and energies by 3.7e-16, now 3.2e-16 and 2.9e-16.)
    double angle = 0, rest = 0;
    auto add = [](double& sum, double& low, double x, double xlow) {
        const double s = sum + x, v = s - sum;
        low += xlow + ((sum - (s - v)) + (x - v));
        sum = s;
    };
    uint32_t tab0 = 0, phased = 0;  // first rotation of the table; those before are in angle
    auto fill = [&](uint32_t first) {
        tab0 = first;
        sync();
        double half = 0, low = 0;
        if (first + lane < rots) {
            const double phi = p[2 * (first + lane) + 1];
            double sy, cy, sz, cz;
            sincos(0.5 * p[2 * (first + lane)], &sy, &cy);
            sincos(phi, &sz, &cz);
            tab[lane][0] = cy;
            tab[lane][1] = sy;
            tab[lane][2] = cz;
            tab[lane][3] = sz;
            if (first + lane >= phased) half = 0.5 * phi;  // tables overlap
        }
#pragma unroll
        for (int d = 1; d < 64; d *= 2) add(half, low, __shfl_xor(half, d), __shfl_xor(low, d));
        phased = first + 64;
        add(angle, rest, half, low);
        sync();
    };
    fill(0);
    const uint32_t sh = m - kVqeReg;
    uint32_t held = sh;  // the register qubits whose amplitudes a[] holds
    // the first layer of |0...0>: qubit q in (cos, sin e^{i phi})
    if (active) {
        auto amp = [&](uint32_t q, bool one) {
            if (q >= rots || q >= n) return double2{one ? 0.0 : 1.0, 0.0};
            return one ? double2{tab[q][1] * tab[q][2], tab[q][1] * tab[q][3]} : double2{tab[q][0], 0.0};
        };
        a[0] = double2{1.0, 0.0};
        for (uint32_t q = 0; q < sh; ++q) a[0] = vqe_mul(a[0], amp(q, tid >> q & 1));
#pragma unroll
        for (int j = 0; j < int(kVqeReg); ++j) {
            const double2 f1 = amp(sh + j, true);
            const double f0 = amp(sh + j, false).x;
#pragma unroll
            for (int k = 0; k < 1 << j; ++k) {
                a[k | 1 << j] = vqe_mul(a[k], f1);
                a[k] = double2{a[k].x * f0, a[k].y * f0};
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) s[vqe_slot(tid) ^ vqe_slot(k << sh)] = a[k];
    }
    sync();
    bool flip = false;
    for (uint32_t r0 = n; r0 < rots; r0 += n, flip = !flip) {
        const uint32_t nq = min(n, rots - r0);
        if (r0 + nq > tab0 + 64) fill(r0);
        for (uint32_t q0 = 0; q0 < nq; q0 += kVqeReg) {
            // registers: qubits p0..p0+3, of which those from q0 on are still to be rotated
            const uint32_t p0 = min(q0, sh), low = (1u << p0) - 1;
            held = p0;
            const uint32_t base = (tid & ~low) << kVqeReg | (tid & low);
            if (active) {
                if (q0 == 0) {
                    const uint32_t at = vqe_slot(vqe_ladder(base, n, flip));
#pragma unroll
                    for (uint32_t k = 0; k < 16; ++k) a[k] = s[at ^ vqe_slot(vqe_ladder(k, n, flip))];
                } else {
#pragma unroll
                    for (uint32_t k = 0; k < 16; ++k) a[k] = s[vqe_slot(base) ^ vqe_slot(k << p0)];
                }
            }
            if (q0 == 0) sync();  // read before others write
            if (active) {
#pragma unroll
                for (uint32_t j = 0; j < kVqeReg; ++j) {
                    const uint32_t q = p0 + j;
                    if (q < q0 || q >= nq) continue;
                    const double* f = tab[r0 + q - tab0];
                    const double cy = f[0], sy = f[1];
                    const double2 ez{f[2], f[3]};
#pragma unroll
                    for (uint32_t k = 0; k < 16; ++k) {
                        if (k >> j & 1) continue;
                        const double2 x = a[k], y = a[k | 1 << j];
                        a[k] = double2{cy * x.x - sy * y.x, cy * x.y - sy * y.y};
                        a[k | 1 << j] = vqe_mul(double2{sy * x.x + cy * y.x, sy * x.y + cy * y.y}, ez);
                    }
                }
#pragma unroll
                for (uint32_t k = 0; k < 16; ++k) s[vqe_slot(base) ^ vqe_slot(k << p0)] = a[k];
            }
            sync();
        }
    }
    // The energy, from the amplitudes of the top four qubits in registers and
    // the partners of other threads in LDS. A lane holds a term's masks and
    // factor for all of its wave.
    if (held != sh && active)
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) a[k] = s[vqe_slot(tid) ^ vqe_slot(k << sh)];
    uint32_t c[16];  // byte offsets of the register indices
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) c[k] = vqe_slot(k << sh) << 4;
    const char* sb = reinterpret_cast<const char*>(s);
    double e = 0;
    for (uint32_t t0 = 0; t0 < I.nterms; t0 += 64) {
        uint32_t masks = 0;
        double factor = 0;
        if (t0 + lane < I.nterms) {
            const uint32_t x = uint32_t(xm[I.toff + t0 + lane]), z = uint32_t(zm[I.toff + t0 + lane]);
            masks = x | z << 16;
            factor = coef[I.toff + t0 + lane];
            if (x) factor *= __popc(x & z) / 2 & 1 ? -2.0 : 2.0;
        }
        const uint32_t nt = min(64u, I.nterms - t0);
        for (uint32_t t = 0; t < nt; ++t) {
            const uint32_t xz = uint32_t(__builtin_amdgcn_readlane(int(masks), int(t))), x = xz & 0xffff, z = xz >> 16;
            const double ft = readlane(factor, t);
            if (!active) continue;
            const uint32_t xr = x >> sh, zr = z >> sh, at = (vqe_slot(tid) ^ vqe_slot(x)) << 4;
            const bool odd = __popc(x & z) & 1;
            bool minus = __popc(tid & z & ((1u << sh) - 1)) & 1;
            double acc;
            if (x == 0) {
                double v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = a[k].x * a[k].x + a[k].y * a[k].y;
                acc = vqe_signed_sum(v, zr);
            } else if (xr >> 3) {
                acc = vqe_pairs<3>(sb, a, at, c, odd, zr);
            } else if (xr >> 2) {
                acc = vqe_pairs<2>(sb, a, at, c, odd, zr);
            } else if (xr >> 1) {
                acc = vqe_pairs<1>(sb, a, at, c, odd, zr);
            } else if (xr) {
                acc = vqe_pairs<0>(sb, a, at, c, odd, zr);
            } else {
                // thread l takes the lower register indices of its pairs with
                // thread l ^ x, which takes the upper ones
                const bool up = tid >> (31 - __clz(int(x))) & 1;
                double2 b[16];
#pragma unroll
                for (int k = 0; k < 8; ++k) b[k] = up ? a[k + 8] : a[k];
                acc = vqe_pairs<3>(sb, b, at ^ (up ? c[8] : 0), c, odd, zr);
                minus ^= up && (zr >> 3 & 1);
            }
            e = fma(ft, minus ? -acc : acc, e);
        }
    }
    e = wave_sum(e);
    if constexpr (WIDE) {
        if (lane == 0) red[threadIdx.x >> 6] = e;
        __syncthreads();
        e = ((red[0] + red[1]) + red[2]) + red[3];
    }
    if (tid == 0) energy[id] = e;
    double sa, ca;
    sincos(angle, &sa, &ca);
    const double2 phase{ca - rest * sa, -(sa + rest * ca)};
    for (uint32_t i = tid; i < A; i += nthr) stamp<double, true>(arena + I.off + i, vqe_mul(phase, s[vqe_slot(i)]));
}

__global__ __launch_bounds__(256) void k_vqe(const VInst* __restrict__ insts, const VUnit* __restrict__ units,
                                             const double* __restrict__ params, const uint64_t* __restrict__ xm,
                                             const uint64_t* __restrict__ zm, const double* __restrict__ coef,
                                             double2* __restrict__ arena, double* __restrict__ energy) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ double tab[4][64][4];
    __shared__ double red[4];
    double2* s = reinterpret_cast<double2*>(smem_raw);
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const VUnit& U = units[blockIdx.x];
    if (U.wide) {
        vqe_run<true>(insts[U.inst[0]], U.inst[0], s, tab[wave], red, params, xm, zm, coef, arena, energy);
    } else if (wave < U.count) {
        // the block's largest instance comes first
        const uint32_t m = max(insts[U.inst[0]].n, kVqeReg);
        vqe_run<false>(insts[U.inst[wave]], U.inst[wave], s + (wave << m), tab[wave], red, params, xm, zm, coef, arena,
                       energy);
    }
}

}  // namespace qcs

using namespace qcs;

struct qcs_vqe {
    uint32_t ninst = 0;
    std::vector<VInst> hinst;
    uint32_t nunits = 0;
    size_t lds = 0;                   // of a block
    VUnit* dunits = nullptr;
    uint64_t* dxm = nullptr;
    uint64_t* dzm = nullptr;
    double* dcoef = nullptr;
    // what an evaluation sends, in one copy: the instances, then the parameters
    std::vector<char> stage;
    char* dstage = nullptr;
    size_t params_cap = 0;
    double2* arena = nullptr;
    double* denergy = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float last_ms = 0;
};

extern "C" {

int qcs_vqe_destroy(qcs_vqe* v) {
    if (!v) return QCS_OK;
    if (v->stream) (void)hipStreamSynchronize(v->stream);
    for (void* p : {static_cast<void*>(v->dunits), static_cast<void*>(v->dxm),
                    static_cast<void*>(v->dzm), static_cast<void*>(v->dcoef), static_cast<void*>(v->dstage),
                    static_cast<void*>(v->arena), static_cast<void*>(v->denergy)})
        if (p) (void)hipFree(p);
    if (v->ev0) (void)hipEventDestroy(v->ev0);
    if (v->ev1) (void)hipEventDestroy(v->ev1);
    if (v->stream) (void)hipStreamDestroy(v->stream);
    delete v;
    return QCS_OK;
}

int qcs_vqe_create(uint32_t ninst, const uint32_t* nqubits, const uint32_t* nterms, const uint64_t* xmask,
                   const uint64_t* zmask, const double* coef, qcs_vqe** out) {
    if (!out || !ninst || !nqubits || !nterms) return set_error(QCS_EINVAL, "null argument");
    *out = nullptr;
    auto* v = new qcs_vqe;
    v->ninst = ninst;
    v->hinst.resize(ninst);
    uint64_t off = 0, toff = 0;
    for (uint32_t i = 0; i < ninst; ++i) {
        const uint32_t n = nqubits[i];
        if (n < 1 || n > kVqeMaxQubits) {
            delete v;
            return set_error(QCS_EINVAL, "instance %u: %u qubits (batched VQE holds 1..%u)", i, n, kVqeMaxQubits);
        }
        VInst& I = v->hinst[i];
        I.off = off;
        I.n = n;
        I.nterms = nterms[i];
        I.toff = uint32_t(toff);
        for (uint32_t t = 0; t < nterms[i]; ++t)
            if ((xmask[toff + t] | zmask[toff + t]) >> n) {
                delete v;
                return set_error(QCS_EINVAL, "instance %u term %u: mask beyond the register", i, t);
            }
        off += uint64_t(1) << n;
        toff += nterms[i];
        if (toff > 0xffffffffull) {
            delete v;
            return set_error(QCS_EINVAL, "too many terms");
        }
    }
    if (toff && (!xmask || !zmask || !coef)) {
        delete v;
        return set_error(QCS_EINVAL, "null term arrays");
    }
    // largest first: the long chains start at once, and a block's four
    // instances are of a size
    std::vector<uint32_t> order(ninst);
    for (uint32_t i = 0; i < ninst; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(),
                     [&](uint32_t a, uint32_t b) { return v->hinst[a].n > v->hinst[b].n; });
    std::vector<VUnit> units;
    for (uint32_t i = 0; i < ninst;) {
        VUnit U{};
        const uint32_t n = v->hinst[order[i]].n;
        U.wide = n > kVqeWaveQubits;
        do
            U.inst[U.count++] = order[i++];
        while (!U.wide && U.count < 4 && i < ninst);
        units.push_back(U);
        v->lds = std::max(v->lds, (U.wide ? 1 : 4) * (sizeof(double2) << std::max(n, kVqeReg)));
    }
    v->nunits = uint32_t(units.size());
    const size_t nt = std::max<uint64_t>(toff, 1);
    if (hipStreamCreateWithFlags(&v->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&v->ev0) != hipSuccess || hipEventCreate(&v->ev1) != hipSuccess) {
        qcs_vqe_destroy(v);
        return set_error(QCS_EDEVICE, "stream creation failed");
    }
    if (hipMalloc(reinterpret_cast<void**>(&v->dunits), sizeof(VUnit) * units.size()) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&v->dxm), sizeof(uint64_t) * nt) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&v->dzm), sizeof(uint64_t) * nt) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&v->dcoef), sizeof(double) * nt) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&v->arena), sizeof(double2) * off) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&v->denergy), sizeof(double) * ninst) != hipSuccess) {
        (void)hipGetLastError();
        qcs_vqe_destroy(v);
        return set_error(QCS_ENOMEM, "batched VQE buffers");
    }
    if ((toff && (hipMemcpy(v->dxm, xmask, sizeof(uint64_t) * toff, hipMemcpyHostToDevice) != hipSuccess ||
                  hipMemcpy(v->dzm, zmask, sizeof(uint64_t) * toff, hipMemcpyHostToDevice) != hipSuccess ||
                  hipMemcpy(v->dcoef, coef, sizeof(double) * toff, hipMemcpyHostToDevice) != hipSuccess)) ||
        hipMemcpy(v->dunits, units.data(), sizeof(VUnit) * units.size(), hipMemcpyHostToDevice) != hipSuccess) {
        qcs_vqe_destroy(v);
        return set_error(QCS_EDEVICE, "batched VQE upload failed");
    }
    *out = v;
    return QCS_OK;
}

int qcs_vqe_evaluate(qcs_vqe* v, const uint32_t* nparams, const double* params, double* energy) {
    if (!v || !nparams || !energy) return set_error(QCS_EINVAL, "null argument");
    uint64_t poff = 0;
    for (uint32_t i = 0; i < v->ninst; ++i) {
        v->hinst[i].nparams = nparams[i];
        v->hinst[i].poff = uint32_t(poff);
        poff += nparams[i];
        if (poff > 0xffffffffull) return set_error(QCS_EINVAL, "too many parameters");
    }
    if (poff && !params) return set_error(QCS_EINVAL, "null parameters");
    const size_t ibytes = sizeof(VInst) * v->ninst, pbytes = sizeof(double) * poff;
    if (!v->dstage || poff > v->params_cap) {
        if (hipStreamSynchronize(v->stream) != hipSuccess) return set_error(QCS_EDEVICE, "sync failed");
        if (v->dstage) (void)hipFree(v->dstage);
        v->dstage = nullptr;
        v->params_cap = 0;
        if (hipMalloc(reinterpret_cast<void**>(&v->dstage), ibytes + pbytes) != hipSuccess) {
            (void)hipGetLastError();
            v->dstage = nullptr;
            return set_error(QCS_ENOMEM, "parameter buffer");
        }
        v->params_cap = poff;
        v->stage.resize(ibytes + pbytes);
    }
    std::memcpy(v->stage.data(), v->hinst.data(), ibytes);
    if (poff) std::memcpy(v->stage.data() + ibytes, params, pbytes);
    if (hipMemcpyAsync(v->dstage, v->stage.data(), ibytes + pbytes, hipMemcpyHostToDevice, v->stream) != hipSuccess ||
        hipEventRecord(v->ev0, v->stream) != hipSuccess)
        return set_error(QCS_EDEVICE, "batched VQE upload failed");
    hipLaunchKernelGGL(k_vqe, dim3(v->nunits), dim3(256), v->lds, v->stream,
                       reinterpret_cast<const VInst*>(v->dstage), v->dunits,
                       reinterpret_cast<const double*>(v->dstage + ibytes), v->dxm, v->dzm, v->dcoef, v->arena, v->denergy);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(QCS_EDEVICE, "k_vqe launch failed: %s", hipGetErrorString(e));
    if (hipEventRecord(v->ev1, v->stream) != hipSuccess ||
        hipMemcpyAsync(energy, v->denergy, sizeof(double) * v->ninst, hipMemcpyDeviceToHost, v->stream) !=
            hipSuccess ||
        hipStreamSynchronize(v->stream) != hipSuccess)
        return set_error(QCS_EDEVICE, "batched VQE evaluation failed");
    (void)hipEventElapsedTime(&v->last_ms, v->ev0, v->ev1);
    return QCS_OK;
}

int qcs_vqe_last_ms(qcs_vqe* v, float* ms) {
    if (!v || !ms) return set_error(QCS_EINVAL, "null argument");
    *ms = v->last_ms;
    return QCS_OK;
}

int qcs_vqe_get_state(qcs_vqe* v, uint32_t inst, double* amps) {
    if (!v || !amps) return set_error(QCS_EINVAL, "null argument");
    if (inst >= v->ninst) return set_error(QCS_EINVAL, "instance out of range");
    const VInst& I = v->hinst[inst];
    if (hipMemcpy(amps, v->arena + I.off, sizeof(double2) << I.n, hipMemcpyDeviceToHost) != hipSuccess)
        return set_error(QCS_EDEVICE, "state download failed");
    return QCS_OK;
}

}  // extern "C"
