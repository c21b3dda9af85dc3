// expect_kernels.hip - Pauli-string expectations, and host vectors streamed
// through the device: inner products with a host vector, diagonal and dense
// operators on the whole register, complex64 conversions.
//
// Pauli strings. A string P = i^{|x & z|} X^x Z^z (per qubit: X if only its
// x bit is set, Z if only its z bit, Y = iXZ if both, identity if neither)
// has (P psi)_s = i^{ny} (-1)^{popcount((s^x) & z)} psi_{s^x}, ny = |x & z|.
// The reference measures such a string after a basis change and averages
// 10000 sampled parities (VQE.h:116-142, with the change of basis at
// :33-44); it leaves this exact form as a TODO (QubitRegister.h:649). Here
// they are evaluated in read-only passes over the state:
//   x = 0:  <P> = sum_s |psi_s|^2 sigma(s), sigma(s) = (-1)^{popcount(s & z)}
//   x != 0: a pair (s, t = s ^ x) adds sigma(s) (kappa a + conj a),
//           a = conj(psi_s) psi_t and kappa = (-1)^{ny}, since
//           sigma(t) = kappa sigma(s); so each term sums sigma(s) Re a (ny
//           even) or sigma(s) Im a (ny odd) over the pairs, whichever of the
//           two stands for s, and <P> = 2 (-1)^{ny/2} S (even) or
//           2 (-1)^{(ny-1)/2} S (odd).
// A pass takes every term whose x mask lies in its tile (k_pauli_tile); a
// mask too wide for a tile has one of its own (k_pauli). All sums are FP64
// with a fixed grid and a fixed combination order.
#include <algorithm>
#include <vector>

#include "common.h"
#include "pauli_plan.h"

namespace qcs {

constexpr int kExThreads = 256;

constexpr uint32_t kFlipBits = 16;  // iteration bits: 2^35 amplitudes over a grid of 2^19 work-items

// One pass's terms, passed by value (kernel arguments, read by scalar loads).
// Iteration k of a work-item visits s = s_thread | s_iter(g(k)), g the Gray
// code, so step k (k >= 1) flips exactly iteration bit b = ctz(k): state bit
// bit[b], and the sign of term j flips by w[b][j] (1 << 31 when z_j holds
// that bit: the sign bit of the double +-1.0).
struct PauliFlip {
    uint32_t w[kFlipBits][kPauliTerms];
    uint64_t bit[kFlipBits];
    uint64_t z[kPauliTerms];
};

// One pass for the terms j < nt that share x (highest bit hbit), the pair
// taken at the index with that bit clear. The grid stride is a power of two,
// so an index splits into disjoint bit sets: s = s_thread | s_iter, s_thread
// from the work-item's index and s_iter from the iteration alone (insert_run
// maps disjoint bit sets to disjoint bit sets). Hence sigma_j(s) =
// sigma_j(s_thread) sigma_j(s_iter): the second factor is the same for the
// whole wave, kept as the high word of a double +-1.0 on the scalar unit and
// updated with one XOR per term and iteration along the Gray walk; the vector
// unit adds conj(psi_s) psi_{s^x} (+-) per term with FP64 FMAs, both parts,
// of which the term needs one; the first factor is applied once per work-item
// at the end.
template <typename T>
__device__ __forceinline__ void pauli_product(const cv<T>* __restrict__ psi, uint64_t s, uint64_t x, double& re,
                                              double& im) {
    const cv<T> u = ldamp<T, true>(psi + s);
    const cv<T> w = ldamp<T, true>(psi + (s ^ x));
    re = double(u.x) * double(w.x) + double(u.y) * double(w.y);
    im = double(u.x) * double(w.y) - double(u.y) * double(w.x);
}

template <typename T, int G>
__global__ __launch_bounds__(kExThreads) void k_pauli(const cv<T>* __restrict__ psi, uint64_t npairs, uint64_t x,
                                                      uint32_t hbit, uint32_t nt, uint32_t niter, uint32_t odd_mask,
                                                      PauliFlip F, double* __restrict__ partial) {
    __shared__ double lds[4][G];
    double ar[G], ai[G];
#pragma unroll
    for (int j = 0; j < G; ++j) ar[j] = ai[j] = 0;
    uint64_t sg[G];  // the per-iteration signs (+-1.0) as bit patterns
#pragma unroll
    for (int j = 0; j < G; ++j) sg[j] = 0x3FF0000000000000ull;
    const uint64_t t = uint64_t(blockIdx.x) * kExThreads + threadIdx.x;
    // a work-item beyond a state smaller than one grid reads index 0 and
    // adds nothing
    const bool live = t < npairs;
    const double wt = live ? 1.0 : 0.0;
    const uint64_t st = live ? insert_run(t, hbit, 1) : 0;
    auto acc = [&](double re, double im, int j) {
        const double sgn = __longlong_as_double(static_cast<long long>(sg[j]));
        ar[j] = fma(re, sgn, ar[j]);
        ai[j] = fma(im, sgn, ai[j]);
    };
    uint64_t sk = 0;
    if (niter >= 2) {
        // two pairs a trip, their loads issued together
        for (uint32_t k = 0; k < niter; k += 2) {
            if (k) {  // Gray step k flips iteration bit ctz(k) >= 1
                const uint32_t b = __builtin_ctz(k);
                sk ^= F.bit[b];
#pragma unroll
                for (int j = 0; j < G; ++j) sg[j] ^= uint64_t(F.w[b][j]) << 32;
            }
            const uint64_t s0 = st | sk, s1 = s0 ^ F.bit[0];  // step k+1 flips bit 0
            double re[2], im[2];
            pauli_product<T>(psi, s0, x, re[0], im[0]);
            pauli_product<T>(psi, s1, x, re[1], im[1]);
#pragma unroll
            for (int j = 0; j < G; ++j) {
                acc(re[0], im[0], j);
                sg[j] ^= uint64_t(F.w[0][j]) << 32;
                acc(re[1], im[1], j);
            }
            sk ^= F.bit[0];
        }
    } else if (niter) {
        double re, im;
        pauli_product<T>(psi, st, x, re, im);
#pragma unroll
        for (int j = 0; j < G; ++j) acc(re, im, j);
    }
    // per term: the part the host needs, the work-item's sign, the wave's sum
    const uint32_t w = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < G; ++j) {
        double v = (odd_mask >> j) & 1 ? ai[j] : ar[j];
        v *= wt;
        if (__popcll(st & F.z[j]) & 1) v = -v;
        v = wave_sum(v);
        if ((threadIdx.x & 63) == 0) lds[w][j] = v;
    }
    __syncthreads();
    if (threadIdx.x < nt)
        partial[threadIdx.x * gridDim.x + blockIdx.x] =
            ((lds[0][threadIdx.x] + lds[1][threadIdx.x]) + lds[2][threadIdx.x]) + lds[3][threadIdx.x];
}

// The terms of a pass that a tile covers. A tile is the 2^t amplitudes that
// differ in the t tile qubits; a term belongs to the pass if its x mask lies
// in them. A block walks over tiles, each thread with the four amplitudes of
// the top two tile qubits in registers and, if the pass has terms with x != 0,
// the tile in LDS, from where it reads the partners of its pairs.
//
// A sum over tiles is kept per thread and register index, so the signs of a z
// mask inside the tile come in only at the end: any number of such terms
// costs the products of their x masks. A slot is two such sums: of the two
// pairs of one x mask, real or imaginary part, or, in passes without pairs,
// of two terms with x = 0 whose z mask leaves the tile. z bits outside the
// tile flip the sign of a sum from tile to tile.
//
// 26 qubits complex128, a Heisenberg chain in a field (101 terms, 25 x masks):
// 5.8 ms in a pass for each x mask and each 16 diagonal terms, 0.71 ms in
// three tile passes. They read the 1 GiB in 190 to 294 us, the more the more
// slots (11 in the slowest), 190 being the rate of a copy's reads: a slot
// costs each wave a trip to LDS. One block of 1024 threads a CU holds two
// tiles in LDS (one barrier a tile) and prefetches the next into registers.
// 27 terms on 27 qubits complex64: 0.51 ms in two passes, now 0.26 ms in one.
constexpr int kPtThreads = 1024;  // of a full tile

template <typename T, bool PAIRS>
__global__ __launch_bounds__(kPtThreads) void k_pauli_tile(const cv<T>* __restrict__ psi, uint64_t amps, uint32_t ntiles,
                                                           PauliTile P, double* __restrict__ partial) {
    __shared__ cv<T> s[2][PAIRS ? 1 << kPtMax : 1];
    __shared__ double red[kPtThreads / 64][kPtTerms];
    const uint32_t tid = threadIdx.x, t = P.t, top = t - 2;
    const bool active = tid < 1u << top;
    uint64_t off = 0, hi[4];
    for (uint32_t i = 0; i < top; ++i) off |= active ? uint64_t(tid >> i & 1) << P.pos[i] : 0;
    // a register of one qubit has two of the four amplitudes; the others'
    // sums stay out of the results
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        hi[k] = uint64_t(k & 1) << P.pos[top] | uint64_t(k >> 1) << P.pos[top + 1];
        if (hi[k] >= amps) hi[k] = 0;
    }
    const bool half = amps < 4;
    uint64_t base = blockIdx.x;
    for (uint32_t i = 0; i < t; ++i) {
        const uint64_t low = (1ull << P.pos[i]) - 1;
        base = ((base & ~low) << 1) | (base & low);
    }
    auto load = [&](cv<T> (&a)[4]) {
        const cv<T>* p = psi + base;
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = ldamp<T, true>(p + hi[k] + off);
    };
    double own[4] = {0, 0, 0, 0}, sum[2 * kPtSlots];
#pragma unroll
    for (int i = 0; i < 2 * kPtSlots; ++i) sum[i] = 0;
    uint32_t neg = 0;  // sums held with the opposite sign
    cv<T> a[4], b[4];
    uint32_t tile = blockIdx.x, buf = 0;
    load(a);
    for (; tile < ntiles; tile += gridDim.x, buf ^= 1) {
        if (PAIRS && active)
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) s[buf][tid | k << top] = a[k];
        if (tile + gridDim.x < ntiles) base = ((base | P.tile_bits) + P.step) & ~P.tile_bits;  // carries pass the tile's bits
        load(b);
        if (PAIRS) __syncthreads();
        // held over the loop, the slots' LDS addresses cost 24 vector registers,
        // their conditions 48 scalar ones, and both spill
        uint32_t l = tid, ns = P.ns, im = P.im;
        asm volatile("" : "+v"(l), "+s"(ns), "+s"(im));
        double w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            w[k] = double(a[k].x) * double(a[k].x) + double(a[k].y) * double(a[k].y);
            own[k] += w[k];
        }
        const double p01 = w[0] + w[1], m01 = w[0] - w[1], p23 = w[2] + w[3], m23 = w[2] - w[3];
#pragma unroll
        for (int j = 0; j < kPtSlots; ++j)
            if (j < int(ns)) {
                if constexpr (!PAIRS) {
#pragma unroll
                    for (int i = 2 * j; i < 2 * j + 2; ++i) {
                        if ((__popc(tile & P.zt[i]) ^ neg >> i) & 1) {
                            neg ^= 1u << i;
                            sum[i] = -sum[i];
                        }
                        const uint32_t c = P.zt[i] >> 30;
                        if (c == 0)
                            sum[i] += p01 + p23;
                        else if (c == 1)
                            sum[i] += m01 + m23;
                        else if (c == 2)
                            sum[i] += p01 - p23;
                        else
                            sum[i] += m01 - m23;
                    }
                } else {
                    if ((__popc(tile & P.zt[j]) ^ neg >> j) & 1) {
                        neg ^= 1u << j;
                        sum[2 * j] = -sum[2 * j];
                        sum[2 * j + 1] = -sum[2 * j + 1];
                    }
                    // the pairs of thread l and thread l ^ x: l takes those of its
                    // register indices 0 and 1, l ^ x of 2 and 3, by the highest
                    // bit of x; a mask on the register qubits leaves each thread
                    // two pairs of its own
                    const uint32_t x = P.x[j], xr = x >> top, xl = x & ((1u << top) - 1);
                    const bool up = xr == 0 && (l >> (31 - __clz(int(xl | 1))) & 1);
                    const bool odd = up || xr == 1;
                    const cv<T> u0 = up ? a[2] : a[0], u1 = odd ? a[3] : a[1];
                    const cv<T> v0 = s[buf][(l | (up ? 2u << top : 0)) ^ x];
                    const cv<T> v1 = s[buf][(l | (odd ? 3u : 1u) << top) ^ x];
                    if (!(im >> j & 1)) {
                        sum[2 * j] = fma(double(u0.x), double(v0.x), fma(double(u0.y), double(v0.y), sum[2 * j]));
                        sum[2 * j + 1] = fma(double(u1.x), double(v1.x), fma(double(u1.y), double(v1.y), sum[2 * j + 1]));
                    } else {
                        sum[2 * j] = fma(double(u0.x), double(v0.y), fma(-double(u0.y), double(v0.x), sum[2 * j]));
                        sum[2 * j + 1] = fma(double(u1.x), double(v1.y), fma(-double(u1.y), double(v1.x), sum[2 * j + 1]));
                    }
                }
            }
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = b[k];
    }
    // per term: the signs of the thread's indices, the wave's sum
    const uint32_t wave = tid >> 6, lane = tid & 63;
    auto put = [&](uint32_t e, double v) {
        v = wave_sum(active ? v : 0.0);
        if (lane == 0) red[wave][e] = v;
    };
    auto sgn = [](uint32_t z, uint32_t i, double v) { return __popc(z & i) & 1 ? -v : v; };
#pragma unroll
    for (int j = 0; j < kPtSlots; ++j)
        if (j < int(P.ns)) {
            const double s0 = neg >> (PAIRS ? j : 2 * j) & 1 ? -sum[2 * j] : sum[2 * j];
            const double s1 = PAIRS && half ? 0 : neg >> (PAIRS ? j : 2 * j + 1) & 1 ? -sum[2 * j + 1] : sum[2 * j + 1];
            const uint32_t x = P.x[j], xr = x >> top, xl = x & ((1u << top) - 1);
            const bool up = xr == 0 && (tid >> (31 - __clz(int(xl | 1))) & 1);
            const uint32_t i0 = tid | (up ? 2u << top : 0), i1 = tid | (up || xr == 1 ? 3u : 1u) << top;
            for (uint32_t e = P.first[j]; e < P.first[j + 1]; ++e) {
                const uint32_t z = P.z[e];
                if (!PAIRS)
                    put(e, sgn(z & ((1u << top) - 1), tid, z >> 15 ? s1 : s0));
                else
                    put(e, sgn(z, i0, s0) + sgn(z, i1, s1));
            }
        }
    if (half) own[2] = own[3] = 0;
    for (uint32_t e = P.first[P.ns]; e < P.nt; ++e) {
        const uint32_t z = P.z[e];
        put(e, (sgn(z, tid, own[0]) + sgn(z, tid | 1u << top, own[1])) +
                   (sgn(z, tid | 2u << top, own[2]) + sgn(z, tid | 3u << top, own[3])));
    }
    __syncthreads();
    if (tid < P.nt) {
        double v = red[0][tid];
        for (uint32_t i = 1; i < blockDim.x / 64; ++i) v += red[i][tid];
        partial[tid * gridDim.x + blockIdx.x] = v;
    }
}

// out[j] = sum of the nb partials of term j = blockIdx.x, in a fixed order
__global__ __launch_bounds__(kExThreads) void k_pauli_final(const double* __restrict__ partial, uint32_t nb,
                                                            double* __restrict__ out) {
    __shared__ double lds[4];
    const double* p = partial + size_t(blockIdx.x) * nb;
    double acc = 0;
    for (uint32_t b = threadIdx.x; b < nb; b += kExThreads) acc += p[b];
    const double t = block_sum256(acc, lds);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

// <psi[0..len) | v[0..len)> partial sums (conj(psi) v), FP64.
template <typename T>
__global__ __launch_bounds__(kExThreads) void k_inner_vec(const cv<T>* __restrict__ psi,
                                                          const double2* __restrict__ v, uint64_t len,
                                                          double* __restrict__ partial) {
    __shared__ double lds[4];
    double re = 0, im = 0;
    const uint64_t stride = uint64_t(gridDim.x) * kExThreads;
    for (uint64_t i = uint64_t(blockIdx.x) * kExThreads + threadIdx.x; i < len; i += stride) {
        const cv<T> a = ldamp<T, true>(psi + i);
        const double2 b = ldamp<double, true>(v + i);
        re += double(a.x) * b.x + double(a.y) * b.y;
        im += double(a.x) * b.y - double(a.y) * b.x;
    }
    const double tr = block_sum256(re, lds);
    const double ti = block_sum256(im, lds);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = tr;
        partial[2 * blockIdx.x + 1] = ti;
    }
}

__global__ __launch_bounds__(kExThreads) void k_inner_final(const double* __restrict__ partial, uint32_t nb,
                                                            double* __restrict__ out) {
    __shared__ double lds[4];
    for (int c = 0; c < 2; ++c) {
        double acc = 0;
        for (uint32_t b = threadIdx.x; b < nb; b += kExThreads) acc += partial[2 * b + c];
        const double t = block_sum256(acc, lds);
        if (threadIdx.x == 0) out[c] = t;
    }
}

// psi[i] *= d[i] for i < len (one amplitude per lane)
template <typename T>
__global__ __launch_bounds__(kExThreads) void k_diag_part(cv<T>* __restrict__ psi, const double2* __restrict__ d,
                                                          uint64_t len) {
    const uint64_t i = uint64_t(blockIdx.x) * kExThreads + threadIdx.x;
    if (i >= len) return;
    const double2 f = ldamp<double, true>(d + i);
    const cv<T> a = ldamp<T, true>(psi + i);
    cv<T> o;
    o.x = T(f.x * double(a.x) - f.y * double(a.y));
    o.y = T(f.x * double(a.y) + f.y * double(a.x));
    stamp<T, true>(psi + i, o);
}

// y[row0 + r] = sum_j M[r][j] x[j] for the rows r < nrows of a row-major
// panel: one wave per row, lanes over the columns (consecutive lanes on
// consecutive matrix entries), FP64 accumulation.
template <typename T>
__global__ __launch_bounds__(kExThreads) void k_gemv_panel(const double2* __restrict__ M, const cv<T>* __restrict__ x,
                                                           cv<T>* __restrict__ y, uint64_t cols, uint64_t row0,
                                                           uint64_t nrows) {
    const uint64_t r = uint64_t(blockIdx.x) * (kExThreads / 64) + (threadIdx.x >> 6);
    if (r >= nrows) return;  // whole waves leave together
    const uint32_t lane = threadIdx.x & 63;
    const double2* row = M + r * cols;
    double re = 0, im = 0;
    for (uint64_t j = lane; j < cols; j += 64) {
        const double2 m = ldamp<double, true>(row + j);
        const cv<T> v = x[j];
        re += m.x * double(v.x) - m.y * double(v.y);
        im += m.x * double(v.y) + m.y * double(v.x);
    }
    re = wave_sum(re);
    im = wave_sum(im);
    if (lane == 0) {
        cv<T> o;
        o.x = T(re);
        o.y = T(im);
        y[row0 + r] = o;
    }
}

__global__ void k_d2f_part(const double2* __restrict__ in, float2* __restrict__ out, uint64_t n) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) out[i] = make_float2(float(in[i].x), float(in[i].y));
}
__global__ void k_f2d_part(const float2* __restrict__ in, double2* __restrict__ out, uint64_t n) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) out[i] = make_double2(double(in[i].x), double(in[i].y));
}

// ---------------------------------------------------------------------------
// Host side.

int ensure_xfer(qcs_register* r, size_t bytes) {
    if (bytes > kXferBytes) return set_error(QCS_EINVAL, "transfer chunk of %zu bytes too large", bytes);
    if (r->xfer && r->xfer_bytes >= bytes) return QCS_OK;
    if (hipStreamSynchronize(r->stream) != hipSuccess) return set_error(QCS_EDEVICE, "sync failed");
    if (r->xfer) (void)hipFree(r->xfer);
    r->xfer = nullptr;
    r->xfer_bytes = 0;
    if (hipMalloc(&r->xfer, bytes) != hipSuccess) {
        (void)hipGetLastError();
        r->xfer = nullptr;
        return set_error(QCS_ENOMEM, "transfer buffer of %zu bytes", bytes);
    }
    r->xfer_bytes = bytes;
    return QCS_OK;
}

// Amplitudes per transfer chunk (16 B each on the host side).
static uint64_t xfer_amps(const qcs_register* r) {
    const uint64_t cap = kXferBytes / 16;
    return r->A < cap ? r->A : cap;
}

static uint32_t grid256(uint64_t n) { return uint32_t((n + 255) / 256); }

// <P> from the sum S of a term's pass.
static double pauli_scale(uint64_t x, uint64_t z) {
    if (!x) return 1;
    const uint32_t ny = uint32_t(__builtin_popcountll(x & z));
    return ny / 2 & 1 ? -2.0 : 2.0;
}

// Terms of one x mask too wide for a tile, kPauliTerms at a time.
template <typename T>
static int pauli_wide(qcs_register* r, const std::vector<uint32_t>& terms, uint64_t x, const uint64_t* zmask,
                      double* out) {
    const uint64_t npairs = r->A / 2;
    const uint32_t hbit = uint32_t(63 - __builtin_clzll(x));
    double* res = r->red + kRedResult;
    for (size_t t0 = 0; t0 < terms.size(); t0 += kPauliTerms) {
        const uint32_t nt = uint32_t(std::min<size_t>(kPauliTerms, terms.size() - t0));
        uint32_t odd = 0;
        // a power-of-two grid (the sign split needs a power-of-two stride)
        uint64_t nb = 1;
        while (nb < uint64_t(kPauliBlocks) && nb * kExThreads * 8 < npairs) nb <<= 1;
        const uint64_t stride = nb * kExThreads;
        const uint32_t lstride = uint32_t(__builtin_ctzll(stride));
        const uint64_t niter = npairs > stride ? npairs / stride : 1;
        const uint32_t ibits = uint32_t(__builtin_ctzll(niter));
        if (ibits > kFlipBits) return set_error(QCS_EINVAL, "state too large for the Pauli pass");
        PauliFlip F{};
        for (uint32_t j = 0; j < nt; ++j) {
            const uint64_t z = zmask[terms[t0 + j]];
            F.z[j] = z;
            if (__builtin_popcountll(x & z) & 1) odd |= 1u << j;
        }
        for (uint32_t b = 0; b < ibits; ++b) {
            const uint32_t kb = lstride + b, pos = kb >= hbit ? kb + 1 : kb;
            F.bit[b] = 1ull << pos;
            for (uint32_t j = 0; j < nt; ++j) F.w[b][j] = uint32_t((F.z[j] >> pos) & 1) << 31;
        }
        const cv<T>* psi = static_cast<const cv<T>*>(r->psi);
        const dim3 grid{unsigned(nb)}, block{unsigned(kExThreads)};
        if (nt <= 8)
            hipLaunchKernelGGL((k_pauli<T, 8>), grid, block, 0, r->stream, psi, npairs, x, hbit, nt, uint32_t(niter), odd,
                               F, r->red);
        else
            hipLaunchKernelGGL((k_pauli<T, kPauliTerms>), grid, block, 0, r->stream, psi, npairs, x, hbit, nt,
                               uint32_t(niter), odd, F, r->red);
        if (const int e = check_launch(r, "k_pauli")) return e;
        hipLaunchKernelGGL(k_pauli_final, dim3(nt), dim3(kExThreads), 0, r->stream, r->red, uint32_t(nb), res);
        if (const int e = check_launch(r, "k_pauli_final")) return e;
        double sums[kPauliTerms];
        if (const int e = fetch(r, res, int(nt), sums)) return e;
        for (uint32_t j = 0; j < nt; ++j) out[terms[t0 + j]] = pauli_scale(x, zmask[terms[t0 + j]]) * sums[j];
    }
    return QCS_OK;
}

template <typename T>
static int pauli_t(qcs_register* r, uint32_t nterms, const uint64_t* xmask, const uint64_t* zmask, double* out) {
    const uint64_t full = r->A - 1;
    for (uint32_t t = 0; t < nterms; ++t)
        if ((xmask[t] | zmask[t]) & ~full) return set_error(QCS_EINVAL, "term %u: mask beyond the register", t);
    PauliPlanner plan(r->n, r->amp_bytes(), nterms, xmask, zmask);
    const uint32_t nb = plan.blocks;
    // the terms whose sums are on their way
    std::vector<uint32_t> batch, terms;
    double* res = r->red + kRedResult;
    auto flush = [&]() -> int {
        if (batch.empty()) return QCS_OK;
        hipLaunchKernelGGL(k_pauli_final, dim3(unsigned(batch.size())), dim3(kExThreads), 0, r->stream, r->red, nb, res);
        if (const int e = check_launch(r, "k_pauli_final")) return e;
        double sums[kPauliResults];
        if (const int e = fetch(r, res, int(batch.size()), sums)) return e;
        for (size_t j = 0; j < batch.size(); ++j) out[batch[j]] = pauli_scale(xmask[batch[j]], zmask[batch[j]]) * sums[j];
        batch.clear();
        return QCS_OK;
    };
    PauliTile P;
    bool pairs = false;
    while (plan.next(P, pairs, terms)) {
        if (batch.size() + terms.size() > size_t(kPauliResults))
            if (const int e = flush()) return e;
        const unsigned threads = std::max(64u, 1u << (P.t - 2));
        double* partial = r->red + batch.size() * nb;
        if (pairs)
            hipLaunchKernelGGL((k_pauli_tile<T, true>), dim3(nb), dim3(threads), 0, r->stream,
                               static_cast<const cv<T>*>(r->psi), r->A, plan.ntiles, P, partial);
        else
            hipLaunchKernelGGL((k_pauli_tile<T, false>), dim3(nb), dim3(threads), 0, r->stream,
                               static_cast<const cv<T>*>(r->psi), r->A, plan.ntiles, P, partial);
        if (const int e = check_launch(r, "k_pauli_tile")) return e;
        batch.insert(batch.end(), terms.begin(), terms.end());
    }
    if (const int e = flush()) return e;
    for (const PauliPlanner::Group& g : plan.wide)
        if (const int e = pauli_wide<T>(r, g.terms, g.x, zmask, out)) return e;
    return QCS_OK;
}

int pauli_expectation(qcs_register* r, uint32_t nterms, const uint64_t* xmask, const uint64_t* zmask, double* out) {
    return r->prec == QCS_COMPLEX128 ? pauli_t<double>(r, nterms, xmask, zmask, out)
                                     : pauli_t<float>(r, nterms, xmask, zmask, out);
}

template <typename T>
static int inner_host_t(qcs_register* r, const double* amps, double* re_im) {
    const uint64_t chunk = xfer_amps(r);
    if (const int e = ensure_xfer(r, chunk * 16)) return e;
    double sre = 0, sim = 0;  // chunk sums added in chunk order
    for (uint64_t off = 0; off < r->A; off += chunk) {
        const uint64_t len = std::min(chunk, r->A - off);
        if (hipMemcpyAsync(r->xfer, amps + 2 * off, len * 16, hipMemcpyHostToDevice, r->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "upload failed");
        const uint32_t nb = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(kRedBlocks, (len + 1023) / 1024)));
        hipLaunchKernelGGL((k_inner_vec<T>), dim3(nb), dim3(kExThreads), 0, r->stream,
                           static_cast<const cv<T>*>(r->psi) + off, static_cast<const double2*>(r->xfer), len, r->red);
        if (const int e = check_launch(r, "k_inner_vec")) return e;
        hipLaunchKernelGGL(k_inner_final, dim3(1), dim3(kExThreads), 0, r->stream, r->red, nb, r->red + kRedResult);
        if (const int e = check_launch(r, "k_inner_final")) return e;
        double z[2];
        if (const int e = fetch(r, r->red + kRedResult, 2, z)) return e;
        sre += z[0];
        sim += z[1];
    }
    re_im[0] = sre;
    re_im[1] = sim;
    return QCS_OK;
}

int inner_host(qcs_register* r, const double* amps, double* re_im) {
    return r->prec == QCS_COMPLEX128 ? inner_host_t<double>(r, amps, re_im) : inner_host_t<float>(r, amps, re_im);
}

template <typename T>
static int diag_host_t(qcs_register* r, const double* diag) {
    const uint64_t chunk = xfer_amps(r);
    if (const int e = ensure_xfer(r, chunk * 16)) return e;
    for (uint64_t off = 0; off < r->A; off += chunk) {
        const uint64_t len = std::min(chunk, r->A - off);
        // pageable source: the copy is ordered after the previous chunk's
        // kernel on this stream, so the buffer is free again
        if (hipMemcpyAsync(r->xfer, diag + 2 * off, len * 16, hipMemcpyHostToDevice, r->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "diagonal upload failed");
        hipLaunchKernelGGL((k_diag_part<T>), dim3(grid256(len)), dim3(kExThreads), 0, r->stream,
                           static_cast<cv<T>*>(r->psi) + off, static_cast<const double2*>(r->xfer), len);
        if (const int e = check_launch(r, "k_diag_part")) return e;
    }
    // the caller may release `diag` once the call returns
    return hipStreamSynchronize(r->stream) == hipSuccess ? QCS_OK : set_error(QCS_EDEVICE, "diagonal sync failed");
}

int apply_diagonal_host(qcs_register* r, const double* diag) {
    return r->prec == QCS_COMPLEX128 ? diag_host_t<double>(r, diag) : diag_host_t<float>(r, diag);
}

// psi <- M psi for a dense row-major 2^n x 2^n matrix in host memory:
// the result goes to the front of the transfer buffer, the matrix streams
// through the rest of it in panels of whole rows, and the result is copied
// over the state at the end.
template <typename T>
static int matrix_host_t(qcs_register* r, const double* mat) {
    const uint64_t A = r->A;
    const size_t ybytes = ((A * sizeof(cv<T>)) + 255) & ~size_t(255);
    const size_t rowbytes = A * 16;
    if (ybytes + rowbytes > kXferBytes) return set_error(QCS_EINVAL, "operator matrix too large for the register");
    const uint64_t rows = std::min<uint64_t>(A, (kXferBytes - ybytes) / rowbytes);
    if (const int e = ensure_xfer(r, ybytes + rows * rowbytes)) return e;
    auto* y = static_cast<cv<T>*>(r->xfer);
    auto* panel = reinterpret_cast<double2*>(static_cast<char*>(r->xfer) + ybytes);
    for (uint64_t r0 = 0; r0 < A; r0 += rows) {
        const uint64_t nr = std::min(rows, A - r0);
        if (hipMemcpyAsync(panel, mat + 2 * r0 * A, nr * rowbytes, hipMemcpyHostToDevice, r->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "matrix upload failed");
        const uint64_t nblk = (nr + 3) / 4;
        hipLaunchKernelGGL((k_gemv_panel<T>), dim3(unsigned(nblk)), dim3(kExThreads), 0, r->stream, panel,
                           static_cast<const cv<T>*>(r->psi), y, A, r0, nr);
        if (const int e = check_launch(r, "k_gemv_panel")) return e;
    }
    if (hipMemcpyAsync(r->psi, y, A * sizeof(cv<T>), hipMemcpyDeviceToDevice, r->stream) != hipSuccess ||
        hipStreamSynchronize(r->stream) != hipSuccess)
        return set_error(QCS_EDEVICE, "operator result copy failed");
    return QCS_OK;
}

int apply_matrix_host(qcs_register* r, const double* mat) {
    return r->prec == QCS_COMPLEX128 ? matrix_host_t<double>(r, mat) : matrix_host_t<float>(r, mat);
}

// complex64 registers: FP64 host amplitudes converted on the device, chunk
// by chunk through the transfer buffer
int convert_upload(qcs_register* r, const double* amps) {
    const uint64_t chunk = xfer_amps(r);
    if (const int e = ensure_xfer(r, chunk * 16)) return e;
    for (uint64_t off = 0; off < r->A; off += chunk) {
        const uint64_t len = std::min(chunk, r->A - off);
        if (hipMemcpyAsync(r->xfer, amps + 2 * off, len * 16, hipMemcpyHostToDevice, r->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "upload failed");
        hipLaunchKernelGGL(k_d2f_part, dim3(grid256(len)), dim3(256), 0, r->stream,
                           static_cast<const double2*>(r->xfer), static_cast<float2*>(r->psi) + off, len);
        if (const int e = check_launch(r, "k_d2f_part")) return e;
    }
    return hipStreamSynchronize(r->stream) == hipSuccess ? QCS_OK : set_error(QCS_EDEVICE, "sync failed");
}

int convert_download(qcs_register* r, double* amps) {
    const uint64_t chunk = xfer_amps(r);
    if (const int e = ensure_xfer(r, chunk * 16)) return e;
    for (uint64_t off = 0; off < r->A; off += chunk) {
        const uint64_t len = std::min(chunk, r->A - off);
        hipLaunchKernelGGL(k_f2d_part, dim3(grid256(len)), dim3(256), 0, r->stream,
                           static_cast<const float2*>(r->psi) + off, static_cast<double2*>(r->xfer), len);
        if (const int e = check_launch(r, "k_f2d_part")) return e;
        if (hipMemcpyAsync(amps + 2 * off, r->xfer, len * 16, hipMemcpyDeviceToHost, r->stream) != hipSuccess ||
            hipStreamSynchronize(r->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "download failed");
    }
    return QCS_OK;
}

}  // namespace qcs
