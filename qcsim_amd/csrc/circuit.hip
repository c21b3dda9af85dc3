// circuit.hip - many gates per pass over the state.
//
// A gate list is cut into passes. A pass owns a set S of t tile qubits: a
// block holds the 2^t amplitudes that differ only in S (one tile) and applies
// to them every gate of the list that acts inside S, in rounds. In a round
// each thread holds the 2^R amplitudes of R register qubits of S and applies
// the round's gates on them in registers; between rounds the tile is
// exchanged through LDS. Qubits on which a gate acts diagonally (its
// controls, the bits of a phase, the target of Rz) may be anywhere: in
// registers, in the thread index or outside the tile.
//
// The state is read and written once per pass instead of once per gate, and
// a register of few qubits (n <= t) runs a whole list in one launch: what
// bounds a gate launch is HBM for large states and the launch itself for
// small ones. The passes are bound by the vector ALUs (8 FMA per amplitude
// and U(2)) and the LDS exchange of each round (32 B per amplitude, the price
// of two U(2)).
// How a list is cut is in circuit_plan.cpp.
#include <algorithm>
#include <vector>

#include "circuit_plan.h"
#include "common.h"

namespace qcs {

// An amplitude: four registers in a row, as LDS reads and writes take them.
typedef double Amp __attribute__((ext_vector_type(2)));

// The operations on one qubit, exchanges and factors, in place on a thread's
// amplitudes a[0..8) for the lanes in `on`. On the device they are one
// statement with its own dispatch: the amplitudes pass through every
// operation of an interpreter, and written in C++ each operation gets
// registers of its own, with copies of all amplitudes before and after it,
// and a branch on the lanes makes the compiler route the whole loop through
// masked control flow (1150 cycles against 480 for a U(2) on a tile of 4096).
// Same operations in the same order as the gate kernels. m: matrix entries.
// The amplitudes are in registers of fixed numbers, so that the halves of one
// can be named here and whole ones outside. A taken branch costs a wave 30
// cycles: matrices are reached over the fewest, then the phases of kOpZ (13.4
// ms against 13.7 with those a branch later, 867 gates on 27 qubits).
#if defined(__HIP_DEVICE_COMPILE__)
#define QA(I, C) QA_##I##C
#define QA_0x "v[32:33]"
#define QA_0y "v[34:35]"
#define QA_1x "v[36:37]"
#define QA_1y "v[38:39]"
#define QA_2x "v[40:41]"
#define QA_2y "v[42:43]"
#define QA_3x "v[44:45]"
#define QA_3y "v[46:47]"
#define QA_4x "v[48:49]"
#define QA_4y "v[50:51]"
#define QA_5x "v[52:53]"
#define QA_5y "v[54:55]"
#define QA_6x "v[56:57]"
#define QA_6y "v[58:59]"
#define QA_7x "v[60:61]"
#define QA_7y "v[62:63]"
#define Q_BIT(I) "s_bitcmp1_b32 %[mask], " #I "\n\ts_cbranch_scc0 9f\n\t"  // to 9 unless bit I of the mask is set
// the orbit {I, K} times the 2x2 matrix
#define Q_GEN(I, K)                                                                                   \
    Q_BIT(I)                                                                                          \
    "v_mul_f64 %[t0], %[i00], " QA(I, y) "\n\t"                                                       \
    "v_mul_f64 %[t1], %[r00], " QA(I, y) "\n\t"                                                       \
    "v_mul_f64 %[t2], %[i10], " QA(I, y) "\n\t"                                                       \
    "v_mul_f64 %[t3], %[r10], " QA(I, y) "\n\t"                                                       \
    "v_fma_f64 %[t0], %[r00], " QA(I, x) ", -%[t0]\n\t"                                               \
    "v_fma_f64 %[t1], %[i00], " QA(I, x) ", %[t1]\n\t"                                                \
    "v_fma_f64 %[t2], %[r10], " QA(I, x) ", -%[t2]\n\t"                                               \
    "v_fma_f64 %[t3], %[i10], " QA(I, x) ", %[t3]\n\t"                                                \
    "v_fma_f64 " QA(I, x) ", %[r01], " QA(K, x) ", %[t0]\n\t"                                         \
    "v_fma_f64 " QA(I, y) ", %[r01], " QA(K, y) ", %[t1]\n\t"                                         \
    "v_fma_f64 %[t2], %[r11], " QA(K, x) ", %[t2]\n\t"                                                \
    "v_fma_f64 %[t3], %[r11], " QA(K, y) ", %[t3]\n\t"                                                \
    "v_fma_f64 " QA(I, x) ", -%[i01], " QA(K, y) ", " QA(I, x) "\n\t"                                 \
    "v_fma_f64 " QA(I, y) ", %[i01], " QA(K, x) ", " QA(I, y) "\n\t"                                  \
    "v_fma_f64 %[t2], -%[i11], " QA(K, y) ", %[t2]\n\t"                                               \
    "v_fma_f64 " QA(K, y) ", %[i11], " QA(K, x) ", %[t3]\n\t"                                         \
    "v_mov_b64 " QA(K, x) ", %[t2]\n9:\n\t"
// the same for the real matrix (m0, m1; m2, m3), and for (m0, i m1; i m2, m3)
#define Q_REAL(I, K)                                                                                  \
    Q_BIT(I)                                                                                          \
    "v_mul_f64 %[t0], %[r01], " QA(I, x) "\n\t"                                                       \
    "v_mul_f64 %[t1], %[r01], " QA(I, y) "\n\t"                                                       \
    "v_mul_f64 " QA(I, x) ", %[r00], " QA(I, x) "\n\t"                                                \
    "v_mul_f64 " QA(I, y) ", %[r00], " QA(I, y) "\n\t"                                                \
    "v_fma_f64 " QA(I, x) ", %[i00], " QA(K, x) ", " QA(I, x) "\n\t"                                  \
    "v_fma_f64 " QA(I, y) ", %[i00], " QA(K, y) ", " QA(I, y) "\n\t"                                  \
    "v_fma_f64 " QA(K, x) ", %[i01], " QA(K, x) ", %[t0]\n\t"                                         \
    "v_fma_f64 " QA(K, y) ", %[i01], " QA(K, y) ", %[t1]\n9:\n\t"
#define Q_IMAG(I, K)                                                                                  \
    Q_BIT(I)                                                                                          \
    "v_mul_f64 %[t0], %[r01], " QA(I, x) "\n\t"                                                       \
    "v_mul_f64 %[t1], %[r01], " QA(I, y) "\n\t"                                                       \
    "v_mul_f64 " QA(I, x) ", %[r00], " QA(I, x) "\n\t"                                                \
    "v_mul_f64 " QA(I, y) ", %[r00], " QA(I, y) "\n\t"                                                \
    "v_fma_f64 " QA(I, x) ", -%[i00], " QA(K, y) ", " QA(I, x) "\n\t"                                 \
    "v_fma_f64 " QA(I, y) ", %[i00], " QA(K, x) ", " QA(I, y) "\n\t"                                  \
    "v_fma_f64 " QA(K, x) ", %[i01], " QA(K, x) ", -%[t1]\n\t"                                        \
    "v_fma_f64 " QA(K, y) ", %[i01], " QA(K, y) ", %[t0]\n9:\n\t"
// a[I] times (R, J)
#define Q_MUL(I, R, J)                                                                                \
    "v_mul_f64 %[t0], " J ", " QA(I, y) "\n\t"                                                        \
    "v_mul_f64 %[t1], " R ", " QA(I, y) "\n\t"                                                        \
    "v_fma_f64 " QA(I, y) ", " J ", " QA(I, x) ", %[t1]\n\t"                                          \
    "v_fma_f64 " QA(I, x) ", " R ", " QA(I, x) ", -%[t0]\n\t"
#define Q_MULB(I, R, J) Q_BIT(I) Q_MUL(I, R, J) "9:\n\t"
#define Q_M0(I) Q_MULB(I, "%[r00]", "%[i00]")
#define Q_M1(I) Q_MULB(I, "%[r01]", "%[i01]")
// a[I] times r00 - i t2 (even register parity) or r00 + i t2 (odd)
#define Q_ZE(I)                                                                                       \
    "v_mul_f64 %[t0], %[t2], " QA(I, y) "\n\t"                                                        \
    "v_mul_f64 %[t1], %[r00], " QA(I, y) "\n\t"                                                       \
    "v_fma_f64 " QA(I, y) ", -%[t2], " QA(I, x) ", %[t1]\n\t"                                         \
    "v_fma_f64 " QA(I, x) ", %[r00], " QA(I, x) ", %[t0]\n\t"
#define Q_ZO(I)                                                                                       \
    "v_mul_f64 %[t0], %[t2], " QA(I, y) "\n\t"                                                        \
    "v_mul_f64 %[t1], %[r00], " QA(I, y) "\n\t"                                                       \
    "v_fma_f64 " QA(I, y) ", %[t2], " QA(I, x) ", %[t1]\n\t"                                          \
    "v_fma_f64 " QA(I, x) ", %[r00], " QA(I, x) ", -%[t0]\n\t"
#define Q_EXCH(I, K)                                                                                  \
    "v_mov_b64 %[t0], " QA(I, x) "\n\t"                                                               \
    "v_mov_b64 %[t1], " QA(I, y) "\n\t"                                                               \
    "v_mov_b64 " QA(I, x) ", " QA(K, x) "\n\t"                                                        \
    "v_mov_b64 " QA(I, y) ", " QA(K, y) "\n\t"                                                        \
    "v_mov_b64 " QA(K, x) ", %[t0]\n\t"                                                               \
    "v_mov_b64 " QA(K, y) ", %[t1]\n\t"
// I and K exchanged if bit M of the mask is set; then times m0 and m1, or both m0
#define Q_SWAP(M, I, K) Q_BIT(M) Q_EXCH(I, K) "9:\n\t"
#define Q_A01(M, I, K) Q_BIT(M) Q_EXCH(I, K) Q_MUL(I, "%[r00]", "%[i00]") Q_MUL(K, "%[r01]", "%[i01]") "9:\n\t"
#define Q_A00(M, I, K) Q_BIT(M) Q_EXCH(I, K) Q_MUL(I, "%[r00]", "%[i00]") Q_MUL(K, "%[r00]", "%[i00]") "9:\n\t"
#define Q_NEG(I)                                                                                      \
    Q_BIT(I) "v_mul_f64 " QA(I, x) ", -1.0, " QA(I, x) "\n\t"                                         \
             "v_mul_f64 " QA(I, y) ", -1.0, " QA(I, y) "\n9:\n\t"
#define Q_IF(CODE, LABEL) "s_cmp_eq_u32 %[code], " #CODE "\n\ts_cbranch_scc1 " #LABEL "f\n\t"
#define Q_DONE "s_branch 8f\n"
__device__ __forceinline__ void tile_simple(Amp (&a)[8], uint32_t code, uint32_t mask, const double (&m)[8],
                                            uint64_t on, uint32_t tid, uint32_t tile) {
    double t0, t1, t2, t3;
    uint64_t save;
    uint32_t v, z;
    // kOpZ: parity of the masked tile-index bits
    const uint32_t zt = __builtin_popcount(tile & uint32_t(__builtin_bit_cast(uint64_t, m[2]))) & 1;
    asm volatile(
        "s_and_saveexec_b64 %[save], %[on]\n\t"
        "s_cbranch_execz 8f\n\t"
        "s_cmp_gt_u32 %[code], 2\n\ts_cbranch_scc1 20f\n\t" Q_IF(1, 21) Q_IF(2, 22)
        Q_GEN(0, 1) Q_GEN(2, 3) Q_GEN(4, 5) Q_GEN(6, 7) Q_DONE
        "21:\n\t" Q_GEN(0, 2) Q_GEN(1, 3) Q_GEN(4, 6) Q_GEN(5, 7) Q_DONE
        "22:\n\t" Q_GEN(0, 4) Q_GEN(1, 5) Q_GEN(2, 6) Q_GEN(3, 7) Q_DONE
        "20:\n\ts_cmp_gt_u32 %[code], 35\n\ts_cbranch_scc1 40f\n\t"
        "s_cmp_gt_u32 %[code], 10\n\ts_cbranch_scc1 30f\n\t" Q_IF(8, 23) Q_IF(9, 24) Q_IF(10, 25)
        Q_IF(5, 26) Q_IF(6, 27)
        Q_REAL(0, 1) Q_REAL(2, 3) Q_REAL(4, 5) Q_REAL(6, 7) Q_DONE
        "26:\n\t" Q_REAL(0, 2) Q_REAL(1, 3) Q_REAL(4, 6) Q_REAL(5, 7) Q_DONE
        "27:\n\t" Q_REAL(0, 4) Q_REAL(1, 5) Q_REAL(2, 6) Q_REAL(3, 7) Q_DONE
        "23:\n\t" Q_IMAG(0, 1) Q_IMAG(2, 3) Q_IMAG(4, 5) Q_IMAG(6, 7) Q_DONE
        "24:\n\t" Q_IMAG(0, 2) Q_IMAG(1, 3) Q_IMAG(4, 6) Q_IMAG(5, 7) Q_DONE
        "25:\n\t" Q_IMAG(0, 4) Q_IMAG(1, 5) Q_IMAG(2, 6) Q_IMAG(3, 7) Q_DONE
        "30:\n\ts_cmp_gt_u32 %[code], 14\n\ts_cbranch_scc1 60f\n\t" Q_IF(13, 31) Q_IF(14, 32)
        Q_SWAP(0, 0, 1) Q_SWAP(2, 2, 3) Q_SWAP(4, 4, 5) Q_SWAP(6, 6, 7) Q_DONE
        "31:\n\t" Q_SWAP(0, 0, 2) Q_SWAP(1, 1, 3) Q_SWAP(4, 4, 6) Q_SWAP(5, 5, 7) Q_DONE
        "32:\n\t" Q_SWAP(0, 0, 4) Q_SWAP(1, 1, 5) Q_SWAP(2, 2, 6) Q_SWAP(3, 3, 7) Q_DONE
        "40:\n\t"
        // t2 = im or -im by the parity of the thread's and the tile's bits
        "s_lshr_b32 %[z], %[mask], 8\n\t"
        "v_and_b32 %[v], %[z], %[tid]\n\t"
        "v_bcnt_u32_b32 %[v], %[v], %[zt]\n\t"
        "v_and_b32 %[v], 1, %[v]\n\t"
        "v_lshlrev_b32 %[v], 1, %[v]\n\t"
        "v_sub_u32 %[v], 1, %[v]\n\t"
        "v_cvt_f64_i32 %[t2], %[v]\n\t"
        "v_mul_f64 %[t2], %[i00], %[t2]\n\t"
        Q_IF(37, 61) Q_IF(38, 62) Q_IF(39, 63) Q_IF(40, 64) Q_IF(41, 65) Q_IF(42, 66) Q_IF(43, 67)
        Q_ZE(0) Q_ZE(1) Q_ZE(2) Q_ZE(3) Q_ZE(4) Q_ZE(5) Q_ZE(6) Q_ZE(7) Q_DONE
        "61:\n\t" Q_ZE(0) Q_ZO(1) Q_ZE(2) Q_ZO(3) Q_ZE(4) Q_ZO(5) Q_ZE(6) Q_ZO(7) Q_DONE
        "62:\n\t" Q_ZE(0) Q_ZE(1) Q_ZO(2) Q_ZO(3) Q_ZE(4) Q_ZE(5) Q_ZO(6) Q_ZO(7) Q_DONE
        "63:\n\t" Q_ZE(0) Q_ZO(1) Q_ZO(2) Q_ZE(3) Q_ZE(4) Q_ZO(5) Q_ZO(6) Q_ZE(7) Q_DONE
        "64:\n\t" Q_ZE(0) Q_ZE(1) Q_ZE(2) Q_ZE(3) Q_ZO(4) Q_ZO(5) Q_ZO(6) Q_ZO(7) Q_DONE
        "65:\n\t" Q_ZE(0) Q_ZO(1) Q_ZE(2) Q_ZO(3) Q_ZO(4) Q_ZE(5) Q_ZO(6) Q_ZE(7) Q_DONE
        "66:\n\t" Q_ZE(0) Q_ZE(1) Q_ZO(2) Q_ZO(3) Q_ZO(4) Q_ZO(5) Q_ZE(6) Q_ZE(7) Q_DONE
        "67:\n\t" Q_ZE(0) Q_ZO(1) Q_ZO(2) Q_ZE(3) Q_ZO(4) Q_ZE(5) Q_ZE(6) Q_ZO(7) Q_DONE
        "60:\n\t" Q_IF(24, 41) Q_IF(25, 42) Q_IF(16, 43) Q_IF(17, 44) Q_IF(18, 45) Q_IF(20, 46) Q_IF(21, 47)
        Q_IF(22, 48) Q_IF(28, 50) Q_IF(29, 51) Q_IF(30, 52) Q_IF(32, 53) Q_IF(33, 54) "s_branch 55f\n"
        "41:\n\t" Q_M0(0) Q_M0(1) Q_M0(2) Q_M0(3) Q_M0(4) Q_M0(5) Q_M0(6) Q_M0(7) Q_DONE
        "42:\n\t" Q_NEG(0) Q_NEG(1) Q_NEG(2) Q_NEG(3) Q_NEG(4) Q_NEG(5) Q_NEG(6) Q_NEG(7) Q_DONE
        "43:\n\t" Q_A01(0, 0, 1) Q_A01(2, 2, 3) Q_A01(4, 4, 5) Q_A01(6, 6, 7) Q_DONE
        "44:\n\t" Q_A01(0, 0, 2) Q_A01(1, 1, 3) Q_A01(4, 4, 6) Q_A01(5, 5, 7) Q_DONE
        "45:\n\t" Q_A01(0, 0, 4) Q_A01(1, 1, 5) Q_A01(2, 2, 6) Q_A01(3, 3, 7) Q_DONE
        "46:\n\t" Q_M0(0) Q_M1(1) Q_M0(2) Q_M1(3) Q_M0(4) Q_M1(5) Q_M0(6) Q_M1(7) Q_DONE
        "47:\n\t" Q_M0(0) Q_M0(1) Q_M1(2) Q_M1(3) Q_M0(4) Q_M0(5) Q_M1(6) Q_M1(7) Q_DONE
        "48:\n\t" Q_M0(0) Q_M0(1) Q_M0(2) Q_M0(3) Q_M1(4) Q_M1(5) Q_M1(6) Q_M1(7) Q_DONE
        "50:\n\t" Q_SWAP(0, 1, 2) Q_SWAP(4, 5, 6) Q_DONE
        "51:\n\t" Q_SWAP(0, 1, 4) Q_SWAP(2, 3, 6) Q_DONE
        "52:\n\t" Q_SWAP(0, 2, 4) Q_SWAP(1, 3, 5) Q_DONE
        "53:\n\t" Q_A00(0, 1, 2) Q_A00(4, 5, 6) Q_DONE
        "54:\n\t" Q_A00(0, 1, 4) Q_A00(2, 3, 6) Q_DONE
        "55:\n\t" Q_A00(0, 2, 4) Q_A00(1, 3, 5)
        "8:\n\ts_mov_b64 exec, %[save]"
        : "+{v[32:35]}"(a[0]), "+{v[36:39]}"(a[1]), "+{v[40:43]}"(a[2]), "+{v[44:47]}"(a[3]), "+{v[48:51]}"(a[4]),
          "+{v[52:55]}"(a[5]), "+{v[56:59]}"(a[6]), "+{v[60:63]}"(a[7]), [t0] "=&v"(t0),
          [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3), [save] "=&s"(save), [v] "=&v"(v), [z] "=&s"(z)
        : [r00] "s"(m[0]), [i00] "s"(m[1]), [r01] "s"(m[2]), [i01] "s"(m[3]), [r10] "s"(m[4]), [i10] "s"(m[5]),
          [r11] "s"(m[6]), [i11] "s"(m[7]), [code] "s"(code), [mask] "s"(mask), [on] "s"(on),
          [tid] "v"(tid), [zt] "s"(zt)
        : "scc");
}
#undef QA
#undef Q_BIT
#undef Q_GEN
#undef Q_MUL
#undef Q_MULB
#undef Q_M0
#undef Q_M1
#undef Q_REAL
#undef Q_IMAG
#undef Q_ZE
#undef Q_ZO
#undef Q_EXCH
#undef Q_SWAP
#undef Q_A01
#undef Q_A00
#undef Q_NEG
#undef Q_IF
#undef Q_DONE
#else
__device__ void tile_simple(Amp (&a)[8], uint32_t code, uint32_t mask, const double (&m)[8], uint64_t on, uint32_t tid,
                            uint32_t tile);
#endif

// Generic blocks: y = M x on the orbit idx[0..D), in the lanes that are on.
template <int R, int D, typename M>
__host__ __device__ __forceinline__ void tile_rows(Amp (&a)[1 << R], const int (&idx)[D], M m, bool on) {
    Amp x[D];
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = a[idx[c]];
#pragma unroll
    for (int r = 0; r < D; ++r) {
        double yr = 0, yi = 0;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            const double mr = m[2 * (r * D + c)], mi = m[2 * (r * D + c) + 1];
            yr += mr * x[c].x - mi * x[c].y;
            yi += mr * x[c].y + mi * x[c].x;
        }
        if (on) {
            a[idx[r]].x = yr;
            a[idx[r]].y = yi;
        }
    }
}

template <int A, int B> __host__ __device__ constexpr int zero2(int i) {  // zero bits inserted at A < B
    const int x = ((i >> A) << (A + 1)) | (i & ((1 << A) - 1));
    return ((x >> B) << (B + 1)) | (x & ((1 << B) - 1));
}

template <int R, int A, int B, typename M>
__host__ __device__ __forceinline__ void tile_gen2(Amp (&a)[1 << R], uint32_t mask, M m, bool on) {
#pragma unroll
    for (int p = 0; p < 1 << (R - 2); ++p) {
        const int i = zero2<A, B>(p);
        const int idx[4] = {i, i | 1 << A, i | 1 << B, i | 1 << A | 1 << B};
        if (mask >> i & 1) tile_rows<R, 4>(a, idx, m, on);
    }
}

template <int R, typename M>
__host__ __device__ __forceinline__ void tile_generic(Amp (&a)[1 << R], uint32_t code, uint32_t mask, M m, bool on) {
    static_assert(R == 3, "register codes are written out for three register qubits");
    if (code == kOpGen2)
        tile_gen2<R, 0, 1>(a, mask, m, on);
    else if (code == kOpGen2 + 1)
        tile_gen2<R, 0, 2>(a, mask, m, on);
    else if (code == kOpGen2 + 2)
        tile_gen2<R, 1, 2>(a, mask, m, on);
    else {
        const int idx[8] = {0, 1, 2, 3, 4, 5, 6, 7};
        tile_rows<R, 8>(a, idx, m, on);
    }
}

// LDS position of tile amplitude i: the low bits of the index are mixed with
// the next ones, so that orbits at any stride of two spread over the banks.
// Linear over XOR.
__host__ __device__ __forceinline__ uint32_t tile_slot(uint32_t i) { return i ^ (i >> 4 & 15); }

__host__ __device__ __forceinline__ uint32_t tile_zero(uint32_t x, uint32_t p) {
    const uint32_t low = (1u << p) - 1;
    return ((x & ~low) << 1) | (x & low);
}

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
    return uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(x >> 32)))) << 32 |
           uint32_t(__builtin_amdgcn_readfirstlane(int(x)));
}

// One pass over a state stored as T, computed in FP64 whatever T: complex64
// amplitudes are rounded once per pass instead of once per gate. (Gate by
// gate in FP32 a 27-qubit circuit of 867 gates came out 1.3e-6 off in its
// expectation values, in dense FP32 blocks 4e-7, in FP64 passes 2e-8.)
//
// 592 gates on 25 qubits in complex128: 8.5 ms, in dense blocks of five qubits
// 19.6 ms; 600 gates on 16 qubits from a graph: 0.37 ms, one launch a gate
// 1.44 ms; the 27-qubit circuit 13.4 ms, in dense blocks 19.2 ms. Vector
// instructions bound a pass of many gates, bytes one of few.
//
// The first and the last round hold the top R tile qubits, the layout of the
// global loads and stores, so they need no LDS. An exchange takes 50 vector
// instructions: the register bits add to a place by XOR of scalars, the places
// of a round's reads serve the writes that end it, and an amplitude stays in
// one register quadruple from the read through all operations to the write.
// (Places formed per amplitude from the thread's index, twice, and amplitudes
// in halves that were moved together for each write, took 170: 8.86 ms on 25
// qubits, 14.6 on 27, 0.395 on 16.)
template <typename T, int R, bool NT>
__global__ __launch_bounds__(1 << (kTileMax - R), 4) void k_tile(cv<T>* __restrict__ psi, TileGeo geo,
                                                                 const uint32_t* __restrict__ stream, uint64_t boff) {
    // aligned to its size, so that places in it are joined by XOR
    extern __shared__ __attribute__((aligned(sizeof(Amp) << kTileMax))) unsigned char smem_raw[];
    typedef __attribute__((address_space(3))) unsigned char* lds_bytes;
    typedef __attribute__((address_space(3))) Amp* lds_amp;
    typedef const __attribute__((address_space(4))) uint32_t* words;
    typedef const __attribute__((address_space(4))) double* reals;
    words w = (words)stream;
    const uint32_t tid = threadIdx.x, t = geo.t;
    const bool active = tid < 1u << (t - R);
    const uint32_t tile = uint32_t(block_id<8>() + boff);
    uint64_t base = tile;
    uint64_t off = 0;
    for (uint32_t i = 0; i < t; ++i) {
        const uint64_t low = (1ull << geo.pos[i]) - 1;
        base = ((base & ~low) << 1) | (base & low);
        if (i < t - R) off |= uint64_t(tid >> i & 1) << geo.pos[i];
    }
    uint64_t hi[1 << R];
#pragma unroll
    for (int k = 0; k < 1 << R; ++k) {
        hi[k] = 0;
#pragma unroll
        for (int i = 0; i < R; ++i) hi[k] |= uint64_t(k >> i & 1) << geo.pos[t - R + i];
    }
    cv<T>* p = psi + (base | off);
    Amp a[1 << R] = {};  // threads past the tile hold zeros, in LDS past the tile's
    if (active) {
#pragma unroll
        for (int k = 0; k < 1 << R; ++k) {
            const cv<T> v = ldamp<T, NT>(p + hi[k]);
            a[k] = Amp{double(v.x), double(v.y)};
        }
    }
    uint32_t regs = 0;
#pragma unroll
    for (uint32_t i = 0; i < R; ++i) regs |= (t - R + i) << (8 * i);
    // The thread's amplitude 0 in LDS, and what the register bits add to a
    // place there (XOR): kept from a round's reads for the writes that end it.
    uint32_t slot = 0, add[R] = {};
    auto layout = [&](uint32_t regs) {
        slot = tid;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            slot = tile_zero(slot, regs >> (8 * i) & 255);
            add[i] = tile_slot(1u << (regs >> (8 * i) & 255)) * uint32_t(sizeof(Amp));
            asm("" : "+s"(add[i]));  // stays a scalar
        }
        slot = uint32_t(reinterpret_cast<uintptr_t>((lds_bytes)smem_raw)) | tile_slot(slot) * uint32_t(sizeof(Amp));
    };
    auto place = [&](int k) {
        uint32_t c = 0;
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (k >> i & 1) c ^= add[i];
        return (lds_amp)(uintptr_t)(slot ^ c);
    };
    layout(regs);
    uint32_t head = w[0], lane = w[1], mask = w[2], blk = w[3];
    for (;;) {
        uint32_t code = head & 0xffff;
        while (code < kOpGen2) {
            // the entries and the next record's head, on their way while the
            // masks are formed
            const reals m = (reals)(w + kHead);
            double f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = m[i];
            w += head >> 16;
            const uint32_t h0 = w[0], h1 = w[1], h2 = w[2], h3 = w[3];
            const uint64_t lanes = __ballot((tid & (lane & 0xffff)) == lane >> 16);
            const uint64_t on = uniform64((tile & blk) == blk ? lanes : 0);
            const bool pick = (mask & kPickBit) && (tile >> (mask >> 16 & 31) & 1);
            f[0] = pick ? f[2] : f[0];
            f[1] = pick ? f[3] : f[1];
            tile_simple(a, code, mask, f, on, tid, tile);
            head = h0;
            lane = h1;
            mask = h2;
            blk = h3;
            code = head & 0xffff;
        }
        if (code == kOpEnd) break;
        const words body = w + kHead;
        w += head >> 16;
        const uint32_t h0 = w[0], h1 = w[1], h2 = w[2], h3 = w[3];  // the next record, ahead of the exchange
        if (code == kOpRound) {
            // from the layout of the round before to this one's; a thread
            // writes back only what it alone has read, so one barrier is enough
#pragma unroll
            for (int k = 0; k < 1 << R; ++k) *place(k) = a[k];
            __syncthreads();
            layout(lane);
#pragma unroll
            for (int k = 0; k < 1 << R; ++k) a[k] = *place(k);
        } else if ((tile & blk) == blk) {
            tile_generic<R>(a, code, mask, (reals)body, (tid & (lane & 0xffff)) == lane >> 16);
        }
        head = h0;
        lane = h1;
        mask = h2;
        blk = h3;
    }
    if (active) {
#pragma unroll
        for (int k = 0; k < 1 << R; ++k) {
            cv<T> v;
            v.x = T(a[k].x);
            v.y = T(a[k].y);
            stamp<T, NT>(p + hi[k], v);
        }
    }
}

// ---------------------------------------------------------------------------
// Host side.

template <typename T>
static int tile_launch(qcs_register* r, const TileGeo& geo, const uint32_t* stream, bool nt) {
    const uint64_t tiles = r->A >> geo.t;
    const unsigned threads = std::max(64u, 1u << (geo.t - kTileReg));
    const size_t shm = std::max<size_t>(sizeof(Amp) << geo.t, sizeof(Amp) * threads << kTileReg);
    for (uint64_t boff = 0; boff < tiles; boff += kMaxBlocks) {
        const unsigned grid = unsigned(std::min(kMaxBlocks, tiles - boff));
        if (nt)
            hipLaunchKernelGGL((k_tile<T, kTileReg, true>), dim3(grid), dim3(threads), shm, r->stream,
                               static_cast<cv<T>*>(r->psi), geo, stream, boff);
        else
            hipLaunchKernelGGL((k_tile<T, kTileReg, false>), dim3(grid), dim3(threads), shm, r->stream,
                               static_cast<cv<T>*>(r->psi), geo, stream, boff);
    }
    return check_launch(r, "k_tile");
}

static int apply_one(qcs_register* r, const qcs_gate& g) {
    const bool dense = (g.flags & QCS_GATE_DENSE) || g.k > 3;
    return dense ? qcs_apply_dense(r, g.k, g.qubits, g.mat)
                 : qcs_apply_gate(r, g.k, g.traits, g.qubits[0], g.qubits[1], g.qubits[2], g.mat);
}

// Whether the gate passes the checks of its entry point.
static bool gate_ok(const qcs_register* r, const qcs_gate& g) {
    if (g.k < 1 || g.k > 5) return false;
    for (uint32_t i = 0; i < g.k; ++i) {
        if (g.qubits[i] >= r->n) return false;
        for (uint32_t j = 0; j < i; ++j)
            if (g.qubits[i] == g.qubits[j]) return false;
    }
    return true;
}

size_t gates_param_bound(const qcs_register* r, const qcs_gate& g) {
    if (g.k > 3) return (r->mat_bytes + 255) & ~size_t(255);
    // its operation, a pass of its own with three rounds, the upload's rounding
    const size_t D = size_t(1) << g.k;
    return 2 * D * D * sizeof(double) + (6 * kHead + kTail) * 4 + 256;
}

// What a pass's stream may take: a staging slot, less its rounding.
static size_t stream_bytes(const qcs_register* r) { return r->mat_bytes - 256; }

template <typename T>
static int run_tiles(qcs_register* r, const qcs_gate* gates, uint32_t n) {
    TilePlanner plan(gates, n, r->n, r->amp_bytes(), stream_bytes(r));
    struct Pass {
        TileGeo geo;
        size_t at;  // first word of its stream
    };
    std::vector<Pass> passes;
    std::vector<uint32_t> words, one;
    size_t batch = 1;  // passes per upload: few at first, so that the GPU starts early
    auto flush = [&]() -> int {
        if (passes.empty()) return QCS_OK;
        const void* dev = nullptr;
        if (const int e = stage_upload(r, words.data(), words.size() * 4, &dev)) return e;
        for (const Pass& p : passes)
            if (const int e = tile_launch<T>(r, p.geo, static_cast<const uint32_t*>(dev) + p.at, plan.big())) return e;
        passes.clear();
        words.clear();
        batch *= 2;
        return QCS_OK;
    };
    Pass p{};
    const qcs_gate* single = nullptr;
    while (plan.next(p.geo, one, &single)) {
        if (single) {
            if (const int e = flush()) return e;
            if (const int e = apply_one(r, *single)) return e;
            continue;
        }
        if ((words.size() + one.size()) * 4 > r->mat_bytes)
            if (const int e = flush()) return e;
        p.at = words.size();
        words.insert(words.end(), one.begin(), one.end());
        passes.push_back(p);
        if (passes.size() >= batch)
            if (const int e = flush()) return e;
    }
    return flush();
}

uint32_t fused_blocks(const qcs_register* r, const qcs_gate* gates, uint32_t n, uint32_t lo, uint32_t hi) {
    return blocks_width(gates, n, r->n, r->amp_bytes(), stream_bytes(r), lo, hi);
}

// The gates in order: in tile passes, or one launch each where a pass does
// not pay. The first gate that its entry point refuses ends the list with
// that error, the gates before it applied.
int run_gates(qcs_register* r, const qcs_gate* gates, uint32_t n) {
    uint32_t ok = 0;
    while (ok < n && gate_ok(r, gates[ok])) ++ok;
    if (r->n < uint32_t(kTileReg)) {
        for (uint32_t i = 0; i < ok; ++i)
            if (const int e = apply_one(r, gates[i])) return e;
    } else if (const int e = r->prec == QCS_COMPLEX128 ? run_tiles<double>(r, gates, ok) : run_tiles<float>(r, gates, ok)) {
        return e;
    }
    return ok < n ? apply_one(r, gates[ok]) : QCS_OK;
}

}  // namespace qcs
