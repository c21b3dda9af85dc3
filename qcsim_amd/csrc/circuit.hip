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
//
// Gates commute when they act diagonally on every qubit they share, so a
// pass takes, in list order, each gate that fits it and commutes with all
// gates left out before it; what is left keeps its order. The gates
// themselves are those of the gate kernels (same traits, same matrix
// entries), applied one by one.
#include <algorithm>
#include <cstring>
#include <vector>

#include "common.h"

namespace qcs {

constexpr int kTileReg = 3;    // register qubits of a round
constexpr int kTileMax = 12;   // tile qubits: 4096 amplitudes, 64 KiB of LDS

struct TileGeo {
    uint32_t t;
    uint8_t pos[kTileMax + 4];  // tile qubits, ascending
};

// An amplitude: four registers in a row, as LDS reads and writes take them.
typedef double Amp __attribute__((ext_vector_type(2)));

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
// The same in C++: what the host compiler sees of the kernel, and a statement
// of what each code does.
__host__ __device__ inline void tile_simple(Amp (&a)[8], uint32_t code, uint32_t mask, const double (&m)[8],
                                            uint64_t on, uint32_t tid, uint32_t tile) {
    if (!on) return;
    auto mul = [](Amp& x, double r, double i) { x = Amp{r * x.x - i * x.y, r * x.y + i * x.x}; };
    for (int i = 0; i < 8; ++i) {
        if (code >= kOpZ) {
            const uint64_t zt = uint32_t(__builtin_bit_cast(uint64_t, m[2]));
            const bool odd = (__builtin_popcount(i & (code - kOpZ)) + __builtin_popcount(tid & mask >> 8) +
                              __builtin_popcount(tile & zt)) & 1;
            mul(a[i], m[0], odd ? m[1] : -m[1]);
            continue;
        }
        if (!(mask >> i & 1)) continue;
        const uint32_t J = code & 3;  // register bit of the one-qubit codes
        if (code < kOpDiagR) {
            if (i >> J & 1) continue;
            Amp &x = a[i], &y = a[i | 1 << J];
            const Amp p = x, q = y;
            if (code >= kOpReal && code < kOpImag) {
                x = Amp{m[0] * p.x + m[1] * q.x, m[0] * p.y + m[1] * q.y};
                y = Amp{m[2] * p.x + m[3] * q.x, m[2] * p.y + m[3] * q.y};
            } else if (code >= kOpImag && code < kOpX) {
                x = Amp{m[0] * p.x - m[1] * q.y, m[0] * p.y + m[1] * q.x};
                y = Amp{m[3] * q.x - m[2] * p.y, m[3] * q.y + m[2] * p.x};
            } else if (code < kOpReal) {
                x = Amp{m[0] * p.x - m[1] * p.y + m[2] * q.x - m[3] * q.y,
                        m[0] * p.y + m[1] * p.x + m[2] * q.y + m[3] * q.x};
                y = Amp{m[4] * p.x - m[5] * p.y + m[6] * q.x - m[7] * q.y,
                        m[4] * p.y + m[5] * p.x + m[6] * q.y + m[7] * q.x};
            } else {
                std::swap(x, y);
                if (code >= kOpAnti) {
                    mul(x, m[0], m[1]);
                    mul(y, m[2], m[3]);
                }
            }
        } else if (code < kOpScale) {
            i >> J & 1 ? mul(a[i], m[2], m[3]) : mul(a[i], m[0], m[1]);
        } else if (code == kOpScale) {
            mul(a[i], m[0], m[1]);
        } else if (code == kOpNeg) {
            mul(a[i], -1, 0);
        } else {
            const uint32_t pair = code & 3;
            const int A = pair == 2 ? 1 : 0, B = pair == 0 ? 1 : 2;
            if (i >> A & 1 || i >> B & 1) continue;
            std::swap(a[i | 1 << A], a[i | 1 << B]);
            if (code >= kOpSwapP) {
                mul(a[i | 1 << A], m[0], m[1]);
                mul(a[i | 1 << B], m[0], m[1]);
            }
        }
    }
}
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
                                                                 const uint32_t* __restrict__ stream, uint32_t words_total,
                                                                 uint64_t boff) {
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
// Planning (host).

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

// CNOT(c, t) Z CNOT(c, t), with Z = exp(i phi) or its conjugate by the parity
// of qubits that include t, is such a gate too, in the parity that c joins or
// leaves: the Rz between two CNOTs of an Ising step, and the ladders around
// the rotations of Pauli strings. Each such sandwich becomes one gate: the
// same factor on the same amplitude (CNOTs move amplitudes unchanged), and a
// gate that any round can take. The gates that are left stay in order.
static std::vector<TileGate> tile_gates(const qcs_gate* gates, uint32_t n, uint32_t nq) {
    std::vector<TileGate> g;
    std::vector<uint8_t> gone;
    std::vector<std::vector<int>> on(nq);  // per qubit, the gates left that touch it
    g.reserve(n);
    auto drop = [&](uint32_t q, int i) { on[q].erase(std::find(on[q].begin(), on[q].end(), i)); };
    for (uint32_t k = 0; k < n; ++k) {
        const TileGate o = tile_gate(gates[k]);
        if (o.op == kOpX && popc(o.ctrl) == 1) {
            const uint32_t t = o.tq[0], c = uint32_t(__builtin_ctzll(o.ctrl));
            auto& ot = on[t];
            auto& oc = on[c];
            const int d = ot.size() > 1 ? ot.back() : -1, x = d >= 0 ? ot[ot.size() - 2] : -1;
            if (d >= 0 && g[x].op == kOpX && g[x].T == o.T && g[x].ctrl == o.ctrl) {
                TileGate& D = g[d];
                const bool has = D.D >> c & 1;
                if (D.op == kOpZ && (has ? oc.size() > 1 && oc.back() == d && oc[oc.size() - 2] == x : oc.back() == x)) {
                    drop(t, x);
                    drop(c, x);
                    gone[x] = 1;
                    D.src = nullptr;
                    D.D ^= 1ull << c;
                    if (has)
                        drop(c, d);
                    else
                        oc.push_back(d);
                    continue;
                }
            }
        }
        for (uint64_t m = o.T | o.D; m; m &= m - 1) on[__builtin_ctzll(m)].push_back(int(g.size()));
        g.push_back(o);
        g.back().src = &gates[k];
        gone.push_back(0);
    }
    size_t kept = 0;
    for (size_t i = 0; i < g.size(); ++i)
        if (!gone[i]) g[kept++] = g[i];
    g.resize(kept);
    return g;
}

// Gates in order with what each still waits for: a linked list of the gates
// not placed yet.
struct TilePlan {
    std::vector<TileGate> g;
    std::vector<int> next;
    int head = -1;
    uint32_t n = 0, t = 0;
    uint64_t all = 0, low = 0;
    size_t max_bytes = 0;  // of a pass's stream

    size_t op_bytes(const TileGate& o) const {
        return (kHead * 4 + 16 * o.nm + 15) / 16 * 16 + (!o.T ? 64 : 0);
    }
};

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

template <typename T>
static int tile_launch(qcs_register* r, const TileGeo& geo, const uint32_t* stream, uint32_t words, bool nt) {
    const uint64_t tiles = r->A >> geo.t;
    const unsigned threads = std::max(64u, 1u << (geo.t - kTileReg));
    const size_t shm = std::max<size_t>(sizeof(Amp) << geo.t, sizeof(Amp) * threads << kTileReg);
    for (uint64_t boff = 0; boff < tiles; boff += kMaxBlocks) {
        const unsigned grid = unsigned(std::min(kMaxBlocks, tiles - boff));
        if (nt)
            hipLaunchKernelGGL((k_tile<T, kTileReg, true>), dim3(grid), dim3(threads), shm, r->stream,
                               static_cast<cv<T>*>(r->psi), geo, stream, words, boff);
        else
            hipLaunchKernelGGL((k_tile<T, kTileReg, false>), dim3(grid), dim3(threads), shm, r->stream,
                               static_cast<cv<T>*>(r->psi), geo, stream, words, boff);
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

template <typename T>
static int run_tiles(qcs_register* r, const qcs_gate* gates, uint32_t n) {
    TilePlan P;
    P.n = r->n;
    P.t = tile_width(r->n);
    P.all = r->n >= 64 ? ~0ull : (1ull << r->n) - 1;
    const bool big = r->A * r->amp_bytes() > (size_t(64) << 20);
    P.low = (1ull << std::min<uint32_t>(r->n, big ? (sizeof(T) == 8 ? 4 : 5) : (sizeof(T) == 8 ? 3 : 4))) - 1;
    P.max_bytes = r->mat_bytes - 256;
    P.g = tile_gates(gates, n, r->n);
    P.next.resize(P.g.size());
    for (size_t i = 0; i < P.g.size(); ++i) P.next[i] = i + 1 < P.g.size() ? int(i + 1) : -1;
    P.head = P.g.empty() ? -1 : 0;

    struct Pass {
        TileGeo geo;
        size_t at;       // first word of its stream
        uint32_t words;  // its length
    };
    std::vector<Pass> passes;
    std::vector<uint32_t> words, one;
    size_t batch = 1;  // passes per upload: few at first, so that the GPU starts early
    auto flush = [&]() -> int {
        if (passes.empty()) return QCS_OK;
        const void* dev = nullptr;
        if (const int e = stage_upload(r, words.data(), words.size() * 4, &dev)) return e;
        for (const Pass& p : passes)
            if (const int e = tile_launch<T>(r, p.geo, static_cast<const uint32_t*>(dev) + p.at, p.words, big))
                return e;
        passes.clear();
        words.clear();
        batch *= 2;
        return QCS_OK;
    };
    std::vector<int> take;
    std::vector<const TileGate*> local;
    while (P.head >= 0) {
        const uint64_t S = tile_choose(P);
        take.clear();
        const double worth = tile_scan(P, S, &take);
        // A pass moves the whole state once: it has to replace launches that
        // move more. Where launches cost more than bytes it has to replace
        // three (us for 2 / 3 / 5 gates on 16 qubits, launches against passes:
        // 10 / 14 / 23 against 12 / 13 / 14; on 20 qubits 15 / 18 / 37 against
        // 18 / 18 / 23; on 25 qubits, by worth, 208 / 382 / 602 against
        // 177 / 211 / 225).
        const bool pass = P.g[P.head].op != kNoTile && (!P.g[P.head].src || (big ? worth > 1.2 : take.size() > 2));
        if (!pass) take.assign(1, P.head);
        int prev = -1;
        size_t k = 0;
        for (int i = P.head; i >= 0 && k < take.size(); i = P.next[i]) {
            if (i == take[k]) {
                ++k;
                (prev < 0 ? P.head : P.next[prev]) = P.next[i];
            } else {
                prev = i;
            }
        }
        if (!pass) {
            if (const int e = flush()) return e;
            if (const int e = apply_one(r, *P.g[take[0]].src)) return e;
            continue;
        }
        local.clear();
        for (const int i : take) local.push_back(&P.g[i]);
        Pass p{};
        uint64_t top = S;
        for (uint64_t x = S; x; x &= x - 1) p.geo.pos[p.geo.t++] = uint8_t(__builtin_ctzll(x));
        while (popc(top) > kTileReg) top &= top - 1;
        one.clear();
        tile_emit(local, tile_rounds(local, S, top), S, r->n, one);
        if ((words.size() + one.size()) * 4 > r->mat_bytes)
            if (const int e = flush()) return e;
        p.at = words.size();
        p.words = uint32_t(one.size());
        words.insert(words.end(), one.begin(), one.end());
        passes.push_back(p);
        if (passes.size() >= batch)
            if (const int e = flush()) return e;
    }
    return flush();
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
