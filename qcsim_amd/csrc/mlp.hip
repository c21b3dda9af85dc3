// mlp.hip - MLP surrogate for QAOA energies: forward, backward and Adam in
// hand-written HIP kernels. No counterpart in the reference.
//
// Network: in -> H -> H -> ... -> 1 (L hidden layers of width H, ReLU), BF16
// weights and activations, FP32 accumulation; FP32 master weights, FP32
// gradients, Adam. Loss: mean squared error. BF16 is stored as the top 16
// bits of an IEEE float, rounded to nearest even (bf16_from), so a CPU
// restatement reproduces every rounding.
//
// Every product is summed in FP32 in ascending order of the summed index,
// one FMA per term. The FP32 matrix instructions (v_mfma_f32_16x16x4_f32)
// do exactly that: their result equals the scalar FMA chain bit for bit
// (checked on the device, denormals included), so the matrix kernels below
// and the vector-ALU kernel for wide networks give the same numbers. The
// BF16 matrix instructions round in another order and are not used.
//
// Two kernels make a training step for networks of up to 256 inputs and 256
// hidden units. Rows of a batch are independent until the weight gradients,
// so k_mlp_rows takes a block of rows through the whole forward pass, the
// loss and the whole backward pass with the activations in LDS; k_mlp_dw
// then sums every layer's weight and bias gradients over the batch and
// applies Adam in its epilogue. Measured on MI355X (17 -> 256 x 3 -> 1,
// batch 4096): 70 us a step, against 5.4 ms for GEMMs and column sums that put
// one block of 256 threads, or 16 blocks, on a sum over the batch.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "common.h"

namespace qcs {

typedef uint16_t bf16;

__host__ __device__ inline bf16 bf16_from(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return bf16(u >> 16);
}
__host__ __device__ inline float bf16_to(bf16 h) { return __builtin_bit_cast(float, uint32_t(h) << 16); }

template <typename T> __device__ inline float ldf(const T* p) { return float(*p); }
template <> __device__ inline float ldf<bf16>(const bf16* p) { return bf16_to(*p); }

enum { EPI_RELU_BF16 = 0, EPI_LINEAR_F32 = 1, EPI_MASK_F32 = 2 };

// C[M x N] = A[M x K] * op(B)[K x N] with an epilogue, on the vector ALUs
// (64x64x16 LDS tiles, 4x4 outputs per thread): the layers of networks wider
// than k_mlp_rows holds. A is M x K row-major (lda), B K x N row-major or,
// with TB_, N x K row-major (ldb).
template <typename TA, typename TB, bool TB_, int EPI>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const TA* __restrict__ A, int lda,
                                              const TB* __restrict__ B, int ldb, float* __restrict__ Cf,
                                              bf16* __restrict__ Cb, int ldc, const float* __restrict__ bias,
                                              const bf16* __restrict__ mask, int ldm) {
    __shared__ float As[16][64 + 4];
    __shared__ float Bs[16][64 + 4];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += 16) {
        for (int e = threadIdx.x; e < 1024; e += 256) {
            // A tile: 64 rows (m) x 16 cols (k)
            const int mm = e >> 4, kk = e & 15;
            const int gm = m0 + mm, gk = k0 + kk;
            float v = 0.f;
            if (gm < M && gk < K) v = ldf<TA>(A + size_t(gm) * lda + gk);
            As[kk][mm] = v;
            // B tile: 16 rows (k) x 64 cols (n)
            const int kb = e >> 6, nb = e & 63;
            const int gkb = k0 + kb, gn = n0 + nb;
            float w = 0.f;
            if (gkb < K && gn < N) w = TB_ ? ldf<TB>(B + size_t(gn) * ldb + gkb) : ldf<TB>(B + size_t(gkb) * ldb + gn);
            Bs[kb][nb] = w;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gm = m0 + ty * 4 + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int gn = n0 + tx * 4 + j;
            if (gn >= N) continue;
            float v = acc[i][j];
            if (EPI == EPI_RELU_BF16) {
                v += bias[gn];
                Cb[size_t(gm) * ldc + gn] = bf16_from(v > 0.f ? v : 0.f);
            } else if (EPI == EPI_LINEAR_F32) {
                Cf[size_t(gm) * ldc + gn] = v + bias[gn];
            } else {
                Cf[size_t(gm) * ldc + gn] = (bf16_to(mask[size_t(gm) * ldm + gn]) > 0.f) ? v : 0.f;
            }
        }
    }
}

// Output layer gradient for MSE: dY = 2 (y - t) / B; per-sample loss terms.
__global__ void k_mse(int Bn, int batch, const float* __restrict__ y, const float* __restrict__ t,
                      float4* __restrict__ dy, float* __restrict__ lossv) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= Bn) return;
    const float d = y[i] - t[i];
    dy[i] = float4{2.f * d / float(batch), 0.f, 0.f, 0.f};
    lossv[i] = d * d;
}

// A batch's inputs as BF16 rows of `ld` (zero past D) and its targets: row r
// is row idx[r] of the data set (or row r with no idx).
__global__ void k_gather(int Bn, int D, int ld, const uint32_t* __restrict__ idx, const float* __restrict__ X,
                         const float* __restrict__ Y, bf16* __restrict__ xb, float* __restrict__ yb) {
    const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= size_t(Bn) * ld) return;
    const int r = int(e / ld), c = int(e % ld);
    const size_t src = idx ? idx[r] : uint32_t(r);
    xb[e] = c < D ? bf16_from(X[src * D + c]) : bf16(0);
    if (c == 0 && Y) yb[r] = Y[src];
}

typedef float fx4 __attribute__((ext_vector_type(4)));

// J consecutive BF16 values and the float of element j.
template <int J> struct bvec;
template <> struct bvec<1> { using type = uint16_t; };
template <> struct bvec<2> { using type = uint32_t; };
__device__ __forceinline__ float bv_get(uint16_t v, int) { return bf16_to(v); }
__device__ __forceinline__ float bv_get(uint32_t v, int j) {
    return __builtin_bit_cast(float, j ? (v & 0xffff0000u) : (v << 16));
}
__device__ __forceinline__ void bv_set(uint16_t& v, int, bf16 b) { v = b; }
__device__ __forceinline__ void bv_set(uint32_t& v, int j, bf16 b) { v |= uint32_t(b) << (16 * j); }

constexpr int kMlpMaxLayers = 9;   // weight layers: at most 8 hidden ones and the output
constexpr int kMlpPad = 256;       // rows of a packed weight matrix are a multiple of this
constexpr int kMlpWide = 256;      // k_mlp_rows: widest layer

struct MlpRows {
    int B, in, L, H;
    int batch;                          // rows of the batch these are of: what its mean is over
    int ldx;                            // LDS rows and stride of the BF16 inputs (multiple of 32)
    int groups;                         // LDS size: groups of 16 columns per row tile
    const float* X;                     // inputs, rows of `in`
    const uint32_t* idx;                // row of X per batch row (null: in order)
    const float* T;                     // targets, by row of X (training)
    const bf16* W[kMlpMaxLayers];       // packed weights, K x NP
    const bf16* Wt[kMlpMaxLayers];      // packed transposes, NP x NP
    const float* bias[kMlpMaxLayers];
    bf16* x0;                           // B x ldx
    bf16* act[kMlpMaxLayers];           // B x NP
    float* dz[kMlpMaxLayers];           // B x NP: gradient before the ReLU of hidden layer l
    float* y;
    float4* dy;                         // (dy, 0, 0, 0): rows k_mlp_dw can load
    float* lossv;
};

// The rows [16 RT b, 16 RT (b + 1)) of a batch through the network, and with
// TRAIN through the loss and back: dz of every hidden layer and the BF16
// activations go to memory for k_mlp_dw.
//
// NW waves split a layer's NP = 16 J NW outputs; J consecutive columns per
// lane, so that one load of J BF16 weights per k feeds J matrix
// instructions (column c J + j of a wave is column c of its j-th 16 x 16
// tile) and the activations come from LDS in the operand order, four k per
// ds_read_b128 (element (row, k) at ((k / 16) 64 + (k % 4) 16 + row) 4 +
// k / 4 % 4). Weights stay in L2 and are loaded chunks ahead of their
// use, across layers too, since they do not depend on the activations. Bound: the FP32 matrix rate (138 TFLOP/s measured)
// for large batches. RT = 1 (16 rows) for batches that would otherwise leave
// CUs idle, RT = 2 halves the weight traffic per row. Measured (17 -> 256 x
// 3 -> 1): training, 4096 rows, 40 us (46 with four waves of J = 4); forward,
// 15360 rows, 49 us (86 TFLOP/s; 105 us per layer and 65536 rows before, on
// the vector ALUs).
template <int J, int NW, int RT, bool TRAIN>
__global__ __launch_bounds__(64 * NW) void k_mlp_rows(MlpRows a) {
    constexpr int NP = 16 * J * NW, CK = NP / 4, CG = CK / 16, NT = 64 * NW;
    constexpr int NS = RT == 1 ? 4 : 2;  // chunks in flight: one block per CU needs more
    using bv = typename bvec<J>::type;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* buf = sm;                              // RT x groups x 64 x 4
    float* wl = buf + RT * a.groups * 256;        // NP: output weights in operand order
    float* dys = wl + NP;                         // 16 RT
    uint32_t* mask = reinterpret_cast<uint32_t*>(dys + 16 * RT);  // L x NT: ReLU signs per thread
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, kk = lane >> 4;
    const int row0 = int(blockIdx.x) * 16 * RT, n0 = wave * 16 * J + c * J;
    const int G = a.groups;

    // The weights in the order the products use them, in chunks of CK k: the
    // forward layers, then (TRAIN) the transposes of layers L-1..1. Chunk i
    // lives in register set i % NS; fetch loads the next one into a set.
    bv wr[NS][CK / 4];
    int fp = 0, fc = 0;
    const int products = TRAIN ? 2 * a.L - 1 : a.L;
    const int chunks0 = (a.ldx + NS * CK - 1) / (NS * CK) * NS;  // of the first product; the others have 4
    auto fetch = [&](bv (&w)[CK / 4]) {
        if (fp >= products) return;
        const bf16* p = (fp < a.L ? a.W[fp] : a.Wt[2 * a.L - 1 - fp]) + size_t(fc * CK + kk) * NP + n0;
#pragma unroll
        for (int s = 0; s < CK / 4; ++s) w[s] = *reinterpret_cast<const bv*>(p + size_t(4 * s) * NP);
        if (++fc == (fp ? 4 : chunks0)) {
            fc = 0;
            ++fp;
        }
    };
    auto at = [&](int rt, int row, int k) {
        return ((rt * G + (k >> 4)) * 64 + (k & 3) * 16 + row) * 4 + ((k >> 2) & 3);
    };
    // inputs: NT / 16 threads per row, RT rows per thread; the row numbers are
    // on their way while the first weights are asked for
    uint32_t src[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = min(row0 + rt * 16 + tid / (NT / 16), a.B - 1);
        src[rt] = a.idx ? a.idx[row] : uint32_t(row);
    }
    uint32_t tsrc[4] = {0, 0, 0, 0};
    if (TRAIN)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = min(row0 + (wave < RT ? wave : 0) * 16 + 4 * kk + r, a.B - 1);
            tsrc[r] = a.idx ? a.idx[row] : uint32_t(row);
        }
#pragma unroll
    for (int i = 0; i < NS; ++i) fetch(wr[i]);
    float target[4] = {0.f, 0.f, 0.f, 0.f};
    if (TRAIN)
#pragma unroll
        for (int r = 0; r < 4; ++r) target[r] = a.T[tsrc[r]];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int r = tid / (NT / 16), row = row0 + rt * 16 + r;
        const float* x = a.X + size_t(src[rt]) * a.in;
        for (int k = tid % (NT / 16); k < a.ldx; k += NT / 16) {
            const bf16 h = row < a.B && k < a.in ? bf16_from(x[min(k, a.in - 1)]) : bf16(0);
            buf[at(rt, r, k)] = bf16_to(h);
            if (TRAIN && row < a.B) a.x0[size_t(row) * a.ldx + k] = h;
        }
    }
    for (int k = tid; k < NP; k += NT)
        wl[((k >> 4) * 4 + (k & 3)) * 4 + ((k >> 2) & 3)] = k < a.H ? bf16_to(a.W[a.L][k]) : 0.f;
    __syncthreads();

    // acc = (rows of buf) x (next matrix in the order) over `groups` x 16 k
    fx4 acc[RT][J];
    auto product = [&](int groups) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[rt][j] = fx4{0.f, 0.f, 0.f, 0.f};
        for (int g0 = 0; g0 < groups; g0 += NS * CG) {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const int g = g0 + i * CG;
                if (g < groups) {
                    // the chunk's activations, then per 16 k the unpacked
                    // weights ahead of their matrix instructions (the barrier
                    // keeps the compiler from pairing each with its unpacking
                    // through one register, which stalls)
                    fx4 x[CG][RT];
                    float w[2][4][J];
#pragma unroll
                    for (int q = 0; q < CG; ++q)
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt)
                            x[q][rt] = *reinterpret_cast<const fx4*>(buf + ((rt * G + min(g + q, G - 1)) * 64 + lane) * 4);
                    auto unpack = [&](int q) {
#pragma unroll
                        for (int s = 0; s < 4; ++s)
#pragma unroll
                            for (int j = 0; j < J; ++j) w[q & 1][s][j] = bv_get(wr[i][4 * q + s], j);
                    };
                    unpack(0);
#pragma unroll
                    for (int q = 0; q < CG; ++q) {
                        if (q + 1 < CG) unpack(q + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        if (g + q < groups) {
#pragma unroll
                            for (int s = 0; s < 4; ++s)
#pragma unroll
                                for (int j = 0; j < J; ++j)
#pragma unroll
                                    for (int rt = 0; rt < RT; ++rt)
                                        acc[rt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q][rt][s], w[q & 1][s][j],
                                                                                          acc[rt][j], 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                fetch(wr[i]);
            }
        }
    };

    for (int l = 0; l < a.L; ++l) {
        float b[J];
#pragma unroll
        for (int j = 0; j < J; ++j) b[j] = a.bias[l][min(n0 + j, a.H - 1)];
        product(l ? NP / 16 : a.ldx / 16);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; ++j) b[j] = n0 + j < a.H ? b[j] : 0.f;
        uint32_t on = 0;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 4 * kk + r;
                bv out{};
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    const float v = acc[rt][j][r] + b[j];
                    const bf16 h = bf16_from(v > 0.f ? v : 0.f);
                    buf[at(rt, row, n0 + j)] = bf16_to(h);
                    bv_set(out, j, h);
                    if (TRAIN) on |= (bf16_to(h) > 0.f ? 1u : 0u) << ((rt * J + j) * 4 + r);
                }
                if (TRAIN && row0 + rt * 16 + row < a.B)
                    *reinterpret_cast<bv*>(a.act[l] + size_t(row0 + rt * 16 + row) * NP + n0) = out;
            }
        if (TRAIN) mask[l * NT + tid] = on;
        __syncthreads();
    }

    // output layer: a wave per 16 rows, the weight vector in every column
    if (wave < RT) {
        fx4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int g = 0; g < NP / 16; ++g) {
            const fx4 x = *reinterpret_cast<const fx4*>(buf + ((wave * G + g) * 64 + lane) * 4);
            const fx4 w = *reinterpret_cast<const fx4*>(wl + (g * 4 + kk) * 4);
#pragma unroll
            for (int s = 0; s < 4; ++s) o = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], w[s], o, 0, 0, 0);
        }
        if (c == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int rr = wave * 16 + 4 * kk + r, row = row0 + rr;
                const float y = o[r] + a.bias[a.L][0];
                float dy = 0.f;
                if (row < a.B) {
                    a.y[row] = y;
                    if (TRAIN) {
                        const float d = y - target[r];
                        dy = 2.f * d / float(a.batch);
                        a.dy[row] = float4{dy, 0.f, 0.f, 0.f};
                        a.lossv[row] = d * d;
                    }
                }
                if (TRAIN) dys[rr] = dy;
            }
        }
    }
    if (!TRAIN) return;
    __syncthreads();

    // backward: dz of the last hidden layer from the output weights, then
    // through the transposed weights; the signs are this thread's own
    for (int l = a.L - 1; l >= 0; --l) {
        if (l < a.L - 1) {
            product(NP / 16);
            __syncthreads();
        }
        const uint32_t on = mask[l * NT + tid];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 4 * kk + r;
                float z[J];
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    const int n = n0 + j;
                    const float v = l == a.L - 1
                                        ? dys[rt * 16 + row] * wl[((n >> 4) * 4 + (n & 3)) * 4 + ((n >> 2) & 3)]
                                        : acc[rt][j][r];
                    z[j] = (on >> ((rt * J + j) * 4 + r)) & 1u ? v : 0.f;
                    if (l > 0) buf[at(rt, row, n)] = z[j];
                }
                if (row0 + rt * 16 + row < a.B) {
                    typedef float fxj __attribute__((ext_vector_type(J)));
                    fxj out;
#pragma unroll
                    for (int j = 0; j < J; ++j) out[j] = z[j];
                    *reinterpret_cast<fxj*>(a.dz[l] + size_t(row0 + rt * 16 + row) * NP + n0) = out;
                }
            }
        __syncthreads();
    }
}

// Adam on one FP32 master weight and its moments.
__device__ __forceinline__ void adam_step(float& w, float& m, float& v, float gi, float lr, float b1, float b2,
                                          float eps, float c1, float c2) {
    m = b1 * m + (1.f - b1) * gi;
    v = b2 * v + (1.f - b2) * gi * gi;
    w = w - lr * (m / c1) / (sqrtf(v / c2) + eps);
}

struct DwLayer {
    const bf16* A;   // layer inputs, B x lda
    const float* Z;  // gradients before the activation, B x ldz
    int lda, ldz, M, N;
    uint32_t woff, boff;      // flat offsets of the weights and biases
    bf16* wp;                 // packed weights (ldw) and transpose (ldt, may be null)
    bf16* wt;
    int ldw, ldt;
    uint32_t block0, nblk;    // first block, column blocks
};

constexpr int kDwRows = 192;  // rows of a slab

struct DwArgs {
    int B, nl;
    uint32_t blocks;          // blocks of the layers; one more sums the loss
    int adam;                 // update the weights, else store the gradients
    int more;                 // go on from the stored gradients: those of the batch's rows before these
    int lossn;                // loss terms to add up
    float *g, *w, *m, *v;
    float lr, b1, b2, eps, c1, c2;
    const float* lossv;
    float* loss;
    DwLayer layer[kMlpMaxLayers];
};

// Weight and bias gradients of every layer, and Adam: dW[m][n] = sum over the
// batch of A[k][m] Z[k][n], k ascending; row M of A is all ones, which makes
// that row the bias gradient. A block owns 32 x 32 outputs, a wave one 16 x
// 16 tile: one FMA chain per output over the whole batch is what the order
// asks for, so the time is the chain (18 ns per 4 rows, 19 us for 4096) and
// one tile per wave spreads the layers over the most CUs. Four waves multiply;
// four others bring slabs of 192 rows to LDS meanwhile, three ahead, one
// barrier a slab. Each matrix instruction keeps the next one of the chain
// waiting, and in that time one of the reads and conversions for later ones is
// issued. The last block adds the loss terms. Measured (17 -> 256 x 3 -> 1,
// 4096 rows): 29 us; with the reads of eight matrix instructions ahead of
// them 36 us; with the multiplying waves bringing the slabs themselves between
// two barriers each 46 us; with branches around the loads 75 us.
__global__ __launch_bounds__(512) void k_mlp_dw(DwArgs a) {
    constexpr int KS = kDwRows, NG = KS / 32, L = 32, NB = 4;  // rows of a slab, in groups of 32; columns; slabs in LDS
    __shared__ __attribute__((aligned(16))) float Zs[NB][KS * L];
    __shared__ __attribute__((aligned(16))) bf16 As[NB][KS * L];
    const int tid = threadIdx.x & 255;
    const bool stager = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // the same in a whole wave
    if (blockIdx.x == a.blocks) {  // not launched without loss terms
        float s = 0.f;
        if (!stager) {
            for (int i = tid; i < a.lossn; i += 256) s += a.lossv[i];
            Zs[0][tid] = s;
        }
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (!stager && tid < o) Zs[0][tid] += Zs[0][tid + o];
            __syncthreads();
        }
        if (threadIdx.x == 0) a.loss[0] = Zs[0][0];
        return;
    }
    int li = 0;
    while (li + 1 < a.nl && blockIdx.x >= a.layer[li + 1].block0) ++li;
    const DwLayer& y = a.layer[li];
    const int M = y.M, N = y.N, lda = y.lda, ldz = y.ldz;
    const int m0 = int((blockIdx.x - y.block0) / y.nblk) * 32, n0 = int((blockIdx.x - y.block0) % y.nblk) * 32;
    const int slabs = (a.B + KS - 1) / KS;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Both kinds of waves pass slabs + 1 barriers. After the first the first two
    // slabs are there, after each later one a slab is used up and one more there.
    if (stager) {
        // Every instruction these waves issue delays the matrix instructions of
        // the others on their SIMD: slabs go from memory to LDS directly, 1 KiB
        // an instruction, at fixed offsets of the thread from a scalar base.
        // Rows past the batch read as zeros through the descriptor's length
        // (which does not see a scalar offset beside it, hence none). A column
        // past the matrix reads one that is there; outputs of other columns are
        // not stored. The 16-byte pieces of a row of Z change
        // places by bit 1 of its index, for the banks of the reads.
        const int zch = (lane & 7) ^ (lane >> 4 & 1) << 2, ach = lane & 3;
        int zo[6], ao[3];
#pragma unroll
        for (int i = 0; i < 6; ++i)
            zo[i] = 4 * (((wave * 6 + i) * 8 + (lane >> 3)) * ldz + (n0 + zch * 4 < ldz ? n0 + zch * 4 : 0));
#pragma unroll
        for (int i = 0; i < 3; ++i)
            ao[i] = 2 * (((wave * 3 + i) * 16 + (lane >> 2)) * lda + (m0 + ach * 8 < lda ? m0 + ach * 8 : 0));
        auto load = [&](int slab) {
            auto rows = [&](const void* base, int bytes) {  // the slab's rows of the batch
                const int left = slab < slabs ? (a.B - slab * KS < KS ? a.B - slab * KS : KS) : 0;
                return __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<char*>(static_cast<const char*>(base)) + size_t(slab < slabs ? slab : 0) * KS * bytes, 0,
                    __builtin_amdgcn_readfirstlane(left * bytes), 0x00020000);
            };
            typedef __attribute__((address_space(3))) void lds_void;
            const auto Z = rows(y.Z, 4 * ldz), A = rows(y.A, 2 * lda);
            float* zs = Zs[slab % NB] + wave * 6 * 256;
            bf16* as = As[slab % NB] + wave * 3 * 512;
#pragma unroll
            for (int i = 0; i < 6; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(Z, (lds_void*)(zs + i * 256), 16, zo[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(A, (lds_void*)(as + i * 512), 16, ao[i], 0, 0, 0);
        };
        // all but the newest slab's nine loads are done
        auto ready = [] {
            __builtin_amdgcn_s_waitcnt(0x0f79);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        load(0);
        load(1);
        load(2);
        ready();
        for (int k = 0; k < slabs; ++k) {
            load(k + 3);
            ready();
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);  // none may land after this block's LDS is another's
        return;
    }
    const int c = lane & 15, kk = lane >> 4, wm = (wave & 1) * 16, wn = (wave >> 1) * 16;
    fx4 acc = {0.f, 0.f, 0.f, 0.f};
    const bool active = m0 + wm <= M && n0 + wn < N;
    // this thread's outputs, and what Adam needs of them: read now, these loads
    // would be most of the kernel's end
    const int n = n0 + wn + c;
    size_t at[4];
    bool mine[4];
    float aw[4], am[4], av[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 4 * kk + r;
        mine[r] = active && n < N && m <= M;
        at[r] = !mine[r] ? 0 : m < M ? y.woff + size_t(m) * N + n : y.boff + size_t(n);
        if (a.more) acc[r] = a.g[at[r]];
        if (a.adam) {
            aw[r] = a.w[at[r]];
            am[r] = a.m[at[r]];
            av[r] = a.v[at[r]];
        }
    }
    // Group by group, across slabs: the operands of the group after the next are
    // read while one is multiplied.
    uint32_t raw[2][8];  // BF16
    float x[2][8], z[3][8];
    const bool one = m0 + wm + c == M;
    auto read = [&](int t, const bf16* pa, const float* pz, int g, int u) {
        raw[t & 1][u] = pa[(32 * g + 4 * u) * L];
        z[t % 3][u] = pz[(32 * g + 4 * u) * L];
    };
    static_assert(NG % 6 == 0, "a slab begins with the first of each register set");
    const int zc = wn + c;
    const bf16* const pa0 = As[0] + kk * L + wm + c;
    const float* const pz0 = Zs[0] + kk * L + (((zc >> 2) ^ (kk >> 1 & 1) << 2) << 2 | (zc & 3));
    __syncthreads();
    auto convert = [&](int t, int u, auto ones) {
        x[t & 1][u] = __builtin_bit_cast(float, raw[t & 1][u] << 16);
        if (ones) x[t & 1][u] = one ? 1.f : x[t & 1][u];
    };
    auto chain = [&](auto ones) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            read(0, pa0, pz0, 0, u);
            read(1, pa0, pz0, 1, u);
            convert(0, u, ones);
        }
        const bf16* pa = pa0;
        const float* pz = pz0;
        for (int k = 0; k < slabs; ++k) {
            const int next = (k + 1) % NB;
            const bf16* const qa = pa0 + next * KS * L;
            const float* const qz = pz0 + next * KS * L;
            // whole slabs: rows past the batch are zero
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                // in order, so that the reads and conversions issue while a matrix
                // instruction keeps the next one waiting
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[g & 1][u], z[g % 3][u], acc, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    convert(g + 1, u, ones);
                    if (g + 2 < NG)
                        read(g + 2, pa, pz, g + 2, u);
                    else
                        read(g + 2, qa, qz, g + 2 - NG, u);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            pa = qa;
            pz = qz;
            __syncthreads();
        }
    };
    if (M >= m0 && M < m0 + 32)  // the column of ones is in this block
        chain(std::true_type{});
    else
        chain(std::false_type{});
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (!mine[r]) continue;
        if (!a.adam) {
            a.g[at[r]] = acc[r];
            continue;
        }
        adam_step(aw[r], am[r], av[r], acc[r], a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
        a.w[at[r]] = aw[r];
        a.m[at[r]] = am[r];
        a.v[at[r]] = av[r];
        const int m = m0 + wm + 4 * kk + r;
        if (m < M) {
            const bf16 h = bf16_from(aw[r]);
            y.wp[size_t(m) * y.ldw + n] = h;
            if (y.wt) y.wt[size_t(n) * y.ldt + m] = h;
        }
    }
}

// Packed BF16 copies of one layer's FP32 weights (M x N): rows of ldw, and
// the transpose in rows of ldt.
__global__ void k_pack(int M, int N, const float* __restrict__ w, bf16* __restrict__ wp, int ldw,
                       bf16* __restrict__ wt, int ldt) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M * N) return;
    const int m = i / N, n = i % N;
    const bf16 h = bf16_from(w[i]);
    wp[size_t(m) * ldw + n] = h;
    if (wt) wt[size_t(n) * ldt + m] = h;
}

}  // namespace qcs

using namespace qcs;

struct qcs_mlp {
    int in = 0, H = 0, L = 0;
    std::vector<int> dims;             // in, H, ..., H, 1
    std::vector<size_t> woff, boff;    // offsets into the flat parameter vector
    size_t nparams = 0;
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // FP32 master / grad / Adam
    // packed BF16 weights: per layer rows of ldw (padded with zeros to a
    // multiple of kMlpPad rows), and the transposes of layers 1..L-1
    bf16* wpack = nullptr;
    std::vector<size_t> poff, toff;
    int ldw = 0, ldx = 0;              // strides of hidden-wide and input rows
    bool rows_kernel = false;          // k_mlp_rows holds the network
    // activations and gradients of the rows in work: a batch's, or of a large
    // batch as many as slice says, one slice after the other
    int slice = 0;
    int cap = 0, rows_cap = 0;  // rows of outputs and loss terms; of the others
    bf16* x0 = nullptr;
    std::vector<bf16*> act;   // outputs of hidden layers (bf16)
    std::vector<float*> dz;   // gradients before their ReLU
    float* out = nullptr;     // network output (fp32)
    float4* dy = nullptr;     // its gradient, one per row
    float *yt = nullptr, *lossv = nullptr;
    bool train_bufs = false;  // the buffers only training needs are there
    float* lsum = nullptr;    // loss sums, one per step of an epoch
    size_t lsum_cap = 0;
    float* xin = nullptr;     // uploaded inputs of forward / gradients
    size_t xin_cap = 0;
    // dataset
    float *dX = nullptr, *dY = nullptr;
    uint32_t* didx = nullptr;
    uint64_t nrows = 0;
    hipStream_t stream = nullptr;
    hipStream_t up = nullptr;    // uploads of forward's input pieces, beside the launches
    hipEvent_t up_ev = nullptr;  // behind the last of them
    uint64_t step = 0;
};

template <typename T> static bool grow(T*& p, size_t& cap, size_t n) {
    if (n <= cap) return true;
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    if (hipMalloc(reinterpret_cast<void**>(&p), sizeof(T) * n) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    cap = n;
    return true;
}

// Buffers for batches of B rows, R of them in work at a time; `train`: those of
// the backward pass too.
static int mlp_reserve(qcs_mlp* n, int B, int R, bool train) {
    if (B < 0) return set_error(QCS_ENOMEM, "mlp activations");  // a batch past 2^31
    if (B <= n->cap && R <= n->rows_cap && (n->train_bufs || !train)) return QCS_OK;
    const size_t all = size_t(std::max(B, n->cap)), rows = size_t(std::max(R, n->rows_cap));
    if (hipStreamSynchronize(n->stream) != hipSuccess) return set_error(QCS_EDEVICE, "sync failed");
    auto fr = [](auto*& p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    };
    fr(n->x0);
    for (auto*& a : n->act) fr(a);
    for (auto*& z : n->dz) fr(z);
    fr(n->out);
    fr(n->dy);
    fr(n->yt);
    fr(n->lossv);
    n->cap = n->rows_cap = 0;
    train = train || n->train_bufs;
    n->train_bufs = false;
    auto get = [](auto*& p, size_t k) { return hipMalloc(reinterpret_cast<void**>(&p), sizeof(*p) * k) == hipSuccess; };
    bool ok = get(n->out, all);
    if (train || !n->rows_kernel) {
        ok = ok && get(n->x0, rows * n->ldx);
        for (auto*& a : n->act) ok = ok && get(a, rows * n->ldw);
    }
    if (train) {
        for (auto*& z : n->dz) ok = ok && get(z, rows * n->ldw);
        ok = ok && get(n->dy, rows) && get(n->yt, rows) && get(n->lossv, all);
    }
    if (!ok) {
        (void)hipGetLastError();
        return set_error(QCS_ENOMEM, "mlp activations");
    }
    n->cap = int(all);
    n->rows_cap = int(rows);
    n->train_bufs = train;
    return QCS_OK;
}

static dim3 ggrid(int M, int N) { return dim3(unsigned((N + 63) / 64), unsigned((M + 63) / 64)); }

template <int J, int NW, int RT, bool TRAIN> static void launch_rows(const MlpRows& a, hipStream_t s) {
    const size_t shm =
        sizeof(float) * (size_t(RT) * a.groups * 256 + 16 * J * NW + 16 * RT + (TRAIN ? a.L * 64 * NW : 0));
    hipLaunchKernelGGL((k_mlp_rows<J, NW, RT, TRAIN>), dim3(unsigned((a.B + 16 * RT - 1) / (16 * RT))), dim3(64 * NW),
                       shm, s, a);
}

template <int J, int NW> static void launch_rows_j(const MlpRows& a, bool train, hipStream_t s) {
    // 32 rows per block once 16 would give every CU more than two blocks
    const bool two = a.B > 16 * 2 * 256;
    if (train)
        two ? launch_rows<J, NW, 2, true>(a, s) : launch_rows<J, NW, 1, true>(a, s);
    else
        two ? launch_rows<J, NW, 2, false>(a, s) : launch_rows<J, NW, 1, false>(a, s);
}

// B rows of X (by idx, or in order) through the network into out; with
// `batch` (targets T, indexed like X) also through the loss, of a batch of that
// many rows, into lossv, and back.
static int mlp_rows(qcs_mlp* n, int B, const float* X, const uint32_t* idx, const float* T, int batch, float* out,
                    float* lossv) {
    const bool train = batch > 0;
    if (n->rows_kernel) {
        MlpRows a{};
        a.B = B;
        a.batch = batch;
        a.in = n->in;
        a.L = n->L;
        a.H = n->H;
        a.ldx = n->ldx;
        a.groups = std::max(n->ldx, n->ldw) / 16;
        a.X = X;
        a.idx = idx;
        a.T = T;
        for (int l = 0; l <= n->L; ++l) {
            a.W[l] = n->wpack + n->poff[l];
            a.Wt[l] = n->wpack + n->toff[l];
            a.bias[l] = n->w + n->boff[l];
        }
        a.x0 = n->x0;
        for (int l = 0; l < n->L; ++l) {
            a.act[l] = n->act[l];
            a.dz[l] = n->dz[l];
        }
        a.y = out;
        a.dy = n->dy;
        a.lossv = lossv;
        if (n->ldw == 64)
            launch_rows_j<1, 4>(a, train, n->stream);
        else if (n->ldw == 128)
            launch_rows_j<1, 8>(a, train, n->stream);
        else
            launch_rows_j<2, 8>(a, train, n->stream);
    } else {
        hipLaunchKernelGGL(k_gather, dim3(unsigned((size_t(B) * n->ldx + 255) / 256)), dim3(256), 0, n->stream, B, n->in,
                           n->ldx, idx, X, T, n->x0, n->yt);
        const bf16* x = n->x0;
        int din = n->in, ld = n->ldx;
        for (int l = 0; l < n->L; ++l) {
            hipLaunchKernelGGL((k_gemm<bf16, bf16, false, EPI_RELU_BF16>), ggrid(B, n->H), dim3(256), 0, n->stream, B,
                               n->H, din, x, ld, n->wpack + n->poff[l], n->ldw, nullptr, n->act[l], n->ldw,
                               n->w + n->boff[l], nullptr, 0);
            x = n->act[l];
            din = n->H;
            ld = n->ldw;
        }
        hipLaunchKernelGGL((k_gemm<bf16, bf16, false, EPI_LINEAR_F32>), ggrid(B, 1), dim3(256), 0, n->stream, B, 1, din,
                           x, ld, n->wpack + n->poff[n->L], 1, out, nullptr, 1, n->w + n->boff[n->L], nullptr, 0);
        if (train) {
            hipLaunchKernelGGL(k_mse, dim3((B + 255) / 256), dim3(256), 0, n->stream, B, batch, out, n->yt, n->dy, lossv);
            // dz_{l} = dz_{l+1} W^T, masked by ReLU' (activation > 0)
            for (int l = n->L - 1; l >= 0; --l) {
                const bool top = l == n->L - 1;
                hipLaunchKernelGGL((k_gemm<float, bf16, true, EPI_MASK_F32>), ggrid(B, n->H), dim3(256), 0, n->stream, B,
                                   n->H, top ? 1 : n->H, top ? reinterpret_cast<const float*>(n->dy) : n->dz[l + 1], top ? 4 : n->ldw,
                                   n->wpack + n->poff[l + 1], top ? 1 : n->ldw, n->dz[l], nullptr, n->ldw, nullptr,
                                   n->act[l], n->ldw);
            }
        }
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? QCS_OK : set_error(QCS_EDEVICE, "mlp rows: %s", hipGetErrorString(e));
}

// Gradients of the rows that mlp_rows has just taken back, added to n->g if
// they are not the batch's first (`more`), into n->g or (adam) straight into the
// weights; with `loss` the sum of the batch's loss terms goes there.
static int mlp_dw(qcs_mlp* n, int B, bool more, int batch, bool adam, float lr, float* loss) {
    DwArgs a{};
    a.B = B;
    a.nl = n->L + 1;
    a.adam = adam;
    a.more = more;
    a.lossn = batch;
    a.g = n->g;
    a.w = n->w;
    a.m = n->m;
    a.v = n->v;
    if (adam) {
        n->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        a.lr = lr;
        a.b1 = b1;
        a.b2 = b2;
        a.eps = 1e-8f;
        a.c1 = 1.f - std::pow(b1, float(n->step));
        a.c2 = 1.f - std::pow(b2, float(n->step));
    }
    a.lossv = n->lossv;
    a.loss = loss;
    for (int l = 0; l <= n->L; ++l) {
        DwLayer& y = a.layer[l];
        y.A = l ? n->act[l - 1] : n->x0;
        y.lda = l ? n->ldw : n->ldx;
        y.Z = l < n->L ? n->dz[l] : reinterpret_cast<const float*>(n->dy);
        y.ldz = l < n->L ? n->ldw : 4;
        y.M = n->dims[l];
        y.N = n->dims[l + 1];
        y.woff = uint32_t(n->woff[l]);
        y.boff = uint32_t(n->boff[l]);
        y.wp = n->wpack + n->poff[l];
        y.ldw = l < n->L ? n->ldw : 1;
        y.wt = l > 0 && l < n->L && n->rows_kernel ? n->wpack + n->toff[l] : nullptr;
        y.ldt = n->ldw;
        y.nblk = uint32_t((y.N + 31) / 32);
        y.block0 = a.blocks;
        a.blocks += y.nblk * uint32_t((y.M + 1 + 31) / 32);
    }
    hipLaunchKernelGGL(k_mlp_dw, dim3(a.blocks + (loss ? 1 : 0)), dim3(512), 0, n->stream, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? QCS_OK : set_error(QCS_EDEVICE, "mlp gradients: %s", hipGetErrorString(e));
}

// A batch of B rows through the network and back, in slices; its gradients and
// loss as mlp_dw leaves them. The sums over the batch go on from slice to slice in
// the order of its rows, so they do not depend on where it is cut.
static int mlp_batch(qcs_mlp* n, int B, const float* X, const uint32_t* idx, const float* T, bool adam, float lr,
                     float* loss) {
    for (size_t b0 = 0; b0 < size_t(B); b0 += n->slice) {
        const int P = int(std::min(size_t(n->slice), B - b0));
        const bool last = b0 + P == size_t(B);
        int e = mlp_rows(n, P, idx ? X : X + b0 * n->in, idx ? idx + b0 : nullptr, idx ? T : T + b0, B, n->out + b0,
                         n->lossv + b0);
        if (!e) e = mlp_dw(n, P, b0 > 0, B, adam && last, lr, last ? loss : nullptr);
        if (e) return e;
    }
    return QCS_OK;
}

// The packed BF16 copies from the FP32 weights.
static int mlp_pack(qcs_mlp* n) {
    for (int l = 0; l <= n->L; ++l) {
        const int M = n->dims[l], N = n->dims[l + 1];
        const bool t = l > 0 && l < n->L && n->rows_kernel;
        hipLaunchKernelGGL(k_pack, dim3(unsigned((size_t(M) * N + 255) / 256)), dim3(256), 0, n->stream, M, N,
                           n->w + n->woff[l], n->wpack + n->poff[l], l < n->L ? n->ldw : 1,
                           t ? n->wpack + n->toff[l] : nullptr, n->ldw);
    }
    return hipGetLastError() == hipSuccess && hipStreamSynchronize(n->stream) == hipSuccess
               ? QCS_OK
               : set_error(QCS_EDEVICE, "weight packing failed");
}

extern "C" {

int qcs_mlp_destroy(qcs_mlp* n) {
    if (!n) return QCS_OK;
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    void* ps[] = {n->w,  n->g,  n->m,     n->v,    n->wpack, n->x0, n->out, n->dy,
                  n->yt, n->xin, n->lossv, n->lsum, n->dX,    n->dY, n->didx};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    for (auto* a : n->act)
        if (a) (void)hipFree(a);
    for (auto* z : n->dz)
        if (z) (void)hipFree(z);
    if (n->up_ev) (void)hipEventDestroy(n->up_ev);
    if (n->up) (void)hipStreamDestroy(n->up);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
    return QCS_OK;
}

int qcs_mlp_create(uint32_t in_dim, uint32_t hidden, uint32_t layers, uint64_t seed, qcs_mlp** out) {
    if (!out || in_dim == 0 || hidden == 0 || layers == 0 || layers > 8) return set_error(QCS_EINVAL, "bad MLP shape");
    auto* n = new qcs_mlp;
    n->in = int(in_dim);
    n->H = int(hidden);
    n->L = int(layers);
    n->dims.push_back(n->in);
    for (int l = 0; l < n->L; ++l) n->dims.push_back(n->H);
    n->dims.push_back(1);
    size_t off = 0;
    for (int l = 0; l <= n->L; ++l) {
        n->woff.push_back(off);
        off += size_t(n->dims[l]) * n->dims[l + 1];
        n->boff.push_back(off);
        off += size_t(n->dims[l + 1]);
    }
    n->nparams = off;
    n->act.assign(n->L, nullptr);
    n->dz.assign(n->L, nullptr);
    // k_mlp_rows holds layers of up to kMlpWide units; wider networks run
    // layer by layer on the vector ALUs
    n->rows_kernel = n->in <= kMlpWide && n->H <= kMlpWide;
    n->ldx = (n->in + 31) / 32 * 32;
    n->ldw = !n->rows_kernel ? (n->H + 31) / 32 * 32 : n->H <= 64 ? 64 : n->H <= 128 ? 128 : 256;
    // of activations and gradients about 1 GiB at a time, in whole slabs of k_mlp_dw
    n->slice = std::max(int((size_t(1) << 30) / (size_t(n->L) * n->ldw * 6 + size_t(n->ldx) * 2)) / kDwRows, 1) * kDwRows;
    auto padded = [](int k) { return size_t((k + kMlpPad - 1) / kMlpPad * kMlpPad); };
    size_t packed = 0;
    for (int l = 0; l <= n->L; ++l) {
        n->poff.push_back(packed);
        packed += l < n->L ? padded(l ? n->ldw : n->ldx) * n->ldw : padded(n->H);
        n->toff.push_back(packed);
        if (l > 0 && l < n->L && n->rows_kernel) packed += padded(n->ldw) * n->ldw;
    }
    // He-uniform initialisation, zero biases
    std::vector<float> w(off, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l <= n->L; ++l) {
        const float lim = std::sqrt(6.f / float(n->dims[l]));
        std::uniform_real_distribution<float> U(-lim, lim);
        for (size_t i = 0; i < size_t(n->dims[l]) * n->dims[l + 1]; ++i) w[n->woff[l] + i] = U(rng);
    }
    bool ok = hipMalloc(reinterpret_cast<void**>(&n->w), sizeof(float) * off) == hipSuccess &&
              hipMalloc(reinterpret_cast<void**>(&n->g), sizeof(float) * off) == hipSuccess &&
              hipMalloc(reinterpret_cast<void**>(&n->m), sizeof(float) * off) == hipSuccess &&
              hipMalloc(reinterpret_cast<void**>(&n->v), sizeof(float) * off) == hipSuccess &&
              hipMalloc(reinterpret_cast<void**>(&n->wpack), sizeof(bf16) * packed) == hipSuccess &&
              hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        qcs_mlp_destroy(n);
        return set_error(QCS_ENOMEM, "mlp allocation failed");
    }
    const std::vector<float> zero(off, 0.f);
    const std::vector<bf16> pzero(packed, bf16(0));
    ok = hipMemcpy(n->w, w.data(), sizeof(float) * off, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->wpack, pzero.data(), sizeof(bf16) * packed, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->m, zero.data(), sizeof(float) * off, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->v, zero.data(), sizeof(float) * off, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        qcs_mlp_destroy(n);
        return set_error(QCS_EDEVICE, "mlp upload failed");
    }
    if (const int e = mlp_pack(n)) {
        qcs_mlp_destroy(n);
        return e;
    }
    *out = n;
    return QCS_OK;
}

uint64_t qcs_mlp_num_params(const qcs_mlp* n) { return n ? n->nparams : 0; }

// FP32 master parameters (the BF16 copies are refreshed on set).
int qcs_mlp_get_params(qcs_mlp* n, float* p) {
    if (!n || !p) return set_error(QCS_EINVAL, "null argument");
    return hipMemcpy(p, n->w, sizeof(float) * n->nparams, hipMemcpyDeviceToHost) == hipSuccess
               ? QCS_OK
               : set_error(QCS_EDEVICE, "download failed");
}

int qcs_mlp_set_params(qcs_mlp* n, const float* p) {
    if (!n || !p) return set_error(QCS_EINVAL, "null argument");
    if (hipMemcpy(n->w, p, sizeof(float) * n->nparams, hipMemcpyHostToDevice) != hipSuccess)
        return set_error(QCS_EDEVICE, "upload failed");
    return mlp_pack(n);
}

// Batches above this run in slices of this many rows.
static constexpr uint32_t kMlpSlice = 65536;
// Inputs are uploaded in pieces of at most this many bytes (what the runtime
// stages at once from pageable memory), on a stream of their own, so that the
// copy of a piece runs while the piece before it is computed; on one stream a
// pageable copy waits for the launches before it. 65536 rows of 17: 471 us
// on one stream, 330 us so. The stream comes with the first call of more than
// one piece: it takes as long to make as the rest of a network (0.9 ms with
// it, 0.5 without).
static constexpr size_t kMlpPiece = size_t(1) << 20;

int qcs_mlp_forward(qcs_mlp* n, const float* x, uint32_t batch, float* y) {
    if (!n || !x || !y || batch == 0) return set_error(QCS_EINVAL, "bad argument");
    for (uint32_t b0 = 0; b0 < batch; b0 += kMlpSlice) {
        const uint32_t B = std::min(kMlpSlice, batch - b0);
        if (const int e = mlp_reserve(n, int(B), n->rows_kernel ? 0 : int(B), false)) return e;
        if (!grow(n->xin, n->xin_cap, size_t(B) * n->in)) return set_error(QCS_ENOMEM, "mlp inputs");
        // wide networks keep one batch's activations: one piece
        const uint32_t fit = uint32_t(kMlpPiece / (sizeof(float) * n->in)) / 512 * 512;
        const uint32_t piece = n->rows_kernel ? std::max(fit, 512u) : B;
        for (uint32_t p0 = 0; p0 < B; p0 += piece) {
            const uint32_t P = std::min(piece, B - p0);
            float* xd = n->xin + size_t(p0) * n->in;
            const bool apart = piece < B;
            if (apart && !n->up && hipStreamCreateWithFlags(&n->up, hipStreamNonBlocking) != hipSuccess)
                return set_error(QCS_EDEVICE, "upload stream");
            if (apart && !n->up_ev && hipEventCreateWithFlags(&n->up_ev, hipEventDisableTiming) != hipSuccess)
                return set_error(QCS_EDEVICE, "upload event");
            if (hipMemcpyAsync(xd, x + size_t(b0 + p0) * n->in, sizeof(float) * P * n->in, hipMemcpyHostToDevice,
                               apart ? n->up : n->stream) != hipSuccess ||
                (apart && (hipEventRecord(n->up_ev, n->up) != hipSuccess ||
                           hipStreamWaitEvent(n->stream, n->up_ev, 0) != hipSuccess)))
                return set_error(QCS_EDEVICE, "input upload failed");
            if (const int e = mlp_rows(n, int(P), xd, nullptr, nullptr, 0, n->out + p0, nullptr)) return e;
        }
        if (hipMemcpyAsync(y + b0, n->out, sizeof(float) * B, hipMemcpyDeviceToHost, n->stream) != hipSuccess ||
            hipStreamSynchronize(n->stream) != hipSuccess)
            return set_error(QCS_EDEVICE, "forward failed");
    }
    return QCS_OK;
}

// Loss and FP32 gradients (flat, same layout as the parameters) of one batch.
int qcs_mlp_gradients(qcs_mlp* n, const float* x, const float* t, uint32_t batch, float* grad, float* loss) {
    if (!n || !x || !t || batch == 0) return set_error(QCS_EINVAL, "bad argument");
    const int B = int(batch);
    if (const int e = mlp_reserve(n, B, std::min(B, n->slice), true)) return e;
    if (!grow(n->xin, n->xin_cap, size_t(B) * (n->in + 1)) || !grow(n->lsum, n->lsum_cap, size_t(4)))
        return set_error(QCS_ENOMEM, "mlp inputs");
    float* td = n->xin + size_t(B) * n->in;
    if (hipMemcpyAsync(n->xin, x, sizeof(float) * B * n->in, hipMemcpyHostToDevice, n->stream) != hipSuccess ||
        hipMemcpyAsync(td, t, sizeof(float) * B, hipMemcpyHostToDevice, n->stream) != hipSuccess)
        return set_error(QCS_EDEVICE, "input upload failed");
    if (const int e = mlp_batch(n, B, n->xin, nullptr, td, false, 0.f, n->lsum)) return e;
    float l = 0;
    if ((grad && hipMemcpyAsync(grad, n->g, sizeof(float) * n->nparams, hipMemcpyDeviceToHost, n->stream) != hipSuccess) ||
        hipMemcpyAsync(&l, n->lsum, sizeof(float), hipMemcpyDeviceToHost, n->stream) != hipSuccess ||
        hipStreamSynchronize(n->stream) != hipSuccess)
        return set_error(QCS_EDEVICE, "gradient download failed");
    if (loss) *loss = l / float(B);
    return QCS_OK;
}

// Train on a device-resident copy of (X, Y): `epochs` passes of shuffled
// mini-batches, Adam with learning rate lr. loss_per_epoch (optional)
// receives the mean training loss of each epoch. An epoch's launches are
// queued without waiting; its step losses are fetched together at its end.
int qcs_mlp_train(qcs_mlp* n, const float* X, const float* Y, uint64_t rows, uint32_t batch, uint32_t epochs, float lr,
                  uint64_t seed, float* loss_per_epoch) {
    if (!n || !X || !Y || rows == 0 || batch == 0) return set_error(QCS_EINVAL, "bad argument");
    if (n->nrows != rows) {
        if (n->dX) (void)hipFree(n->dX);
        if (n->dY) (void)hipFree(n->dY);
        if (n->didx) (void)hipFree(n->didx);
        n->dX = nullptr;
        n->dY = nullptr;
        n->didx = nullptr;
        n->nrows = 0;
        if (hipMalloc(reinterpret_cast<void**>(&n->dX), sizeof(float) * rows * n->in) != hipSuccess ||
            hipMalloc(reinterpret_cast<void**>(&n->dY), sizeof(float) * rows) != hipSuccess ||
            hipMalloc(reinterpret_cast<void**>(&n->didx), sizeof(uint32_t) * rows) != hipSuccess)
            return set_error(QCS_ENOMEM, "dataset allocation failed");
        n->nrows = rows;
    }
    if (hipMemcpy(n->dX, X, sizeof(float) * rows * n->in, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(n->dY, Y, sizeof(float) * rows, hipMemcpyHostToDevice) != hipSuccess)
        return set_error(QCS_EDEVICE, "dataset upload failed");
    const uint64_t steps = rows / batch;
    if (const int e = mlp_reserve(n, int(batch), std::min(int(batch), n->slice), true)) return e;
    if (!grow(n->lsum, n->lsum_cap, size_t(std::max<uint64_t>(steps, 1)))) return set_error(QCS_ENOMEM, "loss buffer");
    std::vector<uint32_t> perm(rows);
    std::vector<float> losses(steps);
    for (uint64_t i = 0; i < rows; ++i) perm[i] = uint32_t(i);
    std::mt19937_64 rng(seed);
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        std::shuffle(perm.begin(), perm.end(), rng);
        // the stream may still read the indices of the epoch before
        if (hipStreamSynchronize(n->stream) != hipSuccess ||
            hipMemcpy(n->didx, perm.data(), sizeof(uint32_t) * rows, hipMemcpyHostToDevice) != hipSuccess)
            return set_error(QCS_EDEVICE, "index upload failed");
        for (uint64_t k = 0; k < steps; ++k) {
            if (const int e = mlp_batch(n, int(batch), n->dX, n->didx + k * batch, n->dY, true, lr, n->lsum + k)) return e;
        }
        if (loss_per_epoch) {
            if (steps && (hipMemcpyAsync(losses.data(), n->lsum, sizeof(float) * steps, hipMemcpyDeviceToHost,
                                         n->stream) != hipSuccess ||
                          hipStreamSynchronize(n->stream) != hipSuccess))
                return set_error(QCS_EDEVICE, "loss download failed");
            double lsum = 0;
            for (const float l : losses) lsum += l / int(batch);
            loss_per_epoch[ep] = steps ? float(lsum / double(steps)) : 0.f;
        }
    }
    return hipStreamSynchronize(n->stream) == hipSuccess ? QCS_OK : set_error(QCS_EDEVICE, "train sync failed");
}

}  // extern "C"
