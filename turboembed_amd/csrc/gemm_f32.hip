// The F32 tier's large products on the BF16 matrix cores. The F32 MFMA
// (v_mfma_f32_32x32x2f32) runs at a sixteenth of the BF16 one's rate, so each
// F32 operand is taken as the sum of three BF16 terms, each rounded to the
// nearest of what the ones before it left, x = x0 + x1 + x2 exactly (the
// split of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019), and a
// product as the six largest of its terms' products, x0 w0 + x0 w1 + x1 w0 +
// x0 w2 + x1 w1 + x2 w0, summed in F32, the five small ones apart from the
// first. |x1| is at most 2^-8 of x's power of two and |x2| 2^-17, so what is
// left out, x1 w2 + x2 w1 + x2 w2, is at most 2^-24 of a product (2^-27.4 in
// the root mean square over normal operands), what one rounding of an F32 sum
// may be off by; with x0 cut off instead, x1 is up to 2^-7, of x's own sign,
// and up to 2^-22 is left out (products 1% faster). And
// the sum of the x0 w0 products rounds once per 16 columns of k where the F32
// MFMA's rounds once per two. (From |x| = 2^-103 up: a smaller one's last
// term falls below BF16's normal range.)
// An infinite or NaN operand's terms differ by NaN, so its sums are NaN here
// whatever the product comes to; and a sum may pass F32's range: a wave with a
// sum that is not finite takes its tiles again on the F32 matrix core.
//
// A workgroup of WM x WN waves per BM x BN output tile. K advances BK columns
// a stage: while one is multiplied, the next one's F32 operands, loaded during
// the stage before, are split and stored to the other LDS buffer and the
// loads of the one after it go out; one barrier a stage. A row of each term's
// LDS plane is padded by 16 bytes, so that the 16-byte fragment reads of
// consecutive rows fall in distinct banks.
//
// Measured (us at 4096 rows, N x K; the F32 MFMA on 128 x 128 tiles, which
// all F32 products took, then on 64 x 64): 768 x 768 here 46 against 81 and
// 54; 2304 x 768 134 (242, 150); 768 x 3072 144 (262, 184); 384 x 1536 54
// (139, 73). A stage's vector work, LDS traffic (six reads and three writes
// of a term per element) and products take about a third of its time each
// and a single workgroup's do not overlap: the 128 x 128 tile runs eight
// waves, not four (768 x 3072: 144 against 190), and 64 x 64 tiles two
// workgroups a CU. BK 16, and the scheduler told to interleave the three,
// were no faster.
#include "kernels.h"
#include "launch.h"
#include "gemm_tile.h"
#include "gemm_more.h"

namespace rocm {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two values' three terms, a pair a word.
__device__ __forceinline__ void split2(float x, float y, uint32_t (&t)[3]) {
    t[0] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)x, (__bf16)y});
    const float x1 = x - __uint_as_float(t[0] << 16), y1 = y - __uint_as_float(t[0] & 0xffff0000u);
    t[1] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)x1, (__bf16)y1});
    const float x2 = x1 - __uint_as_float(t[1] << 16), y2 = y1 - __uint_as_float(t[1] & 0xffff0000u);
    t[2] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)x2, (__bf16)y2});
}

// A 32 x 32 tile on the F32 matrix core, a lane's row of each operand straight
// from memory: four columns of each eight, its half's (K a multiple of 4).
__device__ __forceinline__ floatx16 f32_tile(const float *a, const float *w, int K) {
    const int h = (threadIdx.x & 63) >> 5;
    floatx16 v{};
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8) {
        const int k = k0 + 4 * h;
        const f32x4 x = k < K ? *(const f32x4 *)(a + k) : f32x4{0, 0, 0, 0};
        const f32x4 y = k < K ? *(const f32x4 *)(w + k) : f32x4{0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 4; ++q) v = Mma<float>::run(x[q], y[q], v);
    }
    return v;
}

template <int BM, int BN, int WM, int WN, int BK, Epi KIND>
__global__ void __launch_bounds__(64 * WM * WN) gemm_f32_split_kernel(Span sp, int a_tok, int N, int K,
                                                                      const float *__restrict__ A, int lda,
                                                                      const float *__restrict__ W, EpiArgs e,
                                                                      int grid_n) {
    constexpr int RS = BK * 2 + 16;              // bytes of an LDS row
    constexpr int PLANE = (BM + BN) * RS, BUF = 3 * PLANE;
    constexpr int THREADS = 64 * WM * WN;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;   // MFMA tiles per wave
    constexpr int VROW = BK / 8;                 // 8-value groups in a tile row
    constexpr int LA = BM * VROW / THREADS, LB = BN * VROW / THREADS;
    static_assert(LA * THREADS == BM * VROW && LB * THREADS == BN * VROW, "tile loads split evenly over the threads");
    extern __shared__ __attribute__((aligned(16))) char lds[];   // [2][3][BM + BN] rows

    const Live lv = live_of(sp);
    const int M = lv.tokens;
    // XCD-aware renumbering over the span's own tiles; blocks past them leave.
    const int live = (M + BM - 1) / BM * grid_n;
    if ((int)blockIdx.x >= live) return;
    A += (size_t)lv.tok0 * a_tok;
    place_epilogue<KIND, float>(e, lv);
    const int per = live / 8;
    int b = blockIdx.x;
    if (b < per * 8) b = (b % 8) * per + b / 8;
    const int m0 = b / grid_n * BM, n0 = b % grid_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;

    f32x4 ra[LA][2], rb[LB][2];
    auto load1 = [&](f32x4 (&r)[2], const float *row, int k) {
#pragma unroll
        for (int q = 0; q < 2; ++q) r[q] = k + 4 * q < K ? *(const f32x4 *)(row + k + 4 * q) : f32x4{0, 0, 0, 0};
    };
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int v = tid + THREADS * i;
            load1(ra[i], A + (size_t)min(m0 + v / VROW, M - 1) * lda, k0 + v % VROW * 8);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int v = tid + THREADS * i;
            load1(rb[i], W + (size_t)min(n0 + v / VROW, N - 1) * K, k0 + v % VROW * 8);
        }
    };
    auto store1 = [&](char *at, const f32x4 (&r)[2]) {
        uint32_t t[4][3];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            split2(r[q][0], r[q][1], t[2 * q]);
            split2(r[q][2], r[q][3], t[2 * q + 1]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) *(u32x4 *)(at + p * PLANE) = u32x4{t[0][p], t[1][p], t[2][p], t[3][p]};
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int v = tid + THREADS * i;
            store1(lds + buf * BUF + v / VROW * RS + v % VROW * 16, ra[i]);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int v = tid + THREADS * i;
            store1(lds + buf * BUF + (BM + v / VROW) * RS + v % VROW * 16, rb[i]);
        }
    };

    // The sums of the x0 w0 products, and of the five small terms' products.
    floatx16 acc[TM][TN], low[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = floatx16{};

    const int nk = (K + BK - 1) / BK;
    load(0);
    store(0);
    if (nk > 1) load(BK);
    __syncthreads();
    const int off_a = (wm * (BM / WM) + (lane & 31)) * RS + (lane >> 5) * 16;
    const int off_b = (BM + wn * (BN / WN) + (lane & 31)) * RS + (lane >> 5) * 16;
    for (int kt = 0; kt < nk; ++kt) {
        const char *base = lds + (kt & 1) * BUF;
        if (kt + 1 < nk) store((kt + 1) & 1);
        if (kt + 2 < nk) load((kt + 2) * BK);
#pragma unroll
        for (int s = 0; s < BK / 16; ++s) {
            bf16x8 fa[3][TM], fb[3][TN];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[p][i] = *(const bf16x8 *)(base + p * PLANE + off_a + i * 32 * RS + s * 32);
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[p][j] = *(const bf16x8 *)(base + p * PLANE + off_b + j * 32 * RS + s * 32);
            }
            constexpr int PA[5] = {2, 1, 0, 1, 0}, PB[5] = {0, 1, 2, 0, 1};
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    acc[i][j] = Mma<__bf16>::run(fa[0][i], fb[0][j], acc[i][j]);
#pragma unroll
                    for (int t = 0; t < 5; ++t) low[i][j] = Mma<__bf16>::run(fa[PA[t]][i], fb[PB[t]][j], low[i][j]);
                }
        }
        __syncthreads();
    }
    float z = 0.0f;   // 0 as long as every sum is finite
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] += low[i][j];
#pragma unroll
            for (int r = 0; r < 16; ++r) z = fmaf(acc[i][j][r], 0.0f, z);
        }
    if (__ballot(z != 0.0f) != 0) {   // uniform
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = f32_tile(A + (size_t)min(m0 + wm * (BM / WM) + i * 32 + (lane & 31), M - 1) * lda,
                                     W + (size_t)min(n0 + wn * (BN / WN) + j * 32 + (lane & 31), N - 1) * K, K);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            epilogue_tile<float, KIND>(e, M, N, m0 + wm * (BM / WM) + i * 32, n0 + wn * (BN / WN) + j * 32 + (lane & 31),
                                       acc[i][j]);
}

template <int BM, int BN, int WM, int WN, int BK>
static hipError_t launch(hipStream_t s, const GemmRows &gr, int M, int N, int K, const void *A, int lda, const void *W,
                         const EpiArgs &e) {
    const int gn = (N + BN - 1) / BN, gm = (M + BM - 1) / BM;
    constexpr int bytes = 2 * 3 * (BM + BN) * (BK * 2 + 16);
#define SPLIT_CASE(E)                                                                                               \
    case Epi::E:                                                                                                    \
        enqueue((gemm_f32_split_kernel<BM, BN, WM, WN, BK, Epi::E>), dim3(gn * gm), dim3(64 * WM * WN), bytes, s,   \
                gr.sp, gr.a_tok, N, K, (const float *)A, lda, (const float *)W, e, gn);                             \
        return hipGetLastError();
    switch (e.kind) {
        SPLIT_CASE(Plain)
        SPLIT_CASE(Qkv)
        SPLIT_CASE(Gelu)
        SPLIT_CASE(Residual)
        SPLIT_CASE(QkvRope)
        SPLIT_CASE(Gated)
        SPLIT_CASE(Bias)
    }
#undef SPLIT_CASE
    return hipErrorInvalidValue;
}

hipError_t gemm_f32_split(hipStream_t s, bool wide, const GemmRows &gr, int M, int N, int K, const void *A, int lda,
                          const void *W, const EpiArgs &e) {
    return wide ? launch<128, 128, 2, 4, 32>(s, gr, M, N, K, A, lda, W, e)
                : launch<64, 64, 2, 2, 32>(s, gr, M, N, K, A, lda, W, e);
}

}  // namespace rocm
