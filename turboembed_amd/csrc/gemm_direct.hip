// Products of few rows (a query, a handful of short texts), where the tiled
// kernels leave the chip idle: C = A W^T as gemm.hip has it, on small output
// tiles whose K is shared among the workgroup's waves.
//
// A launch of M <= 256 rows has N / 128 tiles of 128 x 128 a row of tiles (6
// at N = 768), each walking all of K one stage after another behind a
// barrier: time is K / 64 round trips, whatever M. Here a workgroup of KW
// waves takes a 32 x 32 tile and wave w the 64-byte blocks of k w, w + KW,
// ...: operands go straight from memory into the MFMA's registers
// (no LDS and no barrier in the loop, the next U blocks' loads in flight
// while U blocks are multiplied), then the waves' F32 sums meet in LDS and
// each wave adds, in wave order, and stores its share of the tile's registers.
#include "kernels.h"
#include "launch.h"
#include "gemm_tile.h"
#include "gemm_more.h"

namespace rocm {

constexpr int DIRECT_KW = 8;   // waves, each with every eighth 64-byte block of k

template <typename T, Epi KIND>
__global__ void __launch_bounds__(64 * DIRECT_KW) gemm_direct_kernel(Span sp, int a_tok, int N, int K,
                                                              const T *__restrict__ A, int lda,
                                                              const T *__restrict__ W, EpiArgs e, int grid_n, int ks,
                                                              size_t stride) {
    typedef typename Mma<T>::frag frag;
    typedef uint32_t vec4 __attribute__((ext_vector_type(4)));
    constexpr int VEC = 16 / sizeof(T), BLK = 4 * VEC;   // elements in 16 bytes; k columns of a 64-byte block
    constexpr int EPM = Mma<T>::EPM, KW = DIRECT_KW;
    constexpr int U = 3;          // of a wave's blocks, those in flight beside the ones multiplied
    constexpr int NR = 16 / KW;   // of a lane's 16 accumulators, those one wave stores
    __shared__ float sums[KW][16][64];

    const Live lv = live_of(sp);
    const int M = lv.tokens;
    const int b = blockIdx.x;
    if (b >= (M + 31) / 32 * grid_n) return;
    A += (size_t)lv.tok0 * a_tok;
    // Slice y of K: ks columns (whole blocks), its sums at its own stride.
    // (A span whose rows pass a slice's would write into the next: such a
    // launch leaves, and the session never makes one.)
    const int k0 = blockIdx.y * ks, ke = min(K, k0 + ks);
    if constexpr (KIND == Epi::Plain) {
        if (gridDim.y > 1 && (size_t)(lv.tok0 + M) * N > stride) return;
        e.out = (float *)e.out + blockIdx.y * stride;
    }
    place_epilogue<KIND, T>(e, lv);
    const int m0 = b / grid_n * 32, n0 = b % grid_n * 32;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // This lane's rows, those past the operands' last clamped to it, at the
    // half of a block it reads (two 16-byte vectors).
    const T *pa = A + (size_t)min(m0 + (lane & 31), M - 1) * lda + k0 + 2 * VEC * h;
    const T *pb = W + (size_t)min(n0 + (lane & 31), N - 1) * K + k0 + 2 * VEC * h;

    floatx16 acc{};
    struct Set {
        vec4 a[U][2], b[U][2];
    };
    // The blocks of k, and (when K ends inside one) the vectors of the last
    // that are whole: K is a multiple of VEC, and a vector past it reads as 0.
    const int kn = ke - k0, nb = (kn + BLK - 1) / BLK;
    auto load = [&](Set &s, int b0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int blk = b0 + u * KW;
            const bool in = blk < nb;   // uniform
            const int k = blk * BLK;
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const bool ok = in && k + (2 * h + v) * VEC < kn;
                s.a[u][v] = ok ? *(const vec4 *)(pa + k + v * VEC) : vec4{0, 0, 0, 0};
                s.b[u][v] = ok ? *(const vec4 *)(pb + k + v * VEC) : vec4{0, 0, 0, 0};
            }
        }
    };
    auto multiply = [&](const Set &s, int b0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (b0 + u * KW >= nb) break;   // uniform
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int q = 0; q < VEC / EPM; ++q) {
                    frag fa, fb;
                    if constexpr (EPM == 1) {
                        fa = __uint_as_float(s.a[u][v][q]);
                        fb = __uint_as_float(s.b[u][v][q]);
                    } else {
                        fa = __builtin_bit_cast(frag, s.a[u][v]);
                        fb = __builtin_bit_cast(frag, s.b[u][v]);
                    }
                    acc = Mma<T>::run(fa, fb, acc);
                }
        }
    };
    Set s0, s1;
    load(s0, wave);
    for (int b0 = wave; b0 < nb; b0 += 2 * U * KW) {
        load(s1, b0 + U * KW);
        multiply(s0, b0);
        load(s0, b0 + 2 * U * KW);
        multiply(s1, b0 + U * KW);
    }

#pragma unroll
    for (int r = 0; r < 16; ++r) sums[wave][r][lane] = acc[r];
    __syncthreads();
    const int r0 = wave * NR;
    float v[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        v[i] = sums[0][r0 + i][lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) v[i] += sums[w][r0 + i][lane];
    }
    epilogue_tile<T, KIND, NR>(e, M, N, m0, n0 + (lane & 31), v, r0);
}

template <typename T>
static hipError_t launch(hipStream_t s, const GemmRows &gr, int M, int N, int K, const void *A, int lda, const void *W,
                         const EpiArgs &e) {
    const int gn = (N + 31) / 32, gm = (M + 31) / 32;
#define DIRECT_CASE(E)                                                                                              \
    case Epi::E:                                                                                                    \
        enqueue((gemm_direct_kernel<T, Epi::E>), dim3(gn * gm), dim3(64 * DIRECT_KW), 0, s, gr.sp,       \
                gr.a_tok, N, K, (const T *)A, lda, (const T *)W, e, gn, K, (size_t)0);                              \
        return hipGetLastError();
    switch (e.kind) {
        DIRECT_CASE(Plain)
        DIRECT_CASE(Qkv)
        DIRECT_CASE(Gelu)
        DIRECT_CASE(Residual)
        DIRECT_CASE(QkvRope)
        DIRECT_CASE(Gated)
        DIRECT_CASE(Bias)
    }
#undef DIRECT_CASE
    return hipErrorInvalidValue;
}

hipError_t gemm_direct(hipStream_t s, Dt dt, const GemmRows &gr, int M, int N, int K, const void *A, int lda,
                       const void *W, const EpiArgs &e) {
    switch (dt) {
    case Dt::F16: return launch<_Float16>(s, gr, M, N, K, A, lda, W, e);
    case Dt::BF16: return launch<__bf16>(s, gr, M, N, K, A, lda, W, e);
    case Dt::F32: return launch<float>(s, gr, M, N, K, A, lda, W, e);
    default: return hipErrorInvalidValue;
    }
}

// K is cut where each of a slice's waves keeps a block of 64 bytes or more in
// flight: four slices from 48 blocks on (K = 1536 in 16 bits, 768 in F32).
int gemm_slices_of(Dt dt, int M, int N, int K, const EpiArgs &e) {
    if (dt == Dt::I8 || e.kind != Epi::Bias || !e.ws || N % 8 != 0 || !gemm_is_direct(dt, M, N, K, e)) return 1;
    const int blocks = K * (int)dt_bytes(dt) / 64;
    const int slices = blocks >= 48 ? 4 : blocks >= 24 ? 2 : 1;
    return (size_t)slices * M * N <= e.ws_floats ? slices : 1;
}

template <typename T>
static void launch_slices(hipStream_t s, const GemmRows &gr, int M, int N, int K, const void *A, int lda, const void *W,
                          float *ws, int slices, size_t stride) {
    constexpr int BLK = 64 / (int)sizeof(T);
    const int gn = (N + 31) / 32, gm = (M + 31) / 32, ks = ((K + slices - 1) / slices + BLK - 1) / BLK * BLK;
    EpiArgs e;
    e.kind = Epi::Plain;
    e.out = ws;
    e.ldo = N;
    enqueue((gemm_direct_kernel<T, Epi::Plain>), dim3(gn * gm, slices), dim3(64 * DIRECT_KW), 0, s, gr.sp, gr.a_tok, N,
            K, (const T *)A, lda, (const T *)W, e, gn, ks, stride);
}

hipError_t gemm_slices(hipStream_t s, Dt dt, const Span &sp, int M, int N, int K, const void *A, int lda, const void *W,
                       float *ws, int slices, size_t stride) {
    const int vec = 16 / (int)dt_bytes(dt);
    // (Every slice has columns: ceil division leaves the last one some.)
    if (dt == Dt::I8 || !ws || slices < 1 || K % vec != 0 || lda % vec != 0 || stride < (size_t)M * N ||
        (slices - 1) * (((K + slices - 1) / slices + 4 * vec - 1) / (4 * vec) * (4 * vec)) >= K)
        return hipErrorInvalidValue;
    if (M <= 0) return hipSuccess;
    const GemmRows gr{sp, lda};
    switch (dt) {
    case Dt::F16: launch_slices<_Float16>(s, gr, M, N, K, A, lda, W, ws, slices, stride); break;
    case Dt::BF16: launch_slices<__bf16>(s, gr, M, N, K, A, lda, W, ws, slices, stride); break;
    default: launch_slices<float>(s, gr, M, N, K, A, lda, W, ws, slices, stride);
    }
    return hipGetLastError();
}

}  // namespace rocm
