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
                                                              const T *__restrict__ W, EpiArgs e, int grid_n) {
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
    place_epilogue<KIND, T>(e, lv);
    const int m0 = b / grid_n * 32, n0 = b % grid_n * 32;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // This lane's rows, those past the operands' last clamped to it, at the
    // half of a block it reads (two 16-byte vectors).
    const T *pa = A + (size_t)min(m0 + (lane & 31), M - 1) * lda + 2 * VEC * h;
    const T *pb = W + (size_t)min(n0 + (lane & 31), N - 1) * K + 2 * VEC * h;

    floatx16 acc{};
    struct Set {
        vec4 a[U][2], b[U][2];
    };
    // The blocks of k, and (when K ends inside one) the vectors of the last
    // that are whole: K is a multiple of VEC, and a vector past it reads as 0.
    const int nb = (K + BLK - 1) / BLK;
    auto load = [&](Set &s, int b0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int blk = b0 + u * KW;
            const bool in = blk < nb;   // uniform
            const int k = blk * BLK;
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const bool ok = in && k + (2 * h + v) * VEC < K;
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
                gr.a_tok, N, K, (const T *)A, lda, (const T *)W, e, gn);                                            \
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

}  // namespace rocm
