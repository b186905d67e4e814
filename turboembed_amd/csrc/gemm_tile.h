// What the GEMM kernels share: the MFMA of each operand type, a launch's rows,
// and the epilogue of one 32 x 32 tile straight from its registers.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "devmath.h"
#include "kernels.h"

namespace rocm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mma;

typedef int int32x4 __attribute__((ext_vector_type(4)));
typedef int int32x16 __attribute__((ext_vector_type(16)));

template <> struct Mma<_Float16> {
    static constexpr int EPM = 8;   // elements a lane feeds one MFMA
    typedef half8 frag;
    typedef floatx16 acc;
    static __device__ __forceinline__ floatx16 run(frag a, frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

template <> struct Mma<__bf16> {
    static constexpr int EPM = 8;
    typedef bf16x8 frag;
    typedef floatx16 acc;
    static __device__ __forceinline__ floatx16 run(frag a, frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

template <> struct Mma<int8_t> {
    static constexpr int EPM = 16;
    typedef int32x4 frag;
    typedef int32x16 acc;
    static __device__ __forceinline__ int32x16 run(frag a, frag b, int32x16 c) {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
};

template <> struct Mma<float> {
    static constexpr int EPM = 1;
    typedef float frag;
    typedef floatx16 acc;
    static __device__ __forceinline__ floatx16 run(frag a, frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
};

// A gated unit's product act(gate) * up as stored: at an F16 output it
// saturates at F16's largest finite magnitude instead of rounding to
// infinity (a NaN stays NaN), as the reference's CUDA backend stores it
// (core/cuda/rotary.cuh:31-45); BF16 and F32 outputs hold it as it is.
template <typename T> __device__ __forceinline__ float gated_product(float g, float up) {
    const float v = __fmul_rn(g, up);
    if constexpr (std::is_same<T, _Float16>::value) return v > 65504.0f ? 65504.0f : v < -65504.0f ? -65504.0f : v;
    return v;
}

// The rows a GEMM launch multiplies: its span, and how far apart A's token
// rows are for the span's first token (the run's operand rows may be wider
// than the product's K).
struct GemmRows {
    Span sp;
    int a_tok;
};

// The span's first token moves the epilogue's row-major output (and the int8
// activation scales) down to it; the Q, K and V scatter (and the rotary
// epilogue's positions) take it as the token of row 0.
template <Epi KIND, typename OT>
__device__ __forceinline__ void place_epilogue(EpiArgs &e, const Live &lv) {
    e.tok0 = lv.tok0;
    if (e.a_scale) e.a_scale += lv.tok0;
    const size_t rows = (size_t)lv.tok0 * e.ldo;
    if constexpr (KIND == Epi::Plain) e.out = (float *)e.out + rows;
    else if constexpr (KIND == Epi::Bias) e.out = e.out_f32 ? (void *)((float *)e.out + rows) : (void *)((OT *)e.out + rows);
    else if constexpr (KIND == Epi::Gelu || KIND == Epi::Gated) e.out = (OT *)e.out + rows;
    else if constexpr (KIND == Epi::Residual) e.x += rows;
}

// The epilogue of one 32 x 32 MFMA tile, for this lane's column n and its 16
// rows m0 + 8 (r / 4) + 4 (lane / 32) + r % 4, v = acc + bias: all of them, or
// the NR of registers r0 .. r0 + NR - 1 (acc[0] is register r0's). The kind is
// a template argument, so each kernel carries one small epilogue, and what
// depends on the column alone is worked out once per tile.
template <typename T, Epi KIND, int NR = 16, typename ACC>
__device__ __forceinline__ void epilogue_tile(const EpiArgs &e, int M, int N, int mt, int n, const ACC &acc,
                                              int r0 = 0) {
    const int lane = threadIdx.x & 63;
    const int mb = mt + (lane >> 5) * 4;   // row of register r: mb + 8 (r / 4) + r % 4
    const bool col_ok = n < N;
    const float bias = (e.bias && col_ok) ? e.bias[n] : 0.0f;
    if constexpr (KIND == Epi::Plain || KIND == Epi::Gelu || KIND == Epi::Residual || KIND == Epi::Bias) {
        if (!col_ok) return;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int r = r0 + i, m = mb + (r >> 2) * 8 + (r & 3);
            if (m >= M) continue;
            const float v = acc[i] + bias;
            const size_t at = (size_t)m * e.ldo + n;
            if constexpr (KIND == Epi::Plain) ((float *)e.out)[at] = v;
            else if constexpr (KIND == Epi::Bias) {
                if (e.out_f32) ((float *)e.out)[at] = v;
                else if (sizeof(T) == 2 && e.out_bf16) ((__bf16 *)e.out)[at] = from_f32<__bf16>(v);
                else ((T *)e.out)[at] = from_f32<T>(v);
            }
            else if constexpr (KIND == Epi::Gelu)
                ((T *)e.out)[at] = from_f32<T>(sizeof(T) == 2 ? dev_gelu_fast(v) : dev_gelu(v));
            else e.x[at] = e.x[at] + v;
        }
    } else if constexpr (KIND == Epi::Qkv || KIND == Epi::QkvRope) {
        const int which = n / e.hidden, rem = n - which * e.hidden;
        const int head = rem / e.d, c = rem - head * e.d;
        T *out = (T *)e.out + (size_t)which * e.heads * e.tcap * e.d;
        const int half = e.d >> 1, pr = c >> 1;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int r = r0 + i, m = mb + (r >> 2) * 8 + (r & 3);
            float v = acc[i] + bias;
            if constexpr (KIND == Epi::QkvRope) {
                // Columns come pair-adjacent: the partner of n is n ^ 1, in
                // the neighbouring lane (column n sits in lane n % 32).
                const float w = __shfl_xor(v, 1, 64);
                if (which < 2 && col_ok && m < M) {
                    // Rounded products, then their sum or difference, in
                    // every instantiation (no fused multiply-add).
#pragma clang fp contract(off)
                    const int pos = e.pos[e.tok0 + m];
                    const float cs = e.cos[(size_t)pos * half + pr], sn = e.sin[(size_t)pos * half + pr];
                    // (x1, x2) -> (x1 cos - x2 sin, x2 cos + x1 sin)
                    v = (c & 1) ? v * cs + w * sn : v * cs - w * sn;
                }
            }
            if (!col_ok || m >= M) continue;
            // Q and K token-major per head; V transposed per head.
            const size_t t = (size_t)e.tok0 + m;
            const size_t at = which < 2 ? ((size_t)head * e.tcap + t) * e.d + c : ((size_t)head * e.d + c) * e.tcap + t;
            out[at] = from_f32<T>(v);
        }
    } else {   // Gated: out[m, n / 2] = act(gate) * up, gate and up in neighbouring columns
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int r = r0 + i, m = mb + (r >> 2) * 8 + (r & 3);
            const float v = acc[i] + bias;
            const float up = __shfl_xor(v, 1, 64);
            if (!col_ok || m >= M || (n & 1)) continue;
            const float g = e.silu ? dev_silu(v) : sizeof(T) == 2 ? dev_gelu_fast(v) : dev_gelu(v);
            ((T *)e.out)[(size_t)m * e.ldo + (n >> 1)] = from_f32<T>(gated_product<T>(g, up));
        }
    }
}

}  // namespace rocm
