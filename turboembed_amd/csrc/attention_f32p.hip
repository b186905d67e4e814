// Softmax attention on the matrix cores with F32 probabilities: the F32 tier's
// heads of 32 and 64, and F16 and BF16 heads of 32 (attention.hip's operands,
// masks and results; its matrix-core path rounds the probabilities to the
// operand type, this one does not).
//
// One wave per (32 queries, head, row), four to a workgroup, with no LDS and
// no barrier: heads this narrow keep a 32-key block of K and V^T in 16 to 64
// registers, loaded straight from memory while the block before is
// computed, and the waves of a (row, head) pair meet in the caches. Scores
// are computed transposed, S^T = K Q^T, so a lane holds one query (lane % 32)
// and 16 of the block's keys, the other 16 in the lane 32 away; the online
// softmax runs in F32 in base 2, on a score's distance from the maximum (the
// difference first, then the scale: the product less a rounded maximum is off
// by half its ulp, past exp2's range from scores of 1e9 on), and moves its
// maximum only when a score passes it by more than 2^8. The context is computed transposed too, O^T += V^T P^T, from
// P as the score registers hold it:
// - F32 operands: v_mfma_f32_32x32x2f32 for both products, register r of P
//   against the four-key groups of V^T that its keys lie in.
// - 16-bit operands: v_mfma_f32_32x32x16 for the scores (exact products, F32
//   sums), and P as two F16 or three BF16 terms, p = p0 + p1 (+ p2), whose
//   products with V^T are each exact and summed in F32. F16's probabilities
//   are kept 2^7 larger (at most 2^15), so that its second term resolves
//   2^-32 of a query's largest.
// A key that is not live (masked, outside the window, past the row) scores
// minus infinity and its V reads as 0, so nothing of it reaches a live query;
// a query with no live key gets a zero context. So does one whose largest
// score is infinite, and a score that is not a number weighs 0 (queries or
// keys past the operand type's range).
//
// Measured against the scalar kernel of attention.hip, which these heads took
// (a lane a query, its keys read from LDS one by one), us a launch: F16 heads
// of 32, 128 rows of 32-256 tokens in two parts side by side 35 against 187;
// F32 heads of 32, 32 rows of 16-128, 16 against 45; F32 heads of 64, 24 rows
// of 33-300, 94 to 101 against 316. Short rows wait for memory (each wave has
// eight blocks at most there), F32 heads of 64 for the F32 matrix cores and
// the 32-byte pieces in which their rows are read.
#include <type_traits>

#include "kernels.h"
#include "launch.h"
#include "devmath.h"
#include "gemm_tile.h"

namespace rocm {

// The sum of a lane's value and the lane 32 away's, and the larger of the two.
__device__ __forceinline__ float halves_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float halves_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// (By the value's bits, and behind the compiler's back: this source is built
// without NaNs.)
__device__ __forceinline__ bool is_nan(float v) {
    uint32_t u = __float_as_uint(v);
    asm("" : "+v"(u));
    return (u & 0x7fffffffu) > 0x7f800000u;
}

constexpr int F32P_WAVES = 4;

template <typename T, int D>
__global__ void __launch_bounds__(64 * F32P_WAVES) attention_f32p_kernel(const T *__restrict__ qkv, int tcap, int heads,
                                                                         Span sp, int nqb, Packing p,
                                                                         const int32_t *__restrict__ mask, int window,
                                                                         T *__restrict__ ctx) {
    constexpr bool F32 = std::is_same<T, float>::value;
    constexpr int QB = 32 * F32P_WAVES, NO = D / 32;
    constexpr int VEC = 16 / sizeof(T);
    constexpr int KV = F32 ? D / 2 / VEC : D / 16;   // 16-byte vectors of K (and Q) a lane holds
    constexpr int VV = F32 ? 4 : 2;                  // of V^T, per 32 columns of the head
    constexpr float BIAS = std::is_same<T, _Float16>::value ? 7.0f : 0.0f;
    constexpr float RESCALE = 8.0f;
    typedef typename Mma<T>::frag frag;
    typedef T vec __attribute__((ext_vector_type(VEC)));
    // (V^T's rows start at the row's packed token: at any element.)
    typedef T loose __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));

    // XCD-aware numbering, as attention.hip's: a pair's query blocks 8 apart.
    const int L = blockIdx.x;
    const int pair = (L / (8 * nqb)) * 8 + L % 8, qb = (L / 8) % nqb;
    const Live lv = live_of(sp);
    if (pair >= heads * lv.rows) return;
    const int r = lv.row0 + pair / heads, head = pair % heads;
    const int len = p.len[r], start = p.start[r];
    const int lane = threadIdx.x & 63, h = lane >> 5, ql = lane & 31;
    const int qw = qb * QB + 32 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (qw >= len) return;
    const T *Q = qkv + ((size_t)head * tcap + start) * D;
    const T *K = qkv + ((size_t)(heads + head) * tcap + start) * D;
    const T *Vt = qkv + ((size_t)2 * heads + head) * D * tcap + start;
    const int32_t *mk = mask + (size_t)r * lv.seq;
    int k_lo = 0, k_hi = len;
    if (window < INT32_MAX) {
        k_lo = max(0, qw - window) / 32 * 32;
        k_hi = min(len, qw + 32 + window);
    }

    // A lane's columns of K and Q: 16 bytes of each 32, its half's (with F32
    // operands a column a product step). Its key of K: the MFMA row itself, or,
    // so that P's registers hold runs of 8 keys, with bits 2 and 3 exchanged.
    constexpr int KSTEP = 2 * VEC;
    const int kcol = h * VEC;
    const int krow = F32 ? ql : (ql & ~12) | ((ql & 4) << 1) | ((ql & 8) >> 1);
    vec q[KV];
#pragma unroll
    for (int s = 0; s < KV; ++s) q[s] = *(const vec *)(Q + (size_t)min(qw + ql, len - 1) * D + kcol + s * KSTEP);

    struct Block {
        vec k[KV];
        vec v[NO][VV];
        int32_t live;
    };
    // The group of a lane's keys that vector g of V^T covers: 4 of each 8
    // (F32), or 8 of each 16. One wholly past the row reads the row's last.
    constexpr int VGROUP = F32 ? 8 : 16;
    auto load = [&](Block &b, int kb) {
        if (kb >= k_hi) return;   // uniform
        const T *kr = K + (size_t)min(kb + krow, len - 1) * D + kcol;
#pragma unroll
        for (int s = 0; s < KV; ++s) b.k[s] = *(const vec *)(kr + s * KSTEP);
#pragma unroll
        for (int g = 0; g < VV; ++g) {
            const int k0 = kb + VGROUP * g + VEC * h;
            const int at = k0 < len ? k0 : (len - 1) & ~(VEC - 1);
#pragma unroll
            for (int t = 0; t < NO; ++t) b.v[t][g] = *(const loose *)(Vt + (size_t)(32 * t + ql) * tcap + at);
        }
        b.live = mk[min(kb + ql, len - 1)];
    };

    floatx16 o[NO];
#pragma unroll
    for (int t = 0; t < NO; ++t) o[t] = floatx16{};
    float m_run = -INFINITY, lsum = 0.0f;
    const float scale = 1.4426950408889634f / sqrtf((float)D), rescale = RESCALE / scale;

    auto step = [&](Block &b, int kb) {
        if (kb >= k_hi) return;   // uniform
        floatx16 sc{};
#pragma unroll
        for (int s = 0; s < KV; ++s) {
            if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) sc = Mma<T>::run(b.k[s][e], q[s][e], sc);
            } else {
                sc = Mma<T>::run(b.k[s], q[s], sc);
            }
        }
        // This lane's keys in reach: the row's live ones, within the window.
        const uint32_t live = (uint32_t)__ballot(kb + ql < len && b.live != 0);
        const bool all = live == ~0u && (window == INT32_MAX || (kb >= qw + 31 - window && kb + 31 <= qw + window));
        if (!all) {
            uint32_t ok = live;
            if (window < INT32_MAX) {
                const int lo = qw + ql - window - kb, hi = qw + ql + window - kb;   // keys lo .. hi of the block
                ok &= hi < 0 || lo > 31 ? 0u
                                        : (hi >= 31 ? ~0u : (2u << hi) - 1) & (lo <= 0 ? ~0u : ~((1u << lo) - 1));
            }
            const uint32_t word = ok >> (F32 ? 4 * h : 8 * h), vword = live >> (F32 ? 4 * h : 8 * h);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int j = F32 ? 8 * (i >> 2) + (i & 3) : 16 * (i >> 3) + (i & 7);
                sc[i] = (word >> j) & 1u ? sc[i] : -INFINITY;
            }
            // (The wave's queries share V: a live key outside one's window
            // weighs 0 there, and reads as 0 only where it is live to none.)
#pragma unroll
            for (int g = 0; g < VV; ++g)
#pragma unroll
                for (int e = 0; e < VEC; ++e)
#pragma unroll
                    for (int t = 0; t < NO; ++t)
                        b.v[t][g][e] = (vword >> (VGROUP * g + e)) & 1u ? b.v[t][g][e] : (T)0.0f;
        }
        float mx = sc[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sc[i]);
        mx = halves_max(mx);
        if (__ballot(mx > m_run + rescale) != 0) {
            const float m_new = fmaxf(m_run, mx);
            // (Equal: both minus infinity, or infinite by a score past F32.)
            const float f = __builtin_amdgcn_exp2f(m_run == m_new ? 0.0f : (m_run - m_new) * scale);
#pragma unroll
            for (int t = 0; t < NO; ++t) o[t] *= f;
            lsum *= f;
            m_run = m_new;
        }
        const float m = m_run == -INFINITY ? 0.0f : m_run;
        float pr[16], bsum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            pr[i] = __builtin_amdgcn_exp2f(fmaf(sc[i] - m, scale, BIAS));
            bsum += pr[i];
        }
        if (__ballot(is_nan(bsum)) != 0) {   // uniform
            bsum = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                pr[i] = is_nan(pr[i]) ? 0.0f : pr[i];
                bsum += pr[i];
            }
        }
        lsum += bsum;
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
                for (int t = 0; t < NO; ++t) o[t] = Mma<T>::run(b.v[t][i >> 2][i & 3], pr[i], o[t]);
        } else {
            constexpr int TERMS = std::is_same<T, _Float16>::value ? 2 : 3;
#pragma unroll
            for (int n = 0; n < TERMS; ++n)
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    frag pf;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const T x = from_f32<T>(pr[8 * g + e]);
                        pr[8 * g + e] -= (float)x;
                        pf[e] = x;
                    }
#pragma unroll
                    for (int t = 0; t < NO; ++t) o[t] = Mma<T>::run(__builtin_bit_cast(frag, b.v[t][g]), pf, o[t]);
                }
        }
    };
    Block b0, b1;
    load(b0, k_lo);
    for (int kb = k_lo; kb < k_hi; kb += 64) {
        load(b1, kb + 32);
        step(b0, kb);
        load(b0, kb + 64);
        step(b1, kb + 32);
    }

    const float l = halves_sum(lsum);
    if (qw + ql >= len) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    T *out = ctx + (size_t)(start + qw + ql) * heads * D + head * D + 4 * h;
    typedef T vec4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int t = 0; t < NO; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(vec4 *)(out + 32 * t + 8 * g) =
                vec4{from_f32<T>(o[t][4 * g] * inv), from_f32<T>(o[t][4 * g + 1] * inv),
                     from_f32<T>(o[t][4 * g + 2] * inv), from_f32<T>(o[t][4 * g + 3] * inv)};
}

bool attention_f32p_takes(Dt dt, int d) { return d == 32 ? dt != Dt::I8 : d == 64 && dt == Dt::F32; }

hipError_t attention_f32p(hipStream_t s, Dt dt, const void *qkv, int tcap, int heads, int d, const Packing &p,
                          const int32_t *mask, const Span &sp, int max_rows, int max_len, int window, void *ctx) {
    if (!attention_f32p_takes(dt, d)) return hipErrorInvalidValue;
    // (A window over the rows' length is none, and the kernel's sums of a key
    // and a window stay in range.)
    if (window >= max_len) window = INT32_MAX;
    // A 1-D grid of groups of 8 (row, head) pairs times nqb query blocks.
    const int nqb = (max_len + 32 * F32P_WAVES - 1) / (32 * F32P_WAVES), pairs = heads * max_rows;
    const dim3 grid((pairs + 7) / 8 * 8 * nqb), block(64 * F32P_WAVES);
#define F32P(T, D)                                                                                               \
    enqueue((attention_f32p_kernel<T, D>), grid, block, 0, s, (const T *)qkv, tcap, heads, sp, nqb, p, mask, window, \
            (T *)ctx)
    if (dt == Dt::F16) F32P(_Float16, 32);
    else if (dt == Dt::BF16) F32P(__bf16, 32);
    else if (d == 32) F32P(float, 32);
    else F32P(float, 64);
#undef F32P
    return hipGetLastError();
}

}  // namespace rocm
