// The sequence classification head over a rerank run's CLS states, beside
// them on the device: the pooler's dense rows and the classifier's one row
// (reference core/src/session/rerank.rs:166-191) with F64 products and sums,
// each rounded to F32 once, as the host head (rerank.cpp) computes them. A
// product of two F32 values is exact in F64, and a pooler's sum runs from its
// bias in column order, so it has the host's bits; the classifier's is summed
// by the lanes of a wave, F64's last bits off the host's.
//
// The pooler is hidden^2 products a row, which one host thread's chain of
// F64 adds took 38 ms for at 128 rows of 768, 15 times the encoder's run;
// here it takes 48 us, on 16 x 16 tiles of (row, output), a thread each, both
// operands through LDS 64 columns at a time, bound by the F64 chain's latency
// at one or two workgroups a CU; the call is 3400 us.
#include "kernels.h"
#include "launch.h"
#include "devmath.h"

namespace rocm {

constexpr int HEAD_TILE = 16, HEAD_COLS = 64;

__global__ void __launch_bounds__(256) rerank_pooler_kernel(const float *__restrict__ x, int rows, int hidden,
                                                            const float *__restrict__ w, const float *__restrict__ b,
                                                            float *__restrict__ pooled) {
    // (Rows padded by one value: a column of either tile spans the banks.)
    __shared__ float xs[HEAD_TILE][HEAD_COLS + 1], ws[HEAD_TILE][HEAD_COLS + 1];
    const int o0 = blockIdx.x * HEAD_TILE, r0 = blockIdx.y * HEAD_TILE;
    const int o = threadIdx.x % HEAD_TILE, r = threadIdx.x / HEAD_TILE;
    double sum = b && o0 + o < hidden ? (double)b[o0 + o] : 0.0;
    for (int k0 = 0; k0 < hidden; k0 += HEAD_COLS) {
        __syncthreads();
        for (int i = threadIdx.x; i < HEAD_TILE * HEAD_COLS; i += 256) {
            const int t = i / HEAD_COLS, k = k0 + i % HEAD_COLS;
            xs[t][i % HEAD_COLS] = r0 + t < rows && k < hidden ? x[(size_t)(r0 + t) * hidden + k] : 0.0f;
            ws[t][i % HEAD_COLS] = o0 + t < hidden && k < hidden ? w[(size_t)(o0 + t) * hidden + k] : 0.0f;
        }
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < HEAD_COLS; ++k) sum = fma((double)ws[o][k], (double)xs[r][k], sum);
    }
    if (r0 + r < rows && o0 + o < hidden)
        pooled[(size_t)(r0 + r) * hidden + o0 + o] = (float)tanh(sum);
}

// A wave a row: its logit, and whether its state was finite.
__global__ void __launch_bounds__(64) rerank_logit_kernel(const float *__restrict__ x, const float *__restrict__ in,
                                                          int hidden, const float *__restrict__ w, float bias,
                                                          float *__restrict__ logit, int32_t *__restrict__ finite) {
    const size_t row = (size_t)blockIdx.x * hidden;
    double sum = 0.0;
    bool bad = false;
    for (int k = threadIdx.x; k < hidden; k += 64) {
        sum = fma((double)w[k], (double)in[row + k], sum);
        // (Not finite: every exponent bit set.)
        bad = bad || (__float_as_uint(x[row + k]) & 0x7f800000u) == 0x7f800000u;
    }
    sum = wave_sum(sum) + (double)bias;
    const bool any = __ballot(bad) != 0;
    if (threadIdx.x == 0) {
        logit[blockIdx.x] = (float)sum;
        finite[blockIdx.x] = any ? 0 : 1;
    }
}

hipError_t rerank_head(hipStream_t s, const float *x, int rows, int hidden, const float *pooler_w,
                       const float *pooler_b, const float *cls_w, float cls_b, float *pooled, float *logit,
                       int32_t *finite) {
    if (rows <= 0) return hipSuccess;
    const float *in = x;
    if (pooler_w) {
        enqueue(rerank_pooler_kernel, dim3((hidden + HEAD_TILE - 1) / HEAD_TILE, (rows + HEAD_TILE - 1) / HEAD_TILE),
                dim3(256), 0, s, x, rows, hidden, pooler_w, pooler_b, pooled);
        in = pooled;
    }
    enqueue(rerank_logit_kernel, dim3(rows), dim3(64), 0, s, x, in, hidden, cls_w, cls_b, logit, finite);
    return hipGetLastError();
}

}  // namespace rocm
