// The second kernel of the products whose k is split across groups: adds the splits' raw
// sums in split order (deterministic), then the epilogue. HBM-bound in name only: the sums
// are a few MB that the last-level cache holds, so what counts is how many loads a thread
// has in flight: eight splits at a time, four outputs a thread where the rows allow it.
#include "after.h"

namespace ts {

namespace {

// PAIR: two sums an output (gate and up, or the high and the low parts of f32 weights).
template <bool PAIR, int V>
__global__ __launch_bounds__(256) void split_finish_kernel(SplitSum p) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const size_t mn = (size_t)p.m * p.n, i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= mn) return;
    constexpr uint32_t kB = 8;
    const size_t stride = (PAIR ? 2 : 1) * mn;
    vec g = (vec)(0.0f), u = (vec)(0.0f);
    for (uint32_t s0 = 0; s0 < p.splits; s0 += kB) {
        vec tg[kB], tu[kB];
#pragma unroll
        for (uint32_t j = 0; j < kB; j++) {
            const uint32_t s = min(s0 + j, p.splits - 1);  // clamped: read but not added
            tg[j] = *(const vec *)(p.part + s * stride + i);
            if (PAIR) tu[j] = *(const vec *)(p.part + s * stride + mn + i);
        }
#pragma unroll
        for (uint32_t j = 0; j < kB; j++)
            if (s0 + j < p.splits) {
                g += tg[j];
                if (PAIR) u += tu[j];
            }
    }
    float head = p.head ? *p.head : 1.0f;
    const uint32_t n = (uint32_t)(i % p.n);  // V divides n: one row
    if (p.sumsq) {
        const uint32_t m = (uint32_t)(i / p.n);
        float ss = 0.0f;
        for (uint32_t s = 0; s < p.splits; s++) ss += p.sumsq[s * p.m + m];
        head = 1.0f / sqrtf(ss / (float)p.k + p.eps);
    }
#pragma unroll
    for (int e = 0; e < V; e++) {
        float a = g[e] * head, b = u[e] * head;
        if (p.w_scale) {
            a *= bf16_float(p.w_scale[n + e]);
            if (PAIR) b *= bf16_float(p.w_scale[p.n + n + e]);
        }
        float v = !PAIR ? a : p.pair_sum ? a + b : a / (1.0f + expf(-a)) * b;
        if (p.stages & TS_AFTER_ADD) v += p.a0[i + e];
        if (p.after.count) v = after_apply(p.after, v, i + e);
        if (p.out_bf16) ((uint16_t *)p.out)[i + e] = bf16_bits(v);
        else ((float *)p.out)[i + e] = v;
    }
}

}  // namespace

int split_finish(const SplitSum &p, void *stream) {
    const bool pair = (p.stages & TS_AFTER_SILU_MUL) || p.pair_sum;
    const int v = p.n % 4 == 0 ? 4 : 1;
    const size_t threads = (size_t)p.m * p.n / v;
    auto k = pair ? (v == 4 ? split_finish_kernel<true, 4> : split_finish_kernel<true, 1>)
                  : (v == 4 ? split_finish_kernel<false, 4> : split_finish_kernel<false, 1>);
    hipLaunchKernelGGL(k, dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream, p);
    TS_CHECK_LAUNCH("split sums launch");
    return TS_OK;
}

}  // namespace ts
