// lm_latent_parts.h — what the kernels of latent attention share (lm_mix.hip, lm_latent_step.hip): rotary pairs, cache rows, the factors of a
// head's result.
#pragma once
#include "lm_kernels.h"

namespace zg {
namespace lm {

namespace {

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }

// an output value, as it is and / or rounded to bf16 for the matrix product that reads it next
__device__ __forceinline__ void put_row(float* out, bf16_t* out16, size_t at, float v) {
    if (out) out[at] = v;
    if (out16) out16[at] = (bf16_t)cvt_pk_bf16(v, v);
}

__device__ __forceinline__ size_t cache_row(const int* page_table, int max_pages, int page_tokens, int slot, int pos) {
    return (size_t)page_table[(size_t)slot * max_pages + pos / page_tokens] * page_tokens + pos % page_tokens;
}

// pair i of `src` (channels (2i, 2i + 1), or (i, i + dims / 2)) at position pos, rotated by pos * freq[i]; angle and product in fp32
__device__ __forceinline__ void rotate_pair(const float* src, float* dst, int i, int pos, const Rotary& rot, bf16_t* dst16 = nullptr) {
    const float a = (float)pos * rot.freq[i];
    const float c = cosf(a) * rot.amp, s = sinf(a) * rot.amp;
    const int a0 = rot.halves ? i : 2 * i, a1 = rot.halves ? i + rot.dims / 2 : 2 * i + 1;
    const float u = src[a0], v = src[a1];
    put_row(dst, dst16, a0, u * c - v * s);
    put_row(dst, dst16, a1, v * c + u * s);
}

// 1 / (L + exp(sink - mx)) times what brings weights of reference point mx to that denominator's (L: sum of exp(score - mx); mx -inf:
// no keys).  sink null: 1 / L.
__device__ __forceinline__ float sink_norm_f(float mx, float L, const float* sink, int h) {
    if (!sink) return 1.0f / L;
    const float s = sink[h];
    if (s <= mx) return 1.0f / (L + expf(s - mx));
    const float e = expf(mx - s);
    return e / (L * e + 1.0f);
}
__device__ __forceinline__ float head_gate_f(const float* gate, int ldg, size_t m, int h) { return gate ? sigmoid_f(gate[m * ldg + h]) : 1.0f; }

// Keys [lo, hi) of range `split` of a row's n_keys: whole groups of 16.
__device__ __forceinline__ int split_chunk(int n_keys, int n_split) { return ((n_keys + n_split - 1) / n_split + 15) & ~15; }

}  // namespace

}  // namespace lm
}  // namespace zg
