// lm_window_parts.h — the keys a row of windowed attention sees and the shape of its scores (lm_seq.hip, lm_window_step.hip).
#pragma once
#include "lm_kernels.h"

namespace zg {
namespace lm {

namespace {

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }

// The keys a row sees, numbered from 0: first the kept tokens that lie in front of its window (the first `keep` positions of the
// sequence stay visible), then the window's keys up to the row's own position.  Every kernel below walks this numbering, so the
// order of a row's sums depends on its position alone.
struct KeySpan {
    int j_lo, n_first, n_keys;
};
__device__ __forceinline__ KeySpan key_span(int pos, const KeyMask& mask) {
    KeySpan k;
    k.j_lo = mask.chunk > 0 ? pos - pos % mask.chunk : mask.window > 0 ? max(0, pos - mask.window + 1) : 0;
    k.n_first = min(mask.keep, k.j_lo);
    k.n_keys = k.n_first + pos - k.j_lo + 1;
    return k;
}
__device__ __forceinline__ int key_pos(const KeySpan& k, int n) { return n < k.n_first ? n : k.j_lo + (n - k.n_first); }

// a scaled score on its way to the softmax: capped, then less the head's slope per position of distance (fp32); with a gate the
// result is the key's weight itself
__device__ __forceinline__ float shape_score(float sc, const ScoreShape& sh, int h, int dist) {
    if (sh.cap > 0.0f) sc = sh.cap * tanhf(sc / sh.cap);
    if (sh.slope) sc -= sh.slope[h] * (float)dist;
    if (sh.gate) sc = sigmoid_f(sc + sh.gate[h]);
    return sc;
}

}  // namespace

}  // namespace lm
}  // namespace zg
