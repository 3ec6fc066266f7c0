// prefill_epi.h — device helpers shared by the epilogues of the whole-prompt Linears (prefill.hip, prefill_ring.hip, gemm_s4.hip).
#pragma once
#include "zg_kernels.h"

namespace zg {

// 16 significant bits (ZG_GPT_PREFILL_2PLANE)
__device__ __forceinline__ float coarse16(float x) {
    const uint32_t b = __float_as_uint(x);
    return __uint_as_float((b + 0x7fu + ((b >> 8) & 1u)) & ~0xffu);
}

// What is to be done about a Linear's rows that are not for two terms (zg_kernels.h SplitSeen): the marks of x and of w whose rows are worked out again, whether
// the call is refused for them.  (The words are written by the launch in front: scalar loads, which wait for none of the requests in flight.)
struct SeenPlan {
    int x, w;
    bool odd, refused;
};
__device__ __forceinline__ SeenPlan seen_plan(const SplitSeen& seen) {
    typedef const __attribute__((address_space(4))) unsigned* scalar_t;
    const scalar_t words = (scalar_t)reinterpret_cast<unsigned long long>(seen.words);
    SeenPlan p{0, 0, words[SEEN_ODD] == seen.call, false};
    if (words[SEEN_ANY] == seen.call) {
        int n[4] = {0, 0, 0, 0};
#pragma unroll 1
        for (int kind = 0; kind < 4; ++kind) {
            n[kind] = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) n[kind] += words[SEEN_ROWS + 16 * kind + i] == seen.call;
        }
        // either way leaves no sparse rows, and uneven ones of one operand only
        const int uneven_w = n[SEEN_X_SPARSE] + n[SEEN_W_SPARSE] + n[SEEN_W_UNEVEN], uneven_x = n[SEEN_X_SPARSE] + n[SEEN_W_SPARSE] + n[SEEN_X_UNEVEN], rows = min(uneven_w, uneven_x);
        p.x = rows == 0 ? 0 : uneven_w <= uneven_x ? MARK_SPARSE : MARK_UNEVEN;
        p.w = rows == 0 ? 0 : uneven_w <= uneven_x ? MARK_UNEVEN : MARK_SPARSE;
        p.refused = rows > kSeenFew;
    }
    return p;
}
// ... seen by a kernel of the call; the first workgroup tells the host
__device__ __forceinline__ bool seen_refused(const SplitSeen& seen) {
    const SeenPlan p = seen_plan(seen);
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (p.refused) __hip_atomic_store(seen.host, seen.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if ((p.x | p.w) != 0) __hip_atomic_store(seen.host + 1, seen.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (p.odd) __hip_atomic_store(seen.host + 2, seen.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return p.refused;
}

// four consecutive values -> 8 B into each of the two planes (plane stride `plane` elements), times 2^-exp
__device__ __forceinline__ void store_split4(uint16_t* dst, size_t plane, f32x4 v, int exp, int coarse) {
    if (coarse) v = f32x4{coarse16(v.x), coarse16(v.y), coarse16(v.z), coarse16(v.w)};
    uint32_t a[2], b[2];
    split2_f16(ldexpf(v.x, -exp), ldexpf(v.y, -exp), a[0], a[1]);
    split2_f16(ldexpf(v.z, -exp), ldexpf(v.w, -exp), b[0], b[1]);
#pragma unroll
    for (int p = 0; p < kPair; ++p) *reinterpret_cast<u32x2*>(dst + p * plane) = u32x2{a[p], b[p]};
}

__device__ __forceinline__ float gelu_fast(float x) {
    const float k1 = -2.0f * 1.4426950408889634f * 0.7978845608f, k2 = k1 * 0.044715f;
    const float arg = x * fmaf(x * x, k2, k1);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(arg));
}

// Cache append (src/ops.zig:152-157) of four consecutive values of one K or V row into the head-major caches [b][h][ctx][64]:
// element offset `off` = ((b H + head) ctx + t) 64 + d, in the cache's storage form (fp32, fp16 saturating, or the 24-bit pair of
// planes — zg_common.h b24_round).
__device__ __forceinline__ void kv_cache_store4(const PrefillQkv& q, void* cache, size_t off, f32x4 v) {
    if (q.kv_mode == 2) {  // four elements: 8 bytes of the bf16 plane, 4 of the byte plane
        const uint32_t r0 = b24_round(v.x), r1 = b24_round(v.y), r2 = b24_round(v.z), r3 = b24_round(v.w);
        *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(cache) + off) = u32x2{(r0 >> 8) | ((r1 >> 8) << 16), (r2 >> 8) | ((r3 >> 8) << 16)};
        *reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(cache) + q.kv_lo + off) =
            (r0 & 0xffu) | ((r1 & 0xffu) << 8) | ((r2 & 0xffu) << 16) | (r3 << 24);
    } else if (q.kv_mode) {
        _Float16* d = reinterpret_cast<_Float16*>(cache) + off;
        const float lim = 65504.0f;  // saturate: an inf in the cache would poison masked positions (0 * inf)
        d[0] = (_Float16)fminf(fmaxf(v.x, -lim), lim); d[1] = (_Float16)fminf(fmaxf(v.y, -lim), lim);
        d[2] = (_Float16)fminf(fmaxf(v.z, -lim), lim); d[3] = (_Float16)fminf(fmaxf(v.w, -lim), lim);
    } else {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(cache) + off) = v;
    }
}

// ... for four consecutive columns [n, n + 4) of qkv row m (PF_QKV epilogues; columns below E are q: nothing to append)
__device__ __forceinline__ void qkv_cache_store(const PrefillQkv& q, int m, int n, f32x4 v) {
    if (n < q.E) return;
    const int which = n >= 2 * q.E;
    const int e = n - (which ? 2 * q.E : q.E);
    const int b = m / q.P, t = m - b * q.P;
    kv_cache_store4(q, which ? q.v_cache : q.k_cache, (((size_t)b * q.H + (e >> 6)) * q.ctx + t) * 64 + (e & 63), v);
}

}  // namespace zg
