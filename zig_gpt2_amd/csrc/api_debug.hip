// api_debug.hip — test entries of the whole-prompt kernels (include/zgpt2.h): one Linear, one attention, on operands that the caller holds in other forms, with exponents
// that lie a given number of binades above what the data need, as those lie that a model has from its weights.
#include <math.h>

#include <algorithm>
#include <vector>

#include "zg_runtime.h"

using namespace zg;

namespace {

// device scratch of a call, given back when it ends
struct Scratch {
    char* base = nullptr;
    size_t used = 0, room = 0;
    ~Scratch() {
        (void)hipStreamSynchronize(ctx().stream);
        (void)hipFree(base);
    }
    int reserve(size_t bytes) {
        room = bytes;
        ZG_HIP(hipMalloc(reinterpret_cast<void**>(&base), bytes));
        return ZG_OK;
    }
    template <typename T>
    T* take(size_t n) {
        T* p = reinterpret_cast<T*>(base + used);
        used += (n * sizeof(T) + 255) & ~(size_t)255;
        return used <= room ? p : nullptr;
    }
};

template <typename T>
int to_host(std::vector<T>& h, const T* d, size_t n) {
    h.resize(n);
    ZG_HIP(hipMemcpyAsync(h.data(), d, n * sizeof(T), hipMemcpyDeviceToHost, ctx().stream));
    ZG_HIP(hipStreamSynchronize(ctx().stream));
    return ZG_OK;
}
int to_device(int* d, const int* h, size_t n) {
    ZG_HIP(hipMemcpyAsync(d, h, n * sizeof(int), hipMemcpyHostToDevice, ctx().stream));
    ZG_HIP(hipStreamSynchronize(ctx().stream));
    return ZG_OK;
}
// the exponent of the rows' largest value among rows first, first + step, ... (rows of zeros and of values that are not finite: none)
int largest(const std::vector<int>& exps, const std::vector<float>& norms, size_t first = 0, size_t step = 1) {
    int e = -1000;
    for (size_t i = first; i < exps.size(); i += step)
        if (norms[i] > 0.0f && std::isfinite(norms[i])) e = std::max(e, exps[i]);
    return e == -1000 ? 0 : e;
}
template <typename F>
int timed(int repeats, float* us, F&& launch) {
    hipStream_t s = ctx().stream;
    if (us == nullptr) {
        for (int i = 0; i < repeats; ++i) ZG_TRY(launch());
        return ZG_OK;
    }
    hipEvent_t e[2];
    for (hipEvent_t& v : e) ZG_HIP(hipEventCreate(&v));
    int st = launch();
    (void)hipEventRecord(e[0], s);
    for (int i = 0; i < repeats && st == ZG_OK; ++i) st = launch();
    (void)hipEventRecord(e[1], s);
    float ms = 0.0f;
    const hipError_t err = hipEventSynchronize(e[1]) == hipSuccess ? hipEventElapsedTime(&ms, e[0], e[1]) : hipErrorUnknown;
    for (hipEvent_t& v : e) (void)hipEventDestroy(v);
    ZG_TRY(st);
    ZG_HIP(err);
    *us = ms * 1e3f / (float)repeats;
    return ZG_OK;
}

}  // namespace

extern "C" {

int zg_debug_prefill_linear_at(const uint16_t* A, const uint16_t* W, const float* bias, void* C, size_t M, size_t N, size_t K, int epilogue, int force_kernel, int slices, float* ws,
                               size_t ws_floats, int slack, int repeats, float* us) {
    ZG_TRY(require_init());
    ZG_REQUIRE(A && W && C && is_device_ptr(A) && is_device_ptr(W) && is_device_ptr(C) && (!bias || is_device_ptr(bias)) && (!ws || is_device_ptr(ws)),
               ZG_ERR_ARG, "debug_prefill_linear: device pointers");
    ZG_REQUIRE(M >= 1 && M < (1u << 30) && N >= 64 && N < (1u << 30) && K >= 64 && K < (1u << 30) && epilogue >= 0 && epilogue <= 2 && force_kernel >= 0 &&
                   force_kernel <= 3 && slices >= 0 && slack >= 0 && slack <= 64 && repeats >= 1,
               ZG_ERR_ARG, "debug_prefill_linear: arguments");
    const int epi = epilogue == 0 ? PF_F32 : epilogue == 1 ? PF_RESID : PF_GELU_SPLIT;
    hipStream_t s = ctx().stream;
    Scratch at;
    ZG_TRY(at.reserve(M * K * 8 + N * K * 2 + M * 8 + N * 8 + (epi == PF_GELU_SPLIT ? M * N * 4 : 0) + 16 * 256));
    float *x = at.take<float>(M * K), *xn = at.take<float>(M), *wn = at.take<float>(N);
    uint16_t *xp = at.take<uint16_t>(M * K * 2), *wp = at.take<uint16_t>(N * K), *op = at.take<uint16_t>(epi == PF_GELU_SPLIT ? M * N * 2 : 0);
    int *xe = at.take<int>(M), *we = at.take<int>(N), *exps = at.take<int>(2);
    ZG_REQUIRE(exps != nullptr, ZG_ERR_STAGING, "debug_prefill_linear: scratch");
    // the caller's three-term planes stand for fp32 rows, which become two terms with one exponent, as in a prompt's pass
    ZG_TRY(launch_join_planes(A, nullptr, (int)M, (int)K, 3, x, s));
    Split2Job j{x, xp, xe, (int)M};
    j.norms = xn;
    ZG_TRY(launch_split2(j, Split2Job{}, (int)K, s));
    ZG_TRY(launch_plane_bf16(W, (int)N, (int)K, wp, we, wn, s));
    std::vector<int> he;
    std::vector<float> hx, hw, hb(N, 0.0f);
    ZG_TRY(to_host(he, xe, M));
    ZG_TRY(to_host(hx, xn, M));
    ZG_TRY(to_host(hw, wn, N));
    if (bias) ZG_TRY(to_host(hb, bias, N));
    auto top = [](const std::vector<float>& v) {
        float m = 0.0f;
        for (float e : v) m = fmaxf(m, fabsf(e));
        return m;
    };
    const float bound = top(hx) * top(hw) + top(hb);  // no output is larger
    const int e[2] = {largest(he, hx) + slack, (bound > 0.0f && std::isfinite(bound) ? ilogbf(bound) - 14 : 0) + slack};
    ZG_TRY(to_device(exps, e, 2));
    j.one = exps;
    ZG_TRY(launch_split2(j, Split2Job{}, (int)K, s));
    prefill_force_route(force_kernel, slices);
    const int st = timed(repeats, us, [&]() {
        return launch_prefill_gemm(PrefillA{xp, exps, false}, PrefillW{wp, we, 1}, bias, epi == PF_GELU_SPLIT ? static_cast<void*>(op) : C, (int)M, (int)N, (int)K,
                                   epi == PF_GELU_SPLIT ? 0 : (int)N, epi, ws, ws_floats, nullptr, s, nullptr, PlaneOut{exps + 1, 0});
    });
    prefill_force_route(0, 0);
    ZG_TRY(st);
    if (epi == PF_GELU_SPLIT) ZG_TRY(launch_join_planes(op, exps + 1, (int)M, (int)N, kPair, static_cast<bf16_t*>(C), s));
    return ZG_OK;
}

int zg_debug_prefill_linear(const uint16_t* A, const uint16_t* W, const float* bias, void* C, size_t M, size_t N, size_t K, int epilogue, int force_kernel, int slices, float* ws,
                            size_t ws_floats) {
    return zg_debug_prefill_linear_at(A, W, bias, C, M, N, K, epilogue, force_kernel, slices, ws, ws_floats, 0, 1, nullptr);
}

int zg_debug_attn_prefill_at(const float* qkv, uint16_t* out, size_t batch, size_t n_tokens, size_t n_embed, size_t n_heads, const float* k_cache, const float* v_cache, size_t ctx_len,
                             float* ws, size_t ws_floats, int key_tiles, int slack, int repeats, float* us) {
    ZG_TRY(require_init());
    ZG_REQUIRE(qkv && out && is_device_ptr(qkv) && is_device_ptr(out) && (!k_cache || (v_cache && is_device_ptr(k_cache) && is_device_ptr(v_cache))) &&
                   (!ws || is_device_ptr(ws)),
               ZG_ERR_ARG, "debug_attn_prefill: device pointers");
    ZG_REQUIRE(batch >= 1 && n_tokens >= 1 && n_heads >= 1 && n_embed == 64 * n_heads && batch * n_tokens < (1u << 24) && n_embed < (1u << 16) && (!k_cache || ctx_len >= n_tokens) &&
                   key_tiles >= 0 && key_tiles <= 255 && slack >= 0 && slack <= 64 && repeats >= 1,
               ZG_ERR_ARG, "debug_attn_prefill: arguments");
    ZG_REQUIRE(batch * n_tokens * 3 < (1u << 30) && (!k_cache || batch * n_heads * ctx_len < (1u << 30)), ZG_ERR_ARG, "debug_attn_prefill: arguments");
    (void)ws_floats;
    hipStream_t s = ctx().stream;
    const size_t rows = batch * n_tokens, thirds = 3 * rows, strips = k_cache ? batch * n_heads * ctx_len : 0, most = std::max(thirds, strips);
    Scratch at;
    ZG_TRY(at.reserve(std::max(thirds * n_embed, strips * 64) * 4 + most * 8 + 8 * 256));
    uint16_t* planes = at.take<uint16_t>(std::max(thirds * n_embed, strips * 64) * 2);  // of the look for the largest values, then of the output
    int *exps = at.take<int>(most), *own = at.take<int>(kBounds);
    float* norms = at.take<float>(most);
    ZG_REQUIRE(norms != nullptr, ZG_ERR_STAGING, "debug_attn_prefill: scratch");
    std::vector<int> he;
    std::vector<float> hn;
    auto look = [&](const float* x, size_t n, size_t K) -> int {
        Split2Job j{x, planes, exps, (int)n};
        j.norms = norms;
        ZG_TRY(launch_split2(j, Split2Job{}, (int)K, s));
        ZG_TRY(to_host(he, exps, n));
        return to_host(hn, norms, n);
    };
    int e[kBounds] = {0};
    ZG_TRY(look(qkv, thirds, n_embed));  // (a row's q, k and v behind each other)
    for (size_t which = 0; which < 3; ++which) e[PB_Q + which] = largest(he, hn, which, 3) + slack;
    for (int which = 1; which < 3 && k_cache; ++which) {
        ZG_TRY(look(which == 1 ? k_cache : v_cache, strips, 64));
        e[PB_Q + which] = largest(he, hn) + slack;
    }
    ZG_TRY(to_device(own, e, kBounds));
    ZG_TRY(timed(repeats, us, [&]() {
        return launch_attn_prefill(qkv, planes, (int)batch, (int)n_tokens, (int)n_embed, (int)n_heads, k_cache, v_cache, (int)ctx_len, own, 0, s, key_tiles > 0,
                                   reinterpret_cast<unsigned long long*>(ws));
    }));
    return launch_join_planes(planes, own + PB_V, (int)rows, (int)n_embed, kPair, out, s);
}

int zg_debug_attn_prefill(const float* qkv, uint16_t* out, size_t batch, size_t n_tokens, size_t n_embed, size_t n_heads, const float* k_cache, const float* v_cache, size_t ctx_len,
                          float* ws, size_t ws_floats, int key_tiles) {
    return zg_debug_attn_prefill_at(qkv, out, batch, n_tokens, n_embed, n_heads, k_cache, v_cache, ctx_len, ws, ws_floats, key_tiles, 0, 1, nullptr);
}

int zg_debug_prefill_route(int force_kernel, int slices) {
    ZG_REQUIRE(force_kernel >= 0 && (force_kernel <= 3 || force_kernel >= 16) && slices >= 0, ZG_ERR_ARG, "debug_prefill_route: arguments");
    prefill_force_route(force_kernel, slices);
    return ZG_OK;
}

}  // extern "C"
