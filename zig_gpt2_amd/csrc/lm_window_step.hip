// lm_window_step.hip — attention inside a window, a chunk or the whole context in decode steps of few rows: two launches from the projected
// rows to the heads' results (lm_seq.hip has the three-launch form behind a preparation of its own, for heads that a matrix mixes, values that
// are turned, and other sizes).
//
// A step is a chain of dependent launches of 3 to 4 us each, whatever they do, and the three-launch form passes every score through memory.  Here
// a workgroup takes a row, a key head and a share of the row's keys: sixteen lanes hold a key (16 bytes a lane of its channels, and of
// its value), so a wave has eight keys of both in flight and a score is a sum over sixteen lanes; the softmax is a running one per sixteen
// lanes, merged at the end.  Where the rows come as the projection left them, every workgroup rotates its own heads' queries, and the one whose
// share holds the row's own token rotates the key and files the cache row; nobody else reads that row.
// 12 heads of 64 on 3 key heads, chunks of 512, three such layers of twelve: a step of one sequence 375 -> 340 us.
#include "lm_window_parts.h"

#include <stdlib.h>

#include <algorithm>

namespace zg {
namespace lm {

namespace {

struct WindowStepRest {
    const int* page_table;
    float* cache;
    int max_pages, page_tokens, H, n_split;
    float scale;
    Rotary rot;
    ScoreShape shape;
    float *st, *po;
};

// keys of a share: whole groups of 16
__device__ __forceinline__ int share_keys(int n_keys, int n_split) { return ((n_keys + n_split - 1) / n_split + 15) & ~15; }

// rep = H / G <= REP heads read a key head; D, V <= 64 RPL
template <int REP, int RPL, bool PREP>
__global__ __launch_bounds__(256) void window_step_kernel(const int* row_pos, const int* row_slot, const float* q, int ldq, int rep, int G, int D, int V, int window, int chunk,
                                                          int keep, const WindowStepRest a) {
    constexpr int CH = 64 * RPL, NQ = (REP * CH / 2 + 255) / 256;
    __shared__ __attribute__((aligned(16))) float s_q[REP][CH], s_k[CH], s_v[CH], s_acc[4][REP][CH];
    __shared__ float s_m[4][REP], s_l[4][REP];
    const int split = blockIdx.x, m = blockIdx.y, g = blockIdx.z, h0 = g * rep, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kq = lane >> 4, c = lane & 15;
    const float* row = q + (size_t)m * ldq;
    const int pos = row_pos[m];
    const KeySpan span = key_span(pos, KeyMask{window, keep, chunk});
    const int per = share_keys(span.n_keys, a.n_split), k_lo = min(span.n_keys, split * per), k_hi = min(span.n_keys, k_lo + per);
    if (k_lo >= k_hi) return;
    const bool has_new = PREP && k_hi == span.n_keys;
    // the queries, and the token's own key and value, on their way
    const int half = PREP ? a.rot.dims / 2 : 0, qpairs = D / 2;
    auto pair_at = [&](int i, int& x, int& y) {  // channels of pair i: rotated ones first
        const bool turn = i < half && a.rot.halves;
        x = turn ? i : 2 * i;
        y = turn ? i + half : 2 * i + 1;
    };
    float qx[NQ], qy[NQ], fr[NQ], kx = 0.0f, ky = 0.0f, kf = 0.0f, nv[RPL];
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const int idx = tid + 256 * j, hh = min(idx / (CH / 2), rep - 1), i = min(idx % (CH / 2), qpairs - 1);
        int x, y;
        pair_at(i, x, y);
        const float* src = row + (size_t)(h0 + hh) * D;
        qx[j] = src[x];
        qy[j] = src[y];
        fr[j] = half > 0 ? a.rot.freq[min(i, half - 1)] : 0.0f;
    }
    if constexpr (PREP) {
        const int i = min(tid % (CH / 2), qpairs - 1);
        int x, y;
        pair_at(i, x, y);
        const float* src = row + (size_t)(a.H + g) * D;
        kx = src[x];
        ky = src[y];
        kf = half > 0 ? a.rot.freq[min(i, half - 1)] : 0.0f;
#pragma unroll
        for (int r = 0; r < RPL; ++r) nv[r] = row[(size_t)(a.H + G) * D + (size_t)g * V + min(lane + 64 * r, V - 1)];
    }
    const int* pages = a.page_table + (size_t)row_slot[m] * a.max_pages;
    const size_t cstride = (size_t)G * (D + V);
    f32x4 kd[2][RPL], vd[2][RPL];
    auto row_of = [&](int j) { return a.cache + ((size_t)pages[(j / a.page_tokens) % a.max_pages] * a.page_tokens + j % a.page_tokens) * cstride; };
    auto fetch = [&](int base, f32x4 (&k)[2][RPL], f32x4 (&v)[2][RPL]) {
        const float* at[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) at[u] = row_of(key_pos(span, min(base + 4 * u + kq, k_hi - 1)));
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < RPL; ++r) {
                k[u][r] = *reinterpret_cast<const f32x4*>(at[u] + (size_t)g * D + min(4 * c + 64 * r, D - 4));
                v[u][r] = *reinterpret_cast<const f32x4*>(at[u] + (size_t)G * D + (size_t)g * V + min(4 * c + 64 * r, V - 4));
            }
    };
    int base = k_lo + wave * 8;
    fetch(base, kd, vd);
    // q (and the new key) into the LDS, zero beyond D
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const int idx = tid + 256 * j, hh = idx / (CH / 2), i = idx % (CH / 2);
        if (hh >= REP) continue;
        int x, y;
        pair_at(i, x, y);
        float ox = qx[j], oy = qy[j];
        if (PREP && i < half) {
            float sn, cs;
            sincosf((float)pos * fr[j], &sn, &cs);
            ox = (qx[j] * cs - qy[j] * sn) * a.rot.amp;
            oy = (qy[j] * cs + qx[j] * sn) * a.rot.amp;
        }
        const bool in = i < qpairs && hh < rep;
        s_q[hh][in ? x : 2 * i] = in ? ox : 0.0f;
        s_q[hh][in ? y : 2 * i + 1] = in ? oy : 0.0f;
    }
    if constexpr (PREP) {
        if (has_new && tid < CH / 2 && tid < qpairs) {
            int x, y;
            pair_at(tid, x, y);
            float ox = kx, oy = ky;
            if (tid < half) {
                float sn, cs;
                sincosf((float)pos * kf, &sn, &cs);
                ox = (kx * cs - ky * sn) * a.rot.amp;
                oy = (ky * cs + kx * sn) * a.rot.amp;
            }
            s_k[x] = ox;
            s_k[y] = oy;
        }
        if (has_new && wave == 3) {
#pragma unroll
            for (int r = 0; r < RPL; ++r)
                if (lane + 64 * r < V) s_v[lane + 64 * r] = nv[r];
        }
    }
    __syncthreads();
    if (has_new) {
        float* crow = row_of(pos);
        for (int i = tid; i < D + V; i += 256) crow[i < D ? (size_t)g * D + i : (size_t)G * D + (size_t)g * V + i - D] = i < D ? s_k[i] : s_v[i - D];
    }
    f32x4 qv[REP][RPL], acc[REP][RPL];
    float mx[REP], l[REP];
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < REP; ++h) {
        mx[h] = -INFINITY;
        l[h] = 0.0f;
#pragma unroll
        for (int r = 0; r < RPL; ++r) {
            qv[h][r] = *reinterpret_cast<const f32x4*>(&s_q[h][4 * c + 64 * r]);
            acc[h][r] = zero;
        }
    }
    auto take = [&](int at) {
        bool ok[2];
        int dist[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n = at + 4 * u + kq, j = key_pos(span, min(n, k_hi - 1));
            ok[u] = n < k_hi;
            dist[u] = pos - j;
            if (PREP && has_new && j == pos) {
#pragma unroll
                for (int r = 0; r < RPL; ++r) {
                    kd[u][r] = *reinterpret_cast<const f32x4*>(&s_k[min(4 * c + 64 * r, D - 4)]);
                    vd[u][r] = *reinterpret_cast<const f32x4*>(&s_v[min(4 * c + 64 * r, V - 4)]);
                }
            }
#pragma unroll
            for (int r = 0; r < RPL; ++r)
                if (4 * c + 64 * r >= D) kd[u][r] = zero;
        }
#pragma unroll
        for (int h = 0; h < REP; ++h) {
            float s[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float d = 0.0f;
#pragma unroll
                for (int r = 0; r < RPL; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) d = fmaf(qv[h][r][e], kd[u][r][e], d);
                s[u] = shape_score(row16_allsum(d) * a.scale, a.shape, min(h0 + h, a.H - 1), dist[u]);
                if (!ok[u]) s[u] = -INFINITY;
            }
            const float mn = fmaxf(mx[h], fmaxf(s[0], s[1])), ref = mn == -INFINITY ? 0.0f : mn;
            const float alpha = expf(mx[h] - ref), p0 = expf(s[0] - ref), p1 = expf(s[1] - ref);
            l[h] = l[h] * alpha + (p0 + p1);
#pragma unroll
            for (int r = 0; r < RPL; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[h][r][e] = fmaf(p1, vd[1][r][e], fmaf(p0, vd[0][r][e], acc[h][r][e] * alpha));
            mx[h] = mn;
        }
    };
    while (base + 32 < k_hi) {
        f32x4 kn[2][RPL], vn[2][RPL];
        fetch(base + 32, kn, vn);
        take(base);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < RPL; ++r) {
                kd[u][r] = kn[u][r];
                vd[u][r] = vn[u][r];
            }
        base += 32;
    }
    if (base < k_hi) take(base);
    // the four groups of lanes, then the four waves
#pragma unroll
    for (int h = 0; h < REP; ++h) {
        float top = fmaxf(mx[h], __shfl_xor(mx[h], 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float f = top == -INFINITY ? 0.0f : expf(mx[h] - top);
        float lt = l[h] * f;
        lt += __shfl_xor(lt, 16, 64);
        lt += __shfl_xor(lt, 32, 64);
        if (lane == 0) {
            s_m[wave][h] = top;
            s_l[wave][h] = lt;
        }
#pragma unroll
        for (int r = 0; r < RPL; ++r) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float t = acc[h][r][e] * f;
                t += __shfl_xor(t, 16, 64);
                v[e] = t + __shfl_xor(t, 32, 64);
            }
            if (kq == 0) *reinterpret_cast<f32x4*>(&s_acc[wave][h][4 * c + 64 * r]) = v;
        }
    }
    __syncthreads();
    for (int o = tid; o < rep * V; o += 256) {
        const int h = o / V, ch = o % V;
        const float top = fmaxf(fmaxf(s_m[0][h], s_m[1][h]), fmaxf(s_m[2][h], s_m[3][h])), ref = top == -INFINITY ? 0.0f : top;
        float v = 0.0f, lt = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = expf(s_m[w][h] - ref);  // (a wave without keys, or whose scores are all minus infinity: 0)
            v = fmaf(f, s_acc[w][h][ch], v);
            lt = fmaf(f, s_l[w][h], lt);
        }
        const size_t at = ((size_t)m * a.n_split + split) * a.H + h0 + h;
        a.po[at * V + ch] = v;
        if (ch == 0) {
            a.st[at * 2] = top;
            a.st[at * 2 + 1] = lt;
        }
    }
}

// out[m][h V + c] = the shares' sums over their common denominator (with the head's sink), in share order, times the gate; a wave per 64 values
// of a head.  The shares' sums are requested sixteen at a time, the first sixteen in front of everything else; shares without keys hold
// what an earlier step left and are not used.
__global__ __launch_bounds__(256) void window_join_kernel(const float* st, const float* po, const int* row_pos, const float* sink, int H, int V, int n_split, int window,
                                                          int chunk, int keep, float* out, int ldo, const float* gate, int ldg, float factor) {
    const int h = blockIdx.x, m = blockIdx.y, lane = threadIdx.x & 63, c = min((int)threadIdx.x, V - 1);
    const size_t at = (size_t)m * n_split * H + h;
    const int sl = min(lane, n_split - 1);
    float pm = st[(at + (size_t)sl * H) * 2], pl = st[(at + (size_t)sl * H) * 2 + 1];
    float v[16];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int s = 0; s < 16; ++s) v[s] = po[(at + (size_t)min(s0 + s, n_split - 1) * H) * V + c];
    };
    fetch(0);
    const float sk = sink ? sink[h] : -INFINITY;
    const int n_keys = key_span(row_pos[m], KeyMask{window, keep, chunk}).n_keys, per = share_keys(n_keys, n_split), used = (n_keys + per - 1) / per;
    if (lane >= used) pm = -INFINITY, pl = 0.0f;
    const float top = fmaxf(wave_allmax(pm), sk), w = expf(pm - top);
    const float den = wave_allsum(w * pl) + (sink ? expf(sk - top) : 0.0f);
    float a = 0.0f;
    for (int s0 = 0; s0 < used; s0 += 16) {
        if (s0 > 0) fetch(s0);
#pragma unroll
        for (int s = 0; s < 16; ++s)
            if (s0 + s < used) a = fmaf(lane_value(w, s0 + s), v[s], a);
    }
    a /= den;
    if ((int)threadIdx.x >= V) return;
    if (gate) a *= sigmoid_f(gate[(size_t)m * ldg + (size_t)h * V + c]) * factor;
    out[(size_t)m * ldo + (size_t)h * V + c] = a;
}

}  // namespace

int launch_window_step(const WindowStep& a, hipStream_t s, bool* taken) {
    *taken = false;
    for (const char* hook : {"ZGPT2_LM_WINDOW_GENERAL", "ZGPT2_LM_WINDOW_TILES"})  // test hooks: the other forms
        if (const char* e = getenv(hook))
            if (atoi(e) != 0) return ZG_OK;
    // (more rows, or wider heads: a wave's registers end, and the forms of lm_seq.hip have the chip full)
    if (a.M <= 0 || a.M > kGemvMaxRows || a.G <= 0 || a.H % a.G != 0 || a.H / a.G > 8 || a.H > 65535 || a.D < 4 || a.D > 128 || a.V < 4 || a.V > 128 || a.D % 4 != 0 ||
        a.V % 4 != 0 || a.shape.gate || a.n_split < 1 || a.n_split > 64 || !a.ws || a.ws_floats < (size_t)a.M * a.n_split * a.H * (a.V + 2) ||
        (reinterpret_cast<uintptr_t>(a.cache) & 15) != 0)
        return ZG_OK;
    if (a.prep) ZG_REQUIRE(a.prep->dims % 2 == 0 && a.prep->dims <= a.D, ZG_ERR_ARG, "rotary: %d rotated dimensions of %d", a.prep->dims, a.D);
    float* const st = a.ws;
    float* const po = st + (size_t)a.M * a.n_split * a.H * 2;
    const KeyMask mk{a.mask.window, a.mask.window > 0 ? a.mask.keep : 0, a.mask.chunk};
    const WindowStepRest rest{a.page_table, a.cache, a.max_pages, a.page_tokens, a.H, a.n_split, a.scale, a.prep ? *a.prep : Rotary{nullptr, 0, 1.0f, 0}, a.shape, st, po};
    const dim3 grid(a.n_split, a.M, a.G);
    const int rep = a.H / a.G, wide = std::max(a.D, a.V) > 64;
#define ZG_WS(REP, RPL, PREP) \
    window_step_kernel<REP, RPL, PREP><<<grid, 256, 0, s>>>(a.row_pos, a.row_slot, a.q, a.ldq, rep, a.G, a.D, a.V, mk.window, mk.chunk, mk.keep, rest)
#define ZG_WS_P(REP)                                  \
    do {                                              \
        if (a.prep && wide) ZG_WS(REP, 2, true);      \
        else if (a.prep) ZG_WS(REP, 1, true);         \
        else if (wide) ZG_WS(REP, 2, false);          \
        else ZG_WS(REP, 1, false);                    \
    } while (0)
    if (rep == 1) ZG_WS_P(1);
    else if (rep == 2) ZG_WS_P(2);
    else if (rep <= 4) ZG_WS_P(4);
    else ZG_WS_P(8);
#undef ZG_WS
#undef ZG_WS_P
    ZG_HIP(hipGetLastError());
    window_join_kernel<<<dim3(a.H, a.M), (a.V + 63) / 64 * 64, 0, s>>>(st, po, a.row_pos, a.sink, a.H, a.V, a.n_split, mk.window, mk.chunk, mk.keep, a.out, a.ldo, a.out_gate,
                                                                      a.ld_gate, a.out_factor);
    note_kernel("window_step_kernel");
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
