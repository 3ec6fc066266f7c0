// lm_latent_step.hip — latent attention of decode steps of up to eight sequences in two launches: everything from the projected queries to
// the partial sums of a key range, and from those to the heads' values.
//
// A step is a chain of dependent launches of 3 to 4 us each, whatever they do.  In their own launches were: the rotation of the queries
// and the token's cache row, the products that carry the queries into the latent space, the attention, the merge of its key ranges, and the
// products that make values of the weighted latents (lm_mix.hip, lm_linear.hip; steps with several rows of a sequence keep them, since
// a row's keys are then written in the same step).  64 x 256 + 32, 12 heads, six such layers of twelve: a step of one sequence 408 -> 375 us, of
// eight, with the queries' norm inside the product in front (lm_rows.hip), 705 -> 653.
// Long ranges are bound by a wave's own instructions and one round trip a turn of sixteen keys.  us a layer (projections and launches around it
// included), in five launches -> here: 16 heads, 64 x 256 + 64, one row behind 1000 keys 35.8 -> 25.3, behind 16000 98 -> 74; eight rows behind 4000
// 110 -> 86; 64 x 512 + 64, eight rows behind 4000 128 -> 112.
#include <type_traits>

#include "lm_latent_parts.h"

namespace zg {
namespace lm {

namespace {

struct LatentStepRest {
    const int* page_table;
    float* cache;
    const float* wkv;
    float* ws;
    Rotary rot;
    int max_pages, page_tokens, H;
    float scale, eps;
};

// A workgroup per (row, head, key range).  It carries its head's query into the latent space itself (KR x D weights of the head, 16 bytes a
// lane, LPR lanes a weight row), so every range of a head reads them: 32 KB at 64 x 256, beside the range's own keys.  The range that holds
// the row's own token works its cache row out (norm, rotation) and, for the first head, files it; no other workgroup reads that row.
// Everything that does not wait for the row's position is requested at entry; EAGER: the weights too, in front of the exit of ranges without
// keys (few rows; with more the empty ranges' reads would delay the others).
// KR <= 64 KP, R <= 64.
template <int KP, int LPR, bool EAGER>
__global__ __launch_bounds__(256) void latent_step_kernel(const int* row_pos, const int* row_slot, const float* q, const bf16_t* ukT, const float* lat, int ldq, int ld_lat,
                                                          int KR, int R, const LatentStepRest a) {
    constexpr int ND = KP + 1, D = 8 * LPR, RPI = 64 / LPR, NP = KP * LPR / 4, NL = (KP + 3) / 4;
    // weights a lane holds at a time (128 x 512: 146 registers, three workgroups to a compute unit, against 205 and two: 16 heads, six rows 63.5 us a
    // layer : 71.1)
    constexpr int BATCH = EAGER ? NP : 16;
    __shared__ float s_q[ND * 64], s_new[ND * 64], s_m[4], s_l[4], s_red[4];
    __shared__ float s_acc[4][ND * 64];
    const int m = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int DT = KR + R;
    const float* qh = q + (size_t)m * ldq + (size_t)h * (D + R);
    const bool own = lat != nullptr;
    const float* lr = own ? lat + (size_t)m * ld_lat : qh;
    f32x4 q8[2];
    u32x4 wr[NP < BATCH ? NP : BATCH];
    auto fetch_weights = [&](int from) {
#pragma unroll
        for (int j = 0; j < NP && j < BATCH; ++j) {
            if (from + j >= NP) break;
            const int row = min((4 * (from + j) + wave) * RPI + lane / LPR, KR - 1);
            wr[j] = *reinterpret_cast<const u32x4*>(ukT + ((size_t)h * KR + row) * D + (lane % LPR) * 8);
        }
    };
    auto fetch_query = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) q8[i] = *reinterpret_cast<const f32x4*>(qh + (lane % LPR) * 8 + 4 * i);
    };
    if constexpr (EAGER) fetch_weights(0), fetch_query();
    const int pos = row_pos[m], n_keys = pos + 1, chunk = split_chunk(n_keys, kAttnSplits);
    const int k_lo = min(n_keys, (int)blockIdx.z * chunk), k_hi = min(n_keys, k_lo + chunk);
    if (k_lo >= k_hi) return;
    const int* pt = a.page_table + (size_t)row_slot[m] * a.max_pages;
    if constexpr (!EAGER) fetch_weights(0), fetch_query();
    const bool has_new = own && k_hi == n_keys;
    float lv[NL], lw[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int i = own ? min(tid + 256 * j, KR - 1) : 0;
        lv[j] = lr[i];
        lw[j] = own ? a.wkv[i] : 0.0f;
    }
    // thread rt of its half of the workgroup: rotated pair rt, or a channel behind the rotated ones
    const int half = a.rot.dims / 2, rt = tid & 127;
    const int r0 = rt < half ? (a.rot.halves ? rt : 2 * rt) : a.rot.dims + rt - half, r1 = a.rot.halves ? rt + half : 2 * rt + 1;
    const float* rsrc = tid < 128 || !own ? qh + D : lr + KR;
    const bool any = R > 0;  // (without a rotated part: some valid channel)
    const float rx = (any ? rsrc : qh)[any ? min(r0, R - 1) : 0], ry = (any ? rsrc : qh)[any ? min(r1, R - 1) : 0], rf = half > 0 ? a.rot.freq[min(rt, half - 1)] : 0.0f;
    float r[4][ND];
    // (a turn's pages are asked for a turn before its keys, all four at once: behind the store of the token's row the compiler takes a look-up
    // for a vector load of its own, and one that stands between the keys' loads waits for them: four round trips a turn)
    int page[4];
    unsigned place[4], col[ND];  // of the keys looked up last: their pages, their places inside them; byte offsets of this lane's channels
#pragma unroll
    for (int i = 0; i < ND; ++i) col[i] = 4u * (unsigned)min(lane + 64 * i, DT - 1);
    auto look_up = [&](int kb) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned key = (unsigned)min(kb + u, k_hi - 1), at = key / (unsigned)a.page_tokens;
            page[u] = pt[at];
            place[u] = key - at * (unsigned)a.page_tokens;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto fetch = [&](float (&to)[4][ND]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float* row = a.cache + ((size_t)(unsigned)__builtin_amdgcn_readfirstlane(page[u]) * (unsigned)a.page_tokens + place[u]) * (unsigned)DT;
#pragma unroll
            for (int i = 0; i < ND; ++i) to[u][i] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(row) + col[i]);
        }
    };
    const int kb0 = k_lo + wave * 4;
    look_up(kb0);
    fetch(r);
    look_up(kb0 + 16);
    // the query in the latent space
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        if (j > 0 && j % BATCH == 0) {
            __builtin_amdgcn_sched_barrier(0);
            fetch_weights(j);
        }
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s = fmaf(q8[i / 2][2 * (i & 1) + 1], bf16_hi(wr[j % BATCH][i]), fmaf(q8[i / 2][2 * (i & 1)], bf16_lo(wr[j % BATCH][i]), s));
        if constexpr (LPR == 16) s = row16_allsum(s);
        else {  // eight lanes
            s += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(s), 0x141, 0xF, 0xF, true));  // 7 - lane
            s += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(s), 0x4E, 0xF, 0xF, true));   // lane ^ 2
            s += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(s), 0xB1, 0xF, 0xF, true));   // lane ^ 1
        }
        const int row = (4 * j + wave) * RPI + lane / LPR;
        if (lane % LPR == 0 && row < KR) s_q[row] = s;
    }
    if (has_new) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NL; ++j)
            if (tid + 256 * j < KR) ss = fmaf(lv[j], lv[j], ss);
        ss = wave_allsum(ss);
        if (lane == 0) s_red[wave] = ss;
    }
    {   // the rotated parts: the query's by the first two waves, the new key's by the others
        float* to = tid < 128 ? s_q + KR : s_new + KR;
        if (tid < 128 || has_new) {
            if (rt < half) {
                const float ang = (float)pos * rf, cs = cosf(ang) * a.rot.amp, sn = sinf(ang) * a.rot.amp;
                to[r0] = rx * cs - ry * sn;
                to[r1] = ry * cs + rx * sn;
            } else if (rt < R - half) to[r0] = rx;  // (rotated in pairs, the others alone)
        }
    }
    __syncthreads();
    if (has_new) {
        const float rc = 1.0f / sqrtf(((s_red[0] + s_red[1]) + (s_red[2] + s_red[3])) / (float)KR + a.eps);
#pragma unroll
        for (int j = 0; j < NL; ++j)
            if (tid + 256 * j < KR) s_new[tid + 256 * j] = lv[j] * rc * lw[j];
        __syncthreads();
        if (h == 0) {
            float* crow = a.cache + ((size_t)pt[pos / a.page_tokens] * a.page_tokens + pos % a.page_tokens) * DT;
            for (int d = tid; d < DT; d += 256) crow[d] = s_new[d];
        }
    }
    float qd[ND], acc[ND], fresh[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int d = lane + 64 * i;
        qd[i] = d < DT ? s_q[min(d, DT - 1)] : 0.0f;
        fresh[i] = has_new && d < DT ? s_new[min(d, DT - 1)] : 0.0f;
        acc[i] = 0.0f;
    }
    float mx = -INFINITY, l = 0.0f;
    // LAST: the turn that may hold the token's own key, or fewer than four
    auto take = [&](int kb, auto last) {
        constexpr bool LAST = decltype(last)::value;
        if (DT < 64 * ND) {  // (channels behind the last one brought it again, which need not be finite)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < ND; ++i) r[u][i] = lane + 64 * i < DT ? r[u][i] : 0.0f;
        }
        float s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool is_new = LAST && has_new && min(kb + u, k_hi - 1) == pos;
            float part = 0.0f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                if (is_new) r[u][i] = fresh[i];
                part = fmaf(qd[i], r[u][i], part);
            }
            s[u] = part;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[u] = wave_allsum(s[u]) * a.scale;
            if (LAST && kb + u >= k_hi) s[u] = -INFINITY;
        }
        const float mn = fmaxf(fmaxf(mx, s[0]), fmaxf(fmaxf(s[1], s[2]), s[3]));
        const float alpha = expf(mx - mn);  // 0 for the first group (mx = -inf, mn finite: key kb is always valid)
        float pw[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) pw[u] = expf(s[u] - mn);
        l = l * alpha + ((pw[0] + pw[1]) + (pw[2] + pw[3]));
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            float v = acc[i] * alpha;
#pragma unroll
            for (int u = 0; u < 4; ++u) v = fmaf(pw[u], r[u][i], v);
            acc[i] = v;
        }
        mx = mn;
    };
    int kb = kb0;
    for (; kb + 16 < k_hi; kb += 16) {
        float next[4][ND];
        fetch(next);
        look_up(kb + 32);
        take(kb, std::false_type());
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < ND; ++i) r[u][i] = next[u][i];
    }
    if (kb < k_hi) take(kb, std::true_type());
    if (lane == 0) {
        s_m[wave] = mx;
        s_l[wave] = l;
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) s_acc[wave][lane + 64 * i] = acc[i];
    __syncthreads();
    const float M4 = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
    float wgt[4], L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        wgt[w] = M4 == -INFINITY ? 0.0f : expf(s_m[w] - M4);  // a wave without keys: exp(-inf) = 0
        L += wgt[w] * s_l[w];
    }
    float* part = a.ws + (((size_t)m * a.H + h) * kAttnSplits + blockIdx.z) * (KR + 2);
    if (tid == 0) {
        part[0] = M4;
        part[1] = L;
    }
    for (int d = tid; d < KR; d += 256) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) v = fmaf(wgt[w], s_acc[w][d], v);
        part[2 + d] = v;
    }
}

// o[m][h Vd + n] = uv[h][n] . (the merged latent of head h), 4 RW values of a head per workgroup, each of which merges the key ranges itself
// (16 KB of partials at KR = 256; all ranges are requested at entry, those without keys are left out of the sums).  KR <= 256 NC.
template <int RW, int NC>
__global__ __launch_bounds__(256) void latent_values_kernel(const float* ws, const bf16_t* uv, const int* row_pos, const float* gate, const float* sink, int KR, int Vd, int H,
                                                            int ldg, float* out, int ldo) {
    __shared__ __attribute__((aligned(16))) float s_ctx[NC * 256];
    const int m = blockIdx.z, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, n0 = (blockIdx.x * 4 + (tid >> 6)) * RW;
    u32x4 wr[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) wr[r] = *reinterpret_cast<const u32x4*>(uv + ((size_t)h * Vd + min(n0 + r, Vd - 1)) * KR + min(lane * 8, KR - 8));
    const float* part = ws + ((size_t)m * H + h) * kAttnSplits * (KR + 2);
    float v[NC][kAttnSplits];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int s = 0; s < kAttnSplits; ++s) v[c][s] = part[(size_t)s * (KR + 2) + 2 + min(tid + 256 * c, KR - 1)];
    const int ls = min(lane, kAttnSplits - 1);
    float pm = part[(size_t)ls * (KR + 2)], pl = part[(size_t)ls * (KR + 2) + 1];
    const int n_keys = row_pos[m] + 1, chunk = split_chunk(n_keys, kAttnSplits), used = min(kAttnSplits, (n_keys + chunk - 1) / chunk);
    if (lane >= used) pm = -INFINITY, pl = 0.0f;
    const float M = wave_allmax(pm), w = pm == -INFINITY ? 0.0f : expf(pm - M);
    const float L = wave_allsum(lane < used ? w * pl : 0.0f);
    const float gf = head_gate_f(gate, ldg, m, h) * (sink ? sink_norm_f(M, L, sink, h) : 1.0f);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        float a = 0.0f;
#pragma unroll
        for (int s = 0; s < kAttnSplits; ++s) a = s < used ? fmaf(lane_value(w, s), v[c][s], a) : a;
        s_ctx[tid + 256 * c] = sink ? a * gf : a / L * gf;
    }
    __syncthreads();
    f32x4 x[2];
    const int k = min(lane * 8, KR - 8);
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = *reinterpret_cast<const f32x4*>(&s_ctx[k + 4 * i]);
    float mine = 0.0f;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s = fmaf(x[i / 2][2 * (i & 1) + 1], bf16_hi(wr[r][i]), fmaf(x[i / 2][2 * (i & 1)], bf16_lo(wr[r][i]), s));
        s = wave_allsum(lane * 8 < KR ? s : 0.0f);
        mine = lane == r ? s : mine;
    }
    if (lane < RW && n0 + lane < Vd) out[(size_t)m * ldo + (size_t)h * Vd + n0 + lane] = mine;
}

}  // namespace

// The forms these kernels have: heads of 64 or 128 unrotated channels, latents of up to 512 + 64 in whole 16-byte pieces.  And where they pay: each of a
// row's sixteen key ranges reads its head's KR x D weights again.  us a layer, five launches : here, the farthest apart of one to twelve thousand
// keys (E: rows x heads x KR x D / 2^20):
//   KR x D <= 16 K: 128 heads of 64 x 64, eight rows 124 : 105; of 128 x 64 (E 8) 158 : 140; of 64 x 256 (E 16) 136 : 130
//   32 K: 32 heads of 128 x 256, eight rows (E 8) 67.8 : 66.3; 48 heads, six rows (E 9) 79 : 74, eight (E 12) 84.8 : 87.6; 64 heads of 64 x 512, eight (E 16) 99 : 109
//   more: 24 heads of 128 x 320, six rows (E 5.6) 60.6 : 52.8; 16 heads of 128 x 512, six rows (E 6) 67.7 : 63.5, eight (E 8) 56.8 : 57.3; 128 heads, one row
//   (E 8) 94.6 : 97.1, eight (E 64) 207 : 404
bool latent_step_fits(int M, int H, int D, int R, int KR, int Vd, int ldq, int ld_lat) {
    const bool form = (D == 64 || D == 128) && KR >= 8 && KR <= 512 && KR % 8 == 0 && R >= 0 && R <= 64 && R % 4 == 0 && ldq % 4 == 0 && Vd > 0 && H > 0 && H <= 65535 && ld_lat >= 0;
    const long long weights = (long long)KR * D, all = weights * M * H;
    return form && (weights <= 16 * 1024 || all <= (weights <= 32 * 1024 ? 8ll << 20 : 6ll << 20));
}

int launch_latent_step(const LatentStep& a, hipStream_t s, bool* taken) {
    *taken = false;
    const uintptr_t all = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.ukT) | reinterpret_cast<uintptr_t>(a.uv);
    if (a.M <= 0 || a.M > kGemvMaxRows || (all & 15) != 0 || !latent_step_fits(a.M, a.H, a.D, a.R, a.KR, a.Vd, a.ldq, a.ld_lat) || !a.ws ||
        a.ws_floats < (size_t)a.M * a.H * kAttnSplits * (a.KR + 2))
        return ZG_OK;
    ZG_REQUIRE(a.rot.dims % 2 == 0 && a.rot.dims <= a.R, ZG_ERR_ARG, "rotary: %d rotated dimensions of a part of %d", a.rot.dims, a.R);
    const LatentStepRest rest{a.page_table, a.cache, a.wkv, a.ws, a.rot, a.max_pages, a.page_tokens, a.H, a.scale, a.eps};
    const dim3 grid(a.M, a.H, kAttnSplits);
    const bool eager = a.M <= 2;
#define ZG_LS(KP, LPR, EAGER) \
    latent_step_kernel<KP, LPR, EAGER><<<grid, 256, 0, s>>>(a.row_pos, a.row_slot, a.q, a.ukT, a.lat, a.ldq, a.ld_lat, a.KR, a.R, rest)
#define ZG_LS_K(KP)                              \
    do {                                         \
        if (a.D == 64 && eager) ZG_LS(KP, 8, true);   \
        else if (a.D == 64) ZG_LS(KP, 8, false);      \
        else if (eager) ZG_LS(KP, 16, true);          \
        else ZG_LS(KP, 16, false);                    \
    } while (0)
    if (a.KR <= 64) ZG_LS_K(1);
    else if (a.KR <= 128) ZG_LS_K(2);
    else if (a.KR <= 256) ZG_LS_K(4);
    else if (a.KR <= 320) ZG_LS_K(5);
    else ZG_LS_K(8);
#undef ZG_LS
#undef ZG_LS_K
    ZG_HIP(hipGetLastError());
    // values per wave: two where the ranges' merging spreads over idle compute units, four where it is repeated for several rows
    const int rw = a.M <= 2 ? 2 : 4;
    const dim3 vgrid((a.Vd + 4 * rw - 1) / (4 * rw), a.H, a.M);
#define ZG_LV(RW, NC) latent_values_kernel<RW, NC><<<vgrid, 256, 0, s>>>(a.ws, a.uv, a.row_pos, a.gate, a.sink, a.KR, a.Vd, a.H, a.ldg, a.out, a.ldo)
    if (rw == 2 && a.KR <= 256) ZG_LV(2, 1);
    else if (rw == 2) ZG_LV(2, 2);
    else if (a.KR <= 256) ZG_LV(4, 1);
    else ZG_LV(4, 2);
#undef ZG_LV
    note_kernel("latent_step_kernel");
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
