// lm_norm.hip — what happens to a row of the residual stream between two sublayers: the sublayer's output (a row, or the chosen experts'
// rows with their weights) normed and added, the sum normed for the next sublayer and, in designs with a token shift, mixed with the
// normed row of the token before.  Rows of up to 1024 values in whole 16-byte pieces; lm_mix.hip and lm_moe.hip have the general kernels.
//
// Bound by memory: a wave holds a row in its registers (16-byte pieces, all requested in one go), so the two statistics between the
// loads and the stores are sums over one wave and nothing waits for other waves.  A wave takes a run of consecutive rows: the shift's
// row before is the one it has just normed, except for the first of the run, which it works out again.  (Then x must not be updated in
// place, since the run in front of it may have been written already.)
// us per launch, in front with a workgroup per row and two barriers a statistic: 8184 rows of 1024, sum and two norms 27 (of 117 MB) : 55,
// experts' rows added, normed and shifted 32 : 44 + 37 in two launches; 8 rows of 768 3.6 : 6.5 and 5.2 : 7.2.
// ROUTE: the choice of experts on the normed row, which is in the wave's registers; the fp32 row is then nobody's but an fp32 product's.  Norm and
// router's launch : here, us: 8184 rows of 1024, rounded rows 27.6 + 21.7 : 29.6; 333 rows of 768, fp32 4.1 + 5.5 : 7.2 (8.2 with the router in the LDS).
#include "lm_kernels.h"

#include <algorithm>
#include <cstdlib>

namespace zg {
namespace lm {

namespace {

enum { FROM_NOTHING, FROM_ROW, FROM_EXPERTS };
enum { TO_NOTHING, TO_NORM, TO_SHIFT };
enum { ROUTE_NOT, ROUTE_ONE, ROUTE_RUN };  // a row a wave: the router in its registers; runs of rows: in the LDS

// (In front of p what the first loads need: the leading arguments are in registers when a wave starts, the others a cold round trip away.
// from: p.y or p.yexp; shape: rows | waves of a workgroup << 28.)
template <int NV, int FROM, int TO, int ROUTE = ROUTE_NOT>
__global__ __launch_bounds__(256) void norm_rows_kernel(const float* x_in, const float* from, const float* p_wb, const float* p_wn, const float* p_mu, int W, unsigned shape,
                                                        int run, int top, const NormRows p) {
    const int lane = threadIdx.x & 63, M = shape & 0x0fffffff;
    const int first = __builtin_amdgcn_readfirstlane((blockIdx.x * (shape >> 28) + (threadIdx.x >> 6)) * run);
    if (ROUTE != ROUTE_RUN && first >= M) return;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    int at[NV];
    bool in[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        in[j] = lane * 4 + 256 * j < W;
        at[j] = min(lane * 4 + 256 * j, W - 4);
    }
    auto load = [&](const float* row, f32x4 (&v)[NV]) {
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = *reinterpret_cast<const f32x4*>(row + at[j]);
    };
    auto inv_rms = [&](const f32x4 (&v)[NV]) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const f32x4 a = in[j] ? v[j] : zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(a[e], a[e], ss);
        }
        return 1.0f / sqrtf(wave_allsum(ss) / (float)W + p.eps);
    };
    f32x4 wb[NV], wn[NV], mu[NV];
    if constexpr (FROM != FROM_NOTHING) load(p_wb, wb);
    if constexpr (TO != TO_NOTHING) load(p_wn, wn);
    if constexpr (TO == TO_SHIFT) load(p_mu, mu);
    constexpr int NE = ROUTE ? kNormExperts : 1;
    __shared__ u32x2 s_router[ROUTE == ROUTE_RUN ? NE * NV * 64 : 1];  // [expert][piece][lane]: in registers they would leave a SIMD two waves
    u32x2 router[NE][NV];
    float corr = 0.0f;
    f32x4 x_next[NV], y_next[NV];
    const int mine = lane >> 3;  // the expert whose score this lane and its seven neighbours have
    if constexpr (ROUTE) {
        const size_t row = (size_t)min(first, M - 1) * W;
        load(x_in + row, x_next);
        load(from + row, y_next);
        __builtin_amdgcn_sched_barrier(0);
        corr = p.correction[min(mine, p.experts - 1)];
    }
    if constexpr (ROUTE == ROUTE_ONE) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
#pragma unroll
            for (int j = 0; j < NV; ++j) router[e][j] = *reinterpret_cast<const u32x2*>(p.router + (size_t)min(e, p.experts - 1) * W + at[j]);
    }
    if constexpr (ROUTE == ROUTE_RUN) {
        constexpr int ALL = NE * NV * 64, FLY = 2 * NV;  // requests of a thread in flight
        for (int i0 = threadIdx.x; i0 < ALL; i0 += FLY * blockDim.x) {
            u32x2 v[FLY];
#pragma unroll
            for (int f = 0; f < FLY; ++f) {
                const int i = min(i0 + f * (int)blockDim.x, ALL - 1);
                v[f] = *reinterpret_cast<const u32x2*>(p.router + (size_t)min(i / (NV * 64), p.experts - 1) * W + min(i % 64 * 4 + i / 64 % NV * 256, W - 4));
            }
#pragma unroll
            for (int f = 0; f < FLY; ++f)
                if (i0 + f * (int)blockDim.x < ALL) s_router[i0 + f * blockDim.x] = v[f];
        }
        __syncthreads();
        if (first >= M) return;
    }
    // This lane's share of its expert's score of a normed row.
    auto score_share = [&](const f32x4 (&h)[NV]) {
        float z[NE];
        if (ROUTE == ROUTE_RUN) asm volatile("" ::: "memory");  // (read anew for every row)
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            z[e] = 0.0f;
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const f32x4 v = in[j] ? h[j] : zero;
                const u32x2 w = ROUTE == ROUTE_RUN ? s_router[(e * NV + j) * 64 + lane] : router[e][j];
                z[e] = fmaf(v.x, bf16_lo(w.x), z[e]);
                z[e] = fmaf(v.y, bf16_hi(w.x), z[e]);
                z[e] = fmaf(v.z, bf16_lo(w.y), z[e]);
                z[e] = fmaf(v.w, bf16_hi(w.y), z[e]);
            }
        }
#pragma unroll
        for (int d = 32, n = NE / 2; d >= 8; d >>= 1, n >>= 1)  // a lane keeps half of its sums with every step
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const float keep = lane & d ? z[n + i] : z[i], send = lane & d ? z[i] : z[n + i];
                z[i] = keep + __shfl_xor(send, d, 64);
            }
        return z[0];
    };
    // The choices of up to eight rows at once, row `first` + lane % 8: softmax over all experts, the largest by score + correction, the first of equals (NaN: the
    // first expert).  Exchanges between lanes are what costs here, 18 behind each other: a row at a time they took 14 us of 8184 rows.
    auto choose = [&](float (&share)[8], int rows) {
#pragma unroll
        for (int d = 4; d > 0; d >>= 1)
#pragma unroll
            for (int i = 0; i < d; ++i) {
                const float keep = lane & d ? share[d + i] : share[i], send = lane & d ? share[i] : share[d + i];
                share[i] = keep + __shfl_xor(send, d, 64);
            }
        const int row = lane & 7;
        auto over = [&](float v, auto op) {  // over the experts
#pragma unroll
            for (int d = 8; d < 64; d <<= 1) v = op(v, __shfl_xor(v, d, 64));
            return v;
        };
        auto larger = [](float a, float b) { return fmaxf(a, b); };
        const float s = mine < p.experts ? share[0] : -INFINITY;
        const float score = expf(s - over(s, larger)), weight = score / over(score, [](float a, float b) { return a + b; });  // (0 for experts that do not exist)
        float rank = mine < p.experts ? weight + corr : -INFINITY;
        for (int k = 0; k < p.choices; ++k) {
            const bool some = rank > -INFINITY;
            const float best = over(some ? rank : -INFINITY, larger);
            int first_of = some && rank == best ? mine : NE;
#pragma unroll
            for (int d = 8; d < 64; d <<= 1) first_of = min(first_of, __shfl_xor(first_of, d, 64));
            if (first_of == NE) first_of = 0;
            if (mine == first_of) {
                if (row < rows) {
                    p.pick[(size_t)(first + row) * p.choices + k] = mine;
                    p.pick_weight[(size_t)(first + row) * p.choices + k] = weight;
                }
                rank = -INFINITY;
            }
        }
    };
    // row m of the stream with the sublayer's output added
    auto sum = [&](int m, f32x4 (&x)[NV]) {
        load(x_in + (size_t)m * W, x);
        if constexpr (FROM == FROM_NOTHING) return;
        f32x4 y[NV];
        if constexpr (FROM == FROM_ROW) load(from + (size_t)m * W, y);
        else {
#pragma unroll
            for (int j = 0; j < NV; ++j) y[j] = zero;
            for (int k = 0; k < top; k += 2) {
                const size_t a = (size_t)m * top + k, b = a + (k + 1 < top ? 1 : 0);
                const float fa = p.weight[a], fb = p.weight[b];
                f32x4 u[NV], v[NV];
                load(from + (size_t)(p.inv ? p.inv[a] : (int)a) * W, u);
                load(from + (size_t)(p.inv ? p.inv[b] : (int)b) * W, v);
#pragma unroll
                for (int j = 0; j < NV; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[j][e] = fmaf(fa, u[j][e], y[j][e]);
                if (k + 1 < top) {
#pragma unroll
                    for (int j = 0; j < NV; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[j][e] = fmaf(fb, v[j][e], y[j][e]);
                }
            }
        }
        const float r = inv_rms(y);
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[j][e] += y[j][e] * r * (1.0f + wb[j][e]);
    };
    auto norm = [&](const f32x4 (&x)[NV], f32x4 (&h)[NV]) {
        const float r = inv_rms(x);
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) h[j][e] = x[j][e] * r * (1.0f + wn[j][e]);
    };
    f32x4 x[NV], h[NV], before[NV];
    if constexpr (ROUTE) {  // the next row is on its way while this one is scored
        float share[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) share[i] = 0.0f;
        for (int m = first; m < min(first + run, M); ++m) {
            const float r = inv_rms(y_next);
#pragma unroll
            for (int j = 0; j < NV; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] = x_next[j][e] + y_next[j][e] * r * (1.0f + wb[j][e]);
                if (in[j]) *reinterpret_cast<f32x4*>(p.x_out + (size_t)m * W + at[j]) = x[j];
            }
            norm(x, h);
            const size_t next = (size_t)min(m + 1, M - 1) * W;  // (behind the run: not used)
            load(x_in + next, x_next);
            load(from + next, y_next);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if (in[j]) {
                    if (p.out) *reinterpret_cast<f32x4*>(p.out + (size_t)m * W + at[j]) = h[j];
                    if (p.out16) *reinterpret_cast<u32x2*>(p.out16 + (size_t)m * W + at[j]) = u32x2{cvt_pk_bf16(h[j][0], h[j][1]), cvt_pk_bf16(h[j][2], h[j][3])};
                }
            const float z = score_share(h);
#pragma unroll
            for (int i = 0; i < 8; ++i) share[i] = i == m - first ? z : share[i];
        }
        choose(share, min(run, M - first));
        return;
    }
    if constexpr (TO == TO_SHIFT) {
        const int prev = p.row_prev ? p.row_prev[first] : -1;
        if (prev >= 0) {
            sum(prev, x);
            norm(x, before);
        }
    }
    for (int m = first; m < min(first + run, M); ++m) {
        if constexpr (TO == TO_SHIFT) {
            if (!p.row_prev || p.row_prev[m] < 0) load(p.shift_state + (size_t)p.row_slot[m] * p.slot_stride, before);
        }
        sum(m, x);
        if constexpr (FROM != FROM_NOTHING) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if (in[j]) *reinterpret_cast<f32x4*>(p.x_out + (size_t)m * W + at[j]) = x[j];
        }
        if constexpr (TO == TO_NOTHING) continue;
        norm(x, h);
        if constexpr (TO == TO_SHIFT) {
            if (p.shift_out) {
#pragma unroll
                for (int j = 0; j < NV; ++j)
                    if (in[j]) *reinterpret_cast<f32x4*>(p.shift_out + (size_t)p.row_slot[m] * p.slot_stride + at[j]) = h[j];
            }
            const int entry = p.row_entry_if_last ? p.row_entry_if_last[m] : -1;
            if (entry >= 0) {
#pragma unroll
                for (int j = 0; j < NV; ++j)
                    if (in[j]) *reinterpret_cast<f32x4*>(p.last_out + (size_t)entry * W + at[j]) = h[j];
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            f32x4 o = h[j];
            if constexpr (TO == TO_SHIFT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = h[j][e] + (before[j][e] - h[j][e]) * mu[j][e];
                before[j] = h[j];
            }
            if (in[j]) {
                if (p.out) *reinterpret_cast<f32x4*>(p.out + (size_t)m * W + at[j]) = o;
                if (p.out16) *reinterpret_cast<u32x2*>(p.out16 + (size_t)m * W + at[j]) = u32x2{cvt_pk_bf16(o[0], o[1]), cvt_pk_bf16(o[2], o[3])};
            }
        }
    }
}

}  // namespace

int launch_norm_rows(const NormRows& in, hipStream_t s, bool* taken) {
    *taken = false;
    NormRows p = in;
    if (p.M <= 0 || p.M >= (1 << 28) || p.W < 4 || p.W > 1024 || p.W % 4 != 0) return ZG_OK;
    const uintptr_t all = reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.x_out) | reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.yexp) |
                          reinterpret_cast<uintptr_t>(p.wb) | reinterpret_cast<uintptr_t>(p.wn) | reinterpret_cast<uintptr_t>(p.mu) | reinterpret_cast<uintptr_t>(p.out) |
                          reinterpret_cast<uintptr_t>(p.out16) | reinterpret_cast<uintptr_t>(p.shift_state) | reinterpret_cast<uintptr_t>(p.last_out);
    if ((all & 15) != 0 || p.slot_stride % 4 != 0) return ZG_OK;
    const int from = p.yexp ? FROM_EXPERTS : p.y ? FROM_ROW : FROM_NOTHING, to = p.mu ? TO_SHIFT : p.wn ? TO_NORM : TO_NOTHING;
    if (from == FROM_NOTHING && to == TO_NOTHING) return ZG_OK;
    if (p.router && (from != FROM_ROW || to != TO_NORM || p.experts < 1 || p.experts > kNormExperts || p.choices < 1 || p.choices > p.experts || !p.correction || (reinterpret_cast<uintptr_t>(p.router) & 7) != 0))
        return ZG_OK;
    if (from != FROM_NOTHING && to == TO_SHIFT && p.row_prev && p.x == p.x_out) return ZG_OK;  // (a run would read what another has written)
    // Runs as long as 2048 waves are left (a run of eight works out one row in nine twice); few rows a wave each in workgroups of their own.
    p.run = std::max(1, std::min(8, p.M / 2048));
    if (const char* e = getenv("ZGPT2_LM_NORM_RUN")) p.run = std::min(p.router ? 8 : 1 << 28, std::max(1, atoi(e)));  // (test hook: runs in short portions)
    const int waves = (p.M + p.run - 1) / p.run, per_group = p.M <= 64 ? 1 : 4;
    const dim3 grid((waves + per_group - 1) / per_group), block(64 * per_group);
#define ZG_NR(NV, FROM, TO) (norm_rows_kernel<NV, FROM, TO><<<grid, block, 0, s>>>(p.x, p.yexp ? p.yexp : p.y, p.wb, p.wn, p.mu, p.W, (unsigned)p.M | (unsigned)per_group << 28, p.run, p.top, p))
#define ZG_NRR_R(NV, R) (norm_rows_kernel<NV, FROM_ROW, TO_NORM, R><<<grid, block, 0, s>>>(p.x, p.y, p.wb, p.wn, p.mu, p.W, (unsigned)p.M | (unsigned)per_group << 28, p.run, p.top, p))
// (up to 2048 rows are a row a wave and all at once with two waves a SIMD)
#define ZG_NRR(NV) (p.run == 1 && p.M <= 2048 ? ZG_NRR_R(NV, ROUTE_ONE) : ZG_NRR_R(NV, ROUTE_RUN))
#define ZG_NR_V(FROM, TO)                       \
    do {                                        \
        if (p.W <= 256) ZG_NR(1, FROM, TO);     \
        else if (p.W <= 512) ZG_NR(2, FROM, TO); \
        else if (p.W <= 768) ZG_NR(3, FROM, TO); \
        else ZG_NR(4, FROM, TO);                \
    } while (0)
    if (p.router) {
        if (p.W <= 256) ZG_NRR(1);
        else if (p.W <= 512) ZG_NRR(2);
        else if (p.W <= 768) ZG_NRR(3);
        else ZG_NRR(4);
    } else if (from == FROM_NOTHING && to == TO_NORM) ZG_NR_V(FROM_NOTHING, TO_NORM);
    else if (from == FROM_NOTHING) ZG_NR_V(FROM_NOTHING, TO_SHIFT);
    else if (from == FROM_ROW && to == TO_NOTHING) ZG_NR_V(FROM_ROW, TO_NOTHING);
    else if (from == FROM_ROW && to == TO_NORM) ZG_NR_V(FROM_ROW, TO_NORM);
    else if (from == FROM_ROW) ZG_NR_V(FROM_ROW, TO_SHIFT);
    else if (to == TO_NOTHING) ZG_NR_V(FROM_EXPERTS, TO_NOTHING);
    else if (to == TO_NORM) ZG_NR_V(FROM_EXPERTS, TO_NORM);
    else ZG_NR_V(FROM_EXPERTS, TO_SHIFT);
#undef ZG_NR
#undef ZG_NRR
#undef ZG_NRR_R
#undef ZG_NR_V
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
