// lm_scan.hip — the gated recurrences with a decay per key channel (HGRN2, gated linear attention) for prompt portions, in chunks of
// 64 tokens as fp32 matrix products.
//
//   S_t = diag(f_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t          (HGRN2: k_t = 1 - f_t)
//
// Inside a chunk, with P(a, b) the product of the gates f_a .. f_b per channel:
//   end state from zero   B = sum_s (k_s P(s+1, end)) v_s^T
//   output                o_t = sum_(s<=t) A_ts v_s + S_start^T (q_t P(start, t)),     A_ts = sum_d q_t k_s P(s+1, t)
// A gate may be arbitrarily small, so no product is ever divided away: the tokens are cut into blocks of 8 and 16, and a pair (t, s) of
// different blocks meets at the start r of t's block, A_ts = sum_d (q_t P(r, t)) (k_s P(s+1, r-1)) — both factors products of gates, at
// most 1 in size, that at worst underflow where the true value does.  Pairs of one block of 8 are multiplied out token by token.
// The rounding error of a product of n gates is n half ulps, the same as the recurrence's own n multiplications.
//
// What bounds it: the fp32 matrix instruction (64 cycles per 32 x 32 x 2: 12.8 k cycles per chunk and head of 128 x 128 in the output
// kernel, 4 k in the state kernel) and the chunk states, written, carried and read (64 KB per chunk and head).  8 x 1023 tokens, 8 heads of
// 128 x 128: state 47 us, carry 27, output 77 = 151 us per layer; scanned token by token inside chunks it was 265 + 25 + 265.
#include <math.h>
#include <stdlib.h>

#include <algorithm>

#include "lm_kernels.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kChunk = 64;
enum { KIND_HGRN2 = 0, KIND_GLA = 1 };

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float log_sigmoid_f(float z) { return fminf(z, 0.0f) - log1pf(expf(-fabsf(z))); }

struct ScanArgs {
    const float* proj;  // rows [q (H D) | f or k (H D) | v (H V)]
    float* out;
    float* wsB;  // [chunk][H][D][V]
    float* wsA;  // [chunk][H][D]
    const int *ent_start, *ent_len;
    const float *bias, *low;  // HGRN2
    GlaGate gla;
    int ld, ldo, n_entries, H, D, V;
    const float* norm_w = nullptr;  // the norm behind the heads
    float norm_eps = 0.0f;
    bf16_t* out16 = nullptr;
};

__device__ __forceinline__ bool find_chunk(int id, const int* ent_len, int n_entries, int& e, int& c) {
    for (e = 0; e < n_entries; ++e) {
        const int nc = (ent_len[e] + kChunk - 1) / kChunk;
        if (id < nc) {
            c = id;
            return true;
        }
        id -= nc;
    }
    return false;
}

// gate and key of a channel from the projection's values: raw = f's (HGRN2) or k's (GLA) column, z = GLA's gate column
template <int KIND>
__device__ __forceinline__ void gate_of(const ScanArgs& p, int ch, float raw, float z, float& f, float& k) {
    if (KIND == KIND_GLA) {
        f = expf(log_sigmoid_f(z + p.gla.z_bias[ch]) * p.gla.inv_tau);
        k = raw;
    } else {
        const float l = p.low[ch];
        f = l + (1.0f - l) * sigmoid_f(raw + p.bias[ch]);
        k = 1.0f - f;
    }
}

// The gates (and for GLA the keys; for the outputs the queries) of a chunk's tokens into the LDS, rows of LD floats; tokens behind the
// chunk's end and channels beyond D as f = 1, k = q = 0.  All loads of a thread are requested before the first is used.
template <int KIND, int DP, int LD, bool WITH_Q>
__device__ __forceinline__ void load_chunk(const ScanArgs& p, int h, int m0, int n, float* sq, float* sf, float* sk) {
    constexpr int ROWS = 512 / DP, IT = kChunk / ROWS;
    const int i = threadIdx.x % DP, t0 = threadIdx.x / DP, HD = p.H * p.D, ch = h * p.D + min(i, p.D - 1);
    float qv[IT], rv[IT], zv[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const float* row = p.proj + (size_t)(m0 + min(t0 + it * ROWS, n - 1)) * p.ld + ch;
        if (WITH_Q) qv[it] = row[0];
        rv[it] = row[HD];
        zv[it] = KIND == KIND_GLA ? p.gla.z[(size_t)(m0 + min(t0 + it * ROWS, n - 1)) * p.gla.ldz + ch] : 0.0f;
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int t = t0 + it * ROWS;
        const bool ok = t < n && i < p.D;
        float f, k;
        gate_of<KIND>(p, ch, rv[it], zv[it], f, k);
        if (WITH_Q) sq[t * LD + i] = ok ? (KIND == KIND_GLA ? qv[it] * p.gla.q_scale : silu_f(qv[it])) : 0.0f;
        sf[t * LD + i] = ok ? f : 1.0f;
        if (KIND == KIND_GLA) sk[t * LD + i] = ok ? k : 0.0f;
    }
}

// phase A: a (chunk, head)'s end state from zero and the product of its gates.  Eight waves: two halves of the channels x four
// 32-column slices of v; an MFMA step takes tokens s and s + 8 (their LDS rows lie half the banks apart).
template <int KIND, int DP>
__global__ __launch_bounds__(512) void gated_chunk_state_kernel(const ScanArgs p) {
    constexpr int LD = DP + 4;
    __shared__ __attribute__((aligned(16))) float s_f[kChunk * LD];
    __shared__ __attribute__((aligned(16))) float s_k[KIND == KIND_GLA ? kChunk * LD : 4];
    __shared__ float s_F[4 * DP];
    int e, c;
    if (!find_chunk(blockIdx.x, p.ent_len, p.n_entries, e, c)) return;
    const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, kh = lane >> 5;
    const int n = min(kChunk, p.ent_len[e] - c * kChunk), m0 = p.ent_start[e] + c * kChunk, HD = p.H * p.D;
    float* const s_key = KIND == KIND_GLA ? s_k : s_f;  // where the decayed keys end up
    const float* vrow = p.proj + (size_t)m0 * p.ld + 2 * HD + (size_t)h * p.V;
    float vf[32];
    auto load_v = [&](int sl) {  // this lane's column of the slice, tokens 16 g + 8 kh + j
        const int col = min(sl * 32 + r, p.V - 1);
#pragma unroll
        for (int x = 0; x < 32; ++x) vf[x] = vrow[min(16 * (x >> 3) + 8 * kh + (x & 7), n - 1) * p.ld + col];
    };
    load_chunk<KIND, DP, LD, false>(p, h, m0, n, nullptr, s_f, s_k);
    const int sl = blockIdx.z * 4 + (wave >> 1);
    load_v(sl);
    __syncthreads();
    for (int idx = tid; idx < 4 * DP; idx += 512) {  // k_s times the gates behind s in its block of 16
        const int i = idx / DP, d = idx % DP;
        float suf = 1.0f;
#pragma unroll
        for (int t = 15; t >= 0; --t) {
            const int at = (16 * i + t) * LD + d;
            const float f = s_f[at];
            s_key[at] = (KIND == KIND_GLA ? s_k[at] : 1.0f - f) * suf;
            suf *= f;
        }
        s_F[i * DP + d] = suf;
    }
    __syncthreads();
    for (int idx = tid; idx < 3 * DP; idx += 512) {  // ... and the gates of the blocks behind
        const int i = idx / DP, d = idx % DP;
        float g = s_F[(i + 1) * DP + d];
        for (int m = i + 2; m < 4; ++m) g *= s_F[m * DP + d];
#pragma unroll
        for (int t = 0; t < 16; ++t) s_key[(16 * i + t) * LD + d] *= g;
    }
    if (tid < p.D && blockIdx.z == 0) p.wsA[((size_t)blockIdx.x * p.H + h) * p.D + tid] = (s_F[tid] * s_F[DP + tid]) * (s_F[2 * DP + tid] * s_F[3 * DP + tid]);
    __syncthreads();
    constexpr int TILES = DP / 64;  // channel tiles of a wave
    float* B = p.wsB + ((size_t)blockIdx.x * p.H + h) * p.D * p.V;
    if (sl * 32 < p.V) {
        f32x16 acc[TILES];
#pragma unroll
        for (int i = 0; i < TILES; ++i)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[i][x] = 0.0f;
#pragma unroll
        for (int x = 0; x < 32; ++x) {
            const int s = 16 * (x >> 3) + 8 * kh + (x & 7);
            const float v = s < n ? vf[x] : 0.0f;
#pragma unroll
            for (int i = 0; i < TILES; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(s_key[s * LD + ((wave & 1) * TILES + i) * 32 + r], v, acc[i], 0, 0, 0);
        }
        const int col = sl * 32 + r;
#pragma unroll
        for (int i = 0; i < TILES; ++i)
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const int d = ((wave & 1) * TILES + i) * 32 + 8 * (x >> 2) + 4 * kh + (x & 3);
                if (d < p.D && col < p.V) B[(size_t)d * p.V + col] = acc[i][x];
            }
    }
}

// phase C: the outputs of a (chunk, head) from its start state (wsB).  Eight waves; the state and the values come straight from memory as
// matrix operands, half of the state requested in front of the work on the gates, the rest beside the products.  A workgroup alone takes 22 us,
// 5 of them in the matrix cores: A takes the place of gates that have been used and waits in registers until then, so that two workgroups of
// HGRN2 share a compute unit (72 KB each, 128 registers a lane; keys of GLA need an array of their own, and one is alone).  8 x 1023 tokens, 8
// heads of 128 x 128: 77 us against 95 for one workgroup of 89 KB; 6 heads 62 against 69, GLA 78 against 81; 333 tokens, 6 heads: 22 on both.
template <int KIND, int DP>
__global__ __launch_bounds__(512, KIND == KIND_HGRN2 && DP == 128 ? 4 : 2) void gated_chunk_out_kernel(const ScanArgs p) {
    constexpr int LD = DP + 4, LA = kChunk + 4;
    __shared__ __attribute__((aligned(16))) float s_q[kChunk * LD];
    __shared__ __attribute__((aligned(16))) float s_f[kChunk * LD];
    __shared__ __attribute__((aligned(16))) float s_k[KIND == KIND_GLA ? kChunk * LD : 4];
    __shared__ __attribute__((aligned(16))) float s_F[8 * DP];  // gates of every block of 8 multiplied
    int e, c;
    if (!find_chunk(blockIdx.x, p.ent_len, p.n_entries, e, c)) return;
    const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, kh = lane >> 5;
    const int n = min(kChunk, p.ent_len[e] - c * kChunk), m0 = p.ent_start[e] + c * kChunk, HD = p.H * p.D;
    float* const s_key = KIND == KIND_GLA ? s_k : s_f;
    float* const s_A = s_f;  // once gates and keys have been used
    const float* vrow = p.proj + (size_t)m0 * p.ld + 2 * HD + (size_t)h * p.V;
    const float* S0 = p.wsB + ((size_t)blockIdx.x * p.H + h) * p.D * p.V;
    const int mt = wave & 1;  // this wave's 32 tokens
    float Sf[DP / 2], vf[32];
    bool odd_v = false;
    // this lane's column of the slice: channels 8 g + 4 kh + j of the state, tokens alike (channels beyond D and tokens behind the chunk: the last
    // valid ones, met by zeros)
    const int sl = blockIdx.z * 4 + (wave >> 1), col = min(sl * 32 + r, p.V - 1);
    constexpr int SHARE = DP / 4;  // the state in two shares: two workgroups fit a compute unit with at most 128 registers a lane
    auto load_state = [&](int from) {
#pragma unroll
        for (int x = from; x < from + SHARE; ++x) Sf[x] = S0[min(8 * (x >> 2) + 4 * kh + (x & 3), p.D - 1) * p.V + col];
        __builtin_amdgcn_sched_barrier(0);
    };
    load_chunk<KIND, DP, LD, true>(p, h, m0, n, s_q, s_f, s_k);
    __syncthreads();
    load_state(0);

    float near0 = 0.0f, near1 = 0.0f;  // A of token part of the wave's block against s0 and s0 + 4
    const int part = lane & 15, s0 = lane >> 4;
    {  // pairs of one block of 8 (a wave's own): lane (s, part) carries k_s P(s+1, t) of its channels from t to t, for s and s + 4
        constexpr int PARTS = DP / 64;
        f32x4 a0[PARTS], a1[PARTS];
        for (int t = 0; t < 8; ++t) {
            float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
            for (int j = 0; j < PARTS; ++j) {
                const int at = (8 * wave + t) * LD + 4 * (part + 16 * j);
                const f32x4 f = *reinterpret_cast<const f32x4*>(&s_f[at]), q = *reinterpret_cast<const f32x4*>(&s_q[at]);
                f32x4 k;
                if (KIND == KIND_GLA) k = *reinterpret_cast<const f32x4*>(&s_k[at]);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float kv = KIND == KIND_GLA ? k[u] : 1.0f - f[u];
                    a0[j][u] = t == s0 ? kv : a0[j][u] * f[u];
                    a1[j][u] = t == s0 + 4 ? kv : a1[j][u] * f[u];
                    x0 = fmaf(q[u], a0[j][u], x0);
                    x1 = fmaf(q[u], a1[j][u], x1);
                }
            }
            x0 = row16_allsum(x0);
            x1 = row16_allsum(x1);
            if (part == t) {
                near0 = t >= s0 ? x0 : 0.0f;
                near1 = t >= s0 + 4 ? x1 : 0.0f;
            }
        }
    }
    __syncthreads();
    for (int idx = tid; idx < 8 * DP; idx += 512) {  // blocks of 8: q_t P(start, t), k_s P(s+1, end)
        const int b = idx / DP, d = idx % DP;
        float f[8], pre = 1.0f, suf = 1.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int at = (8 * b + t) * LD + d;
            f[t] = s_f[at];
            pre *= f[t];
            s_q[at] *= pre;
        }
        s_F[b * DP + d] = pre;
#pragma unroll
        for (int t = 7; t >= 0; --t) {
            const int at = (8 * b + t) * LD + d;
            s_key[at] = (KIND == KIND_GLA ? s_k[at] : 1.0f - f[t]) * suf;
            suf *= f[t];
        }
    }
    __syncthreads();
    // a 16 x 16 tile of A: tokens 16 i + .. against 16 j + ..; the gates of the blocks between multiply the queries
    const int m16 = lane & 15, kg = lane >> 4;
    auto pair_tile = [&](int i, int j) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int d0 = 0; d0 < DP; d0 += 16) {
            f32x4 q = *reinterpret_cast<const f32x4*>(&s_q[(16 * i + m16) * LD + d0 + 4 * kg]);
            const f32x4 k = *reinterpret_cast<const f32x4*>(&s_key[(16 * j + m16) * LD + d0 + 4 * kg]);
            for (int b = 2 * j + 2; b < 2 * i; ++b) q *= *reinterpret_cast<const f32x4*>(&s_F[b * DP + d0 + 4 * kg]);
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q[u], k[u], acc, 0, 0, 0);
        }
        return acc;  // element x: token 16 i + 4 kg + x against token 16 j + m16
    };
    f32x4 half = {0.0f, 0.0f, 0.0f, 0.0f}, cross = half;
    if (wave < 4) half = pair_tile(wave, wave);  // the second half of a block of 16 against its first
    __syncthreads();
    for (int idx = tid; idx < kChunk * (DP / 4); idx += 512) {  // blocks of 16: the halves meet
        const int t = idx / (DP / 4), d = (idx % (DP / 4)) * 4, b = t >> 3;
        f32x4* v = reinterpret_cast<f32x4*>((b & 1) ? &s_q[t * LD + d] : &s_key[t * LD + d]);
        *v *= *reinterpret_cast<const f32x4*>(&s_F[(b ^ 1) * DP + d]);
    }
    __syncthreads();
    // blocks of 16 against earlier ones; the last two waves have the zeros behind the diagonal that a product of 32 tokens meets
    const int ti = wave < 1 ? 1 : wave < 3 ? 2 : wave < 6 ? 3 : wave == 6 ? 0 : 2, tj = wave < 1 ? 0 : wave < 3 ? wave - 1 : wave < 6 ? wave - 3 : wave == 6 ? 1 : 3;
    if (wave < 6) cross = pair_tile(ti, tj);
    __syncthreads();
    load_state(SHARE);
    if (part < 8) {
        s_A[(8 * wave + part) * LA + 8 * wave + s0] = near0;
        s_A[(8 * wave + part) * LA + 8 * wave + s0 + 4] = near1;
    }
    if (wave < 4 && (kg >= 2) == (m16 < 8))
#pragma unroll
        for (int x = 0; x < 4; ++x) s_A[(16 * wave + 4 * kg + x) * LA + 16 * wave + m16] = kg >= 2 ? half[x] : 0.0f;
#pragma unroll
    for (int x = 0; x < 4; ++x) s_A[(16 * ti + 4 * kg + x) * LA + 16 * tj + m16] = cross[x];
    for (int idx = tid; idx < 48 * (DP / 4); idx += 512) {  // the queries from the chunk's start
        const int t = 16 + idx / (DP / 4), d = (idx % (DP / 4)) * 4;
        f32x4* v = reinterpret_cast<f32x4*>(&s_q[t * LD + d]);
        f32x4 g = *v;
        for (int b = 0; b < 2 * (t >> 4); ++b) g *= *reinterpret_cast<const f32x4*>(&s_F[b * DP + d]);
        *v = g;
    }
    __syncthreads();
    f32x16 acc;
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[x] = 0.0f;
    if (sl * 32 < p.V) {
        auto state_share = [&](int from) {
#pragma unroll
            for (int g = from / 4; g < (from + SHARE) / 4; ++g) {
                const f32x4 q = *reinterpret_cast<const f32x4*>(&s_q[(32 * mt + r) * LD + 8 * g + 4 * kh]);
#pragma unroll
                for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(q[u], Sf[4 * g + u], acc, 0, 0, 0);
            }
        };
        state_share(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 32; ++x) vf[x] = vrow[min(8 * (x >> 2) + 4 * kh + (x & 3), n - 1) * p.ld + col];
        __builtin_amdgcn_sched_barrier(0);
        state_share(SHARE);
        // A is zero above its diagonal, but zero times a value that is not finite is not: such values are left out here and added below,
        // token by token, to the outputs at and behind them only
        odd_v = false;
#pragma unroll
        for (int x = 0; x < 32; ++x) odd_v = odd_v || !(fabsf(vf[x]) <= 3.4028235e38f);
        const bool any_odd = __any(odd_v);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            if (g >= 4 && mt == 0) break;
            const f32x4 a = *reinterpret_cast<const f32x4*>(&s_A[(32 * mt + r) * LA + 8 * g + 4 * kh]);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float v = vf[4 * g + u];
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], fabsf(v) <= 3.4028235e38f ? v : 0.0f, acc, 0, 0, 0);
            }
        }
        if (any_odd)
            for (int s = 0; s < n; ++s) {
                const float v = vrow[(size_t)s * p.ld + col];
                if (!(fabsf(v) <= 3.4028235e38f))
#pragma unroll
                    for (int x = 0; x < 16; ++x) {
                        const int t = 32 * mt + 8 * (x >> 2) + 4 * kh + (x & 3);
                        if (t >= s) acc[x] = fmaf(s_A[t * LA + s], v, acc[x]);
                    }
            }
    }
    const bool mine = sl * 32 + r < p.V;
    if (!p.norm_w) {
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const int t = 32 * mt + 8 * (x >> 2) + 4 * kh + (x & 3);
            if (t < n && mine) p.out[(size_t)(m0 + t) * p.ldo + h * p.V + col] = acc[x];
        }
        return;
    }
    // The norm behind the head (its channels are all here): a launch of its own read and wrote the outputs again, 18 us for 8184 tokens of 8 heads
    // beside the 81 of this kernel, which takes 84 with the norm; 333 tokens of 6 heads 4.3 beside 21.9, here 23.4.
    float ss[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) ss[x] = mine ? acc[x] * acc[x] : 0.0f;
#pragma unroll
    for (int d = 16; d > 1; d >>= 1)  // over the 32 columns: a lane keeps half of its tokens with every step
#pragma unroll
        for (int i = 0; i < d / 2; ++i) {
            const float keep = r & d ? ss[d / 2 + i] : ss[i], send = r & d ? ss[i] : ss[d / 2 + i];
            ss[i] = keep + __shfl_xor(send, d, 64);
        }
    ss[0] += __shfl_xor(ss[0], 1, 64);
    float* const s_ss = s_F;         // [token][wave of 32 columns]
    float* const s_inv = s_F + 256;  // [token]
    const int x0 = r >> 1;
    s_ss[(32 * mt + 8 * (x0 >> 2) + 4 * kh + (x0 & 3)) * 4 + (wave >> 1)] = ss[0];
    __syncthreads();
    if (tid < kChunk) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(&s_ss[tid * 4]);
        s_inv[tid] = 1.0f / sqrtf(((v.x + v.y) + (v.z + v.w)) / (float)p.V + p.norm_eps);
    }
    __syncthreads();
    const float w = p.norm_w[col];
    constexpr int PITCH = 128 * 2 + 16;  // bytes of a row of the image
    char* const img = reinterpret_cast<char*>(s_q);
    static_assert(kChunk * PITCH <= sizeof(s_q), "the outputs fit the queries' place");
#pragma unroll
    for (int x = 0; x < 16; ++x) {
        const int t = 32 * mt + 8 * (x >> 2) + 4 * kh + (x & 3);
        const float v = acc[x] * s_inv[t] * w;
        if (p.out16) *reinterpret_cast<bf16_t*>(img + t * PITCH + (sl * 32 + r) * 2) = (bf16_t)cvt_pk_bf16(v, v);
        else if (t < n && mine) p.out[(size_t)(m0 + t) * p.ldo + h * p.V + col] = v;
    }
    if (!p.out16) return;
    __syncthreads();
    const int per = p.V / 8;
    for (int idx = tid; idx < n * per; idx += 512) {
        const int t = idx / per, c = (idx - t * per) * 8;
        *reinterpret_cast<u32x4*>(p.out16 + (size_t)(m0 + t) * p.ldo + h * p.V + c) = *reinterpret_cast<const u32x4*>(img + t * PITCH + c * 2);
    }
}

// One token of every entry (decode steps), HGRN2, and the norm behind the head: a workgroup per (entry, head), four value channels a lane
// (CW lanes a row of the state), the key channels dealt over the rest of the 512 threads.  A step reads and writes each state once, so
// everything is requested at entry: the rows of the state before the gates that scale them.  8 entries, 6 heads of 128 x 128: 6.0 us,
// 8.0 for the token-by-token scan's kernel and 4.0 for the norm's launch behind it.
constexpr int kStepRows = 8;  // rows of the state in flight per thread
template <int CW>
__global__ __launch_bounds__(512) void gated_step_kernel(const float* proj, float* state, size_t slot_stride, const int* ent_start, const int* ent_slot, int ld, int H,
                                                         int D, int V, const float* bias, const float* low, float* out, int ldo, const float* w, float eps) {
    constexpr int GROUPS = 512 / CW;
    __shared__ float s_q[256], s_f[256], s_red[8];
    __shared__ __attribute__((aligned(16))) float s_o[GROUPS][CW * 4 + 4];
    const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, c = tid % CW, r = tid / CW;
    const size_t m = ent_start[e];
    float* S = state + (size_t)ent_slot[e] * slot_stride + (size_t)h * D * V;
    const float* row = proj + m * ld;
    const int HD = H * D, col = min(c * 4, V - 4);
    const bool ok = c * 4 < V;
    f32x4 s[kStepRows];
#pragma unroll
    for (int u = 0; u < kStepRows; ++u) s[u] = *reinterpret_cast<const f32x4*>(S + (size_t)min(r + GROUPS * u, D - 1) * V + col);
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = row[2 * HD + h * V + col + i];
    const int gi = h * D + min(tid, D - 1);
    const float gq = row[gi], gf = row[HD + gi], gl = low[gi], gb = bias[gi], gw = w[min(tid, V - 1)];
    if (tid < D) {
        s_q[tid] = gq / (1.0f + expf(-gq));
        s_f[tid] = gl + (1.0f - gl) / (1.0f + expf(-(gf + gb)));
    }
    __syncthreads();
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i0 = 0; i0 < D; i0 += GROUPS * kStepRows) {
        if (i0 > 0) {
#pragma unroll
            for (int u = 0; u < kStepRows; ++u) s[u] = *reinterpret_cast<const f32x4*>(S + (size_t)min(i0 + r + GROUPS * u, D - 1) * V + col);
        }
#pragma unroll
        for (int u = 0; u < kStepRows; ++u) {
            const int i = i0 + r + GROUPS * u;
            if (i < D && ok) {
                const float f = s_f[i], q = s_q[i];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    s[u][k] = fmaf(f, s[u][k], (1.0f - f) * v[k]);
                    o[k] = fmaf(s[u][k], q, o[k]);
                }
                *reinterpret_cast<f32x4*>(S + (size_t)i * V + col) = s[u];
            }
        }
    }
    *reinterpret_cast<f32x4*>(&s_o[r][c * 4]) = o;
    __syncthreads();
    float a = 0.0f;
    if (tid < V) {
#pragma unroll
        for (int k = 0; k < GROUPS; ++k) a += s_o[k][tid];
    }
    const float ss = wave_allsum(a * a);
    if ((tid & 63) == 0) s_red[tid >> 6] = ss;
    __syncthreads();
    if (tid < V) {
        const float rms = ((s_red[0] + s_red[1]) + (s_red[2] + s_red[3])) + ((s_red[4] + s_red[5]) + (s_red[6] + s_red[7]));
        out[m * ldo + h * V + tid] = a * (1.0f / sqrtf(rms / (float)V + eps)) * gw;
    }
}

}  // namespace

int launch_gated_step(const float* proj, int ld, float* out, int ldo, float* state, size_t slot_stride, const int* ent_start, const int* ent_slot,
                      int n_entries, int H, int D, int V, const float* bias, const float* low, const float* w, float eps, hipStream_t s, bool* taken) {
    *taken = false;
    if (n_entries <= 0 || D > 256 || V < 4 || V > 256 || V % 4 != 0 || slot_stride % 4 != 0 || (reinterpret_cast<uintptr_t>(state) & 15) != 0 || H > 65535)
        return ZG_OK;
    const dim3 grid(n_entries, H);
#define ZG_GSTEP(CW) gated_step_kernel<CW><<<grid, 512, 0, s>>>(proj, state, slot_stride, ent_start, ent_slot, ld, H, D, V, bias, low, out, ldo, w, eps)
    if (V <= 32) ZG_GSTEP(8);
    else if (V <= 64) ZG_GSTEP(16);
    else if (V <= 128) ZG_GSTEP(32);
    else ZG_GSTEP(64);
#undef ZG_GSTEP
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

int launch_gated_chunks(const float* proj, int ld, float* out, int ldo, float* state, size_t slot_stride, const int* ent_start, const int* ent_len,
                        const int* ent_slot, int n_entries, int M, int H, int D, int V, const float* bias, const float* low, float* ws, size_t ws_floats,
                        const GlaGate* gla, hipStream_t s, bool* taken, HeadNorm* norm) {
    *taken = false;
    const int n_chunks = (M + kChunk - 1) / kChunk + n_entries;
    const size_t hf = (size_t)H * D * V;
    if (D > 128 || !ws || ws_floats < (size_t)n_chunks * (hf + (size_t)H * D) || H > 65535) return ZG_OK;
    ScanArgs p;
    p.proj = proj; p.ld = ld; p.out = out; p.ldo = ldo; p.ent_start = ent_start; p.ent_len = ent_len; p.n_entries = n_entries;
    p.H = H; p.D = D; p.V = V; p.bias = bias; p.low = low; p.gla = gla ? *gla : GlaGate();
    p.wsB = ws;
    p.wsA = ws + (size_t)n_chunks * hf;
    if (norm && V <= 128 && (!norm->out16 || (V % 8 == 0 && ldo % 8 == 0 && (reinterpret_cast<uintptr_t>(norm->out16) & 15) == 0))) {  // (a workgroup has whole heads)
        p.norm_w = norm->w; p.norm_eps = norm->eps; p.out16 = norm->out16;
        norm->done = true;
    }
    const dim3 grid(n_chunks, H, (V + 127) / 128);
    for (int phase = 0; phase < 2; ++phase) {
#define ZG_CHUNK(KIND, DP)                                                            \
    do {                                                                              \
        if (phase == 0) gated_chunk_state_kernel<KIND, DP><<<grid, 512, 0, s>>>(p);   \
        else gated_chunk_out_kernel<KIND, DP><<<grid, 512, 0, s>>>(p);                \
    } while (0)
        if (gla && D <= 64) ZG_CHUNK(KIND_GLA, 64);
        else if (gla) ZG_CHUNK(KIND_GLA, 128);
        else if (D <= 64) ZG_CHUNK(KIND_HGRN2, 64);
        else ZG_CHUNK(KIND_HGRN2, 128);
#undef ZG_CHUNK
        ZG_HIP(hipGetLastError());
        if (phase == 0) ZG_TRY(launch_state_carry(state, slot_stride, ent_len, ent_slot, n_entries, H, D, V, p.wsB, p.wsA, D, kChunk, s));
    }
    note_kernel("gated_chunk_out_kernel");
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
