// lm_linear.hip — the linear maps of the layered-model tier: C = act(A B^T) with fp32 activation rows A and bf16 weights B.
//
// Behind one launcher:
//   * steps of up to 8 rows: lm_gemv_at_once_kernel (lm_gemv.hip; one or two rows in whole 16-byte pieces), lm_rows_kernel (lm_rows.hip;
//                      three rows and more, lists of experts), and for what these leave
//   * lm_gemv_kernel   (long rows: lm_gemv_ks_kernel) a wave owns two weight rows, its lanes split K in 16-byte pieces, the
//                      activation rows come straight from the cache hierarchy, sums are fp32 FMAs in both precision modes.
//   * gemm_s4_kernel   (gemm_s4.hip) plain products of prompt portions whose rows are rounded already, where they fill the chip several times.
//   * lm_stream_kernel (lm_stream.hip) the other products of rounded rows, and those of 32-bit mode, whose K is whole steps of 64, experts' among them.
//   * lm_wide_kernel   prompt portions that fill the chip: 128 x 128 or 64 x 64 tiles staged through the LDS.
//   * lm_deep_kernel   short portions: 32-wide tiles with K split over the waves of a workgroup.
//                      Both multiply with v_mfma_f32_32x32x16_bf16: bf16 mode rounds the activations on their way there, 32-bit mode
//                      multiplies their exact three-term bf16 split (the weights are bf16), fp32 accumulation.
//   * lm_gemm_kernel   any alignment, any K: 64 x 64 tiles, one LDS buffer, the fp32 instruction in 32-bit mode.
// All understand the same addressing: a row gather for A, one matrix per grid.z batch (heads), a matrix chosen per batch by
// an index array (the expert of an assignment), and row groups sorted by expert with their offsets in device memory.
#include <stdlib.h>

#include <algorithm>

#include <type_traits>

#include "lm_linear_args.h"
#include "zg_kernels.h"

namespace zg {
namespace lm {

namespace {


// eight consecutive weights of row `w` from column k, zero beyond K
__device__ __forceinline__ void load_w8(const bf16_t* w, int k, int K, bool vec, float out[8]) {
    if (vec && k + 8 <= K) {
        const u32x4 p = *reinterpret_cast<const u32x4*>(w + k);
        out[0] = bf16_lo(p.x); out[1] = bf16_hi(p.x); out[2] = bf16_lo(p.y); out[3] = bf16_hi(p.y);
        out[4] = bf16_lo(p.z); out[5] = bf16_hi(p.z); out[6] = bf16_lo(p.w); out[7] = bf16_hi(p.w);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = (k + i < K) ? __uint_as_float((uint32_t)w[k + i] << 16) : 0.0f;
    }
}

__device__ __forceinline__ f32x4 load_a4(const float* a, int k, int K, bool vec) {
    if (a == nullptr) return f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (vec && k + 4 <= K) return *reinterpret_cast<const f32x4*>(a + k);
    f32x4 r;
    r.x = (k + 0 < K) ? a[k + 0] : 0.0f;
    r.y = (k + 1 < K) ? a[k + 1] : 0.0f;
    r.z = (k + 2 < K) ? a[k + 2] : 0.0f;
    r.w = (k + 3 < K) ? a[k + 3] : 0.0f;
    return r;
}

// ------------------------------------------------------------------------------------------------ few rows
// Rows that enter through the polynomial a N(z) + b N(z^2) + c N(z^3) + e (N divides the row by its root mean square): the statistics
// are sums over the same row, so one pass gathers them beside the products with z, z^2, z^3 and 1, and they meet at the end.
struct PolySums {
    float q1 = 0.0f, q2 = 0.0f, q3 = 0.0f;  // sums of z^2, z^4, z^6
    float d0[4] = {0.0f, 0.0f, 0.0f, 0.0f}, d1[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // the two weight rows with z, z^2, z^3, 1
    __device__ __forceinline__ void add(float z, float w0, float w1) {
        const float q = z * z, c = q * z;
        q1 += q;
        q2 = fmaf(q, q, q2);
        q3 = fmaf(c, c, q3);
        d0[0] = fmaf(z, w0, d0[0]); d1[0] = fmaf(z, w1, d1[0]);
        d0[1] = fmaf(q, w0, d0[1]); d1[1] = fmaf(q, w1, d1[1]);
        d0[2] = fmaf(c, w0, d0[2]); d1[2] = fmaf(c, w1, d1[2]);
        d0[3] += w0; d1[3] += w1;
    }
    __device__ __forceinline__ void add8(const f32x4& a0, const f32x4& a1, const float* w0, const float* w1) {
        add(a0.x, w0[0], w1[0]); add(a0.y, w0[1], w1[1]); add(a0.z, w0[2], w1[2]); add(a0.w, w0[3], w1[3]);
        add(a1.x, w0[4], w1[4]); add(a1.y, w0[5], w1[5]); add(a1.z, w0[6], w1[6]); add(a1.w, w0[7], w1[7]);
    }
    __device__ __forceinline__ void reduce_wave() {
        q1 = wave_allsum(q1);
        q2 = wave_allsum(q2);
        q3 = wave_allsum(q3);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            d0[i] = wave_allsum(d0[i]);
            d1[i] = wave_allsum(d1[i]);
        }
    }
};
__device__ __forceinline__ float poly_value(const LinArgs& p, float q1, float q2, float q3, const float* d) {
    const float K = (float)p.K, eps = p.poly_eps;
    return (p.a_poly[0] / sqrtf(q1 / K + eps) * d[0] + p.a_poly[1] / sqrtf(q2 / K + eps) * d[1]) +
           (p.a_poly[2] / sqrtf(q3 / K + eps) * d[2] + p.a_poly[3] * d[3]);
}

template <int MR, bool POLY = false>
__device__ __forceinline__ void gemv_body(const LinArgs& p, const int z) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = blockIdx.x * 8 + wave * 2;
    if (n0 >= p.N) return;
    if (p.z_group && p.z_group[z] >= p.z_limit) return;
    const bf16_t* B = p.B + (long long)(p.z_group ? p.z_group[z] : z) * p.b_zoff;
    const float* A = p.A + (long long)z * p.a_zoff;
    float* C = p.C + (long long)z * p.c_zoff;
    const float* arow[MR];
    float asc[MR], agate[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        arow[m] = nullptr;
        asc[m] = agate[m] = 1.0f;
        if (m < p.M) {
            const int rid = p.z_group ? z * p.M + m : m;
            const int src = (p.a_rows ? p.a_rows[rid] : rid) / p.a_div;
            arow[m] = A + (long long)src * p.lda;
            if (p.a_glu > 0 && p.glu_scale) asc[m] = p.glu_scale[rid];
            if (p.a_glu > 0 && p.glu_gate_col >= 0) agate[m] = 1.0f / (1.0f + expf(-arow[m][p.glu_gate_col]));
        }
    }
    const bool two = n0 + 1 < p.N;
    const bf16_t* w0 = B + (long long)n0 * p.ldb;
    const bf16_t* w1 = B + (long long)(two ? n0 + 1 : n0) * p.ldb;
    float acc0[MR], acc1[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc0[m] = acc1[m] = 0.0f;
    PolySums ps[POLY ? MR : 1];
    // two K pieces per trip, all four weight vectors requested before the first is used: rows of up to 1024 columns cost one
    // memory round trip
    constexpr int U = MR <= 2 ? 2 : 1;
    for (int k = lane * 8; k < p.K; k += 512 * U) {
        float wa[U][8], wb[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            load_w8(w0, k + 512 * u, p.K, p.b_vec, wa[u]);
            load_w8(w1, k + 512 * u, p.K, p.b_vec, wb[u]);
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            f32x4 av[U][2];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int kk = k + 512 * u;
                f32x4 a0 = load_a4(arow[m], kk, p.K, p.a_vec), a1 = load_a4(arow[m], kk + 4, p.K, p.a_vec);
                if (p.a_glu > 0 && arow[m]) {  // rows [gate | up]: silu(gate) * up
                    const f32x4 u0 = load_a4(arow[m] + p.a_glu, kk, p.K, p.a_vec && p.a_glu % 4 == 0);
                    const f32x4 u1 = load_a4(arow[m] + p.a_glu, kk + 4, p.K, p.a_vec && p.a_glu % 4 == 0);
                    a0.x = glu_on_load(a0.x, u0.x, p, asc[m]) * agate[m]; a0.y = glu_on_load(a0.y, u0.y, p, asc[m]) * agate[m];
                    a0.z = glu_on_load(a0.z, u0.z, p, asc[m]) * agate[m]; a0.w = glu_on_load(a0.w, u0.w, p, asc[m]) * agate[m];
                    a1.x = glu_on_load(a1.x, u1.x, p, asc[m]) * agate[m]; a1.y = glu_on_load(a1.y, u1.y, p, asc[m]) * agate[m];
                    a1.z = glu_on_load(a1.z, u1.z, p, asc[m]) * agate[m]; a1.w = glu_on_load(a1.w, u1.w, p, asc[m]) * agate[m];
                }
                av[u][0] = a0;
                av[u][1] = a1;
            }
            if constexpr (POLY) {
#pragma unroll
                for (int u = 0; u < U; ++u) ps[m].add8(av[u][0], av[u][1], wa[u], wb[u]);
                continue;
            }
            float s0 = acc0[m], s1 = acc1[m];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const f32x4 a0 = av[u][0], a1 = av[u][1];
                s0 = fmaf(a0.x, wa[u][0], s0); s1 = fmaf(a0.x, wb[u][0], s1);
                s0 = fmaf(a0.y, wa[u][1], s0); s1 = fmaf(a0.y, wb[u][1], s1);
                s0 = fmaf(a0.z, wa[u][2], s0); s1 = fmaf(a0.z, wb[u][2], s1);
                s0 = fmaf(a0.w, wa[u][3], s0); s1 = fmaf(a0.w, wb[u][3], s1);
                s0 = fmaf(a1.x, wa[u][4], s0); s1 = fmaf(a1.x, wb[u][4], s1);
                s0 = fmaf(a1.y, wa[u][5], s0); s1 = fmaf(a1.y, wb[u][5], s1);
                s0 = fmaf(a1.z, wa[u][6], s0); s1 = fmaf(a1.z, wb[u][6], s1);
                s0 = fmaf(a1.w, wa[u][7], s0); s1 = fmaf(a1.w, wb[u][7], s1);
            }
            acc0[m] = s0;
            acc1[m] = s1;
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        if constexpr (POLY) {
            ps[m].reduce_wave();
            acc0[m] = poly_value(p, ps[m].q1, ps[m].q2, ps[m].q3, ps[m].d0);
            acc1[m] = poly_value(p, ps[m].q1, ps[m].q2, ps[m].q3, ps[m].d1);
        }
        const float s0 = POLY ? acc0[m] : wave_allsum(acc0[m]), s1 = POLY ? acc1[m] : wave_allsum(acc1[m]);
        if (lane == 0 && m < p.M) {
            C[(long long)m * p.ldc + n0] = finish(s0, n0, p);
            if (two) C[(long long)m * p.ldc + n0 + 1] = finish(s1, n0 + 1, p);
        }
    }
}

template <int MR, bool POLY>
__global__ __launch_bounds__(256) void lm_gemv_kernel(const LinArgs p) {
    gemv_body<MR, POLY>(p, blockIdx.z);
}

// Two products of one-row batches in one launch: batches [0, nz_a) are product a's, the rest product b's (the chosen experts and the
// expert every token uses read the same rows; a decode step saves a dependent launch per product).
__global__ __launch_bounds__(256) void lm_gemv_pair_kernel(const LinArgs a, const LinArgs b, int nz_a) {
    if ((int)blockIdx.z < nz_a) gemv_body<1>(a, blockIdx.z);
    else gemv_body<1>(b, blockIdx.z - nz_a);
}

// The same for long rows (K >= 1536; at 1024 columns half the lanes of a quarter idle and it measured 6 % slower): a workgroup owns two weight rows and its four waves split K into quarters, so a matrix of
// a few MB is requested whole in one go by thousands of waves instead of trip by trip by a few hundred (a 1600 x 1600 matrix:
// 800 workgroups, every 16-byte piece in flight at once); the quarter sums meet in the LDS.  The summation order of an output
// depends on K alone.
template <int MR, bool POLY>
__global__ __launch_bounds__(256) void lm_gemv_ks_kernel(const LinArgs p) {
    __shared__ float s_part[4][MR][POLY ? 11 : 2];
    const int z = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = blockIdx.x * 2;
    if (p.z_group && p.z_group[z] >= p.z_limit) return;
    const bf16_t* B = p.B + (long long)(p.z_group ? p.z_group[z] : z) * p.b_zoff;
    const float* A = p.A + (long long)z * p.a_zoff;
    float* C = p.C + (long long)z * p.c_zoff;
    const float* arow[MR];
    float asc[MR], agate[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        arow[m] = nullptr;
        asc[m] = agate[m] = 1.0f;
        if (m < p.M) {
            const int rid = p.z_group ? z * p.M + m : m;
            const int src = (p.a_rows ? p.a_rows[rid] : rid) / p.a_div;
            arow[m] = A + (long long)src * p.lda;
            if (p.a_glu > 0 && p.glu_scale) asc[m] = p.glu_scale[rid];
            if (p.a_glu > 0 && p.glu_gate_col >= 0) agate[m] = 1.0f / (1.0f + expf(-arow[m][p.glu_gate_col]));
        }
    }
    const bf16_t* w0 = B + (long long)n0 * p.ldb;
    const bf16_t* w1 = B + (long long)min(n0 + 1, p.N - 1) * p.ldb;
    float acc0[MR], acc1[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc0[m] = acc1[m] = 0.0f;
    PolySums ps[POLY ? MR : 1];
    const int kq = (((p.K + 3) / 4) + 7) & ~7;  // a wave's quarter of K, a multiple of 8
    const int k_lo = wave * kq, k_hi = min(p.K, k_lo + kq);
    constexpr int U = 2;
    for (int k = k_lo + lane * 8; k < k_hi; k += 512 * U) {
        float wa[U][8], wb[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            load_w8(w0, k + 512 * u, k_hi, p.b_vec, wa[u]);
            load_w8(w1, k + 512 * u, k_hi, p.b_vec, wb[u]);
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float s0 = acc0[m], s1 = acc1[m];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int kk = k + 512 * u;
                f32x4 a0 = load_a4(arow[m], kk, k_hi, p.a_vec), a1 = load_a4(arow[m], kk + 4, k_hi, p.a_vec);
                if (p.a_glu > 0 && arow[m]) {  // rows [gate | up]: silu(gate) * up
                    const f32x4 u0 = load_a4(arow[m] + p.a_glu, kk, k_hi, p.a_vec && p.a_glu % 4 == 0);
                    const f32x4 u1 = load_a4(arow[m] + p.a_glu, kk + 4, k_hi, p.a_vec && p.a_glu % 4 == 0);
                    a0.x = glu_on_load(a0.x, u0.x, p, asc[m]) * agate[m]; a0.y = glu_on_load(a0.y, u0.y, p, asc[m]) * agate[m];
                    a0.z = glu_on_load(a0.z, u0.z, p, asc[m]) * agate[m]; a0.w = glu_on_load(a0.w, u0.w, p, asc[m]) * agate[m];
                    a1.x = glu_on_load(a1.x, u1.x, p, asc[m]) * agate[m]; a1.y = glu_on_load(a1.y, u1.y, p, asc[m]) * agate[m];
                    a1.z = glu_on_load(a1.z, u1.z, p, asc[m]) * agate[m]; a1.w = glu_on_load(a1.w, u1.w, p, asc[m]) * agate[m];
                }
                if constexpr (POLY) {
                    ps[m].add8(a0, a1, wa[u], wb[u]);
                    continue;
                }
                s0 = fmaf(a0.x, wa[u][0], s0); s1 = fmaf(a0.x, wb[u][0], s1);
                s0 = fmaf(a0.y, wa[u][1], s0); s1 = fmaf(a0.y, wb[u][1], s1);
                s0 = fmaf(a0.z, wa[u][2], s0); s1 = fmaf(a0.z, wb[u][2], s1);
                s0 = fmaf(a0.w, wa[u][3], s0); s1 = fmaf(a0.w, wb[u][3], s1);
                s0 = fmaf(a1.x, wa[u][4], s0); s1 = fmaf(a1.x, wb[u][4], s1);
                s0 = fmaf(a1.y, wa[u][5], s0); s1 = fmaf(a1.y, wb[u][5], s1);
                s0 = fmaf(a1.z, wa[u][6], s0); s1 = fmaf(a1.z, wb[u][6], s1);
                s0 = fmaf(a1.w, wa[u][7], s0); s1 = fmaf(a1.w, wb[u][7], s1);
            }
            acc0[m] = s0;
            acc1[m] = s1;
        }
    }
    if constexpr (POLY) {
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            ps[m].reduce_wave();
            if (lane == 0) {
                float* o = s_part[wave][m];
                o[0] = ps[m].q1; o[1] = ps[m].q2; o[2] = ps[m].q3;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[3 + i] = ps[m].d0[i];
                    o[7 + i] = ps[m].d1[i];
                }
            }
        }
        __syncthreads();
        if (threadIdx.x < MR * 2) {
            const int m = threadIdx.x >> 1, c = threadIdx.x & 1;
            auto sum4 = [&](int i) { return (s_part[0][m][i] + s_part[1][m][i]) + (s_part[2][m][i] + s_part[3][m][i]); };
            const float d[4] = {sum4(3 + 4 * c), sum4(4 + 4 * c), sum4(5 + 4 * c), sum4(6 + 4 * c)};
            if (m < p.M && n0 + c < p.N) C[(long long)m * p.ldc + n0 + c] = finish(poly_value(p, sum4(0), sum4(1), sum4(2), d), n0 + c, p);
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const float t0 = wave_allsum(acc0[m]), t1 = wave_allsum(acc1[m]);
        if (lane == 0) {
            s_part[wave][m][0] = t0;
            s_part[wave][m][1] = t1;
        }
    }
    __syncthreads();
    if (threadIdx.x < MR * 2) {
        const int m = threadIdx.x >> 1, c = threadIdx.x & 1;
        if (m < p.M && n0 + c < p.N)
            C[(long long)m * p.ldc + n0 + c] = finish((s_part[0][m][c] + s_part[1][m][c]) + (s_part[2][m][c] + s_part[3][m][c]), n0 + c, p);
    }
}

// ------------------------------------------------------------------------------------------------ matrix cores
// Both kernels below multiply bf16 tiles with v_mfma_f32_32x32x16_bf16 and accumulate in fp32.  NP = 1: the activations are rounded
// to bf16 on their way to the matrix cores.  NP = 3 (32-bit mode): an activation is the exact sum of three bf16 terms and the
// weights are bf16 as they are, so three products give the fp32 product exactly, at 5 times the rate of the fp32 instruction.
// Both take 16-byte pieces: aligned operands, K a multiple of 8.

// f(step<0>()) ... f(step<N - 1>()): indices known to the compiler, for rings kept in registers
template <int I>
using step = std::integral_constant<int, I>;
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unroll(F&& f) {
    if constexpr (I < N) {
        f(step<I>());
        unroll<N, I + 1>(f);
    }
}

// Eight consecutive activations in flight: fp32 as they are, or already rounded to bf16 by the kernel that wrote them.
template <typename AT>
struct Act8;
template <>
struct Act8<float> {
    f32x4 a, b;
    __device__ __forceinline__ void load(const float* row, int k) {
        a = *reinterpret_cast<const f32x4*>(row + k);
        b = *reinterpret_cast<const f32x4*>(row + k + 4);
    }
    __device__ __forceinline__ void clear() { a = b = f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
    template <int NP>
    __device__ __forceinline__ Planes8<NP> planes() const { return to_planes<NP>(a, b); }
};
__device__ __forceinline__ u32x4 load_b8(const bf16_t* row, int k) { return *reinterpret_cast<const u32x4*>(row + k); }
template <>
struct Act8<bf16_t> {
    u32x4 v;
    __device__ __forceinline__ void load(const bf16_t* row, int k) { v = load_b8(row, k); }
    __device__ __forceinline__ void clear() { v = u32x4{0u, 0u, 0u, 0u}; }
    template <int NP>
    __device__ __forceinline__ Planes8<NP> planes() const {
        static_assert(NP == 1, "rounded activations have one term");
        return Planes8<1>{{v}};
    }
};

template <typename AT>
__device__ __forceinline__ const AT* a_row(const LinArgs& p, int m) {
    const AT* A;
    if constexpr (std::is_same<AT, float>::value) A = p.A;
    else A = p.A16;
    return A + (long long)blockIdx.z * p.a_zoff + (long long)((p.a_rows ? p.a_rows[m] : m) / p.a_div) * p.lda;
}
// output (m, n), finished
__device__ __forceinline__ void put(const LinArgs& p, int m, int n, float v) {
    const long long at = (long long)blockIdx.z * p.c_zoff + (long long)m * p.ldc + n;
    v = finish(v, n, p);
    if (p.C) p.C[at] = v;
    if (p.C16) p.C16[at] = (bf16_t)cvt_pk_bf16(v, v);
}

// Three terms: a weight that is infinite meets terms that are zero, and the sum is NaN where an fp32 sum is an infinity.  The outputs
// (bit b of `which`: at(b)) that came out NaN again, as plain fp32 sums (one that has become NaN ends at once).
template <typename F>
__device__ __forceinline__ void again(const LinArgs& p, const TileAt& t, unsigned which, F&& at) {
#pragma unroll 1
    for (; which != 0; which &= which - 1) {
        int m, n;
        at(__builtin_ctz(which), m, n);
        const float* a = a_row<float>(p, m);
        const bf16_t* b = t.B + (long long)n * p.ldb;
        float s = 0.0f;
#pragma unroll 1
        for (int k = 0; k < p.K && s == s; k += 8) {
            Act8<float> x;
            x.load(a, k);
            const u32x4 w = load_b8(b, k);
#pragma unroll
            for (int i = 0; i < 4; ++i) s = fmaf(i < 2 ? x.a[2 * i + 1] : x.b[2 * i - 3], bf16_hi(w[i]), fmaf(i < 2 ? x.a[2 * i] : x.b[2 * i - 4], bf16_lo(w[i]), s));
        }
        put(p, m, n, s);
    }
}

// What bounds it: the bytes a compute unit takes in (31 to 37 B per clock beside matrix products) and, per K step, one LDS round trip.
// 8184 x 3072 x 1024 takes 106 us (490 TFLOP/s; before, with one LDS buffer and 64 x 64 tiles, 176), 8184 x 1024 x 4096 107 us
// (640 TFLOP/s; 274), 333 x 768 x 3072 17.5 us (95): there the reads of a step's fragments, which the compiler had paired with a
// wait for each product, and loads under a condition, which it waited for at every step, were three quarters of the time.
// Enough rows to fill the chip: 64 TM x 64 TN tiles, four waves in a 2 x 2 arrangement of TM x TN MFMA tiles each.  Operands pass
// through two LDS buffers (rows of BK elements, their 16-byte chunks swizzled by the row so that the fragment reads of eight
// consecutive rows hit different banks); the registers hold the K step behind the one in the LDS, so a load has a whole step of
// MFMAs to arrive, and there is one barrier per step.
template <typename AT, int NP, int TM, int TN, int AHEAD>
__global__ __launch_bounds__(256, 2) void lm_wide_kernel(const LinArgs p) {
    constexpr int BM = 64 * TM, BN = 64 * TN, BK = NP == 1 ? 64 : 32, CH = BK / 8;
    constexpr int AC = BM * CH / 256, BC = BN * CH / 256;
    __shared__ __attribute__((aligned(16))) bf16_t As[2][NP][BM * BK];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[2][BN * BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wy = wave >> 1, wx = wave & 1;
    TileAt t;
    if (!find_tile(p, p.N, BM, BN, t)) return;
    auto swz = [](int row) { return CH == 8 ? row & 7 : (row >> 1) & 3; };  // (row & 31 decides)

    const AT* a_src[AC];
    const bf16_t* b_src[BC];
    int a_lds[AC], b_lds[BC];
    const int kc = (tid % CH) * 8;  // this thread's chunk of every row it fetches
#pragma unroll
    for (int j = 0; j < AC; ++j) {
        const int row = (tid + 256 * j) / CH;
        a_src[j] = a_row<AT>(p, min(t.m0 + row, t.m_end - 1));  // (rows beyond the edge: some valid row, never stored)
        a_lds[j] = row * BK + (((tid % CH) ^ swz(row)) * 8);
    }
#pragma unroll
    for (int j = 0; j < BC; ++j) {
        const int row = (tid + 256 * j) / CH;
        b_src[j] = t.B + (long long)min(t.n0 + row, p.N - 1) * p.ldb;
        b_lds[j] = row * BK + (((tid % CH) ^ swz(row)) * 8);
    }
    Act8<AT> a_ring[AHEAD][AC];
    u32x4 b_ring[AHEAD][BC];
    auto fetch = [&](auto slot, int k0) {
        const int k = min(k0 + kc, p.K - 8);  // (columns beyond K: valid ones, zeroed when stashed)
#pragma unroll
        for (int j = 0; j < AC; ++j) a_ring[slot][j].load(a_src[j], k);
#pragma unroll
        for (int j = 0; j < BC; ++j) b_ring[slot][j] = load_b8(b_src[j], k);
    };
    const int n_steps = (p.K + BK - 1) / BK;
    auto stash = [&](auto slot, int buf, int s) {
        auto& a_reg = a_ring[slot];
        auto& b_reg = b_ring[slot];
        if (s == n_steps - 1 && s * BK + kc >= p.K) {  // chunks beyond K
#pragma unroll
            for (int j = 0; j < AC; ++j) a_reg[j].clear();
#pragma unroll
            for (int j = 0; j < BC; ++j) b_reg[j] = u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int j = 0; j < AC; ++j) {
            const Planes8<NP> pl = a_reg[j].template planes<NP>();
#pragma unroll
            for (int q = 0; q < NP; ++q) *reinterpret_cast<u32x4*>(&As[buf][q][a_lds[j]]) = pl.v[q];
        }
#pragma unroll
        for (int j = 0; j < BC; ++j) *reinterpret_cast<u32x4*>(&Bs[buf][b_lds[j]]) = b_reg[j];
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // The fragments of a step: all requested before the first product, so that the LDS latency is paid once per step.
    const int fr = lane & 31, kh = lane >> 5;
    int a_at[TM], b_at[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_at[i] = ((wy * TM + i) * 32 + fr) * BK;
#pragma unroll
    for (int j = 0; j < TN; ++j) b_at[j] = ((wx * TN + j) * 32 + fr) * BK;
    const int fswz = swz(fr);  // (32 rows apart the swizzle repeats)
    u32x4 af[CH / 2][NP][TM], bf[CH / 2][TN];
    auto read = [&](int cur) {
#pragma unroll
        for (int kk = 0; kk < CH / 2; ++kk) {
            const int c = ((2 * kk + kh) ^ fswz) * 8;
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[kk][j] = *reinterpret_cast<const u32x4*>(&Bs[cur][b_at[j] + c]);
#pragma unroll
            for (int q = NP - 1; q >= 0; --q)
#pragma unroll
                for (int i = 0; i < TM; ++i) af[kk][q][i] = *reinterpret_cast<const u32x4*>(&As[cur][q][a_at[i] + c]);
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
            for (int q = NP - 1; q >= 0; --q)  // the smallest terms first
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[kk][q][i]), __builtin_bit_cast(bf16x8, bf[kk][j]),
                                                                            acc[i][j], 0, 0, 0);
    };
    // Step s is fetched AHEAD steps before it is stashed, and stashed while the step in front of it is multiplied.  Fetches and stashes
    // are unconditional (beyond the last step they repeat valid addresses and nobody reads what they leave): a fetch under a
    // condition would make the compiler wait for every load at every stash.
    unroll<AHEAD>([&](auto i) { fetch(i, i * BK); });
    stash(step<0>(), 0, 0);
    fetch(step<0>(), AHEAD * BK);
    __syncthreads();
    int cur = 0, s = 0;
    auto body = [&](auto i) {
        constexpr int nx = (decltype(i)::value + 1) % AHEAD;
        read(cur);
        stash(step<nx>(), cur ^ 1, s + 1);
        fetch(step<nx>(), (s + 1 + AHEAD) * BK);
        multiply();
        // order: the fragment reads, then between the products what the next steps need
        constexpr int products = CH / 2 * NP * TM * TN;
        __builtin_amdgcn_sched_group_barrier(0x100, CH / 2 * (NP * TM + TN), 0);
#pragma unroll
        for (int x = 0; x < products; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, (AC * NP + BC + products - 1) / products, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, (AC * 2 + BC + products - 1) / products, 0);
        }
        cur ^= 1;
        ++s;
        __syncthreads();
    };
    for (int g = n_steps / AHEAD; g > 0; --g) unroll<AHEAD>(body);
    if constexpr (AHEAD > 1)
        unroll<AHEAD - 1>([&](auto i) {
            if (s < n_steps) body(i);
        });

    // accumulator element e of a 32 x 32 tile: row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
    auto row_of = [&](int i, int e) { return t.m0 + (wy * TM + i) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); };
    auto column_of = [&](int j) { return t.n0 + (wx * TN + j) * 32 + (lane & 31); };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = column_of(j);
            if (n >= p.N) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = row_of(i, e);
                if (m < t.m_end) put(p, m, n, acc[i][j][e]);
            }
        }
    if constexpr (NP > 1) {
        static_assert(TM * TN <= 2, "an output, a bit");
        f32x16 all = acc[0][0];  // (NaN if one of them is)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = i == 0 ? 1 : 0; j < TN; ++j) all += acc[i][j];
        const float sum = (((all[0] + all[1]) + (all[2] + all[3])) + ((all[4] + all[5]) + (all[6] + all[7]))) +
                          (((all[8] + all[9]) + (all[10] + all[11])) + ((all[12] + all[13]) + (all[14] + all[15])));
        if (__builtin_expect(sum != sum, 0)) {
            unsigned which = 0;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        if (acc[i][j][e] != acc[i][j][e] && row_of(i, e) < t.m_end && column_of(j) < p.N) which |= 1u << ((i * TN + j) * 16 + e);
            again(p, t, which, [&](int b, int& m, int& n) {
                m = row_of((b >> 4) / TN, b & 15);
                n = column_of((b >> 4) % TN);
            });
        }
    }
}

// Too few tiles to fill the chip (portions of some hundred rows): 32 TM x 32 TN tiles, the four waves of a workgroup split K and meet
// in the LDS.  Nothing is staged: a lane loads its own fragments (16 consecutive k of a row, both halves of a wave the whole
// 128-byte line), no wave waits for another before the end, and a tile's time is a quarter of its K.  Bound by latency: 37 x 2304 x
// 768 takes 6.5 us (15.9 before); in 32-bit mode 333 x 768 x 768 9.5 us (31.6 with the fp32 instruction).
template <typename AT, int NP, int TM, int TN, int AHEAD>
__global__ __launch_bounds__(256, 2) void lm_deep_kernel(const LinArgs p) {
    constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32;
    __shared__ float part[4][TM * TN * 16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, kh = lane >> 5;
    TileAt t;
    if (!find_tile(p, p.N, BM, BN, t)) return;
    const AT* a_src[TM];
    const bf16_t* b_src[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_src[i] = a_row<AT>(p, min(t.m0 + 32 * i + r, t.m_end - 1));
#pragma unroll
    for (int j = 0; j < TN; ++j) b_src[j] = t.B + (long long)min(t.n0 + 32 * j + r, p.N - 1) * p.ldb;
    const int kq = ((p.K + 4 * BK - 1) / (4 * BK)) * BK;
    const int k_lo = wave * kq, k_hi = min(p.K, k_lo + kq);

    Act8<AT> a_reg[AHEAD][TM][2];
    u32x4 b_reg[AHEAD][TN][2];
    auto fetch = [&](auto s, int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int kw = k0 + 16 * kh + 8 * h, k = min(kw, p.K - 8);
#pragma unroll
            for (int i = 0; i < TM; ++i) a_reg[s][i][h].load(a_src[i], k);
#pragma unroll
            for (int j = 0; j < TN; ++j) b_reg[s][j][h] = load_b8(b_src[j], k);
        }
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    auto multiply = [&](auto s, int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = k0 + 16 * kh + 8 * h < p.K;  // (beyond K the clamped load brought columns that were there before)
            bf16x8 bf[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[j] = __builtin_bit_cast(bf16x8, in ? b_reg[s][j][h] : u32x4{0u, 0u, 0u, 0u});
            Planes8<NP> pl[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                Act8<AT> a = a_reg[s][i][h];
                if (!in) a.clear();
                pl[i] = a.template planes<NP>();
            }
#pragma unroll
            for (int q = NP - 1; q >= 0; --q)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, pl[i].v[q]), bf[j], acc[i][j], 0, 0, 0);
        }
    };
    unroll<AHEAD>([&](auto i) {
        if (k_lo + i * BK < k_hi) fetch(i, k_lo + i * BK);
    });
    for (int k0 = k_lo; k0 < k_hi; k0 += AHEAD * BK)
        unroll<AHEAD>([&](auto i) {
            const int k = k0 + i * BK;
            if (k < k_hi) {
                multiply(i, k);
                if (k + AHEAD * BK < k_hi) fetch(i, k + AHEAD * BK);
            }
        });
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) part[wave][(i * TN + j) * 16 + e][lane] = acc[i][j][e];
    __syncthreads();
    constexpr int SHARE = TM * TN * 4;  // accumulator elements this wave sums and stores
    auto place = [&](int x, int& m, int& n) {
        const int el = wave * SHARE + x, e = el & 15, ij = el >> 4, i = ij / TN, j = ij % TN;
        n = t.n0 + 32 * j + r;
        m = t.m0 + 32 * i + 8 * (e >> 2) + 4 * kh + (e & 3);
    };
    float all = 0.0f;  // (NaN if one of them is)
    auto sum = [&](int x) {
        const int el = wave * SHARE + x;
        return (part[0][el][lane] + part[1][el][lane]) + (part[2][el][lane] + part[3][el][lane]);
    };
#pragma unroll
    for (int x = 0; x < SHARE; ++x) {
        const float v = sum(x);
        int m, n;
        place(x, m, n);
        if (n < p.N && m < t.m_end) put(p, m, n, v);
        if (NP > 1) all += v;
    }
    if (NP > 1 && __builtin_expect(all != all, 0)) {
        unsigned which = 0;
#pragma unroll 1
        for (int x = 0; x < SHARE; ++x) {
            const float v = sum(x);
            int m, n;
            place(x, m, n);
            if (v != v && n < p.N && m < t.m_end) which |= 1u << x;
        }
        again(p, t, which, place);
    }
}

template <bool F32>
struct Tile {
    static constexpr int BK = F32 ? 16 : 32;
    static constexpr int LDS_K = F32 ? 17 : 40;  // row stride in elements: conflict-free fragment reads
    typedef typename std::conditional<F32, float, bf16_t>::type elem;
};

// Operands that 16-byte loads cannot take (odd leading dimensions, K no multiple of 8): 64 x 64 tiles, one buffer, a value at a time.
template <bool F32>
__global__ __launch_bounds__(256) void lm_gemm_kernel(const LinArgs p) {
    typedef Tile<F32> T;
    typedef typename T::elem elem;
    constexpr int WT = 1, BM = 64 * WT, BN = 64 * WT, BK = T::BK, LK = T::LDS_K;
    __shared__ __attribute__((aligned(16))) elem As[BM * LK];
    __shared__ __attribute__((aligned(16))) elem Bs[BN * LK];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wy = wave >> 1, wx = wave & 1;
    const int z = blockIdx.z;
    const bf16_t* B = p.B;
    int m0, m_end;
    if (p.grp_off) {  // find the row group this tile belongs to
        int tile = blockIdx.y, e = 0, lo = 0, hi = 0;
        for (; e < p.n_groups; ++e) {
            lo = p.grp_off[e];
            hi = p.grp_off[e + 1];
            const int nt = (hi - lo + BM - 1) / BM;
            if (tile < nt) break;
            tile -= nt;
        }
        if (e >= p.n_groups) return;
        m0 = lo + tile * BM;
        m_end = hi;
        B += (long long)e * p.b_zoff;
    } else {
        m0 = blockIdx.y * BM;
        m_end = p.M;
        B += (long long)(p.z_group ? p.z_group[z] : z) * p.b_zoff;
    }
    const float* A = p.A + (long long)z * p.a_zoff;
    float* C = p.C + (long long)z * p.c_zoff;
    const int n0 = blockIdx.x * BN;

    // global -> register assignment of this thread (fixed over the K loop)
    constexpr int A_VEC_PER_ROW = BK / 4;                 // float4 per A row of the tile
    constexpr int A_LOADS = BM * A_VEC_PER_ROW / 256;     // per thread
    constexpr int B_VEC_PER_ROW = BK / 8;                 // 8 bf16 per vector
    constexpr int B_LOADS = (BN * B_VEC_PER_ROW + 255) / 256;
    const float* a_src[A_LOADS];
    int a_r[A_LOADS], a_k[A_LOADS];
#pragma unroll
    for (int j = 0; j < A_LOADS; ++j) {
        const int v = tid + 256 * j;
        a_r[j] = v / A_VEC_PER_ROW;
        a_k[j] = (v % A_VEC_PER_ROW) * 4;
        const int m = m0 + a_r[j];
        a_src[j] = nullptr;
        if (m < m_end) {
            const int rid = p.z_group ? z * p.M + m : m;
            const int src = (p.a_rows ? p.a_rows[rid] : rid) / p.a_div;
            a_src[j] = A + (long long)src * p.lda;
        }
    }
    const bf16_t* b_src[B_LOADS];
    int b_r[B_LOADS], b_k[B_LOADS];
#pragma unroll
    for (int j = 0; j < B_LOADS; ++j) {
        const int v = tid + 256 * j;
        b_r[j] = v / B_VEC_PER_ROW;
        b_k[j] = (v % B_VEC_PER_ROW) * 8;
        const int n = n0 + b_r[j];
        b_src[j] = (b_r[j] < BN && n < p.N) ? B + (long long)n * p.ldb : nullptr;
    }

    f32x16 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    f32x4 a_reg[A_LOADS];
    float b_reg[B_LOADS][8];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) a_reg[j] = load_a4(a_src[j], k0 + a_k[j], p.K, p.a_vec);
#pragma unroll
        for (int j = 0; j < B_LOADS; ++j) {
            if (b_src[j]) {
                load_w8(b_src[j], k0 + b_k[j], p.K, p.b_vec, b_reg[j]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) b_reg[j][i] = 0.0f;
            }
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) {
            elem* d = &As[a_r[j] * LK + a_k[j]];
            if constexpr (F32) {
                d[0] = a_reg[j].x; d[1] = a_reg[j].y; d[2] = a_reg[j].z; d[3] = a_reg[j].w;
            } else {
                u32x2 pk;
                pk.x = cvt_pk_bf16(a_reg[j].x, a_reg[j].y);
                pk.y = cvt_pk_bf16(a_reg[j].z, a_reg[j].w);
                *reinterpret_cast<u32x2*>(d) = pk;
            }
        }
#pragma unroll
        for (int j = 0; j < B_LOADS; ++j) {
            if (b_r[j] < BN) {
                elem* d = &Bs[b_r[j] * LK + b_k[j]];
                if constexpr (F32) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) d[i] = b_reg[j][i];
                } else {
                    u32x4 pk;  // the values are bf16 already: the conversion is exact
                    pk.x = cvt_pk_bf16(b_reg[j][0], b_reg[j][1]);
                    pk.y = cvt_pk_bf16(b_reg[j][2], b_reg[j][3]);
                    pk.z = cvt_pk_bf16(b_reg[j][4], b_reg[j][5]);
                    pk.w = cvt_pk_bf16(b_reg[j][6], b_reg[j][7]);
                    *reinterpret_cast<u32x4*>(d) = pk;
                }
            }
        }
    };

    fetch(0);
    for (int k0 = 0; k0 < p.K; k0 += BK) {
        __syncthreads();  // the previous step's fragment reads are done
        stash();
        __syncthreads();
        if (k0 + BK < p.K) fetch(k0 + BK);  // in flight beside the MFMAs
        const int r = lane & 31, kh = lane >> 5;
        if constexpr (F32) {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 2) {
                float af[WT], bf[WT];
#pragma unroll
                for (int i = 0; i < WT; ++i) af[i] = As[((wy * WT + i) * 32 + r) * LK + kk + kh];
#pragma unroll
                for (int j = 0; j < WT; ++j) bf[j] = Bs[((wx * WT + j) * 32 + r) * LK + kk + kh];
#pragma unroll
                for (int i = 0; i < WT; ++i)
#pragma unroll
                    for (int j = 0; j < WT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], acc[i][j], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 16) {
                bf16x8 af[WT], bf[WT];
#pragma unroll
                for (int i = 0; i < WT; ++i)
                    af[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&As[((wy * WT + i) * 32 + r) * LK + kk + kh * 8]));
#pragma unroll
                for (int j = 0; j < WT; ++j)
                    bf[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&Bs[((wx * WT + j) * 32 + r) * LK + kk + kh * 8]));
#pragma unroll
                for (int i = 0; i < WT; ++i)
#pragma unroll
                    for (int j = 0; j < WT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
            }
        }
    }

    // accumulator element e of a 32 x 32 tile: row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            const int n = n0 + (wx * WT + j) * 32 + (lane & 31);
            if (n >= p.N) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + (wy * WT + i) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (m < m_end) C[(long long)m * p.ldc + n] = finish(acc[i][j][e], n, p);
            }
        }
}

}  // namespace

namespace {
// Plain products of rounded rows with enough tiles of 256 x 192 go to the persistent kernel of the large-batch Linears (gemm_s4.hip), whose
// hand-scheduled four waves read the LDS less for every product: 8184 x 3072 x 1024 67 against 78 us (lm_stream.hip); 8184 x 4096 x 1024 with max(., 0)^2
// and a rounded result 68 against 85; 8184 x 1536 x 384 20.5 against 23.6.  Its time goes by rounds of 256 tiles, each what 640 tiles of 128 x 128
// cost there: 8184 x 1024 x 1024 (512 of those) 29.1 against 25.3, 8184 x 672 x 1024 25.7 against 21.9, 2048 x 3072 x 768 23.7 against 19.5.
// Products that kernel cannot take (columns in no whole pieces of eight) come here from 112 tiles on: 1791 x 3072 x 768 23.2 against 24.5 on the
// staged tiles.
bool takes_persistent(const Linear& L) {
    const char* form = getenv("ZGPT2_LM_GEMM_TILE");  // test hook: 256 = here at any number of tiles, another = never
    const long long tiles = (long long)((L.M + 255) / 256) * ((L.N + 191) / 192), fine = (long long)((L.M + 127) / 128) * ((L.N + 127) / 128);
    const bool pays = form ? atoi(form) == 256 : getenv("ZGPT2_LM_STREAM") ? false : stream_fits(L, false) ? fine >= 640 * ((tiles + 255) / 256) : tiles >= 112;
    GemmPlanes pl{};
    pl.lda = L.lda;
    pl.ldb = L.ldb;
    pl.kpp = L.K / 64;
    pl.npairs = 1;
    const bool one_result = (L.C != nullptr) != (L.C16 != nullptr);
    return !L.grp_off && !L.z_group && L.nz == 1 && !L.a_rows && L.a_div == 1 && (L.act == ACT_NONE || L.act == ACT_RELU2) && one_result && L.K >= 128 && L.K % 64 == 0 && L.lda % 8 == 0 &&
           L.ldb % 8 == 0 && L.lda >= L.K && L.ldc >= L.N && (L.C || (L.N % 8 == 0 && L.ldc % 8 == 0)) && gemm_s4_args_ok(pl, L.ldc) &&
           ((reinterpret_cast<uintptr_t>(L.A16) | reinterpret_cast<uintptr_t>(L.B) | reinterpret_cast<uintptr_t>(L.C) | reinterpret_cast<uintptr_t>(L.C16)) & 15) == 0 &&
           (size_t)L.M * L.ldc * 4 < ((size_t)1 << 32) && (size_t)L.N * L.ldb < (1u << 30) && (size_t)L.M * L.lda < (1u << 30) && pays;
}
bool takes_k_split(const Linear& L) { return L.K >= 1536 && L.M <= 2 && L.nz <= 4; }
}  // namespace

int launch_linear_pair(const Linear& A, const Linear& B, bool f32, hipStream_t s) {
    bool taken = false;
    if (getenv("ZGPT2_LM_NO_ROWS") == nullptr) ZG_TRY(launch_rows(A, &B, s, &taken));
    if (taken) return ZG_OK;
    ZG_TRY(launch_gemv_at_once(A, &B, nullptr, s, &taken));
    if (taken) return ZG_OK;
    const bool one_launch = A.M == 1 && B.M == 1 && A.nz >= 1 && B.nz >= 1 && A.N > 0 && B.N > 0 && !A.grp_off && !B.grp_off && !takes_k_split(A) &&
                            !takes_k_split(B) && A.K > 0 && B.K > 0 && A.A && A.B && A.C && B.A && B.B && B.C && A.a_div >= 1 && B.a_div >= 1 &&
                            A.nz + B.nz <= 65535;
    if (!one_launch) {
        ZG_TRY(launch_linear(A, f32, s));
        return launch_linear(B, f32, s);
    }
    const dim3 grid((std::max(A.N, B.N) + 7) / 8, 1, A.nz + B.nz);
    lm_gemv_pair_kernel<<<grid, 256, 0, s>>>(make_args(A), make_args(B), A.nz);
    note_kernel("lm_gemv_pair_kernel");
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}


namespace {
template <typename AT, int NP>
int launch_tiles(const Linear& L, const LinArgs& p, hipStream_t s) {
    auto tiles = [&](int bm, int bn) { return (long long)((L.N + bn - 1) / bn) * ((L.M + bm - 1) / bm + (L.grp_off ? L.n_groups : 0)); };
    int force = 0;  // 128, 64 or 32: that form at any size (tests run small ragged shapes through all of them)
    if (const char* e = getenv("ZGPT2_LM_GEMM_TILE")) force = atoi(e) == 256 ? 0 : atoi(e);
    auto grid = [&](int bm, int bn) { return dim3((unsigned)tiles(bm, bn), 1, L.nz); };
    ZG_REQUIRE(tiles(32, 32) < (1LL << 31) && L.nz <= 65535, ZG_ERR_UNSUPPORTED, "linear: %d rows in %d batches exceed the grid", L.M, L.nz);
    // Which form (us per launch, both sides measured on an MI355X):
    //   * 320 tiles of 128 x 128 and more fill the chip: 8184 x 1024 x 1024 35.6 against 44.4 with 64 x 64 tiles, 1791 x 3072 x 768 (336
    //     tiles) 28.0 against 29.3; below, the smaller tiles do: 1791 x 768 x 1536 (84 tiles) 18.1 against 28.2.
    //   * up to 256 tiles of 32 x 32 a compute unit has one of them at most: 37 x 2304 x 768 6.5 against 7.5 with 64 x 64 tiles; with
    //     more, their rows are fetched too often: 333 x 2304 x 768 (792) 19.3 against 8.3.
    //   * three terms are bound by their products rather than by the staging: 333 x 768 x 768 9.5 in 32 x 64 tiles with K split
    //     against 14.4 staged, 333 x 2304 x 768 (396 tiles) 15.2 against 15.7; from there on staged 64 x 128 tiles:
    //     333 x 3072 x 768 18.3 against 22.2, 1023 x 2304 x 768 26.5 against 32.
    const bool deep = force ? force == 32 : tiles(32, 32) <= 256;
    const char* which;
#define ZG_TILES(kernel, TM, TN, AHEAD, bm, bn) (kernel<AT, NP, TM, TN, AHEAD><<<grid(bm, bn), 256, 0, s>>>(p), which = #kernel "<" #TM ", " #TN ">")
    if (deep) ZG_TILES(lm_deep_kernel, 1, 1, 3, 32, 32);
    else if constexpr (NP == 1) {
        // (two steps ahead where rounded activations leave the registers for it: 8184 x 3072 x 1024 88.7 against 92.6)
        if (force ? force == 128 : tiles(128, 128) >= 320) ZG_TILES(lm_wide_kernel, 2, 2, (std::is_same<AT, float>::value ? 1 : 2), 128, 128);
        else ZG_TILES(lm_wide_kernel, 1, 1, 2, 64, 64);
    } else {
        if (force ? force == 128 : tiles(32, 64) > 512) ZG_TILES(lm_wide_kernel, 1, 2, 2, 64, 128);
        else ZG_TILES(lm_deep_kernel, 1, 2, 3, 32, 64);
    }
#undef ZG_TILES
    note_kernel("%s x %d", which, NP);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}
}  // namespace

int launch_linear_gated(const Linear& L, int F, int kind, float* h, bf16_t* h16, bool f32, hipStream_t s, bool* taken) {
    *taken = false;
    if (F <= 0 || L.act != ACT_NONE || L.bias || kind == GLU_CLIPPED || L.M <= 0 || L.a_glu) return ZG_OK;
    Linear g = L;
    g.N = 2 * F; g.glu_out = F; g.glu_kind = kind; g.C = h; g.C16 = nullptr; g.ldc = F; g.c_zoff = F;
    if (L.M > kGemvMaxRows || L.grp_off) {  // prompt portions
        if (h16) g.C = nullptr, g.C16 = h16;
        return launch_stream(g, f32, s, taken);
    }
    if (getenv("ZGPT2_LM_NO_ROWS") != nullptr) return ZG_OK;
    return launch_rows(g, nullptr, s, taken);
}

int launch_linear_normed(const Linear& L, const NormIn& n, hipStream_t s, bool* taken) {
    *taken = false;
    const uintptr_t all = reinterpret_cast<uintptr_t>(n.x) | reinterpret_cast<uintptr_t>(n.y) | reinterpret_cast<uintptr_t>(n.wb) | reinterpret_cast<uintptr_t>(n.wn) |
                          reinterpret_cast<uintptr_t>(n.x_out);
    if (L.M != 1 || (all & 15) != 0 || n.x == n.x_out || L.a_glu || L.a_poly || L.a_rows || L.z_group) return ZG_OK;
    return launch_gemv_at_once(L, nullptr, &n, s, taken);
}

int launch_linear_row_norm(const Linear& L, hipStream_t s, bool* taken) {
    *taken = false;
    if (!L.a_norm || L.M <= 0 || L.M > kGemvMaxRows || L.grp_off || L.a_poly) return ZG_OK;
    if (getenv("ZGPT2_LM_NO_ROWS") == nullptr) ZG_TRY(launch_rows(L, nullptr, s, taken));
    return *taken ? ZG_OK : launch_gemv_at_once(L, nullptr, nullptr, s, taken);
}

int launch_linear(const Linear& L, bool f32, hipStream_t s) {
    if (L.M <= 0 || L.N <= 0 || L.nz <= 0) return ZG_OK;
    const bool tiled = L.grp_off || L.M > kGemvMaxRows;
    ZG_REQUIRE(L.K > 0 && L.B && (tiled ? (L.A || (L.A16 && !f32)) && (L.C || L.C16) : L.A && L.C && !L.C16), ZG_ERR_ARG, "linear: empty operand");
    ZG_REQUIRE(L.a_div >= 1, ZG_ERR_ARG, "linear: a_div %d", L.a_div);
    ZG_REQUIRE(!L.a_norm, ZG_ERR_ARG, "linear: a norm on load is launch_linear_row_norm's");
    ZG_REQUIRE(!L.a_poly || (L.M <= kPolyMaxRows && L.a_glu == 0 && !L.grp_off), ZG_ERR_ARG, "linear: the polynomial activation on load is for %d rows at most",
               kPolyMaxRows);
    const LinArgs p = make_args(L);
    if (!L.grp_off && L.M <= kGemvMaxRows) {
        bool taken = false;
        if (getenv("ZGPT2_LM_NO_ROWS") == nullptr) ZG_TRY(launch_rows(L, nullptr, s, &taken));
        if (taken) return ZG_OK;
        ZG_TRY(launch_gemv_at_once(L, nullptr, nullptr, s, &taken));
        if (taken) return ZG_OK;
        if (takes_k_split(L)) {  // long rows, one or two of them, few batches: K split over the waves, two weight rows per workgroup
            const dim3 gks((L.N + 1) / 2, 1, L.nz);  // (from four rows on the activations are re-read by too many workgroups: measured slower)
            if (L.a_poly) {
                if (L.M == 1) lm_gemv_ks_kernel<1, true><<<gks, 256, 0, s>>>(p);
                else lm_gemv_ks_kernel<2, true><<<gks, 256, 0, s>>>(p);
            } else if (L.M == 1) lm_gemv_ks_kernel<1, false><<<gks, 256, 0, s>>>(p);
            else lm_gemv_ks_kernel<2, false><<<gks, 256, 0, s>>>(p);
            note_kernel("lm_gemv_ks_kernel<%d>", L.M);
            ZG_HIP(hipGetLastError());
            return ZG_OK;
        }
        const dim3 grid((L.N + 7) / 8, 1, L.nz);
        if (L.a_poly && L.M == 1) lm_gemv_kernel<1, true><<<grid, 256, 0, s>>>(p);
        else if (L.a_poly) lm_gemv_kernel<2, true><<<grid, 256, 0, s>>>(p);
        else if (L.M == 1) lm_gemv_kernel<1, false><<<grid, 256, 0, s>>>(p);
        else if (L.M == 2) lm_gemv_kernel<2, false><<<grid, 256, 0, s>>>(p);
        else if (L.M <= 4) lm_gemv_kernel<4, false><<<grid, 256, 0, s>>>(p);
        else lm_gemv_kernel<8, false><<<grid, 256, 0, s>>>(p);
        note_kernel("lm_gemv_kernel<%d>", L.M == 1 ? 1 : L.M == 2 ? 2 : L.M <= 4 ? 4 : 8);
        ZG_HIP(hipGetLastError());
        return ZG_OK;
    }
    ZG_REQUIRE(L.a_glu == 0, ZG_ERR_ARG, "linear: the gated activation on load is for steps of few rows");
    ZG_REQUIRE(!(L.z_group && L.grp_off), ZG_ERR_ARG, "linear: a matrix per batch and row groups exclude each other");
    ZG_REQUIRE(L.z_limit == 0x7fffffff, ZG_ERR_ARG, "linear: skipped batches are for steps of few rows");
    const bool rounded = L.A16 && !f32;
    const bool persistent = rounded && takes_persistent(L);
    if (!persistent) {
        bool taken = false;
        ZG_TRY(launch_stream(L, f32, s, &taken));
        if (taken) return ZG_OK;
    }
    if (persistent) {
        GemmPlanes pl{};
        pl.lda = L.lda;
        pl.ldb = L.ldb;
        pl.kpp = L.K / 64;
        pl.npairs = 1;
        note_kernel("gemm_s4_kernel");
        if (L.act == ACT_RELU2) return launch_gemm_s4_relu2(L.A16, L.B, L.bias, L.C ? static_cast<void*>(L.C) : L.C16, L.M, L.N, pl, L.ldc, L.C == nullptr, s);
        return launch_gemm_s4(L.A16, L.B, L.bias, L.C ? static_cast<void*>(L.C) : L.C16, L.M, L.N, pl, L.ldc, false, L.C == nullptr, 192, s);
    }
    const bool a_vec = rounded ? (reinterpret_cast<uintptr_t>(L.A16) & 15) == 0 && L.lda % 8 == 0 && L.a_zoff % 8 == 0 : p.a_vec != 0;
    if (a_vec && p.b_vec && L.K % 8 == 0 && !L.z_group && !toy_product(L, f32)) {
        if (f32) return launch_tiles<float, 3>(L, p, s);
        return rounded ? launch_tiles<bf16_t, 1>(L, p, s) : launch_tiles<float, 1>(L, p, s);
    }
    ZG_REQUIRE(L.A && L.C && !L.C16, ZG_ERR_ARG, "linear: rounded rows need 16-byte pieces");
    const dim3 grid((L.N + 63) / 64, (L.M + 63) / 64 + (L.grp_off ? L.n_groups : 0), L.nz);
    ZG_REQUIRE(grid.y <= 65535 && grid.z <= 65535, ZG_ERR_UNSUPPORTED, "linear: %d rows in %d batches exceed the grid", L.M, L.nz);
    if (f32) lm_gemm_kernel<true><<<grid, 256, 0, s>>>(p);
    else lm_gemm_kernel<false><<<grid, 256, 0, s>>>(p);
    note_kernel("lm_gemm_kernel<%s>", f32 ? "true" : "false");
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
