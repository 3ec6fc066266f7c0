// lm_gemv.hip — the linear maps of decode steps of one or two rows, operands in whole 16-byte pieces.
//
// A step of one sequence is a chain of some hundred launches that each read a few MB: its time is the chain's latency, and a launch's
// latency is the number of memory round trips it makes.  Here everything a wave reads (its share of two weight rows and of the
// activations) is requested at entry, unconditionally and at clamped addresses, before anything is used: one round trip.  (In the
// general kernel, lm_gemv_kernel, every piece is loaded under its own bounds check and waited for inside it.)
//
// One row, us a launch inside a replayed step, this against the general kernel: 768 columns 4.3 : 5.6, 3072 columns through the polynomial
// 4.7 : 7.4.  With the sum and the two norms in front of a product inside it 4.45, where their own launch took 5.25 more.
// What a row needs before its products (norms, the polynomial) is worked out while the weights are on their way and shared by four weight rows
// (the rule is at the launch): the polynomial had met its weights power by power, eleven sums and fifteen operations an element, where its
// statistics now meet over the workgroup first and an element is one product a weight row: 4.0 -> 3.2 us a launch.
// Both, 64 tokens of one sequence (768 wide, twelve layers, twelve feed-forwards through it) 19.4 -> 18.8 ms.
//
// Short rows: a wave has two or four whole weight rows.  Long rows (K of 1536 and more): a workgroup has them, its four waves a quarter of K each.
#include "lm_linear_args.h"

#include <algorithm>

namespace zg {
namespace lm {

namespace {

enum { GEMV_PLAIN, GEMV_GLU, GEMV_POLY, GEMV_NORM, GEMV_RMS };

// sums of N values over the lanes of a wave, each in every lane
template <int N>
__device__ __forceinline__ void wave_sums(float (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_allsum(v[i]);
}

// What the loads at entry need.  These travel as the leading arguments (14 dwords at most), which a wave finds in its registers; anything else
// of a launch's arguments is a round trip to memory of its own, cold in a step that has a new block of them for every launch.  Behind one
// such round trip a step of one sequence took 448 us, of eight 823; without it, here and in lm_rows.hip, 408 and 737, and with the norms, the
// router and the recurrence's step done alike 705.
struct GemvAt {
    const float* A;
    const bf16_t* B;
    int K, N, ldb, lda, a_zoff, b_zoff, a_glu;
    const float* a_norm = nullptr;  // GEMV_RMS: the rows' norm weights
    float eps = 0.0f;
    const float* a_poly = nullptr;  // GEMV_POLY: its four factors
};

// NR: weight rows of a wave (SPLIT: of a workgroup).  INDIRECT: rows through an array, or a matrix chosen by a list
template <int MR, int U, int KIND, bool SPLIT, bool INDIRECT, int NR = 2>
__device__ __forceinline__ void gemv_body(const GemvAt& t, const LinArgs& p, const int z, const NormIn& pre) {
    constexpr int NS = KIND == GEMV_RMS ? NR + 1 : NR;  // sums of a row: the products, then that of squares
    __shared__ float s_part[SPLIT ? 4 : 1][MR][NS], s_pow[4][MR][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = SPLIT ? blockIdx.x * NR : (blockIdx.x * 4 + wave) * NR;
    if (n0 >= t.N) return;
    if (INDIRECT && p.z_group && p.z_group[z] >= p.z_limit) return;
    const bf16_t* B = t.B + (long long)(INDIRECT && p.z_group ? p.z_group[z] : z) * t.b_zoff;
    const bf16_t* w[NR];
#pragma unroll
    for (int c = 0; c < NR; ++c) w[c] = B + (long long)min(n0 + c, t.N - 1) * t.ldb;
    const int kq = SPLIT ? (((t.K + 3) / 4) + 7) & ~7 : t.K;  // a wave's share of K, whole pieces of 8
    const int k_lo = SPLIT ? wave * kq : 0, k_hi = SPLIT ? min(t.K, k_lo + kq) : t.K;
    int at[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = k_lo + lane * 8 + 512 * u;
        in[u] = k < k_hi;
        at[u] = min(k, t.K - 8);
    }
    u32x4 wr[NR][U];
    f32x4 a[MR][U][2], g[KIND == GEMV_GLU ? MR : 1][U][2], nw[U][2];
    float asc[MR], agate[MR];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NR; ++c) wr[c][u] = *reinterpret_cast<const u32x4*>(w[c] + at[u]);
    if constexpr (KIND == GEMV_NORM) {
        // the row is norm(x + norm(y) (1 + wb)) (1 + wn): every wave works it out for itself, the first one keeps the sum
        f32x4 y[U][2], vb[U][2], vn[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[0][u][i] = *reinterpret_cast<const f32x4*>(pre.x + at[u] + 4 * i);
                y[u][i] = *reinterpret_cast<const f32x4*>(pre.y + at[u] + 4 * i);
                vb[u][i] = *reinterpret_cast<const f32x4*>(pre.wb + at[u] + 4 * i);
                vn[u][i] = *reinterpret_cast<const f32x4*>(pre.wn + at[u] + 4 * i);
            }
        float ss = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (in[u]) ss = fmaf(y[u][i][e], y[u][i][e], ss);
        const float r = 1.0f / sqrtf(wave_allsum(ss) / (float)t.K + pre.eps);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[0][u][i][e] += y[u][i][e] * r * (1.0f + vb[u][i][e]);
                    if (in[u]) s2 = fmaf(a[0][u][i][e], a[0][u][i][e], s2);
                }
                if (n0 == 0 && in[u]) *reinterpret_cast<f32x4*>(pre.x_out + at[u] + 4 * i) = a[0][u][i];
            }
        const float r2 = 1.0f / sqrtf(wave_allsum(s2) / (float)t.K + pre.eps);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[0][u][i][e] = a[0][u][i][e] * r2 * (1.0f + vn[u][i][e]);
    } else {
        float d[4];
        if constexpr (KIND == GEMV_POLY) {
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i] = t.a_poly[i];
        }
        const float* A = t.A + (long long)z * t.a_zoff;
        if constexpr (KIND == GEMV_RMS) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) nw[u][i] = *reinterpret_cast<const f32x4*>(t.a_norm + at[u] + 4 * i);
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const int rid = INDIRECT && p.z_group ? z * p.M + m : m;
            const float* row = A + (long long)(INDIRECT ? (p.a_rows ? p.a_rows[rid] : rid) / p.a_div : rid) * t.lda;
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[m][u][i] = *reinterpret_cast<const f32x4*>(row + at[u] + 4 * i);
                    if constexpr (KIND == GEMV_GLU) g[m][u][i] = *reinterpret_cast<const f32x4*>(row + t.a_glu + at[u] + 4 * i);
                }
            asc[m] = KIND == GEMV_GLU && p.glu_scale ? p.glu_scale[rid] : 1.0f;
            agate[m] = KIND == GEMV_GLU && p.glu_gate_col >= 0 ? 1.0f / (1.0f + expf(-row[p.glu_gate_col])) : 1.0f;
        }
        if constexpr (KIND == GEMV_POLY) {
            // the row is d0 n(v) + d1 n(v^2) + d2 n(v^3) + d3, every power divided by its root mean square: the workgroup's four shares meet, and the
            // row is worked out, while the weights are on their way
            static_assert(SPLIT, "the polynomial's rows are long");
            float q[MR][3];
#pragma unroll
            for (int m = 0; m < MR; ++m) {
#pragma unroll
                for (int i = 0; i < 3; ++i) q[m][i] = 0.0f;
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = in[u] ? a[m][u][i][e] : 0.0f, v2 = v * v, v3 = v2 * v;
                            q[m][0] += v2;
                            q[m][1] = fmaf(v2, v2, q[m][1]);
                            q[m][2] = fmaf(v3, v3, q[m][2]);
                        }
                wave_sums(q[m]);
            }
            if (lane == 0) {
#pragma unroll
                for (int m = 0; m < MR; ++m)
#pragma unroll
                    for (int i = 0; i < 3; ++i) s_pow[wave][m][i] = q[m][i];
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                float f[3];
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    f[i] = d[i] / sqrtf(((s_pow[0][m][i] + s_pow[1][m][i]) + (s_pow[2][m][i] + s_pow[3][m][i])) / (float)t.K + t.eps);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = a[m][u][i][e], v2 = v * v;
                            a[m][u][i][e] = fmaf(f[2], v2 * v, fmaf(f[1], v2, fmaf(f[0], v, d[3])));
                        }
            }
        }
    }
    ZG_PIN(p.C);
    ZG_PIN(p.bias);
    ZG_PIN(p.act);
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const u32x4 none = {0u, 0u, 0u, 0u};
    float sum[MR][NS];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int i = 0; i < NS; ++i) sum[m][i] = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        float wf[NR][8];
#pragma unroll
        for (int c = 0; c < NR; ++c) {
            const u32x4 v = in[u] ? wr[c][u] : none;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wf[c][2 * i] = bf16_lo(v[i]);
                wf[c][2 * i + 1] = bf16_hi(v[i]);
            }
        }
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f32x4 x = a[m][u][i];
                if constexpr (KIND == GEMV_GLU) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = glu_on_load(x[e], g[m][u][i][e], p, asc[m]) * agate[m];
                }
                if (!in[u]) x = zero;
                if constexpr (KIND == GEMV_RMS) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sum[m][NR] = fmaf(x[e], x[e], sum[m][NR]);
                        x[e] *= nw[u][i][e];
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) sum[m][r] = fmaf(x[e], wf[r][4 * i + e], sum[m][r]);
                }
            }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) wave_sums(sum[m]);
    float* C = p.C + (long long)z * p.c_zoff;
    if constexpr (!SPLIT) {
        if (lane < NR && n0 + lane < t.N) {
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                float v = sum[m][0];
#pragma unroll
                for (int r = 1; r < NR; ++r) v = lane == r ? sum[m][r] : v;
                if constexpr (KIND == GEMV_RMS) v *= 1.0f / sqrtf(sum[m][NR] / (float)t.K + t.eps);
                C[(long long)m * p.ldc + n0 + lane] = finish(v, n0 + lane, p);
            }
        }
    } else {
        if (lane == 0) {
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int i = 0; i < NS; ++i) s_part[wave][m][i] = sum[m][i];
        }
        __syncthreads();
        const int m = threadIdx.x / NR, c = threadIdx.x % NR;
        if (m < MR && n0 + c < t.N) {
            auto sum4 = [&](int i) { return (s_part[0][m][i] + s_part[1][m][i]) + (s_part[2][m][i] + s_part[3][m][i]); };
            float v = sum4(c);
            if constexpr (KIND == GEMV_RMS) v *= 1.0f / sqrtf(sum4(NR) / (float)t.K + t.eps);
            C[(long long)m * p.ldc + n0 + c] = finish(v, n0 + c, p);
        }
    }
}

template <int MR, int U, int KIND, bool SPLIT, bool INDIRECT, int NR>
__global__ __launch_bounds__(256) void lm_gemv_at_once_kernel(const float* A, const bf16_t* B, const float* a_poly, int K, int N, int ldb, int lda, int a_zoff,
                                                              int b_zoff, int a_glu, float poly_eps, const LinArgs p) {
    gemv_body<MR, U, KIND, SPLIT, INDIRECT, NR>(GemvAt{A, B, K, N, ldb, lda, a_zoff, b_zoff, a_glu, nullptr, poly_eps, a_poly}, p, blockIdx.z, NormIn());
}
template <int U, int NR>
__global__ __launch_bounds__(256) void lm_gemv_normed_kernel(const float* x, const float* y, const float* wb, const float* wn, const bf16_t* B, int K, int N, int ldb,
                                                             float eps, float* x_out, const LinArgs p) {
    gemv_body<1, U, GEMV_NORM, false, false, NR>(GemvAt{nullptr, B, K, N, ldb, 0, 0, 0, 0}, p, 0, NormIn{x, y, wb, wn, x_out, eps});
}
template <int MR, int U, bool SPLIT, int NR>
__global__ __launch_bounds__(256) void lm_gemv_row_norm_kernel(const float* A, const bf16_t* B, const float* a_norm, int K, int N, int ldb, int lda, float eps, const LinArgs p,
                                                               const TailArgs tail) {
    if (blockIdx.y > 0) return move_tails(tail);
    gemv_body<MR, U, GEMV_RMS, SPLIT, false, NR>(GemvAt{A, B, K, N, ldb, lda, 0, 0, 0, a_norm, eps}, p, 0, NormIn());
}
// batches [0, za) are product a's, the rest product b's
template <int U, int KIND>
__global__ __launch_bounds__(256) void lm_gemv_at_once_pair_kernel(const LinArgs a, const LinArgs b, int za) {
    auto one = [](const LinArgs& p, int z) {
        gemv_body<1, U, KIND, false, true>(GemvAt{p.A, p.B, p.K, p.N, p.ldb, p.lda, (int)p.a_zoff, (int)p.b_zoff, p.a_glu}, p, z, NormIn());
    };
    if ((int)blockIdx.z < za) one(a, blockIdx.z);
    else one(b, blockIdx.z - za);
}

constexpr int kLongRow = 1536;  // from here on K is split over the waves

int kind_of(const Linear& L) { return L.a_poly ? GEMV_POLY : L.a_glu > 0 ? GEMV_GLU : GEMV_PLAIN; }
bool pieces_ok(const Linear& L, const LinArgs& p) {
    return L.M >= 1 && L.M <= 2 && !L.grp_off && !L.C16 && !L.glu_out && L.N > 0 && L.nz >= 1 && L.nz <= 65535 && L.K >= 8 && L.K % 8 == 0 && L.A && L.B && L.C &&
           p.a_vec && p.b_vec && L.a_glu % 4 == 0 && L.a_div >= 1 && L.a_zoff <= 0x7fffffff && L.b_zoff <= 0x7fffffff;
}

}  // namespace

int launch_gemv_at_once(const Linear& A, const Linear* B, const NormIn* norm, hipStream_t s, bool* taken) {
    *taken = false;
    const LinArgs a = make_args(A), b = B ? make_args(*B) : a;
    if (!pieces_ok(A, a) || (B && (!pieces_ok(*B, b) || B->M != A.M || kind_of(*B) != kind_of(A) || A.nz + B->nz > 65535))) return ZG_OK;
    const int kind = norm ? (int)GEMV_NORM : A.a_norm ? (int)GEMV_RMS : kind_of(A);
    if (kind == GEMV_RMS && (B || kind_of(A) != GEMV_PLAIN || A.nz != 1 || A.a_rows || A.z_group || A.a_div != 1 || (reinterpret_cast<uintptr_t>(A.a_norm) & 15) != 0)) return ZG_OK;
    const int k_min = B ? std::min(A.K, B->K) : A.K, k_max = B ? std::max(A.K, B->K) : A.K;
    // (batches of long rows fill the chip without the split)
    const bool split = k_min >= kLongRow && A.nz + (B ? B->nz : 0) <= 4;
    if (kind == GEMV_POLY && !split) return ZG_OK;
    if (norm && (split || B || A.M != 1 || A.nz != 1)) return ZG_OK;
    if (B && (split || A.M != 1)) return ZG_OK;
    const int share = split ? (((k_max + 3) / 4) + 7) & ~7 : k_max, pieces = (share + 511) / 512;
    if (pieces > (norm ? 2 : 3)) return ZG_OK;
    const bool indirect = A.z_group || A.a_rows || A.a_div != 1;
    // Where every wave prepares the row for itself, four weight rows share a preparation once two would be more workgroups than compute units (some
    // then have two, each with the row's reads and arithmetic; up to there more waves are ahead).  One row, us a launch, four rows : two, 768 ->
    // 3072 behind the two norms 3.68 : 4.24, 768 -> 1680 2.88 : 3.92, 1536 -> 768 behind its own 2.80 : 2.96.  Without a preparation two: 768 ->
    // 3072 2.96 : 2.76, 768 -> 2304 2.84 : 2.76, 3072 -> 768 3.04 : 2.92, 768 -> 50264 12.3 : 12.0.
    const bool four = !B && !indirect && A.nz == 1 && (kind == GEMV_NORM || kind == GEMV_RMS || kind == GEMV_POLY) && A.N > 256 * (split ? 2 : 8);
    const int rows = (split ? 1 : 4) * (four ? 4 : 2);
    const dim3 grid((std::max(A.N, B ? B->N : 0) + rows - 1) / rows, A.a_norm && A.tail ? 2 : 1, A.nz + (B ? B->nz : 0));
#define ZG_GV(MR, U, KIND, SPLIT)                                                                                                                   \
    do {                                                                                                                                            \
        if (indirect) ZG_GV_I(MR, U, KIND, SPLIT, true, 2);                                                                                         \
        else if (four) ZG_GV_I(MR, U, KIND, SPLIT, false, (KIND == GEMV_POLY ? 4 : 2));                                                             \
        else ZG_GV_I(MR, U, KIND, SPLIT, false, 2);                                                                                                 \
    } while (0)
#define ZG_GV_I(MR, U, KIND, SPLIT, IND, NR)                                                                                                        \
    lm_gemv_at_once_kernel<MR, U, KIND, SPLIT, IND, NR><<<grid, 256, 0, s>>>(a.A, a.B, a.a_poly, a.K, a.N, a.ldb, a.lda, (int)a.a_zoff, (int)a.b_zoff, a.a_glu, a.poly_eps, a)
#define ZG_GV_P(KIND)                                                                              \
    do {                                                                                           \
        if (pieces == 1) lm_gemv_at_once_pair_kernel<1, KIND><<<grid, 256, 0, s>>>(a, b, A.nz);      \
        else if (pieces == 2) lm_gemv_at_once_pair_kernel<2, KIND><<<grid, 256, 0, s>>>(a, b, A.nz); \
        else lm_gemv_at_once_pair_kernel<3, KIND><<<grid, 256, 0, s>>>(a, b, A.nz);                  \
    } while (0)
#define ZG_GV_U(MR, KIND, SPLIT)                      \
    do {                                              \
        if (pieces == 1) ZG_GV(MR, 1, KIND, SPLIT);   \
        else if (pieces == 2) ZG_GV(MR, 2, KIND, SPLIT); \
        else ZG_GV(MR, 3, KIND, SPLIT);               \
    } while (0)
#define ZG_GV_M(KIND, SPLIT)                    \
    do {                                        \
        if (A.M == 1) ZG_GV_U(1, KIND, SPLIT);  \
        else ZG_GV_U(2, KIND, SPLIT);           \
    } while (0)
    if (B && kind == GEMV_GLU) ZG_GV_P(GEMV_GLU);
    else if (B) ZG_GV_P(GEMV_PLAIN);
    else if (norm) {
#define ZG_GV_N(U, NR) lm_gemv_normed_kernel<U, NR><<<grid, 256, 0, s>>>(norm->x, norm->y, norm->wb, norm->wn, a.B, a.K, a.N, a.ldb, norm->eps, norm->x_out, a)
        if (pieces == 1 && four) ZG_GV_N(1, 4);
        else if (pieces == 1) ZG_GV_N(1, 2);
        else if (four) ZG_GV_N(2, 4);
        else ZG_GV_N(2, 2);
#undef ZG_GV_N
    } else if (kind == GEMV_RMS) {
#define ZG_GV_R(MR, U)                               \
    do {                                             \
        if (split && four) ZG_GV_RN(MR, U, true, 4); \
        else if (split) ZG_GV_RN(MR, U, true, 2);    \
        else if (four) ZG_GV_RN(MR, U, false, 4);    \
        else ZG_GV_RN(MR, U, false, 2);              \
    } while (0)
#define ZG_GV_RN(MR, U, SPLIT, NR) \
    lm_gemv_row_norm_kernel<MR, U, SPLIT, NR><<<grid, 256, 0, s>>>(a.A, a.B, a.a_norm, a.K, a.N, a.ldb, a.lda, a.norm_eps, a, tail_args(A))
#define ZG_GV_RU(MR)                     \
    do {                                 \
        if (pieces == 1) ZG_GV_R(MR, 1); \
        else if (pieces == 2) ZG_GV_R(MR, 2); \
        else ZG_GV_R(MR, 3);             \
    } while (0)
        if (A.M == 1) ZG_GV_RU(1);
        else ZG_GV_RU(2);
#undef ZG_GV_R
#undef ZG_GV_RN
#undef ZG_GV_RU
    } else if (kind == GEMV_POLY) ZG_GV_M(GEMV_POLY, true);
    else if (kind == GEMV_GLU && split) ZG_GV_M(GEMV_GLU, true);
    else if (kind == GEMV_GLU) ZG_GV_M(GEMV_GLU, false);
    else if (split) ZG_GV_M(GEMV_PLAIN, true);
    else ZG_GV_M(GEMV_PLAIN, false);
#undef ZG_GV
#undef ZG_GV_I
#undef ZG_GV_P
#undef ZG_GV_U
#undef ZG_GV_M
    note_kernel("lm_gemv_at_once_kernel<%d>", A.M);
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
