// lm_rows.hip — the linear maps of decode steps of 3 to 8 rows on the matrix cores, and the chosen experts' products of such steps.
//
// A workgroup owns 16 weight rows; its four waves take K in turns of 64 columns and meet in the LDS.  The weights are the MFMA's rows,
// straight from memory (a lane loads 32 bytes of its row, four lanes a 128-byte line).  The activations stay fp32: a value is the exact
// sum of three bf16 terms, the eight rows' leading and middle terms are the sixteen columns of one product, their last terms, under the
// middle ones, half of a second one.  Everything a wave needs is requested at entry for K up to 1024, four turns ahead beyond.
//
// The general kernel (lm_gemv_kernel) reads all rows for every two weight rows: 8 x 24 KB of activations through each wave for 3 KB of
// weights at K = 768.  Here they are read once per 16 weight rows.
//
// Gated feed-forwards: a workgroup owns eight gate rows and the eight rows they gate, and writes the activated values.  (Applied where the
// second product reads its rows, every workgroup of it repeated the activation: 15.7 us against 7.5 for eight experts of
// 768 x 768 and 16 assignments; the first product stays at 9.4.)
//
// Chosen experts: a workgroup takes an EXPERT's 16 weight rows and the (up to eight) assignments that chose it, found in the step's
// list on the device; experts nobody chose cost an empty workgroup, and one chosen by several rows is read once.
#include "lm_linear_args.h"

#include <algorithm>

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(4))) float acc4;

constexpr int kTurn = 64;  // columns of K a wave takes at a time

__device__ __forceinline__ int nth_bit(unsigned long long m, int n) {  // position of the n-th set bit (n < 8)
#pragma unroll
    for (int i = 0; i < 7; ++i)
        if (i < n) m &= m - 1;
    return __builtin_ctzll(m);
}

template <int I>
using step = std::integral_constant<int, I>;

enum { ROWS_PLAIN, ROWS_GLU_ON_LOAD, ROWS_GLU_OUT, ROWS_RMS };
// What the loads at entry need (leading arguments, see lm_gemv.hip).
struct RowsAt {
    const float* A;
    const bf16_t* B;
    const int* z_group;
    int K, N, M, ldb, lda, a_zoff, b_zoff, a_div;
    const float* a_norm = nullptr;  // ROWS_RMS: the rows' norm weights
    float eps = 0.0f;
};
// rows and matrices in a row; a matrix per list entry; either, and rows through an array; a list of at least as many entries as there are matrices
enum { FORM_PLAIN, FORM_LIST, FORM_ANY, FORM_FULL_LIST };
// TURNS > 0: every wave's turns are at most TURNS, all in flight at once; 0: any number, four in flight.
template <int TURNS, int KIND, int FORM, int WAVES = 4>
__device__ __forceinline__ void rows_body(const RowsAt& t, const LinArgs& p, const int z, float (*part)[16][17]) {
    // (nearly every matrix of a full list is somebody's: its rows are asked for in front of the list.  16 rows on 8 experts of 768 x 768: 6.5 us
    // against 7.0.  Gated products, bound by the terms they make, gain nothing: 8.6 against 8.2)
    constexpr bool EARLY = FORM == FORM_FULL_LIST && TURNS > 0;
    constexpr bool GLU = KIND == ROWS_GLU_ON_LOAD, OUT = KIND == ROWS_GLU_OUT, RMS = KIND == ROWS_RMS, ARRAY = FORM == FORM_ANY;
    const bool list = FORM == FORM_LIST || FORM == FORM_FULL_LIST || (FORM == FORM_ANY && t.z_group != nullptr);
    // (gated products: eight gates and the eight values they gate)
    constexpr int half = OUT ? 8 : 16;
    const int n0 = blockIdx.x * half, n_out = OUT ? t.N / 2 : t.N;
    if (n0 >= n_out) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kg = lane >> 4, m = col & 7;
    const int w_row = OUT ? (col & 8 ? n_out : 0) + min(n0 + (col & 7), n_out - 1) : min(n0 + col, t.N - 1);
    const bf16_t* w = t.B + (long long)z * t.b_zoff + (long long)w_row * t.ldb;
    constexpr int RING = TURNS > 0 ? TURNS : 4;
    u32x4 wr[RING][2];
    auto fetch_w = [&](int slot, int turn) {
#pragma unroll
        for (int j = 0; j < 2; ++j) wr[slot][j] = *reinterpret_cast<const u32x4*>(w + min(turn * kTurn + 16 * kg + 8 * j, t.K - 8));
    };
    unsigned long long left = 0;  // assignments of this expert that are still to do
    if (list) {
        const int mine = t.z_group[min(lane, t.M - 1)];
        if constexpr (EARLY) {
#pragma unroll
            for (int i = 0; i < TURNS; ++i) fetch_w(i, wave + WAVES * i);
            __builtin_amdgcn_sched_barrier(0);
        }
        left = __ballot(lane < t.M && mine == z);
        if (left == 0) return;
    }
    do {
        const int n_rows = list ? min(8, __popcll(left)) : t.M;
        // (columns without a row compute on the last one's and are not stored)
        const int rid = list ? nth_bit(left, min(m, n_rows - 1)) : min(m, n_rows - 1);
        const float* a = t.A + (long long)(list ? rid : z) * t.a_zoff + (long long)(FORM == FORM_PLAIN ? rid : (ARRAY && p.a_rows ? p.a_rows[rid] : rid) / t.a_div) * t.lda;
        const float asc = GLU && p.glu_scale ? p.glu_scale[rid] : 1.0f;
        const float agate = GLU && p.glu_gate_col >= 0 ? 1.0f / (1.0f + expf(-a[p.glu_gate_col])) : 1.0f;
        const int n_turns = (t.K + kTurn - 1) / kTurn;
        f32x4 ar[RING][4], ur[GLU || RMS ? RING : 1][4];
        float ss = 0.0f;  // (RMS) squares of the lane's share of its row
        auto fetch = [&](int slot, int turn) {
            if constexpr (!EARLY) fetch_w(slot, turn);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int k = min(turn * kTurn + 16 * kg + 8 * j, t.K - 8);
                ar[slot][2 * j] = *reinterpret_cast<const f32x4*>(a + k);
                ar[slot][2 * j + 1] = *reinterpret_cast<const f32x4*>(a + k + 4);
                if constexpr (GLU || RMS) {  // the values a gate multiplies, or the norm's weights
                    const float* u = RMS ? t.a_norm : a + p.a_glu;
                    ur[slot][2 * j] = *reinterpret_cast<const f32x4*>(u + k);
                    ur[slot][2 * j + 1] = *reinterpret_cast<const f32x4*>(u + k + 4);
                }
            }
        };
        acc4 acc1 = {0.0f, 0.0f, 0.0f, 0.0f}, acc2 = acc1;
        auto multiply = [&](int slot, int turn) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                f32x4 x = ar[slot][2 * j], y = ar[slot][2 * j + 1];
                u32x4 wv = wr[slot][j];
                if constexpr (GLU) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        x[u] = glu_on_load(x[u], ur[slot][2 * j][u], p, asc) * agate;
                        y[u] = glu_on_load(y[u], ur[slot][2 * j + 1][u], p, asc) * agate;
                    }
                }
                if (turn * kTurn + kTurn > t.K && turn * kTurn + 16 * kg + 8 * j >= t.K) {  // columns beyond K: the clamped load brought earlier ones
                    x = y = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    wv = u32x4{0u, 0u, 0u, 0u};
                }
                if constexpr (RMS) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        ss = fmaf(x[u], x[u], fmaf(y[u], y[u], ss));
                        x[u] *= ur[slot][2 * j][u];
                        y[u] *= ur[slot][2 * j + 1][u];
                    }
                }
                const Planes8<3> pl = to_planes<3>(x, y);
                const u32x4 zero = {0u, 0u, 0u, 0u};
                const bf16x8 wf = __builtin_bit_cast(bf16x8, wv);
                acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(bf16x8, col < 8 ? zero : pl.v[2]), acc2, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(bf16x8, col < 8 ? pl.v[0] : pl.v[1]), acc1, 0, 0, 0);
            }
        };
        if constexpr (TURNS > 0) {
#pragma unroll
            for (int i = 0; i < TURNS; ++i) fetch(i, wave + WAVES * i);
#pragma unroll
            for (int i = 0; i < TURNS; ++i) multiply(i, wave + WAVES * i);  // (a turn behind the last one multiplies zeros)
        } else {
#pragma unroll
            for (int i = 0; i < RING; ++i) fetch(i, wave + WAVES * i);
            for (int turn = wave; turn < n_turns; turn += WAVES * RING) {
#pragma unroll
                for (int i = 0; i < RING; ++i) {
                    multiply(i, turn + WAVES * i);
                    fetch(i, turn + WAVES * (i + RING));
                }
            }
        }
        // element e: weight row 4 kg + e, column col (leading terms, or middle and last ones).  An infinite sum of the leading terms is the
        // result: the other terms of what met the infinity may be zero, and zero times infinity is not
#pragma unroll
        for (int e = 0; e < 4; ++e) part[wave][4 * kg + e][col] = col < 8 ? acc1[e] : acc1[e] + acc2[e];
        __shared__ float s_ss[RMS ? 4 * WAVES : 1][8];
        if constexpr (RMS) {
            if (col < 8) s_ss[4 * wave + kg][m] = ss;
        }
        __syncthreads();
        const int row = threadIdx.x & 15, om = threadIdx.x >> 4;
        if (om < n_rows && row < half && n0 + row < n_out) {
            auto sum = [&](int r) {
                float hi = 0.0f, mid = 0.0f;
#pragma unroll
                for (int i = 0; i < WAVES; i += 4) {
                    hi += (part[i][r][om] + part[i + 1][r][om]) + (part[i + 2][r][om] + part[i + 3][r][om]);
                    mid += (part[i][r][om + 8] + part[i + 1][r][om + 8]) + (part[i + 2][r][om + 8] + part[i + 3][r][om + 8]);
                }
                return fabsf(hi) <= 3.4028235e38f ? hi + mid : hi;
            };
            float v = sum(row);
            if constexpr (RMS) {
                float q = 0.0f;
#pragma unroll
                for (int i = 0; i < 4 * WAVES; ++i) q += s_ss[i][om];
                v *= 1.0f / sqrtf(q / (float)t.K + t.eps);
            }
            float* C = p.C + (list ? (long long)nth_bit(left, om) * p.c_zoff : (long long)z * p.c_zoff + (long long)om * p.ldc);
            C[n0 + row] = OUT ? glu_on_load(v, sum(row + 8), p, 1.0f) : finish(v, n0 + row, p);
        }
        if (!list) return;
        for (int i = 0; i < 8 && left; ++i) left &= left - 1;
        if (left) __syncthreads();
    } while (left);
}

// batches [0, za) are product a's, the rest product b's
template <int TURNS, int KIND>
__global__ __launch_bounds__(256) void lm_rows_kernel(const LinArgs a, const LinArgs b, int za) {
    __shared__ float part[4][16][17];
    auto one = [&](const LinArgs& p, int z) {
        rows_body<TURNS, KIND, FORM_ANY>(RowsAt{p.A, p.B, p.z_group, p.K, p.N, p.M, p.ldb, p.lda, (int)p.a_zoff, (int)p.b_zoff, p.a_div}, p, z, part);
    };
    if ((int)blockIdx.z < za) one(a, blockIdx.z);
    else one(b, blockIdx.z - za);
}
// one product, rows in their order
template <int TURNS, int KIND, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void lm_rows_one_kernel(const float* A, const bf16_t* B, int K, int N, int M, int ldb, int lda, int a_zoff, int b_zoff, const LinArgs p) {
    __shared__ float part[WAVES][16][17];
    rows_body<TURNS, KIND, FORM_PLAIN, WAVES>(RowsAt{A, B, nullptr, K, N, M, ldb, lda, a_zoff, b_zoff, 1}, p, blockIdx.z, part);
}
template <int TURNS>
__global__ __launch_bounds__(256) void lm_rows_norm_kernel(const float* A, const bf16_t* B, const float* a_norm, int K, int N, int M, int ldb, int lda, float eps, const LinArgs p,
                                                           const TailArgs tail) {
    if (blockIdx.y > 0) return move_tails(tail);
    __shared__ float part[4][16][17];
    rows_body<TURNS, ROWS_RMS, FORM_PLAIN>(RowsAt{A, B, nullptr, K, N, M, ldb, lda, 0, 0, 1, a_norm, eps}, p, blockIdx.z, part);
}
template <int TURNS, int KIND, int FORM>
__global__ __launch_bounds__(256) void lm_rows_list_kernel(const float* A, const bf16_t* B, const int* z_group, int K, int N, int M, int ldb, int lda, int a_zoff, int b_zoff,
                                                           int a_div, const LinArgs p) {
    __shared__ float part[4][16][17];
    rows_body<TURNS, KIND, FORM>(RowsAt{A, B, z_group, K, N, M, ldb, lda, a_zoff, b_zoff, a_div}, p, blockIdx.z, part);
}

// One product of very many weight rows (the vocabulary): a workgroup makes the activations' terms once and takes every gridDim.x-th 16 weight
// rows, the next ones on their way beside the products.  Bound by the memory: 8 rows x 768 of 50257 weight rows (77 MB) 24.4 us against 30.6 for 3142
// workgroups that each made the terms again (9 us of vector work and as much again of activations read).
template <int TURNS>
__global__ __launch_bounds__(256) void lm_rows_many_kernel(const float* A, const bf16_t* B, int K, int N, int M, int ldb, int lda, const LinArgs p) {
    __shared__ float part[2][4][16][17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kg = lane >> 4, n_tiles = (N + 15) / 16;
    u32x4 wr[2][TURNS][2], first[TURNS][2], second[TURNS][2];  // leading and middle terms (columns 0 .. 7 and 8 .. 15), and under the middle ones the last
    int k_at[TURNS][2];
    auto fetch = [&](auto buf, int tile) {
        const bf16_t* w = B + (size_t)min(min(tile, n_tiles - 1) * 16 + col, N - 1) * ldb;
#pragma unroll
        for (int i = 0; i < TURNS; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) wr[buf][i][j] = *reinterpret_cast<const u32x4*>(w + k_at[i][j]);
    };
#pragma unroll
    for (int i = 0; i < TURNS; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) k_at[i][j] = min((wave + 4 * i) * kTurn + 16 * kg + 8 * j, K - 8);
    fetch(step<0>(), blockIdx.x);
    const float* a = A + (size_t)min(col & 7, M - 1) * lda;
#pragma unroll
    for (int i = 0; i < TURNS; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool beyond = (wave + 4 * i) * kTurn + 16 * kg + 8 * j >= K;  // (the clamped load brings earlier columns: they weigh nothing)
            const Planes8<3> pl = to_planes<3>(*reinterpret_cast<const f32x4*>(a + k_at[i][j]), *reinterpret_cast<const f32x4*>(a + k_at[i][j] + 4));
            const u32x4 zero = {0u, 0u, 0u, 0u};
            first[i][j] = beyond ? zero : col < 8 ? pl.v[0] : pl.v[1];
            second[i][j] = beyond || col < 8 ? zero : pl.v[2];
        }
    auto body = [&](auto buf, int tile) {
        constexpr int b = decltype(buf)::value;
        fetch(step<1 - b>(), tile + gridDim.x);
        acc4 acc1 = {0.0f, 0.0f, 0.0f, 0.0f}, acc2 = acc1;
#pragma unroll
        for (int i = 0; i < TURNS; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const u32x4 zero = {0u, 0u, 0u, 0u};
                const bool beyond = (wave + 4 * i) * kTurn + kTurn > K && (wave + 4 * i) * kTurn + 16 * kg + 8 * j >= K;
                const bf16x8 wf = __builtin_bit_cast(bf16x8, beyond ? zero : wr[b][i][j]);
                acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(bf16x8, second[i][j]), acc2, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(bf16x8, first[i][j]), acc1, 0, 0, 0);
            }
#pragma unroll
        for (int e = 0; e < 4; ++e) part[b][wave][4 * kg + e][col] = col < 8 ? acc1[e] : acc1[e] + acc2[e];
        __syncthreads();  // (the tile after next writes this place again: everybody has passed the next tile's barrier by then)
        const int row = threadIdx.x & 15, om = threadIdx.x >> 4, n = tile * 16 + row;
        if (om < M && n < N) {
            const float hi = (part[b][0][row][om] + part[b][1][row][om]) + (part[b][2][row][om] + part[b][3][row][om]);
            const float mid = (part[b][0][row][om + 8] + part[b][1][row][om + 8]) + (part[b][2][row][om + 8] + part[b][3][row][om + 8]);
            p.C[(long long)om * p.ldc + n] = finish(fabsf(hi) <= 3.4028235e38f ? hi + mid : hi, n, p);
        }
    };
    for (int tile = blockIdx.x; tile < n_tiles; tile += 2 * gridDim.x) {
        body(step<0>(), tile);
        if (tile + (int)gridDim.x < n_tiles) body(step<1>(), tile + gridDim.x);  // (uniform)
    }
}

// a product in the form the kernel takes: plain rows, or a list of one-row batches with the matrix chosen by a list (M: its length);
// false: neither
bool rows_form(const Linear& L, LinArgs& p, int& nz) {
    if (L.grp_off || L.a_poly || L.C16 || L.K < 8 || L.N <= 0 || !L.A || !L.B || !L.C || L.a_div < 1) return false;
    p = make_args(L);
    nz = L.nz;
    if (L.a_zoff > 0x7fffffff || L.b_zoff > 0x7fffffff) return false;
    if (L.z_group) {
        if (L.M != 1 || L.nz > 64 || L.n_groups <= 0 || L.n_groups > 65535) return false;
        p.M = L.nz;
        nz = L.n_groups;  // (entries of the list that name no matrix are left alone, as z_limit asks)
        if (L.z_limit < L.n_groups) return false;
    } else if (L.M == 1 && L.nz > 1 && L.b_zoff == 0 && !L.a_rows) {  // one-row batches of one matrix
        if (L.a_zoff > 0x7fffffff || L.c_zoff > 0x7fffffff || L.a_div != 1) return false;
        p.M = L.nz;
        p.lda = (int)L.a_zoff;
        p.ldc = (int)L.c_zoff;
        nz = 1;
    }
    // Where it pays (us per launch, this against the general kernel): 3 rows 2304 x 768 4.3 : 5.6, 8 rows 4.9 : 9.5, 8 rows of the
    // vocabulary 31 : 75.  Beyond K = 1024 a compute unit's intake binds it and the general kernel's finer tiles spread over more of them: 3
    // rows 768 x 3072 9.4 : 8.5, 4 rows 9.9 : 9.2, 8 rows 11.9 : 14.8.
    // Lists: an expert nobody chose costs a grid plane of empty workgroups, one chosen twice saves a reading, so the line rises with the number
    // of experts.  Steps of four such layers, us, this against the general kernel, experts of 768 x 768: 8 of them, 8 assignments 172 : 168, 16
    // 189 : 197, 32 206 : 239; 32 of them, 16 214 : 209, 24 231 : 235; 64, 16 227 : 217, 24 247 : 248, 32 257 : 265; 256, 8 (one row) 323 : 270,
    // 32 352 : 337, 48 376 : 383.
    const bool pays = L.z_group ? p.M >= 14 + L.n_groups / 8 : p.M >= (L.K <= 1024 ? 3 : 6);
    if (L.glu_out && L.a_glu) return false;
    if (L.a_norm && (L.z_group || L.a_rows || L.a_glu || L.glu_out || nz != 1 || p.a_div != 1 || (reinterpret_cast<uintptr_t>(L.a_norm) & 15) != 0)) return false;
    return pays && (L.z_group || p.M <= 8) && p.a_vec && p.b_vec && L.K % 8 == 0 && L.a_glu % 4 == 0 && nz <= 65535;
}

}  // namespace

int launch_rows(const Linear& A, const Linear* B, hipStream_t s, bool* taken) {
    *taken = false;
    LinArgs a, b;
    int za = 0, zb = 0;
    if (!rows_form(A, a, za)) return ZG_OK;
    b = a;
    if (B && (a.a_norm || B->a_norm || !rows_form(*B, b, zb) || za + zb > 65535 || (a.a_glu > 0) != (b.a_glu > 0) || a.glu_out || b.glu_out)) return ZG_OK;
    const int turns = (std::max(a.K, b.K) + kTurn - 1) / kTurn;
    auto tiles = [](const LinArgs& p) { return p.glu_out ? (p.glu_out + 7) / 8 : (p.N + 15) / 16; };
    const dim3 grid(std::max(tiles(a), tiles(b)), A.a_norm && A.tail ? 2 : 1, za + zb);
    const int per_wave = (turns + 3) / 4;
    const bool one = !B && !a.a_rows && a.a_glu == 0 && (a.z_group || a.a_div == 1);
    // (rows beyond 1024 columns: sixteen waves, and every turn in flight again.  8 rows 768 x 3072 10.9 us against 12.8 with four waves and a ring)
    const int per_16 = (turns + 15) / 16;
    const bool wide = one && !a.z_group && !a.a_norm && a.glu_out == 0 && per_wave > 4 && per_16 <= 4;
    const bool many = one && !a.z_group && !a.a_norm && a.glu_out == 0 && per_wave <= 4 && za == 1 && tiles(a) >= 1024;
    const bool full = a.z_group && a.M >= za;
#define ZG_ROWS_ARGS a.A, a.B, a.K, a.N, a.M, a.ldb, a.lda, (int)a.a_zoff, (int)a.b_zoff, a
#define ZG_ROWS_LIST a.A, a.B, a.z_group, a.K, a.N, a.M, a.ldb, a.lda, (int)a.a_zoff, (int)a.b_zoff, a.a_div, a
#define ZG_ROWS_ONE(T, KIND)                                                                                      \
    do {                                                                                                          \
        if (full) lm_rows_list_kernel<T, KIND, T && KIND == ROWS_PLAIN ? FORM_FULL_LIST : FORM_LIST><<<grid, 256, 0, s>>>(ZG_ROWS_LIST);                \
        else if (a.z_group) lm_rows_list_kernel<T, KIND, FORM_LIST><<<grid, 256, 0, s>>>(ZG_ROWS_LIST);           \
        else lm_rows_one_kernel<T, KIND, 4><<<grid, 256, 0, s>>>(ZG_ROWS_ARGS);                                   \
    } while (0)
#define ZG_ROWS(T)                                                                                \
    do {                                                                                          \
        if (a.a_norm) lm_rows_norm_kernel<T><<<grid, 256, 0, s>>>(a.A, a.B, a.a_norm, a.K, a.N, a.M, a.ldb, a.lda, a.norm_eps, a, tail_args(A)); \
        else if (one && a.glu_out > 0) ZG_ROWS_ONE(T, ROWS_GLU_OUT);                                   \
        else if (one) ZG_ROWS_ONE(T, ROWS_PLAIN);                                                 \
        else if (a.a_glu > 0) lm_rows_kernel<T, ROWS_GLU_ON_LOAD><<<grid, 256, 0, s>>>(a, b, za);      \
        else if (a.glu_out > 0) lm_rows_kernel<T, ROWS_GLU_OUT><<<grid, 256, 0, s>>>(a, b, za);   \
        else lm_rows_kernel<T, ROWS_PLAIN><<<grid, 256, 0, s>>>(a, b, za);                        \
    } while (0)
    const int share = (tiles(a) + 1023) / 1024, groups = (tiles(a) + share - 1) / share;
#define ZG_ROWS_MANY(T) lm_rows_many_kernel<T><<<groups, 256, 0, s>>>(a.A, a.B, a.K, a.N, a.M, a.ldb, a.lda, a)
    if (wide && per_16 == 2) lm_rows_one_kernel<2, ROWS_PLAIN, 16><<<grid, 1024, 0, s>>>(ZG_ROWS_ARGS);
    else if (wide && per_16 == 3) lm_rows_one_kernel<3, ROWS_PLAIN, 16><<<grid, 1024, 0, s>>>(ZG_ROWS_ARGS);
    else if (wide) lm_rows_one_kernel<4, ROWS_PLAIN, 16><<<grid, 1024, 0, s>>>(ZG_ROWS_ARGS);
    else if (many && per_wave == 1) ZG_ROWS_MANY(1);
    else if (many && per_wave == 2) ZG_ROWS_MANY(2);
    else if (many && per_wave == 3) ZG_ROWS_MANY(3);
    else if (many) ZG_ROWS_MANY(4);
    else if (per_wave == 1) ZG_ROWS(1);
    else if (per_wave == 2) ZG_ROWS(2);
    else if (per_wave == 3) ZG_ROWS(3);
    else if (per_wave == 4) ZG_ROWS(4);
    else ZG_ROWS(0);
#undef ZG_ROWS
#undef ZG_ROWS_ONE
#undef ZG_ROWS_MANY
#undef ZG_ROWS_ARGS
#undef ZG_ROWS_LIST
    note_kernel("lm_rows_kernel<%d>", per_wave <= 4 ? per_wave : 0);
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
