// lm_linear_args.h — what the kernels behind launch_linear share (lm_linear.hip, lm_rows.hip): the launch's arguments, what happens to
// an activation on its way in and to an output on its way out, and the exact split of fp32 values into bf16 terms.
#pragma once
#include <type_traits>

#include "lm_kernels.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

struct LinArgs {
    const float* A;
    const bf16_t* B;
    float* C;
    const int* a_rows;
    const int* z_group;
    const int* grp_off;
    long long a_zoff, b_zoff, c_zoff;
    int lda, ldb, ldc;
    int M, N, K;
    int a_div, act, n_groups, a_glu;
    float act_a, act_b;
    const float* bias;
    int z_limit;
    int glu_kind;
    float glu_limit;
    const float* glu_scale;
    int glu_gate_col;
    const float* a_poly;
    float poly_eps;
    const float* a_norm;
    float norm_eps;
    const bf16_t* A16;  // the same rows as bf16 (tiled kernels), or null
    bf16_t* C16;        // the result rounded to bf16, beside or instead of C (tiled kernels), or null
    int glu_out;        // > 0: gated product (Linear::glu_out)
    int a_vec, b_vec;  // 16-byte loads allowed (alignment of base, leading dimension and batch offsets)
};

// output n on its way out: the bias, then the activation
__device__ __forceinline__ float finish(float v, int n, const LinArgs& p) {
    const int act = p.act;
    if (p.bias) v += p.bias[n];
    if (act == ACT_SCALE_SOFTCAP) {
        v *= p.act_a;
        if (p.act_b > 0.0f) v = p.act_b * tanhf(v / p.act_b);
    } else if (act == ACT_RELU2) {
        v = fmaxf(v, 0.0f);
        v = v * v;
    } else if (act == ACT_GELU_ERF) {
        v = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));
    }
    return v;
}

// the gated activation of a [gate | up] row, applied where a product reads it (sc: the row's factor, clipped form only)
__device__ __forceinline__ float glu_on_load(float g, float u, const LinArgs& p, float sc) {
    if (p.glu_kind == GLU_CLIPPED) {
        g = fminf(g * sc, p.glu_limit);
        u = fminf(fmaxf(u * sc, -p.glu_limit), p.glu_limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    if (p.glu_kind == GLU_GELU) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
    return g / (1.0f + expf(-g)) * u;
}

// eight consecutive fp32 values -> NP planes of eight bf16 (packed pairs)
template <int NP>
struct Planes8 {
    u32x4 v[NP];
};
// the upper bf16 half of a value (truncated), and what is left of it (nothing of an infinity or NaN)
__device__ __forceinline__ float term_left(float x) {
    const uint32_t b = __float_as_uint(x);
    const float r = x - __uint_as_float(b & 0xFFFF0000u);
    return (b & 0x7F800000u) == 0x7F800000u ? 0.0f : r;
}
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }
template <int NP>
__device__ __forceinline__ Planes8<NP> to_planes(const f32x4& a, const f32x4& b) {
    Planes8<NP> o;
    if constexpr (NP == 1) {
        o.v[0] = u32x4{cvt_pk_bf16(a.x, a.y), cvt_pk_bf16(a.z, a.w), cvt_pk_bf16(b.x, b.y), cvt_pk_bf16(b.z, b.w)};
    } else {
        float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int t = 0; t < NP; ++t) {  // 24 mantissa bits = 8 + 8 + 8: what the third term leaves is zero
            o.v[t] = u32x4{upper_halves(x[0], x[1]), upper_halves(x[2], x[3]), upper_halves(x[4], x[5]), upper_halves(x[6], x[7])};
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (t + 1 < NP) x[i] = t == 0 ? term_left(x[i]) : x[i] - __uint_as_float(__float_as_uint(x[i]) & 0xFFFF0000u);
        }
    }
    return o;
}

// The tile of a workgroup: rows [m0, m_end) of A / C, columns from n0, the matrix.  Consecutive workgroups go to the eight XCDs in
// turn, so the tile list is dealt in eight contiguous runs: the tiles of one run share their A rows in that XCD's L2.
struct TileAt {
    const bf16_t* B;
    int m0, m_end, n0;
};
__device__ __forceinline__ bool find_tile(const LinArgs& p, int N, int BM, int BN, TileAt& t) {
    const int n_tiles = (N + BN - 1) / BN, total = gridDim.x, id = blockIdx.x;
    const int q = total >> 3, r = total & 7, x = id & 7;
    const int at = x * q + min(x, r) + (id >> 3);
    int mt = at / n_tiles;
    t.n0 = (at - mt * n_tiles) * BN;
    t.B = p.B + (long long)blockIdx.z * p.b_zoff;
    t.m0 = mt * BM;
    t.m_end = p.M;
    if (p.grp_off) {  // the row group this tile belongs to: 64 groups' tile counts summed across the lanes at a time
        const int lane = threadIdx.x & 63;
        for (int e0 = 0;; e0 += 64) {
            if (e0 >= p.n_groups) return false;
            const int e = min(e0 + lane, p.n_groups - 1);
            const int lo = p.grp_off[e], hi = p.grp_off[e + 1];
            const int own = e0 + lane < p.n_groups ? (hi - lo + BM - 1) / BM : 0;
            int upto = own;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(upto, d, 64);
                if (lane >= d) upto += o;
            }
            const unsigned long long past = __ballot(mt < upto);
            if (past) {
                const int l = __builtin_ctzll(past);
                t.B = p.B + (long long)(e0 + l) * p.b_zoff;
                t.m0 = __shfl(lo, l, 64) + (mt - __shfl(upto - own, l, 64)) * BM;
                t.m_end = __shfl(hi, l, 64);
                break;
            }
            mt -= __shfl(upto, 63, 64);
        }
    }
    return t.m0 < t.m_end;
}
inline LinArgs make_args(const Linear& L) {
    LinArgs p;
    p.A = L.A; p.B = L.B; p.C = L.C; p.a_rows = L.a_rows; p.z_group = L.z_group; p.grp_off = L.grp_off;
    p.a_zoff = L.a_zoff; p.b_zoff = L.b_zoff; p.c_zoff = L.c_zoff;
    p.lda = L.lda; p.ldb = L.ldb; p.ldc = L.ldc; p.M = L.M; p.N = L.N; p.K = L.K;
    p.a_div = L.a_div; p.act = L.act; p.n_groups = L.grp_off ? L.n_groups : 0; p.a_glu = L.a_glu;
    p.act_a = L.act_a; p.act_b = L.act_b; p.bias = L.bias; p.z_limit = L.z_limit; p.glu_kind = L.glu_kind; p.glu_limit = L.glu_limit; p.glu_scale = L.glu_scale;
    p.glu_gate_col = L.glu_gate_col;
    p.A16 = L.A16; p.C16 = L.C16; p.glu_out = L.glu_out;
    p.a_poly = L.a_poly;
    p.poly_eps = L.poly_eps;
    p.a_norm = L.a_norm;
    p.norm_eps = L.norm_eps;
    p.a_vec = ((reinterpret_cast<uintptr_t>(L.A) & 15) == 0 && L.lda % 4 == 0 && L.a_zoff % 4 == 0) ? 1 : 0;
    p.b_vec = ((reinterpret_cast<uintptr_t>(L.B) & 15) == 0 && L.ldb % 8 == 0 && L.b_zoff % 8 == 0) ? 1 : 0;
    return p;
}

}  // namespace

namespace {
// What rides in a launch of row-normed products (Linear::tail), in the second row of the grid.
struct TailArgs {
    ConvArgs cv;
    const int* slot = nullptr;
    int M = 0;
};
inline TailArgs tail_args(const Linear& L) {
    TailArgs t;
    if (L.tail) t.cv = *L.tail, t.slot = L.tail_slot, t.M = L.M;
    return t;
}
__device__ __forceinline__ void move_tails(const TailArgs& t) {
    const int per = (t.cv.C + 255) / 256;
    for (int b = blockIdx.x; b < t.M * per; b += gridDim.x) {
        const int m = b / per, c = (b - m * per) * 256 + threadIdx.x;
        if (c < t.cv.C) move_tail(t.cv, t.slot[m], m, c);
    }
}
}  // namespace

// lm_rows.hip: steps of 3 to 8 rows on the matrix cores.  *taken = false: not a form it has (nothing launched).
int launch_rows(const Linear& a, const Linear* b, hipStream_t s, bool* taken);
// 32-bit products of a few columns exist in toy models only.  There the last bits of a sum that cancels almost entirely can decide a row, and at
// any number of rows they stay what the fp32 instruction makes them: 5.5 us against 3.4 at K = 64.
inline bool toy_product(const Linear& L, bool f32) { return f32 && L.K < 128 && L.nz == 1; }
// lm_stream.hip: prompt portions whose K is whole steps of 64.  *taken as above.
bool stream_fits(const Linear& L, bool f32);
int launch_stream(const Linear& a, bool f32, hipStream_t s, bool* taken);
// lm_gemv.hip: steps of one or two rows whose operands are whole 16-byte pieces.  *taken as above.
int launch_gemv_at_once(const Linear& a, const Linear* b, const NormIn* norm, hipStream_t s, bool* taken);

}  // namespace lm
}  // namespace zg
