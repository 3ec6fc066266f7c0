// lm_window_rows.hip — windowed attention of prompt portions whose heads keep their own weights: scores, softmax and weighted values of 32
// consecutive rows and a head in one pass over their keys, in true fp32 (v_mfma_f32_32x32x2_f32) in both precision modes.
//
// What bounds it: the fp32 matrix instruction (4096 cycles a wave and tile of 32 keys with heads of 64 channels) and the vector work beside it (some
// 600 instructions).  In four launches with the scores in a workspace, 12 heads on 3 in chunks of 512 took 50 (scores) + 20 (their maxima and
// sums) + 79 (values) + 16 us (shares added) for 58 blocks of 32 rows on up to 512 keys, here 60; 42 + 13 + 52 + 10 for 64 blocks on up to 256,
// here 36; 24 + 11 + 24 + 8 for 16 blocks, here 33.
// Scores and values are multiplied transposed (S^T = K Q^T, O^T = V^T P^T): a lane's column is a query, its maximum and sum are the lane's own, and
// the weights are the second product's operand as they lie.  A wave takes a head, the waves of a workgroup heads of a key head and, so that two
// share a SIMD, every ks-th tile of the keys; what these found meets in the LDS.
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "lm_window_parts.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kHalf = 32;  // channels of half a head at most

struct RowsArgs {
    const float *q, *cache, *sink, *out_gate;
    float* out;
    bf16_t* out16;
    const int *ent_start, *ent_len, *row_pos, *row_slot, *page_table;
    KeyMask mask;
    ScoreShape shape;
    float scale, out_factor;
    int ldq, ldo, ld_gate, H, G, D, V, max_pages, page_tokens, n_entries, hw, ks;
};

__device__ __forceinline__ float both_halves_max(float v) { return fmaxf(v, __shfl_xor(v, 32, 64)); }

// exp(x) for x <= 0 (x log2 e in two pieces; below what fp32 holds: 0)
__device__ __forceinline__ float exp_of(float x) {
    x = x < -150.0f ? -150.0f : x;  // (NaN stays)
    const float t = x * 1.44269502f, rest = fmaf(x, 1.44269502f, -t) + x * 1.92596303e-8f;
    const float p = __builtin_amdgcn_exp2f(t);
    return fmaf(p, rest * 0.693147182f, p);
}

// 32 CT >= V; SHAPED: scores are capped or lose the head's slope
template <int CT, bool SHAPED>
__global__ __launch_bounds__(512, 2) void window_rows_kernel(const RowsArgs a) {
    extern __shared__ __attribute__((aligned(16))) float s_mem[];  // a wave's tile of keys; behind the last, what the waves behind the first key range found: [wave][CT * 16 + 2][64]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, kh = lane >> 5;
    // the block's entry: 64 entries' block counts summed across the lanes at a time (the rows with the most keys first)
    int at = gridDim.x - 1 - blockIdx.x, e = -1, b = 0;
    for (int e0 = 0; e0 < a.n_entries; e0 += 64) {
        const int own = e0 + lane < a.n_entries ? (a.ent_len[min(e0 + lane, a.n_entries - 1)] + 31) / 32 : 0;
        int upto = own;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int below = __shfl_up(upto, d, 64);
            if (lane >= d) upto += below;
        }
        const unsigned long long past = __ballot(at < upto);
        if (past) {
            const int l = __builtin_ctzll(past);
            e = e0 + l;
            b = __builtin_amdgcn_readfirstlane(at - __shfl(upto - own, l, 64));
            break;
        }
        at -= __shfl(upto, 63, 64);
    }
    if (e < 0) return;
    const int rep = a.H / a.G, groups = (rep + a.hw - 1) / a.hw, g = blockIdx.y / groups, hi = blockIdx.y % groups * a.hw + wave % a.hw, range = wave / a.hw;
    const int h = g * rep + min(hi, rep - 1);
    const int m0 = a.ent_start[e] + 32 * b, nrows = min(32, a.ent_len[e] - 32 * b), pos0 = a.row_pos[m0], pos_last = pos0 + nrows - 1;
    // the block's keys, numbered like a row's: the kept tokens in front of the first row's window, then everything to the last row's position
    const KeySpan blk = key_span(pos0, a.mask), mine = key_span(pos0 + r, a.mask);
    const int lo_last = key_span(pos_last, a.mask).j_lo;
    const int n_blk = blk.n_first + pos_last - blk.j_lo + 1, n_tiles = (n_blk + 31) / 32;
    const int* pages = a.page_table + (size_t)a.row_slot[m0] * a.max_pages;
    const int Dh = a.D / 2;
    const size_t cstride = (size_t)a.G * (a.D + a.V);
    const int k_at = g * a.D, v_at = a.G * a.D + g * a.V;
    float* const s_k = s_mem + wave * 32 * 64;  // rows of 64 channels, their 16-byte pieces swizzled by the row
    float qreg[kHalf];
    f32x4 knext[8];  // the tile behind the one in the LDS, asked for in whole rows (16 lanes to a row; a lane asking for its own row half fetched every line eight times)
    uint64_t krow = 0;  // cache row of key lane % 32 of that tile
    int pos_next, page_next;  // (a tile's pages are asked for a tile before its keys)
    {
        const float* qr = a.q + (size_t)(m0 + min(r, nrows - 1)) * a.ldq + (size_t)h * a.D + kh * Dh;
#pragma unroll
        for (int t = 0; t < kHalf; t += 4) {
            const f32x4 x = t < Dh ? *reinterpret_cast<const f32x4*>(qr + t) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            qreg[t] = x.x; qreg[t + 1] = x.y; qreg[t + 2] = x.z; qreg[t + 3] = x.w;
        }
    }
    auto look_up = [&](int tile) {  // key 32 tile + r of the block (keys behind the last: the last, never weighed)
        pos_next = key_pos(blk, min(32 * min(tile, n_tiles - 1) + r, n_blk - 1));
        const int page = pos_next / a.page_tokens;
        pos_next -= page * a.page_tokens;
        page_next = pages[page % a.max_pages];
    };
    auto row_of = [&](int key) {
        const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)krow, key, 64), hi32 = (uint32_t)__shfl((int)(uint32_t)(krow >> 32), key, 64);
        return reinterpret_cast<const float*>((uint64_t)hi32 << 32 | lo);
    };
    auto fetch = [&]() {  // the tile looked up last
        krow = reinterpret_cast<uint64_t>(a.cache + ((size_t)page_next * a.page_tokens + pos_next) * cstride);
#pragma unroll
        for (int i = 0; i < 8; ++i) knext[i] = *reinterpret_cast<const f32x4*>(row_of(4 * i + (lane >> 4)) + k_at + min((lane & 15) * 4, a.D - 4));
    };
    f32x16 o[CT];
    int v_col[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        v_col[c] = v_at + min(c * 32 + r, a.V - 1);
#pragma unroll
        for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;
    }
    // what this lane's query sees, in the block's numbering: [0, n_keep) and [n_lo, n_hi]
    const int n_hi = min(n_blk - 1, blk.n_first + pos0 + r - blk.j_lo), n_lo = blk.n_first + mine.j_lo - blk.j_lo;
    const int n_keep = blk.n_first + max(0, mine.n_first - blk.j_lo);
    float mx = -INFINITY, l = 0.0f;
    auto file_keys = [&]() {  // the tile asked for last into the LDS
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(s_k + (4 * i + (lane >> 4)) * 64 + ((lane & 15) ^ ((4 * i + (lane >> 4)) & 15)) * 4) = knext[i];
    };
    auto sees_all = [&](int tile) {  // every row sees every key of the tile
        const int n0 = 32 * tile, j0 = blk.j_lo + n0 - blk.n_first;
        return n0 >= blk.n_first && j0 >= lo_last && j0 + 31 <= pos0;
    };
    // the tile in the LDS against the queries; element i: key 8 (i / 4) + 4 half + i % 4 of the tile, query lane % 32
    auto scores = [&](int tile, bool whole, f32x16& s) {
        float kreg[kHalf];
#pragma unroll
        for (int t = 0; t < kHalf; t += 4) {
            const f32x4 x = t < Dh ? *reinterpret_cast<const f32x4*>(s_k + r * 64 + (((kh * Dh + t) / 4) ^ (r & 15)) * 4) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            kreg[t] = x.x; kreg[t + 1] = x.y; kreg[t + 2] = x.z; kreg[t + 3] = x.w;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < kHalf; ++t) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kreg[t], qreg[t], s, 0, 0, 0);
        auto score_at = [&](int i) { return 32 * tile + 8 * (i >> 2) + 4 * kh + (i & 3); };
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = SHAPED ? shape_score(s[i] * a.scale, a.shape, h, pos0 + r - key_pos(blk, score_at(i))) : s[i] * a.scale;
        if (!whole)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int n = score_at(i);
                s[i] = n <= n_hi && (n >= n_lo || n < n_keep) ? s[i] : -INFINITY;
            }
    };
    bool odd = false;  // some masked key may have values that are not finite
    auto body = [&](int tile) {
        file_keys();
        float v[CT][16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float* vr = row_of(8 * (i >> 2) + 4 * kh + (i & 3));
#pragma unroll
            for (int c = 0; c < CT; ++c) v[c][i] = vr[v_col[c]];
        }
        fetch();
        look_up(tile + 2 * a.ks);
        const bool whole = sees_all(tile);
        f32x16 s;
        scores(tile, whole, s);
        float top = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) top = fmaxf(top, s[i]);
        top = fmaxf(mx, both_halves_max(top));
        if (__any(top > mx)) {
            const float f = mx == top ? 1.0f : expf(mx - top);  // (none so far: 0)
            l *= f;
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[c][i] *= f;
            mx = top;
        }
        const float ref = mx == -INFINITY ? 0.0f : mx;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = exp_of(s[i] - ref);
            l += s[i];
        }
        if (!whole) {  // a masked weight is zero, but zero times a value that is not finite is not: such values wait until the other tiles are done
            float z = 0.0f;
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < 16; ++i) z = fmaf(v[c][i], 0.0f, z);
            if (__builtin_expect(__any(z != z), 0)) {
                odd = true;
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = fabsf(v[c][i]) <= 3.4028235e38f ? v[c][i] : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int c = 0; c < CT; ++c) o[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[c][i], s[i], o[c], 0, 0, 0);
    };
    if (hi < rep && range < n_tiles) {
        look_up(range);
        fetch();
        look_up(range + a.ks);
        for (int tile = range; tile < n_tiles; tile += a.ks) body(tile);
    }
    if (__builtin_expect(odd, 0)) {  // what waited, key by key, for the rows that see it
        const float ref = mx == -INFINITY ? 0.0f : mx;
#pragma unroll 1
        for (int tile = range; tile < n_tiles; tile += a.ks) {
            if (sees_all(tile)) continue;
            look_up(tile);
            fetch();
            file_keys();
            f32x16 s;
            scores(tile, false, s);
#pragma unroll
            for (int i = 0; i < 16; ++i) s_k[(8 * (i >> 2) + 4 * kh + (i & 3)) * 32 + r] = exp_of(s[i] - ref);  // (the keys have been used)
#pragma unroll 1
            for (int key = 0; key < 32; ++key) {
                const int n = 32 * tile + key;
                const float* vr = row_of(key) + v_at;
                const float p = s_k[key * 32 + r];
                const bool sees = n <= n_hi && (n >= n_lo || n < n_keep);
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int x = 0; x < 16; ++x) {
                        const float y = vr[min(c * 32 + 8 * (x >> 2) + 4 * kh + (x & 3), a.V - 1)];
                        if (sees && !(fabsf(y) <= 3.4028235e38f)) o[c][x] = fmaf(p, y, o[c][x]);
                    }
            }
        }
    }
    __syncthreads();
    l += __shfl_xor(l, 32, 64);  // (the halves hold different keys' weights)
    constexpr int PART = (CT * 16 + 2) * 64;
    if (range > 0) {
        float* part = s_mem + (size_t)((range - 1) * a.hw + wave % a.hw) * PART + lane;
        part[0] = mx;
        part[64] = l;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 16; ++i) part[(2 + c * 16 + i) * 64] = o[c][i];
    }
    __syncthreads();
    if (range > 0 || hi >= rep) return;
    for (int k = 1; k < a.ks; ++k) {
        const float* part = s_mem + (size_t)((k - 1) * a.hw + wave % a.hw) * PART + lane;
        const float m2 = part[0], top = fmaxf(mx, m2), ref = top == -INFINITY ? 0.0f : top, f1 = expf(mx - ref), f2 = expf(m2 - ref);
        l = l * f1 + part[64] * f2;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[c][i] = o[c][i] * f1 + part[(2 + c * 16 + i) * 64] * f2;
        mx = top;
    }
    if (r >= nrows) return;
    const float sk = a.sink ? a.sink[h] : -INFINITY, top = fmaxf(mx, sk), f = expf(mx - top) / (l * expf(mx - top) + (a.sink ? expf(sk - top) : 0.0f));
    const size_t m = m0 + r, col = (size_t)h * a.V;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {  // channels c 32 + 8 (i / 4) + 4 half + ..
            const int ch = c * 32 + 2 * i + 4 * kh;
            if (ch >= a.V) continue;  // (V is whole pieces of four)
            f32x4 y = {o[c][i] * f, o[c][i + 1] * f, o[c][i + 2] * f, o[c][i + 3] * f};
            if (a.out_gate)
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] *= sigmoid_f(a.out_gate[m * a.ld_gate + col + ch + u]) * a.out_factor;
            if (a.out16) *reinterpret_cast<u32x2*>(a.out16 + m * a.ldo + col + ch) = u32x2{cvt_pk_bf16(y.x, y.y), cvt_pk_bf16(y.z, y.w)};
            else *reinterpret_cast<f32x4*>(a.out + m * a.ldo + col + ch) = y;
        }
}

}  // namespace

int launch_window_rows(const WindowStep& w, const int* ent_start, const int* ent_len, int n_entries, bf16_t* out16, hipStream_t s, bool* taken) {
    *taken = false;
    // test hooks: other forms of these steps
    for (const char* hook : {"ZGPT2_LM_WINDOW_GENERAL", "ZGPT2_LM_WINDOW_NO_TILES", "ZGPT2_LM_WINDOW_NO_ROWS"}) {
        const char* v = getenv(hook);
        if (v && strcmp(v, "0") != 0) return ZG_OK;
    }
    const uintptr_t all = reinterpret_cast<uintptr_t>(w.q) | reinterpret_cast<uintptr_t>(w.cache) | (out16 ? reinterpret_cast<uintptr_t>(out16) : reinterpret_cast<uintptr_t>(w.out));
    if (w.M <= kGemvMaxRows || !ent_start || n_entries <= 0 || w.D > 2 * kHalf || w.D % 8 != 0 || w.V > 64 || w.V % 4 != 0 || w.ldq % 4 != 0 || w.ldo % 4 != 0 || (all & 15) != 0 || w.shape.gate || w.H % w.G != 0)
        return ZG_OK;
    const int rep = w.H / w.G;
    RowsArgs a;
    a.q = w.q; a.cache = w.cache; a.sink = w.sink; a.out_gate = w.out_gate; a.out = w.out; a.out16 = out16;
    a.ent_start = ent_start; a.ent_len = ent_len; a.row_pos = w.row_pos; a.row_slot = w.row_slot; a.page_table = w.page_table;
    a.mask = w.mask; a.shape = w.shape; a.scale = w.scale; a.out_factor = w.out_factor;
    a.ldq = w.ldq; a.ldo = w.ldo; a.ld_gate = w.ld_gate; a.H = w.H; a.G = w.G; a.D = w.D; a.V = w.V; a.max_pages = w.max_pages; a.page_tokens = w.page_tokens; a.n_entries = n_entries;
    // Heads of a workgroup (its waves beyond them share the keys).  A compute unit has room for one workgroup, so the price is rounds of 256 workgroups
    // times a wave's longest range of the keys, in tiles of 32, and two tiles for the rest; fewer heads read the keys more often and have to
    // promise a tenth.  The grid holds counted blocks alone: with empty ones among 256 the last were a round of their own.  us a layer, one : two : four
    // heads (or the two named): 64 blocks of 12 heads on 3 (256 keys at most) 46 : 41 : 36, 58 (512) 62 : 59 : 60, 16 (512) 31 : 33 : 54; 16 sequences of one row,
    // 16 heads on 4 behind 4000 keys one 136, two 233; 32 sequences, 10 heads on 2 behind 4000 keys two 224, four 419; 25 heads on 5 behind 1000 two 142, four
    // 227; 48 sequences, 24 heads on 4 behind 100 keys two 71, four 69; 200 rows of 32 heads on 8 behind 4000 keys one 156, two 269.
    const int blocks = w.blocks > 0 ? w.blocks : (w.M + 31) / 32 + n_entries;
    auto price = [&](int hw) {
        const long long groups = (long long)blocks * w.G * ((rep + hw - 1) / hw);
        return (double)((groups + 255) / 256) * (2.0 + (double)w.keys / (32 * (8 / hw)));
    };
    a.hw = std::min(rep, 4);
    for (int hw = a.hw - 1; hw >= 1; --hw)
        if (price(hw) < 0.9 * price(a.hw)) a.hw = hw;
    a.ks = 8 / a.hw;
    const dim3 grid(blocks, w.G * ((rep + a.hw - 1) / a.hw));
    if (grid.y > 65535) return ZG_OK;
    const int ct = (w.V + 31) / 32;
    const size_t lds = std::max((size_t)a.hw * a.ks * 32 * 64, (size_t)(a.ks - 1) * a.hw * (ct * 16 + 2) * 64) * sizeof(float);
    const bool shaped = w.shape.cap > 0.0f || w.shape.slope;
#define ZG_ROWS(CT) (shaped ? window_rows_kernel<CT, true><<<grid, 64 * a.hw * a.ks, lds, s>>>(a) : window_rows_kernel<CT, false><<<grid, 64 * a.hw * a.ks, lds, s>>>(a))
    if (ct == 1) ZG_ROWS(1);
    else ZG_ROWS(2);
#undef ZG_ROWS
    ZG_HIP(hipGetLastError());
    note_kernel("window_rows_kernel<%d>", ct);
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
