// Greedy decode of two to eight sequences in lock step as a resident kernel: decode_resident.hip's cut of a Block over the XCDs and its
// hand-overs, the products on the matrix cores.  A generation alone, launches -> here: GPT-2 124M, 8 sequences, 75 + 181 tokens 57.7 -> 35.8 ms
// (33 + 991 322 -> 218), 4 sequences, 40 + 216 60.1 -> 34.3, 2 sequences 244 -> 133 us a step; char model, 8 sequences, 256 tokens 36.8 -> 15.5 ms.  bf16 weights: an activation travels as
// the exact three-term bf16 split of its fp32 value (zg_common.h split3_pk), split once by the thread that makes it, all three terms and a
// tag of 16 bits in ONE word; a wave multiplies 16 weight rows with the terms of all sequences (v_mfma_f32_16x16x32_bf16: columns of a
// product are terms x sequences), the waves split K and meet in the LDS.  A wave polls for the words its own lanes multiply, laid out as they
// ask for them, and the lanes that share a sequence hand its terms round (DPP): through the LDS and a barrier 40.4 ms.
//
// Per Block: x -> A c_attn -> q, k, v -> B attention -> C merge + c_proj -> (all XCDs) -> x -> D c_fc + GELU -> h -> E mlp c_proj -> (all XCDs) -> x.
// The thread that adds up a column of x (bias, residual, eight partial sums) also multiplies it with the gain of the LayerNorm that
// follows; mean and variance arrive as sums of 8 columns beside it and are applied to the product's outputs (LayerNorm linearised, as
// in gemv_ksplit.hip).
//
// What bounds it (8 sequences, 256 tokens, 13 us a Block): x is 48 KB of words for every workgroup, twice a Block, weights 60, keys and values 64:
// the compute unit's one queue of vector memory (27 to 64 B a cycle).  Measured and left out: a look at the sums alone before
// the columns are asked for (+2 %, a round trip more), pauses between looks (+0.5 %), keys of the next Block asked for beside the MLP
// (+2 %), c_proj's weights behind the merge instead of in front of c_attn (+1 %), partial sums polled by their column's thread alone (+0.6 %).
#include "decode_resident_parts.h"
#include "zg_once.h"

#include <type_traits>

namespace zg {

namespace {

using namespace resident;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef unsigned short u16;
constexpr int kPause = 8;                     // x 64 cycles before the first look at words of other XCDs
constexpr int kAfterX = 22;                   // before the first loads of a Block, behind the far words of the one in front (0: +1 %; 36: +1 %; 60: +3 %)
constexpr int kAfterA = 20;                   // before the fetches of a Block, behind c_attn's words
constexpr int kMostSplits = 4;                // workgroups that share the positions of a (head, sequence)

// three terms and the low half of the tag
__device__ __forceinline__ u64 terms(unsigned tag, float v) {
    uint32_t hi, mid, lo;
    split3_pk(v, 0.0f, hi, mid, lo);
    return ((u64)((tag << 16) | (lo & 0xffffu)) << 32) | (u64)((mid << 16) | (hi & 0xffffu));
}

// a lane's value and the ones 16 lanes (rows 0 and 1, 2 and 3) or 32 lanes away: both, on both lanes
__device__ __forceinline__ void rows_apart_16(unsigned v, unsigned& a, unsigned& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void rows_apart_32(unsigned v, unsigned& a, unsigned& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = r[0];
    b = r[1];
}
// over the lanes with the same lane & 7, on all of them
__device__ __forceinline__ float sum_over_8(float v) {
    v += dpp_row_ror<8>(v);
    unsigned a, b;
    rows_apart_16(__float_as_uint(v), a, b);
    v = __uint_as_float(a) + __uint_as_float(b);
    rows_apart_32(__float_as_uint(v), a, b);
    return __uint_as_float(a) + __uint_as_float(b);
}
// over the lanes 16 apart, or those with the same lane & 7, on all of them: the largest value, of equal ones the lowest index
template <bool EIGHT>
__device__ __forceinline__ void best_over(float& v, int& i) {
    const float own = v;
    unsigned a, b;
    if (EIGHT) v = fmaxf(v, dpp_row_ror<8>(v));
    rows_apart_16(__float_as_uint(v), a, b);
    v = fmaxf(__uint_as_float(a), __uint_as_float(b));
    rows_apart_32(__float_as_uint(v), a, b);
    v = fmaxf(__uint_as_float(a), __uint_as_float(b));
    int c = own == v ? i : 0x7fffffff;
    if (EIGHT) c = min(c, __builtin_amdgcn_update_dpp(0, c, 0x128, 0xF, 0xF, true));
    rows_apart_16((unsigned)c, a, b);
    c = min((int)a, (int)b);
    rows_apart_32((unsigned)c, a, b);
    i = min((int)a, (int)b);
}

template <int NW, int NH, int MB>
struct Spots {  // words
    static constexpr int E = 64 * NW, F = E / 2, CPR = 2 * NW;
    static constexpr int OW = (CPR * 8 + 63) / 64;             // waves that own columns of x
    static constexpr int sums = 2 * kRanks * OW * 8;           // (sum, sum of squares) of 8 columns by (workgroup, wave, sequence)
    static constexpr int block = (CPR * 8 + 15) & ~15;         // partial sums of a workgroup, all sequences
    static constexpr int qkv = 0, att = qkv + 8 * NH * 192, ml = att + 8 * NH * kMostSplits * 64, x1 = ml + 8 * NH * kMostSplits * 2, st1 = x1 + 8 * E, h = st1 + sums,
                         x2 = h + 8 * F, st2 = x2 + 8 * E, best = st2 + sums, near_words = best + kRanks * 8 * 2;
    static constexpr int far1 = kXcds * near_words, far2 = far1 + kXcds * kRanks * block, pick = far2 + kXcds * kRanks * block, words = pick + kXcds * 16;
};

// LDS, bytes of the dynamic part
template <int NW, int NH, int MB>
struct Hall {
    static constexpr int E = 64 * NW, F = E / 2, CPR = 2 * NW;
    static constexpr int turns(int bytes) { return (bytes + 4095) / 4096; }
    static constexpr int nA = turns(6 * NH * E * 2), nC = turns(CPR * NH * 64 * 2), nD = turns(NW * E * 2), nE = turns(CPR * F * 2);
    static constexpr int step = 3 * MB * 64 + 64;              // the terms of 32 columns of all sequences (64 more: consecutive steps start in other banks)
    static constexpr int TI = (CPR + 15) / 16;                 // tiles of 16 rows of C and E
    static constexpr int A = 0, C = A + 2 * nA * 4096, D = C + nC * 4096, Eo = D + nD * 4096, X = Eo + nE * 4096, acc = X + (E / 32) * step,
                         far_ = acc + (128 * NW + 16) * TI * 4, bytes = far_ + kXcds * CPR * 8 * 4;
};

template <int NW, int NH, int MB>
__global__ __launch_bounds__(64 * (NW + 4)) void decode_resident_batch_kernel(const ResidentArgs a) {
    typedef Spots<NW, NH, MB> P;
    typedef Hall<NW, NH, MB> R;
    constexpr int E = 64 * NW, F = E / 2, CPR = 2 * NW, NT = 64 * NW;
    constexpr int HC = NH * 64, TI = R::TI, OW = P::OW;
    constexpr int MX = MB / 2, MF = MB / 4;                        // sequences of a thread's pair of columns of x (two groups), of h (four groups)
    constexpr int NS = (P::sums / 2 + NT - 1) / NT, NF8 = (kXcds * CPR * 4 + NT - 1) / NT;
    constexpr int CJ = 2 * NH * TI;                                // (K step, tile) pairs of C
    static_assert(CJ <= NW && 2 * R::nA + R::nC + R::nD + R::nE + 20 < 64 && OW <= NW && 8 * 32 * NH <= NT, "shapes");
    static_assert(R::bytes + 10 * 1024 <= 160 * 1024, "LDS");

    extern __shared__ __attribute__((aligned(16))) char s_hall[];
    __shared__ float s_vec[2][192];                                // c2, c3 of the rows of A (12 each) and D (20 each); biases of the columns (32 each); ln_1 g, ln_2 g (32 each)
    __shared__ __attribute__((aligned(16))) float s_sum[2][8][NW];
    __shared__ __attribute__((aligned(16))) float s_new[192];      // q, k, v
    __shared__ __attribute__((aligned(16))) float s_o[16][64];
    __shared__ __attribute__((aligned(16))) float s_m[4], s_l[4];
    __shared__ float s_bv[16][8];
    __shared__ int s_bi[16][8];
    __shared__ int s_tok[8];
    __shared__ unsigned s_rank, s_go, s_fail;

    // (made opaque once a Block: what follows from them is made again where it is used instead of being kept, and spilled, for all Blocks)
    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto anew = [&]() {
        tid = (int)fresh((unsigned)tid);
        lane = tid & 63;
    };
    const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7u;  // HW_REG_XCC_ID
    if (tid == 0) {
        s_fail = 0u;
        s_go = join(a.ctl, xcc, (unsigned)a.s0, a.start_limit, &s_rank);
    }
    __syncthreads();
    if (s_go != 1u) {
        if (tid == 0) __hip_atomic_store(a.withdrawn, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    const int k = __builtin_amdgcn_readfirstlane((int)xcc), r = __builtin_amdgcn_readfirstlane((int)s_rank);
    const int H = a.n_heads, M = a.batch;
    const int nh = k < H ? (H - k + kXcds - 1) / kXcds : 0;       // heads of this XCD: k, k + 8, ...
    const int pairs = nh * M;                                     // (head, sequence)
    const int G = pairs > 0 ? min(kRanks / pairs, kMostSplits) : 1;  // workgroups of a pair
    const int my = r / G, sp = r % G;                             // this workgroup's
    const int ih = my < pairs ? my / M : 0, im = my < pairs ? my % M : 0;
    const int head = (k < H ? k : 0) + kXcds * ih;
    // positions 0 .. T - 1 in chunks of 64: a split's, this workgroup's (c0 .. c1 - 1), the splits there are
    int cps, c0, c1, n_sp;
    auto divide = [&](int T) {
        const int n = (T + 63) >> 6;
        cps = __builtin_amdgcn_readfirstlane((n + G - 1) / G);
        n_sp = __builtin_amdgcn_readfirstlane((n + cps - 1) / cps);
        c0 = sp * cps;
        c1 = min(c0 + cps, n);
        return my < pairs && c0 < n;
    };
    u64* const near = a.words + (size_t)k * P::near_words;
    u64* const far1 = a.words + P::far1;
    u64* const far2 = a.words + P::far2;
    u64* const picks = a.words + P::pick;
    auto row_A = [&](int j) {  // row j of this workgroup's 6 nh rows of c_attn
        const int n = r * 6 * nh + j, i = n / 192, part = (n % 192) / 64;
        return part * E + (k + kXcds * i) * 64 + (n & 63);
    };
    const unsigned hall = lds_at(s_hall);

    // the waves' shares of something, neighbours in the LDS
    auto sum_shares = [&](unsigned at) {
        if constexpr (NW % 4 == 0) {
            f32x4 v[NW / 4];
#pragma unroll
            for (int q = 0; q < NW / 4; ++q) v[q] = lds_read<f32x4>(at + q * 16);
            f32x4 s = v[0];
#pragma unroll
            for (int q = 1; q < NW / 4; ++q) s += v[q];
            return (s.x + s.y) + (s.z + s.w);
        } else {
            f32x2 v[NW / 2];
#pragma unroll
            for (int q = 0; q < NW / 2; ++q) v[q] = lds_read<f32x2>(at + q * 8);
            f32x2 s = v[0];
#pragma unroll
            for (int q = 1; q < NW / 2; ++q) s += v[q];
            return s.x + s.y;
        }
    };
    auto stats = [&](int m, float& mean, float& rstd) {
        const unsigned at = fresh(lds_at(&s_sum[0][m][0]));
        const float sx = sum_shares(at), sxx = sum_shares(at + 8 * NW * 4);
        mean = sx * (1.0f / (float)E);
        rstd = __builtin_amdgcn_rsqf(sxx * (1.0f / (float)E) - mean * mean + 1e-5f);
    };

    // ---- the vocabulary's rows: 16 of them with all sequences, by any wave
    auto head_tiles = [&](bool last) {
        const int V = a.vocab, tiles = (V + 15) >> 4, row16 = lane & 15, g4 = lane >> 4, m = lane & 15;
        float bv = -3.0e38f;
        int bi = 0x7fffffff;
        for (int j = wave; j * kXcds * kRanks + k * kRanks + r < tiles; j += NW + 4) {
            const int tile = j * kXcds * kRanks + k * kRanks + r;
            const gchar* const p = base_at(a.wte);
            const unsigned off = fresh((unsigned)(min(tile * 16 + row16, V - 1) * E) * 2u + (unsigned)g4 * 16u);
            constexpr int KS = E / 32, RING = 8;
            u32x4 wr[RING];
            f32x4 c2, c3;
#pragma unroll
            for (int t = 0; t < RING; ++t) wr[t] = *(gptr<const u32x4>)(p + off + t * 64);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned q = fresh((unsigned)min(tile * 16 + g4 * 4 + i, V - 1) * 4u);
                c2[i] = *(gptr<const float>)(base_at(a.lm_c2) + q);
                c3[i] = *(gptr<const float>)(base_at(a.lm_c3) + q);
            }
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < KS; ++t) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, wr[t % RING]);
                if (t + RING < KS) wr[t % RING] = *(gptr<const u32x4>)(p + off + (t + RING) * 64);
                const unsigned at = fresh(hall + R::X + (unsigned)t * R::step + (unsigned)(g4 * 16));
                if (MB == 8) {
                    acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, lds_read<u32x4>(at + (16u + (m & 7)) * 64u)), acc1, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, lds_read<u32x4>(at + (unsigned)m * 64u)), acc, 0, 0, 0);
                } else {
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, lds_read<u32x4>(at + (unsigned)min(m, 11) * 64u)), acc, 0, 0, 0);
                }
            }
            float mean, rstd;
            stats(m & 7, mean, rstd);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float s = MB == 8 ? (acc1[i] + dpp_row_ror<8>(acc[i])) + acc[i] : (dpp_row_ror<8>(acc[i]) + dpp_row_ror<12>(acc[i])) + acc[i];
                const float y = fmaf(rstd, fmaf(-mean, c2[i], s), c3[i]);
                const int row = tile * 16 + g4 * 4 + i;
                if (m < M && row < V) {
                    if (y > bv) {
                        bv = y;
                        bi = row;
                    }
                    if (last) *(gptr<float>)(base_at(a.logits) + fresh((unsigned)(m * V + row) * 4u)) = y;
                }
            }
        }
        best_over<false>(bv, bi);
        if (lane < 8) {
            s_bv[wave][lane] = bv;
            s_bi[wave][lane] = bi;
        }
    };

    // ---- weights: memory -> LDS, in pieces of 1 KB: pieces p0, p0 + dp, ... of a Block's matrices by one wave.  Rows of 16-byte units, unit u
    // of row j at u ^ (j & 7): the 16 rows a product reads at once lie in different banks
    auto from = [&](const void* base, int l, size_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)base_at(base, (size_t)l * a.w_stride), 0, (int)bytes, 0x00020000);
    };
    constexpr int uE = E / 8, uF = F / 8, uC = HC / 8;
    auto unit = [](int c, int u_row) { return (c % u_row) ^ ((c / u_row) & 7); };
    auto unit_at = [&](int p, int most) { return min((int)fresh((unsigned)(p * 64 + lane)), most); };
    auto fetch_A = [&](int l, int copy, int p0, int dp) {
        const auto b = from(a.c_attn_w, l, 3 * (size_t)E * E * 2);
#pragma unroll 1
        for (int p = p0; p < R::nA * 4; p += dp) {
            const int c = unit_at(p, max(6 * nh * uE - 1, 0));
            dma16(b, (unsigned)((nh > 0 ? row_A(c / uE) : 0) * E) * 2u + (unsigned)unit(c, uE) * 16u, hall + R::A + copy * R::nA * 4096 + p * 1024);
        }
    };
    auto fetch_C = [&](int l, int p0, int dp) {
        const auto b = from(a.c_proj_w, l, (size_t)E * E * 2);
#pragma unroll 1
        for (int p = p0; p < R::nC * 4; p += dp) {
            const int c = unit_at(p, CPR * uC - 1), u = unit(c, uC), i_h = u / 8;
            dma16(b, (unsigned)((r * CPR + c / uC) * E + ((k < H ? k : 0) + kXcds * (i_h < nh ? i_h : 0)) * 64) * 2u + (unsigned)(u % 8) * 16u, hall + R::C + p * 1024);
        }
    };
    auto fetch_D = [&](int l, int p0, int dp) {
        const auto b = from(a.c_fc_w, l, 4 * (size_t)E * E * 2);
#pragma unroll 1
        for (int p = p0; p < R::nD * 4; p += dp) {
            const int c = unit_at(p, NW * uE - 1);
            dma16(b, (unsigned)((k * F + r * NW + c / uE) * E) * 2u + (unsigned)unit(c, uE) * 16u, hall + R::D + p * 1024);
        }
    };
    auto fetch_E = [&](int l, int p0, int dp) {
        const auto b = from(a.mlp_proj_w, l, 4 * (size_t)E * E * 2);
#pragma unroll 1
        for (int p = p0; p < R::nE * 4; p += dp) {
            const int c = unit_at(p, CPR * uF - 1);
            dma16(b, (unsigned)((r * CPR + c / uF) * 4 * E + k * F) * 2u + (unsigned)unit(c, uF) * 16u, hall + R::Eo + p * 1024);
        }
    };
    auto fetch_V = [&](int l, int to, int w4) {
        const int q = min(w4, 2);  // 0: rows of A and D, 1: biases, 2: gains
        const float* v = q == 0 ? (lane < 12 ? a.c_attn_c2 : lane < 24 ? a.c_attn_c3 : lane < 44 ? a.c_fc_c2 : a.c_fc_c3)
                                : q == 1 ? (lane < 32 ? a.c_proj_b : a.mlp_proj_b) : (lane < 32 ? a.ln_1_g : a.ln_2_g);
        const int jA = lane < 12 ? lane : lane - 12;
        const int n = q == 0 ? (lane < 24 ? (jA < 6 * nh ? row_A(jA) : 0) : k * F + r * NW + min(lane < 44 ? lane - 24 : lane - 44, NW - 1))
                             : r * CPR + min(lane & 31, CPR - 1);
        const float* const p = reinterpret_cast<const float*>(reinterpret_cast<const char*>(v) + (size_t)l * a.w_stride) + n;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_at(&s_vec[to][q * 64])), "v"(p) : "memory", "m0");
    };

    if (wave >= NW) {
        // =========================================================================================== fetch and attend
        const int fw = wave - NW;
        // (in front of loads that are not always made: the registers would be kept for the rows they held before)
        auto forget = [&](KeyRows& x) {
            asm volatile("" : "=v"(x.k[0][0]), "=v"(x.k[0][1]), "=v"(x.k[1][0]), "=v"(x.k[1][1]));
            asm volatile("" : "=v"(x.v[0]), "=v"(x.v[1]), "=v"(x.v[2]), "=v"(x.v[3]));
        };
        // chunk c of 64 positions of this workgroup's (head, sequence): 16 a wave
        auto load_KV = [&](KeyRows& to, int l, int T, int c) {
            const size_t slab = (size_t)l * a.kv_stride + ((size_t)im * H + head) * a.ctx * 256;
            load_rows(to, a.k_cache + slab, a.v_cache + slab, a.ctx, c * 64 + fw * 16, T, lane);
        };
        int vp = 0;
        fetch_V(0, 0, fw);
        fetch_A(0, 0, fw, 4);
        in_flight<0>();
        barrier();  // B0
        for (int s = a.s0; s < a.s1; ++s) {
            const int T = s + 1;
            const bool here = divide(T);
            for (int l = 0; l < a.n_layer; ++l) {
                const int ln = l + 1 < a.n_layer ? l + 1 : 0;
                anew();
                if (nh > 0) {
                    __builtin_amdgcn_s_sleep(kAfterX);
                    if (!here) {
                        fetch_C(l, fw, 4);
                        barrier();  // B1a
                        __builtin_amdgcn_s_sleep(kAfterA);
                    } else {
                        // (asked for here: c_attn and its hand-over take longer than they do; across Blocks they would want 64 registers all along)
                        KeyRows kv[2];
                        load_KV(kv[0], l, T, c0);
                        fetch_C(l, fw, 4);
                        barrier();  // B1a
                        forget(kv[1]);
                        if (c0 + 1 < c1) load_KV(kv[1], l, T, c0 + 1);
                        barrier();  // B2
                        // ---- B
                        float m = kNone, lsum = 0.0f;
                        f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
                        for (int c = c0;;) {
                            if (c + 1 < c1) attend_rows<2, false>(kv, c * 64 + fw * 16, T, lane, s_new, m, lsum, o);  // one chunk or two
                            else attend_rows<1, false>(kv, c * 64 + fw * 16, T, lane, s_new, m, lsum, o);
                            c += 2;
                            if (c >= c1) break;
                            load_KV(kv[0], l, T, c);
                            forget(kv[1]);
                            if (c + 1 < c1) load_KV(kv[1], l, T, c + 1);
                        }
                        put_share(fw, lane, m, lsum, o, s_o, s_m, s_l);
                        barrier();  // B3
                    }
                } else {
                    barrier();  // B1
                }
                if (!(here && cps > 1)) {
                    fetch_D(l, fw, 4);
                    fetch_E(l, fw, 4);
                    fetch_V(ln, vp ^ 1, fw);
                    fetch_A(ln, vp ^ 1, fw, 4);
                }
                if (nh > 0) {
                    in_flight<R::nD + R::nE + 1 + R::nA>();  // C has arrived (behind the attention's rows where there were any)
                    barrier();  // B4
                    barrier();  // B4a
                }
                barrier();  // B4b
                in_flight<R::nE + 1 + R::nA>();  // D has
                barrier();  // B5
                barrier();  // B5a
                in_flight<0>();
                barrier();  // B6
                barrier();  // B6a
                barrier();  // B6b
                vp ^= 1;
            }
            if (s >= a.n_prompt) {
                barrier();  // B7
                head_tiles(s + 1 == a.s1);
                barrier();  // B8
            }
            barrier();  // B9
            if (s_fail != 0u) return;
            barrier();  // B10
        }
        return;
    }

    // ================================================================================================ rows and words
    Waiter w{a.spin_limit, &s_fail};
    int vp = 0;
    const unsigned all_words = (unsigned)P::words * 8u;
    // 16 bytes, two words, of lanes' own addresses: all of them checked by `ok`, asked for again until it holds
    auto words_at = [&](u64* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base_at(base), 0, (int)all_words, 0x00020000); };
    auto again = [&](unsigned& n) {  // another look?
        asm volatile("" ::: "memory");
        if (n >= w.limit) {
            s_fail = 1u;
            w.limit = 0u;
            return false;
        }
        ++n;
        return true;
    };
    auto load16 = [&](__amdgpu_buffer_rsrc_t b, unsigned i) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, (int)fresh(i * 8u), 0, 16)); };
    // Words of x and h lie as the lanes of a product ask for them, 1 KB at a time: columns [64 w, 64 w + 64) of x are wave w's two K steps, and
    // the MB lanes that share a sequence's columns in a product (its three terms) have a half or a quarter of them each.
    auto x_at = [](int col, int m) {
        const int w = col >> 6, i = col >> 5 & 1, g = col >> 3 & 3, u = col & 7;
        return MB == 8 ? ((w * 4 + (u >> 1)) * 64 + g * 16 + i * 8 + m) * 2 + (u & 1) : ((w * 2 + (u >> 1 & 1)) * 64 + g * 16 + (i * 2 + (u >> 2)) * 4 + m) * 2 + (u & 1);
    };
    auto h_at = [](int col, int m) {
        const int w = col >> 5, g = col >> 3 & 3, u = col & 7;
        return MB == 8 ? ((w * 2 + (u >> 1 & 1)) * 64 + g * 16 + (u >> 2) * 8 + m) * 2 + (u & 1) : (w * 64 + g * 16 + (u >> 1) * 4 + m) * 2 + (u & 1);
    };
    auto lane_of = [&]() { return (lane & ~(MB - 1)) | min(lane & (MB - 1), M - 1); };  // (sequences that are not there: the last one's words)
    // term 0, 1, 2 of a pair of columns
    auto term = [](const u32x4& v, int i) { return i == 2 ? __builtin_amdgcn_perm(v.w, v.y, 0x05040100u) : __builtin_amdgcn_perm(v.z, v.x, i ? 0x07060302u : 0x05040100u); };
    // the lanes of quarter `bank` take `v` of the lanes `by` quarters on, the others keep theirs
    auto from_quarter = [](uint32_t old, uint32_t v, auto by, auto bank) {
        constexpr int d = decltype(by)::value & 3, ctrl = d == 0 ? 0xE4 : 0x120 | (16 - 4 * d);
        return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, ctrl, 0xF, 1 << decltype(bank)::value, false);
    };
    auto from_half = [](uint32_t old, uint32_t v, auto bank) {  // the lanes of half `bank` take the other half's
        return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, 0x128, 0xF, decltype(bank)::value ? 0xC : 0x3, false);
    };
    // terms of columns (c, c + 1) of sequence m: their place among the K steps' operands in the LDS
    auto put_terms = [&](int c, int m, const u32x4& v) {
        const unsigned at = fresh(hall + R::X + (unsigned)(c >> 5) * R::step + (unsigned)m * 64u + (unsigned)(c & 31) * 2u);
        typedef __attribute__((address_space(3))) uint32_t lds_u32;
        *(lds_u32*)(uintptr_t)(at) = (v.x & 0xffffu) | (v.z << 16);
        *(lds_u32*)(uintptr_t)(at + MB * 64u) = (v.x >> 16) | (v.z & 0xffff0000u);
        *(lds_u32*)(uintptr_t)(at + 2 * MB * 64u) = (v.y & 0xffffu) | (v.w << 16);
    };
    // x of `tag`: this wave's 64 columns of all sequences as its lanes multiply them (x_at), and the waves' shares of its sums
    auto get_x = [&](unsigned at_x, unsigned at_st, unsigned tag, u32x4 (&v)[MX]) {
        const auto b = words_at(near);
        u32x4 st[NS];
        for (unsigned n = 0;;) {
            bool ok = true;
#pragma unroll
            for (int j = 0; j < MX; ++j) v[j] = load16(b, at_x + (unsigned)((wave * MX + j) * 64 + lane_of()) * 2u);
#pragma unroll
            for (int i = 0; i < NS; ++i) st[i] = load16(b, at_st + 2u * (unsigned)min(tid + i * NT, P::sums / 2 - 1));
#pragma unroll
            for (int j = 0; j < MX; ++j) ok = ok && (v[j].y >> 16) == (tag & 0xffffu) && (v[j].w >> 16) == (tag & 0xffffu);
#pragma unroll
            for (int i = 0; i < NS; ++i) ok = ok && st[i].y == tag && st[i].w == tag;
            if (ok || !again(n)) break;
        }
        float sx = __uint_as_float(st[0].x), sxx = __uint_as_float(st[0].z);
        if (NS > 1 && tid + NT < P::sums / 2) {
            sx += __uint_as_float(st[NS - 1].x);
            sxx += __uint_as_float(st[NS - 1].z);
        }
        sx = sum_over_8(sx);  // pair tid: sequence tid & 7
        sxx = sum_over_8(sxx);
        if (lane < 8) {
            s_sum[0][lane][wave] = sx;
            s_sum[1][lane][wave] = sxx;
        }
    };
    // N K steps from `ws` on (weights: rows of u_row units at `at_w`) times operands' steps of the same numbers, 16 rows from row0 on
    auto product = [&](auto n_steps, unsigned at_w, int u_row, int row0, int ws, f32x4& acc) {
        constexpr int N = decltype(n_steps)::value;
        const int row = row0 + (lane & 15), g = lane >> 4, n = lane & 15;
        const unsigned at_r = fresh(at_w + (unsigned)(row * u_row) * 16u), sw = (unsigned)(row & 7);
        const unsigned at_x = fresh(hall + R::X + (unsigned)ws * R::step + (unsigned)g * 16u);
        u32x4 wt[N], top[N], low[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            wt[i] = lds_read<u32x4>(at_r + (((unsigned)((ws + i) * 4 + g)) ^ sw) * 16u);
            if (MB == 8) low[i] = lds_read<u32x4>(at_x + i * R::step + (16u + (n & 7)) * 64u);
            top[i] = lds_read<u32x4>(at_x + i * R::step + (unsigned)(MB == 8 ? n : min(n, 11)) * 64u);
        }
        f32x4 s_low = {0.0f, 0.0f, 0.0f, 0.0f}, s_top = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (MB == 8) s_low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[i]), __builtin_bit_cast(bf16x8, low[i]), s_low, 0, 0, 0);
            s_top = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[i]), __builtin_bit_cast(bf16x8, top[i]), s_top, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc[i] = MB == 8 ? (s_low[i] + dpp_row_ror<8>(s_top[i])) + s_top[i] : (dpp_row_ror<8>(s_top[i]) + dpp_row_ror<12>(s_top[i])) + s_top[i];
    };
    // The same with the operands made from the words this wave has: N = 2, x; 1, h.  The weights are in wt already (row lane & 15)
    auto weights = [&](auto n_steps, unsigned at_w, int u_row, int row0, int ws, u32x4* wt) {
        const int row = row0 + (lane & 15), g = lane >> 4;
        const unsigned at_r = fresh(at_w + (unsigned)(row * u_row) * 16u), sw = (unsigned)(row & 7);
#pragma unroll
        for (int i = 0; i < decltype(n_steps)::value; ++i) wt[i] = lds_read<u32x4>(at_r + (((unsigned)((ws + i) * 4 + g)) ^ sw) * 16u);
    };
    constexpr std::integral_constant<int, 0> k0{};
    constexpr std::integral_constant<int, 1> k1{};
    constexpr std::integral_constant<int, 2> k2{};
    constexpr std::integral_constant<int, 3> k3{};
    auto operands = [&](auto n_steps, const u32x4* v, u32x4* top, u32x4* low) {
        constexpr int N = decltype(n_steps)::value;
        if constexpr (MB == 8) {
            const bool first = (lane & 8) == 0;
            if constexpr (N == 2) {  // (a lane has all columns of K step lane / 8 & 1)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t hi = term(v[j], 0), mid = term(v[j], 1), lo = term(v[j], 2);
                    top[0][j] = from_half(hi, mid, k1);
                    top[1][j] = from_half(mid, hi, k0);
                    low[0][j] = first ? lo : 0u;
                    low[1][j] = first ? 0u : lo;  // (columns 8 to 15 of that product: added in the end)
                }
            } else {  // (the first or the last four columns)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t hi = term(v[j], 0), mid = term(v[j], 1), lo = term(v[j], 2);
                    top[0][j] = from_half(hi, mid, k1);
                    top[0][2 + j] = from_half(mid, hi, k0);
                    low[0][j] = first ? lo : 0u;
                    low[0][2 + j] = from_half(0u, lo, k0);
                }
            }
        } else {
            auto all_terms = [&](auto from_q, const u32x4& w) {  // of the pair of columns that quarter from_q has: leading, middle, last term to quarters 0, 1, 2
                constexpr int q = decltype(from_q)::value;
                uint32_t x = from_quarter(0u, term(w, 0), std::integral_constant<int, q>{}, k0);
                x = from_quarter(x, term(w, 1), std::integral_constant<int, q - 1>{}, k1);
                return from_quarter(x, term(w, 2), std::integral_constant<int, q - 2>{}, k2);
            };
            if constexpr (N == 2) {  // (quarter 2 i + h has half h of K step i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    top[0][j] = all_terms(k0, v[j]);
                    top[0][2 + j] = all_terms(k1, v[j]);
                    top[1][j] = all_terms(k2, v[j]);
                    top[1][2 + j] = all_terms(k3, v[j]);
                }
            } else {
                top[0][0] = all_terms(k0, v[0]);
                top[0][1] = all_terms(k1, v[0]);
                top[0][2] = all_terms(k2, v[0]);
                top[0][3] = all_terms(k3, v[0]);
            }
        }
    };
    auto multiply = [&](auto n_steps, const u32x4* wt, const u32x4* top, const u32x4* low, f32x4& acc) {
        f32x4 s_low = {0.0f, 0.0f, 0.0f, 0.0f}, s_top = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < decltype(n_steps)::value; ++i) {
            if (MB == 8) s_low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[i]), __builtin_bit_cast(bf16x8, low[i]), s_low, 0, 0, 0);
            s_top = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[i]), __builtin_bit_cast(bf16x8, top[i]), s_top, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc[i] = MB == 8 ? ((s_low[i] + dpp_row_ror<8>(s_low[i])) + dpp_row_ror<8>(s_top[i])) + s_top[i]
                             : (dpp_row_ror<8>(s_top[i]) + dpp_row_ror<12>(s_top[i])) + s_top[i];
    };
    // (row, sequence) of 16 x 8 outputs: thread row * 8 + sequence finds the waves' shares at the same place
    auto acc_at = [&](int tile, int t) { return hall + R::acc + (unsigned)(tile * (128 * NW + 16) + t * NW + (t >> 5) * 4) * 4u; };  // (four words between the lanes' quarters: banks)
    auto share = [&](int tile, int of, const f32x4& acc) {
        if ((lane & 15) < 8) {
            const unsigned at = fresh(acc_at(tile, (lane >> 4) * 32 + (lane & 7)) + (unsigned)of * 4u);
            typedef __attribute__((address_space(3))) float lds_f32;
#pragma unroll
            for (int i = 0; i < 4; ++i) *(lds_f32*)(uintptr_t)(at + i * 8 * NW * 4) = acc[i];
        }
    };
    auto total = [&](int tile, int t) { return sum_shares(fresh(acc_at(tile, t))); };
    float* const s_far = reinterpret_cast<float*>(s_hall + R::far_);
    // thread -> column oc of this workgroup, sequence om, which it owns
    auto om = [&]() { return tid & 7; };
    auto oc = [&]() { return tid >> 3; };
    auto owns = [&]() { return oc() < CPR && om() < M; };
    auto ocol = [&]() { return r * CPR + min(oc(), CPR - 1); };
    float res = 0.0f;
    // x (in res) -> its terms times `gain`, sums of 8 columns
    auto put_x = [&](unsigned to_x, unsigned at_st, unsigned tag, float gain) {
        if (owns()) put_near(near, to_x, terms(tag, res * gain));
        if (wave < OW) {
            const float v = owns() ? res : 0.0f;
            const float sx = sum_over_8(v), sxx = sum_over_8(v * v);
            if (lane < 8) {
                const unsigned to = at_st + (unsigned)((r * OW + wave) * 16 + 2 * lane);
                put_near(near, to, tagged(tag, sx));
                put_near(near, to + 1u, tagged(tag, sxx));
            }
        }
    };
    // the eight partial sums of every column
    auto gather = [&](u64* from, int n_from, unsigned tag) {
        const auto b = words_at(from);
        __builtin_amdgcn_s_sleep(kPause);
        u32x4 v[NF8];
        for (unsigned n = 0;;) {
            bool ok = true;
#pragma unroll
            for (int i = 0; i < NF8; ++i) {
                const int u = min(tid + i * NT, kXcds * CPR * 4 - 1), q = u / (CPR * 4);
                v[i] = load16(b, (unsigned)((min(q, n_from - 1) * kRanks + r) * P::block + 2 * (u % (CPR * 4))));
                ok = ok && v[i].y == tag && v[i].w == tag;
            }
            if (ok || !again(n)) break;
        }
#pragma unroll
        for (int i = 0; i < NF8; ++i) {
            const int u = tid + i * NT;
            if (u < n_from * CPR * 4) *reinterpret_cast<f32x2*>(&s_far[u * 2]) = f32x2{__uint_as_float(v[i].x), __uint_as_float(v[i].z)};
        }
    };
    auto add_up = [&](int n_from, float bias) {
        if (oc() < CPR) {
            const unsigned at = fresh((unsigned)tid);
            float v[kXcds], y = 0.0f;
#pragma unroll
            for (int q = 0; q < kXcds; ++q) v[q] = s_far[q * CPR * 8 + at];
#pragma unroll
            for (int q = 0; q < kXcds; ++q) y += q < n_from ? v[q] : 0.0f;
            res += y + bias;
        }
    };
    __builtin_amdgcn_s_setprio(3);
    if (tid < 8) s_tok[tid] = tid < M && a.s0 > a.prompt_len[min(tid, M - 1)] ? a.out_tokens[(size_t)min(tid, M - 1) * a.out_stride + max(a.s0 - 1, 0)] : 0;
    const int np = a.prompt_len[min(om(), M - 1)];
    const float fin_g = a.ln_f_g[ocol()];
    barrier();  // B0
    for (int s = a.s0; s < a.s1; ++s) {
        const int T = s + 1;
        const bool here = divide(T), newest = sp == n_sp - 1;  // attends; to position T - 1 too
        const unsigned tag0 = a.tag0 + (unsigned)(s - a.s0) * (unsigned)(a.n_layer + 2);
        int tok = 0;
        if (owns()) {
            tok = s < np ? a.prompt[(size_t)om() * a.out_stride + s] : s == np ? a.prompt[(size_t)om() * a.out_stride + np - 1] : s_tok[om()];
            if (s < np && k == 0 && r == 0 && oc() == 0) a.out_tokens[(size_t)om() * a.out_stride + s] = tok;
            auto value = [&](const void* base, size_t row) -> float {
                return __uint_as_float((uint32_t)(reinterpret_cast<const bf16_t*>(base)[row * E + ocol()]) << 16);
            };
            res = value(a.wte, (size_t)tok) + value(a.wpe, (size_t)s);
        }
        put_x(P::x2 + (unsigned)x_at(ocol(), om()), P::st2, tag0, s_vec[vp][128 + min(oc(), 31)]);
        for (int l = 0; l < a.n_layer; ++l) {
            const unsigned tag = tag0 + 1u + (unsigned)l;
            anew();
            if (nh > 0) {
                // ---- A
                {
                    u32x4 wt[2], v[MX], top[2], low[2];
                    f32x4 acc;
                    weights(k2, hall + R::A + vp * R::nA * 4096, E / 8, 0, 2 * wave, wt);
                    get_x(P::x2, P::st2, tag - 1u, v);
                    operands(k2, v, top, low);
                    multiply(k2, wt, top, low, acc);
                    share(0, wave, acc);
                }
                const int jA = tid >> 3, nA = r * 6 * nh + jA;
                const bool hasA = jA < 6 * nh && om() < M;
                // (what the outputs are made with and where they go: known before the last share is)
                const unsigned toA = fresh(P::qkv + (unsigned)(om() * NH * 192 + nA));
                const float c2A = s_vec[vp][min(jA, 11)], c3A = s_vec[vp][12 + min(jA, 11)];
                barrier();  // B1a
                float yA = 0.0f;
                if (jA < 6 * nh) {
                    float mean, rstd;
                    stats(om(), mean, rstd);
                    yA = fmaf(rstd, fmaf(-mean, c2A, total(0, tid)), c3A);
                    if (hasA) put_near(near, toA, tagged(tag, yA));
                }
                if (here) {
                    if (tid < 192 && (tid < 64 || newest)) s_new[tid] = w.get(near, P::qkv + (unsigned)(im * NH * 192 + ih * 192 + tid), tag);
                    barrier();  // B2
                    // While four waves attend to more than 64 positions: the rest of this Block's weights and the next one's first.  What a
                    // thread polls for next returns behind them, but takes as long; and with it they are known to have arrived, long before
                    // anyone multiplies with them.  (124M, 8 sequences, 256 tokens 41.8 -> 41.0 ms, 1024 255 -> 247; up to 64 positions the attending
                    // waves fetch behind their attention: char model, 8 sequences 17.3 against 17.7 ms)
                    if (cps > 1) {
                        const int ln = l + 1 < a.n_layer ? l + 1 : 0;
                        fetch_D(l, wave, NW);
                        fetch_E(l, wave, NW);
                        if (wave < 3) fetch_V(ln, vp ^ 1, wave);
                        fetch_A(ln, vp ^ 1, wave, NW);
                    }
                    barrier();  // B3
                    if (wave == 0) {
                        float m, lsum, o;
                        merge_waves(lane, s_o, s_m, s_l, m, lsum, o);
                        const unsigned to = (unsigned)((im * NH + ih) * kMostSplits + sp);
                        if (lane < 2) put_near(near, P::ml + to * 2u + lane, tagged(tag, lane ? lsum : m));
                        put_near(near, P::att + to * 64u + lane, tagged(tag, o));
                    }
                }
                if (hasA) {  // the cache, while the partials are on their way
                    const int row = row_A(jA), part = row / E, c = row % E;
                    gchar *const kb = base_at(a.k_cache, (size_t)l * a.kv_stride), *const vb = base_at(a.v_cache, (size_t)l * a.kv_stride);
                    if (part > 0) *(gptr<float>)((part == 1 ? kb : vb) + (((size_t)(om() * H + (c >> 6)) * a.ctx + (T - 1)) * 64 + (c & 63)) * 4) = yA;
                }
                // ---- C: two columns of a sequence a thread, merged over the splits
                {
                    const int c2 = tid % (HC / 2), m = tid / (HC / 2), i_h = c2 >> 5;
                    if (m < MB) {
                        u32x4 z4 = {0u, 0u, 0u, 0u};
                        if (m < M && i_h < nh) {
                            const auto b = words_at(near);
                            u32x4 o4[kMostSplits], m4[kMostSplits];
                            for (unsigned n = 0;;) {
                                bool ok = true;
#pragma unroll
                                for (int q = 0; q < kMostSplits; ++q) {
                                    const unsigned at = (unsigned)((m * NH + i_h) * kMostSplits + min(q, n_sp - 1));
                                    if (q < n_sp) {
                                        o4[q] = load16(b, P::att + at * 64u + 2u * (unsigned)(c2 & 31));
                                        m4[q] = load16(b, P::ml + at * 2u);
                                    }
                                }
#pragma unroll
                                for (int q = 0; q < kMostSplits; ++q)
                                    if (q < n_sp) ok = ok && o4[q].y == tag && o4[q].w == tag && m4[q].y == tag && m4[q].w == tag;
                                if (ok || !again(n)) break;
                            }
                            float mx = kNone, lsum = 0.0f, z0 = 0.0f, z1 = 0.0f;
#pragma unroll
                            for (int q = 0; q < kMostSplits; ++q)
                                if (q < n_sp) mx = fmaxf(mx, __uint_as_float(m4[q].x));
#pragma unroll
                            for (int q = 0; q < kMostSplits; ++q)
                                if (q < n_sp) {
                                    const float e = __expf(__uint_as_float(m4[q].x) - mx);
                                    lsum = fmaf(e, __uint_as_float(m4[q].z), lsum);
                                    z0 = fmaf(e, __uint_as_float(o4[q].x), z0);
                                    z1 = fmaf(e, __uint_as_float(o4[q].z), z1);
                                }
                            const float inv = 1.0f / lsum;
                            const u64 t0 = terms(0u, z0 * inv), t1 = terms(0u, z1 * inv);
                            z4 = u32x4{(uint32_t)t0, (uint32_t)(t0 >> 32), (uint32_t)t1, (uint32_t)(t1 >> 32)};
                        }
                        put_terms(2 * c2, m, z4);
                    }
                }
                barrier();  // B4
                if (wave < CJ) {
                    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                    const int ws = wave % (2 * NH), ti = wave / (2 * NH);
                    if (ws < 2 * nh) product(k1, hall + R::C, HC / 8, ti * 16, ws, acc);
                    share(ti, ws, acc);
                }
                barrier();  // B4a
                if (tid < CPR * 8) {
                    float y = 0.0f;
                    const unsigned at = fresh(acc_at(tid >> 7, tid & 127));
                    f32x2 v[NH];
#pragma unroll
                    for (int q = 0; q < NH; ++q) v[q] = lds_read<f32x2>(at + q * 8);
#pragma unroll
                    for (int q = 0; q < NH; ++q) y += q < nh ? v[q].x + v[q].y : 0.0f;
                    if (om() < M) put_far(far1, (unsigned)((k * kRanks + r) * P::block + tid), tagged(tag, y));
                    else put_far(far1, (unsigned)((k * kRanks + r) * P::block + tid), tagged(tag, 0.0f));
                }
            } else {
                barrier();  // B1 (the helpers' fetches of vectors take the place of the Block's in front)
                if constexpr (NW < kFar1From)  // far2 has been read here (decode_resident_order.h)
                    if (tid < CPR * 8) put_far(far1, (unsigned)((k * kRanks + r) * P::block + tid), tagged(tag, 0.0f));
            }
            unsigned to_x = fresh(P::x1 + (unsigned)x_at(ocol(), om()));
            float bias = s_vec[vp][64 + min(oc(), 31)], gain = s_vec[vp][160 + min(oc(), 31)];
            gather(far1, kFar1From, tag);
            barrier();  // B4b
            add_up(kFar1From, bias);
            put_x(to_x, P::st1, tag, gain);
            barrier();  // B5
            // ---- D
            {
                u32x4 wt[2], v[MX], top[2], low[2];
                f32x4 acc;
                weights(k2, hall + R::D, E / 8, 0, 2 * wave, wt);
                get_x(P::x1, P::st1, tag, v);
                operands(k2, v, top, low);
                multiply(k2, wt, top, low, acc);
                share(0, wave, acc);
            }
            const unsigned toD = fresh(P::h + (unsigned)h_at(r * NW + min(oc(), NW - 1), om()));
            const float c2D = s_vec[vp][24 + min(oc(), NW - 1)], c3D = s_vec[vp][44 + min(oc(), NW - 1)];
            barrier();  // B5a
            if (oc() < NW) {
                float mean, rstd;
                stats(om(), mean, rstd);
                const float y = gelu_ref(fmaf(rstd, fmaf(-mean, c2D, total(0, tid)), c3D));
                if (om() < M) put_near(near, toD, terms(tag, y));
            }
            barrier();  // B6
            // ---- E
            {
                u32x4 wt[TI], v[MF], top[1], low[1];
#pragma unroll
                for (int ti = 0; ti < TI; ++ti) weights(k1, hall + R::Eo, F / 8, ti * 16, wave, wt + ti);
                const auto b = words_at(near);
                for (unsigned n = 0;;) {
                    bool ok = true;
#pragma unroll
                    for (int j = 0; j < MF; ++j) {
                        v[j] = load16(b, P::h + (unsigned)((wave * MF + j) * 64 + lane_of()) * 2u);
                        ok = ok && (v[j].y >> 16) == (tag & 0xffffu) && (v[j].w >> 16) == (tag & 0xffffu);
                    }
                    if (ok || !again(n)) break;
                }
                operands(k1, v, top, low);
#pragma unroll
                for (int ti = 0; ti < TI; ++ti) {
                    f32x4 acc;
                    multiply(k1, wt + ti, top, low, acc);
                    share(ti, wave, acc);
                }
            }
            barrier();  // B6a
            if (tid < CPR * 8) put_far(far2, (unsigned)((k * kRanks + r) * P::block + tid), tagged(tag, total(tid >> 7, tid & 127)));
            to_x = fresh(P::x2 + (unsigned)x_at(ocol(), om()));
            bias = s_vec[vp][96 + min(oc(), 31)];
            vp ^= 1;
            gain = l + 1 < a.n_layer ? s_vec[vp][128 + min(oc(), 31)] : fin_g;
            gather(far2, kXcds, tag);
            barrier();  // B6b
            add_up(kXcds, bias);
            put_x(to_x, P::st2, tag, gain);
        }
        const bool last = s + 1 == a.s1;
        if (s >= a.n_prompt) {  // ---- ln_f + lm_head + argmax (main.zig:189-194, :337)
            {
                u32x4 v[MX];
                get_x(P::x2, P::st2, tag0 + (unsigned)a.n_layer, v);
                const int q = lane >> 3 & 1, c = 64 * wave + (lane >> 4) * 8 + (MB == 8 ? q * 32 : q * 32 + (lane >> 2 & 1) * 4);
#pragma unroll
                for (int j = 0; j < MX; ++j) put_terms(c + 2 * j, lane & (MB - 1), v[j]);
            }
            barrier();  // B7
            head_tiles(last);
            barrier();  // B8
            const unsigned tag = tag0 + (unsigned)a.n_layer + 1u;
            static_assert(NW + 4 <= 16, "two waves' bests a lane");
            // (value, index): two words, in one store
            auto put_pair = [&](u64* base, unsigned at, float v, int i, auto scope) {
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(v), tag, (unsigned)i, tag}, words_at(base), (int)fresh(at * 8u), 0, scope);
            };
            constexpr std::integral_constant<int, 0> in_xcd{};
            constexpr std::integral_constant<int, 16> everywhere{};
            if (wave == 0) {  // the workgroup's: lane -> (waves lane >> 3 and that + 8, sequence lane & 7)
                const int q = lane >> 3, q8 = min(q + 8, NW + 3);
                float v = s_bv[min(q, NW + 3)][lane & 7];
                int i = s_bi[min(q, NW + 3)][lane & 7];
                better(v, i, s_bv[q8][lane & 7], s_bi[q8][lane & 7]);
                best_over<true>(v, i);
                if (lane < 8) put_pair(near, P::best + (unsigned)(r * 16 + 2 * lane), v, i, in_xcd);
            }
            auto pair_at = [&](u64* base, unsigned at, float& v, int& i) {
                const auto b = words_at(base);
                u32x4 p;
                for (unsigned n = 0;;) {
                    p = load16(b, at);
                    if ((p.y == tag && p.w == tag) || !again(n)) break;
                }
                v = __uint_as_float(p.x);
                i = (int)p.z;
            };
            if (r == 0 && wave == 0) {  // the XCD's: lane -> (workgroup lane >> 3 + 8 q, sequence lane & 7)
                float v = -3.0e38f;
                int i = 0x7fffffff;
                const auto b = words_at(near);
                u32x4 p[4];
                for (unsigned n = 0;;) {
                    bool ok = true;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        p[q] = load16(b, P::best + (unsigned)(((lane >> 3) + 8 * q) * 16 + 2 * (lane & 7)));
                        ok = ok && p[q].y == tag && p[q].w == tag;
                    }
                    if (ok || !again(n)) break;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) better(v, i, __uint_as_float(p[q].x), (int)p[q].z);
                best_over<true>(v, i);
                if (lane < 8) put_pair(picks, (unsigned)(k * 16 + 2 * lane), v, i, everywhere);
            }
            if (wave == 0) {
                float v;
                int i;
                __builtin_amdgcn_s_sleep(kPause);
                pair_at(picks, (unsigned)((lane >> 3) * 16 + 2 * (lane & 7)), v, i);
                best_over<true>(v, i);
                // logits that are all NaN: index 0, never one behind the table (embed_step_kernel)
                if (lane < 8) {
                    s_tok[lane] = (unsigned)i < (unsigned)a.vocab ? i : 0;
                    if (lane < M && k == 0 && r == 0) {
                        if (s >= np) a.out_tokens[(size_t)lane * a.out_stride + s] = s_tok[lane];
                        if (last) {  // for the launches that may follow: one partial holds the pick
                            a.part_val[(size_t)lane * a.n_part] = v;
                            a.part_idx[(size_t)lane * a.n_part] = i;
                        }
                    }
                }
            }
        }
        barrier();  // B9
        if (s_fail != 0u) {  // a wait ran out: results are worthless and everyone leaves
            if (tid == 0) __hip_atomic_store(a.fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
        barrier();  // B10
        if (last) {
            if (owns() && k == 0) a.x[(size_t)om() * E + ocol()] = res;
            if (k == 0 && r == 0) {
                if (s >= a.n_prompt)
                    for (int q = tid; q < M * a.n_part; q += NT)
                        if (q % a.n_part != 0) {
                            a.part_val[q] = -3.0e38f;
                            a.part_idx[q] = 0x7fffffff;
                        }
                if (owns() && oc() == 0) a.cur_token[om()] = tok;
                if (tid == 0) {
                    a.ctrl->seq_len = T;
                    a.ctrl->step = T;
                    a.ctl->done = (unsigned)T;
                }
            }
        }
    }
}

template <int NW, int NH, int MB>
int launch(const ResidentArgs& a, hipStream_t s) {
    note_kernel("decode_resident_batch_kernel<%d, %d, %d>", NW, NH, MB);
    constexpr int kOneEach = Hall<NW, NH, MB>::bytes > 84 * 1024 ? Hall<NW, NH, MB>::bytes : 84 * 1024;  // more than half of a compute unit's LDS: one workgroup each
    static OncePerDevice once;
    int dev = 0;
    ZG_HIP(hipGetDevice(&dev));
    ZG_TRY(once.run(dev, [&]() -> int {
        ZG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&decode_resident_batch_kernel<NW, NH, MB>), hipFuncAttributeMaxDynamicSharedMemorySize, kOneEach));
        return ZG_OK;
    }));
    hipLaunchKernelGGL((decode_resident_batch_kernel<NW, NH, MB>), dim3(kXcds * kRanks), dim3(64 * (NW + 4)), kOneEach, s, a);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace

size_t resident_batch_words(size_t n_embed) {
    switch (n_embed / 64) {
        case 6: return Spots<6, 1, 8>::words;
        case 8: return Spots<8, 1, 8>::words;
        case 12: return Spots<12, 2, 8>::words;
        default: return 0;
    }
}

int launch_decode_resident_batch(const ResidentArgs& a, int n_embed, hipStream_t s) {
    ZG_REQUIRE(a.batch >= 2 && a.batch <= 8, ZG_ERR_ARG, "resident decode: %d sequences", a.batch);
#define ZG_CASE(nw, nh) \
    case nw:            \
        return a.batch <= 4 ? launch<nw, nh, 4>(a, s) : launch<nw, nh, 8>(a, s);
    switch (n_embed / 64) {
        ZG_CASE(6, 1)
        ZG_CASE(8, 1)
        ZG_CASE(12, 2)
    }
#undef ZG_CASE
    set_error("resident decode: n_embed %d", n_embed);
    return ZG_ERR_UNSUPPORTED;
}

}  // namespace zg
