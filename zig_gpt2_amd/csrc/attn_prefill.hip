// attn_prefill.hip — causal scaled_dot_product_attention for all n prompt positions at once (src/ops.zig:249-307: per head
// two sgemm calls and a softmax per query row; the reference runs it once per token, src/main.zig:331-334), on the
// matrix cores at fp32 accuracy.
//
// Numerics.  q, k, v arrive as fp32 (the c_attn rows).  Every operand of a matrix product is the two-term fp16 split of its value
// times a power of two (zg_common.h split2_f16; the powers follow from the weights, launch_prefill_bounds, those of the probabilities
// from their largest, 2^kDefer), and a product a . b is the three plane products hi hi, hi lo, lo hi: every fp16 x fp16 product is exact in fp32 and the
// MFMA accumulates in fp32.  The probabilities are split the same way after the softmax.
//
// Structure.  A workgroup = four waves = four consecutive 32-query blocks of one head (128 queries) against a range of 32-key
// tiles; the K / V tiles are shared: the four waves fetch a tile as fp32 (a quarter each, coalesced 256-byte rows), split it
// once and write the planes into LDS — K as [key][64] rows with the 16-byte chunks XOR-swizzled for ds_read_b128 fragment
// reads, V as four [32 keys][16 d] sub-tiles read back TRANSPOSED by ds_read_b64_tr_b16 (the MFMA wants 8 consecutive keys
// per lane; tools/microbench/tr_read_probe.hip pins the lane map) — double buffered, one barrier per tile, the next tile's
// global loads in flight under the current tile's products.  Everything is computed transposed (S^T = K Q^T, O^T = V^T P^T):
// the query is the lane, so every per-query statistic is one register of one lane and P needs no transpose between the two
// products (the k index of an MFMA step only has to agree between its operands: the keys a lane holds after S^T are the keys
// its P fragment multiplies).  A few prompts have too few such workgroups: theirs are blocks of 32 queries (attn_prefill_block_kernel below).
#include <type_traits>

#include "prefill_epi.h"
#include "zg_kernels.h"

namespace zg {
namespace {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

constexpr int kKPlane = 32 * 128;        // one K plane of a tile: [32 keys][64 d] bf16
constexpr int kVBlock = 32 * 32 + 128;   // one 16-d block of a V plane: [32 keys][16 d] bf16, + 128 B: the two blocks a half-wave reads
                                         // in one ds_read_b64_tr_b16 then lie 288 dwords apart — the two halves of the 64 banks
constexpr int kVPlane = 4 * kVBlock;
constexpr int kLds = 2 * kPair * kKPlane + 2 * kPair * kVPlane;  // K ring + V ring, two slots each: 34816 B
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kDefer = 8.0f;  // log2 units
constexpr float kProbUp = 7.0f;  // probabilities are made 2^7 times as large: at most 2^15

// A query's 32 scores of a tile sit in two lanes (l and l ^ 32, 16 keys each): v_permlane32_swap hands every lane both halves'
// values (vdst = {lower half's, lower half's}, src0 = {upper half's, upper half's}) — no LDS crossbar, no select
__device__ __forceinline__ float both_halves_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_halves_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ f16x8 frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return __builtin_bit_cast(f16x8, u32x4{a, b, c, d}); }

// One instruction stream per wave, software-pipelined over the key tiles so that the matrix pipe and the vector ALU of a SIMD
// work side by side WITHIN a wave (the first version ran S -> softmax -> split -> PV -> staging in sequence: 48 MFMAs = 1.5 k
// cycles of a 6.4 k-cycle tile, 45 % matrix-busy with two waves per SIMD):
//   phase A   S^T(t + 1) = K(t + 1) Q^T  (12 MFMAs)   beside   exp / sum / split of tile t's scores
//   phase B   O^T += V(t)^T P(t)^T       (12 MFMAs)   beside   split + LDS write of the tiles in flight: K(t + 2), V(t + 1)
// so K runs one tile ahead of V through its own two-slot ring; one barrier per tile.  The loop body has no branch (tiles above a
// wave's diagonal are computed fully masked: its siblings need the tile anyway, the barrier would make it wait for them), only
// the rare rescale of the running maximum sits in front of phase A.
// K / V rows of (sequence b, head h), key t: 64 floats at ksrc / vsrc + b kv.stride_b + h kv.stride_h + t kv.stride_t bytes — the k / v
// columns of the qkv rows, or the head-major fp32 caches the c_attn epilogue has just appended to (then the Linear need not
// store those columns at all).
struct AttnKv {
    const char* ksrc;
    const char* vsrc;
    size_t stride_b, stride_h;
    unsigned stride_t;
};
__global__ __launch_bounds__(256, 2) void attn_prefill_pl_kernel(const float* __restrict__ qkv, uint16_t* __restrict__ out, int P, int E, const AttnKv kv,
                                                                 const int* __restrict__ exps, int coarse, unsigned long long* stamps) {
    const int exp_q = exps[PB_Q], exp_k = exps[PB_K], exp_v = exps[PB_V];
    const float s_back = ldexpf(1.0f, exp_q + exp_k);  // scores leave the products 2^-(exp_q + exp_k) times as large
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l31 = lane & 31, hl = lane >> 5;
    // grid (H, B, groups): the dispatcher hands out workgroups in linear order, x fastest — the longest groups of EVERY
    // (sequence, head) first, the short ones fill the tail (with the groups innermost the last sequence's 32-tile group started
    // when the rest of the chip was nearly done: 1.0 waves per SIMD on average instead of 2)
    const int g = (int)gridDim.z - 1 - (int)blockIdx.z;
    const int h = blockIdx.x, b = blockIdx.y;
    const int nqb = (P + 31) >> 5;
    const int n_t = min(4 * g + 4, nqb);  // key tiles
#ifdef ZG_STAMPS  // diagnostic build: every workgroup's start / end (s_memrealtime, 100 MHz) and where it ran
    const unsigned long long stamp0 = __builtin_amdgcn_s_memrealtime();
#endif
    const int qb = 4 * g + wave, tq = qb * 32 + l31;
    const size_t row0 = (size_t)b * P;
    const int ld = 3 * E;

    // Q^T fragments (B operand of S^T = K Q^T): lane = query, 8 consecutive d per 16-d slice.  Scaled by log2(e) / sqrt(64) before the
    // split (one fp32 rounding, as the reference's own alpha of sgemm, ops.zig:275) so that the softmax runs on bare v_exp_f32.
    f16x8 qf[kPair][4];
    {
        const float sc = ldexpf(0.125f * kLog2e, -exp_q);
        const float* qp = qkv + (row0 + min(tq, P - 1)) * ld + h * 64 + hl * 8;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(qp + 16 * ks), c = *reinterpret_cast<const f32x4*>(qp + 16 * ks + 4);
            uint32_t w[4][kPair];
            split2_f16(a.x * sc, a.y * sc, w[0][0], w[0][1]);
            split2_f16(a.z * sc, a.w * sc, w[1][0], w[1][1]);
            split2_f16(c.x * sc, c.y * sc, w[2][0], w[2][1]);
            split2_f16(c.z * sc, c.w * sc, w[3][0], w[3][1]);
#pragma unroll
            for (int p = 0; p < kPair; ++p) qf[p][ks] = frag(w[0][p], w[1][p], w[2][p], w[3][p]);
        }
    }

    // staging: wave w fetches keys 8 w .. 8 w + 7 of a tile.  K: 16 lanes x 16 B = one 256-byte head row per key (its LDS row is 128
    // contiguous bytes: 32 banks).  V: a 16-lane group takes ONE 16-d block of four keys, the 128 contiguous bytes that block is in
    // LDS (with K's map the four blocks of a row, 288 dwords apart, met on the same banks: a third of all LDS cycles were conflicts).
    // The loads go through a buffer descriptor — the lane's part of the address is fixed, the tile a scalar offset — and rows past
    // the last sequence read as zero (rows past P of another sequence read its first rows: finite, and masked).
    // The descriptors end behind key P - 1 of this (sequence, head): later keys read as zero (a cache row past the prompt may hold
    // anything, and 0 x NaN would poison the second product; the scores of such keys are masked anyway).
    const size_t kv_base = (size_t)b * kv.stride_b + (size_t)h * kv.stride_h;
    const unsigned kv_bytes = (unsigned)(P - 1) * kv.stride_t + 256u;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kv.ksrc + kv_base), 0, kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kv.vsrc + kv_base), 0, kv_bytes, 0x00020000);
    const int skey = wave * 8 + (lane >> 4), sd0 = (lane & 15) * 4;
    const int vkey = wave * 8 + ((lane & 15) >> 2), vd0 = 16 * (lane >> 4) + 4 * (lane & 3);
    const unsigned kvo = (unsigned)skey * kv.stride_t + (unsigned)sd0 * 4u, vvo = (unsigned)vkey * kv.stride_t + (unsigned)vd0 * 4u;
    const unsigned row4 = 4u * kv.stride_t;  // four keys further on
    auto tile_off = [&](int kt) { return (unsigned)kt * 32u * kv.stride_t; };
    auto load_k = [&](int kt, u32x4(&kr)[2]) {
        const unsigned so = tile_off(kt);
        kr[0] = __builtin_amdgcn_raw_buffer_load_b128(rk, kvo, so, 0);
        kr[1] = __builtin_amdgcn_raw_buffer_load_b128(rk, kvo + row4, so, 0);
    };
    auto load_v = [&](int kt, u32x4(&vr)[2]) {
        const unsigned so = tile_off(kt);
        vr[0] = __builtin_amdgcn_raw_buffer_load_b128(rv, vvo, so, 0);
        vr[1] = __builtin_amdgcn_raw_buffer_load_b128(rv, vvo + row4, so, 0);
    };
    char* const kring = lds;                        // [2 slots][2 planes][32 keys][64 d]
    char* const vring = lds + 2 * kPair * kKPlane;  // [2 slots][2 planes][4 d blocks][32 keys][16 d]
    const float k_up = ldexpf(1.0f, -exp_k), v_up = ldexpf(1.0f, -exp_v);
    const int kaddr = skey * 128 + (((sd0 >> 3) ^ ((skey >> 1) & 7)) << 4) + ((sd0 >> 2) & 1) * 8;  // (key + 4: same swizzle term + 2)
    const int kaddr1 = (skey + 4) * 128 + (((sd0 >> 3) ^ (((skey + 4) >> 1) & 7)) << 4) + ((sd0 >> 2) & 1) * 8;
    const int vaddr = (vd0 >> 4) * kVBlock + vkey * 32 + (vd0 & 15) * 2;
    auto store_k = [&](int slot, const u32x4(&kr)[2]) {
        char* st = kring + slot * kPair * kKPlane;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const f32x4 v = __builtin_bit_cast(f32x4, kr[j]) * k_up;
            uint32_t a[kPair], c[kPair];
            split2_f16(v.x, v.y, a[0], a[1]);
            split2_f16(v.z, v.w, c[0], c[1]);
#pragma unroll
            for (int p = 0; p < kPair; ++p) *reinterpret_cast<u32x2*>(st + p * kKPlane + (j ? kaddr1 : kaddr)) = u32x2{a[p], c[p]};
        }
    };
    auto store_v = [&](int slot, const u32x4(&vr)[2]) {
        char* st = vring + slot * kPair * kVPlane;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const f32x4 v = __builtin_bit_cast(f32x4, vr[j]) * v_up;
            uint32_t a[kPair], c[kPair];
            split2_f16(v.x, v.y, a[0], a[1]);
            split2_f16(v.z, v.w, c[0], c[1]);
#pragma unroll
            for (int p = 0; p < kPair; ++p) *reinterpret_cast<u32x2*>(st + p * kVPlane + vaddr + j * 4 * 32) = u32x2{a[p], c[p]};
        }
    };

    // fragment addresses: K rows by key = l31; V blocks by the 16-lane group (d block) and the lane's place in the 4 x 16 read
    const int koff = l31 * 128, kswz = (l31 >> 1) & 7;
    const int voff = ((lane >> 4) & 1) * kVBlock + (4 * hl + ((lane & 15) >> 2)) * 32 + (lane & 3) * 8;
    constexpr int PK[3] = {1, 0, 0}, PQ[3] = {0, 1, 0};  // the plane pairs (k or v plane, q or p plane), smallest first
    // S^T = K Q^T of the tile in K slot `slot`: ONE accumulator chain, the 12 MFMAs back to back (an MFMA that follows another one on
    // the same accumulator must follow it directly: anything issued between them costs the accumulate forwarding, ~43 cycles —
    // MI355X_MICROARCH.md, per-instruction constants).  Two chains taking the plane pairs in turn — which let this wave's own vector
    // work issue between MFMAs — cost 16 additions per tile to join and ran 1 % slower (89.6 against 90.6 us at 8 x 1023, same box):
    // the SIMD's other wave fills the matrix pipe's shadow anyway (tools/microbench/pingpong_probe.hip).
    auto s_tile = [&](int slot, f32x16& sa) __attribute__((always_inline)) {
        const char* kp = kring + slot * kPair * kKPlane;
#pragma unroll
        for (int r = 0; r < 16; ++r) sa[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            f16x8 kf[kPair];
#pragma unroll
            for (int p = 0; p < kPair; ++p) kf[p] = *reinterpret_cast<const f16x8*>(kp + p * kKPlane + koff + (((2 * ks + hl) ^ kswz) << 4));
#pragma unroll
            for (int t = 0; t < 3; ++t) sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[PK[t]], qf[PQ[t]][ks], sa, 0, 0, 0);
        }
    };

    f32x16 o0, o1;
#pragma unroll
    for (int r = 0; r < 16; ++r) o0[r] = o1[r] = 0.0f;
    float mrun = -INFINITY, lrun = 0.0f;  // reference point of the exponentials (log2 units) and running sum of this lane's query

    // ---- prologue: K(0), V(0), K(1) staged; S(0); K(2), V(1) in flight
    u32x4 kr[2], vr[2];
    f32x16 sc;
    {
        u32x4 k1[2];
        load_k(0, kr);
        load_v(0, vr);
        load_k(1, k1);
        store_k(0, kr);
        store_v(0, vr);
        store_k(1, k1);
        load_k(2, kr);
        load_v(1, vr);
        __syncthreads();
        s_tile(0, sc);
        __syncthreads();  // (K slot 0 is rewritten in the first tile's phase B: every wave must have read K(0) out)
    }

    // tile kt (slot parity SLOT = kt & 1), WITH_S = a next tile exists
    auto body = [&](auto SLOT_T, auto WITH_S_T, int kt) {
        constexpr int SLOT = decltype(SLOT_T)::value;
        constexpr bool WITH_S = decltype(WITH_S_T)::value;
        // sc[r] = log2(e) / 8 * q . k / s_back of key kt * 32 + (r & 3) + 8 (r >> 2) + 4 hl against query tq
        if (kt >= qb) {  // diagonal tile (and the tiles past it, which a sibling wave needs): position tq sees keys 0 .. tq
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = kt * 32 + (r & 3) + 8 * (r >> 2) + 4 * hl;
                sc[r] = key <= tq ? sc[r] : -INFINITY;
            }
        }
        float mx = sc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[r]);
        mx = both_halves_max(mx);
        // The reference point of the exponentials moves only when some query's maximum grew by more than 2^kDefer since it was
        // set (fp32 accumulators: probabilities up to 2^kDefer lose nothing, and their planes have the same bits) — the rescale
        // of the 32 output registers then runs on a few tiles of a row instead of all.  Everything at the old reference (O, l) is
        // rescaled at the decision, before any probability of this tile exists.
        if (__builtin_amdgcn_ballot_w64(mx * s_back > mrun + kDefer) != 0) {
            const float mnew = fmaxf(mrun, mx * s_back);
            const float corr = mnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mrun - mnew);  // (a row that has seen no key yet)
            lrun *= corr;
            mrun = mnew;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                o0[r] *= corr;
                o1[r] *= corr;
            }
        }
        // ---- phase A: the next tile's scores beside this tile's probabilities
        f32x16 sn;
        if constexpr (WITH_S) s_tile(SLOT ^ 1, sn);
        const float mref = kProbUp - fmaxf(mrun, -1e30f);  // (all keys masked so far: 2^(-inf - mref) = 0, not NaN)
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            sc[r] = __builtin_amdgcn_exp2f(fmaf(sc[r], s_back, mref));
            psum += sc[r];
        }
        lrun += both_halves_sum(psum);
        f16x8 pf[kPair][2];  // P^T fragments: registers 8 s' .. 8 s' + 7 are the lane's 8 keys of key slice s'
#pragma unroll
        for (int sp = 0; sp < 2; ++sp) {
            uint32_t w[4][kPair];
#pragma unroll
            for (int e = 0; e < 4; ++e) split2_f16(sc[8 * sp + 2 * e], sc[8 * sp + 2 * e + 1], w[e][0], w[e][1]);
#pragma unroll
            for (int p = 0; p < kPair; ++p) pf[p][sp] = frag(w[0][p], w[1][p], w[2][p], w[3][p]);
        }
        // ---- phase B: O^T += V^T P^T beside the staging of the tiles in flight.  The lane's V fragment = keys 16 s' + 4 hl + {0..3, 8..11}
        // of head dimension l31 (+ 32).
        const char* vp = vring + SLOT * kPair * kVPlane + voff;
#pragma unroll
        for (int sp = 0; sp < 2; ++sp) {
            f16x8 vf[2][kPair];
#pragma unroll
            for (int dh = 0; dh < 2; ++dh)
#pragma unroll
                for (int p = 0; p < kPair; ++p) {
                    const char* a = vp + p * kVPlane + 2 * dh * kVBlock + 16 * sp * 32;
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(a));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(a + 8 * 32));
                    vf[dh][p] = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
#pragma unroll
            for (int t = 0; t < 3; ++t) {  // the two halves of the head dimension in turn: two accumulator chains
                o0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[0][PK[t]], pf[PQ[t]][sp], o0, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[1][PK[t]], pf[PQ[t]][sp], o1, 0, 0, 0);
            }
        }
        store_k(SLOT, kr);       // K(kt + 2): the slot K(kt) left in the previous tile's phase A
        store_v(SLOT ^ 1, vr);   // V(kt + 1): the slot V(kt - 1) left in the previous tile's phase B
        load_k(kt + 3, kr);
        load_v(kt + 2, vr);
        if constexpr (WITH_S) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = sn[r];
        }
        __syncthreads();
    };
    {
        using T = std::true_type;
        using F = std::false_type;
        int i = 0;
        for (; i + 2 < n_t; i += 2) {
            body(std::integral_constant<int, 0>{}, T{}, i);
            body(std::integral_constant<int, 1>{}, T{}, i + 1);
        }
        if (n_t - i == 2) {
            body(std::integral_constant<int, 0>{}, T{}, i);
            body(std::integral_constant<int, 1>{}, F{}, i + 1);
        } else {
            body(std::integral_constant<int, 0>{}, F{}, i);
        }
    }
#ifdef ZG_STAMPS
    if (tid == 0 && stamps != nullptr) {
        unsigned long long* st = stamps + 4 * ((size_t)(blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x);
        st[0] = stamp0;
        st[1] = __builtin_amdgcn_s_memrealtime();
        st[2] = (unsigned long long)__builtin_amdgcn_s_getreg((4 << 0) | (0 << 6) | (31 << 11)) |         // HW_REG_HW_ID
                ((unsigned long long)__builtin_amdgcn_s_getreg((20 << 0) | (0 << 6) | (31 << 11)) << 32);  // HW_REG_XCC_ID
        st[3] = (unsigned long long)n_t;
    }
#endif
    if (qb >= nqb || tq >= P) return;

    // O^T: the lane holds d = (r & 3) + 8 (r >> 2) + 4 hl (+ 32 in o1) of its query
    const float inv = 1.0f / lrun;  // softmax divides by the sum (ops.zig:239); the c_proj GEMM takes the rows as planes (a mean of v's: they leave with v's exponent)
    uint16_t* hi = out + (row0 + tq) * kPair * E + h * 64;
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
        const int d = 8 * gq + 4 * hl;
        store_split4(hi + d, E, f32x4{o0[gq * 4] * inv, o0[gq * 4 + 1] * inv, o0[gq * 4 + 2] * inv, o0[gq * 4 + 3] * inv}, 0, coarse);
        store_split4(hi + 32 + d, E, f32x4{o1[gq * 4] * inv, o1[gq * 4 + 1] * inv, o1[gq * 4 + 2] * inv, o1[gq * 4 + 3] * inv}, 0, coarse);
    }
}

// A workgroup per query block of 32 rows of one (sequence, head): its waves take the block's key tiles in turn, each straight from memory into
// fragments (a lane has a key of K, a head dimension of V), and their (m, l, O) meet in the LDS.  No barrier before that, no wave that
// waits for another's staging, four times as many workgroups: what bounds prompts of a few sequences is how little of the chip the groups of
// 128 queries fill and one tile's chain of latencies behind another's.  But every block splits the keys and values it sees again, four times as often.
// us a launch, 12 heads, beside the kernel above (its key ranges cut over workgroups, with the launch that merged them): 1 x 64 tokens 4.9 : 7.0,
// 1 x 300 8.5 : 16.0, 1 x 1023 21 : 27, 4 x 300 13 : 21, 8 x 150 9.2 : 18.8, 2 x 1023 31 : 36; 25 heads 1 x 400 12.4 : 20.6, 2 x 400 17 : 23.
// Eight waves a block are slower from 1 x 300 on (9.0; 2 x 1023 36).
constexpr int kBlockWaves = 4;
__global__ __launch_bounds__(kBlockWaves * 64, 2) void attn_prefill_block_kernel(const float* __restrict__ qkv, uint16_t* __restrict__ out, int P, int E, const AttnKv kv,
                                                                        const int* __restrict__ exps, int coarse) {
    constexpr int PITCH = 68;  // floats of a query's row of a wave's partial sums
    __shared__ __attribute__((aligned(16))) float s_part[kBlockWaves * 32 * PITCH];
    __shared__ float s_m[kBlockWaves * 32], s_l[kBlockWaves * 32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l31 = lane & 31, hl = lane >> 5;
    const int h = blockIdx.x, b = blockIdx.y, qb = (int)gridDim.z - 1 - (int)blockIdx.z, tq = qb * 32 + l31;  // (the longest first)
    const size_t row0 = (size_t)b * P;
    const int exp_q = exps[PB_Q], exp_k = exps[PB_K], exp_v = exps[PB_V];
    // (the descriptors end behind key P - 1: later keys read as zero)
    const size_t kv_base = (size_t)b * kv.stride_b + (size_t)h * kv.stride_h;
    const unsigned kv_bytes = (unsigned)(P - 1) * kv.stride_t + 256u;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kv.ksrc + kv_base), 0, kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kv.vsrc + kv_base), 0, kv_bytes, 0x00020000);
    const unsigned kvo = (unsigned)l31 * kv.stride_t + (unsigned)hl * 32u, vvo = (unsigned)(4 * hl) * kv.stride_t + (unsigned)l31 * 4u;
    u32x4 kr[8];
    uint32_t vr[2][2][8];  // [16 keys][d, d + 32][key of the fragment]
    auto load_k = [&](int kt) {
        const unsigned so = (unsigned)kt * 32u * kv.stride_t;
#pragma unroll
        for (int i = 0; i < 8; ++i) kr[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, kvo + 64u * (i >> 1) + 16u * (i & 1), so, 0);
    };
    auto load_v = [&](int kt) {
#pragma unroll
        for (int sp = 0; sp < 2; ++sp)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned so = (unsigned)(kt * 32 + 16 * sp + (j & 3) + 8 * (j >> 2)) * kv.stride_t;
#pragma unroll
                for (int dh = 0; dh < 2; ++dh) vr[sp][dh][j] = __builtin_amdgcn_raw_buffer_load_b32(rv, vvo + 128u * dh, so, 0);
            }
    };
    f32x4 qr[8];
    {
        const float* qp = qkv + (row0 + min(tq, P - 1)) * 3 * E + h * 64 + hl * 8;
#pragma unroll
        for (int i = 0; i < 8; ++i) qr[i] = *reinterpret_cast<const f32x4*>(qp + 16 * (i >> 1) + 4 * (i & 1));
    }
    load_k(min(wave, qb));
    load_v(min(wave, qb));
    const float s_back = ldexpf(1.0f, exp_q + exp_k), k_up = ldexpf(1.0f, -exp_k), v_up = ldexpf(1.0f, -exp_v), q_up = ldexpf(0.125f * kLog2e, -exp_q);
    // eight values times a power of two -> their two planes
    auto planes = [](const float(&x)[8], float up, f16x8(&to)[kPair]) {
        uint32_t w[4][kPair];
#pragma unroll
        for (int e = 0; e < 4; ++e) split2_f16(x[2 * e] * up, x[2 * e + 1] * up, w[e][0], w[e][1]);
#pragma unroll
        for (int p = 0; p < kPair; ++p) to[p] = frag(w[0][p], w[1][p], w[2][p], w[3][p]);
    };
    f16x8 qf[4][kPair];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const f32x4 a = qr[2 * ks], c = qr[2 * ks + 1];
        const float x[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
        planes(x, q_up, qf[ks]);
    }
    constexpr int PK[3] = {1, 0, 0}, PQ[3] = {0, 1, 0};  // the plane pairs, smallest first
    f32x16 o0, o1;
#pragma unroll
    for (int r = 0; r < 16; ++r) o0[r] = o1[r] = 0.0f;
    float mrun = -INFINITY, lrun = 0.0f;
    for (int kt = wave; kt <= qb; kt += kBlockWaves) {
        f32x16 sc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const f32x4 a = __builtin_bit_cast(f32x4, kr[2 * ks]), c = __builtin_bit_cast(f32x4, kr[2 * ks + 1]);
            const float x[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
            f16x8 kf[kPair];
            planes(x, k_up, kf);
#pragma unroll
            for (int t = 0; t < 3; ++t) sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[PK[t]], qf[ks][PQ[t]], sc, 0, 0, 0);
        }
        if (kt + kBlockWaves <= qb) load_k(kt + kBlockWaves);
        if (kt == qb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = kt * 32 + (r & 3) + 8 * (r >> 2) + 4 * hl <= tq ? sc[r] : -INFINITY;
        }
        float mx = sc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[r]);
        mx = both_halves_max(mx);
        if (__builtin_amdgcn_ballot_w64(mx * s_back > mrun + kDefer) != 0) {
            const float mnew = fmaxf(mrun, mx * s_back);
            const float corr = mnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mrun - mnew);
            lrun *= corr;
            mrun = mnew;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                o0[r] *= corr;
                o1[r] *= corr;
            }
        }
        const float mref = kProbUp - fmaxf(mrun, -1e30f);
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            sc[r] = __builtin_amdgcn_exp2f(fmaf(sc[r], s_back, mref));
            psum += sc[r];
        }
        lrun += both_halves_sum(psum);
#pragma unroll
        for (int sp = 0; sp < 2; ++sp) {
            f16x8 pf[kPair], vf[2][kPair];
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = sc[8 * sp + j];
            planes(x, 1.0f, pf);
#pragma unroll
            for (int dh = 0; dh < 2; ++dh) {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = __uint_as_float(vr[sp][dh][j]);
                planes(x, v_up, vf[dh]);
            }
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                o0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[0][PK[t]], pf[PQ[t]], o0, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[1][PK[t]], pf[PQ[t]], o1, 0, 0, 0);
            }
        }
        if (kt + kBlockWaves <= qb) load_v(kt + kBlockWaves);
    }
    // O^T: the lane holds d = (r & 3) + 8 (r >> 2) + 4 hl (+ 32 in o1) of its query.  (a wave without a tile: m = -inf, nothing else)
    float* mine = s_part + (wave * 32 + l31) * PITCH + 4 * hl;
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
        *reinterpret_cast<f32x4*>(mine + 8 * gq) = f32x4{o0[gq * 4], o0[gq * 4 + 1], o0[gq * 4 + 2], o0[gq * 4 + 3]};
        *reinterpret_cast<f32x4*>(mine + 32 + 8 * gq) = f32x4{o1[gq * 4], o1[gq * 4 + 1], o1[gq * 4 + 2], o1[gq * 4 + 3]};
    }
    if (hl == 0) {
        s_m[wave * 32 + l31] = mrun;
        s_l[wave * 32 + l31] = lrun;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 8 / kBlockWaves; ++it) {
        const int q = it * 4 * kBlockWaves + (tid >> 4), d = (tid & 15) * 4, t = qb * 32 + q;
        float m = s_m[q], l = 0.0f;
#pragma unroll
        for (int w = 1; w < kBlockWaves; ++w) m = fmaxf(m, s_m[w * 32 + q]);
        f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < kBlockWaves; ++w) {
            const float c = __builtin_amdgcn_exp2f(s_m[w * 32 + q] - m);
            l = fmaf(c, s_l[w * 32 + q], l);
            o += *reinterpret_cast<const f32x4*>(s_part + (w * 32 + q) * PITCH + d) * c;
        }
        if (t < P) store_split4(out + (row0 + t) * kPair * E + h * 64 + d, E, o * (1.0f / l), 0, coarse);
    }
}

}  // namespace

// out[M][kPair E] = planes of (causal attention of the q / k / v columns of qkv[M][3E]), M = B P rows ordered (b, t).
// k_cache / v_cache != null: K and V come from the head-major fp32 caches [b][h][ctx][64] (positions 0 .. P - 1 just appended
// by the c_attn epilogue) instead of the k / v columns of qkv.  by_groups (test hook): groups of 128 queries at any size.  stamps: diagnostic builds.
int launch_attn_prefill(const float* qkv, uint16_t* out, int B, int P, int E, int H, const float* k_cache, const float* v_cache, int ctx, const int* exps, int coarse,
                        hipStream_t s, bool by_groups, unsigned long long* stamps) {
    ZG_REQUIRE(E == H * 64, ZG_ERR_UNSUPPORTED, "attention prefill: head_dim must be 64 (n_embed %d, %d heads)", E, H);
    const int nqb = (P + 31) / 32, ng = (nqb + 3) / 4;
    ZG_REQUIRE(nqb < 65536, ZG_ERR_UNSUPPORTED, "attention prefill: %d positions", P);
    AttnKv kv;
    if (k_cache != nullptr) {  // head-major fp32 caches [b][h][ctx][64]
        kv = AttnKv{reinterpret_cast<const char*>(k_cache), reinterpret_cast<const char*>(v_cache), (size_t)H * ctx * 256, (size_t)ctx * 256, 256u};
    } else {  // the k / v columns of the qkv rows
        kv = AttnKv{reinterpret_cast<const char*>(qkv + E), reinterpret_cast<const char*>(qkv + 2 * E), (size_t)P * 3 * E * 4, (size_t)256, (unsigned)(3 * E * 4)};
    }
    ZG_REQUIRE((size_t)P * kv.stride_t < ((size_t)1 << 31), ZG_ERR_SHAPE, "attention prefill: rows beyond a 32-bit buffer descriptor");
    // Groups of 128 queries once there is one for every compute unit; below, blocks of 32.  us, 12 heads, groups : blocks: 8 x 300 (288 groups)
    // 18.1 : 18.6, 3 x 1023 (288) 39 : 40, 8 x 500 (384) 27 : 33; 25 heads 2 x 700 (300) 29 : 32.  240 groups of 4 x 600 31 : 26.
    if (!by_groups && (long)B * H * ng < 256)
        attn_prefill_block_kernel<<<dim3(H, B, nqb), kBlockWaves * 64, 0, s>>>(qkv, out, P, E, kv, exps, coarse);
    else
        attn_prefill_pl_kernel<<<dim3(H, B, ng), 256, kLds, s>>>(qkv, out, P, E, kv, exps, coarse, stamps);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace zg
