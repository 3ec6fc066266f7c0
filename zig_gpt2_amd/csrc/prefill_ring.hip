// prefill_ring.hip — the Linears of the whole-prompt pass (src/ops.zig:21-46 for M = batch x prompt rows) where the large tiles leave the chip
// idle: prompts of some hundred rows.
//
// A = the activation planes [M][2 K] (hi | lo), W = the one plane [N][K] of a bf16 weight, or the two [2][N][K] of an fp32 weight (zg_common.h split2_f16).
// All the products of a K step of 64 columns (two; four, or five with a third plane; three of an op-tier Linear in one piece, four of one in slices) are made from ONE staging of the planes, where the 128-row kernels of prefill.hip
// walk an fp32 weight in two passes that each stage the activations again and meet in slabs.
// What bounds it: a compute unit takes in some 30 bytes a clock (32 KB a step of a 64 x 64 tile of an fp32 weight: 1100 clocks, beside 384 or 512 of
// products).  So tiles are small while they are few, and no operand is staged twice for one tile.  The planes arrive by LDS-DMA in a ring of
// K steps; a step costs one barrier; its fragments were read beside the products of the step before.  The leading products of a step are a sum
// of their own, added to the steps' before it beside the products of the next, so that neither they nor the small ones are rounded at the size of
// the whole.  Tiles of 128 x 128 (fp32 weights, some thousand rows) stage 64 KB for what four tiles of 64 x 64 stage 128 KB for; their leading
// products are a sum of four steps (a second set has no registers), and what the epilogue needs is fetched behind the products.  us, 768 columns,
// 128 x 64 : 128 x 128: 1000 x 3072 33 : 28, 1500 x 2304 37 : 30; 3072 columns 1500 x 768 in slices, with the reduction 53 : 39; 2000 x 2304 (two rounds
// for three) 50 : 53.  With one plane of a bf16 weight they are no faster than the 128-row kernel of prefill.hip (1000 x 3072 22 : 21): not built.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "prefill_epi.h"
#include "zg_kernels.h"
#include "zg_once.h"

namespace zg {

namespace {

typedef __attribute__((address_space(3))) char* lds_at_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kBk = 64, kRow = 128, kCh = 8;  // columns of K of a step; bytes and 16-byte chunks of a row of them

// (written here, not by the builtin: the compiler would wait for every request in flight in front of any read of the LDS.  m0: the address of
// the wave's 1 KB piece; the wait state is what a request needs behind a write of m0)
__device__ __forceinline__ void dma_16(unsigned lds, const u32x4& rsrc, unsigned v_off, unsigned s_off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(v_off), "s"(rsrc), "s"(s_off) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void arrive() {  // N requests may be in flight; what was read of the LDS is here; every wave has come this far
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ u32x4 rsrc_of(const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, 0x80000000u, 0x00020000u};
}

// PF_LINEAR: the fp32 operands themselves, for outputs that are not finite (plain_sum); ldc is then the number of columns, N the same in whole 64s
struct RawRows {
    const float *x, *w;
};

// 2 x 2 waves of TM x TN 32 x 32 tiles; NW planes of the weight (3: the last bits of an fp32 one as well); ST steps in the ring.  blockIdx.y: the K slice (PF_PARTIAL, PF_LINEAR_PART).
// ALL: a prompt's fp32 Linears make the product of the two second terms as well.  With three products short sums, the rest of which is near to exact, left a small
// model's logits further from 64 bits than six of three bf16 terms; the fourth hides beside the staging (300 rows 10.3 -> 10.8 us, 14.2 -> 14.2, 13.9 ->
// 14.1; 1 x 300 tokens 850 -> 866).  Models of fewer than 512 columns: few rows have the weight's last bits as a third plane, more rows NEAR, totals that keep what an addition
// rounds away (both are too dear: 337 us for 1 x 9 tokens of the char model, where a third plane alone takes 296, NEAR alone 306 and three exact terms took 295).
// Errors against 64 bits of that model, twelve weights by eight prompts, e-7, three exact terms / NEAR / third plane: 1 x 9 tokens 2.92 / 2.97 / 2.91, 2 x 20 3.02 / 3.00 / 2.95,
// 1 x 64 2.91 / 2.90 / 2.79, 3 x 40 2.99 / 2.96 / 2.87, 1 x 130 3.03 / 2.79 / 2.75.
template <int EPI, int TM, int TN, int NW, int ST, bool NEAR>
__global__ __launch_bounds__(256, 1) void prefill_ring_kernel(const uint16_t* A, const uint16_t* W, const int* ex_a, const int* ex_w, const float* bias, int M, int N, int K, int n_sp_each,
                                                              void* C, int ldc, const PrefillQkv qa, const PlaneOut po, const RawRows raw, const SplitSeen seen) {
    // (in front of C what the first loads need: the leading arguments are in registers when a wave starts.  n_sp_each: K slices, and whether A's rows have exponents of their own)
    const int n_sp = n_sp_each >> 1;
    const bool a_each = n_sp_each & 1;
    constexpr int BM = 64 * TM, BN = 64 * TN, PA = BM / 32, PB = BN / 32, A_PLANE = BM * kRow, B_PLANE = BN * kRow, SLOT = kPair * A_PLANE + NW * B_PLANE;
    constexpr int REQ = kPair * PA + NW * PB;  // 1 KB pieces (8 rows) a wave asks for in a step
    extern __shared__ __attribute__((aligned(1024))) char s_ring[];
    const unsigned lds0 = (unsigned)(unsigned long)(lds_at_t)s_ring;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wy = wave >> 1, wx = wave & 1;
    // workgroups go round the eight XCDs: each gets a run of the tiles, row tiles of a column tile next to each other (the weights are read once)
    const int tiles_m = (M + BM - 1) / BM, n_tiles = tiles_m * ((N + BN - 1) / BN), q8 = n_tiles >> 3, r8 = n_tiles & 7, xcd = blockIdx.x & 7;
    const int tile = xcd * q8 + min(xcd, r8) + (int)(blockIdx.x >> 3);
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
    const int in_row = lane >> 3, chunk = (lane & 7) ^ in_row;  // (every eighth row the swizzle repeats)
    const u32x4 ra = rsrc_of(A), rb = rsrc_of(W);
    unsigned va[PA], vb[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) va[i] = (unsigned)min(m0 + (wave + 4 * i) * 8 + in_row, M - 1) * (unsigned)(kPair * K) * 2u + chunk * 16u;  // (rows beyond the edge: never stored)
#pragma unroll
    for (int i = 0; i < PB; ++i) vb[i] = (unsigned)(TN == 1 ? n0 + (wave + 4 * i) * 8 + in_row : min(n0 + (wave + 4 * i) * 8 + in_row, N - 1)) * (unsigned)K * 2u + chunk * 16u;
    const int nk = K / kBk, t0 = nk * (int)blockIdx.y / n_sp, steps = nk * ((int)blockIdx.y + 1) / n_sp - t0;
    auto request = [&](int slot, int s) {
        const unsigned off = (unsigned)(t0 + min(s, steps - 1)) * kRow, to = lds0 + slot * SLOT + wave * 1024;
#pragma unroll
        for (int p = 0; p < kPair; ++p)
#pragma unroll
            for (int i = 0; i < PA; ++i) dma_16(to + p * A_PLANE + i * 4096, ra, va[i], off + (unsigned)p * (unsigned)K * 2u);
#pragma unroll
        for (int p = 0; p < NW; ++p)
#pragma unroll
            for (int i = 0; i < PB; ++i) dma_16(to + kPair * A_PLANE + p * B_PLANE + i * 4096, rb, vb[i], off + (unsigned)p * (unsigned)N * (unsigned)K * 2u);
    };
    constexpr bool ALL = NW >= 2 && EPI != PF_LINEAR;
    constexpr int NL = TN == 2 ? 1 : 2;  // leading products by the step's parity, or (registers) one sum of four steps
    f32x16 lead[NL][TM][TN], small[TM][TN], total[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) lead[0][i][j][e] = lead[NL - 1][i][j][e] = small[i][j][e] = total[i][j][e] = 0.0f;
    auto gather = [&](f32x16& to, f32x16& from, f32x16& rest) {  // NEAR: what the addition rounds away joins the small products
        if constexpr (NEAR) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float t = to[e], y = from[e], sum = t + y, z = sum - t;
                rest[e] += (t - (sum - z)) + (y - z);
                to[e] = sum;
            }
        } else to += from;
#pragma unroll
        for (int e = 0; e < 16; ++e) from[e] = 0.0f;
    };
    const int fr = lane & 31, kh = lane >> 5, fswz = fr & 7;
    u32x4 af[2][kCh / 2][kPair][TM], bf[2][kCh / 2][NW][TN];  // of the step that is multiplied, and of the one behind it on its way
    auto read = [&](auto b, int slot) {
        const char* base = s_ring + slot * SLOT;
#pragma unroll
        for (int kk = 0; kk < kCh / 2; ++kk) {
            const int c = ((2 * kk + kh) ^ fswz) * 16;
#pragma unroll
            for (int p = 0; p < NW; ++p)
#pragma unroll
                for (int j = 0; j < TN; ++j) bf[b][kk][p][j] = *reinterpret_cast<const u32x4*>(base + kPair * A_PLANE + p * B_PLANE + ((wx * TN + j) * 32 + fr) * kRow + c);
#pragma unroll
            for (int p = 0; p < kPair; ++p)
#pragma unroll
                for (int i = 0; i < TM; ++i) af[b][kk][p][i] = *reinterpret_cast<const u32x4*>(base + p * A_PLANE + ((wy * TM + i) * 32 + fr) * kRow + c);
        }
    };
    // (the operands change places: an accumulator's registers are then runs of four columns of a row)
    auto multiply = [&](auto b) {
        auto one = [&](f32x16& acc, int kk, int pa, int pw, int i, int j) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, bf[b][kk][pw][j]), __builtin_bit_cast(f16x8, af[b][kk][pa][i]), acc, 0, 0, 0);
        };
        constexpr int now = NL == 2 ? (int)decltype(b)::value : 0;
        if constexpr (NL == 2)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) gather(total[i][j], lead[1 - now][i][j], small[i][j]);
#pragma unroll
        for (int kk = 0; kk < kCh / 2; ++kk)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (ALL) one(small[i][j], kk, 1, 1, i, j);
                    one(small[i][j], kk, 1, 0, i, j);
                    one(lead[now][i][j], kk, 0, 0, i, j);
                    if constexpr (NW >= 2) one(small[i][j], kk, 0, 1, i, j);
                    if constexpr (NW == 3) one(small[i][j], kk, 0, 2, i, j);
                }
    };
    // what the epilogue needs besides the sums, on its way before the requests
    const int cc = (lane & 7) * 4, n_w = n0 + wx * TN * 32 + cc;
    i32x4 col_exp[TN];
    f32x4 bv[TN];
    int row_exp[TM][4];
    auto fetch_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = TN == 1 ? n_w : min(n_w + 32 * j, N - 4);  // (N: whole pieces of 32)
            col_exp[j] = *reinterpret_cast<const i32x4*>(ex_w + n);
            bv[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (EPI == PF_LINEAR) {
                if (bias)
#pragma unroll
                    for (int e = 0; e < 4; ++e) bv[j][e] = bias[min(n + e, ldc - 1)];
            } else if (EPI != PF_PARTIAL && EPI != PF_LINEAR_PART && bias) {
                bv[j] = *reinterpret_cast<const f32x4*>(bias + n);
            }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r8i = 0; r8i < 4; ++r8i) row_exp[i][r8i] = ex_a[a_each ? min(m0 + (wy * TM + i) * 32 + 8 * r8i + (lane >> 3), M - 1) : 0];
    };
    if (TN == 1) fetch_scales();  // (larger tiles have no registers for them beside the products)
#pragma unroll
    for (int s = 0; s < ST; ++s) request(s, s);
    int out_exp = 0;  // the epilogue's arguments, fetched under the first requests
    if (EPI == PF_GELU_SPLIT) {
        out_exp = *po.exp;
        ZG_PIN(out_exp);
    }
    ZG_PIN(C); ZG_PIN(ldc);
    if (EPI == PF_QKV) {
        ZG_PIN(qa.P); ZG_PIN(qa.E); ZG_PIN(qa.H); ZG_PIN(qa.ctx); ZG_PIN(qa.kv_mode); ZG_PIN(qa.kv_lo); ZG_PIN(qa.k_cache); ZG_PIN(qa.v_cache);
    }
    if ((EPI == PF_LINEAR || EPI == PF_LINEAR_PART) && seen_refused(seen)) {  // (every wave alike; its requests still write the ring)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), said to the compiler: with scalar loads in flight it would wait for all fragments at once
    arrive<(ST - 1) * REQ>();
    read(std::integral_constant<int, 0>(), 0);
    int slot = 0, s = 0;
    // Step s: its fragments have been read, so its slot takes step s + ST; those of s + 1 are read beside its products.
    auto body = [&](auto b) {
        constexpr int other = 1 - decltype(b)::value;
        arrive<(ST - 2) * REQ>();
        request(slot, s + ST);
        slot = slot == ST - 1 ? 0 : slot + 1;
        __builtin_amdgcn_sched_barrier(0);
        read(std::integral_constant<int, other>(), slot);
        multiply(b);
        constexpr int products = kCh / 2 * TM * TN * (NW + 1 + ALL), reads = kCh / 2 * (kPair * TM + NW * TN);
#pragma unroll
        for (int x = 0; x < products; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x100, (reads + products - 1) / products, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (NL == 1 && other == 0 && (s & 2))
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) gather(total[i][j], lead[0][i][j], small[i][j]);
        ++s;
    };
    for (int pairs = steps >> 1; pairs > 0; --pairs) {
        body(std::integral_constant<int, 0>());
        body(std::integral_constant<int, 1>());
    }
    if (steps & 1) body(std::integral_constant<int, 0>());
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the requests behind the last step still write the ring)
    if (TN > 1) fetch_scales();
    if constexpr (NEAR)
#pragma unroll
        for (int ij = 0; ij < TM * TN; ++ij)
#pragma unroll
            for (int l = 0; l < NL; ++l) gather(total[ij / TN][ij % TN], lead[l][ij / TN][ij % TN], small[ij / TN][ij % TN]);

    // element e of a 32 x 32 tile: column 8 (e / 4) + 4 (lane / 32) + e % 4, row lane % 32.  Every wave turns its rows in an image of its own
    // (its accesses to the LDS are in order), so that eight lanes store 128 bytes of a row.
    constexpr int PITCH = 32 * 4 + 16;
    static_assert(4 * 32 * PITCH <= SLOT, "the images fit the ring");
    char* img = s_ring + wave * 32 * PITCH;
#pragma unroll
    for (int ij = 0; ij < TM * TN; ++ij) {
        const int i = ij / TN, j = ij % TN, n = n_w + 32 * j;
        if (TN > 1 && n >= N) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4 v;  // (of the two leading sums one is in the total already, and zero)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (total[i][j][4 * g + e] + (NL == 2 ? lead[0][i][j][4 * g + e] + lead[NL - 1][i][j][4 * g + e] : lead[0][i][j][4 * g + e])) + small[i][j][4 * g + e];
            *reinterpret_cast<f32x4*>(img + fr * PITCH + (8 * g + 4 * kh) * 4) = v;
        }
#pragma unroll
        for (int r8i = 0; r8i < 4; ++r8i) {
            const int r = 8 * r8i + (lane >> 3), m = m0 + (wy * TM + i) * 32 + r;
            f32x4 v = *reinterpret_cast<const f32x4*>(img + r * PITCH + cc * 4);
            if (m >= M) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ldexpf(v[e], row_exp[i][r8i] + col_exp[j][e]) + bv[j][e];
            if constexpr (EPI == PF_GELU_SPLIT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gelu_fast(v[e]);
                store_split4(reinterpret_cast<uint16_t*>(C) + (size_t)m * kPair * N + n, N, v, out_exp, po.coarse);
            } else if constexpr (EPI == PF_LINEAR) {
                float* y = reinterpret_cast<float*>(C) + (size_t)m * ldc + n;
                if ((ldc & 3) == 0 && n < ldc) {
                    *reinterpret_cast<f32x4*>(y) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < ldc) y[e] = v[e];
                }
                if (odd(v[0]) + odd(v[1]) + odd(v[2]) + odd(v[3]) > 0.0f)
#pragma unroll 1
                    for (int e = 0; e < 4; ++e)
                        if (n + e < ldc && odd(v[e]) > 0.0f) y[e] = plain_sum(raw.x + (size_t)m * K, raw.w + (size_t)(n + e) * K, K) + bv[j][e];
            } else if constexpr (EPI == PF_PARTIAL || EPI == PF_LINEAR_PART) {  // C: slabs [n_sp][M][N]
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + ((size_t)blockIdx.y * M + m) * N + n) = v;
            } else {
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + (size_t)m * ldc + n) = v;
                if constexpr (EPI == PF_QKV) qkv_cache_store(qa, m, n, v);
            }
        }
    }
}

template <int EPI, int TM, int TN, int NW, int ST, bool NEAR = false>
int launch_ring(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int ldc, int n_sp, const PrefillQkv& qa, const PlaneOut& po, hipStream_t s,
                const RawRows& raw = RawRows{}, const SplitSeen& seen = SplitSeen{}) {
    constexpr int LDS = ST * (kPair * 64 * TM + NW * 64 * TN) * kRow;
    static_assert(LDS <= 160 * 1024, "the ring fits the LDS");
    static OncePerDevice raised;
    int device = 0;
    ZG_HIP(hipGetDevice(&device));
    ZG_TRY(raised.run(device, []() -> int {
        ZG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_ring_kernel<EPI, TM, TN, NW, ST, NEAR>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        return ZG_OK;
    }));
    const int tiles = ((M + 64 * TM - 1) / (64 * TM)) * ((N + 64 * TN - 1) / (64 * TN));
    prefill_ring_kernel<EPI, TM, TN, NW, ST, NEAR><<<dim3(tiles, n_sp), 256, LDS, s>>>(A.p, W.p, A.exp, W.exps, bias, M, N, K, 2 * n_sp + A.each, C, ldc, qa, po, raw, seen);
    note_kernel("prefill_ring_kernel<%d, %d>", TM, NW);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

template <int EPI>
int launch_ring_epi(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int ldc, int tm, int n_sp, const PrefillQkv& qa, const PlaneOut& po,
                    hipStream_t s, const SplitSeen& seen = SplitSeen{}) {
    if constexpr (EPI != PF_LINEAR_PART)
        if (W.rest && tm == 1) return launch_ring<EPI, 1, 1, 3, 4>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s);
    if (W.planes == 2 && std::min(N, K) < (int)kNearColumns)
        return tm == 1   ? launch_ring<EPI, 1, 1, 2, 4, true>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen)
               : tm == 2 ? launch_ring<EPI, 2, 1, 2, 3, true>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen)
                         : launch_ring<EPI, 2, 2, 2, 2, true>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen);
    if (W.planes == 2)
        return tm == 1   ? launch_ring<EPI, 1, 1, 2, 4>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen)
               : tm == 2 ? launch_ring<EPI, 2, 1, 2, 3>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen)
                         : launch_ring<EPI, 2, 2, 2, 2>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s, RawRows{}, seen);
    if constexpr (EPI == PF_LINEAR_PART) ZG_REQUIRE(false, ZG_ERR_ARG, "linear: %d planes", W.planes);
    else return tm == 1 ? launch_ring<EPI, 1, 1, 1, 5>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s) : launch_ring<EPI, 2, 1, 1, 3>(A, W, bias, C, M, N, K, ldc, n_sp, qa, po, s);
}

// the slabs [n_sp][M][Np] of a Linear added, and its bias: a thread four columns of a row
__global__ __launch_bounds__(256) void linear_ring_finish_kernel(const float* __restrict__ slabs, int n_sp, int M, int Np, const float* __restrict__ bias, float* __restrict__ Y, int N,
                                                                 const float* __restrict__ X, const float* __restrict__ W, int K, const SplitSeen seen) {
    if (seen_plan(seen).refused) return;
    const int n4 = (N + 3) / 4;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)M * n4) return;
    const int m = (int)(i / n4), n = (int)(i % n4) * 4;
    const float* p = slabs + (size_t)m * Np + n;
    const size_t slab = (size_t)M * Np;
    f32x4 v = *reinterpret_cast<const f32x4*>(p);
    for (int s0 = 1; s0 < n_sp; s0 += 4) {
        f32x4 t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const f32x4*>(p + (size_t)min(s0 + u, n_sp - 1) * slab);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s0 + u < n_sp) v += t[u];
    }
    float* y = Y + (size_t)m * N + n;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (n + e >= N) break;
        const float b = bias ? bias[n + e] : 0.0f, sum = v[e] + b;
        y[e] = odd(v[e]) > 0.0f ? plain_sum(X + (size_t)m * K, W + (size_t)(n + e) * K, K) + b : sum;
    }
}

}  // namespace

namespace {
size_t whole(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
size_t whole64(size_t n) { return (n + 63) / 64 * 64; }
// tiles of form t: 64 x 64, 128 x 64, 128 x 128
long ring_tiles(long M, long N, int t) { return (M + (t == 1 ? 63 : 127)) / (t == 1 ? 64 : 128) * ((N + (t == 3 ? 127 : 63)) / (t == 3 ? 128 : 64)); }
// us of a K step of two weight planes, by form.  A round of workgroups costs 4.5 us besides: 768 columns in one round 11.7, 17 and 27.
constexpr double kStepUs[4] = {0.0, 0.55, 1.02, 1.85};
}  // namespace

size_t linear_ring_scratch(size_t M, size_t N, size_t K, int n_sp) {
    const size_t Np = whole64(N);
    return whole(M * K * 4) + whole(Np * K * 4) + whole(M * 4) + whole(Np * 4) + whole((M + N) * 4) + (n_sp > 1 ? whole((size_t)n_sp * M * Np * 4) : 0);
}

static std::atomic<unsigned long long> g_linear_ring_launches{0};
unsigned long long linear_ring_launch_count() { return g_linear_ring_launches.load(std::memory_order_relaxed); }

int launch_linear_ring(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, int tm, int n_sp, char* scratch, SplitSeen* in, hipStream_t s) {
    const int Np = (int)whole64(N);
    ZG_REQUIRE(M > 0 && N > 0 && K % kBk == 0 && n_sp >= 1 && n_sp <= K / kBk && tm >= 1 && tm <= 3 && (size_t)M * K * 4 < ((size_t)1 << 31) && (size_t)Np * K * 4 < ((size_t)1 << 31),
               ZG_ERR_UNSUPPORTED, "linear: %d x %d x %d", M, N, K);
    uint16_t *xp = reinterpret_cast<uint16_t*>(scratch), *wp = reinterpret_cast<uint16_t*>(scratch += whole((size_t)M * K * 4));
    int *xe = reinterpret_cast<int*>(scratch += whole((size_t)Np * K * 4)), *we = reinterpret_cast<int*>(scratch += whole((size_t)M * 4));
    in->marks = reinterpret_cast<int*>(scratch += whole((size_t)Np * 4));
    float* slabs = reinterpret_cast<float*>(scratch += whole(((size_t)M + N) * 4));
    const SplitSeen seen = *in;
    // (the weight's rows beyond N hold whatever the scratch held: their columns are never stored)
    ZG_TRY(launch_split2(Split2Job{X, xp, xe, M}, Split2Job{W, wp, we, N, (size_t)Np * K}, K, s, seen));
    const PrefillA A{xp, xe, true};
    const PrefillW P{wp, we, 2};
    g_linear_ring_launches.fetch_add(1, std::memory_order_relaxed);
    if (n_sp == 1) {
        const PrefillQkv none{};
        const RawRows raw{X, W};
        ZG_TRY(tm == 1   ? (launch_ring<PF_LINEAR, 1, 1, 2, 4>(A, P, bias, Y, M, Np, K, N, 1, none, PlaneOut{}, s, raw, seen))
               : tm == 2 ? (launch_ring<PF_LINEAR, 2, 1, 2, 3>(A, P, bias, Y, M, Np, K, N, 1, none, PlaneOut{}, s, raw, seen))
                         : (launch_ring<PF_LINEAR, 2, 2, 2, 2>(A, P, bias, Y, M, Np, K, N, 1, none, PlaneOut{}, s, raw, seen)));
        return ZG_OK;
    }
    ZG_TRY(launch_ring_epi<PF_LINEAR_PART>(A, P, nullptr, slabs, M, Np, K, Np, tm, n_sp, PrefillQkv{}, PlaneOut{}, s, seen));
    const size_t quads = (size_t)M * ((N + 3) / 4);
    linear_ring_finish_kernel<<<(unsigned)((quads + 255) / 256), 256, 0, s>>>(slabs, n_sp, M, Np, bias, Y, N, X, W, K, seen);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

// Priced in us like the prompts' Linears below, with 3 for the launch that adds slabs.  It takes a Linear of 1536 columns and more where the kernel that splits in its own staging
// has few slices of K to add up, whose chains are then so long that this kernel is closer to 64 bits as well (e-7 of the result, that kernel : this: 700 x 1600 x 1600 1.67 : 1.38,
// 2048 x 3072 x 768 2.35 : 1.64, 400 x 6400 x 1600 2.81 : 1.43), and where it is cheap beside the persistent one (rounds of 256 x 192 tiles: one of
// 1600 columns 90 predicted, 95 measured; beside several rounds here, which are a sixth longer than predicted, 0.85 of that) and beside the kernel that splits in its
// own staging.  There the pass over both operands counts, which for few rows is the weight's and most of the call (this kernel behind it: within 9 % over the shapes of
// linear_tiles_us).  us of a call, without : with: 3072 -> 768 700 rows 48 : 44; 1600 -> 1600 700 rows 49 : 45, 1200 66 : 46; 1600 -> 4800 256 rows 50 : 46,
// 700 103 : 63; 6400 -> 1600 420 rows 100 : 84, 1200 204 : 131; 4800 -> 5120 300 rows 154 : 117; not taken: 4800 -> 5120 128 rows 66 : 84,
// 6400 -> 6400 128 rows 103 : 147, 300 205 : 208; 6400 -> 9601 64 rows 83 : 210, 256 270 : 330; 4096 -> 1024 478 rows 47 : 48; 1600 -> 4800 1500 rows 119 : 139.
int linear_ring_route(size_t M, size_t N, size_t K, int* tm) {
    if (K < 1536 || linear_tiles_slices(M, N, K) > (K < 3072 ? 2 : 4)) return 0;
    const int nk = (int)(K / kBk);
    const double slab = (double)M * (double)whole64(N) * 8.0 / 4e6;
    auto rounds = [](long n) { return (double)((n + 255) / 256); };
    int best = 0;
    double best_us = rounds((long)((M + 255) / 256 * ((N + 191) / 192))) * (3.2 * nk + 10.0) * 0.85;
    for (int t = 1; t <= 3; ++t) {
        const long tiles = ring_tiles((long)M, (long)N, t);
        const long most = std::max(1l, std::min(256 / tiles, (long)nk / 3));
        for (long n = 1; n <= most; ++n) {
            const double us = rounds(tiles * n) * (4.5 + (double)((nk + n - 1) / n) * kStepUs[t]) + (n > 1 ? (double)n * slab + 3.0 : 0.0);
            if (us < best_us) {
                best = (int)n;
                best_us = us;
                *tm = t;
            }
        }
    }
    if (best > 0 && linear_tiles_pay(M, N, K, true) && linear_split_us(M, N, K) + 0.78 * best_us > 0.97 * linear_tiles_us(M, N, K)) return 0;
    return best;
}

// K slices of the launch (1 unless it is a residual Linear, whose slices meet in slabs) and rows of a tile (64 tm); 0: the 128-row kernels take it.
// Both sides are priced in us.  bf16 weights: by what one compute unit takes in (65 bytes a ns), 3 us for each round of workgroups, and slabs at
// 4 TB/s.  At K = 768: 300 x 3072 predicts 9 here and 14 there (measured 10.5 and 16.6), 800 x 3072 41 and 15 (31.7, 20.4); K = 3072: 300 x 768
// 10 and 13 (14.3, 16.1), 800 x 768 28 and 18 (27.6, 24.7).  fp32 weights: by the steps of the three tile forms and of the 128-row kernel (1 us for 128 columns):
// 300 x 3072 11 and 33 (11.8, 27), 1000 x 768 x 3072 27 and 39 (28, 40), 1500 x 3072 x 768 41 and 54 (39, 56), 2000 x 768 x 3072 50 and 58 (52, 66).
// bf16: beyond a few hundred rows what wins by less than a microsecond is lost again in the reduce kernel behind it, which finds one slab where
// it found several (a whole prompt of 4 x 200 rows of 768 columns: 1377 us against 1359, 8 x 255 of 384: 600 against 588).
int prefill_ring_route(int M, int N, int K, bool resid, bool planes, size_t ws_floats, bool force, int* tm) {
    if (!planes && M > 700 && !force) return 0;
    const int nk = K / kBk;
    const double slab = (double)M * N * 8.0 / 4e6;
    auto rounds = [](long n) { return (double)((n + 255) / 256); };
    int best = 0;
    double best_us = 0.0;
    for (int t = 1; t <= (planes ? 3 : 2); ++t) {
        const long tiles = ring_tiles(M, N, t);
        int n_sp = resid ? (int)std::max(1l, std::min(256 / tiles, (long)nk / 3)) : 1;
        while (resid && n_sp > 1 && (size_t)n_sp * M * N > ws_floats) --n_sp;
        if (resid && (size_t)n_sp * M * N > ws_floats) continue;
        const double us = (planes ? rounds(tiles * n_sp) * (4.5 + (nk + n_sp - 1) / n_sp * kStepUs[t]) : rounds(tiles * n_sp) * (3.0 + (nk + n_sp - 1) / n_sp * (16.0 * t + 8.0) / 65.0)) +
                          (resid ? n_sp * slab : 0.0);
        if (best == 0 || us < best_us) {
            best = n_sp;
            best_us = us;
            *tm = t;
        }
    }
    if (best == 0 || force) return best;
    const bool wide = prefill_rows_wide(M, N, planes ? 2 : 1);
    const int bn = wide ? 256 : 128;
    const long tiles = (long)((M + 127) / 128) * ((N + bn - 1) / bn);
    const int passes = planes ? 2 : 1;
    const int n_sp = (int)std::max(1l, std::min(planes ? (256 + 2 * tiles - 1) / (2 * tiles) : 256 / tiles, (long)nk / 3));
    const double us = rounds(tiles * n_sp * passes) * (planes ? 4.5 + (nk + n_sp - 1) / n_sp * bn / 128.0 : 3.0 + (nk + n_sp - 1) / n_sp * (32.0 + bn / 8.0) / 65.0) +
                      (resid || n_sp * passes > 1 ? n_sp * passes * slab : 0.0) + (!resid && n_sp * passes > 1 ? 3.0 : 0.0);
    return best_us + (planes || M <= 256 ? 0.0 : 1.0) <= us ? best : 0;
}

int launch_prefill_ring(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int ldc, int epi, int tm, int n_sp, const PrefillQkv& qa,
                        const PlaneOut& po, hipStream_t s) {
    ZG_REQUIRE(M > 0 && N % 64 == 0 && K % kBk == 0 && n_sp >= 1 && n_sp <= K / kBk && (size_t)M * kPair * K * 2 < ((size_t)1 << 31) &&
                   (size_t)N * K * 2 * (W.planes + W.rest) < ((size_t)1 << 31),
               ZG_ERR_UNSUPPORTED, "prefill gemm: operands of %d x %d x %d beyond 2 GiB", M, N, K);
    switch (epi) {
        case PF_F32: return launch_ring_epi<PF_F32>(A, W, bias, C, M, N, K, ldc, tm, 1, qa, po, s);
        case PF_PARTIAL: return launch_ring_epi<PF_PARTIAL>(A, W, nullptr, C, M, N, K, ldc, tm, n_sp, qa, po, s);
        case PF_GELU_SPLIT: return launch_ring_epi<PF_GELU_SPLIT>(A, W, bias, C, M, N, K, ldc, tm, 1, qa, po, s);
        case PF_QKV: return launch_ring_epi<PF_QKV>(A, W, bias, C, M, N, K, ldc, tm, 1, qa, po, s);
    }
    ZG_REQUIRE(false, ZG_ERR_ARG, "prefill gemm: epilogue %d", epi);
}

}  // namespace zg
