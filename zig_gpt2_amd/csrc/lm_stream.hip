// lm_stream.hip — the products of prompt portions (rows rounded to bf16 already, or fp32 rows in 32-bit mode; bf16 weights, K a multiple of 64):
// operands by LDS-DMA through a ring of K steps.
//
// What bounded the staged tiles (lm_wide_kernel, lm_linear.hip) was the way of an operand: into registers, through a swizzle into the LDS, a
// barrier, and two K steps in flight at most.  Here a wave only names addresses (buffer_load ... lds, the swizzle in which chunk of a row a
// lane asks for), ST - 1 K steps are in flight, and a K step costs one barrier: what a step waits for was requested ST - 1 steps ago, and the slot
// that barrier frees takes the step ST - 1 ahead.  The number of requests in flight is the same at every step (behind the last one it is
// repeated), so the wait is a constant.  Rows are gathered where they are asked for, so experts' grouped products take this form too.
// Results leave through the LDS as 16-byte pieces of whole rows.
#include "lm_linear_args.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "zg_once.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((address_space(3))) char* lds_at_t;

// (written here, not by the builtin: the compiler would wait for every request in flight in front of any read of the LDS.  m0: the address of
// the wave's 1 KB piece; the wait state is what a request needs behind a write of m0)
__device__ __forceinline__ void dma_16(unsigned lds, const u32x4& rsrc, unsigned v_off, unsigned s_off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(v_off), "s"(rsrc), "s"(s_off) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void arrive() {  // N requests may be in flight; what was read of the LDS is here; every wave has come this far
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

constexpr int kBk = 64;  // columns of K of a step
enum { STREAM_PLAIN, STREAM_GLU };
__device__ __forceinline__ float silu_gate(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// (an output that came out NaN, again as a plain fp32 sum: the terms of an infinity meet infinite weights as zeros)
__device__ __forceinline__ float plain_sum(const float* a, const bf16_t* b, int K) {
    float s = 0.0f;
#pragma unroll 1
    for (int k = 0; k < K && s == s; k += 2) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(b + k);
        s = fmaf(a[k + 1], bf16_hi(w), fmaf(a[k], bf16_lo(w), s));
    }
    return s;
}

// The three terms of eight values, cut off rather than rounded.  What an infinity leaves is NaN, and the outputs it reaches are worked out again.
__device__ __forceinline__ Planes8<3> terms_of(const u32x4& lo, const u32x4& hi) {
    Planes8<3> o;
    uint32_t x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o.v[t][i] = __builtin_amdgcn_perm(x[2 * i + 1], x[2 * i], 0x07060302u);
#pragma unroll
            for (int e = 2 * i; e < 2 * i + 2; ++e)
                if (t < 2) x[e] = __float_as_uint(__uint_as_float(x[e]) - __uint_as_float(x[e] & 0xFFFF0000u));
        }
    return o;
}

// 2 x 2 waves of TM x TN 32 x 32 tiles, two workgroups to a compute unit.  STREAM_GLU (TN = 2): a wave's first column tile is 32 gates, its second the 32 columns they gate.
// F32 (32-bit mode): rows of fp32, multiplied as their exact three bf16 terms, the smallest first.  They pass the LDS as they are (4 bytes a value
// where three terms take 6), and the terms are made from the fragments, beside the products of the fragments in front of them.  That work
// bounds it (190 vector instructions a wave and K step beside 12 products), so KG = 2 groups of waves take half the columns of a step each.
template <int TM, int TN, int ST, int KIND, bool F32, int KG>
__global__ __launch_bounds__(256 * KG, 2) void lm_stream_kernel(const LinArgs p) {
    constexpr bool GLU = KIND == STREAM_GLU;
    constexpr int BM = 64 * TM, BN = 64 * TN, OUT_N = GLU ? BN / 2 : BN, ROW = kBk * 2, CH = kBk / 8;  // (a row of a step: 128 bytes, 8 chunks)
    constexpr int ROW_A = F32 ? 2 * ROW : ROW, NP = F32 ? 3 : 1, AH = F32 ? 2 : 1, WAVES = 4 * KG, KK = CH / 2 / KG;
    constexpr int PA = BM * ROW_A / (1024 * WAVES), PB = BN / (8 * WAVES), SLOT = BM * ROW_A + BN * ROW;  // 1 KB pieces a wave asks for, bytes of a step
    static_assert(!GLU || TN == 2, "a tile of gates and a tile of what they gate");
    static_assert(F32 ? TM == 1 && KG == 2 : KG == 1, "halves of K: fp32 rows, one tile of them");
    extern __shared__ __attribute__((aligned(1024))) char s_ring[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wg = wave >> 2, wy = (wave >> 1) & 1, wx = wave & 1;
    const unsigned lds0 = (unsigned)(unsigned long)(lds_at_t)s_ring;
    const int n_all = GLU ? p.glu_out : p.N;
    TileAt t;
    if (!find_tile(p, n_all, BM, OUT_N, t)) return;
    auto rsrc_of = [](const void* base) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)), 0x80000000u,
                     0x00020000u};
    };
    const u32x4 ra = F32 ? rsrc_of(p.A + (long long)blockIdx.z * p.a_zoff) : rsrc_of(p.A16 + (long long)blockIdx.z * p.a_zoff), rb = rsrc_of(t.B);
    const int in_row = lane >> 3, chunk = (lane & 7) ^ in_row;  // (every eighth row the swizzle repeats)
    // (fp32 rows: 16 chunks, four rows to a piece)
    const int in_row_a = F32 ? lane >> 4 : in_row, chunk_a = F32 ? (lane & 15) ^ ((wave * 4 + in_row_a) & 15) : chunk;
    unsigned va[PA], vb[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int m = min(t.m0 + (wave + WAVES * i) * (F32 ? 4 : 8) + in_row_a, t.m_end - 1);  // (rows beyond the edge: some valid row, never stored)
        va[i] = (unsigned)((p.a_rows ? p.a_rows[m] : m) / p.a_div) * (unsigned)p.lda * (F32 ? 4u : 2u) + chunk_a * 16u;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int r = (wave + WAVES * i) * 8 + in_row;  // row of the tile of weights: [wave column][gates | gated] of 32 each, or as they are
        const int n = GLU ? min(t.n0 + (r / 64) * 32 + r % 32, n_all - 1) + (r & 32 ? n_all : 0) : min(t.n0 + r, n_all - 1);
        vb[i] = (unsigned)n * (unsigned)p.ldb * 2u + chunk * 16u;
    }
    const int steps = p.K / kBk;
    auto request = [&](int slot, int s) {
        const unsigned at = (unsigned)min(s, steps - 1), to = lds0 + slot * SLOT + wave * 1024;
#pragma unroll
        for (int i = 0; i < PA; ++i) dma_16(to + i * 1024 * WAVES, ra, va[i], at * ROW_A);
#pragma unroll
        for (int i = 0; i < PB; ++i) dma_16(to + BM * ROW_A + i * 1024 * WAVES, rb, vb[i], at * ROW);
    };
    f32x16 acc[TM][TN], small[TM][TN];  // (the second and third terms' products have sums of their own, so that they are not rounded at the first's size)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = small[i][j][e] = 0.0f;
    const int fr = lane & 31, kh = lane >> 5, fswz = fr & 7;
    // The operands change places: an accumulator's registers are then runs of four columns of a row (lane % 32: the row).
    u32x4 af[2][KK][TM][AH], bf[2][KK][TN];  // of the step that is multiplied, and of the one behind it on its way
    auto read = [&](auto b, int slot) {
        const char* base = s_ring + slot * SLOT;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int at = KK * wg + kk, c = ((2 * at + kh) ^ fswz) * 16;
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[b][kk][j] = *reinterpret_cast<const u32x4*>(base + BM * ROW_A + ((wx * TN + j) * 32 + fr) * ROW + c);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int h = 0; h < AH; ++h)
                    af[b][kk][i][h] = *reinterpret_cast<const u32x4*>(base + ((wy * TM + i) * 32 + fr) * ROW_A + (F32 ? ((4 * at + 2 * kh + h) ^ (fr & 15)) * 16 : c));
        }
    };
    // (a fragment's terms are made beside the products of the one in front of it)
    Planes8<NP> terms[2][TM];
    auto split = [&](auto b, int kk, auto to) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (F32) terms[to][i] = terms_of(af[b][kk][i][0], af[b][kk][i][AH - 1]);
            else terms[to][i].v[0] = af[b][kk][i][0];
        }
    };
    auto multiply = [&](auto b) {
        constexpr int other = 1 - decltype(b)::value;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            if (!F32) split(b, kk, std::integral_constant<int, 0>());
            else if (kk + 1 < KK) kk % 2 ? split(b, kk + 1, std::integral_constant<int, 0>()) : split(b, kk + 1, std::integral_constant<int, 1>());
            else split(std::integral_constant<int, other>(), 0, std::integral_constant<int, 0>());
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int q = NP - 1; q >= 0; --q)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x16& to = q > 0 ? small[i][j] : acc[i][j];
                        to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bf[b][kk][j]), __builtin_bit_cast(bf16x8, terms[F32 ? kk % 2 : 0][i].v[q]), to, 0, 0, 0);
                    }
        }
    };
#pragma unroll
    for (int s = 0; s < ST; ++s) request(s, s);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), said to the compiler: with scalar loads in flight it would wait for all fragments at once
    arrive<(ST - 1) * (PA + PB)>();
    read(std::integral_constant<int, 0>(), 0);
    if (F32) split(std::integral_constant<int, 0>(), 0, std::integral_constant<int, 0>());
    int slot = 0, s = 0;
    // Step s: its fragments have been read, so its slot takes step s + ST; those of s + 1 are read beside its products.
    auto body = [&](auto b) {
        constexpr int other = 1 - decltype(b)::value;
        arrive<(ST - 2) * (PA + PB)>();
        request(slot, s + ST);
        slot = slot == ST - 1 ? 0 : slot + 1;
        __builtin_amdgcn_sched_barrier(0);
        read(std::integral_constant<int, other>(), slot);
        multiply(b);
        // order: a read in front of every product while there are any (fp32: two), behind it what makes terms
        constexpr int products = KK * TM * TN * NP, reads = KK * (TM * AH + TN);
#pragma unroll
        for (int x = 0; x < products; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x100, F32 ? 2 : (reads + products - 1) / products, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (F32) __builtin_amdgcn_sched_group_barrier(0x002, (KK * TM * 44 + products - 1) / products, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        ++s;
    };
    for (int pairs = steps >> 1; pairs > 0; --pairs) {
        body(std::integral_constant<int, 0>());
        body(std::integral_constant<int, 1>());
    }
    if (steps & 1) body(std::integral_constant<int, 0>());
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the requests behind the last step still write the ring)

    if (F32)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[0][j] += small[0][j];
    // element e of a 32 x 32 tile: column 8 (e / 4) + 4 (lane / 32) + e % 4, row lane % 32.  Every wave turns its rows in an image of its own.
    constexpr int WN_OUT = OUT_N / 2, PITCH = WN_OUT * 4 + 16;  // columns of a wave, bytes of a row of its image
    constexpr int REGION = KG > 1 ? TN * 4096 + 512 : 32 * PITCH;
    static_assert(4 * REGION <= ST * SLOT && 32 * PITCH <= REGION, "the images fit the ring");
    char* img = s_ring + (wave & 3) * REGION;
    if constexpr (KG > 1) {  // the second half of the columns joins the first
        f32x4* part = reinterpret_cast<f32x4*>(img) + lane;
        if (wg == 1)
#pragma unroll
            for (int x = 0; x < TN * 4; ++x) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[0][x / 4][x % 4 * 4 + e];
                part[x * 64] = v;
            }
        __syncthreads();
        if (wg == 1) return;
#pragma unroll
        for (int x = 0; x < TN * 4; ++x) {
            const f32x4 v = part[x * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[0][x / 4][x % 4 * 4 + e] += v[e];
        }
    }
    const bool to16 = p.C == nullptr;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < (GLU ? 1 : TN); ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = GLU ? silu_gate(acc[i][0][4 * g + e], acc[i][TN - 1][4 * g + e]) : acc[i][j][4 * g + e];
                *reinterpret_cast<f32x4*>(img + fr * PITCH + (32 * j + 8 * g + 4 * kh) * 4) = v;
            }
        // (a wave's accesses to the LDS are in order)
        constexpr int PER = WN_OUT / 8;  // runs of eight columns of a row
#pragma unroll 1
        for (int q = lane; q < 32 * PER; q += 64) {
            const int r = q / PER, c = q % PER * 8, m = t.m0 + (wy * TM + i) * 32 + r, n = t.n0 + wx * WN_OUT + c;
            f32x4 v[2] = {*reinterpret_cast<const f32x4*>(img + r * PITCH + c * 4), *reinterpret_cast<const f32x4*>(img + r * PITCH + c * 4 + 16)};
            if (m >= t.m_end || n >= n_all) continue;
            const bool half = n + 8 > n_all;  // (four columns)
            if constexpr (F32) {
                const f32x4 z = v[0] + v[1];
                const float sum = (z.x + z.y) + (z.z + z.w);
                if (__builtin_expect(sum != sum, 0)) {
                    const float* a = p.A + (long long)blockIdx.z * p.a_zoff + (long long)((p.a_rows ? p.a_rows[m] : m) / p.a_div) * p.lda;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (v[e / 4][e % 4] != v[e / 4][e % 4] && n + e < n_all) {
                            const bf16_t* b = t.B + (long long)(n + e) * p.ldb;
                            const float y = plain_sum(a, b, p.K);
                            v[e / 4][e % 4] = GLU ? silu_gate(y, plain_sum(a, b + (long long)n_all * p.ldb, p.K)) : y;
                        }
                }
            }
            if (!GLU && (p.act != ACT_NONE || p.bias)) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e / 4][e % 4] = finish(v[e / 4][e % 4], min(n + e, n_all - 1), p);
            }
            const long long at = (long long)blockIdx.z * p.c_zoff + (long long)m * p.ldc + n;
            if (to16) {
                const u32x4 r = to_planes<1>(v[0], v[1]).v[0];
                if (half) *reinterpret_cast<u32x2*>(p.C16 + at) = u32x2{r.x, r.y};
                else *reinterpret_cast<u32x4*>(p.C16 + at) = r;
            } else {
                *reinterpret_cast<f32x4*>(p.C + at) = v[0];
                if (!half) *reinterpret_cast<f32x4*>(p.C + at + 4) = v[1];
            }
        }
    }
}

template <int TM, int TN, int ST, int KIND, bool F32 = false, int KG = 1>
int launch_form(const LinArgs& p, int nz, hipStream_t s) {
    constexpr int BM = 64 * TM, BN = 64 * TN, LDS = ST * (BM * (F32 ? 2 : 1) + BN) * kBk * 2;
    static_assert(2 * LDS <= 160 * 1024, "two workgroups to a compute unit");
    static OncePerDevice raised;
    int device = 0;
    ZG_HIP(hipGetDevice(&device));
    ZG_TRY(raised.run(device, []() -> int {
        ZG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&lm_stream_kernel<TM, TN, ST, KIND, F32, KG>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        return ZG_OK;
    }));
    const int n = KIND == STREAM_GLU ? p.glu_out : p.N, out_n = KIND == STREAM_GLU ? BN / 2 : BN;
    const long long tiles = (long long)((n + out_n - 1) / out_n) * ((p.M + BM - 1) / BM + p.n_groups);
    ZG_REQUIRE(tiles < (1LL << 31), ZG_ERR_UNSUPPORTED, "linear: %d rows exceed the grid", p.M);
    lm_stream_kernel<TM, TN, ST, KIND, F32, KG><<<dim3((unsigned)tiles, 1, nz), 256 * KG, LDS, s>>>(p);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace

bool stream_fits(const Linear& L, bool f32) {
    if (toy_product(L, f32) || (f32 ? !L.A : !L.A16) || L.z_group || L.a_glu || L.a_poly || L.a_norm || L.K < kBk || L.K % kBk != 0 || (L.C != nullptr) == (L.C16 != nullptr) || L.nz < 1 || L.nz > 65535 ||
        (L.glu_out > 0 && L.glu_kind != GLU_SILU))
        return false;
    const int n_out = L.glu_out > 0 ? L.glu_out : L.N;
    const uintptr_t all = (f32 ? reinterpret_cast<uintptr_t>(L.A) : reinterpret_cast<uintptr_t>(L.A16)) | reinterpret_cast<uintptr_t>(L.B) | reinterpret_cast<uintptr_t>(L.C) | reinterpret_cast<uintptr_t>(L.C16);
    const int of_a = f32 ? 4 : 8, of_c = L.C16 ? 8 : 4;
    return (all & 15) == 0 && L.lda % of_a == 0 && L.ldb % 8 == 0 && L.a_zoff % of_a == 0 && L.b_zoff % 8 == 0 && L.c_zoff % of_c == 0 && L.ldc % of_c == 0 && n_out % 4 == 0 &&
           (size_t)L.M * L.lda < (f32 ? 1u << 29 : 1u << 30) && (size_t)L.N * L.ldb < (1u << 30);  // (32-bit offsets of bytes)
}

int launch_stream(const Linear& L, bool f32, hipStream_t s, bool* taken) {
    *taken = false;
    int force = 0;  // test hooks: 1 to 4 that form at any size, -1 none; the forms of lm_linear.hip by theirs
    if (const char* e = getenv("ZGPT2_LM_STREAM")) force = atoi(e);
    else if (getenv("ZGPT2_LM_GEMM_TILE")) force = -1;
    if (force < 0 || !stream_fits(L, f32)) return ZG_OK;
    const LinArgs p = make_args(L);
    const bool glu = L.glu_out > 0;
    const int n_out = glu ? L.glu_out : L.N;
    auto tiles = [&](int bm, int bn) { return (long long)((n_out + bn - 1) / bn) * ((L.M + bm - 1) / bm + (L.grp_off ? L.n_groups : 0)) * L.nz; };
    // Which form.  A compute unit takes in some 30 bytes a clock whatever the form (64 x 64 x 64 steps 590 clocks each, whether one workgroup
    // or two share it), so few tiles are small ones, and large ones as soon as they fill the chip.  us per launch, 64 x 64 : 128 x 64 :
    // 128 x 128 : the staged tiles of lm_linear.hip (or the persistent kernel *):
    //   333 x 768 x 768 (72 tiles of 64 x 64) 5.7 : 7.3 : 10.6 : 7.0     900 x 768 x 3072 (180) 13.8 : 18.7 : 33 : 16.1    500 x 2048 x 3072 (256) 18.4 : 23.7 : 43 : 19.8
    //   1400 x 768 x 3072 (264) 16.6 : 19.1 : 33 : 25.8      450 x 2304 x 768 (288) 10.4 : 7.9 : 11.2 : 11.1             2048 x 768 x 3072 (384) 21.5 : 20.1 : 33 : 27.8
    //   2048 x 1456 x 768 (192 of 128 x 128) 14.0 : 13.2 : 13.5 : 14.7   1023 x 3072 x 768 (192) 16.0 : 14.1 : 14.7 : 15.3   2048 x 3072 x 768 (384) 29.8 : 22.2 : 19.5 : 23.7*
    //   8184 x 1024 x 1024 (512) 39.5 : 33.3 : 25.3 : 29.1*  8184 x 672 x 1024 (384) 26.8 : 23.1 : 21.9 : 25.7*
    // Below 32 rows the tiles with K over the waves keep ahead (16 x 768 x 3072 13.2 : 11.8).
    // 32-bit mode, us per launch, 64 x 64 : 64 x 128 : the staged tiles or those with K over the waves:
    //   333 x 768 x 768 (72 tiles of 64 x 64) 9.4 : 11.3 : 10.2     333 x 768 x 3072 (72) 25.4 : 32.5 : 27.9     333 x 2304 x 768 (216) 10.1 : 11.9 : 17.3
    //   333 x 3072 x 768 (288) 14.7 : 12.5 : 17.7     1023 x 2304 x 768 (576) 21.0 : 18.7 : 25.2     2048 x 3072 x 768 (1536) 48.7 : 36.8 : 43.8
    // up to 256 tiles of 32 x 32 those with K over the waves keep ahead (200 x 768 x 768 (168) 9.2 : 11.1 : 7.9; 40 x 3072 x 3072 (192) 25.6 : 44 : 20.6).
    int form = force;
    if (!force && f32) {
        if (tiles(32, 32) * (glu ? 2 : 1) <= 256) return ZG_OK;
        form = tiles(64, 64) <= 256 ? 3 : 2;
    } else if (!force && glu) form = tiles(128, 64) >= 256 ? 1 : 4;
    else if (!force && L.M <= 32 && !L.grp_off) return ZG_OK;
    else if (!force) form = tiles(64, 64) <= 272 ? 3 : tiles(128, 128) < 256 ? 2 : 1;
    if (f32 && glu) ZG_TRY((launch_form<1, 2, 2, STREAM_GLU, true, 2>(p, L.nz, s)));
    else if (f32 && form <= 2) ZG_TRY((launch_form<1, 2, 2, STREAM_PLAIN, true, 2>(p, L.nz, s)));
    else if (f32) ZG_TRY((launch_form<1, 1, 3, STREAM_PLAIN, true, 2>(p, L.nz, s)));
    else if (glu && form == 1) ZG_TRY((launch_form<2, 2, 2, STREAM_GLU>(p, L.nz, s)));
    else if (glu) ZG_TRY((launch_form<1, 2, 3, STREAM_GLU>(p, L.nz, s)));
    else if (form == 1) ZG_TRY((launch_form<2, 2, 2, STREAM_PLAIN>(p, L.nz, s)));
    else if (form == 2) ZG_TRY((launch_form<2, 1, 3, STREAM_PLAIN>(p, L.nz, s)));
    else ZG_TRY((launch_form<1, 1, 4, STREAM_PLAIN>(p, L.nz, s)));
    note_kernel("lm_stream_kernel<%d>", form);
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
