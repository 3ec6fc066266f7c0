// lm_stream.hip — the products of prompt portions whose rows are rounded already (bf16 A, bf16 weights, K a multiple of 64): operands by LDS-DMA
// through a ring of K steps.
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

// 2 x 2 waves of TM x TN 32 x 32 tiles, two workgroups to a compute unit.  STREAM_GLU (TN = 2): a wave's first column tile is 32 gates, its second the 32 columns they gate.
template <int TM, int TN, int ST, int KIND>
__global__ __launch_bounds__(256, 2) void lm_stream_kernel(const LinArgs p) {
    constexpr bool GLU = KIND == STREAM_GLU;
    constexpr int BM = 64 * TM, BN = 64 * TN, OUT_N = GLU ? BN / 2 : BN, ROW = kBk * 2, CH = kBk / 8;  // (a row of a step: 128 bytes, 8 chunks)
    constexpr int PA = BM / 32, PB = BN / 32, SLOT = (BM + BN) * ROW;  // 1 KB pieces (8 rows) a wave asks for, bytes of a step
    static_assert(!GLU || TN == 2, "a tile of gates and a tile of what they gate");
    extern __shared__ __attribute__((aligned(1024))) char s_ring[];
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wy = wave >> 1, wx = wave & 1;
    const unsigned lds0 = (unsigned)(unsigned long)(lds_at_t)s_ring;
    const int n_all = GLU ? p.glu_out : p.N;
    TileAt t;
    if (!find_tile(p, n_all, BM, OUT_N, t)) return;
    auto rsrc_of = [](const void* base) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)), 0x80000000u,
                     0x00020000u};
    };
    const u32x4 ra = rsrc_of(p.A16 + (long long)blockIdx.z * p.a_zoff), rb = rsrc_of(t.B);
    const int in_row = lane >> 3, chunk = (lane & 7) ^ in_row;  // (every eighth row the swizzle repeats)
    unsigned va[PA], vb[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int m = min(t.m0 + (wave + 4 * i) * 8 + in_row, t.m_end - 1);  // (rows beyond the edge: some valid row, never stored)
        va[i] = (unsigned)((p.a_rows ? p.a_rows[m] : m) / p.a_div) * (unsigned)p.lda * 2u + chunk * 16u;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int r = (wave + 4 * i) * 8 + in_row;  // row of the tile of weights: [wave column][gates | gated] of 32 each, or as they are
        const int n = GLU ? min(t.n0 + (r / 64) * 32 + r % 32, n_all - 1) + (r & 32 ? n_all : 0) : min(t.n0 + r, n_all - 1);
        vb[i] = (unsigned)n * (unsigned)p.ldb * 2u + chunk * 16u;
    }
    const int steps = p.K / kBk;
    auto request = [&](int slot, int s) {
        const unsigned off = (unsigned)min(s, steps - 1) * ROW, to = lds0 + slot * SLOT + wave * 1024;
#pragma unroll
        for (int i = 0; i < PA; ++i) dma_16(to + i * 4096, ra, va[i], off);
#pragma unroll
        for (int i = 0; i < PB; ++i) dma_16(to + BM * ROW + i * 4096, rb, vb[i], off);
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    const int fr = lane & 31, kh = lane >> 5, fswz = fr & 7;
    // The operands change places: an accumulator's registers are then runs of four columns of a row (lane % 32: the row).
    u32x4 af[2][CH / 2][TM], bf[2][CH / 2][TN];  // of the step that is multiplied, and of the one behind it on its way
    auto read = [&](auto b, int slot) {
        const char* base = s_ring + slot * SLOT;
#pragma unroll
        for (int kk = 0; kk < CH / 2; ++kk) {
            const int c = ((2 * kk + kh) ^ fswz) * 16;
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[b][kk][j] = *reinterpret_cast<const u32x4*>(base + BM * ROW + ((wx * TN + j) * 32 + fr) * ROW + c);
#pragma unroll
            for (int i = 0; i < TM; ++i) af[b][kk][i] = *reinterpret_cast<const u32x4*>(base + ((wy * TM + i) * 32 + fr) * ROW + c);
        }
    };
    auto multiply = [&](auto b) {
#pragma unroll
        for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bf[b][kk][j]), __builtin_bit_cast(bf16x8, af[b][kk][i]), acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < ST; ++s) request(s, s);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), said to the compiler: with scalar loads in flight it would wait for all fragments at once
    arrive<(ST - 1) * (PA + PB)>();
    read(std::integral_constant<int, 0>(), 0);
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
        // order: a read in front of every product while there are any
        constexpr int products = CH / 2 * TM * TN, reads = CH / 2 * (TM + TN);
#pragma unroll
        for (int x = 0; x < products; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x100, (reads + products - 1) / products, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
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

    // element e of a 32 x 32 tile: column 8 (e / 4) + 4 (lane / 32) + e % 4, row lane % 32.  Every wave turns its rows in an image of its own.
    constexpr int WN_OUT = OUT_N / 2, PITCH = WN_OUT * 4 + 16;  // columns of a wave, bytes of a row of its image
    static_assert(4 * 32 * PITCH <= ST * SLOT, "the images fit the ring");
    char* img = s_ring + wave * 32 * PITCH;
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
            if (!GLU && (p.act != ACT_NONE || p.bias)) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e / 4][e % 4] = finish(v[e / 4][e % 4], n + e, p);
            }
            const long long at = (long long)blockIdx.z * p.c_zoff + (long long)m * p.ldc + n;
            if (to16) *reinterpret_cast<u32x4*>(p.C16 + at) = to_planes<1>(v[0], v[1]).v[0];
            else {
                *reinterpret_cast<f32x4*>(p.C + at) = v[0];
                *reinterpret_cast<f32x4*>(p.C + at + 4) = v[1];
            }
        }
    }
}

template <int TM, int TN, int ST, int KIND>
int launch_form(const LinArgs& p, int nz, hipStream_t s) {
    constexpr int BM = 64 * TM, BN = 64 * TN, LDS = ST * (BM + BN) * kBk * 2;
    static_assert(2 * LDS <= 160 * 1024, "two workgroups to a compute unit");
    static OncePerDevice raised;
    int device = 0;
    ZG_HIP(hipGetDevice(&device));
    ZG_TRY(raised.run(device, []() -> int {
        ZG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&lm_stream_kernel<TM, TN, ST, KIND>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        return ZG_OK;
    }));
    const int n = KIND == STREAM_GLU ? p.glu_out : p.N, out_n = KIND == STREAM_GLU ? BN / 2 : BN;
    const long long tiles = (long long)((n + out_n - 1) / out_n) * ((p.M + BM - 1) / BM + p.n_groups);
    ZG_REQUIRE(tiles < (1LL << 31), ZG_ERR_UNSUPPORTED, "linear: %d rows exceed the grid", p.M);
    lm_stream_kernel<TM, TN, ST, KIND><<<dim3((unsigned)tiles, 1, nz), 256, LDS, s>>>(p);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace

bool stream_fits(const Linear& L) {
    if (!L.A16 || L.z_group || L.a_glu || L.a_poly || L.a_norm || L.K < kBk || L.K % kBk != 0 || (L.C != nullptr) == (L.C16 != nullptr) || L.nz < 1 || L.nz > 65535 ||
        (L.glu_out > 0 && L.glu_kind != GLU_SILU))
        return false;
    const int n_out = L.glu_out > 0 ? L.glu_out : L.N;
    const uintptr_t all = reinterpret_cast<uintptr_t>(L.A16) | reinterpret_cast<uintptr_t>(L.B) | reinterpret_cast<uintptr_t>(L.C) | reinterpret_cast<uintptr_t>(L.C16);
    return (all & 15) == 0 && L.lda % 8 == 0 && L.ldb % 8 == 0 && L.a_zoff % 8 == 0 && L.b_zoff % 8 == 0 && L.c_zoff % 8 == 0 && L.ldc % 8 == 0 && n_out % 8 == 0 &&
           (size_t)L.M * L.lda < (1u << 30) && (size_t)L.N * L.ldb < (1u << 30);  // (32-bit offsets of bytes)
}

int launch_stream(const Linear& L, hipStream_t s, bool* taken) {
    *taken = false;
    int force = 0;  // test hooks: 1 to 4 that form at any size, -1 none; the forms of lm_linear.hip by theirs
    if (const char* e = getenv("ZGPT2_LM_STREAM")) force = atoi(e);
    else if (getenv("ZGPT2_LM_GEMM_TILE")) force = -1;
    if (force < 0 || !stream_fits(L)) return ZG_OK;
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
    int form = force;
    if (!force && glu) form = tiles(128, 64) >= 256 ? 1 : 4;
    else if (!force && L.M <= 32 && !L.grp_off) return ZG_OK;
    else if (!force) form = tiles(64, 64) <= 272 ? 3 : tiles(128, 128) < 256 ? 2 : 1;
    if (glu && form == 1) ZG_TRY((launch_form<2, 2, 2, STREAM_GLU>(p, L.nz, s)));
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
