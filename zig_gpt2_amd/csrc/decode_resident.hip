// Greedy decode of ONE sequence as a resident kernel: the whole chip stays inside one launch for up to 64 tokens, some 3.5 ms (GPT.forward + the
// argmax of generate, src/main.zig:178-195, :322-342), and the phases of a Block meet through tagged words instead of launch
// boundaries.  Measured: GPT-2 124M 208 -> 110 us a token (256 tokens; 1024: 207 -> 121), fp32 weights 277 -> 147, the char model 92 -> 36.
//
// What bounded it: a step was 62 dependent launches (124M) of 2.7-4 us each, most of that the boundary, the first loads behind it
// and the fetch of weights nobody could request ahead.  What a hand-over inside a kernel costs depends on how far it goes:
//   within an XCD (32 workgroups, one L2)   0.93 us: a store without scope bits stops in that L2, a load with sc1 passes the L1 and finds it there
//   across XCDs (memory side)               1.2 us, where a word is polled by one workgroup of every XCD only
//   a launch boundary                       1.5-1.9 us in front of a kernel that has loaded nothing yet
// (768-word vectors, every word with its tag.)  So a Block is cut like tensor parallelism, an XCD in a device's place: XCD k owns heads
// k, k + 8, ... and an eighth of the MLP's columns.  Per Block five hand-overs stay inside an XCD and two cross:
//   A  ln_1 + c_attn of the XCD's heads          -> q, k, v      (XCD)
//   B  attention, 64 positions a workgroup       -> partials     (XCD)
//   C  merge + c_proj over the XCD's columns     -> partial sums (all XCDs); a workgroup adds the eight of its E / 32 columns,
//                                                   bias and residual, which stays in registers -> x (XCD)
//   D  ln_2 + c_fc + GELU, an eighth             -> h            (XCD)
//   E  mlp c_proj over that eighth               -> partial sums (all XCDs) -> x (XCD)
// A Block takes 8 to 9 us at 124M; the hand-overs alone 7, the vocabulary's 77 MB 13 of a step's 110 (5.9 TB/s), its pick 2.
//
// What else it needed (us a token at 124M, 256 tokens, as each came in):
//   149  weights of the next Block requested into registers by the waves that poll: a poll returns behind them, loads of a wave being in order
//   163  fetched into the LDS by four waves of their own
//   136  words of other XCDs gathered into one store on cache lines of their own, and not looked at for their first 0.2 us: every
//        store to a line that eight XCDs poll invalidates it in all of them
//   119  the fetches where nobody's word waits behind them in the compute unit's one queue of vector memory (27 B a cycle with fetches in it)
//   117  fewer registers in the vocabulary's loop: a spill there waits for the rows in flight
//   112  no rows requested behind a wave's last (8.25 a half wave: 12 were)
//   110  the pick's value first and then its index; the attention's weights without readlane, and a longer pause behind it
//
// Safety: every workgroup must be resident before any may wait for another.  Workgroups register; the last one commits, and
// one that has waited too long withdraws the launch for all (a compare-and-swap decides, so all agree): then nothing has been
// touched, launches behind it leave at once, and the last one of the generation (decode_rest.hip), which needs no particular number of
// workgroups, runs the steps that are missing.  Behind the commitment every wait is bounded as well (fault word).
#include "decode_resident_parts.h"
#include "zg_once.h"

namespace zg {

namespace {

using namespace resident;
constexpr int kFar = 32;         // words of a workgroup's partial sums: two cache lines of its own
// Pauses, x 64 cycles, measured at 124M and the char model: before the first look at words of other XCDs (0: +4 %; 16: +1 %); before the
// fetches of a Block, behind c_attn's words (0: +10 %; 12: +3 %; 24: +1 %) and behind the attention (4: +5 %; 12: +0.5 %; 32: +2 %)
constexpr int kFarSleep = 8, kAfterA = 20, kAfterB = 18;

// ------------------------------------------------------------------------------------------------ pieces of rows in registers
// N consecutive elements of a row, at a byte offset of 32 bits from a scalar base (the address costs a lane one register)
template <typename WT, int N>
struct Piece;
template <>
struct Piece<bf16_t, 2> {
    uint32_t r;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) { r = *(gptr<const uint32_t>)(base + off); }
    __device__ __forceinline__ void load_lds(unsigned at) { r = lds_read<uint32_t>(at); }
    __device__ __forceinline__ float at(int i) const { return i ? bf16_hi(r) : bf16_lo(r); }
};
template <>
struct Piece<bf16_t, 4> {
    u32x2 r;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) { r = *(gptr<const u32x2>)(base + off); }
    __device__ __forceinline__ void load_lds(unsigned at) { r = lds_read<u32x2>(at); }
    __device__ __forceinline__ float at(int i) const { return i & 1 ? bf16_hi(r[i >> 1]) : bf16_lo(r[i >> 1]); }
};
template <>
struct Piece<bf16_t, 8> {
    u32x4 r;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) { r = *(gptr<const u32x4>)(base + off); }
    __device__ __forceinline__ void load_lds(unsigned at) { r = lds_read<u32x4>(at); }
    __device__ __forceinline__ float at(int i) const { return i & 1 ? bf16_hi(r[i >> 1]) : bf16_lo(r[i >> 1]); }
};
template <>
struct Piece<float, 2> {
    f32x2 r;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) { r = *(gptr<const f32x2>)(base + off); }
    __device__ __forceinline__ void load_lds(unsigned at) { r = lds_read<f32x2>(at); }
    __device__ __forceinline__ float at(int i) const { return i ? r.y : r.x; }
};
template <>
struct Piece<float, 4> {
    f32x4 r;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) { r = *(gptr<const f32x4>)(base + off); }
    __device__ __forceinline__ void load_lds(unsigned at) { r = lds_read<f32x4>(at); }
    __device__ __forceinline__ float at(int i) const { return r[i]; }
};
template <>
struct Piece<float, 8> {
    f32x4 a, b;
    __device__ __forceinline__ void load(const gchar* base, unsigned off) {
        a = *(gptr<const f32x4>)(base + off);
        b = *(gptr<const f32x4>)(base + off + 16);
    }
    __device__ __forceinline__ void load_lds(unsigned at) {
        a = lds_read<f32x4>(at);
        b = lds_read<f32x4>(at + 16);
    }
    __device__ __forceinline__ float at(int i) const { return i < 4 ? a[i & 3] : b[i & 3]; }
};

// acc[0 .. 3] += piece . z, z at the same elements
template <typename WT, int N>
__device__ __forceinline__ void fma_piece(const Piece<WT, N>& w, const float* z, float (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i & 3] = fmaf(w.at(i), z[i], acc[i & 3]);
}
// ------------------------------------------------------------------------------------------------ the words' places
// per XCD: q | k | v of its heads, attention partials, x behind c_proj, h, x behind the MLP; then, for all: partial sums, picks
template <int NW, int NH>
struct Places {
    static constexpr int E = 64 * NW;
    static constexpr int qkv = 0, att = qkv + NH * 192, x1 = att + ((kRanks * kPartStride + 15) & ~15), h = x1 + E, x2 = h + E / 2, best = x2 + E, near_words = best + 2 * kRanks;
    static constexpr int far1 = kXcds * near_words, far2 = far1 + kXcds * kRanks * kFar, pick = far2 + kXcds * kRanks * kFar, words = pick + kXcds * 16;
};

// The LDS, in bytes from the start of the dynamic part.  Blocks of weights end on whole turns of the four fetching waves (4 KiB).
template <typename WT, int NW, int NH>
struct Room {
    static constexpr int E = 64 * NW, F = E / 2, CPR = 2 * NW, WB = sizeof(WT);
    static constexpr int turns(int bytes) { return (bytes + 4095) / 4096; }
    static constexpr int nA = turns(6 * NH * E * WB), nC = turns(CPR * NH * 64 * WB), nD = turns(NW * E * WB), nE = turns(CPR * F * WB);
    static constexpr int copies = sizeof(WT) == 2 ? 2 : 1;   // of A and C; fp32: no room for the next Block's beside this one's
    static constexpr int uG = (E * 4 + 1023) / 1024;         // 1 KB pieces of a vector of E floats
    static constexpr int small = 2 * uG * 256;               // floats: ln_1 g | ln_2 g | c2, c3 of the rows of A and D | biases of the columns
    static constexpr int nV = (2 * uG + 2 + 3) / 4, vec = small + 128;
    static constexpr int A = 0, C = A + copies * nA * 4096, D = C + copies * nC * 4096, Eo = D + nD * 4096, V = Eo + nE * 4096, bytes = V + 2 * 4 * vec;
};

// NW: waves of a workgroup that have rows and words = n_embed / 64.  NH: most heads of an XCD.
// Four more waves fetch the weights into the LDS and attend: loads of a wave return in order, so a wave with weights on their way
// would learn of a word's arrival only behind them (measured: 1 us a Block at the first crossing).  A thread polls one word: what
// it finds is the data, and a second word would be a second round trip (700 cycles of 2200 for a hand-over).
template <typename WT, int NW, int NH>
__global__ __launch_bounds__(64 * (NW + 4)) void decode_resident_kernel(const ResidentArgs a) {
    typedef Places<NW, NH> P;
    typedef Room<WT, NW, NH> R;
    constexpr int E = 64 * NW, F = E / 2, CPR = 2 * NW;            // F: columns of the MLP an XCD owns; CPR: columns of x a workgroup adds up
    constexpr unsigned WB = sizeof(WT);
    constexpr int CH = NW % 4 == 0 ? 4 : 2, NC = NW / CH;          // a lane's pieces of a row of E (wave) or of F (half a wave)
    constexpr int RA = (6 * NH + NW - 1) / NW;                     // rows of c_attn a wave has
    constexpr int HC = NH * 64, CC = 2 * NH;                       // columns of c_proj an XCD owns, a lane's share of them
    constexpr int NG = (NW - 1) * 64 / HC;                         // splits gathered at a time; the last wave has their maxima and sums
    constexpr int AW = 4, MS = kRanks / NH;                        // attention: waves, most splits of a head
    constexpr int LC = NW % 4 == 0 ? 8 : 4, LN = 2 * NW / LC, LR = sizeof(WT) == 2 ? 2 : 1;  // lm_head: pieces of a row (half a wave), rows in flight
    static_assert(CH * NC == NW && LC * LN == 2 * NW && 8 * CPR <= E && NW <= 12 && 2 * NH * MS <= 64 && NG >= 1, "shapes");
    static_assert(R::nD + R::nE + R::nA + R::nC + R::nV + 8 < 64, "vmcnt counts to 63");
    static_assert(R::bytes + 24 * 1024 <= 160 * 1024, "LDS");

    extern __shared__ __attribute__((aligned(16))) char s_room[];
    __shared__ __attribute__((aligned(16))) float s_z[2][E];
    __shared__ float2 s_stat[2][16];
    __shared__ __attribute__((aligned(16))) float s_new[192];  // q, k, v
    __shared__ __attribute__((aligned(16))) float s_o[4 * AW][64];
    __shared__ __attribute__((aligned(16))) float s_m[AW], s_l[AW];
    __shared__ __attribute__((aligned(16))) float s_part[MS][HC];
    __shared__ __attribute__((aligned(8))) float s_ml[NH][MS][2];
    __shared__ __attribute__((aligned(16))) float s_h[F];
    __shared__ float s_out[CPR];
    __shared__ float s_bv[16];
    __shared__ int s_bi[16];
    __shared__ unsigned s_rank, s_go, s_fail;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7u;  // HW_REG_XCC_ID
    // ---- register; all workgroups resident, or nobody starts
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
    const int H = a.n_heads;
    const int nh = k < H ? (H - k + kXcds - 1) / kXcds : 0;       // heads of this XCD: k, k + 8, ...
    const int G = nh > 0 ? kRanks / nh : kRanks;                  // workgroups of a head
    const int hi = min(r / G, NH - 1), sp = r % G;                // this workgroup's head and 64 positions
    const int head = (k < H ? k : 0) + kXcds * (hi < nh ? hi : 0);
    u64* const near = a.words + (size_t)k * P::near_words;
    u64* const far1 = a.words + P::far1;
    u64* const far2 = a.words + P::far2;
    u64* const picks = a.words + P::pick;
    // row j of this workgroup's 6 nh rows of c_attn: among the XCD's words, and in the matrix
    auto word_A = [&](int j) { return r * 6 * nh + j; };
    auto row_A = [&](int j) {
        const int n = word_A(j), ih = n / 192, part = (n % 192) / 64;
        return part * E + (k + kXcds * ih) * 64 + (n & 63);
    };

    // The two kinds of waves run loops of their own that meet at the barriers (numbered; B2 and B3 where the workgroup attends, B4
    // where its XCD has heads, B7 and B8 where the step ends in a pick).
    if (wave >= NW) {
        // =========================================================================================== fetch and attend
        const int fw = wave - NW, ft = tid - E;
        auto from = [&](const void* base, int l, size_t bytes) {
            return __builtin_amdgcn_make_buffer_rsrc((void*)base_at(base, (size_t)l * a.w_stride), 0, (int)bytes, 0x00020000);
        };
        constexpr int uE = E * (int)WB / 16, uF = F * (int)WB / 16, uC = HC * (int)WB / 16, uH = 64 * (int)WB / 16;  // 16-byte units of a row
        const unsigned room = lds_at(s_room) + (unsigned)fw * 1024u;
        unsigned oA[R::nA], oC[R::nC], oE[R::nE];
#pragma unroll
        for (int i = 0; i < R::nA; ++i) {
            const int c = min(i * 256 + ft, max(6 * nh * uE - 1, 0));
            oA[i] = (unsigned)((nh > 0 ? row_A(c / uE) : 0) * E) * WB + (unsigned)(c % uE) * 16u;
        }
#pragma unroll
        for (int i = 0; i < R::nC; ++i) {
            const int c = min(i * 256 + ft, CPR * uC - 1), ih = c % uC / uH;
            oC[i] = (unsigned)((r * CPR + c / uC) * E + ((k < H ? k : 0) + kXcds * (ih < nh ? ih : 0)) * 64) * WB + (unsigned)(c % uH) * 16u;
        }
#pragma unroll
        for (int i = 0; i < R::nE; ++i) {
            const int c = min(i * 256 + ft, CPR * uF - 1);
            oE[i] = (unsigned)((r * CPR + c / uF) * 4 * E + k * F) * WB + (unsigned)(c % uF) * 16u;
        }
        auto fetch_A = [&](int l, int copy) {
            const auto b = from(a.c_attn_w, l, 3 * (size_t)E * E * WB);
#pragma unroll
            for (int i = 0; i < R::nA; ++i) dma16(b, oA[i], room + R::A + (R::copies == 2 ? copy : 0) * R::nA * 4096 + i * 4096);
        };
        auto fetch_C = [&](int l, int copy) {
            const auto b = from(a.c_proj_w, l, (size_t)E * E * WB);
#pragma unroll
            for (int i = 0; i < R::nC; ++i) dma16(b, oC[i], room + R::C + (R::copies == 2 ? copy : 0) * R::nC * 4096 + i * 4096);
        };
        auto fetch_D = [&](int l) {
            const auto b = from(a.c_fc_w, l, 4 * (size_t)E * E * WB);
            const unsigned o = (unsigned)((k * F + r * NW) * E) * WB;
#pragma unroll
            for (int i = 0; i < R::nD; ++i) dma16(b, o + fresh((unsigned)min(i * 256 + ft, NW * uE - 1)) * 16u, room + R::D + i * 4096);
        };
        auto fetch_E = [&](int l) {
            const auto b = from(a.mlp_proj_w, l, 4 * (size_t)E * E * WB);
#pragma unroll
            for (int i = 0; i < R::nE; ++i) dma16(b, oE[i], room + R::Eo + i * 4096);
        };
        // c2, c3 of the rows of A (12 each), of D (20 each); c_proj and MLP bias of the columns (32 each)
        auto fetch_V = [&](int l, int to) {
            const unsigned at_v = lds_at(s_room) + R::V + (unsigned)to * (4u * R::vec);
#pragma unroll
            for (int i = 0; i < R::nV; ++i) {
                const int u = i * 4 + fw;
                if (u < 2 * R::uG) {
                    const int c = (u < R::uG ? u : u - R::uG) * 64 + lane;
                    dma16(from(u < R::uG ? a.ln_1_g : a.ln_2_g, l, E * 4), (unsigned)min(c, E / 4 - 1) * 16u, at_v + (unsigned)u * 1024u);
                } else {
                    const int q = min(u - 2 * R::uG, 1);  // 0: rows of A and D, 1: columns (again where nothing is left)
                    const float* v = q == 0 ? (lane < 12 ? a.c_attn_c2 : lane < 24 ? a.c_attn_c3 : lane < 44 ? a.c_fc_c2 : a.c_fc_c3)
                                            : (lane < 32 ? a.c_proj_b : a.mlp_proj_b);
                    const int jA = lane < 12 ? lane : lane - 12;
                    const int n = q == 0 ? (lane < 24 ? (jA < 6 * nh ? row_A(jA) : 0) : k * F + r * NW + min(lane < 44 ? lane - 24 : lane - 44, NW - 1))
                                         : r * CPR + min(lane & 31, CPR - 1);
                    const float* const p = reinterpret_cast<const float*>(reinterpret_cast<const char*>(v) + (size_t)l * a.w_stride) + n;
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(at_v + 4u * R::small + (unsigned)q * 256u), "v"(p) : "memory", "m0");
                }
            }
        };
        KeyRows kv;
        auto load_KV = [&](int l, int T) {  // the cache rows in front of position T - 1
            const size_t slab = (size_t)l * a.kv_stride + (size_t)head * a.ctx * 256;
            load_rows(kv, a.k_cache + slab, a.v_cache + slab, a.ctx, sp * 64 + fw * 16, T, lane);
        };
        constexpr int nKV = 8;
        int vp = 0;
        auto attends = [&](int T) { return hi < nh && sp < (T + 63) >> 6; };
        fetch_V(0, 0);
        fetch_A(0, 0);
        if (R::copies == 2) fetch_C(0, 0);
        if (attends(a.s0 + 1)) load_KV(0, a.s0 + 1);
        in_flight<0>();
        barrier();  // B0
        for (int s = a.s0; s < a.s1; ++s) {
            const int T = s + 1;
            for (int l = 0; l < a.n_layer; ++l) {
                const int ln = l + 1 < a.n_layer ? l + 1 : 0, Tn = l + 1 < a.n_layer ? T : T + 1;
                barrier();  // B1
                if (attends(T)) {  // (here since B6; nobody waits for them behind the fetches)
                    asm volatile("" ::"v"(kv.k[0][0]), "v"(kv.k[0][1]), "v"(kv.v[0]), "v"(kv.v[1]));
                    asm volatile("" ::"v"(kv.k[1][0]), "v"(kv.k[1][1]), "v"(kv.v[2]), "v"(kv.v[3]));
                }
                if (R::copies == 1 && nh > 0) fetch_C(l, 0);
                if (nh > 0) {
                    if (!attends(T)) {
                        __builtin_amdgcn_s_sleep(kAfterA);
                    } else {
                        barrier();  // B2
                        // ---- B
                        float m = kNone, lsum = 0.0f;
                        f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
                        attend_rows<1, true>(&kv, sp * 64 + fw * 16, T, lane, s_new, m, lsum, o);
                        put_share(fw, lane, m, lsum, o, s_o, s_m, s_l);
                        barrier();  // B3
                        __builtin_amdgcn_s_sleep(kAfterB);
                    }
                }
                fetch_D(l);
                fetch_E(l);
                fetch_V(ln, vp ^ 1);
                if (R::copies == 2) {
                    fetch_A(ln, vp ^ 1);
                    if (nh > 0) fetch_C(ln, vp ^ 1);
                }
                if (nh > 0) {
                    if (R::copies == 1) in_flight<R::nD + R::nE + R::nV>();  // C has arrived
                    barrier();  // B4
                    barrier();  // B4a
                    if (R::copies == 1) fetch_A(ln, 0);
                    if (attends(Tn)) {
                        load_KV(ln, Tn);
                        in_flight<R::nE + R::nV + R::nA + (R::copies == 2 ? R::nC : 0) + nKV>();  // D has
                    } else {
                        in_flight<R::nE + R::nV + R::nA + (R::copies == 2 ? R::nC : 0)>();
                    }
                } else {
                    in_flight<R::nE + R::nV + (R::copies == 2 ? R::nA : 0)>();
                }
                barrier();  // B5
                in_flight<0>();
                barrier();  // B6
                barrier();  // B6a
                vp ^= 1;
            }
            if (s >= a.n_prompt) {
                barrier();  // B7
                barrier();  // B8
                barrier();  // B9
            }
            barrier();  // B10
            if (s_fail != 0u) return;
            barrier();  // B11
        }
        return;
    }

    // ================================================================================================ rows and words
    const int colC = l32 * CC;                                    // column among the XCD's
    const int owner = tid < 8 * CPR ? tid >> 3 : -1;              // column of this workgroup a thread helps to add up
    const int ocol = r * CPR + (owner < 0 ? 0 : owner);
    Waiter w{a.spin_limit, &s_fail};
    int vp = 0;
    const unsigned room = lds_at(s_room);
    auto vec = [&](int i) { return lds_read<float>(room + R::V + (unsigned)(vp * R::vec + i) * 4u); };
    constexpr int v_small = R::small;
    // x of this thread's column -> LDS as z, with the row's sums
    auto spread = [&](int b, float x, float z) {
        s_z[b][tid] = z;
        const float sx = wave_allsum(x), sxx = wave_allsum(x * x);
        if (lane == 0) s_stat[b][wave] = float2{sx, sxx};
        barrier();  // B1, B5, B7
    };
    auto stats = [&](int b, float& mean, float& rstd) {
        const float2 v = lane < NW ? s_stat[b][lane] : float2{0.0f, 0.0f};
        const float sx = row16_allsum(v.x), sxx = row16_allsum(v.y);
        mean = lane_value(sx, 0) * (1.0f / (float)E);
        rstd = __builtin_amdgcn_rsqf(lane_value(sxx, 0) * (1.0f / (float)E) - mean * mean + 1e-5f);
    };
    auto dot_wave = [&](const Piece<WT, CH> (&wt)[NC], const float* z) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            float v[CH];
            lds_floats<CH>(z + j * 64 * CH + lane * CH, v);
            fma_piece<WT, CH>(wt[j], v, acc);
        }
        return wave_allsum((acc[0] + acc[1]) + (acc[2] + acc[3]));
    };
    float x, res;
    // the eight partial sums of a column, bias and residual -> x, for this XCD's workgroups
    auto add_up = [&](const u64* from, int n_from, int bias, unsigned to, unsigned tag) {
        if (owner >= 0) {
            const int q = tid & 7;
            const float b = vec(bias + owner);
            __builtin_amdgcn_s_sleep(kFarSleep);
            float v = q < n_from ? w.get(from, (q * kRanks + r) * kFar + owner, tag) : 0.0f;
            v = sum8(v);
            res += v + b;
            if (q == 0) put_near(near, to + ocol, tagged(tag, res));
        }
    };
    __builtin_amdgcn_s_setprio(3);  // in front of the fetching waves wherever both want to issue (1 us a token)
    int pick = a.s0 > a.n_prompt ? a.out_tokens[a.s0 - 1] : 0;
    const float fin_g = a.ln_f_g[tid], fin_b = a.ln_f_b[tid];
    barrier();  // B0
    for (int s = a.s0; s < a.s1; ++s) {
        const int T = s + 1, n_sp = (T + 63) >> 6;
        const unsigned tag0 = a.tag0 + (unsigned)(s - a.s0) * (unsigned)(a.n_layer + 1);
        const int tok = __builtin_amdgcn_readfirstlane(s < a.n_prompt ? a.prompt[s] : s == a.n_prompt ? a.prompt[a.n_prompt - 1] : pick);
        if (s < a.n_prompt && k == 0 && r == 0 && tid == 0) a.out_tokens[s] = tok;
        {
            const gchar *const te = base_at(a.wte, (size_t)tok * E * WB), *const pe = base_at(a.wpe, (size_t)s * E * WB);
            const unsigned b0 = fresh((unsigned)tid * WB), b1 = fresh((unsigned)ocol * WB);
            auto value = [](const gchar* p, unsigned b) -> float {
                if (sizeof(WT) == 2) return __uint_as_float((uint32_t)*(gptr<const bf16_t>)(p + b) << 16);
                return *(gptr<const float>)(p + b);
            };
            x = value(te, b0) + value(pe, b0);
            res = value(te, b1) + value(pe, b1);
        }
        for (int l = 0; l < a.n_layer; ++l) {
            const unsigned tag = tag0 + (unsigned)l;
            spread(0, x, x * vec(tid));  // B1
            if (nh > 0) {
                float yA[RA];
                {   // ---- A
                    float mean, rstd;
                    stats(0, mean, rstd);
#pragma unroll
                    for (int i = 0; i < RA; ++i) {
                        const int j = wave + NW * i;
                        if (j < 6 * nh) {
                            Piece<WT, CH> wA[NC];
#pragma unroll
                            for (int q = 0; q < NC; ++q)
                                wA[q].load_lds(room + R::A + (R::copies == 2 ? vp : 0) * R::nA * 4096 + j * E * WB + (unsigned)(q * 64 * CH + lane * CH) * WB);
                            const float S1 = dot_wave(wA, s_z[0]);
                            yA[i] = fmaf(rstd, fmaf(-mean, vec(v_small + j), S1), vec(v_small + 12 + j));
                            if (lane == 0) put_near(near, P::qkv + word_A(j), tagged(tag, yA[i]));
                        }
                    }
                }
                if (hi < nh && sp < n_sp) {
                    if (tid < 192 && (tid < 64 || sp == n_sp - 1)) {  // the newest position's key and value: where it belongs
                        const float v = w.get(near, P::qkv + hi * 192 + tid, tag);
                        s_new[tid] = v;
                    }
                    barrier();  // B2
                    barrier();  // B3
                    if (wave == 0) {
                        float m, lsum, o;
                        merge_waves(lane, s_o, s_m, s_l, m, lsum, o);
                        const unsigned to = P::att + (hi * G + sp) * kPartStride + lane;
                        if (lane < 2) put_near(near, to + 64, tagged(tag, lane ? lsum : m));
                        put_near(near, to, tagged(tag, o));
                    }
                }
#pragma unroll
                for (int i = 0; i < RA; ++i) {  // the cache, while the partials are on their way
                    const int j = wave + NW * i;
                    if (j < 6 * nh) {
                        const int row = row_A(j), part = row / E, c = row % E;
                        if (part > 0 && lane == 0)
                            *(gptr<float>)base_at((part == 1 ? a.k_cache : a.v_cache) + (size_t)l * a.kv_stride + ((size_t)(c >> 6) * a.ctx + (T - 1)) * 256 + (c & 63) * 4) = yA[i];
                    }
                }
                // ---- C
                Piece<WT, CC> wC;
                if (wave == NW - 1) {
                    const int ih = lane / (2 * MS), q = lane / 2 % MS;
                    if (ih < nh && q < n_sp) s_ml[ih][q][lane & 1] = w.get(near, P::att + (ih * G + q) * kPartStride + 64 + (lane & 1), tag);
                } else {
                    const int c = tid % HC, ih = c >> 6;
                    if (ih < nh)
                        for (int q = tid / HC; q < n_sp; q += NG) s_part[q][c] = w.get(near, P::att + (ih * G + q) * kPartStride + (c & 63), tag);
                }
                barrier();  // B4
                {
                    wC.load_lds(room + R::C + (R::copies == 2 ? vp : 0) * R::nC * 4096 + ((2 * wave + half) * HC + colC) * WB);
                    const int ih = colC >> 6;
                    float z[CC], zo[CC], acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    float m = kNone, lsum = 0.0f;
#pragma unroll
                    for (int c = 0; c < CC; ++c) z[c] = 0.0f;
                    for (int q0 = 0; q0 < n_sp; q0 += 4) {  // four splits at a time: their reads overlap
                        f32x2 ml[4];
                        float mn = m;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            ml[q] = *reinterpret_cast<const f32x2*>(s_ml[ih][min(q0 + q, n_sp - 1)]);
                            mn = fmaxf(mn, ml[q].x);
                        }
                        const float e0 = __expf(m - mn);
                        lsum *= e0;
#pragma unroll
                        for (int c = 0; c < CC; ++c) z[c] *= e0;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            if (q0 + q < n_sp) {
                                const float e = __expf(ml[q].x - mn);
                                lsum = fmaf(e, ml[q].y, lsum);
                                lds_floats<CC>(&s_part[q0 + q][colC], zo);
#pragma unroll
                                for (int c = 0; c < CC; ++c) z[c] = fmaf(e, zo[c], z[c]);
                            }
                        }
                        m = mn;
                    }
                    fma_piece<WT, CC>(wC, z, acc);
                    const float y = group_allsum<32>(ih < nh ? ((acc[0] + acc[1]) + (acc[2] + acc[3])) * (1.0f / lsum) : 0.0f);
                    if (l32 == 0) s_out[2 * wave + half] = y;
                    barrier();  // B4a
                    if (tid < CPR) put_far(far1, (k * kRanks + r) * kFar + tid, tagged(tag, s_out[tid]));
                }
            } else if constexpr (NW < kFar1From) {  // far2 has been read here (decode_resident_order.h)
                if (tid < CPR) put_far(far1, (k * kRanks + r) * kFar + tid, tagged(tag, 0.0f));
            }
            add_up(far1, kFar1From, v_small + 64, P::x1, tag);
            x = w.get(near, P::x1 + tid, tag);
            // ---- D
            spread(1, x, x * vec(R::uG * 256 + tid));  // B5
            {
                Piece<WT, CH> wD[NC];
#pragma unroll
                for (int q = 0; q < NC; ++q) wD[q].load_lds(room + R::D + (unsigned)(wave * E + q * 64 * CH + lane * CH) * WB);
                float mean, rstd;
                stats(1, mean, rstd);
                const float S1 = dot_wave(wD, s_z[1]);
                const float y = gelu_ref(fmaf(rstd, fmaf(-mean, vec(v_small + 24 + wave), S1), vec(v_small + 44 + wave)));
                if (lane == 0) put_near(near, P::h + r * NW + wave, tagged(tag, y));
            }
            // ---- E
            if (tid < F) s_h[tid] = w.get(near, P::h + tid, tag);
            barrier();  // B6
            {
                float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    Piece<WT, CH> wE;
                    wE.load_lds(room + R::Eo + (unsigned)((2 * wave + half) * F + j * 32 * CH + l32 * CH) * WB);
                    float z[CH];
                    lds_floats<CH>(s_h + j * 32 * CH + l32 * CH, z);
                    fma_piece<WT, CH>(wE, z, acc);
                }
                const float y = group_allsum<32>((acc[0] + acc[1]) + (acc[2] + acc[3]));
                if (l32 == 0) s_out[2 * wave + half] = y;
                barrier();  // B6a
                if (tid < CPR) put_far(far2, (k * kRanks + r) * kFar + tid, tagged(tag, s_out[tid]));
            }
            add_up(far2, kXcds, v_small + 96, P::x2, tag);
            x = w.get(near, P::x2 + tid, tag);
            vp ^= 1;
        }
        const bool last = s + 1 == a.s1;
        float v = -3.0e38f;
        int i = 0x7fffffff;
        if (s >= a.n_prompt) {  // ---- ln_f + lm_head + argmax (main.zig:189-194, :337)
            const int wg = k * kRanks + r, V = a.vocab;
            const int pairs = (V + 1) >> 1, per = (pairs + kXcds * kRanks - 1) / (kXcds * kRanks);  // two rows at a time, half a wave each
            const int p_end = min((wg + 1) * per, pairs), nj = (p_end - wg * per - wave + NW - 1) / NW;  // (negative: this wave has none)
            Piece<WT, LC> ring[LR][LN];
            auto row_of = [&](int j) { return 2 * (wg * per + wave + NW * j) + half; };
            auto fetch = [&](Piece<WT, LC> (&to)[LN], int j) {
                const unsigned b = fresh((unsigned)(min(row_of(j), V - 1) * E + l32 * LC) * WB);
                const gchar* const p = base_at(a.wte);
#pragma unroll
                for (int q = 0; q < LN; ++q) to[q].load(p, b + q * 32 * LC * WB);
            };
#pragma unroll
            for (int u = 0; u < LR; ++u) fetch(ring[u], u);
            spread(0, x, 0.0f);  // B7
            {
                float mean, rstd;
                stats(0, mean, rstd);
                s_z[1][tid] = fmaf((x - mean) * rstd, fin_g, fin_b);
                barrier();  // B8
            }
            const unsigned at_z = lds_at(&s_z[1][l32 * LC]);  // (read again for every row: in registers z would push others out to memory)
            auto row_dot = [&](const Piece<WT, LC> (&of)[LN], int j, auto behind) {
                float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 0; q < LN; ++q) {
                    float z[LC];
#pragma unroll
                    for (int d = 0; d < LC; d += 4) {
                        const f32x4 v4 = lds_read<f32x4>(fresh(at_z) + (unsigned)(q * 32 * LC + d) * 4u);
                        z[d] = v4.x; z[d + 1] = v4.y; z[d + 2] = v4.z; z[d + 3] = v4.w;
                    }
                    fma_piece<WT, LC>(of[q], z, acc);
                }
                behind();
                const float y = group_allsum<32>((acc[0] + acc[1]) + (acc[2] + acc[3]));
                const int row = row_of(j);
                const bool has = (row >> 1) < p_end && row < V;
                if (has && y > v) {  // rows of a lane ascend: the first of equal values stays
                    v = y;
                    i = row;
                }
                if (last && has && l32 == 0) *(gptr<float>)(base_at(a.logits) + fresh((unsigned)row * 4u)) = y;
            };
            int j0 = 0;
            for (; j0 + LR < nj; j0 += LR) {
#pragma unroll
                for (int u = 0; u < LR; ++u) row_dot(ring[u], j0 + u, [&]() { fetch(ring[u], j0 + u + LR); });
            }
#pragma unroll
            for (int u = 0; u < LR; ++u) row_dot(ring[u], j0 + u, []() {});
            {
                const float v1 = lane_value(v, 32);
                const int i1 = __builtin_amdgcn_readlane(i, 32);
                v = lane_value(v, 0);
                i = __builtin_amdgcn_readlane(i, 0);
                better(v, i, v1, i1);
                if (lane == 0) {
                    s_bv[wave] = v;
                    s_bi[wave] = i;
                }
            }
            barrier();  // B9
            const unsigned tag = tag0 + (unsigned)a.n_layer;
            if (wave == 0) {  // the workgroup's, the XCD's, all of them: (value, index) in neighbouring words, a lane has one of the two
                auto pair_up = [&](float word_) {
                    const float other = __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(word_), 0xB1, 0xF, 0xF, true));
                    v = lane & 1 ? -3.0e38f : word_;
                    i = lane & 1 ? 0x7fffffff : __float_as_int(other);
                };
                v = s_bv[min(lane, NW - 1)];
                i = s_bi[min(lane, NW - 1)];
                argmax_row(v, i);  // (the first row has them all)
                if (lane < 2) put_near(near, P::best + 2 * r + lane, tagged(tag, lane ? __int_as_float(i) : v));
                if (r == 0) {
                    pair_up(w.get(near, P::best + lane, tag));
                    argmax_wave(v, i);
                    if (lane < 2) put_far(picks, 16 * k + lane, tagged(tag, lane ? __int_as_float(i) : v));
                }
                __builtin_amdgcn_s_sleep(kFarSleep);
                pair_up(w.get(picks, (unsigned)((lane >> 1 & 7) * 16 + (lane & 1)), tag));
                argmax_row(v, i);
                if (lane == 0) {
                    s_bv[12] = v;
                    s_bi[12] = i;
                }
            }
        }
        barrier();  // B10
        if (s_fail != 0u) {  // a wait ran out: results are worthless and everyone leaves
            if (tid == 0) __hip_atomic_store(a.fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
        if (s >= a.n_prompt) {
            v = s_bv[12];
            i = s_bi[12];
            // logits that are all NaN: index 0, never one behind the table (embed_step_kernel)
            pick = __builtin_amdgcn_readfirstlane((unsigned)i < (unsigned)a.vocab ? i : 0);
            if (k == 0 && r == 0) {
                if (tid == 0) a.out_tokens[s] = pick;
                if (last)  // for the launches that may follow: one partial holds the pick
                    for (int q = tid; q < a.n_part; q += E) {
                        a.part_val[q] = q == 0 ? v : -3.0e38f;
                        a.part_idx[q] = q == 0 ? i : 0x7fffffff;
                    }
            }
        }
        if (last && k == 0 && r == 0) {
            a.x[tid] = x;
            if (tid == 0) {
                a.cur_token[0] = tok;
                a.ctrl->seq_len = T;
                a.ctrl->step = T;
                a.ctl->done = (unsigned)T;
            }
        }
        barrier();  // B11
    }
}

template <typename WT, int NW, int NH>
int launch(const ResidentArgs& a, hipStream_t s) {
    note_kernel("decode_resident_kernel<%s, %d, %d>", sizeof(WT) == 2 ? "unsigned short" : "float", NW, NH);
    constexpr int kOneEach = Room<WT, NW, NH>::bytes > 84 * 1024 ? Room<WT, NW, NH>::bytes : 84 * 1024;  // more than half of a compute unit's LDS: one workgroup each
    static OncePerDevice once;
    int dev = 0;
    ZG_HIP(hipGetDevice(&dev));
    ZG_TRY(once.run(dev, [&]() -> int {
        ZG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&decode_resident_kernel<WT, NW, NH>), hipFuncAttributeMaxDynamicSharedMemorySize, kOneEach));
        return ZG_OK;
    }));
    hipLaunchKernelGGL((decode_resident_kernel<WT, NW, NH>), dim3(kXcds * kRanks), dim3(64 * (NW + 4)), kOneEach, s, a);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace

// (Two layers at least: the cache rows of the next step's first layer are requested during the last layer of this one, which has to be
// another for the newest row to be known to have arrived.  Rows of the vocabulary are found by 32-bit offsets of bytes.)
// Widths: the kernels are built for 384, 512 and 768, what was there to measure.  640 (10 waves with rows, heads on eight XCDs as 2, 2, 1, ...) would
// be another instance and has not been; from 832 on a workgroup of n_embed / 64 + 4 waves is more than the 1024 threads there are.
bool resident_shape(size_t n_embed, size_t n_heads, size_t ctx, size_t n_layer, size_t vocab) {
    if (n_heads * 64 != n_embed || n_heads > 16 || n_layer < 2 || vocab < 1 || vocab > 0xffffffffu / (n_embed * 4)) return false;
    const size_t nw = n_embed / 64;
    if (nw != 6 && nw != 8 && nw != 12) return false;
    return ctx <= 64 * (n_heads > 8 ? kRanks / 2 : kRanks);  // a workgroup attends to 64 positions of one head
}

size_t resident_words(size_t n_embed, size_t batch) {
    if (batch > 1) return resident_batch_words(n_embed);
    switch (n_embed / 64) {
        case 6: return Places<6, 1>::words;
        case 8: return Places<8, 1>::words;
        case 12: return Places<12, 2>::words;
        default: return 0;
    }
}

int launch_decode_resident(const ResidentArgs& a, int n_embed, int weight_type, hipStream_t s) {
    ZG_REQUIRE(resident_shape((size_t)n_embed, (size_t)a.n_heads, (size_t)a.ctx, (size_t)a.n_layer, (size_t)a.vocab) && a.s0 >= 0 && a.s0 < a.s1 && a.s1 <= a.ctx && a.n_prompt >= 1, ZG_ERR_ARG, "resident decode: bad arguments");
    if (a.batch > 1) {
        ZG_REQUIRE(weight_type == WT_BF16, ZG_ERR_UNSUPPORTED, "resident decode: several sequences with fp32 weights");
        return launch_decode_resident_batch(a, n_embed, s);
    }
#define ZG_CASE(nw, nh)                                                         \
    case nw:                                                                     \
        return weight_type == WT_BF16 ? launch<bf16_t, nw, nh>(a, s) : launch<float, nw, nh>(a, s);
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
