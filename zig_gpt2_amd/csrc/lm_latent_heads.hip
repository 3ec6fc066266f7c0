// lm_latent_heads.hip — latent attention of prompt portions, over keys and values of the heads' own.
//
// In the latent space a (query, key) pair of a head costs KR + R products for its score and KR for its value (544 with latents of 256 + 32); with the
// key uk c and the value uv c of the head itself it costs D + R and V (160).  What brings queries into the latent space and results out of it, two
// launches in front and behind, becomes one launch that brings every cached latent into the heads', and the queries are read where the projection left them.
// A portion pays for the keys in front of it again, so it has to have enough rows (latent_heads_fit).
// us a layer, latents of 256 + 32, in the latent space : here, bf16 mode: 8 x 1023 tokens, 16 heads: queries 33, tiles 9, attention 107, values 25 : keys 28, attention 42;
// 8 x 256 tokens, 12 heads: 8 + 8 + 29 + 8 : 13.6 + 15.2.  The attention is bound by the vector work of its softmax beside ten products a tile, the keys'
// launch by a workgroup's chain from the weights over its tiles.  32-bit mode, 1 x 333 tokens, 12 heads: queries 9 + 3, attention 32, values 9 : 8.4 + 15.7.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "lm_latent_parts.h"
#include "lm_quotient.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;

// 32 cached tokens of one entry, as the waves' fragments of 1 KB: the rotated key part, which all heads share (two pieces of 16 channels), the angles
// of its positions ([token][pair] cosine and sine, what the queries are rotated by), and for every head four pieces of its keys (16 channels each) and
// four of its values ([16 tokens][32 channels]).  A piece is [lane] 16 bytes; which 16 of a fragment's 32 x 16 values are a lane's is the matrix
// instruction's layout of results, so that a result is a fragment as it lies: of 16 channels (tokens) a lane has 4 half + 0..3 and 8 + 4 half + 0..3.
// In 32-bit mode the same values are fp32, pieces of 8 channels (tokens) of which a lane has 4 half + 0..3.
constexpr int kD = 64, kR = 32, kV = 64;
template <bool F32>
struct Record {
    static constexpr int EL = F32 ? 4 : 2, ANGLES = 32 * kR * EL, HEADS = ANGLES + 32 * (kR / 2) * 8, VALUES = 32 * kD * EL, HEAD = VALUES + 32 * kV * EL;
    static __host__ __device__ constexpr size_t bytes(int H) { return HEADS + (size_t)H * HEAD; }
};

struct Entry {
    int first_tile, tiles;      // key tiles of the entries in front of it, its own
    int start, len, pos, slot;  // first row, rows, position of the first row, cache slot
};
__device__ __forceinline__ int below(int v, int lane) {  // the sum over this lane and those below
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}
// ITEMS: item `id` of the attention, its entry, head and block of BQ rows; else the entry of key tile `id`.  Entries are looked at 64 at a time.
// Items of the same blocks from the end are neighbours, those with the most keys first: workgroups that start together and share a compute unit (every
// 32nd of an XCD) have blocks of all lengths, and a head's blocks meet in one XCD where entries times heads are a multiple of eight.
template <bool ITEMS>
__device__ __forceinline__ bool find(int id, const int* ent_start, const int* ent_len, const int* ent_slot, int n_entries, const int* row_pos, int bq, int H, Entry& at, int& h, int& block) {
    const int lane = threadIdx.x & 63;
    int tiles_before = 0;
    for (int e0 = 0; e0 < n_entries; e0 += 64) {
        const int e = min(e0 + lane, n_entries - 1);
        const int len = e0 + lane < n_entries ? ent_len[e] : 0, start = ent_start[e], slot = ent_slot[e];
        const int pos = row_pos[start], tiles = len > 0 ? (pos + len + 31) / 32 : 0, blocks = (len + bq - 1) / bq;
        const int t = below(tiles, lane), all_tiles = __builtin_amdgcn_readlane(t, 63);
        int l = -1;
        if constexpr (ITEMS) {
            const int all = __builtin_amdgcn_readlane(below(blocks, lane), 63) * H;
            if (id < all)
                for (int level = 0;; ++level) {
                    const unsigned long long has = __ballot(blocks > level);
                    const int n = __builtin_popcountll(has);
                    if (id < n * H) {
                        h = id / n;
                        l = __builtin_ctzll(__ballot((has >> lane & 1ull) && __builtin_popcountll(has & ((1ull << lane) - 1ull)) == id - h * n));
                        block = __builtin_amdgcn_readlane(blocks, l) - 1 - level;
                        break;
                    }
                    id -= n * H;
                }
            else id -= all;
        } else if (id < tiles_before + all_tiles) l = __builtin_ctzll(__ballot(id < tiles_before + t));
        if (l >= 0) {
            at.start = __builtin_amdgcn_readlane(start, l);
            at.len = __builtin_amdgcn_readlane(len, l);
            at.pos = __builtin_amdgcn_readlane(pos, l);
            at.slot = __builtin_amdgcn_readlane(slot, l);
            at.tiles = __builtin_amdgcn_readlane(tiles, l);
            at.first_tile = tiles_before + __builtin_amdgcn_readlane(t, l) - at.tiles;
            return true;
        }
        tiles_before += all_tiles;
    }
    return false;
}

__device__ __forceinline__ u32x4 eight(const f32x16& v, int at) {
    return u32x4{cvt_pk_bf16(v[at], v[at + 1]), cvt_pk_bf16(v[at + 2], v[at + 3]), cvt_pk_bf16(v[at + 4], v[at + 5]), cvt_pk_bf16(v[at + 6], v[at + 7])};
}

struct KeysArgs {
    const float* cache;
    const bf16_t *ukT, *uv;
    const int *ent_start, *ent_len, *ent_slot, *row_pos, *page_table;
    char* out;
    int H, n_entries, max_pages, page_tokens, n_tiles, per;
    Rotary rot;
};

constexpr int kMostTiles = 8;  // of a workgroup
struct KeysShared {
    int row[32 * kMostTiles], tokens[kMostTiles], pos[kMostTiles];  // cache rows of the tiles' tokens; how many a tile has; position of its first
    unsigned bad[3];                                                // tokens with a latent value that is not finite (as bf16)
};

// The keys (or the values) of two heads for `per` tiles of 32 cached tokens: a wave keeps the weights of 32 channels (by KR: 64 registers) and passes the
// tiles by them.  The tiles come from the cache in whole rows, two tiles ahead, and turn into fragments of bf16 in the LDS.
// Keys are multiplied as uk c^T and values as c uv^T, so that either result lies as the attention's fragment.
// A latent with a value that is not finite is left out (a weight of zero times it would reach queries that do not see the key), and its rotated part
// says so (NaN): the queries that see the key come out NaN.  Values are kept finite for the same reason.
// F32 (32-bit mode): a latent as its exact three bf16 terms, three products each, the second and third terms' with sums of their own; one buffer.
template <int KS, bool V, bool F32>  // KR = 16 KS
__device__ __forceinline__ void head_keys(const KeysArgs& a, char* s_mem, KeysShared& sh) {
    typedef Record<F32> REC;
    constexpr int NP = F32 ? 3 : 1;
    constexpr int KR = 16 * KS, DT = KR + kR, NL = KR / 32, CH = KR / 4, STEP = 1024 + 16;  // 16-byte pieces of a tile a lane loads; of a row; bytes from k-step to k-step
    constexpr int PITCH = V ? KR * 2 + 8 : kD * 2, HEAD = V ? 64 * PITCH : KR * PITCH, NW = KR / 16;  // of the weights in the LDS (other banks); 16-byte pieces a lane loads
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, hf = lane >> 5, j = wave & 1;  // channels 32 j ..
    const int t0 = blockIdx.x * a.per, t_end = min(a.n_tiles, t0 + a.per), h = 2 * blockIdx.y + (wave >> 1);
    const int n = t_end - t0;
    const bool shared_part = !V && blockIdx.y == 0;
    u32x4 raw[NW];  // the weights' rows
#pragma unroll
    for (int i = 0; i < NW; ++i)
        raw[i] = reinterpret_cast<const u32x4*>((V ? a.uv : a.ukT) + (size_t)min((int)(2 * blockIdx.y) + i / (NW / 2), a.H - 1) * KR * 64)[tid + 256 * (i % (NW / 2))];
    __builtin_amdgcn_sched_barrier(0);
    // Where the tokens of the tiles lie: looked up here, so that the loop's loads are rows alone (a page asked for there was waited for together with the
    // rows in flight: 8184 tokens of 16 heads 33 us, here 29).
    {
        Entry at;
        at.first_tile = at.tiles = 0;
        int none = 0;
        for (int l = 0; l < n; ++l) {
            if (t0 + l >= at.first_tile + at.tiles && !find<false>(t0 + l, a.ent_start, a.ent_len, a.ent_slot, a.n_entries, a.row_pos, 32, a.H, at, none, none)) return;
            const int pos = (t0 + l - at.first_tile) * 32, tokens = min(32, at.pos + at.len - pos);
            if (tid >> 5 == l) {
                const int at_pos = pos + min(tid & 31, tokens - 1);  // (beyond the last token: it again)
                sh.row[tid] = a.page_table[(size_t)at.slot * a.max_pages + at_pos / a.page_tokens] * a.page_tokens + at_pos % a.page_tokens;
                sh.tokens[l] = tokens;
                sh.pos[l] = pos;
            }
        }
    }
    if (tid < 3) sh.bad[tid] = 0;
    const float freq = a.rot.freq[tid % (kR / 2)];
    f32x4 next[2][NL], rope_next[2];
    auto fetch = [&](auto which, int l) {  // (no such tile: the last again, not used)
        const int* row = sh.row + min(l, n - 1) * 32;
#pragma unroll
        for (int i = 0; i < NL; ++i) next[which][i] = *reinterpret_cast<const f32x4*>(a.cache + (size_t)row[(tid + 256 * i) / CH] * DT + (tid + 256 * i) % CH * 4);
        rope_next[which] = *reinterpret_cast<const f32x4*>(a.cache + (size_t)row[tid >> 3] * DT + KR + (tid & 7) * 4);
    };
    // The weights by way of the LDS: ukT is [KR][64] for the queries' way into the latent space and is read back transposed.
    u32x4 w[KS];
    {
        __syncthreads();
        fetch(std::integral_constant<int, 0>(), 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int x = tid + 256 * (i % (NW / 2));
            char* to = s_mem + i / (NW / 2) * HEAD + (V ? x / (KR / 8) * PITCH + x % (KR / 8) * 16 : x * 16);
            *reinterpret_cast<u32x2*>(to) = u32x2{raw[i].x, raw[i].y};
            *reinterpret_cast<u32x2*>(to + 8) = u32x2{raw[i].z, raw[i].w};
        }
    }
    __syncthreads();
    const int i16 = lane & 15, G = (lane >> 4) & 1;
    typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;
    const char* s_w = s_mem + (wave >> 1) * HEAD;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if constexpr (V) {
            const char* p = s_w + (j * 32 + r) * PITCH + (s * 16 + 4 * hf) * 2;
            const u32x2 lo = *reinterpret_cast<const u32x2*>(p), hi = *reinterpret_cast<const u32x2*>(p + 16);
            w[s] = u32x4{lo.x, lo.y, hi.x, hi.y};
        } else {
            const char* p = s_w + (s * 16 + 4 * hf + (i16 >> 2)) * PITCH + (j * 32 + 16 * G + 4 * (i16 & 3)) * 2;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 8 * PITCH));
            w[s] = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
    __syncthreads();
    fetch(std::integral_constant<int, 1>(), 1);
    int slot = 0;
    auto body = [&](auto buf, int l) {
        const int keys = __builtin_amdgcn_readfirstlane(sh.tokens[l]), pos = sh.pos[l];
        const f32x4 rope = rope_next[buf];
        char* const tile = s_mem + (F32 ? 0 : buf * (KS * STEP));
        if (F32) __syncthreads();  // (the tile in front has been read)
        constexpr unsigned kTop = F32 ? 0x7F800000u : 0x7F7F8000u;  // from here on a value is not finite, rounds to an infinity
        unsigned most = 0;
#pragma unroll
        for (int i = 0; i < NL; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) most = max(most, __float_as_uint(next[buf][i][u]) & 0x7FFFFFFFu);
        if (__builtin_expect(keys < 32 || __any(most >= kTop), 0)) {
            unsigned bad = 0;
#pragma unroll
            for (int i = 0; i < NL; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int key = (tid + 256 * i) / CH;
                    const bool fine = (__float_as_uint(next[buf][i][u]) & 0x7FFFFFFFu) < kTop;
                    bad |= fine ? 0u : 1u << key;
                    next[buf][i][u] = fine && key < keys ? next[buf][i][u] : 0.0f;
                }
            if (bad) atomicOr(&sh.bad[slot], bad);  // (tokens beyond the last repeat it, and nobody sees them)
        }
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int key = (tid + 256 * i) / CH, c = (tid + 256 * i) % CH;
            f32x4 v = next[buf][i];
            // (k-steps lie 16 bytes more than their size apart, so that a row's pieces go to different banks)
            char* const to = tile + (c >> 2) * STEP + ((c & 1) * 32 + key) * 16 + ((c >> 1) & 1) * 8;
            if constexpr (!F32) *reinterpret_cast<u32x2*>(to) = u32x2{cvt_pk_bf16(v.x, v.y), cvt_pk_bf16(v.z, v.w)};
            else
#pragma unroll
                for (int t = 0; t < 3; ++t) {  // 24 mantissa bits = 8 + 8 + 8, cut off
                    uint32_t b[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        b[u] = __float_as_uint(v[u]);
                        v[u] -= __uint_as_float(b[u] & 0xFFFF0000u);
                    }
                    *reinterpret_cast<u32x2*>(to + t * (KS * STEP)) = u32x2{__builtin_amdgcn_perm(b[1], b[0], 0x07060302u), __builtin_amdgcn_perm(b[3], b[2], 0x07060302u)};
                }
        }
        __syncthreads();
        fetch(buf, l + 2);
        char* rec = a.out + (size_t)(t0 + l) * REC::bytes(a.H);
        if (shared_part) {
            const int key = tid >> 3, c = tid & 7;
            f32x4 v = key < keys ? rope : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (c == 0 && (sh.bad[slot] >> key & 1u)) v.x = __uint_as_float(0x7FC00000u);
            if (F32) *reinterpret_cast<f32x4*>(rec + (c >> 1) * 1024 + ((c & 1) * 32 + key) * 16) = v;
            else *reinterpret_cast<u32x2*>(rec + (c >> 2) * 1024 + ((c & 1) * 32 + key) * 16 + ((c >> 1) & 1) * 8) = u32x2{cvt_pk_bf16(v.x, v.y), cvt_pk_bf16(v.z, v.w)};
}
        if (V)  // (the angles of a tile, 64 a wave, dealt over the heads: with all in the first head's workgroups 1.3 us more)
#pragma unroll 1
            for (int x = wave * (int)gridDim.y + (int)blockIdx.y; x < 32 * (kR / 2) / 64; x += 4 * (int)gridDim.y) {
                const float angle = (float)(pos + 4 * x + lane / (kR / 2)) * freq;
                reinterpret_cast<f32x2*>(rec + REC::ANGLES)[64 * x + lane] = f32x2{cosf(angle) * a.rot.amp, sinf(angle) * a.rot.amp};
            }
        f32x16 acc, small;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = small[e] = 0.0f;
        auto part = [&](int x) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(tile + x * STEP + lane * 16)); };  // k-step x % KS of term x / KS
        constexpr int AHEAD = 4;  // (fragments on their way)
        bf16x8 c[AHEAD];
#pragma unroll
        for (int x = 0; x < AHEAD; ++x) c[x] = part(NP * KS - 1 - x);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < NP * KS; ++x) {  // the smallest term first
            const int at = NP * KS - 1 - x;
            const bf16x8 ws = __builtin_bit_cast(bf16x8, w[at % KS]);
            f32x16& to = at >= KS ? small : acc;
            to = V ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[x % AHEAD], ws, to, 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x16_bf16(ws, c[x % AHEAD], to, 0, 0, 0);
            if (x + AHEAD < NP * KS) c[x % AHEAD] = part(at - AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (F32) acc += small;
        if (V) {
            constexpr float kMost = F32 ? 3.40282347e38f : 3.38953139e38f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {  // (NaN stays)
                acc[e] = acc[e] > kMost ? kMost : acc[e];
                acc[e] = acc[e] < -kMost ? -kMost : acc[e];
            }
        }
        if (h < a.H) {
            char* to = rec + REC::HEADS + (size_t)h * REC::HEAD + (V ? REC::VALUES : 0) + lane * 16;
            if constexpr (F32) {
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(to + (4 * j + g) * 1024) = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
            } else {
#pragma unroll
                for (int x = 0; x < 2; ++x) *reinterpret_cast<u32x4*>(to + (V ? 2 * x + j : 2 * j + x) * 1024) = eight(acc, 8 * x);
            }
        }
        if (tid == 0) sh.bad[slot == 0 ? 2 : slot - 1] = 0;  // (the slot of the tile in front: read before this tile's barrier, written next behind the next one's)
        slot = slot == 2 ? 0 : slot + 1;
    };
    for (int l = 0; l < n; l += 2) {
        body(std::integral_constant<int, 0>(), l);
        if (l + 1 < n) body(std::integral_constant<int, 1>(), l + 1);
    }
}

template <int KS, bool F32>
__global__ __launch_bounds__(256, 2) void latent_head_keys_kernel(const KeysArgs a) {
    constexpr int KR = 16 * KS, TILES = (F32 ? 3 : 2) * KS * 1040, WEIGHTS = 2 * 64 * (KR * 2 + 8);
    __shared__ __attribute__((aligned(1024))) char s_mem[TILES > WEIGHTS ? TILES : WEIGHTS];
    __shared__ KeysShared sh;
    if (blockIdx.z == 0) head_keys<KS, false, F32>(a, s_mem, sh);
    else head_keys<KS, true, F32>(a, s_mem, sh);
}

struct HeadsArgs {
    const float* q;
    const char* keys;
    bf16_t* out;
    float* out32;
    const float *gate, *sink;
    const int *ent_start, *ent_len, *ent_slot, *row_pos;
    int ldq, ldo, ldg, H, n_entries, halves;
    float scale;
};

// A query's rotated part, channel 8 i + 4 half + u of it in v[8 + i][u], by its position's cosines and sines.
__device__ __forceinline__ void rotate(f32x4 (&v)[12], const f32x2* cs, int halves, int hf) {
    if (halves) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const f32x2 c = cs[8 * i + 4 * hf + u];
                const float x = v[8 + i][u], y = v[10 + i][u];
                v[8 + i][u] = x * c.x - y * c.y;
                v[10 + i][u] = y * c.x + x * c.y;
            }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 4; u += 2) {
                const f32x2 c = cs[4 * i + 2 * hf + u / 2];
                const float x = v[8 + i][u], y = v[8 + i][u + 1];
                v[8 + i][u] = x * c.x - y * c.y;
                v[8 + i][u + 1] = y * c.x + x * c.y;
            }
    }
}

// A wave takes 32 queries of one head.  KW = 1: the four waves of a workgroup have queries behind each other and share the tiles of 32 keys; KW = 4: they
// have the same queries and every fourth tile each, and meet in the LDS.  Tiles arrive by DMA as whole fragments, two (four) to a buffer, in two buffers.
// Both products are computed transposed (S^T = K Q^T, O^T = V^T P^T): a lane's column is a query, so the running maximum and sum are the lane's, and the
// probabilities a lane computed are the ones it has to feed back.  Scores, softmax and both accumulations are fp32.
template <int KW>
__global__ __launch_bounds__(256, KW == 1 ? 4 : 2) void latent_heads_kernel(const HeadsArgs a) {
    typedef Record<false> REC;
    constexpr int S = KW == 1 ? 2 : 4, BQ = 32 * (4 / KW), TILE = 2048 + REC::HEAD, PIECES = S * TILE / 1024;  // tiles of a buffer, queries of a workgroup
    __shared__ __attribute__((aligned(1024))) char s_k[2][S * TILE];
    Entry at;
    int h = 0, block = 0;
    if (!find<true>(blockIdx.x, a.ent_start, a.ent_len, a.ent_slot, a.n_entries, a.row_pos, BQ, a.H, at, h, block)) return;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q0 = block * BQ + (KW == 1 ? 32 * wave : 0);  // the wave's first query, in the entry
    const int nq = min(32, at.len - q0);                    // (none: the wave only brings tiles)
    const int m_first = at.start + q0, pos_first = at.pos + q0, qpos = pos_first + r;
    const int my_tiles = nq > 0 ? (pos_first + nq + 31) / 32 : 0, n_tiles = (at.pos + min(at.len, block * BQ + BQ) + 31) / 32, n_iter = (n_tiles + S - 1) / S;
    const size_t record = REC::bytes(a.H);
    const char* src = a.keys + (size_t)at.first_tile * record + lane * 16;
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)&s_k[0][0];
    auto request = [&](int it, int buf) {
#pragma unroll
        for (int i = 0; i < PIECES / 4; ++i) {
            const int p = wave + 4 * i, j = p / 10, x = p - 10 * j;  // (beyond the last tile: the last, not used)
            const char* g = src + (size_t)min(it * S + j, n_tiles - 1) * record + (x < 2 ? x * 1024 : REC::HEADS + h * REC::HEAD + (x - 2) * 1024);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds0 + buf * (S * TILE) + p * 1024), "v"(g) : "memory", "m0");
        }
    };
    static_assert(TILE == 10 * 1024, "ten pieces of a tile");
    request(0, 0);
    bf16x8 qf[6];
    {
        const float* qr = a.q + (size_t)(m_first + (nq > 0 ? min(r, nq - 1) : -q0)) * a.ldq + (size_t)h * (kD + kR) + 4 * hf;  // (beyond the block: some valid row, never stored)
        f32x4 v[12];
#pragma unroll
        for (int i = 0; i < 12; ++i) v[i] = *reinterpret_cast<const f32x4*>(qr + 8 * i);
        const int kp = min(qpos, at.pos + at.len - 1);
        rotate(v, reinterpret_cast<const f32x2*>(a.keys + (size_t)(at.first_tile + kp / 32) * record + REC::ANGLES) + (kp % 32) * (kR / 2), a.halves, hf);
#pragma unroll
        for (int k = 0; k < 6; ++k)
            qf[k] = __builtin_bit_cast(bf16x8, u32x4{cvt_pk_bf16(v[2 * k].x, v[2 * k].y), cvt_pk_bf16(v[2 * k].z, v[2 * k].w), cvt_pk_bf16(v[2 * k + 1].x, v[2 * k + 1].y),
                                                     cvt_pk_bf16(v[2 * k + 1].z, v[2 * k + 1].w)});
    }
    f32x16 o[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;
    float mx = -INFINITY, lsum = 0.0f;  // maximum in units of log2
    const float to_log2 = a.scale * 1.44269502f;
    // vmcnt(0): this wave's pieces have landed; lgkmcnt(0), said to the compiler: with scalar loads in flight it would wait for all fragments at once
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
    for (int it = 0; it < n_iter; ++it) {
        if (it + 1 < n_iter) request(it + 1, (it + 1) & 1);
#pragma unroll
        for (int j = 0; j < (KW == 1 ? S : 1); ++j) {
            const int jt = KW == 1 ? j : wave, kt = it * S + jt;
            if (kt >= my_tiles) continue;
            const char* K = s_k[it & 1] + jt * TILE + lane * 16;
            auto piece = [&](int x) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(K + x * 1024)); };
            bf16x8 kf[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) kf[k] = piece(k < 4 ? 2 + k : k - 4);
            f32x16 sacc;
#pragma unroll
            for (int i = 0; i < 16; ++i) sacc[i] = 0.0f;
#pragma unroll
            for (int k = 0; k < 6; ++k) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[k], qf[k], sacc, 0, 0, 0);
            bf16x8 vf[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) vf[x] = piece(6 + x);
            if (kt * 32 + 31 > pos_first) {  // some query does not see the whole tile
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kt * 32 + 8 * (i >> 2) + 4 * hf + (i & 3) > qpos) sacc[i] = -INFINITY;
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, sacc[i]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64)) * to_log2;
            // The reference point of the exponentials moves only when some query's maximum grew by more than 2^11 (the weights stay far inside fp32 and bf16 range)
            if (__any(tmax > mx + 11.0f)) {  // also the first tile (mx = -inf)
                const float mn = tmax > mx + 11.0f ? tmax : mx;
                const float alpha = mx == mn ? 1.0f : __builtin_amdgcn_exp2f(mx - mn);  // mx = -inf, mn finite: 0
                lsum *= alpha;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[t][i] *= alpha;
                mx = mn;
            }
            const float mref = fmaxf(mx, -1e30f);  // (no key seen so far: 2^(-inf) = 0, not NaN)
            uint32_t pk[8];
            float part[2] = {0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(sacc[2 * i], to_log2, -mref)), p1 = __builtin_amdgcn_exp2f(fmaf(sacc[2 * i + 1], to_log2, -mref));
                part[i & 1] += p0 + p1;
                pk[i] = cvt_pk_bf16(p0, p1);
            }
            lsum += part[0] + part[1];
            const bf16x8 pf[2] = {__builtin_bit_cast(bf16x8, u32x4{pk[0], pk[1], pk[2], pk[3]}), __builtin_bit_cast(bf16x8, u32x4{pk[4], pk[5], pk[6], pk[7]})};
#pragma unroll
            for (int x = 0; x < 4; ++x) o[x & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x], pf[x >> 1], o[x & 1], 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the next tiles' pieces
        __syncthreads();
    }
    float L = lsum + __shfl_xor(lsum, 32, 64);
    // Results leave through the LDS as 16-byte pieces of whole rows.
    constexpr int PITCH = kV * 2 + 16;
    const size_t row = (size_t)(at.start + q0 + (nq > 0 ? min(r, nq - 1) : -q0));
    if constexpr (KW == 1) {
        if (nq <= 0) return;
        char* const img = &s_k[0][0] + wave * (32 * PITCH);
        const float gf = head_gate_f(a.gate, a.ldg, row, h) * (a.sink ? sink_norm_f(mx * 0.69314718055994531f, L, a.sink, h) : 1.0f), inv = 1.0f / L;
        auto value = [&](float v) { return (a.sink ? v : quotient(v, L, inv)) * gf; };
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; i += 4)
                *reinterpret_cast<u32x2*>(img + r * PITCH + (t * 32 + 2 * i + 4 * hf) * 2) = u32x2{cvt_pk_bf16(value(o[t][i]), value(o[t][i + 1])), cvt_pk_bf16(value(o[t][i + 2]), value(o[t][i + 3]))};
        // (a wave's accesses to the LDS are in order)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int qr = 8 * x + (lane >> 3), c = (lane & 7) * 8;
            const u32x4 v = *reinterpret_cast<const u32x4*>(img + qr * PITCH + c * 2);
            if (qr < nq) *reinterpret_cast<u32x4*>(a.out + (size_t)(m_first + qr) * a.ldo + h * kV + c) = v;
        }
    } else {
        // (maximum, sum, values) of every wave; each then has a quarter of the channels
        float* const part = reinterpret_cast<float*>(&s_k[0][0]);
        char* const img = &s_k[0][0] + 4 * 34 * 256;
        float* mine = part + wave * 34 * 64 + lane;
        mine[0] = mx;
        mine[64] = L;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[(2 + t * 16 + i) * 64] = o[t][i];
        __syncthreads();
        float top = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; ++k) top = fmaxf(top, part[k * 34 * 64 + lane]);
        const float ref = fmaxf(top, -1e30f);
        float sum = 0.0f, v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float* p = part + k * 34 * 64 + lane;
            const float f = __builtin_amdgcn_exp2f(p[0] - ref);
            sum = fmaf(p[64], f, sum);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = fmaf(p[(2 + 8 * wave + e) * 64], f, v[e]);
        }
        const float gf = head_gate_f(a.gate, a.ldg, row, h) * (a.sink ? sink_norm_f(top * 0.69314718055994531f, sum, a.sink, h) : 1.0f), inv = 1.0f / sum;
        auto value = [&](float x) { return (a.sink ? x : quotient(x, sum, inv)) * gf; };
#pragma unroll
        for (int i = 0; i < 2; ++i)  // channels 32 (wave / 2) + 16 (wave % 2) + 8 i + 4 half + ..
            *reinterpret_cast<u32x2*>(img + r * PITCH + (16 * wave + 8 * i + 4 * hf) * 2) =
                u32x2{cvt_pk_bf16(value(v[4 * i]), value(v[4 * i + 1])), cvt_pk_bf16(value(v[4 * i + 2]), value(v[4 * i + 3]))};
        __syncthreads();
        const int qr = tid >> 3, c = (tid & 7) * 8;
        if (qr < nq) *reinterpret_cast<u32x4*>(a.out + (size_t)(m_first + qr) * a.ldo + h * kV + c) = *reinterpret_cast<const u32x4*>(img + qr * PITCH + c * 2);
    }
}

// exp(x) for x <= 0 (x log2 e in two pieces; below what fp32 holds: 0)
__device__ __forceinline__ float exp_of(float x) {
    x = x < -150.0f ? -150.0f : x;  // (NaN stays)
    const float t = x * 1.44269502f, rest = fmaf(x, 1.44269502f, -t) + x * 1.92596303e-8f;
    const float p = __builtin_amdgcn_exp2f(t);
    return fmaf(p, rest * 0.693147182f, p);
}

// 32-bit mode: the same in true fp32 (v_mfma_f32_32x32x2_f32), 32 queries of a head to a workgroup, whose four waves take every fourth tile.  Keys and
// values go from memory to registers, whole fragments of 1 KB, 20 of them a tile beside 80 products of 64 cycles, which bound it.
__global__ __launch_bounds__(256, 2) void latent_heads_f32_kernel(const HeadsArgs a) {
    typedef Record<true> REC;
    __shared__ __attribute__((aligned(16))) float s_part[4 * 34 * 64];
    __shared__ __attribute__((aligned(16))) float s_img[32 * (kV + 4)];
    Entry at;
    int h = 0, block = 0;
    if (!find<true>(blockIdx.x, a.ent_start, a.ent_len, a.ent_slot, a.n_entries, a.row_pos, 32, a.H, at, h, block)) return;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q0 = block * 32, nq = min(32, at.len - q0), m_first = at.start + q0, pos_first = at.pos + q0, qpos = pos_first + r, n_tiles = (pos_first + nq + 31) / 32;
    const size_t record = REC::bytes(a.H), row = (size_t)(m_first + min(r, nq - 1));  // (beyond the block: some valid row, never stored)
    const char* src = a.keys + (size_t)at.first_tile * record + lane * 16;
    f32x4 q[12];
    {
        const float* qr = a.q + row * a.ldq + (size_t)h * (kD + kR) + 4 * hf;
#pragma unroll
        for (int i = 0; i < 12; ++i) q[i] = *reinterpret_cast<const f32x4*>(qr + 8 * i);
        const int kp = min(qpos, at.pos + at.len - 1);
        rotate(q, reinterpret_cast<const f32x2*>(a.keys + (size_t)(at.first_tile + kp / 32) * record + REC::ANGLES) + (kp % 32) * (kR / 2), a.halves, hf);
    }
    f32x16 o[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;
    float mx = -INFINITY, lsum = 0.0f;
    f32x4 k[12];
    auto fetch = [&](int kt) {  // (beyond the last tile: the last, not used)
        const char* g = src + (size_t)min(kt, n_tiles - 1) * record;
#pragma unroll
        for (int i = 0; i < 12; ++i) k[i] = *reinterpret_cast<const f32x4*>(g + (i < 8 ? REC::HEADS + (size_t)h * REC::HEAD + i * 1024 : (i - 8) * 1024));
    };
    fetch(wave);
    for (int kt = wave; kt < n_tiles; kt += 4) {
        f32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const f32x4*>(src + (size_t)kt * record + REC::HEADS + (size_t)h * REC::HEAD + REC::VALUES + i * 1024);
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int i = 0; i < 12; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) s = __builtin_amdgcn_mfma_f32_32x32x2f32(k[i][u], q[i][u], s, 0, 0, 0);
        fetch(kt + 4);
        float top = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] *= a.scale;
        if (kt * 32 + 31 > pos_first) {  // some query does not see the whole tile
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (kt * 32 + 8 * (i >> 2) + 4 * hf + (i & 3) > qpos) s[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) top = fmaxf(top, s[i]);
        top = fmaxf(mx, fmaxf(top, __shfl_xor(top, 32, 64)));
        if (__any(top > mx)) {
            const float f = mx == top ? 1.0f : exp_of(mx - top);  // (none so far: 0)
            lsum *= f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[t][i] *= f;
            mx = top;
        }
        const float ref = mx == -INFINITY ? 0.0f : mx;
        float part[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = exp_of(s[i] - ref);
            part[i & 1] += s[i];
        }
        lsum += part[0] + part[1];
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t) o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[4 * t + (i >> 2)][i & 3], s[i], o[t], 0, 0, 0);
    }
    float* mine = s_part + wave * 34 * 64 + lane;
    mine[0] = mx;
    mine[64] = lsum + __shfl_xor(lsum, 32, 64);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) mine[(2 + t * 16 + i) * 64] = o[t][i];
    __syncthreads();
    float top = -INFINITY, sum = 0.0f, v[8];  // a quarter of the channels to a wave
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, s_part[w * 34 * 64 + lane]);
    const float ref = top == -INFINITY ? 0.0f : top;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float* p = s_part + w * 34 * 64 + lane;
        const float f = exp_of(p[0] - ref);
        sum = fmaf(p[64], f, sum);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = fmaf(p[(2 + 8 * wave + e) * 64], f, v[e]);
    }
    const float gf = head_gate_f(a.gate, a.ldg, row, h) * (a.sink ? sink_norm_f(top, sum, a.sink, h) : 1.0f), inv = 1.0f / sum;
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // channels 16 wave + 8 i + 4 half + ..
        f32x4 y;
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = (a.sink ? v[4 * i + u] : quotient(v[4 * i + u], sum, inv)) * gf;
        *reinterpret_cast<f32x4*>(s_img + r * (kV + 4) + 16 * wave + 8 * i + 4 * hf) = y;
    }
    __syncthreads();
#pragma unroll
    for (int x = tid; x < 32 * kV / 4; x += 256) {
        const int qr = x / (kV / 4), c = x % (kV / 4) * 4;
        if (qr < nq) *reinterpret_cast<f32x4*>(a.out32 + (size_t)(m_first + qr) * a.ldo + h * kV + c) = *reinterpret_cast<const f32x4*>(s_img + qr * (kV + 4) + c);
    }
}

}  // namespace

size_t latent_heads_record(int H, int D, int R, int KR, int Vd, int rot_dims, bool f32) {
    return D == kD && R == kR && Vd == kV && rot_dims == kR && (KR == 128 || KR == 256) ? (f32 ? Record<true>::bytes(H) : Record<false>::bytes(H)) : 0;
}

bool latent_heads_fit(const LatentHeads& a) {
    const uintptr_t all = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.cache) | reinterpret_cast<uintptr_t>(a.ukT) | reinterpret_cast<uintptr_t>(a.uv) |
                          reinterpret_cast<uintptr_t>(a.ws) | reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.out32);
    const size_t record = latent_heads_record(a.H, a.D, a.R, a.KR, a.Vd, a.rot.dims, a.out32 != nullptr);
    const PortionSize& p = a.size;
    const char* force = getenv("ZGPT2_LM_LATENT_HEADS");  // test hook: -1 never, 1 or 4 that form of the attention at any size
    const int f = force ? atoi(force) : 0;
    if (f < 0 || record == 0 || !a.ws || p.rows == 0 || p.tiles * record > a.ws_bytes || a.ldq % 4 != 0 || a.ldo % 8 != 0 || (all & 15) != 0 || !(a.scale > 0.0f)) return false;
    if ((long long)p.blocks * a.H >= (1LL << 31) || a.H > 65535) return false;
    // A key costs KR (D + V) products a head whoever sees it, a pair saves 2 KR - D - V.  Portions of few rows behind much are let in as long as that is a
    // short launch: up to 8192 keys of 12 heads (28 us) every shape was faster, whole steps of 9 rows and more on the 12-layer stacks, in the latent space : here,
    // us: 1 x 9 rows behind nothing 909 : 856, behind 1000 1110 : 906, behind 7000 2166 : 1238; 8 x 2 behind 900 1152 : 1069; 8 x 64 behind 256 1399 : 1313.
    // In 32-bit mode the keys' launch is dearer (8 x 2 behind 900 1303 : 1326, 8 x 16 behind 900 1482 : 1490, 8 x 64 behind 900 2093 : 1868, 1 x 9 behind 7000
    // 3023 : 2062, 1 x 9 990 : 967, 1 x 1000 2475 : 1812): there many sequences with few rows stay where they were.
    const bool f32 = a.out32 != nullptr;
    const bool brief = p.all_keys * a.H <= 8192 * 12 && (!f32 || p.all_keys * a.H <= 1024 * 12 || p.all_keys <= 2 * p.longest);
    return f > 0 || brief || (double)(p.all_keys - p.rows) * a.KR * (a.D + a.Vd) <= (f32 ? 2.0 : 0.5) * (double)p.pairs * (2 * a.KR - a.D - a.Vd);
}

int launch_latent_heads(const LatentHeads& a, hipStream_t s) {
    const PortionSize& p = a.size;
    KeysArgs k;
    k.cache = a.cache; k.ukT = a.ukT; k.uv = a.uv; k.ent_start = a.ent_start; k.ent_len = a.ent_len; k.ent_slot = a.ent_slot; k.row_pos = a.row_pos; k.page_table = a.page_table;
    k.out = a.ws; k.H = a.H; k.n_entries = a.n_entries; k.max_pages = a.max_pages; k.page_tokens = a.page_tokens; k.n_tiles = (int)p.tiles; k.rot = a.rot;
    // two workgroups a compute unit where there are as many tiles
    const int pairs = (a.H + 1) / 2;
    k.per = (int)std::max(1ll, std::min<long long>(kMostTiles, (long long)p.tiles * pairs * 2 / 512));
    const dim3 kg((unsigned)((p.tiles + k.per - 1) / k.per), (unsigned)pairs, 2);
    const bool f32 = a.out32 != nullptr;
    if (a.KR == 128) f32 ? latent_head_keys_kernel<8, true><<<kg, 256, 0, s>>>(k) : latent_head_keys_kernel<8, false><<<kg, 256, 0, s>>>(k);
    else f32 ? latent_head_keys_kernel<16, true><<<kg, 256, 0, s>>>(k) : latent_head_keys_kernel<16, false><<<kg, 256, 0, s>>>(k);
    ZG_HIP(hipGetLastError());
    HeadsArgs h;
    h.q = a.q; h.keys = a.ws; h.out = a.out; h.out32 = a.out32; h.gate = a.gate; h.sink = a.sink; h.ent_start = a.ent_start; h.ent_len = a.ent_len; h.ent_slot = a.ent_slot; h.row_pos = a.row_pos;
    h.ldq = a.ldq; h.ldo = a.ldo; h.ldg = a.ldg; h.H = a.H; h.n_entries = a.n_entries; h.halves = a.rot.halves; h.scale = a.scale;
    // Blocks of 128 queries once there are some for most compute units.  us a step of the 12-layer stack, 32 : 128 queries (workgroups of the latter): 1 x 1000 rows
    // (96) 1399 : 1445, 8 x 128 behind 800 (96) 1651 : 1672, 8 x 250 (192) 1755 : 1721, 8 x 256 behind 256 (192) 1847 : 1813.
    const char* force = getenv("ZGPT2_LM_LATENT_HEADS");
    const bool wide = force && atoi(force) > 0 ? atoi(force) == 1 : (long long)p.wide_blocks * a.H >= 160;
    if (f32) latent_heads_f32_kernel<<<(unsigned)(p.blocks * a.H), 256, 0, s>>>(h);
    else if (wide) latent_heads_kernel<1><<<(unsigned)(p.wide_blocks * a.H), 256, 0, s>>>(h);
    else latent_heads_kernel<4><<<(unsigned)(p.blocks * a.H), 256, 0, s>>>(h);
    ZG_HIP(hipGetLastError());
    if (f32) note_kernel("latent_heads_f32_kernel");
    else note_kernel("latent_heads_kernel<%d>", wide ? 1 : 4);
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
