// decode_resident_parts.h — what the resident decode kernels share (decode_resident.hip: one sequence, decode_resident_batch.hip: two to eight in lock step)
#pragma once
#include "decode_resident_order.h"
#include "zg_common.h"
#include "zg_kernels.h"

#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the words of the resident kernels rest on what gfx950's caches do (decode_resident_order.h)"
#endif

namespace zg {
namespace resident {

constexpr float kNone = -1e30f;  // score of a position that is not there

typedef unsigned long long u64;

// A base that stays in scalar registers, an offset that is made again where it is used: without them the compiler keeps some
// sixty loop-invariant 64-bit addresses of every lane in registers it then has to spill.
typedef __attribute__((address_space(1))) char gchar;  // (said to be global memory: the compiler cannot see through the asm)
typedef __attribute__((address_space(1))) u64 gword;
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
__device__ __forceinline__ gchar* base_at(const void* p, size_t off = 0) {
    const char* q = reinterpret_cast<const char*>(p) + off;
    asm volatile("" : "+s"(q));
    return (gchar*)const_cast<char*>(q);
}
__device__ __forceinline__ unsigned fresh(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

// ------------------------------------------------------------------------------------------------ words with tags
__device__ __forceinline__ u64 tagged(unsigned tag, float v) { return ((u64)tag << 32) | (u64)__float_as_uint(v); }
__device__ __forceinline__ gword* word(const u64* base, unsigned i) { return (gword*)(base_at(base) + fresh(i * 8u)); }
// word i of base.  Within the XCD: no bit of a wider scope, the word stays in this L2 (decode_resident_order.h: what this rests on)
__device__ __forceinline__ void put_near(u64* base, unsigned i, u64 v) { __hip_atomic_store(word(base, i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
// for every XCD: written through
__device__ __forceinline__ void put_far(u64* base, unsigned i, u64 v) { __hip_atomic_store(word(base, i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

struct Waiter {
    unsigned limit;  // polls of one wait; 0 once one has run out
    unsigned* fail;  // LDS
    __device__ __forceinline__ u64 wait(const gword* p, unsigned tag) {
        u64 v;
        for (unsigned n = 0;; ++n) {
            v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((unsigned)(v >> 32) == tag) break;
            if (n >= limit) {
                *fail = 1u;
                limit = 0u;
                break;
            }
        }
        return v;
    }
    __device__ __forceinline__ float get(const u64* base, unsigned i, unsigned tag) { return __uint_as_float((unsigned)wait(word(base, i), tag)); }
};

// LDS is exchanged between waves, vector memory is not: loads in flight stay in flight (a __syncthreads() drains them)
__device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ------------------------------------------------------------------------------------------------ the LDS
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ unsigned lds_at(const void* p) { return (unsigned)(uintptr_t)(lds_char*)(p); }
template <typename T>
__device__ __forceinline__ T lds_read(unsigned at) { return *(const __attribute__((address_space(3))) T*)(uintptr_t)at; }
// sum over eight consecutive lanes, on all of them, the same bits on all of them (commutative pairs)
__device__ __forceinline__ float sum8(float v) {
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0xB1, 0xF, 0xF, true));
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x4E, 0xF, 0xF, true));
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x141, 0xF, 0xF, true));
    return v;
}

__device__ __forceinline__ void better(float& v, int& i, float ov, int oi) {  // the larger value, of equal ones the lower index
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

// the largest value and of equal ones the lowest index: over the 16 lanes of a row; over the wave, on all lanes.  (First the value, then the
// index among those that have it: a step is one instruction each, where pairs take five that depend on each other.)
__device__ __forceinline__ int row_min(int i) {
#define ZG_MIN_STEP(N) i = min(i, __builtin_amdgcn_update_dpp(0, i, 0x120 | N, 0xF, 0xF, true));
    ZG_MIN_STEP(8) ZG_MIN_STEP(4) ZG_MIN_STEP(2) ZG_MIN_STEP(1)
#undef ZG_MIN_STEP
    return i;
}
__device__ __forceinline__ void argmax_row(float& v, int& i) {
    const float own = v;
    v = fmaxf(v, dpp_row_ror<8>(v));
    v = fmaxf(v, dpp_row_ror<4>(v));
    v = fmaxf(v, dpp_row_ror<2>(v));
    v = fmaxf(v, dpp_row_ror<1>(v));
    i = row_min(own == v ? i : 0x7fffffff);
}
__device__ __forceinline__ void argmax_wave(float& v, int& i) {
    const float own = v;
    v = wave_allmax(v);
    const int c = row_min(own == v ? i : 0x7fffffff);
    i = min(min(__builtin_amdgcn_readlane(c, 0), __builtin_amdgcn_readlane(c, 16)), min(__builtin_amdgcn_readlane(c, 32), __builtin_amdgcn_readlane(c, 48)));
}

template <int N>
__device__ __forceinline__ void lds_floats(const float* p, float* out) {
    if (N == 2) {
        const float2 v = *reinterpret_cast<const float2*>(p);
        out[0] = v.x;
        out[1] = v.y;
    } else {
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(p + i);
            out[i] = v.x; out[i + 1] = v.y; out[i + 2] = v.z; out[i + 3] = v.w;
        }
    }
}

// ------------------------------------------------------------------------------------------------ weights: memory -> LDS
// 64 lanes x 16 bytes from the lanes' offsets into the LDS from `to` on.  In flight until vmcnt says otherwise.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t from, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(off), "s"(from) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void in_flight() {  // at most N of this wave's vector memory operations
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// ------------------------------------------------------------------------------------------------ attention
// 16 positions of a head, by a wave.  Eight lanes have a position's key, 16 lanes (a row) its values, four each: of eight positions a row has the
// values of the two that it scores, so that a weight is in its row already (or eight lanes away).  readlane for all of them: 0.15 us more
struct KeyRows {
    f32x4 k[2][2], v[4];
};
// The rows from p0 on.  This XCD's workgroups wrote them: past the L1 (sc1), whose lines may be older.  Positions that are not there yet re-read the
// last one that is; they weigh nothing
__device__ __forceinline__ void load_rows(KeyRows& to, char* k_rows, char* v_rows, int ctx, int p0, int T, int lane) {
    const int bytes = ctx * 256, last = max(T - 2, 0);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(k_rows, 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(v_rows, 0, bytes, 0x00020000);
    const int l8 = (int)fresh((unsigned)lane);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int off = min(p0 + i * 8 + (l8 >> 3), last) * 256 + (l8 & 7) * 32;
        to.k[i][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 16));
        to.k[i][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off + 16, 0, 16));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        to.v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, min(p0 + i / 2 * 8 + i % 2 + (l8 >> 4) * 2, last) * 256 + (l8 & 15) * 16, 0, 16));
}
template <typename Op>
__device__ __forceinline__ float over_rows(float v, Op op) { return op(op(lane_value(v, 0), lane_value(v, 16)), op(lane_value(v, 32), lane_value(v, 48))); }

// N pieces of 16 positions, the first from p0 on and 64 apart, their dependent steps side by side: running maximum and sum, o four columns of every
// fourth position.  s_new: query, key and value of position T - 1 in the LDS, read where they are used (two pieces in flight take 64 registers)
template <int N, bool FIRST>
__device__ __forceinline__ void attend_rows(const KeyRows* kv, int p0, int T, int lane, const float* s_new, float& m, float& lsum, f32x4& o) {
    float sc[2 * N], mn = m;
    {
        const unsigned at = fresh(lds_at(&s_new[(lane & 7) * 8]));
        const f32x4 q0 = lds_read<f32x4>(at), q1 = lds_read<f32x4>(at + 16), n0 = lds_read<f32x4>(at + 256), n1 = lds_read<f32x4>(at + 272);
#pragma unroll
        for (int i = 0; i < 2 * N; ++i) {
            const KeyRows& x = kv[i / 2];
            const int t = p0 + i / 2 * 64 + i % 2 * 8 + (lane >> 3);
            const bool nw = t == T - 1;
            float acc0 = 0.0f, acc1 = 0.0f;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                acc0 = fmaf(q0[d], nw ? n0[d] : x.k[i % 2][0][d], acc0);
                acc1 = fmaf(q1[d], nw ? n1[d] : x.k[i % 2][1][d], acc1);
            }
            const float dot = sum8(acc0 + acc1) * 0.125f;  // 1 / sqrt(64): ops.zig:275
            sc[i] = t < T ? dot : kNone;
        }
    }
    {
        float top = sc[0];
#pragma unroll
        for (int i = 1; i < 2 * N; ++i) top = fmaxf(top, sc[i]);
        mn = fmaxf(mn, over_rows(fmaxf(top, dpp_row_ror<8>(top)), [](float x, float y) { return fmaxf(x, y); }));
    }
    const f32x4 vn = lds_read<f32x4>(fresh(lds_at(&s_new[128 + (lane & 15) * 4])));
    if (!FIRST) {
        const float e0 = __expf(m - mn);
        lsum *= e0;
        o *= e0;
    }
#pragma unroll
    for (int i = 0; i < 2 * N; ++i) {
        const int tb = p0 + i / 2 * 64 + i % 2 * 8;
        const float p = tb + (lane >> 3) < T ? __expf(sc[i] - mn) : 0.0f, other = dpp_row_ror<8>(p);
        lsum += p + other;
        if (N == 2) __builtin_amdgcn_sched_barrier(0);  // (the values, last to arrive, are not waited for earlier: 2 % of long contexts)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int tj = tb + q + (lane >> 4) * 2;
            const float pq = (lane >> 3 & 1) == q ? p : other;
#pragma unroll
            for (int d = 0; d < 4; ++d) o[d] = fmaf(pq, tj == T - 1 ? vn[d] : tj < T ? kv[i / 2].v[i % 2 * 2 + q][d] : 0.0f, o[d]);
        }
    }
    m = mn;
}
// What wave w of four has, for merge_waves
__device__ __forceinline__ void put_share(int w, int lane, float m, float lsum, const f32x4& o, float (*s_o)[64], float* s_m, float* s_l) {
    lsum = over_rows(lsum, [](float x, float y) { return x + y; });
    *reinterpret_cast<f32x4*>(&s_o[w * 4 + (lane >> 4)][(lane & 15) * 4]) = o;
    if (lane == 0) {
        s_m[w] = m;
        s_l[w] = lsum;
    }
}
// by one wave: the four waves' maxima, sums and (a lane a column) values
__device__ __forceinline__ void merge_waves(int lane, const float (*s_o)[64], const float* s_m, const float* s_l, float& m, float& lsum, float& o) {
    const f32x4 m4 = *reinterpret_cast<const f32x4*>(s_m), l4 = *reinterpret_cast<const f32x4*>(s_l);
    m = fmaxf(fmaxf(m4.x, m4.y), fmaxf(m4.z, m4.w));
    o = lsum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float e = __expf(m4[i] - m);
        o = fmaf(e, (s_o[4 * i][lane] + s_o[4 * i + 1][lane]) + (s_o[4 * i + 2][lane] + s_o[4 * i + 3][lane]), o);
        lsum = fmaf(e, l4[i], lsum);
    }
}

// ------------------------------------------------------------------------------------------------ the start
// By one thread of every workgroup: register; the last one commits if the steps in front have run and every XCD has 32, one that has
// waited too long (behind a withdrawn launch: at once) withdraws the launch for all.  1: all workgroups are resident; 2: nothing may be touched.
__device__ inline unsigned join(ResidentCtl* ctl, unsigned xcc, unsigned s0, unsigned start_limit, unsigned* rank) {
    *rank = __hip_atomic_fetch_add(&ctl->reg[xcc], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned before = __hip_atomic_fetch_add(&ctl->total, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (before == (unsigned)(kXcds * kRanks) - 1u) {
        bool ok = ctl->done == s0;
        for (int i = 0; i < kXcds; ++i) ok = ok && __hip_atomic_load(&ctl->reg[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)kRanks;
        unsigned open = 0u;
        __hip_atomic_compare_exchange_strong(&ctl->state, &open, ok ? 1u : 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    for (unsigned n = 0;; ++n) {
        const unsigned st = __hip_atomic_load(&ctl->state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (st != 0u) return st;
        if (n >= start_limit || ctl->done != s0) {  // (final: no other launch is running)
            unsigned open = 0u;
            __hip_atomic_compare_exchange_strong(&ctl->state, &open, 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return open == 0u ? 2u : open;
        }
        __builtin_amdgcn_s_sleep(2);
    }
}

}  // namespace resident
}  // namespace zg
