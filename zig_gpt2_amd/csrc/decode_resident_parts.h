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
