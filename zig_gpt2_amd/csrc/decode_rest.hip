// What is left of a greedy generation whose resident launches were withdrawn (decode_resident.hip: other kernels held compute units for longer
// than a launch waits for all of its workgroups), on the stream behind them, so that the stream's end is the generation's end.
//
// This kernel needs no particular number of workgroups.  Those that have started by the time the first one closes the list share the work:
// every one of them is running, so they may wait for each other; later ones leave at once.  A phase of a Block is one product or the
// attention, spread over all waves of the members, activations in memory, a barrier over the members behind each.  It is no fast path (124M, one
// sequence, an otherwise idle chip: 0.79 ms a token, eight sequences 1.95; the launch chain 0.21 and 0.27) and takes over rarely: the handle then stays with the
// launch chain for some generations.  Behind launches that ran it costs an empty launch a generation.
#include "decode_resident_parts.h"

namespace zg {

namespace {

using namespace resident;
constexpr int kWaves = 8, kGroups = 128;  // (256: barriers cost more than their loads gain, 1.00 : 0.79 ms a token; 64: 0.96)
constexpr unsigned kClosed = 1u << 31;

template <typename WT>
__device__ __forceinline__ void load8(const WT* p, float (&v)[8]) {
    if constexpr (sizeof(WT) == 2) {
        const u32x4 r = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = bf16_lo(r[i]);
            v[2 * i + 1] = bf16_hi(r[i]);
        }
    } else {
        const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = a[i];
            v[4 + i] = b[i];
        }
    }
}
template <typename WT>
__device__ __forceinline__ float element(const void* base, size_t i) {
    if constexpr (sizeof(WT) == 2) return __uint_as_float((uint32_t) reinterpret_cast<const bf16_t*>(base)[i] << 16);
    return reinterpret_cast<const float*>(base)[i];
}

template <typename WT>
__global__ __launch_bounds__(64 * kWaves) void decode_rest_kernel(const RestArgs p) {
    __shared__ float s_m[kWaves], s_l[kWaves], s_o[kWaves][64], s_bv[kWaves][8], s_v[8];
    __shared__ int s_bi[kWaves][8], s_i[8], s_pick[8], s_tok[8];
    __shared__ unsigned s_id, s_n, s_from, s_fail;
    const ResidentArgs& a = p.r;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    ResidentCtl* const ctl = a.ctl;
    if (tid == 0) {
        s_fail = 0u;
        s_n = 0u;
        s_from = __hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (behind a wait that ran out nothing is worth running: the call that drains the stream fails)
        if (s_from < (unsigned)a.s1 && __hip_atomic_load(a.fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == 0u) {
            s_id = __hip_atomic_fetch_add(&ctl->joined, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (s_id == 0u) {
                for (unsigned n = 0; n < p.patience && __hip_atomic_load(&ctl->joined, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < gridDim.x; ++n) __builtin_amdgcn_s_sleep(2);
                s_n = __hip_atomic_fetch_or(&ctl->joined, kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&ctl->members, s_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else if (!(s_id & kClosed)) {  // (the first one is running and closes the list without waiting for anyone)
                do s_n = __hip_atomic_load(&ctl->members, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                while (s_n == 0u);
            }
        }
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane((int)s_n), id = __builtin_amdgcn_readfirstlane((int)s_id);
    if (n == 0) return;
    const int from = __builtin_amdgcn_readfirstlane((int)s_from);
    const int E = p.n_embed, F = 4 * E, M = a.batch, H = a.n_heads, V = a.vocab;
    const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7u;  // HW_REG_XCC_ID
    unsigned barriers = 0u;
    // every member's stores in front of it are seen by every member behind it; false: a wait ran out.  The last one to arrive tells the others, a
    // line for an XCD: all of them polling the word they count in made a barrier 3 times as long
    auto meet = [&]() -> bool {
        __syncthreads();
        if (tid == 0) {
            ++barriers;
            __threadfence();
            if (__hip_atomic_fetch_add(&ctl->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == barriers * (unsigned)n - 1u)
                for (int x = 0; x < kXcds; ++x) __hip_atomic_store(&ctl->passed[x][0], barriers, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (unsigned t = 0; (int)(__hip_atomic_load(&ctl->passed[xcc][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - barriers) < 0; ++t) {
                if (t >= a.spin_limit) {
                    s_fail = 1u;
                    __hip_atomic_store(a.fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            __threadfence();
        }
        __syncthreads();
        return s_fail == 0u;
    };
    auto at_layer = [&](const auto* base, int l) { return reinterpret_cast<decltype(base)>(reinterpret_cast<const char*>(base) + (size_t)l * a.w_stride); };
    float mean[8], rstd[8];
    auto stats = [&]() {
#pragma unroll
        for (int m = 0; m < 8; ++m)
            if (m < M) {
                float sx = 0.0f, sxx = 0.0f;
                for (int e = lane; e < E; e += 64) {
                    const float x = a.x[(size_t)m * E + e];
                    sx += x;
                    sxx = fmaf(x, x, sxx);
                }
                mean[m] = wave_allsum(sx) * (1.0f / (float)E);
                rstd[m] = __builtin_amdgcn_rsqf(wave_allsum(sxx) * (1.0f / (float)E) - mean[m] * mean[m] + 1e-5f);
            }
    };
    // out(row, y) for every row of w [N][K] that is this wave's: lane m < M has the product with sequence m of in [M][K]
    auto rows = [&](const void* w, int N, int K, const float* in, const float* gain, const float* c2, const float* c3, auto out) {
        for (int row = id * kWaves + wave; row < N; row += n * kWaves) {
            float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            for (int k = lane * 8; k < K; k += 512) {
                float wf[8], g[8], z[8];
                load8(reinterpret_cast<const WT*>(w) + (size_t)row * K + k, wf);
                if (gain != nullptr) load8(gain + k, g);
#pragma unroll
                for (int m = 0; m < 8; ++m)
                    if (m < M) {
                        load8(in + (size_t)m * K + k, z);
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[m] = fmaf(wf[i], gain != nullptr ? z[i] * g[i] : z[i], acc[m]);
                    }
            }
            float y = 0.0f;
#pragma unroll
            for (int m = 0; m < 8; ++m)
                if (m < M) {
                    const float S = wave_allsum(acc[m]);
                    const float v = gain != nullptr ? fmaf(rstd[m], fmaf(-mean[m], c2[row], S), c3[row]) : S;
                    y = lane == m ? v : y;
                }
            if (lane < M) out(row, y);
        }
    };
    if (tid < M) s_pick[tid] = from > a.prompt_len[tid] ? a.out_tokens[(size_t)tid * a.out_stride + from - 1] : 0;
    const int np = a.prompt_len[min(tid, M - 1)];
    for (int s = from; s < a.s1; ++s) {
        const int T = s + 1;
        const bool last = T == a.s1;
        __syncthreads();
        if (tid < M) {
            const int* const prompt = a.prompt + (size_t)tid * a.out_stride;
            s_tok[tid] = s < np ? prompt[s] : s == np ? prompt[np - 1] : s_pick[tid];
            if (s < np && id == 0) a.out_tokens[(size_t)tid * a.out_stride + s] = s_tok[tid];
        }
        __syncthreads();
        for (int i = id * 64 * kWaves + tid; i < M * E; i += n * 64 * kWaves)
            a.x[i] = element<WT>(a.wte, (size_t)s_tok[i / E] * E + i % E) + element<WT>(a.wpe, (size_t)s * E + i % E);
        if (!meet()) break;
        for (int l = 0; l < a.n_layer; ++l) {
            float* const kc = reinterpret_cast<float*>(a.k_cache + (size_t)l * a.kv_stride);
            float* const vc = reinterpret_cast<float*>(a.v_cache + (size_t)l * a.kv_stride);
            stats();
            rows(at_layer(reinterpret_cast<const char*>(a.c_attn_w), l), 3 * E, E, a.x, at_layer(a.ln_1_g, l), at_layer(a.c_attn_c2, l), at_layer(a.c_attn_c3, l), [&](int row, float y) {
                const int part = row / E, c = row % E;
                if (part == 0) p.q[(size_t)lane * E + c] = y;
                else (part == 1 ? kc : vc)[((size_t)(lane * H + (c >> 6)) * a.ctx + (T - 1)) * 64 + (c & 63)] = y;
            });
            if (!meet()) break;
            for (int pair = id; pair < M * H; pair += n) {  // (sequence, head): four positions of a wave at a time, a lane has a dimension
                const float q = p.q[(size_t)(pair / H) * E + (pair % H) * 64 + lane];
                const float *const kh = kc + (size_t)pair * a.ctx * 64, *const vh = vc + (size_t)pair * a.ctx * 64;
                float m = kNone, sum = 0.0f, o = 0.0f;
                for (int t0 = wave; t0 < T; t0 += 4 * kWaves) {
                    float k4[4], v4[4], sc[4], mn = m;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int t = min(t0 + j * kWaves, T - 1);
                        k4[j] = kh[(size_t)t * 64 + lane];
                        v4[j] = vh[(size_t)t * 64 + lane];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float dot = wave_allsum(q * k4[j]) * 0.125f;  // 1 / sqrt(64): ops.zig:275
                        sc[j] = t0 + j * kWaves < T ? dot : kNone;
                        mn = fmaxf(mn, sc[j]);
                    }
                    const float e0 = __expf(m - mn);
                    sum *= e0;
                    o *= e0;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const bool there = t0 + j * kWaves < T;
                        const float e = there ? __expf(sc[j] - mn) : 0.0f;
                        sum += e;
                        o = fmaf(e, there ? v4[j] : 0.0f, o);
                    }
                    m = mn;
                }
                s_o[wave][lane] = o;
                if (lane == 0) {
                    s_m[wave] = m;
                    s_l[wave] = sum;
                }
                __syncthreads();
                if (wave == 0) {
                    float mx = kNone, l8 = 0.0f, o8 = 0.0f;
#pragma unroll
                    for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, s_m[w]);
#pragma unroll
                    for (int w = 0; w < kWaves; ++w) {
                        const float e = __expf(s_m[w] - mx);
                        l8 = fmaf(e, s_l[w], l8);
                        o8 = fmaf(e, s_o[w][lane], o8);
                    }
                    p.z[(size_t)(pair / H) * E + (pair % H) * 64 + lane] = o8 / l8;
                }
                __syncthreads();
            }
            if (!meet()) break;
            const float *const b1 = at_layer(a.c_proj_b, l), *const b2 = at_layer(a.mlp_proj_b, l);
            rows(at_layer(reinterpret_cast<const char*>(a.c_proj_w), l), E, E, p.z, nullptr, nullptr, nullptr, [&](int row, float y) { a.x[(size_t)lane * E + row] += y + b1[row]; });
            if (!meet()) break;
            stats();
            rows(at_layer(reinterpret_cast<const char*>(a.c_fc_w), l), F, E, a.x, at_layer(a.ln_2_g, l), at_layer(a.c_fc_c2, l), at_layer(a.c_fc_c3, l),
                 [&](int row, float y) { p.h[(size_t)lane * F + row] = gelu_ref(y); });
            if (!meet()) break;
            rows(at_layer(reinterpret_cast<const char*>(a.mlp_proj_w), l), E, F, p.h, nullptr, nullptr, nullptr, [&](int row, float y) { a.x[(size_t)lane * E + row] += y + b2[row]; });
            if (!meet()) break;
        }
        if (s_fail != 0u) break;
        if (s >= a.n_prompt) {  // ---- ln_f + lm_head + argmax (main.zig:189-194, :337)
            float bv = -3.0e38f;
            int bi = 0x7fffffff;
            stats();
            rows(a.wte, V, E, a.x, a.ln_f_g, a.lm_c2, a.lm_c3, [&](int row, float y) {
                if (y > bv) {  // rows of a wave ascend: the first of equal values stays
                    bv = y;
                    bi = row;
                }
                if (last) a.logits[(size_t)lane * V + row] = y;
            });
            if (lane < 8) {
                s_bv[wave][lane] = bv;
                s_bi[wave][lane] = bi;
            }
            __syncthreads();
            if (tid < M) {
                for (int w = 1; w < kWaves; ++w) better(bv, bi, s_bv[w][tid], s_bi[w][tid]);
                p.best_v[tid * kGroups + id] = bv;
                p.best_i[tid * kGroups + id] = bi;
            }
            if (!meet()) break;
            if (wave < M) {
                float v = -3.0e38f;
                int i = 0x7fffffff;
                for (int g = lane; g < n; g += 64) better(v, i, p.best_v[wave * kGroups + g], p.best_i[wave * kGroups + g]);
                argmax_wave(v, i);
                if (lane == 0) {
                    s_v[wave] = v;
                    s_i[wave] = i;
                    s_pick[wave] = (unsigned)i < (unsigned)V ? i : 0;  // logits that are all NaN: index 0 (embed_step_kernel)
                }
            }
            __syncthreads();
            if (id == 0 && tid < M && s >= np) a.out_tokens[(size_t)tid * a.out_stride + s] = s_pick[tid];
            if (id == 0 && last)  // for the launches that may follow: one partial holds the pick
                for (int g = tid; g < M * a.n_part; g += 64 * kWaves) {
                    const bool first = g % a.n_part == 0;
                    a.part_val[g] = first ? s_v[g / a.n_part] : -3.0e38f;
                    a.part_idx[g] = first ? s_i[g / a.n_part] : 0x7fffffff;
                }
        }
    }
    if (id != 0 || s_fail != 0u) return;
    if (tid < M) a.cur_token[tid] = s_tok[tid];
    if (tid == 0) {
        a.ctrl->seq_len = a.s1;
        a.ctrl->step = a.s1;
        ctl->rest_steps += (unsigned)(a.s1 - from);
        ctl->rest_members = (unsigned)n;
        __hip_atomic_store(&ctl->done, (unsigned)a.s1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace

size_t decode_rest_floats() { return 2 * 8 * (size_t)kGroups; }

int launch_decode_rest(const RestArgs& a, int weight_type, hipStream_t s) {
    ZG_REQUIRE(a.r.batch >= 1 && a.r.batch <= 8 && a.n_embed % 64 == 0 && a.r.s1 <= a.r.ctx, ZG_ERR_ARG, "rest of a generation: bad arguments");
    if (weight_type == WT_BF16) decode_rest_kernel<bf16_t><<<kGroups, 64 * kWaves, 0, s>>>(a);
    else decode_rest_kernel<float><<<kGroups, 64 * kWaves, 0, s>>>(a);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace zg
