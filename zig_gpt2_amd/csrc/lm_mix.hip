// lm_mix.hip — the row-wise and sequence-wise kernels of the layered-model tier: embedding, RMS norms (with the token shift and
// the residual sum fused in), the gated linear recurrence (HGRN2) and the latent attention over a paged cache of latents.
// Everything here is fp32 in both precision modes: norms, gates, the recurrent state, positions, angles, scores and weights.
#include <math.h>
#include <stdlib.h>

#include <algorithm>

#include "lm_latent_parts.h"
#include "lm_quotient.h"

namespace zg {
namespace lm {

namespace {

__device__ __forceinline__ float block_allsum(float v, float* s_red) {
    v = wave_allsum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    float t = 0.0f;
    for (int w = 0; w < nw; ++w) t += s_red[w];
    return t;
}

// 1 / sqrt(mean(v^2) + eps) of one row, the same summation order wherever a row is normed (a row normed again as somebody's
// predecessor gives the bits its own workgroup got).
__device__ __forceinline__ float row_inv_rms(const float* v, int n, float eps, float* s_red) {
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) ss = fmaf(v[i], v[i], ss);
    ss = block_allsum(ss, s_red);
    return 1.0f / sqrtf(ss / (float)n + eps);
}

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }

__global__ __launch_bounds__(256) void embed_kernel(const bf16_t* table, const int* ids, float* x, float* x_copy, float scale, int W, int vocab,
                                                    int* flag, const int* row_pos, const float* pos_freq) {
    const int m = blockIdx.x, id = ids[m];
    const bool ok = id >= 0 && id < vocab;
    if (!ok && threadIdx.x == 0) *flag = 1;
    const bf16_t* row = table + (size_t)(ok ? id : 0) * W;
    const float fpos = row_pos ? (float)row_pos[m] : 0.0f;
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
        float v = ok ? __uint_as_float((uint32_t)row[i] << 16) * scale : 0.0f;
        if (row_pos) {  // entries (2j, 2j + 1) = (sin, cos) of the fp32 product position x frequency j
            const float a = fpos * pos_freq[i >> 1];
            v += (i & 1) ? cosf(a) : sinf(a);
        }
        x[(size_t)m * W + i] = v;
        if (x_copy) x_copy[(size_t)m * W + i] = v;
    }
}

// Rows of up to 256 * kRowRegs floats are held in registers between the statistics and the result: every operand is requested
// in one go at the top of the kernel, so a one-row step (decoding) pays one memory round trip instead of one per pass.
constexpr int kRowRegs = 16;

__global__ __launch_bounds__(256) void norm_shift_kernel(const float* x, const float* w, const float* mu, float eps, float* out, int W,
                                                         const int* row_prev, const int* row_slot, const float* shift_state,
                                                         size_t slot_stride, const int* row_entry_if_last, float* last_out, bf16_t* out16) {
    __shared__ float s_red[8];
    const int m = blockIdx.x;
    const float* xr = x + (size_t)m * W;
    const int entry = row_entry_if_last ? row_entry_if_last[m] : -1;
    const int pm = mu ? row_prev[m] : -1;
    const float* xp = (mu && pm >= 0) ? x + (size_t)pm * W : nullptr;
    const float* hp = (mu && pm < 0) ? shift_state + (size_t)row_slot[m] * slot_stride : nullptr;
    if (W <= 256 * kRowRegs) {
        float xv[kRowRegs], pv[kRowRegs], wv[kRowRegs], mv[kRowRegs];
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            const bool ok = i < W;
            xv[j] = ok ? xr[i] : 0.0f;
            wv[j] = ok ? w[i] : 0.0f;
            mv[j] = (ok && mu) ? mu[i] : 0.0f;
            pv[j] = !ok ? 0.0f : xp ? xp[i] : hp ? hp[i] : 0.0f;
        }
        float ss = 0.0f;  // the same order as row_inv_rms: element i of thread t is t + 256 j, j ascending
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) ss = fmaf(xv[j], xv[j], ss);
        ss = block_allsum(ss, s_red);
        const float r = 1.0f / sqrtf(ss / (float)W + eps);
        float rp = 0.0f;
        if (xp) {
            float sp = 0.0f;
#pragma unroll
            for (int j = 0; j < kRowRegs; ++j) sp = fmaf(pv[j], pv[j], sp);
            sp = block_allsum(sp, s_red);
            rp = 1.0f / sqrtf(sp / (float)W + eps);
        }
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < W) {
                const float g = 1.0f + wv[j];
                const float h = xv[j] * r * g;
                const float before = xp ? pv[j] * rp * g : pv[j];
                put_row(out, out16, (size_t)m * W + i, mu ? h + (before - h) * mv[j] : h);
                if (entry >= 0) last_out[(size_t)entry * W + i] = h;
            }
        }
        return;
    }
    const float r = row_inv_rms(xr, W, eps, s_red);
    if (mu == nullptr) {
        for (int i = threadIdx.x; i < W; i += blockDim.x) {
            const float h = xr[i] * r * (1.0f + w[i]);
            put_row(out, out16, (size_t)m * W + i, h);
            if (entry >= 0) last_out[(size_t)entry * W + i] = h;
        }
        return;
    }
    float rp = 0.0f;
    if (xp) rp = row_inv_rms(xp, W, eps, s_red);
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
        const float g = 1.0f + w[i];
        const float h = xr[i] * r * g;
        const float before = xp ? xp[i] * rp * g : hp[i];
        put_row(out, out16, (size_t)m * W + i, h + (before - h) * mu[i]);
        if (entry >= 0) last_out[(size_t)entry * W + i] = h;
    }
}

__global__ __launch_bounds__(256) void commit_rows_kernel(float* dst, size_t slot_stride, const float* src, size_t src_stride, const int* slots,
                                                          int width, size_t dst_set_stride, size_t src_set_stride) {
    const int e = blockIdx.x, set = blockIdx.y;
    float* d = dst + (size_t)slots[e] * slot_stride + set * dst_set_stride;
    const float* s = src + (size_t)e * src_stride + set * src_set_stride;
    for (int i = threadIdx.x; i < width; i += blockDim.x) d[i] = s[i];
}

__global__ __launch_bounds__(256) void norm_add_kernel(const float* x, float* out, const float* y, const float* w, float eps, int W) {
    __shared__ float s_red[8];
    const int m = blockIdx.x;
    const float* yr = y + (size_t)m * W;
    const float r = row_inv_rms(yr, W, eps, s_red);
    for (int i = threadIdx.x; i < W; i += blockDim.x) out[(size_t)m * W + i] = x[(size_t)m * W + i] + yr[i] * r * (1.0f + w[i]);
}

__global__ __launch_bounds__(256) void copy_floats_kernel(const float* x, float* out, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = x[i];
}

// x += norm(y) * (1 + wb), then h = norm(x) * (1 + wn): the norm behind the mixer, the residual sum and the norm in front of the
// feed-forward in one pass over the row
__global__ __launch_bounds__(256) void norm_add_norm_kernel(float* x, const float* y, const float* wb, const float* wn, float eps, float* h, int W,
                                                            bf16_t* h16) {
    __shared__ float s_red[8];
    const int m = blockIdx.x;
    const float* yr = y + (size_t)m * W;
    float* xr = x + (size_t)m * W;
    if (W <= 256 * kRowRegs) {
        float yv[kRowRegs], xv[kRowRegs], bv[kRowRegs], nv[kRowRegs];
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            const bool ok = i < W;
            yv[j] = ok ? yr[i] : 0.0f;
            xv[j] = ok ? xr[i] : 0.0f;
            bv[j] = ok ? wb[i] : 0.0f;
            nv[j] = ok ? wn[i] : 0.0f;
        }
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) ss = fmaf(yv[j], yv[j], ss);
        ss = block_allsum(ss, s_red);
        const float r = 1.0f / sqrtf(ss / (float)W + eps);
        float s2 = 0.0f;
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            xv[j] += yv[j] * r * (1.0f + bv[j]);  // (rows beyond W: 0 + 0)
            s2 = fmaf(xv[j], xv[j], s2);
        }
        s2 = block_allsum(s2, s_red);
        const float r2 = 1.0f / sqrtf(s2 / (float)W + eps);
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < W) {
                xr[i] = xv[j];
                put_row(h, h16, (size_t)m * W + i, xv[j] * r2 * (1.0f + nv[j]));
            }
        }
        return;
    }
    const float r = row_inv_rms(yr, W, eps, s_red);
    for (int i = threadIdx.x; i < W; i += blockDim.x) xr[i] += yr[i] * r * (1.0f + wb[i]);  // each thread rereads only what it wrote
    float ss = 0.0f;
    for (int i = threadIdx.x; i < W; i += blockDim.x) ss = fmaf(xr[i], xr[i], ss);
    ss = block_allsum(ss, s_red);
    const float r2 = 1.0f / sqrtf(ss / (float)W + eps);
    for (int i = threadIdx.x; i < W; i += blockDim.x) put_row(h, h16, (size_t)m * W + i, xr[i] * r2 * (1.0f + wn[i]));
}

// Steps of one row per entry (decoding): the sum behind a pass's last sublayer and the NEXT pass's norm + token shift in one
// launch, the row held in registers:
//   y = a sublayer's output row, or sum_k weight[k] * yexp[m top + k] (the chosen experts, in choice order)
//   x += norm(y) (1 + wb);   h = norm(x) (1 + wn);   out = h + (state[slot] - h) mu;   last_out[entry] = h
// (the predecessor of a decoded token is always the row its slot keeps)
__global__ __launch_bounds__(256) void sum_norm_shift_kernel(float* x, const float* y, const float* yexp, const float* weight, int top, const float* wb,
                                                             const float* wn, const float* mu, float eps, float* out, int W, const int* row_slot,
                                                             const float* shift_state, size_t slot_stride, const int* row_entry_if_last,
                                                             float* last_out) {
    __shared__ float s_red[8];
    const int m = blockIdx.x;
    float* xr = x + (size_t)m * W;
    const float* hp = shift_state + (size_t)row_slot[m] * slot_stride;
    const int entry = row_entry_if_last[m];
    float yv[kRowRegs], xv[kRowRegs], bv[kRowRegs], nv[kRowRegs], mv[kRowRegs], pv[kRowRegs];
#pragma unroll
    for (int j = 0; j < kRowRegs; ++j) {
        const int i = threadIdx.x + 256 * j;
        const bool ok = i < W;
        float v = 0.0f;
        if (ok) {
            if (yexp) {
                for (int k = 0; k < top; ++k) v = fmaf(weight[m * top + k], yexp[(size_t)(m * top + k) * W + i], v);
            } else {
                v = y[(size_t)m * W + i];
            }
        }
        yv[j] = v;
        xv[j] = ok ? xr[i] : 0.0f;
        bv[j] = ok ? wb[i] : 0.0f;
        nv[j] = ok ? wn[i] : 0.0f;
        mv[j] = ok ? mu[i] : 0.0f;
        pv[j] = ok ? hp[i] : 0.0f;
    }
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < kRowRegs; ++j) ss = fmaf(yv[j], yv[j], ss);
    ss = block_allsum(ss, s_red);
    const float r = 1.0f / sqrtf(ss / (float)W + eps);
    float s2 = 0.0f;
#pragma unroll
    for (int j = 0; j < kRowRegs; ++j) {
        xv[j] += yv[j] * r * (1.0f + bv[j]);
        s2 = fmaf(xv[j], xv[j], s2);
    }
    s2 = block_allsum(s2, s_red);
    const float r2 = 1.0f / sqrtf(s2 / (float)W + eps);
#pragma unroll
    for (int j = 0; j < kRowRegs; ++j) {
        const int i = threadIdx.x + 256 * j;
        if (i < W) {
            const float h = xv[j] * r2 * (1.0f + nv[j]);
            xr[i] = xv[j];
            out[(size_t)m * W + i] = h + (pv[j] - h) * mv[j];
            if (entry >= 0) last_out[(size_t)entry * W + i] = h;
        }
    }
}

__global__ __launch_bounds__(256) void norm_gather_kernel(const float* x, const int* rows, const float* w, float eps, float* out, int W, float one) {
    __shared__ float s_red[8];
    const int j = blockIdx.x;
    const float* xr = x + (size_t)rows[j] * W;
    const float r = row_inv_rms(xr, W, eps, s_red);
    for (int i = threadIdx.x; i < W; i += blockDim.x) out[(size_t)j * W + i] = xr[i] * r * (one + w[i]);
}

// Side-by-side sublayers: the residual sum the layer before left open, then the two norms of the same row from one statistic.
// Rows of up to 256 * kRowRegs floats stay in registers between the statistic and the results.
__device__ __forceinline__ float open_sums_at(const OpenSums& add, size_t m, int i, int W, float v) {
    if (add.sa) {  // a factor per channel on either sublayer's result
        float a = add.a ? add.a[m * W + i] : 0.0f;
        if (add.bias) a = fmaf(add.w, add.bias[i], a);
        v = fmaf(add.sa[i], a, v);
    } else if (add.a) {
        v += add.a[m * W + i];
    }
    const float sb = add.sb ? add.sb[i] : 1.0f;
    if (add.exp) {  // in choice order: the sum does not depend on the batch
        float e = 0.0f;
        for (int k = 0; k < add.top; ++k) {
            const size_t as = m * add.top + k;
            const float y = add.pick && add.pick[as] >= add.n_exp ? add.ident[m * W + i] : add.exp[as * W + i];
            e = add.exp_w ? fmaf(add.exp_w[as], y, e) : e + y;
        }
        if (add.b) e += add.b[m * W + i];
        v = fmaf(sb, e, v);
    } else if (add.b) {
        v = fmaf(sb, add.b[m * W + i], v);
    }
    if (add.bias && !add.sa) v = fmaf(add.w, add.bias[i], v);
    return v;
}

__global__ __launch_bounds__(256) void norm_two_kernel(float* x, const OpenSums add, const float* wa, const float* wb, float eps, float* ha, float* hb,
                                                       int W, bf16_t* ha16, bf16_t* hb16) {
    __shared__ float s_red[8];
    const int m = blockIdx.x;
    float* xr = x + (size_t)m * W;
    const bool adds = add.any();
    auto value = [&](int i) { return adds ? open_sums_at(add, (size_t)m, i, W, xr[i]) : xr[i]; };
    if (W <= 256 * kRowRegs) {
        float v[kRowRegs];
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            v[j] = i < W ? value(i) : 0.0f;
            ss = fmaf(v[j], v[j], ss);
        }
        ss = block_allsum(ss, s_red);
        const float r = 1.0f / sqrtf(ss / (float)W + eps);
#pragma unroll
        for (int j = 0; j < kRowRegs; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < W) {
                if (adds) xr[i] = v[j];
                put_row(ha, ha16, (size_t)m * W + i, v[j] * r * wa[i]);
                if (wb) put_row(hb, hb16, (size_t)m * W + i, v[j] * r * wb[i]);
            }
        }
        return;
    }
    float ss = 0.0f;
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
        const float v = value(i);
        if (adds) xr[i] = v;  // (each thread reads back only what it wrote itself)
        ss = fmaf(v, v, ss);
    }
    ss = block_allsum(ss, s_red);
    const float r = 1.0f / sqrtf(ss / (float)W + eps);
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
        const float v = xr[i];
        put_row(ha, ha16, (size_t)m * W + i, v * r * wa[i]);
        if (wb) put_row(hb, hb16, (size_t)m * W + i, v * r * wb[i]);
    }
}

__global__ __launch_bounds__(256) void add_two_kernel(float* x, const OpenSums add, size_t n, int W) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] = open_sums_at(add, i / W, (int)(i % W), W, x[i]);
}

// one wave per (row, head) vector
__global__ __launch_bounds__(256) void norm_plain_kernel(float* v, int ld, int rows_per_m, int width, int n_vec, const float* w, float eps, bf16_t* out16) {
    const int vec = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (vec >= n_vec) return;
    const size_t at = (size_t)(vec / rows_per_m) * ld + (size_t)(vec % rows_per_m) * width;
    float* p = v + at;
    float ss = 0.0f;
    for (int i = lane; i < width; i += 64) ss = fmaf(p[i], p[i], ss);
    ss = wave_allsum(ss);
    const float r = 1.0f / sqrtf(ss / (float)width + eps);
    for (int i = lane; i < width; i += 64) put_row(out16 ? nullptr : v, out16, at + i, p[i] * r * w[i]);
}

// ------------------------------------------------------------------------------------------------ norms without statistics
// n(v) = tanh(alpha v) * w + b, nw = [w (W) | b (W) | alpha]: elementwise, so a thread takes four neighbours of a row (rows whose
// width is no multiple of four: one) and every sum around the norm rides in the same pass.
__device__ __forceinline__ float tanh_norm_f(const float* nw, int W, int i, float alpha, float v) { return fmaf(tanhf(alpha * v), nw[i], nw[W + i]); }

template <int VW>
__global__ __launch_bounds__(256) void tanh_norm_kernel(float* x, const float* pre, const float* nw, const int* rows, float* out, size_t n, int W) {
    const size_t idx = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VW;
    if (idx >= n) return;
    const size_t j = idx / W;
    const int i = (int)(idx % W);
    const size_t src = (rows ? (size_t)rows[j] : j) * W + i;
    const float ap = pre ? pre[2 * W] : 0.0f, an = nw ? nw[2 * W] : 0.0f;
    float v[VW];
    if (VW == 4) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(x + src);
        v[0] = t.x; v[VW > 1 ? 1 : 0] = t.y; v[VW > 2 ? 2 : 0] = t.z; v[VW > 3 ? 3 : 0] = t.w;
    } else {
        v[0] = x[src];
    }
    if (pre) {
#pragma unroll
        for (int u = 0; u < VW; ++u) v[u] = tanh_norm_f(pre, W, i + u, ap, v[u]);
        if (VW == 4) *reinterpret_cast<f32x4*>(x + src) = f32x4{v[0], v[VW > 1 ? 1 : 0], v[VW > 2 ? 2 : 0], v[VW > 3 ? 3 : 0]};
        else x[src] = v[0];
    }
    if (!nw) return;
#pragma unroll
    for (int u = 0; u < VW; ++u) v[u] = tanh_norm_f(nw, W, i + u, an, v[u]);
    if (VW == 4) *reinterpret_cast<f32x4*>(out + idx) = f32x4{v[0], v[VW > 1 ? 1 : 0], v[VW > 2 ? 2 : 0], v[VW > 3 ? 3 : 0]};
    else out[idx] = v[0];
}

template <int VW>
__global__ __launch_bounds__(256) void tanh_sum_norm_kernel(float* x, const SumParts y, const float* nb, float mult, const float* nn, float* h, size_t n,
                                                            int W) {
    const size_t idx = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VW;
    if (idx >= n) return;
    const size_t m = idx / W;
    const int i = (int)(idx % W);
    auto load = [&](const float* p, float* v) {
        if (VW == 4) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(p);
            v[0] = t.x; v[VW > 1 ? 1 : 0] = t.y; v[VW > 2 ? 2 : 0] = t.z; v[VW > 3 ? 3 : 0] = t.w;
        } else {
            v[0] = p[0];
        }
    };
    float a[VW], t[VW], xv[VW];
#pragma unroll
    for (int u = 0; u < VW; ++u) a[u] = 0.0f;
    load(x + idx, xv);
    if (y.a) load(y.a + idx, a);
    for (int k = 0; k < y.top; ++k) {  // in choice order: the sum does not depend on the batch
        const size_t as = m * y.top + k;
        const float wk = y.exp_w ? y.exp_w[as] : 1.0f;
        load(y.exp + (size_t)(y.inv ? y.inv[as] : as) * W + i, t);
#pragma unroll
        for (int u = 0; u < VW; ++u) a[u] = fmaf(wk, t[u], a[u]);
    }
    if (y.b) {
        load(y.b + idx, t);
#pragma unroll
        for (int u = 0; u < VW; ++u) a[u] += t[u];
    }
    const float ab = nb[2 * W], an = nn ? nn[2 * W] : 0.0f;
#pragma unroll
    for (int u = 0; u < VW; ++u) xv[u] = fmaf(mult, tanh_norm_f(nb, W, i + u, ab, a[u]), xv[u]);
    if (VW == 4) *reinterpret_cast<f32x4*>(x + idx) = f32x4{xv[0], xv[VW > 1 ? 1 : 0], xv[VW > 2 ? 2 : 0], xv[VW > 3 ? 3 : 0]};
    else x[idx] = xv[0];
    if (!nn) return;
#pragma unroll
    for (int u = 0; u < VW; ++u) t[u] = tanh_norm_f(nn, W, i + u, an, xv[u]);
    if (VW == 4) *reinterpret_cast<f32x4*>(h + idx) = f32x4{t[0], t[VW > 1 ? 1 : 0], t[VW > 2 ? 2 : 0], t[VW > 3 ? 3 : 0]};
    else h[idx] = t[0];
}

// ------------------------------------------------------------------------------------------------ HGRN2
// A column j of a head's state S[D][V] is held by G consecutive lanes, 16 rows each (D <= 16 G).  The token loop is serial; the
// gates and values of the next SB tokens are staged in the LDS (rows beyond D padded with q = 0, f = 1: they stay zero).
//
// Long entries are cut into chunks of kScanChunk tokens that run side by side (the recurrence is linear in S):
//   phase A   every chunk from a zero state: its end state B_c and the product A_c of its gates per row
//   phase B   S_start(c + 1) = A_c * S_start(c) + B_c down the chunks of an entry (elementwise; S_start overwrites B in place)
//   phase C   every chunk again from its true start state, now writing the outputs
// Short steps (decoding, small portions) run the same kernel once per entry, from the slot's state and back into it.
constexpr int kScanRows = 16;
constexpr int kScanChunk = 64;
enum { SCAN_DIRECT = 0, SCAN_A = 1, SCAN_C = 2 };

// which (entry, chunk) a workgroup of the chunked phases works on; false: none
__device__ __forceinline__ bool scan_find_chunk(int id, const int* ent_len, int n_entries, int& e, int& c) {
    for (e = 0; e < n_entries; ++e) {
        const int nc = (ent_len[e] + kScanChunk - 1) / kScanChunk;
        if (id < nc) {
            c = id;
            return true;
        }
        id -= nc;
    }
    return false;
}

// KIND SCAN_LIN: linear attention with a fixed decay per head on the same layout — the staged "gate" array holds silu(k), the weight of
// the token's value in the state's row, and every row decays by decay[h]:  S <- decay S + k v^T  (q, k, v through silu).
// KIND SCAN_GLA: gated linear attention — q (times a factor), k and v unchanged, and one decay per key channel,
// f = sigmoid(z + bias)^(1 / tau) = exp(log sigmoid(z + bias) / tau) in fp32, staged beside k:  S <- diag(f) S + k v^T.
enum { SCAN_HGRN2 = 0, SCAN_LIN = 1, SCAN_GLA = 2 };
__device__ __forceinline__ float log_sigmoid_f(float z) { return fminf(z, 0.0f) - log1pf(expf(-fabsf(z))); }

template <int G, int KIND>
__global__ __launch_bounds__(256) void hgrn2_scan_kernel(const float* proj, int ld, float* out, int ldo, float* state, size_t slot_stride,
                                                         const int* ent_start, const int* ent_len, const int* ent_slot, int n_entries, int H, int D,
                                                         int V, int mode, int SB, float* wsB, float* wsA, const float* bias, const float* low,
                                                         const float* decay, const GlaGate gla) {
    constexpr bool LIN = KIND == SCAN_LIN, GLA = KIND == SCAN_GLA;
    extern __shared__ __attribute__((aligned(16))) float s_scan[];
    constexpr int Dp = G * kScanRows;
    const int cols = blockDim.x / G;
    float* sq = s_scan;             // [SB][Dp]
    float* sf = sq + SB * Dp;       // [SB][Dp]
    float* sv = sf + SB * Dp;       // [SB][cols]
    float* sk = sv + SB * cols;     // [SB][Dp] (SCAN_GLA: the keys; the gate array holds the decays)
    const int h = blockIdx.y;
    const int jl = threadIdx.x / G, g = threadIdx.x % G, j0 = blockIdx.z * cols, j = j0 + jl;
    const bool col_ok = j < V;
    const int HD = H * D;
    int e, c = 0, t_lo, t_hi;
    if (mode == SCAN_DIRECT) {
        e = blockIdx.x;
        t_lo = 0;
        t_hi = ent_len[e];
    } else {
        if (!scan_find_chunk(blockIdx.x, ent_len, n_entries, e, c)) return;
        t_lo = c * kScanChunk;
        t_hi = min(ent_len[e], t_lo + kScanChunk);
    }
    const int m0 = ent_start[e];
    const size_t head_floats = (size_t)D * V;
    const float dec = LIN ? decay[h] : 0.0f;
    float* S_slot = state + (size_t)ent_slot[e] * slot_stride + (size_t)h * head_floats;
    float* S_ws = wsB ? wsB + ((size_t)blockIdx.x * H + h) * head_floats : nullptr;
    const float* S_in = mode == SCAN_DIRECT ? S_slot : mode == SCAN_C ? S_ws : nullptr;
    float S[kScanRows], A[kScanRows];
#pragma unroll
    for (int r = 0; r < kScanRows; ++r) {
        const int i = g * kScanRows + r;
        S[r] = (S_in && col_ok && i < D) ? S_in[(size_t)i * V + j] : 0.0f;
        A[r] = 1.0f;
    }
    for (int tb = t_lo; tb < t_hi; tb += SB) {
        const int nb = min(SB, t_hi - tb);
        __syncthreads();  // the previous block has been consumed
        for (int idx = threadIdx.x; idx < nb * Dp; idx += blockDim.x) {
            const int tt = idx / Dp, i = idx % Dp;
            const float* row = proj + (size_t)(m0 + tb + tt) * ld;
            // the gates are activated on their way into the LDS: q = silu(.), f = low + (1 - low) sigmoid(. + bias)
            float qv = 0.0f, fv = LIN ? 0.0f : 1.0f, kv = 0.0f;
            if (i < D) {
                if (GLA) {
                    qv = row[h * D + i] * gla.q_scale;
                    kv = row[HD + h * D + i];
                    fv = expf(log_sigmoid_f(gla.z[(size_t)(m0 + tb + tt) * gla.ldz + h * D + i] + gla.z_bias[h * D + i]) * gla.inv_tau);
                } else {
                    qv = silu_f(row[h * D + i]);
                    if (LIN) {
                        fv = silu_f(row[HD + h * D + i]);
                    } else {
                        const float l = low[h * D + i];
                        fv = l + (1.0f - l) * sigmoid_f(row[HD + h * D + i] + bias[h * D + i]);
                    }
                }
            }
            sq[idx] = qv;
            sf[idx] = fv;
            if (GLA) sk[idx] = kv;
        }
        for (int idx = threadIdx.x; idx < nb * cols; idx += blockDim.x) {
            const int tt = idx / cols, jj = idx % cols;
            const float vin = j0 + jj < V ? proj[(size_t)(m0 + tb + tt) * ld + 2 * HD + h * V + j0 + jj] : 0.0f;
            sv[idx] = LIN ? silu_f(vin) : vin;
        }
        __syncthreads();
        for (int tt = 0; tt < nb; ++tt) {
            const f32x4* q4 = reinterpret_cast<const f32x4*>(sq + tt * Dp + g * kScanRows);
            const f32x4* f4 = reinterpret_cast<const f32x4*>(sf + tt * Dp + g * kScanRows);
            const f32x4* k4 = reinterpret_cast<const f32x4*>(sk + tt * Dp + g * kScanRows);
            const float v = sv[tt * cols + jl];
            float o = 0.0f;
#pragma unroll
            for (int r4 = 0; r4 < kScanRows / 4; ++r4) {
                const f32x4 qq = q4[r4], ff = f4[r4];
                const f32x4 kk = GLA ? k4[r4] : ff;
                const float qv[4] = {qq.x, qq.y, qq.z, qq.w}, fv[4] = {ff.x, ff.y, ff.z, ff.w}, kv[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = r4 * 4 + u;
                    S[r] = GLA ? fmaf(fv[u], S[r], kv[u] * v) : LIN ? fmaf(dec, S[r], fv[u] * v) : fmaf(fv[u], S[r], (1.0f - fv[u]) * v);
                    o = fmaf(S[r], qv[u], o);
                    if (mode == SCAN_A) A[r] *= LIN ? dec : fv[u];
                }
            }
            if (mode != SCAN_A) {
#pragma unroll
                for (int off = 1; off < G; off <<= 1) o += __shfl_xor(o, off, 64);
                if (g == 0 && col_ok) out[(size_t)(m0 + tb + tt) * ldo + h * V + j] = o;
            }
        }
    }
    float* S_out = mode == SCAN_DIRECT ? S_slot : mode == SCAN_A ? S_ws : nullptr;
    if (S_out) {
#pragma unroll
        for (int r = 0; r < kScanRows; ++r) {
            const int i = g * kScanRows + r;
            if (col_ok && i < D) S_out[(size_t)i * V + j] = S[r];
        }
    }
    if (mode == SCAN_A && blockIdx.z == 0 && jl == 0) {
#pragma unroll
        for (int r = 0; r < kScanRows; ++r) {
            const int i = g * kScanRows + r;
            if (i < D) wsA[((size_t)blockIdx.x * H + h) * D + i] = A[r];
        }
    }
}

// phase B: a thread per VEC state elements in a row walks the chunks of its entry.  Bound by the memory: every chunk's state is read and written.
// 8 entries of 16 chunks, 8 heads of 128 x 128: 142 MB in 27.4 us with two elements a thread against 29.2 with one; 24 heads of 128 x 64, 60 chunks of
// 8 entries 20.1 against 22.3.
template <int VEC>
__global__ __launch_bounds__(256) void hgrn2_carry_kernel(float* state, size_t slot_stride, const int* ent_len, const int* ent_slot, int n_entries, int H,
                                                          int D, int V, float* wsB, const float* wsA, int a_rows, int chunk) {
    typedef __attribute__((ext_vector_type(VEC))) float vec;
    const int e = blockIdx.y;
    const size_t n = (size_t)H * D * V, idx = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    if (idx >= n) return;
    int first = 0;
    for (int k = 0; k < e; ++k) first += (ent_len[k] + chunk - 1) / chunk;
    const int nc = (ent_len[e] + chunk - 1) / chunk;
    const size_t ai = idx / ((size_t)V * (D / a_rows)), na = (size_t)H * a_rows;  // the decay of the element's (head, row), or of its head
    vec* slot = reinterpret_cast<vec*>(state + (size_t)ent_slot[e] * slot_stride + idx);
    vec S = *slot;
    for (int c0 = 0; c0 < nc; c0 += 8) {  // eight chunks' operands requested together: the chain itself is eight multiply-adds
        vec Bv[8];
        float Av[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = min(c0 + u, nc - 1);
            Bv[u] = *reinterpret_cast<const vec*>(wsB + (size_t)(first + c) * n + idx);
            Av[u] = wsA[(size_t)(first + c) * na + ai];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c0 + u < nc) {
                *reinterpret_cast<vec*>(wsB + (size_t)(first + c0 + u) * n + idx) = S;  // the chunk's start state for phase C
#pragma unroll
                for (int i = 0; i < VEC; ++i) S[i] = fmaf(Av[u], S[i], Bv[u][i]);
            }
    }
    if (nc > 0) *slot = S;
}

// ------------------------------------------------------------------------------------------------ linear attention, chunks on the matrix cores
// With ONE decay per head the recurrence S <- lambda S + k v^T, o = S^T q of a chunk of n <= 32 tokens is three matrix products
// (true fp32, v_mfma_f32_32x32x2_f32; q, k, v through silu on load):
//   state   B = sum_j lambda^(n-1-j) k_j v_j^T                       the chunk's end state from zero          (phase A, per chunk)
//   carry   S_start(c + 1) = lambda^n S_start(c) + B_c               down the chunks of an entry              (hgrn2_carry_kernel)
//   output  o_i = sum_(j<=i) lambda^(i-j) (q_i . k_j) v_j + lambda^(i+1) S_start^T q_i                        (phase C, per chunk)
// A workgroup takes a (chunk, head); lane (r, half) of a wave holds channels half * Dh .. of row r (the order inside a dot product
// is free), tokens half * 16 .. where the tokens are the product's inner dimension.
constexpr int kLinChunk = 32;
typedef __attribute__((ext_vector_type(16))) float f32x16_lin;

__device__ __forceinline__ float decay_pow(float lam, float l2, int n) { return n <= 0 ? 1.0f : (lam <= 0.0f ? 0.0f : exp2f((float)n * l2)); }

__device__ __forceinline__ bool lin_find_chunk(int id, const int* ent_len, int n_entries, int& e, int& c) {
    for (e = 0; e < n_entries; ++e) {
        const int nc = (ent_len[e] + kLinChunk - 1) / kLinChunk;
        if (id < nc) {
            c = id;
            return true;
        }
        id -= nc;
    }
    return false;
}

__global__ __launch_bounds__(256) void linear_chunk_state_kernel(const float* __restrict__ proj, int ld, const int* ent_start, const int* ent_len,
                                                                 int n_entries, int H, int D, int V, const float* decay, float* __restrict__ wsB,
                                                                 float* __restrict__ wsA) {
    int e, c;
    if (!lin_find_chunk(blockIdx.x, ent_len, n_entries, e, c)) return;
    const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, kh = lane >> 5;
    const int n = min(kLinChunk, ent_len[e] - c * kLinChunk), m0 = ent_start[e] + c * kLinChunk, HD = H * D;
    const float lam = decay[h], l2 = lam > 0.0f ? log2f(lam) : 0.0f;
    const float* kbase = proj + (size_t)m0 * ld + HD + (size_t)h * D;
    const float* vbase = proj + (size_t)m0 * ld + 2 * HD + (size_t)h * V;
    float* B = wsB + ((size_t)blockIdx.x * H + h) * D * V;
    const int tilesD = (D + 31) / 32, tilesV = (V + 31) / 32;
    for (int tile = blockIdx.z * 4 + wave; tile < tilesD * tilesV; tile += 4 * gridDim.z) {
        const int d0 = (tile / tilesV) * 32, v0 = (tile % tilesV) * 32;
        float a[16], b[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {  // token j is the inner dimension: weight lambda^(n - 1 - j) on the key
            const int j = kh * 16 + t;
            a[t] = (j < n && d0 + r < D) ? kbase[(size_t)j * ld + d0 + r] : 0.0f;
            b[t] = (j < n && v0 + r < V) ? vbase[(size_t)j * ld + v0 + r] : 0.0f;
        }
        f32x16_lin acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < 16; ++t)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(silu_f(a[t]) * decay_pow(lam, l2, n - 1 - (kh * 16 + t)), silu_f(b[t]), acc, 0, 0, 0);
        // accumulator element i: row 8 (i / 4) + 4 half + i % 4, column r
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int d = d0 + 8 * (i >> 2) + 4 * kh + (i & 3);
            if (d < D && v0 + r < V) B[(size_t)d * V + v0 + r] = acc[i];
        }
    }
    if (blockIdx.z == 0)
        for (int i = threadIdx.x; i < D; i += blockDim.x) wsA[((size_t)blockIdx.x * H + h) * D + i] = decay_pow(lam, l2, n);
}

template <int DH>
__global__ __launch_bounds__(256) void linear_chunk_out_kernel(const float* __restrict__ proj, int ld, float* __restrict__ out, int ldo,
                                                               const int* ent_start, const int* ent_len, int n_entries, int H, int D, int V,
                                                               const float* decay, const float* __restrict__ wsB) {
    __shared__ float s_p[4][32][33];
    int e, c;
    if (!lin_find_chunk(blockIdx.x, ent_len, n_entries, e, c)) return;
    const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, kh = lane >> 5;
    const int n = min(kLinChunk, ent_len[e] - c * kLinChunk), m0 = ent_start[e] + c * kLinChunk, HD = H * D, Dh = (D + 1) / 2;
    const float lam = decay[h], l2 = lam > 0.0f ? log2f(lam) : 0.0f;
    const float* S = wsB + ((size_t)blockIdx.x * H + h) * D * V;  // the chunk's start state (the carry left it here)
    const float* qrow = proj + (size_t)(m0 + min(r, n - 1)) * ld + (size_t)h * D + kh * Dh;
    const float* krow = qrow + HD;
    const float* vbase = proj + (size_t)m0 * ld + 2 * HD + (size_t)h * V;
    float qreg[DH], kreg[DH];
    // 16-byte loads where a lane's run of channels starts on a 16-byte boundary and is a multiple of four long
    const bool vec = D % 8 == 0 && ld % 4 == 0 && (reinterpret_cast<uintptr_t>(proj) & 15) == 0;
    if (vec) {
#pragma unroll
        for (int t = 0; t < DH; t += 4) {
            const bool ok = r < n && t < Dh;
            const f32x4 a = ok ? *reinterpret_cast<const f32x4*>(qrow + t) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            const f32x4 b = ok ? *reinterpret_cast<const f32x4*>(krow + t) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            qreg[t] = a.x; qreg[t + 1] = a.y; qreg[t + 2] = a.z; qreg[t + 3] = a.w;
            kreg[t] = b.x; kreg[t + 1] = b.y; kreg[t + 2] = b.z; kreg[t + 3] = b.w;
        }
    } else {
#pragma unroll
        for (int t = 0; t < DH; ++t) {
            const bool ok = r < n && t < Dh && kh * Dh + t < D;
            qreg[t] = ok ? qrow[t] : 0.0f;
            kreg[t] = ok ? krow[t] : 0.0f;
        }
    }
#pragma unroll
    for (int t = 0; t < DH; ++t) {
        qreg[t] = silu_f(qreg[t]);
        kreg[t] = silu_f(kreg[t]);
    }
    f32x16_lin acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < DH; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(qreg[t], kreg[t], acc, 0, 0, 0);
    // element i: query 8 (i / 4) + 4 half + i % 4, key r: the decay of their distance, nothing for keys behind the query
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int qi = 8 * (i >> 2) + 4 * kh + (i & 3);
        s_p[wave][qi][r] = (r <= qi && qi < n) ? acc[i] * decay_pow(lam, l2, qi - r) : 0.0f;
    }
    __syncthreads();
    const float carry = decay_pow(lam, l2, r + 1);  // what the start state has decayed to when token r reads it
#pragma unroll
    for (int t = 0; t < DH; ++t) qreg[t] *= carry;
    const int tilesV = (V + 31) / 32;
    for (int vt = wave; vt < tilesV; vt += 4) {
        const int v0 = vt * 32;
        const bool col_ok = v0 + r < V;
        float vv[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const int j = kh * 16 + t;
            vv[t] = (j < n && col_ok) ? vbase[(size_t)j * ld + v0 + r] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < 16; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s_p[wave][r][kh * 16 + t], silu_f(vv[t]), acc, 0, 0, 0);
#pragma unroll
        for (int t0 = 0; t0 < DH; t0 += 16) {  // the start state's share, 16 state rows requested at a time
            float sv[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int t = t0 + u, ch = kh * Dh + t;
                sv[u] = (t < DH && t < Dh && ch < D && col_ok) ? S[(size_t)ch * V + v0 + r] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 16; ++u)
                if (t0 + u < DH) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(qreg[min(t0 + u, DH - 1)], sv[u], acc, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int qi = 8 * (i >> 2) + 4 * kh + (i & 3);
            if (qi < n && col_ok) out[(size_t)(m0 + qi) * ldo + (size_t)h * V + v0 + r] = acc[i];
        }
    }
}

// ------------------------------------------------------------------------------------------------ latent attention
__global__ __launch_bounds__(256) void latent_prep_kernel(const float* proj, int ld, int q_rank, int KR, int R, const float* wq, const float* wkv,
                                                          float eps, Rotary rot, const int* row_pos, const int* row_slot, const int* page_table,
                                                          int max_pages, int page_tokens, float* cq, float* cache, bf16_t* cq16) {
    __shared__ float s_red[8];
    const int m = blockIdx.x, pos = row_pos[m];
    const float* row = proj + (size_t)m * ld;
    float* crow = cache + cache_row(page_table, max_pages, page_tokens, row_slot[m], pos) * (size_t)(KR + R);
    const float* kr = row + q_rank + KR;
    if (q_rank + KR <= 1024) {  // both parts in registers, requested in one go with their weights
        const int n = q_rank + KR;
        float v[4], w[4], sq = 0.0f, sc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = min((int)threadIdx.x + 256 * j, n - 1);
            v[j] = row[i];
            w[j] = i < q_rank ? wq[i] : wkv[i - q_rank];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < q_rank) sq = fmaf(v[j], v[j], sq);
            else if (i < n) sc = fmaf(v[j], v[j], sc);
        }
        sq = wave_allsum(sq);
        sc = wave_allsum(sc);
        if ((threadIdx.x & 63) == 0) {
            s_red[threadIdx.x >> 6] = sq;
            s_red[4 + (threadIdx.x >> 6)] = sc;
        }
        __syncthreads();
        const float rq = 1.0f / sqrtf(((s_red[0] + s_red[1]) + (s_red[2] + s_red[3])) / (float)q_rank + eps);
        const float rc = 1.0f / sqrtf(((s_red[4] + s_red[5]) + (s_red[6] + s_red[7])) / (float)KR + eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < q_rank) put_row(cq16 ? nullptr : cq, cq16, (size_t)m * q_rank + i, v[j] * rq * w[j]);
            else if (i < n) crow[i - q_rank] = v[j] * rc * w[j];
        }
    } else {
        const float rq = row_inv_rms(row, q_rank, eps, s_red);
        const float rc = row_inv_rms(row + q_rank, KR, eps, s_red);
        for (int i = threadIdx.x; i < q_rank; i += blockDim.x) put_row(cq16 ? nullptr : cq, cq16, (size_t)m * q_rank + i, row[i] * rq * wq[i]);
        for (int i = threadIdx.x; i < KR; i += blockDim.x) crow[i] = row[q_rank + i] * rc * wkv[i];
    }
    for (int i = threadIdx.x; i < rot.dims / 2; i += blockDim.x) rotate_pair(kr, crow + KR, i, pos, rot);
    for (int i = rot.dims + threadIdx.x; i < R; i += blockDim.x) crow[KR + i] = kr[i];
}

__global__ __launch_bounds__(256) void q_rotary_kernel(const float* q, int ldq, float* qa, int ldqa, int H, int D, int R, int KR, Rotary rot,
                                                       const int* row_pos, bf16_t* qa16) {
    const int m = blockIdx.x, pos = row_pos[m], half = rot.dims / 2;
    for (int idx = threadIdx.x; idx < H * half; idx += blockDim.x) {
        const int h = idx / half, i = idx % half;
        const size_t at = (size_t)m * ldqa + (size_t)h * (KR + R) + KR;
        rotate_pair(q + (size_t)m * ldq + (size_t)h * (D + R) + D, qa16 ? nullptr : qa + at, i, pos, rot, qa16 ? qa16 + at : nullptr);
    }
    const int rest = R - rot.dims;
    for (int idx = threadIdx.x; idx < H * rest; idx += blockDim.x) {
        const int h = idx / rest, i = rot.dims + idx % rest;
        put_row(qa16 ? nullptr : qa, qa16, (size_t)m * ldqa + (size_t)h * (KR + R) + KR + i, q[(size_t)m * ldq + (size_t)h * (D + R) + D + i]);
    }
}

// Queries projected directly: blockIdx.y == 0 rotates the heads' query parts into qa (neither qa nor qa16: not asked for), blockIdx.y == 1 (layers with latents of their
// own) norms the latent, rotates the shared key part and files both in the token's cache row.
__global__ __launch_bounds__(256) void latent_direct_prep_kernel(const float* proj, int ld, int H, int D, int R, int KR, int kv_col, const float* wkv,
                                                                 float eps, Rotary rot, const int* row_pos, const int* row_slot, const int* page_table,
                                                                 int max_pages, int page_tokens, float* qa, float* cache, bf16_t* qa16) {
    __shared__ float s_red[8];
    const int m = blockIdx.x, pos = row_pos[m], half = rot.dims / 2;
    const float* row = proj + (size_t)m * ld;
    if (blockIdx.y == 0 && (qa || qa16)) {
        const int rest = R - rot.dims, per = half + rest;
        for (int idx = threadIdx.x; idx < H * per; idx += blockDim.x) {
            const int h = idx / per, i = idx % per;
            const float* src = row + (size_t)h * (D + R) + D;
            const size_t at = ((size_t)m * H + h) * (KR + R) + KR;
            float* dst = qa16 ? nullptr : qa + at;
            bf16_t* dst16 = qa16 ? qa16 + at : nullptr;
            if (i < half) rotate_pair(src, dst, i, pos, rot, dst16);
            else put_row(dst, dst16, rot.dims + i - half, src[rot.dims + i - half]);
        }
        return;
    }
    const float* lat = row + kv_col;
    const float rc = row_inv_rms(lat, KR, eps, s_red);
    float* crow = cache + cache_row(page_table, max_pages, page_tokens, row_slot[m], pos) * (size_t)(KR + R);
    for (int i = threadIdx.x; i < KR; i += blockDim.x) crow[i] = lat[i] * rc * wkv[i];
    const float* kr = lat + KR;
    for (int i = threadIdx.x; i < half; i += blockDim.x) rotate_pair(kr, crow + KR, i, pos, rot);
    for (int i = rot.dims + threadIdx.x; i < R; i += blockDim.x) crow[KR + i] = kr[i];
}

// One workgroup per (row, head).  The lanes of a wave split the KR + R dimensions of a cache row (ND per lane); a wave walks
// its share of the keys four at a time with a running (maximum, sum, weighted latent) and the four waves are merged at the end.
// With n_split > 1 (decode steps: few rows, long key ranges) grid.z workgroups share a row's keys in ranges of whole groups of 16
// and leave (maximum, sum, weighted latent) partials in ws for latent_merge_kernel.
// gate (may be null): head h's result is multiplied by sigmoid(gate[m ldg + h]) where it is written.
// 8 rows, 12 heads on latents of 256 + 32, some 300 keys: 4.6 us and 3.2 for the merge (13.4 and 4.6 with loads under their own bounds
// checks and ranges of 64 keys and more: four dependent round trips instead of one).
template <int ND>
__global__ __launch_bounds__(256) void latent_attention_kernel(const float* qa, float* ctx, int H, int KR, int R, float scale, const int* row_pos,
                                                               const int* row_slot, const int* page_table, int max_pages, int page_tokens,
                                                               const float* cache, float* ws, int n_split, const float* gate, int ldg,
                                                               const float* sink) {
    __shared__ float s_m[4], s_l[4];
    __shared__ float s_acc[4][ND * 64];
    const int m = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int DT = KR + R, n_keys = row_pos[m] + 1, slot = row_slot[m];
    int k_lo = 0, k_hi = n_keys;
    if (n_split > 1) {
        const int chunk = split_chunk(n_keys, n_split);
        k_lo = min(n_keys, (int)blockIdx.z * chunk);
        k_hi = min(n_keys, k_lo + chunk);
    }
    const float* qrow = qa + ((size_t)m * H + h) * DT;
    float q[ND], acc[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int d = lane + 64 * i;
        const float v = qrow[min(d, DT - 1)];
        q[i] = d < DT ? v : 0.0f;
        acc[i] = 0.0f;
    }
    float mx = -INFINITY, l = 0.0f;
    const int* pt = page_table + (size_t)slot * max_pages;
    for (int kb = k_lo + wave * 4; kb < k_hi; kb += 16) {
        float r[4][ND], s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int key = kb + u < k_hi ? kb + u : kb;
            const float* row = cache + ((size_t)pt[key / page_tokens] * page_tokens + key % page_tokens) * DT;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                r[u][i] = row[min(lane + 64 * i, DT - 1)];  // (unconditional: every load in flight before the first is used)
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float part = 0.0f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                if (lane + 64 * i >= DT) r[u][i] = 0.0f;
                part = fmaf(q[i], r[u][i], part);
            }
            s[u] = part;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[u] = wave_allsum(s[u]) * scale;
            if (kb + u >= k_hi) s[u] = -INFINITY;
        }
        const float mn = fmaxf(fmaxf(mx, s[0]), fmaxf(fmaxf(s[1], s[2]), s[3]));
        const float alpha = expf(mx - mn);  // 0 for the first group (mx = -inf, mn finite: key kb is always valid)
        float pw[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) pw[u] = expf(s[u] - mn);
        l = l * alpha + ((pw[0] + pw[1]) + (pw[2] + pw[3]));
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            float a = acc[i] * alpha;
#pragma unroll
            for (int u = 0; u < 4; ++u) a = fmaf(pw[u], r[u][i], a);
            acc[i] = a;
        }
        mx = mn;
    }
    if (lane == 0) {
        s_m[wave] = mx;
        s_l[wave] = l;
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) s_acc[wave][lane + 64 * i] = acc[i];
    __syncthreads();
    const float M4 = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
    float wgt[4], L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        wgt[w] = M4 == -INFINITY ? 0.0f : expf(s_m[w] - M4);  // a wave without keys: exp(-inf) = 0; a range without keys: all zero
        L += wgt[w] * s_l[w];
    }
    if (n_split > 1) {
        float* part = ws + (((size_t)m * H + h) * n_split + blockIdx.z) * (KR + 2);
        if (threadIdx.x == 0) {
            part[0] = M4;
            part[1] = L;
        }
        for (int d = threadIdx.x; d < KR; d += blockDim.x) {
            float a = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) a = fmaf(wgt[w], s_acc[w][d], a);
            part[2 + d] = a;
        }
        return;
    }
    float* out = ctx + ((size_t)m * H + h) * KR;
    const float gf = head_gate_f(gate, ldg, m, h) * (sink ? sink_norm_f(M4, L, sink, h) : 1.0f);
    for (int d = threadIdx.x; d < KR; d += blockDim.x) {
        float a = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) a = fmaf(wgt[w], s_acc[w][d], a);
        out[d] = sink ? a * gf : a / L * gf;
    }
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;

// Tiles of 32 cached rows as the matrix cores read them: bf16, rows of 16 NKS dimensions (zeros behind the last one) padded so that
// four consecutive rows start 16 or 48 banks apart, 16-byte chunks swizzled by the row's second bit pair — then a fragment read of
// 16 rows, and a transposed read of four, touch every bank once.
template <int NKS>
struct KeyTile {
    static constexpr int DT = NKS * 16, LD = DT + ((DT / 2) % 64 == 0 ? 32 : 0);  // elements per row
    static constexpr int BYTES = 32 * LD * 2, PIECES = BYTES / 1024;
    static_assert(BYTES % 1024 == 0 && LD % 32 == 0, "a tile is whole 1 KB pieces");
};
constexpr int kLog2eBits = 0x3fb8aa3b;  // log2(e)

// Entries of a step, one per lane (64 at a time): the rows of entry e cut into blocks of 32 queries, its cached rows (this step's
// included) into tiles of 32 keys.  Finds the entry of query block `id` (of BQ queries) and the key tiles of the entries in front of it.
// Everything the caller needs of the entry comes out of the same two loads, in front of the scan.
struct EntryAt {
    int block, first_tile;
    int start, len, pos, slot;  // of the entry: first row, rows, position of the first row, cache slot
};
template <int BQ = 32>
__device__ __forceinline__ bool find_entry(int id, const int* ent_start, const int* ent_len, const int* ent_slot, int n_entries, const int* row_pos, EntryAt& at) {
    const int lane = threadIdx.x & 63;
    int tiles_before = 0;
    for (int e0 = 0; e0 < n_entries; e0 += 64) {
        const int e = min(e0 + lane, n_entries - 1);
        const int len = e0 + lane < n_entries ? ent_len[e] : 0, start = ent_start[e], slot = ent_slot[e];
        const int pos = len > 0 ? row_pos[start] : 0;
        const int blocks = (len + BQ - 1) / BQ, tiles = len > 0 ? (pos + len + 31) / 32 : 0;
        int b = blocks, t = tiles;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int ob = __shfl_up(b, d, 64), ot = __shfl_up(t, d, 64);
            if (lane >= d) {
                b += ob;
                t += ot;
            }
        }
        const unsigned long long past = __ballot(id < b);
        if (past) {
            const int l = __builtin_ctzll(past);
            at.start = __builtin_amdgcn_readlane(start, l);
            at.len = __builtin_amdgcn_readlane(len, l);
            at.pos = __builtin_amdgcn_readlane(pos, l);
            at.slot = __builtin_amdgcn_readlane(slot, l);
            at.block = id - __builtin_amdgcn_readlane(b - blocks, l);
            at.first_tile = tiles_before + __builtin_amdgcn_readlane(t - tiles, l);
            return true;
        }
        id -= __builtin_amdgcn_readlane(b, 63);
        tiles_before += __builtin_amdgcn_readlane(t, 63);
    }
    return false;
}

// The cached rows of every entry of the step as key tiles, back to back in entry order.  Each tile is read by every query block
// behind it and by all heads: converting it once (8 x 1023 rows of 288 values: 9 us) took the conversion, the page table and the
// 4-byte loads out of loops that ran 16 times over every tile.
// A tile is multiplied for queries in front of some of its keys too, with weight zero, and zero times a value that is not finite is not
// zero: such values of the latent part are left out, and the row's last column, which only the scores read, says so (NaN): the queries that see
// the key come out NaN, the others do not meet it.
template <int NKS>
__global__ __launch_bounds__(256) void latent_tiles_kernel(const float* cache, int DT, int KR, const int* ent_start, const int* ent_len, const int* ent_slot,
                                                           int n_entries, const int* row_pos, const int* page_table, int max_pages, int page_tokens,
                                                           bf16_t* tiles) {
    typedef KeyTile<NKS> T;
    __shared__ unsigned s_bad;  // rows with a latent value that is not finite (as bf16)
    const int e = blockIdx.y, lane = threadIdx.x & 63;
    const int len = ent_len[e];
    if (len <= 0) return;
    const int n_keys = row_pos[ent_start[e] + len - 1] + 1;
    if ((int)blockIdx.x * 32 >= n_keys) return;
    if (threadIdx.x == 0) s_bad = 0;
    __syncthreads();
    int first = 0;  // tiles of the entries in front
    for (int e0 = 0; e0 < e; e0 += 64) {
        const int o = e0 + lane, ol = o < e ? ent_len[o] : 0;
        int t = ol > 0 ? (row_pos[ent_start[o] + ol - 1] + 32) / 32 : 0;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) t += __shfl_xor(t, d, 64);
        first += t;
    }
    bf16_t* out = tiles + (size_t)(first + blockIdx.x) * (T::BYTES / 2);
    const int* pt = page_table + (size_t)ent_slot[e] * max_pages;
    const bool vec = DT % 4 == 0 && (reinterpret_cast<uintptr_t>(cache) & 15) == 0;
    for (int idx = threadIdx.x; idx < 32 * (T::LD / 8); idx += 256) {
        const int key = idx / (T::LD / 8), c = idx % (T::LD / 8), kpos = blockIdx.x * 32 + key;
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = 0.0f;
        if (kpos < n_keys) {
            const float* row = cache + ((size_t)pt[kpos / page_tokens] * page_tokens + kpos % page_tokens) * DT;
            if (vec && c * 8 + 8 <= DT) {
                const f32x4 a = *reinterpret_cast<const f32x4*>(row + c * 8), b = *reinterpret_cast<const f32x4*>(row + c * 8 + 4);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (c * 8 + u < DT) v[u] = row[c * 8 + u];
            }
            bool bad = false;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c * 8 + u < KR && !(fabsf(v[u]) < 3.3961775e38f)) {  // (from here on it rounds to an infinity)
                    v[u] = 0.0f;
                    bad = true;
                }
            if (bad) atomicOr(&s_bad, 1u << key);
        }
        *reinterpret_cast<u32x4*>(out + key * T::LD + (c ^ ((key >> 2) & 3)) * 8) =
            u32x4{cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]), cvt_pk_bf16(v[4], v[5]), cvt_pk_bf16(v[6], v[7])};
    }
    __syncthreads();
    if (threadIdx.x < 32 && (s_bad >> threadIdx.x & 1u) != 0) {
        constexpr int c = T::DT / 8 - 1;  // (behind the 32 NT value columns of every kernel that reads these tiles)
        out[threadIdx.x * T::LD + (c ^ ((threadIdx.x >> 2) & 3)) * 8 + 7] = 0x7FC0;
    }
}

// Prompt portions in bf16 mode: the same attention on the matrix cores.  A workgroup takes 32 consecutive queries of one entry and
// four heads (one per wave), which share the tiles of 32 keys that arrive by DMA in two LDS buffers, one barrier per tile.  Both
// products are computed transposed (S^T = K Q^T, O^T = C^T P^T): a lane's column is a query, so the running maximum and sum are
// per-lane values and the probabilities a lane computed are exactly the eight per k-step it has to feed back (keys {0-3, 8-11} from
// the lower half-wave, {4-7, 12-15} from the upper one); the latent part is read back transposed from the same rows the scores used
// (ds_read_b64_tr_b16).  Scores, softmax and both accumulations are fp32; q, cache rows and probabilities enter the products as bf16.
// Bound by the matrix cores and the LDS together: a fragment of keys (1 KB) serves one product (32 cycles), so the four SIMDs of a
// compute unit ask the LDS for its whole 128 B per clock; two workgroups per compute unit hide the softmax of one under the
// products of the other (hence 256 registers a lane: 72 of queries, 128 of sums).  The blocks with the most keys are dealt first.
// 8 x 1023 tokens, 16 heads on latents of 256 + 32: 116 us and 9 for the tiles (73 GFLOP: 585 TFLOP/s); 827 us when every workgroup
// converted and transposed its own tiles behind three barriers.
template <int NKS, int NT>  // 16 NKS >= KR + R (score dimensions), 32 NT >= KR (latent dimensions)
__global__ __launch_bounds__(256, NKS > 18 ? 1 : 2) void latent_attention_mfma_kernel(const float* qa, const bf16_t* qa16, float* ctx, bf16_t* ctx16, int H, int KR, int R, float scale,
                                                                       const int* ent_start, const int* ent_len, const int* ent_slot, int n_entries, const int* row_pos,
                                                                       const bf16_t* tiles, const float* gate, int ldg, const float* sink) {
    typedef KeyTile<NKS> T;
    static_assert(NT * 32 < T::DT, "the latent part lies inside the rows, in front of their last column");
    __shared__ __attribute__((aligned(1024))) char Ks[2][T::BYTES];
    EntryAt at;
    if (!find_entry(gridDim.x - 1 - blockIdx.x, ent_start, ent_len, ent_slot, n_entries, row_pos, at)) return;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.y * 4 + wave;
    const bool head_ok = h < H;
    const int m_first = at.start + at.block * 32, nq = min(32, at.len - at.block * 32);
    const int pos_first = at.pos + at.block * 32, qpos = pos_first + r, DT = KR + R;
    const int n_tiles = (pos_first + nq + 31) / 32;
    const char* src = reinterpret_cast<const char*>(tiles) + (size_t)at.first_tile * T::BYTES + lane * 16;

    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)&Ks[0][0];
    auto request = [&](int kt, int buf) {
        const char* g = src + (size_t)kt * T::BYTES;
#pragma unroll
        for (int pc = 0; pc < (T::PIECES + 3) / 4; ++pc) {
            const int i = wave + 4 * pc;
            // (written here, not by the builtin: the compiler would wait for the next tile in front of this tile's latent part)
            if (i < T::PIECES)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds0 + buf * T::BYTES + i * 1024), "v"(g + i * 1024) : "memory", "m0");
        }
    };
    request(0, 0);
    bf16x8 qf[NKS];
    {
        const size_t q_at = ((size_t)(m_first + (r < nq ? r : 0)) * H + (head_ok ? h : 0)) * DT;  // (beyond the block: some valid row, never stored)
        const float* qrow = qa + q_at;
        auto round8 = [](const f32x4& a, const f32x4& b) {
            return __builtin_bit_cast(bf16x8, u32x4{cvt_pk_bf16(a.x, a.y), cvt_pk_bf16(a.z, a.w), cvt_pk_bf16(b.x, b.y), cvt_pk_bf16(b.z, b.w)});
        };
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        if (qa16) {  // rounded by their producers (DT is a multiple of 8)
            const u32x4 none = {0u, 0u, 0u, 0u};
            u32x4 q8[NKS];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) q8[ks] = *reinterpret_cast<const u32x4*>(qa16 + q_at + min(ks * 16 + 8 * hf, DT - 8));
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, ks * 16 + 8 * hf < DT ? q8[ks] : none);
        } else if (DT % 4 == 0 && (reinterpret_cast<uintptr_t>(qa) & 15) == 0) {
            f32x4 q4[2 * NKS];
#pragma unroll
            for (int i = 0; i < 2 * NKS; ++i) q4[i] = *reinterpret_cast<const f32x4*>(qrow + min((i >> 1) * 16 + 8 * hf + 4 * (i & 1), DT - 4));
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int d = ks * 16 + 8 * hf;
                qf[ks] = round8(d + 4 <= DT ? q4[2 * ks] : zero, d + 8 <= DT ? q4[2 * ks + 1] : zero);
            }
        } else {
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                f32x4 ab[2] = {zero, zero};
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (ks * 16 + 8 * hf + u < DT) ab[u >> 2][u & 3] = qrow[ks * 16 + 8 * hf + u];
                qf[ks] = round8(ab[0], ab[1]);
            }
        }
    }
    f32x16 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;
    float mx = -INFINITY, lsum = 0.0f;  // maximum in units of log2
    const float to_log2 = scale * __uint_as_float(kLog2eBits);

    // byte offsets inside a tile: this lane's key row for the scores (even and odd k-steps), its rows for the transposed reads
    const int swz = (r >> 2) & 3;
    const int k_even = r * T::LD * 2 + ((0 + hf) ^ swz) * 16, k_odd = r * T::LD * 2 + ((2 + hf) ^ swz) * 16;
    const int i16 = lane & 15, G = (lane >> 4) & 1, vc = 2 * G + ((i16 & 3) >> 1);
    const int v_lo = (4 * hf + (i16 >> 2)) * T::LD * 2 + ((vc ^ hf) * 16) + (i16 & 1) * 8;
    const int v_hi = (8 + 4 * hf + (i16 >> 2)) * T::LD * 2 + ((vc ^ (hf + 2)) * 16) + (i16 & 1) * 8;
    typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

    // vmcnt(0): this wave's pieces have landed; lgkmcnt(0), said to the compiler: with scalar loads in flight it would wait for all fragments at once
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
    for (int kt = 0; kt < n_tiles; ++kt) {
        const char* K = Ks[kt & 1];
        if (kt + 1 < n_tiles) request(kt + 1, (kt + 1) & 1);
        if (head_ok) {
            // fragments are requested AHEAD products before they are used (left alone, the compiler pairs each request with its product and
            // waits out the LDS latency 34 times per tile)
            constexpr int AHEAD = 5;
            auto key_part = [&](int ks) { return *reinterpret_cast<const u32x4*>(K + ((ks & 1) ? k_odd : k_even) + (ks >> 1) * 64); };
            u32x4 kf[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) kf[i] = key_part(i);
            __builtin_amdgcn_sched_barrier(0);
            f32x16 sacc;
#pragma unroll
            for (int i = 0; i < 16; ++i) sacc[i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[ks % AHEAD]), qf[ks], sacc, 0, 0, 0);
                if (ks + AHEAD < NKS) kf[ks % AHEAD] = key_part(ks + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
            float tmax = -INFINITY;
            if (kt * 32 + 31 > pos_first) {  // some query does not see the whole tile
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kt * 32 + 8 * (i >> 2) + 4 * hf + (i & 3) > qpos) sacc[i] = -INFINITY;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                sacc[i] *= to_log2;
                tmax = fmaxf(tmax, sacc[i]);
            }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
            // The reference point of the exponentials moves only when some query's maximum grew by more than 2^11 (the weights stay far
            // inside fp32 and bf16 range): the accumulators are rescaled on few tiles instead of on every one.
            if (__any(tmax > mx + 11.0f)) {  // also the first tile (mx = -inf)
                const float mn = tmax > mx + 11.0f ? tmax : mx;
                const float alpha = mx == mn ? 1.0f : __builtin_amdgcn_exp2f(mx - mn);  // mx = -inf, mn finite: 0
                lsum *= alpha;
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[t][i] *= alpha;
                mx = mn;
            }
            const float mref = fmaxf(mx, -1e30f);  // (no key seen so far: 2^(-inf) = 0, not NaN)
            uint32_t pk[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float p0 = __builtin_amdgcn_exp2f(sacc[2 * i] - mref), p1 = __builtin_amdgcn_exp2f(sacc[2 * i + 1] - mref);
                lsum += p0 + p1;
                pk[i] = cvt_pk_bf16(p0, p1);
            }
            const bf16x8 pf[2] = {__builtin_bit_cast(bf16x8, u32x4{pk[0], pk[1], pk[2], pk[3]}), __builtin_bit_cast(bf16x8, u32x4{pk[4], pk[5], pk[6], pk[7]})};
            auto value_part = [&](int x) {  // 16 keys x 32 dimensions, transposed
                const int off = (x / NT) * 16 * T::LD * 2 + (x % NT) * 64;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(K + v_lo + off));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(K + v_hi + off));
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            };
            bf16x8 vf[AHEAD];
#pragma unroll
            for (int i = 0; i < (AHEAD < 2 * NT ? AHEAD : 2 * NT); ++i) vf[i] = value_part(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int x = 0; x < 2 * NT; ++x) {
                o[x % NT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x % AHEAD], pf[x / NT], o[x % NT], 0, 0, 0);
                if (x + AHEAD < 2 * NT) vf[x % AHEAD] = value_part(x + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the next tile's pieces
        __syncthreads();
    }
    if (!head_ok) return;
    const float L = lsum + __shfl_xor(lsum, 32, 64);
    if (ctx16) {  // (KR is a multiple of 8)
        // A lane has a query's values: turned in the tiles' place, half of the dimensions at a time, they leave as 16-byte pieces of whole rows.
        // (8 bytes a lane to 32 rows, divided one by one: 6.1 us behind the last tile, 3.3 so; 2.0 with one reciprocal a
        // row, whose quotients are a last bit off: these are the division's.)
        constexpr int P = NT * 16, PITCH = P * 2 + 16;
        static_assert(32 * PITCH <= T::BYTES / 2, "a wave's rows fit its half of a tile's place");
        char* const img = &Ks[0][0] + wave * (T::BYTES / 2);
        const size_t row = (size_t)(m_first + min(r, nq - 1));
        const float gf = head_gate_f(gate, ldg, row, h) * (sink ? sink_norm_f(mx * 0.69314718055994531f, L, sink, h) : 1.0f), inv = 1.0f / L;
        auto value = [&](float v) { return (sink ? v : quotient(v, L, inv)) * gf; };
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int t = 0; t < NT / 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; i += 4) {
                    const f32x16& v = o[half * (NT / 2) + t];
                    *reinterpret_cast<u32x2*>(img + r * PITCH + (t * 32 + 8 * (i >> 2) + 4 * hf) * 2) = u32x2{cvt_pk_bf16(value(v[i]), value(v[i + 1])), cvt_pk_bf16(value(v[i + 2]), value(v[i + 3]))};
                }
            // (a wave's accesses to the LDS are in order)
#pragma unroll
            for (int q = 0; q < P / 16; ++q) {
                const int u = q * 64 + lane, qr = u / (P / 8), c = u % (P / 8) * 8;
                const u32x4 v = *reinterpret_cast<const u32x4*>(img + qr * PITCH + c * 2);
                if (qr < nq && half * P + c < KR) *reinterpret_cast<u32x4*>(ctx16 + ((size_t)(m_first + qr) * H + h) * KR + half * P + c) = v;
            }
        }
        return;
    }
    if (r >= nq) return;
    const size_t out_at = ((size_t)(m_first + r) * H + h) * KR;
    float* out = ctx + out_at;
    const float gf = head_gate_f(gate, ldg, (size_t)(m_first + r), h) * (sink ? sink_norm_f(mx * 0.69314718055994531f, L, sink, h) : 1.0f);
    const bool vec = KR % 4 == 0 && (reinterpret_cast<uintptr_t>(ctx) & 15) == 0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
            const int d = t * 32 + 8 * (i >> 2) + 4 * hf;
            f32x4 v;
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = sink ? o[t][i + u] * gf : o[t][i + u] / L * gf;
            if (vec) {
                if (d < KR) *reinterpret_cast<f32x4*>(out + d) = v;
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (d + u < KR) out[d + u] = v[u];
            }
        }
}

// Prompt portions in 32-bit mode: the same attention on the matrix cores' fp32 products.  A workgroup takes 16 consecutive queries of one
// entry and one head; its four waves take every fourth tile of 16 keys and are merged at the end.  Transposed as above (S^T = K Q^T,
// O^T = C^T P^T): a lane's column is a query, and its four probabilities are the four it has to feed back.  Which of the 16 dimensions of
// a piece a lane group multiplies is free as long as both operands agree, so that every load is 16 bytes: four consecutive dimensions of
// a key for the scores; for the latent part four consecutive dimensions of one of the lane group's own keys, a row of four result tiles.
// Keys go from the cache to registers (18 loads of 16 bytes a tile and 16 for the latent part, 34 KB against 4.3 k cycles of products: what
// a compute unit can take in beside them); the latent part of a tile is requested piece by piece under its scores, the next tile's keys
// under this tile's sums.  A masked key must not reach the sums as 0 x infinity: the tiles on the diagonal look whether a value is not
// finite, and then add key by key.
// 333 tokens, 12 heads on latents of 256 + 32: 31 us against 118.8 with a wave per key row and its dimensions over the lanes.
template <int NKS, int NV, bool EXACT>  // 16 NKS >= KR + R (score dimensions), 64 NV >= KR (latent dimensions); EXACT: equal
__global__ __launch_bounds__(256, EXACT && NKS <= 18 ? 2 : 1) void latent_attention_f32_kernel(const float* qa, float* ctx, int H, int KR, int R, float scale,
    const int* ent_start, const int* ent_len, const int* ent_slot, int n_entries, const int* row_pos, const int* page_table, int max_pages,
    int page_tokens, const float* cache, const float* gate, int ldg, const float* sink) {
    static_assert(4 * NV <= NKS, "the latent part is requested under the scores");
    constexpr int LDO = NV * 64 + 4;
    __shared__ __attribute__((aligned(16))) float s_o[2][16][LDO];
    __shared__ f32x4 s_q[NKS][64];
    __shared__ float s_m[4][16], s_l[4][16];
    EntryAt at;
    if (!find_entry<16>(gridDim.x - 1 - blockIdx.x, ent_start, ent_len, ent_slot, n_entries, row_pos, at)) return;
    const int tid = threadIdx.x, lane = tid & 63, q = lane & 15, g = lane >> 4, h = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m_first = at.start + at.block * 16, nq = min(16, at.len - at.block * 16), DT = KR + R;
    const int pos_first = at.pos + at.block * 16, qpos = pos_first + q, n_keys = pos_first + nq, n_tiles = (n_keys + 15) / 16;
    const int* pt = page_table + (size_t)at.slot * max_pages;
    // piece c of a row of scores, of the latent part: where they end inside the last pieces, some valid piece (zeroed, never stored)
    auto k_at = [&](int c) { return EXACT ? c * 16 + g * 4 : min(c * 16 + g * 4, DT - 4); };
    auto v_at = [&](int d) { return EXACT ? d : min(d, KR - 4); };
    auto row_of = [&](int tile) {  // cache row of key 16 tile + q
        const int key = min(tile * 16 + q, n_keys - 1);
        return pt[key / page_tokens] * page_tokens + key % page_tokens;
    };
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 kf[NKS], vf[4 * NV], acc[4 * NV];
    const float* qrow = qa + ((size_t)(m_first + min(q, nq - 1)) * H + h) * DT;
    int row = row_of(min(wave, n_tiles - 1));
    {
        const float* kp = cache + (size_t)row * DT;
#pragma unroll
        for (int c = 0; c < NKS; ++c) kf[c] = *reinterpret_cast<const f32x4*>(kp + k_at(c));
    }
    for (int c = wave; c < NKS; c += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(qrow + k_at(c));
        s_q[c][lane] = EXACT || c * 16 + g * 4 < DT ? v : zero;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4 * NV; ++i) acc[i] = zero;
    float mx = -INFINITY, l = 0.0f;
    for (int kt = wave; kt < n_tiles; kt += 4) {
        const float* vp[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) vp[i] = cache + (size_t)__shfl(row, g * 4 + i, 64) * DT;
        const int next_row = row_of(min(kt + 4, n_tiles - 1));
        f32x4 s0 = zero, s1 = zero, qn = s_q[0][lane];
#pragma unroll
        for (int c = 0; c < NKS; ++c) {
            if (c < 4 * NV) vf[c] = *reinterpret_cast<const f32x4*>(vp[c / NV] + v_at((c % NV) * 64 + q * 4));
            const f32x4 k = EXACT || c * 16 + g * 4 < DT ? kf[c] : zero, qc = qn;
            qn = s_q[c + 1 < NKS ? c + 1 : 0][lane];
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.x, qc.x, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.y, qc.y, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.z, qc.z, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.w, qc.w, s1, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int key0 = kt * 16 + g * 4;
        float p[4], top = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[i] = key0 + i <= qpos ? (s0[i] + s1[i]) * scale : -INFINITY;
            top = fmaxf(top, p[i]);
        }
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float mn = fmaxf(mx, top), base = mn == -INFINITY ? 0.0f : mn;  // (no key of the tile, and none before, is this query's)
        const float alpha = expf(mx - base);
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = expf(p[i] - base);
        l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
        mx = mn;
#pragma unroll
        for (int i = 0; i < 4 * NV; ++i) acc[i] *= alpha;
        bool by_key = false;
        if (kt * 16 + 15 > pos_first) {  // (uniform) some query of the block does not see the whole tile
            float z = 0.0f;
#pragma unroll
            for (int j = 0; j < 4 * NV; ++j) z += (vf[j].x * 0.0f + vf[j].y * 0.0f) + (vf[j].z * 0.0f + vf[j].w * 0.0f);
            by_key = __any(!(z == 0.0f));
        }
        const float* kp = cache + (size_t)next_row * DT;
        if (__builtin_expect(by_key, 0)) {
#pragma unroll 1
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float pj = __shfl(p[i], j * 16 + q, 64);
                    const float* v = cache + (size_t)__shfl(row, j * 4 + i, 64) * DT;
                    const bool seen = kt * 16 + j * 4 + i <= qpos;
#pragma unroll
                    for (int b = 0; b < 4 * NV; ++b) {  // the four dimensions of result row 4 g + b % 4
                        const f32x4 x = *reinterpret_cast<const f32x4*>(v + v_at((b >> 2) * 64 + g * 16 + (b & 3) * 4));
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            acc[(b >> 2) * 4 + t][b & 3] = seen ? fmaf(pj, x[t], acc[(b >> 2) * 4 + t][b & 3]) : acc[(b >> 2) * 4 + t][b & 3];
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
#pragma unroll
            for (int b = 0; b < 4 * NV; ++b) vf[b] = zero;
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < NKS; ++j) {
            kf[j] = *reinterpret_cast<const f32x4*>(kp + k_at(j));
            if (j < 4 * NV) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[(j % NV) * 4 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j][t], p[j / NV], acc[(j % NV) * 4 + t], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        row = next_row;
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) {
        s_m[wave][q] = mx;
        s_l[wave][q] = l;
    }
    __syncthreads();
    const float top = fmaxf(fmaxf(s_m[0][q], s_m[1][q]), fmaxf(s_m[2][q], s_m[3][q]));
    const float w = top == -INFINITY ? 0.0f : expf(mx - top);  // (a wave without keys: 0)
#pragma unroll
    for (int i = 0; i < 4 * NV; ++i) acc[i] *= w;
    for (int half = 1; half >= 0; --half) {  // waves 2 and 3 leave their sums, waves 0 and 1 add theirs
        if (wave >> 1 == half) {
#pragma unroll
            for (int b = 0; b < 4 * NV; ++b) {
                f32x4* o = reinterpret_cast<f32x4*>(&s_o[wave & 1][q][(b >> 2) * 64 + g * 16 + (b & 3) * 4]);
                f32x4 v;
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = acc[(b >> 2) * 4 + t][b & 3];
                *o = half ? v : *o + v;
            }
        }
        __syncthreads();
    }
    for (int i = tid; i < 16 * (KR >> 2); i += 256) {
        const int qi = i / (KR >> 2), d = (i - qi * (KR >> 2)) * 4;
        if (qi >= nq) break;
        float mq = fmaxf(fmaxf(s_m[0][qi], s_m[1][qi]), fmaxf(s_m[2][qi], s_m[3][qi])), L = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) L += (mq == -INFINITY ? 0.0f : expf(s_m[k][qi] - mq)) * s_l[k][qi];
        const size_t m = m_first + qi;
        const float gf = head_gate_f(gate, ldg, m, h) * (sink ? sink_norm_f(mq, L, sink, h) : 1.0f / L);
        const f32x4 v = *reinterpret_cast<const f32x4*>(&s_o[0][qi][d]) + *reinterpret_cast<const f32x4*>(&s_o[1][qi][d]);
        *reinterpret_cast<f32x4*>(ctx + (m * H + h) * KR + d) = v * gf;
    }
}

// ctx[m][h] from the partials of latent_attention_kernel, in a fixed order (the result does not depend on timing); only the
// ranges that held keys are read
__global__ __launch_bounds__(256) void latent_merge_kernel(const float* ws, float* ctx, int H, int KR, int n_split, const int* row_pos, const float* gate,
                                                           int ldg, const float* sink) {
    __shared__ float s_w[64];
    __shared__ float s_L, s_M;
    const int m = blockIdx.x, h = blockIdx.y, n_keys = row_pos[m] + 1;
    const int chunk = split_chunk(n_keys, n_split);
    const int used = min(n_split, (n_keys + chunk - 1) / chunk);
    const float* part = ws + ((size_t)m * H + h) * n_split * (KR + 2);
    if (threadIdx.x < 64) {
        const int sidx = threadIdx.x;
        const float pm = sidx < used ? part[(size_t)sidx * (KR + 2)] : -INFINITY;
        const float M = wave_allmax(pm);
        const float w = pm == -INFINITY ? 0.0f : expf(pm - M);
        s_w[sidx] = w;
        const float L = wave_allsum(sidx < used ? w * part[(size_t)sidx * (KR + 2) + 1] : 0.0f);
        if (sidx == 0) {
            s_L = L;
            s_M = M;
        }
    }
    __syncthreads();
    float* out = ctx + ((size_t)m * H + h) * KR;
    const float L = s_L, gf = head_gate_f(gate, ldg, m, h) * (sink ? sink_norm_f(s_M, L, sink, h) : 1.0f);
    for (int d = threadIdx.x; d < KR; d += blockDim.x) {
        float a = 0.0f;
        for (int s0 = 0; s0 < used; s0 += 16) {  // sixteen partials in flight (those beyond the last repeat it with weight 0)
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = part[(size_t)min(s0 + u, used - 1) * (KR + 2) + 2 + d];
#pragma unroll
            for (int u = 0; u < 16; ++u)
                if (s0 + u < used) a = fmaf(s_w[s0 + u], v[u], a);
        }
        out[d] = sink ? a * gf : a / L * gf;
    }
}

// the next step's rows: the tokens this one drew, one position further; also to host memory
__global__ __launch_bounds__(64) void advance_rows_kernel(const int* tok, int M, int* ids, int* pos, int* seen) {
    const int r = blockIdx.x * 64 + threadIdx.x;
    if (r >= M) return;
    const int t = tok[r];
    ids[r] = t;
    pos[r] += 1;
    seen[r] = t;
}

__global__ __launch_bounds__(64) void new_pages_kernel(int* table, const NewPages pages) {
#pragma unroll
    for (int i = 0; i < kGemvMaxRows; ++i)
        if ((int)threadIdx.x == i && i < pages.n) table[pages.at[i]] = pages.page[i];
}

// The largest of a workgroup's values and its index (the smaller one of equals), in every thread; s_v, s_i: four each.
__device__ __forceinline__ void block_argmax(float& best, int& bi, float* s_v, int* s_i) {
    const float wbest = wave_allmax(best);
    int cand = (best == wbest) ? bi : 0x7fffffff;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) cand = min(cand, __shfl_xor(cand, off, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        s_v[wave] = wbest;
        s_i[wave] = cand;
    }
    __syncthreads();
    best = s_v[0];
    bi = s_i[0];
    for (int w = 1; w < 4; ++w)
        if (s_v[w] > best || (s_v[w] == best && s_i[w] < bi)) {
            best = s_v[w];
            bi = s_i[w];
        }
}

__global__ __launch_bounds__(256) void next_token_kernel(const NextToken a) {
    __shared__ float s_v[4], s_red[4];
    __shared__ int s_i[4];
    const int m = blockIdx.x, tid = threadIdx.x, at = min(tid * 4, a.W - 4);
    const bool in = tid * 4 < a.W;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const int part = min(tid, a.n_parts - 1);
    float best = a.part_val[(size_t)m * a.n_parts + part];
    int bi = a.part_idx[(size_t)m * a.n_parts + part];
    const f32x4 wn = *reinterpret_cast<const f32x4*>(a.wn + at);
    f32x4 mu = zero, before = zero;
    if (a.mu) {
        mu = *reinterpret_cast<const f32x4*>(a.mu + at);
        before = *reinterpret_cast<const f32x4*>(a.last_h + (size_t)m * a.W + at);
    }
    if (tid >= a.n_parts || !(best > -INFINITY)) bi = 0x7fffffff, best = -INFINITY;
    block_argmax(best, bi, s_v, s_i);
    if (bi == 0x7fffffff) bi = 0;  // (no logit is a number)
    const u32x2 e = *reinterpret_cast<const u32x2*>(a.table + (size_t)bi * a.W + at);
    if (tid == 0) {
        const int n = a.count[m] + 1;  // the step's number, from 1
        a.ids[m] = bi;
        a.pos[m] += 1;
        a.count[m] = n;
        a.seen[(n % a.ahead) * a.seen_stride + m] = bi;
    }
    const f32x4 x = {bf16_lo(e.x) * a.scale, bf16_hi(e.x) * a.scale, bf16_lo(e.y) * a.scale, bf16_hi(e.y) * a.scale};
    float ss = in ? fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, x.w * x.w))) : 0.0f;
    ss = wave_allsum(ss);
    if ((tid & 63) == 0) s_red[tid >> 6] = ss;
    __syncthreads();
    const float r = 1.0f / sqrtf(((s_red[0] + s_red[1]) + (s_red[2] + s_red[3])) / (float)a.W + a.eps);
    if (!in) return;
    f32x4 h, o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = x[i] * r * (1.0f + wn[i]);
        o[i] = a.mu ? h[i] + (before[i] - h[i]) * mu[i] : h[i];
    }
    *reinterpret_cast<f32x4*>(a.x + (size_t)m * a.W + at) = x;
    *reinterpret_cast<f32x4*>(a.h + (size_t)m * a.W + at) = o;
    if (a.mu) {
        *reinterpret_cast<f32x4*>(a.shift_state + (size_t)a.row_slot[m] * a.slot_stride + at) = before;
        *reinterpret_cast<f32x4*>(a.last_h + (size_t)m * a.W + at) = h;
    }
}

// Stage 1: block (row, part) finds the maximum and its first index in its slice of the row; stage 2 (parts == 1 in the grid,
// n_parts > 0 as argument): one block per row combines the parts.  The first maximum wins; a row of NaNs gives index 0.
__global__ __launch_bounds__(256) void row_argmax_kernel(const float* logits, int n, float* max_out, int* idx_out, float* part_val, int* part_idx,
                                                         int n_parts, int combine) {
    __shared__ float s_v[4];
    __shared__ int s_i[4];
    const int row = blockIdx.x;
    float best = -INFINITY;
    int bi = 0x7fffffff;
    if (!combine) {
        const int per = (n + n_parts - 1) / n_parts, lo = blockIdx.y * per, hi = min(n, lo + per);
        const float* r = logits + (size_t)row * n;
        for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) {
            const float v = r[i];
            if (v > best) {  // ascending i per thread: the first maximum stays
                best = v;
                bi = i;
            }
        }
    } else {
        for (int i = threadIdx.x; i < n_parts; i += blockDim.x) {
            const float v = part_val[(size_t)row * n_parts + i];
            const int ix = part_idx[(size_t)row * n_parts + i];
            if (v > best || (v == best && ix < bi)) {
                best = v;
                bi = ix;
            }
        }
    }
    block_argmax(best, bi, s_v, s_i);
    if (threadIdx.x == 0) {
        const float v = best;
        int ix = bi;
        if (!combine) {
            part_val[(size_t)row * n_parts + blockIdx.y] = v;
            part_idx[(size_t)row * n_parts + blockIdx.y] = ix;
        } else {
            if (ix == 0x7fffffff) ix = 0;
            if (max_out) max_out[row] = v;
            if (idx_out) idx_out[row] = ix;
        }
    }
}

}  // namespace

int launch_embed(const bf16_t* table, const int* ids, float* x, float* x_copy, float scale, int M, int W, int vocab, int* flag, const int* row_pos,
                 const float* pos_freq, hipStream_t s) {
    if (M <= 0) return ZG_OK;
    embed_kernel<<<M, 256, 0, s>>>(table, ids, x, x_copy, scale, W, vocab, flag, pos_freq ? row_pos : nullptr, pos_freq);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_norm_shift(const float* x, const float* w, const float* mu, float eps, float* out, int M, int W, const int* row_prev,
                      const int* row_slot, const float* shift_state, size_t slot_stride, const int* row_entry_if_last, float* last_out,
                      hipStream_t s, bf16_t* out16) {
    if (M <= 0) return ZG_OK;
    NormRows r;
    r.x = x; r.wn = w; r.mu = mu; r.eps = eps; r.out = out; r.out16 = out16; r.M = M; r.W = W; r.row_prev = row_prev; r.row_slot = row_slot;
    r.shift_state = shift_state; r.slot_stride = slot_stride; r.row_entry_if_last = row_entry_if_last; r.last_out = last_out;
    bool taken = false;
    if (mu || !row_entry_if_last) ZG_TRY(launch_norm_rows(r, s, &taken));  // (without a shift it keeps no last rows)
    if (taken) return ZG_OK;
    norm_shift_kernel<<<M, 256, 0, s>>>(x, w, mu, eps, out, W, row_prev, row_slot, shift_state, slot_stride, row_entry_if_last, last_out, out16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_commit_rows(float* dst, size_t slot_stride, const float* src, size_t src_stride, const int* slots, int n_entries, int width,
                       int n_sets, size_t dst_set_stride, size_t src_set_stride, hipStream_t s) {
    if (n_entries <= 0 || n_sets <= 0) return ZG_OK;
    commit_rows_kernel<<<dim3(n_entries, n_sets), 256, 0, s>>>(dst, slot_stride, src, src_stride, slots, width, dst_set_stride, src_set_stride);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_norm_add(const float* x, float* out, const float* y, const float* w, float eps, int M, int W, hipStream_t s) {
    if (M <= 0) return ZG_OK;
    NormRows r;
    r.x = x; r.x_out = out; r.y = y; r.wb = w; r.eps = eps; r.M = M; r.W = W;
    bool taken = false;
    ZG_TRY(launch_norm_rows(r, s, &taken));
    if (taken) return ZG_OK;
    norm_add_kernel<<<M, 256, 0, s>>>(x, out, y, w, eps, W);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_copy_floats(const float* x, float* out, size_t n, hipStream_t s) {
    if (n == 0) return ZG_OK;
    copy_floats_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, out, n);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_norm_add_norm(float* x, const float* y, const float* wb, const float* wn, float eps, float* h, int M, int W, hipStream_t s, bf16_t* h16) {
    if (M <= 0) return ZG_OK;
    NormRows r;
    r.x = x; r.x_out = x; r.y = y; r.wb = wb; r.wn = wn; r.eps = eps; r.out = h; r.out16 = h16; r.M = M; r.W = W;
    bool taken = false;
    ZG_TRY(launch_norm_rows(r, s, &taken));
    if (taken) return ZG_OK;
    norm_add_norm_kernel<<<M, 256, 0, s>>>(x, y, wb, wn, eps, h, W, h16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_sum_norm_shift(float* x, const float* y, const float* yexp, const float* weight, int top, const float* wb, const float* wn, const float* mu,
                          float eps, float* out, int M, int W, const int* row_slot, const float* shift_state, size_t slot_stride,
                          const int* row_entry_if_last, float* last_out, hipStream_t s, bool* taken) {
    *taken = false;
    if (M <= 0 || W > 256 * kRowRegs) return ZG_OK;  // wider rows: the caller's separate launches
    sum_norm_shift_kernel<<<M, 256, 0, s>>>(x, y, yexp, weight, top, wb, wn, mu, eps, out, W, row_slot, shift_state, slot_stride, row_entry_if_last,
                                            last_out);
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

int launch_norm_gather(const float* x, const int* rows, const float* w, float eps, float* out, int n_rows, int W, bool plain, hipStream_t s) {
    if (n_rows <= 0) return ZG_OK;
    norm_gather_kernel<<<n_rows, 256, 0, s>>>(x, rows, w, eps, out, W, plain ? 0.0f : 1.0f);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_norm_two(float* x, const OpenSums& add, const float* wa, const float* wb, float eps, float* ha, float* hb, int M, int W, hipStream_t s, bf16_t* ha16,
                    bf16_t* hb16) {
    if (M <= 0) return ZG_OK;
    norm_two_kernel<<<M, 256, 0, s>>>(x, add, wa, wb, eps, ha, hb, W, ha16, hb16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_add_two(float* x, const OpenSums& add, int M, int W, hipStream_t s) {
    const size_t n = (size_t)M * W;
    if (n == 0 || !add.any()) return ZG_OK;
    add_two_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, add, n, W);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_tanh_norm(float* x, const float* pre, const float* nw, const int* rows, float* out, int n_rows, int W, hipStream_t s) {
    const size_t n = (size_t)n_rows * W;
    if (n == 0) return ZG_OK;
    ZG_REQUIRE((pre || nw) && (!nw || out) && !(pre && rows), ZG_ERR_ARG, "tanh norm: nothing to do, no output, or an in-place norm of gathered rows");
    const bool vec = W % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (vec) tanh_norm_kernel<4><<<(unsigned)((n / 4 + 255) / 256), 256, 0, s>>>(x, pre, nw, rows, out, n, W);
    else tanh_norm_kernel<1><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, pre, nw, rows, out, n, W);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_tanh_sum_norm(float* x, const SumParts& y, const float* nb, float mult, const float* nn, float* h, int M, int W, hipStream_t s) {
    const size_t n = (size_t)M * W;
    if (n == 0) return ZG_OK;
    ZG_REQUIRE(nb && (!nn || h) && (y.top == 0 || y.exp), ZG_ERR_ARG, "tanh norm behind a sum: no norm, no output, or no rows of the experts");
    const uintptr_t al = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(y.a) |
                         reinterpret_cast<uintptr_t>(y.exp) | reinterpret_cast<uintptr_t>(y.b);
    if (W % 4 == 0 && (al & 15) == 0) tanh_sum_norm_kernel<4><<<(unsigned)((n / 4 + 255) / 256), 256, 0, s>>>(x, y, nb, mult, nn, h, n, W);
    else tanh_sum_norm_kernel<1><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, y, nb, mult, nn, h, n, W);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_norm_plain(float* v, int ld, int rows_per_m, int width, int M, const float* w, float eps, hipStream_t s, bf16_t* out16) {
    const int n_vec = M * rows_per_m;
    if (n_vec <= 0) return ZG_OK;
    norm_plain_kernel<<<(n_vec + 3) / 4, 256, 0, s>>>(v, ld, rows_per_m, width, n_vec, w, eps, out16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_state_carry(float* state, size_t slot_stride, const int* ent_len, const int* ent_slot, int n_entries, int H, int D, int V, float* wsB,
                       const float* wsA, int a_rows, int chunk, hipStream_t s) {
    const size_t n = (size_t)H * D * V;
    if (n_entries <= 0 || n == 0) return ZG_OK;
    ZG_REQUIRE(a_rows == 1 || a_rows == D, ZG_ERR_ARG, "state carry: %d decays per head of %d rows", a_rows, D);
    // two elements a thread where rows, slots and pointers allow
    const bool two = V % 2 == 0 && slot_stride % 2 == 0 && ((reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(wsB)) & 7) == 0;
    const int per = two ? 512 : 256;
    const dim3 grid((unsigned)((n + per - 1) / per), n_entries);
    if (two) hgrn2_carry_kernel<2><<<grid, 256, 0, s>>>(state, slot_stride, ent_len, ent_slot, n_entries, H, D, V, wsB, wsA, a_rows, chunk);
    else hgrn2_carry_kernel<1><<<grid, 256, 0, s>>>(state, slot_stride, ent_len, ent_slot, n_entries, H, D, V, wsB, wsA, a_rows, chunk);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_hgrn2_scan(const float* proj, int ld, float* out, int ldo, float* state, size_t slot_stride, const int* ent_start,
                      const int* ent_len, const int* ent_slot, int n_entries, int M, int H, int D, int V, const float* bias, const float* low,
                      float* ws, size_t ws_floats, int longest, hipStream_t s, const float* decay, const GlaGate* gla, HeadNorm* norm) {
    if (n_entries <= 0) return ZG_OK;
    ZG_REQUIRE(!gla || (gla->z && gla->z_bias && !decay), ZG_ERR_ARG, "gated linear attention: its gate needs z and a bias, and no fixed decay");
    const GlaGate gg = gla ? *gla : GlaGate();
    ZG_REQUIRE(D >= 1 && D <= 16 * kScanRows, ZG_ERR_UNSUPPORTED, "hgrn2: %d key channels per head (at most %d)", D, 16 * kScanRows);
    if (decay && M > kGemvMaxRows && D <= 128 && ws && getenv("ZGPT2_LM_LINEAR_NO_CHUNKS") == nullptr) {
        // a scalar decay per head: chunks of kLinChunk tokens as matrix products (prompt portions; the test hook sends them through the scan)
        const int n_chunks = (M + kLinChunk - 1) / kLinChunk + n_entries;
        const size_t hf = (size_t)H * D * V;
        if (ws_floats >= (size_t)n_chunks * (hf + (size_t)H * D) && n_chunks <= 65535 && H <= 65535) {
            float* cB = ws;
            float* cA = ws + (size_t)n_chunks * hf;
            const dim3 grid(n_chunks, H);
            const int tiles = ((D + 31) / 32) * ((V + 31) / 32);
            linear_chunk_state_kernel<<<dim3(n_chunks, H, std::min(16, (tiles + 3) / 4)), 256, 0, s>>>(proj, ld, ent_start, ent_len, n_entries, H, D, V, decay, cB, cA);
            ZG_HIP(hipGetLastError());
            ZG_TRY(launch_state_carry(state, slot_stride, ent_len, ent_slot, n_entries, H, D, V, cB, cA, D, kLinChunk, s));
            const int dh = (D + 1) / 2;
            if (dh <= 8) linear_chunk_out_kernel<8><<<grid, 256, 0, s>>>(proj, ld, out, ldo, ent_start, ent_len, n_entries, H, D, V, decay, cB);
            else if (dh <= 16) linear_chunk_out_kernel<16><<<grid, 256, 0, s>>>(proj, ld, out, ldo, ent_start, ent_len, n_entries, H, D, V, decay, cB);
            else if (dh <= 32) linear_chunk_out_kernel<32><<<grid, 256, 0, s>>>(proj, ld, out, ldo, ent_start, ent_len, n_entries, H, D, V, decay, cB);
            else linear_chunk_out_kernel<64><<<grid, 256, 0, s>>>(proj, ld, out, ldo, ent_start, ent_len, n_entries, H, D, V, decay, cB);
            ZG_HIP(hipGetLastError());
            return ZG_OK;
        }
    }
    // Entries of more than 32 tokens: chunks as matrix products (us per layer of 6 heads of 128 x 128, everything else of the layer
    // included: one entry of 33 tokens 61.6 against 61.0 token by token, of 129 65.7 against 141, of 1023 79 against 155 in scanned
    // chunks; eight entries of 33 tokens 73 against 97).  The test hook sends them through the scan.
    if (!decay && M > kGemvMaxRows && longest > 32 && getenv("ZGPT2_LM_SCAN_NO_CHUNKS") == nullptr) {
        bool taken = false;
        ZG_TRY(launch_gated_chunks(proj, ld, out, ldo, state, slot_stride, ent_start, ent_len, ent_slot, n_entries, M, H, D, V, bias, low, ws, ws_floats, gla, s,
                                   &taken, norm));
        if (taken) return ZG_OK;
    }
    int G = 1;
    while (G * kScanRows < D) G <<= 1;
    const int Dp = G * kScanRows;
    int threads = ((V * G + 63) / 64) * 64;
    if (threads > 256) threads = 256;
    const int cols = threads / G;
    const int SB = std::max(1, std::min(kScanChunk, std::min((gla ? 2560 : 4096) / Dp, 8192 / cols)));
    const size_t lds = ((size_t)(gla ? 3 : 2) * SB * Dp + (size_t)SB * cols) * sizeof(float);
    // chunked when the step is long enough to pay for two passes, and the workspace holds every chunk's state
    const int max_chunks = (M + kScanChunk - 1) / kScanChunk + n_entries;
    const size_t head_floats = (size_t)H * D * V, need = (size_t)max_chunks * (head_floats + (size_t)H * D);
    const bool chunked = M >= 4 * kScanChunk && ws && ws_floats >= need;
    float* wsB = chunked ? ws : nullptr;
    float* wsA = chunked ? ws + (size_t)max_chunks * head_floats : nullptr;
#define ZG_SCAN_L(G_, KIND_, grid_x, mode)                                                                                                  \
    hgrn2_scan_kernel<G_, KIND_><<<dim3(grid_x, H, (V + cols - 1) / cols), threads, lds, s>>>(proj, ld, out, ldo, state, slot_stride, ent_start,    \
                                                                                               ent_len, ent_slot, n_entries, H, D, V, mode, SB, wsB, \
                                                                                               wsA, bias, low, decay, gg)
#define ZG_SCAN(G_, grid_x, mode)                         \
    do {                                                  \
        if (gla) ZG_SCAN_L(G_, SCAN_GLA, grid_x, mode);   \
        else if (decay) ZG_SCAN_L(G_, SCAN_LIN, grid_x, mode); \
        else ZG_SCAN_L(G_, SCAN_HGRN2, grid_x, mode);     \
    } while (0)
#define ZG_SCAN_G(grid_x, mode)                    \
    switch (G) {                                   \
        case 1: ZG_SCAN(1, grid_x, mode); break;   \
        case 2: ZG_SCAN(2, grid_x, mode); break;   \
        case 4: ZG_SCAN(4, grid_x, mode); break;   \
        case 8: ZG_SCAN(8, grid_x, mode); break;   \
        default: ZG_SCAN(16, grid_x, mode); break; \
    }
    if (!chunked) {
        ZG_SCAN_G(n_entries, SCAN_DIRECT);
        ZG_HIP(hipGetLastError());
        return ZG_OK;
    }
    ZG_SCAN_G(max_chunks, SCAN_A);
    ZG_HIP(hipGetLastError());
    ZG_TRY(launch_state_carry(state, slot_stride, ent_len, ent_slot, n_entries, H, D, V, wsB, wsA, D, kScanChunk, s));
    ZG_SCAN_G(max_chunks, SCAN_C);
    ZG_HIP(hipGetLastError());
#undef ZG_SCAN_G
#undef ZG_SCAN
#undef ZG_SCAN_L
    return ZG_OK;
}

int launch_latent_prep(const float* proj, int ld, int M, int q_rank, int KR, int R, const float* wq, const float* wkv, float eps, Rotary rot,
                       const int* row_pos, const int* row_slot, const int* page_table, int max_pages, int page_tokens, float* cq,
                       float* cache, hipStream_t s, bf16_t* cq16) {
    if (M <= 0) return ZG_OK;
    ZG_REQUIRE(rot.dims % 2 == 0 && rot.dims <= R, ZG_ERR_ARG, "rotary: %d rotated dimensions of a part of %d", rot.dims, R);
    latent_prep_kernel<<<M, 256, 0, s>>>(proj, ld, q_rank, KR, R, wq, wkv, eps, rot, row_pos, row_slot, page_table, max_pages, page_tokens, cq,
                                         cache, cq16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_latent_direct_prep(const float* proj, int ld, int M, int H, int D, int R, int KR, int kv_col, const float* wkv, float eps, Rotary rot,
                              const int* row_pos, const int* row_slot, const int* page_table, int max_pages, int page_tokens, float* qa, float* cache,
                              hipStream_t s, bf16_t* qa16) {
    if (M <= 0) return ZG_OK;
    ZG_REQUIRE(rot.dims % 2 == 0 && rot.dims <= R, ZG_ERR_ARG, "rotary: %d rotated dimensions of a part of %d", rot.dims, R);
    const int parts = (qa || qa16 ? 1 : 0) + (cache ? 1 : 0);
    if (parts == 0) return ZG_OK;
    latent_direct_prep_kernel<<<dim3(M, parts), 256, 0, s>>>(proj, ld, H, D, R, KR, kv_col, wkv, eps, rot, row_pos, row_slot, page_table, max_pages,
                                                                     page_tokens, qa, cache, qa16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_q_rotary(const float* q, int ldq, float* qa, int ldqa, int M, int H, int D, int R, int KR, Rotary rot, const int* row_pos,
                    hipStream_t s, bf16_t* qa16) {
    if (M <= 0 || R <= 0) return ZG_OK;
    q_rotary_kernel<<<M, 256, 0, s>>>(q, ldq, qa, ldqa, H, D, R, KR, rot, row_pos, qa16);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

size_t latent_tile_elems(int KR, int R) {  // elements of a key tile in the launch's workspace, 0: the latent is larger than its tiles hold
    const int DT = KR + R;
    if (DT <= 96 && KR <= 64) return KeyTile<6>::BYTES / 2;
    if (DT <= 160 && KR <= 128) return KeyTile<10>::BYTES / 2;
    if (DT <= 288 && KR <= 256) return KeyTile<18>::BYTES / 2;
    if (DT <= 384 && KR <= 320) return KeyTile<24>::BYTES / 2;
    return 0;
}

int launch_latent_attention_tiles(const float* qa, float* ctx, int M, int H, int KR, int R, float scale, const int* ent_start, const int* ent_len,
                                  const int* ent_slot, int n_entries, const int* row_pos, const int* page_table, int max_pages, int page_tokens,
                                  const float* cache, bf16_t* ws, size_t ws_elems, size_t n_tiles, int max_keys, hipStream_t s, bool* taken,
                                  const float* gate, int ldg, const float* sink, const bf16_t* qa16, bf16_t* ctx16) {
    *taken = false;
    if (M <= 0 || n_entries <= 0) return ZG_OK;
    const size_t tile = latent_tile_elems(KR, R);
    if (tile == 0 || !ws || n_tiles * tile > ws_elems || n_entries > 65535) return ZG_OK;  // the caller's general kernel
    const dim3 cgrid((max_keys + 31) / 32, n_entries), grid((M + 31) / 32 + n_entries, (H + 3) / 4);
#define ZG_ATT_T(NKS_, NT_)                                                                                                                          \
    do {                                                                                                                                             \
        latent_tiles_kernel<NKS_><<<cgrid, 256, 0, s>>>(cache, KR + R, KR, ent_start, ent_len, ent_slot, n_entries, row_pos, page_table, max_pages,      \
                                                        page_tokens, ws);                                                                            \
        ZG_HIP(hipGetLastError());                                                                                                                   \
        latent_attention_mfma_kernel<NKS_, NT_><<<grid, 256, 0, s>>>(qa, qa16, ctx, ctx16, H, KR, R, scale, ent_start, ent_len, ent_slot, n_entries, row_pos, ws, gate, ldg, \
                                                                     sink);                                                                          \
    } while (0)
    if (tile == KeyTile<6>::BYTES / 2) ZG_ATT_T(6, 2);
    else if (tile == KeyTile<10>::BYTES / 2) ZG_ATT_T(10, 4);
    else if (tile == KeyTile<18>::BYTES / 2) ZG_ATT_T(18, 8);
    else ZG_ATT_T(24, 10);
#undef ZG_ATT_T
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

// Prompt portions in 32-bit mode.  (The general kernel stays for latents beyond the tiles and rows that are no whole 16-byte pieces.)
int launch_latent_attention_f32(const float* qa, float* ctx, int M, int H, int KR, int R, float scale, const int* ent_start, const int* ent_len,
                                const int* ent_slot, int n_entries, const int* row_pos, const int* page_table, int max_pages, int page_tokens,
                                const float* cache, hipStream_t s, bool* taken, const float* gate, int ldg, const float* sink) {
    *taken = false;
    const size_t tile = latent_tile_elems(KR, R);
    if (M <= 0 || n_entries <= 0 || tile == 0 || KR % 4 != 0 || R % 4 != 0 || H > 65535 ||
        ((reinterpret_cast<uintptr_t>(qa) | reinterpret_cast<uintptr_t>(ctx) | reinterpret_cast<uintptr_t>(cache)) & 15) != 0)
        return ZG_OK;
    const dim3 grid((M + 15) / 16 + n_entries, H);
#define ZG_ATT_FX(NKS_, NV_, EXACT_)                                                                                                           \
    latent_attention_f32_kernel<NKS_, NV_, EXACT_><<<grid, 256, 0, s>>>(qa, ctx, H, KR, R, scale, ent_start, ent_len, ent_slot, n_entries, row_pos, \
                                                                        page_table, max_pages, page_tokens, cache, gate, ldg, sink)
#define ZG_ATT_F(NKS_, NV_)                                                             \
    if (KR + R == 16 * NKS_ && KR == 64 * NV_) ZG_ATT_FX(NKS_, NV_, true);              \
    else ZG_ATT_FX(NKS_, NV_, false)
    if (tile == KeyTile<6>::BYTES / 2) { ZG_ATT_F(6, 1); }
    else if (tile == KeyTile<10>::BYTES / 2) { ZG_ATT_F(10, 2); }
    else if (tile == KeyTile<18>::BYTES / 2) { ZG_ATT_F(18, 4); }
    else { ZG_ATT_F(24, 5); }
#undef ZG_ATT_F
#undef ZG_ATT_FX
    ZG_HIP(hipGetLastError());
    *taken = true;
    return ZG_OK;
}

int launch_latent_attention(const float* qa, float* ctx, int M, int H, int KR, int R, float scale, const int* row_pos, const int* row_slot,
                            const int* page_table, int max_pages, int page_tokens, const float* cache, float* ws, size_t ws_floats,
                            hipStream_t s, const float* gate, int ldg, const float* sink) {
    if (M <= 0) return ZG_OK;
    const int nd = (KR + R + 63) / 64;
    ZG_REQUIRE(nd <= 16, ZG_ERR_UNSUPPORTED, "latent attention: %d cached dimensions per token (at most 1024)", KR + R);
    // decode steps: the keys of a row in up to kAttnSplits ranges (a fixed grid, so that a captured step can be replayed at any
    // sequence length; ranges beyond the row's keys leave empty partials)
    int n_split = 1;
    if (M <= kGemvMaxRows && ws && ws_floats >= (size_t)M * H * kAttnSplits * (KR + 2) && (long long)max_pages * page_tokens > 128) n_split = kAttnSplits;
    const dim3 grid(M, H, n_split);
#define ZG_ATT(ND_)                                                                                                                           \
    latent_attention_kernel<ND_><<<grid, 256, 0, s>>>(qa, ctx, H, KR, R, scale, row_pos, row_slot, page_table, max_pages, page_tokens, cache, ws, \
                                                      n_split, gate, ldg, sink)
    if (nd <= 1) ZG_ATT(1);
    else if (nd <= 2) ZG_ATT(2);
    else if (nd <= 3) ZG_ATT(3);
    else if (nd <= 4) ZG_ATT(4);
    else if (nd <= 5) ZG_ATT(5);
    else if (nd <= 6) ZG_ATT(6);
    else if (nd <= 9) ZG_ATT(9);
    else if (nd <= 12) ZG_ATT(12);
    else ZG_ATT(16);
#undef ZG_ATT
    ZG_HIP(hipGetLastError());
    if (n_split > 1) {
        latent_merge_kernel<<<dim3(M, H), 256, 0, s>>>(ws, ctx, H, KR, n_split, row_pos, gate, ldg, sink);
        ZG_HIP(hipGetLastError());
    }
    return ZG_OK;
}

int launch_advance_rows(const int* tok, int M, int* ids, int* pos, int* seen, hipStream_t s) {
    if (M <= 0) return ZG_OK;
    advance_rows_kernel<<<(M + 63) / 64, 64, 0, s>>>(tok, M, ids, pos, seen);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_new_pages(int* table, const NewPages& pages, hipStream_t s) {
    if (pages.n <= 0) return ZG_OK;
    ZG_REQUIRE(pages.n <= kGemvMaxRows, ZG_ERR_ARG, "new pages: %d at a time", pages.n);
    new_pages_kernel<<<1, 64, 0, s>>>(table, pages);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_argmax_parts(const float* logits, int rows, int n, float* part_val, int* part_idx, int* n_parts, hipStream_t s) {
    *n_parts = std::max(1, std::min(kArgmaxParts, (n + 1023) / 1024));
    if (rows <= 0) return ZG_OK;
    row_argmax_kernel<<<dim3(rows, *n_parts), 256, 0, s>>>(logits, n, nullptr, nullptr, part_val, part_idx, *n_parts, 0);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_next_token(const NextToken& a, int M, hipStream_t s) {
    if (M <= 0) return ZG_OK;
    ZG_REQUIRE(a.W >= 4 && a.W <= 1024 && a.W % 4 == 0 && a.n_parts >= 1 && a.n_parts <= 256 && a.ahead >= 1, ZG_ERR_ARG, "next token: rows of %d, %d parts", a.W, a.n_parts);
    next_token_kernel<<<M, 256, 0, s>>>(a);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int launch_row_argmax(const float* logits, int rows, int n, float* max_out, int* idx_out, float* part_val, int* part_idx, hipStream_t s) {
    if (rows <= 0) return ZG_OK;
    const int parts = std::max(1, std::min(kArgmaxParts, (n + 1023) / 1024));
    row_argmax_kernel<<<dim3(rows, parts), 256, 0, s>>>(logits, n, nullptr, nullptr, part_val, part_idx, parts, 0);
    ZG_HIP(hipGetLastError());
    row_argmax_kernel<<<dim3(rows, 1), 256, 0, s>>>(logits, n, max_out, idx_out, part_val, part_idx, parts, 1);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
