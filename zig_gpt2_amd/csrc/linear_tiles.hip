// linear_tiles.hip — fp32 Linears of nine rows to some thousand (y = x W^T + bias, src/ops.zig:21-46) in one pass over both operands, and of
// two to fifteen rows (linear_few_kernel and linear_few_mfma_kernel, below).
//
// Both operands are split exactly into three bf16 terms on their way into the LDS (x = hi + mid + lo) and the six products above 2^-24 of
// the leading one are summed, as the persistent kernel for many rows does (gemm_s4.hip); here no planes are written to memory first, and
// the tiles are small enough to use the whole chip: 64 x 64, and K in slices over grid.z while there are too few of them (each slice leaves
// a slab, linear_slabs_kernel adds them).  The leading products have sums of their own, so that the small ones are not rounded at their size.
#include "prefill_epi.h"
#include "zg_kernels.h"

#include <algorithm>
#include <atomic>

namespace zg {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kBk = 32, kChunks = kBk / 8;  // columns of K a step stages, 16-byte pieces of a row of them
constexpr int kAheadSteps = 3;

// rows of 32 bf16 (64 bytes): pieces swizzled by the row, so that a fragment read of eight rows touches every bank once
__device__ __forceinline__ int lds_at(int row, int piece) { return row * kBk + ((piece ^ ((row >> 1) & 3)) * 8); }

struct Terms {
    u32x4 v[3];  // hi, mid, lo of eight values
};
__device__ __forceinline__ Terms split8(const f32x4& a, const f32x4& b) {
    Terms t;
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        split3_pk(x[2 * i], x[2 * i + 1], h, m, l);
        t.v[0][i] = h;
        t.v[1][i] = m;
        t.v[2][i] = l;
    }
    return t;
}

// What bounds it: the LDS, which takes 24 KB of terms and gives 48 KB of fragments a step, beside 384 cycles of products.
__global__ __launch_bounds__(256, 2) void linear_tiles_kernel(const float* __restrict__ X, const float* __restrict__ W, const float* __restrict__ bias,
                                                              float* __restrict__ Y, int M, int N, int K, int steps) {
    __shared__ __attribute__((aligned(16))) bf16_t As[2][3][64 * kBk];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[2][3][64 * kBk];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wy = wave >> 1, wx = wave & 1;
    // consecutive workgroups go to the eight XCDs in turn: each gets a contiguous run of the tiles, row tiles of one column tile together
    const int tiles_m = (M + 63) / 64, total = gridDim.x, q = total >> 3, r8 = total & 7, xcd = blockIdx.x & 7;
    const int at = xcd * q + min(xcd, r8) + (int)(blockIdx.x >> 3);
    const int m0 = (at % tiles_m) * 64, n0 = (at / tiles_m) * 64;
    const int k_first = blockIdx.z * steps * kBk;
    steps = min(steps, (K - k_first) / kBk);

    const int row = tid / kChunks, piece = tid % kChunks, to = lds_at(row, piece);
    const float* x = X + (size_t)min(m0 + row, M - 1) * K + k_first + piece * 8;  // (rows beyond the edge: some valid row, never stored)
    const float* w = W + (size_t)min(n0 + row, N - 1) * K + k_first + piece * 8;
    f32x4 xr[kAheadSteps][2], wr[kAheadSteps][2];
    auto fetch = [&](int slot, int s) {
        const int k = min(s, steps - 1) * kBk;  // (beyond the last step: fetched again, not used)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            xr[slot][i] = *reinterpret_cast<const f32x4*>(x + k + 4 * i);
            wr[slot][i] = *reinterpret_cast<const f32x4*>(w + k + 4 * i);
        }
    };
    auto stash = [&](int slot, int buf) {
        const Terms a = split8(xr[slot][0], xr[slot][1]), b = split8(wr[slot][0], wr[slot][1]);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            *reinterpret_cast<u32x4*>(&As[buf][t][to]) = a.v[t];
            *reinterpret_cast<u32x4*>(&Bs[buf][t][to]) = b.v[t];
        }
    };
    f32x16 lead, small;
#pragma unroll
    for (int e = 0; e < 16; ++e) lead[e] = small[e] = 0.0f;
    const int fr = lane & 31, kh = lane >> 5;
    bf16x8 af[2][3], bf[2][3];
    auto read = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                af[kk][t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&As[buf][t][lds_at(wy * 32 + fr, 2 * kk + kh)]));
                bf[kk][t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&Bs[buf][t][lds_at(wx * 32 + fr, 2 * kk + kh)]));
            }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][2], bf[kk][0], small, 0, 0, 0);
            lead = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][0], bf[kk][0], lead, 0, 0, 0);
            small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][1], bf[kk][1], small, 0, 0, 0);
            small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][0], bf[kk][2], small, 0, 0, 0);
            small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][1], bf[kk][0], small, 0, 0, 0);
            small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][0], bf[kk][1], small, 0, 0, 0);
        }
    };
#pragma unroll
    for (int i = 0; i < kAheadSteps; ++i) fetch(i, i);
    stash(0, 0);
    fetch(0, kAheadSteps);
    __syncthreads();
    int buf = 0;
    for (int s0 = 0; s0 < steps; s0 += kAheadSteps) {
#pragma unroll
        for (int i = 0; i < kAheadSteps; ++i) {
            if (s0 + i < steps) {  // (uniform)
                const int nx = (i + 1) % kAheadSteps;
                read(buf);
                stash(nx, buf ^ 1);
                fetch(nx, s0 + i + 1 + kAheadSteps);
                multiply();
                buf ^= 1;
                __syncthreads();
            }
        }
    }
    // element e of the wave's 32 x 32: row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
    float* y = Y + (gridDim.z > 1 ? (size_t)blockIdx.z * M * N : 0);
    const int n = n0 + wx * 32 + fr;
    if (n >= N) return;
    const float b = bias != nullptr && gridDim.z == 1 ? bias[n] : 0.0f;
    float worst = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int m = m0 + wy * 32 + 8 * (e >> 2) + 4 * kh + (e & 3);
        const float v = lead[e] + (small[e] + b);
        worst = fmaxf(worst, odd(v));
        if (m < M) y[(size_t)m * N + n] = v;
    }
    if (__builtin_expect(worst != 0.0f, 0) && gridDim.z == 1)  // (slabs: where they meet)
#pragma unroll 1
        for (int e = 0; e < 16; ++e) {
            const int m = m0 + wy * 32 + 8 * (e >> 2) + 4 * kh + (e & 3);
            if (m < M && odd(y[(size_t)m * N + n]) != 0.0f) y[(size_t)m * N + n] = plain_sum(X + (size_t)m * K, W + (size_t)n * K, K) + b;
        }
}

__global__ __launch_bounds__(256) void linear_slabs_kernel(const float* __restrict__ slabs, int n_slabs, const float* __restrict__ bias, float* __restrict__ Y,
                                                           size_t n, int N, const float* __restrict__ X, const float* __restrict__ W, int K) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int here = (int)min((size_t)4, n - i);
    if (here == 4 && n % 4 == 0) {
        for (int s = 0; s < n_slabs; ++s) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(slabs + s * n + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += t[e];
        }
    } else {
        for (int s = 0; s < n_slabs; ++s)
            for (int e = 0; e < here; ++e) v[e] += slabs[s * n + i + e];
    }
    float worst = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        worst = fmaxf(worst, odd(v[e]));
        if (e < here) Y[i + e] = v[e] + (bias ? bias[(i + e) % N] : 0.0f);
    }
    if (__builtin_expect(worst != 0.0f, 0))
#pragma unroll 1
        for (int e = 0; e < here; ++e) {
            const size_t m = (i + e) / N, c = (i + e) % N;
            if (odd(Y[i + e]) != 0.0f) Y[i + e] = plain_sum(X + m * K, W + c * K, K) + (bias ? bias[c] : 0.0f);
        }
}

constexpr int kLongRow = 1536;

// Two to eight rows: a wave multiplies R weight rows with all of them, two pieces of 512 columns in flight; long rows (SPLIT) are cut over the
// four waves of a workgroup.  Everything is loaded at clamped addresses without a condition, and the workgroups are small enough for
// every compute unit to have one.  A call, us, this against the general kernel: 8 rows 768 -> 3072 15.4 : 20.0, 6400 -> 1600 26 : 32, 2 rows
// 768 -> 50257 32 : 47, 1600 -> 4800 17.0 : 22.8.
template <int MR, int R, bool SPLIT>
__global__ __launch_bounds__(256) void linear_few_kernel(const float* __restrict__ X, const float* __restrict__ W, const float* __restrict__ bias,
                                                         float* __restrict__ Y, int M, int N, int K) {
    __shared__ float s_part[SPLIT ? 4 : 1][MR * R];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = SPLIT ? blockIdx.x * R : (blockIdx.x * 4 + wave) * R;
    if (n0 >= N) return;
    const int kq = SPLIT ? (((K + 3) / 4) + 7) & ~7 : K, k_lo = SPLIT ? wave * kq : 0, k_hi = SPLIT ? min(K, k_lo + kq) : K;
    f32x4 xr[2][MR][2], wr[2][R][2];
    auto fetch = [&](int slot, int k0) {
        const int k = min(k0 + lane * 8, K - 8);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int r = 0; r < R; ++r) wr[slot][r][i] = *reinterpret_cast<const f32x4*>(W + (size_t)min(n0 + r, N - 1) * K + k + 4 * i);
#pragma unroll
            for (int m = 0; m < MR; ++m) xr[slot][m][i] = *reinterpret_cast<const f32x4*>(X + (size_t)min(m, M - 1) * K + k + 4 * i);
        }
    };
    float sum[MR][R];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) sum[m][r] = 0.0f;
    auto add = [&](int slot, int k0) {
        if (k0 + lane * 8 >= k_hi) return;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[m][r] = fmaf(xr[slot][m][i][e], wr[slot][r][i][e], sum[m][r]);
    };
    fetch(0, k_lo);
    fetch(1, k_lo + 512);
    for (int k0 = k_lo; k0 < k_hi; k0 += 1024) {
        add(0, k0);
        fetch(0, k0 + 1024);
        add(1, k0 + 512);
        fetch(1, k0 + 1536);
    }
    float mine = 0.0f;  // lane m R + r: the sum of row m, weight row n0 + r
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float v = wave_allsum(sum[m][r]);
            mine = lane == m * R + r ? v : mine;
        }
    if constexpr (SPLIT) {
        if (lane < MR * R) s_part[wave][lane] = mine;
        __syncthreads();
        if (wave != 0 || lane >= MR * R) return;
        mine = (s_part[0][lane] + s_part[1][lane]) + (s_part[2][lane] + s_part[3][lane]);
    }
    const int m = lane / R, n = n0 + lane % R;
    if (lane < MR * R && m < M && n < N) Y[(size_t)m * N + n] = mine + (bias ? bias[n] : 0.0f);
}

// Five to fifteen rows: a workgroup multiplies sixteen weight rows with all of them, its waves pieces of 32 columns in turn, by the matrix
// cores' fp32 products: a weight and an activation are loaded once a workgroup and nothing is summed over lanes.  RING pieces of a wave in
// flight, at clamped addresses without a condition.  Eight sums a lane keep the chains of additions short and meet in 64 bits: against 64 bits
// the outputs are as near as those of the kernels it took over from, or nearer (rms of 768 columns 5.8e-8 of the outputs' own, 8.2e-8 and 7.2e-8
// there; with 32-bit sums 8.0e-8).
// What bounds it: latency, the launch and one round of loads, and where a workgroup has many pieces the intake of its compute unit.  A call, us,
// repeated on the same buffers, those kernels -> this one: 8 rows 768 -> 3072 15.2 -> 13.8 (on new buffers every call 15.0 -> 14.4), 768 -> 50257 55 -> 46,
// 1600 -> 6400 28.2 -> 23.8, 12 rows 768 -> 768 18.8 -> 14.3, 520 -> 600 25.8 -> 13.1, 768 -> 50257 57 -> 49.
template <int RING>
__global__ __launch_bounds__(512) void linear_few_mfma_kernel(const float* __restrict__ X, const float* __restrict__ W, const float* __restrict__ bias,
                                                                    float* __restrict__ Y, int M, int N, int K) {
    constexpr int kWaves = 8;
    __shared__ double s_part[kWaves][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = lane & 15, n0 = blockIdx.x * 16;
    const int on = n0 + (tid & 15), om = tid >> 4;  // the output a thread ends with
    const float b = bias != nullptr ? bias[min(on, N - 1)] : 0.0f;
    const float* const w = W + (size_t)min(n0 + row, N - 1) * K;
    const float* const x = X + (size_t)min(row, M - 1) * K;
    const int k_lane = wave * 32 + (lane >> 4) * 8;
    f32x4 wr[RING][2], xr[RING][2];
    auto fetch = [&](int slot, int p) {
        const int k = min(k_lane + p * kWaves * 32, K - 8);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            wr[slot][i] = *reinterpret_cast<const f32x4*>(w + k + 4 * i);
            xr[slot][i] = *reinterpret_cast<const f32x4*>(x + k + 4 * i);
        }
    };
    f32x4 acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int slot, int p) {
        const bool in = k_lane + p * kWaves * 32 < K;  // (K is whole eights)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? wr[slot][i >> 2][i & 3] : 0.0f, in ? xr[slot][i >> 2][i & 3] : 0.0f, acc[i], 0, 0, 0);
    };
    const int mine = ((K + 31) / 32 - wave + kWaves - 1) / kWaves;  // pieces of this wave
#pragma unroll
    for (int i = 0; i < RING; ++i) fetch(i, i);
    int p = 0;
    for (; p + RING < mine; p += RING) {
#pragma unroll
        for (int i = 0; i < RING; ++i) {
            multiply(i, p + i);
            fetch(i, p + i + RING);
        }
    }
#pragma unroll
    for (int i = 0; i < RING; ++i) multiply(i, p + i);  // (pieces beyond K: zeros)
#pragma unroll
    for (int e = 0; e < 4; ++e)
        s_part[wave][e][lane] = (((double)acc[0][e] + acc[1][e]) + ((double)acc[2][e] + acc[3][e])) + (((double)acc[4][e] + acc[5][e]) + ((double)acc[6][e] + acc[7][e]));
    __syncthreads();
    if (tid >= 256 || on >= N || om >= M) return;
    // element e of a lane's four: weight row 4 (lane / 16) + e, row of X lane % 16
    const int at = ((tid & 15) >> 2) * 16 + om, e = tid & 3;
    double v[kWaves];
#pragma unroll
    for (int i = 0; i < kWaves; ++i) v[i] = s_part[i][e][at];
    Y[(size_t)om * N + on] = (float)((((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]))) + b);
}

// The outputs of marked rows of X and of W again: every wave looks through the marks and takes its share of a marked row's outputs, a dot product at a time (one
// row of 8192 x 768 x 3072: 20 us, half of it the look through the marks).
constexpr int kMarkedGroups = 512;
__global__ __launch_bounds__(256) void linear_marked_rows_kernel(const float* __restrict__ X, const float* __restrict__ W, const float* __restrict__ bias, float* __restrict__ Y,
                                                                 int M, int N, int K, const SplitSeen seen) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)), all = M + N;
    const SeenPlan p = seen_plan(seen);
    auto redo = [&](int at) {
        const bool of_w = at >= M;
        const int row = of_w ? at - M : at;
        const float* mine = (of_w ? W : X) + (size_t)row * K;
        for (int o = wave; o < (of_w ? M : N); o += 4 * kMarkedGroups) {
            const float* other = (of_w ? X : W) + (size_t)o * K;
            float s = 0.0f;
            for (int k = 4 * lane; k < K; k += 256) {
                const f32x4 a = *reinterpret_cast<const f32x4*>(mine + k), b = *reinterpret_cast<const f32x4*>(other + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) s = fmaf(a[e], b[e], s);
            }
            s = wave_allsum(s);
            const int m = of_w ? o : row, n = of_w ? row : o;
            if (lane == 0) Y[(size_t)m * N + n] = s + (bias ? bias[n] : 0.0f);
        }
    };
    for (int base = 0; base < all; base += 1024) {
        i32x4 mark[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) mark[u] = reinterpret_cast<const i32x4*>(seen.marks)[min(base / 4 + 64 * u + lane, (all - 1) / 4)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int first = base + 256 * u + e, at = first + 4 * lane;
                unsigned long long some = __ballot(at < all && (mark[u][e] & (MARK_ODD | (at >= M ? p.w : p.x))) != 0);
                for (; some != 0; some &= some - 1) redo(first + 4 * __builtin_ctzll(some));
            }
    }
}

}  // namespace

bool linear_tiles_pay(size_t M, size_t N, size_t K, bool planes) {
    // Against the persistent kernel behind its splitting pass, whose time goes by rounds of 256 tiles of 256 x 192 whether they are full or not.
    // From 640 columns on that kernel takes three products of fp16 terms (us of a call, this : that): 768 -> 3072 1023 rows (768 tiles)
    // 50 : 66, 1300 (1008) 62 : 67, 1500 (1152) 69 : 67, 2048 (1536) 83 : 68; 768 -> 1031 4096 rows (1088) 70 : 68; 1600 -> 1600 1500 rows (600) 80 : 101,
    // 2048 (800) 107 : 101; 6400 -> 1600 1500 rows (600) 278 : 337, 2048 (800) 384 : 342; 3072 -> 768 4096 rows (768) 161 : 185, 6000 (1128) 240 : 192.
    // Below, and for rows that are not for two terms, six of bf16: 128 -> 3072 1856 rows (1392 tiles) and more.
    const size_t tiles = ((M + 63) / 64) * ((N + 63) / 64), rounds = (((M + 255) / 256) * ((N + 191) / 192) + 255) / 256;
    // Where the splitting pass leaves the last level's cache it is priced as well: 6400 -> 9601 420 rows 440 : 469, 512 458 : 486 (predicted 453 : 499 and 453 : 504).
    if (tiles <= (!planes || K < kSplit2MinK ? 1400 : K < 1024 ? 1100 : 800) * rounds) return true;
    return planes && K >= kSplit2MinK && linear_split_mb(M, N, K) > 240.0 && linear_tiles_us(M, N, K) < (double)rounds * (3.2 * (double)(K / 64) + 10.0) + linear_split_us(M, N, K);
}

// 13 us, 0.44 a step of 32 columns of the compute unit with the most tiles, and the slabs (within 5 % over 40 to 1200 rows of 14 shapes of 1536 to 8192 columns)
double linear_tiles_us(size_t M, size_t N, size_t K) {
    const size_t slices = linear_tiles_slices(M, N, K), steps = (K / kBk + slices - 1) / slices, tiles = ((M + 63) / 64) * ((N + 63) / 64) * slices;
    return 13.0 + 0.44 * (double)((tiles + 255) / 256 * steps) + (slices > 1 ? 2e-6 * (double)slices * (double)M * (double)N : 0.0);
}

// The pass that splits both operands in two terms, and the launches: 4 bytes read and 4 written a value, dearer where they leave the last level's cache
double linear_split_mb(size_t M, size_t N, size_t K) { return (double)(M + N) * (double)K * 8e-6; }
double linear_split_us(size_t M, size_t N, size_t K) {
    const double mb = linear_split_mb(M, N, K);
    return 9.0 + 0.144 * mb + 0.257 * std::max(0.0, mb - 240.0) + 0.0027 * (double)K;
}

int launch_linear_marked_rows(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, const SplitSeen& seen, hipStream_t s) {
    ZG_REQUIRE(M > 0 && N > 0 && M < (1 << 30) && N < (1 << 30) && K > 0 && K % 4 == 0, ZG_ERR_ARG, "linear: %d x %d x %d", M, N, K);
    linear_marked_rows_kernel<<<kMarkedGroups, 256, 0, s>>>(X, W, bias, Y, M, N, K, seen);
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

int linear_tiles_slices(size_t M, size_t N, size_t K) {
    // two workgroups a compute unit, slices of at least four steps
    const size_t tiles = ((M + 63) / 64) * ((N + 63) / 64), steps = K / kBk;
    size_t s = std::min<size_t>({(512 + tiles - 1) / tiles, steps / 4, 16});
    s = std::max<size_t>(1, s);
    const size_t per = (steps + s - 1) / s;
    return (int)((steps + per - 1) / per);  // (none is empty)
}

int launch_linear_tiles(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, float* slabs, hipStream_t s) {
    ZG_REQUIRE(M > 0 && N > 0 && K > 0 && K % kBk == 0, ZG_ERR_UNSUPPORTED, "linear tiles: M=%d N=%d K=%d", M, N, K);
    const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64);
    ZG_REQUIRE(tiles < (1LL << 31) - 8, ZG_ERR_UNSUPPORTED, "linear tiles: %d x %d outputs exceed the grid", M, N);
    const int slices = linear_tiles_slices(M, N, K), steps = (K / kBk + slices - 1) / slices;
    ZG_REQUIRE(slices == 1 || slabs != nullptr, ZG_ERR_ARG, "linear tiles: %d slices and no room for their slabs", slices);
    linear_tiles_kernel<<<dim3((unsigned)tiles, 1, slices), 256, 0, s>>>(X, W, bias, slices > 1 ? slabs : Y, M, N, K, steps);
    ZG_HIP(hipGetLastError());
    if (slices > 1) {
        const size_t n = (size_t)M * N;
        linear_slabs_kernel<<<(unsigned)((n + 1023) / 1024), 256, 0, s>>>(slabs, slices, bias, Y, n, N, X, W, K);
        ZG_HIP(hipGetLastError());
    }
    note_kernel("linear_tiles_kernel");
    return ZG_OK;
}

static std::atomic<unsigned long long> g_few_mfma_launches{0};
unsigned long long linear_few_mfma_launch_count() { return g_few_mfma_launches.load(std::memory_order_relaxed); }

// linear_few_mfma_kernel, or linear_few_kernel and the tiles; a call's us on the same buffers, this : those.  Nine rows to fifteen (12 rows 768 -> 768 14.3 : 18.8,
// 768 -> 3072 14.3 : 20.6, 1600 -> 1600 18.4 : 20.7; K in no whole 64s, as 520 -> 600, 13.1 : 25.8): the tiles, which have sixteen rows and more,
// catch up where long rows make a compute unit's share long (16 rows 1600 -> 4800 25.0 : 24.0, 3072 -> 768 21.4 : 22.4, 6400 -> 1600 35.5 : 30.7);
// rows shorter than their 128 columns stay on the general kernels.  Five to eight: linear_few_kernel has more workgroups and is ahead until they
// are more than the compute units (8 rows 768 -> 768 13.0 : 12.8, 1024 -> 1024 13.7 : 12.9, 768 -> 2304 13.7 : 15.4; its long rows 1536 -> 384
// 16.6 : 14.3, 1600 -> 1600 17.5 : 19.3, 3072 -> 1031 19.4 : 18.9; between them 1528 -> 2000 16.9 : 14.7); short rows are ahead at once here
// (384 -> 384 12.7 : 13.2).
static bool few_on_mfma(size_t M, size_t N, size_t K) {
    if (M > 15) return false;
    if (M > 8) return K >= 128 && (K <= 1024 || (K <= 1792 && N <= 4096));
    if (M < 5 || (K < 256 && N > 6144)) return false;  // (so short and so many: still the general kernel, by linear_few_ok)
    return K <= 512 || (K <= 1024 && N > 2048) || (K >= kLongRow && K <= 1792 && N > 1024);
}

bool linear_few_ok(size_t M, size_t N, size_t K) {
    if (K < 64 || K > 8192 || K % 8 != 0 || N >= (1u << 30)) return false;
    if (few_on_mfma(M, N, K)) return true;
    // Beyond four rows every workgroup's share of the activations outweighs its weights: with more than some three workgroups a compute unit
    // the general kernel, which reads them less often, is faster (6400 -> 1600, 400 of them, 26 : 32; 1200 of 1600 columns 32.9 : 27.9).
    const size_t groups = K >= kLongRow ? (N + 3) / 4 : (N + 7) / 8;
    // One row stays on the general kernels: a generation through op-tier calls with host buffers measured 782 tokens/s with it here, 819 there.
    return M >= 2 && M <= 8 && (M <= 4 || groups <= 768);
}

int launch_linear_few(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, hipStream_t s) {
    ZG_REQUIRE(M >= 1 && M <= 15 && N > 0 && K >= 8 && K % 8 == 0, ZG_ERR_UNSUPPORTED, "linear: M=%d N=%d K=%d", M, N, K);
    if (few_on_mfma(M, N, K)) {
        const int each = (K + 255) / 256;  // pieces of a wave
#define ZG_FEW(RING) linear_few_mfma_kernel<RING><<<(N + 15) / 16, 512, 0, s>>>(X, W, bias, Y, M, N, K)
        if (each == 1) ZG_FEW(1);
        else if (each == 2) ZG_FEW(2);
        else if (each == 3) ZG_FEW(3);
        else ZG_FEW(4);
#undef ZG_FEW
        note_kernel("linear_few_kernel");  // (the two have one name; the count says which)
        g_few_mfma_launches.fetch_add(1, std::memory_order_relaxed);
        ZG_HIP(hipGetLastError());
        return ZG_OK;
    }
    ZG_REQUIRE(M <= 8, ZG_ERR_UNSUPPORTED, "linear: M=%d N=%d K=%d", M, N, K);
    const bool split = K >= kLongRow;
#define ZG_FEW(MR)                                                                                             \
    do {                                                                                                       \
        if (split) linear_few_kernel<MR, 4, true><<<(N + 3) / 4, 256, 0, s>>>(X, W, bias, Y, M, N, K);         \
        else linear_few_kernel<MR, 2, false><<<(N + 7) / 8, 256, 0, s>>>(X, W, bias, Y, M, N, K);              \
    } while (0)
    if (M <= 2) ZG_FEW(2);
    else if (M <= 4) ZG_FEW(4);
    else ZG_FEW(8);
#undef ZG_FEW
    note_kernel("linear_few_kernel");
    ZG_HIP(hipGetLastError());
    return ZG_OK;
}

}  // namespace zg
