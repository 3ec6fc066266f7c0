// lm_absorb.hip — latent attention of prompt portions: the queries as its key tiles want them, in one launch: the unrotated part carried into the
// latent space head by head (q ukT^T), the rotated part behind it, both rounded to bf16.
//
// What bounds it: the memory (8184 rows of 16 heads: 50 MB of queries come, 75 MB go; 27 us at 4.6 TB/s).  As a product of one K step on the staged
// tiles it took 57.6 us, whose results left as single values of two bytes, and 11.7 for a rotation in a launch of its own; here 32.9.  A wave
// keeps its 64 weight rows and passes blocks of 64 rows by them: the rows are asked for whole, a block ahead, by the workgroup, rounded into the
// LDS, and the results turn there into 16-byte pieces.  (Every wave asking for its own fragments, 16 bytes of 32 rows at a time: 66.7 us, for the
// lines of a load are fetched one by one.)
#include <algorithm>

#include "lm_latent_parts.h"

namespace zg {
namespace lm {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kRows = 64, kPitch = 64 * 2 + 16;

// D = 16 DK.  A workgroup: a head, 256 columns of its latent (a wave 64, whose weights it keeps), `blocks` times 64 rows one after the other.
template <int DK>
__global__ __launch_bounds__(256, 2) void latent_queries_kernel(const float* q, const bf16_t* ukT, bf16_t* qa, int ldq, int M, int H, int R, int KR, int blocks, const int* row_pos, Rotary rot) {
    constexpr int D = 16 * DK, PITCH_A = D * 2 + 16, LA = D / 16, RPT = D / 4;  // 16-byte pieces of a query a lane loads; lanes to a row
    __shared__ __attribute__((aligned(16))) char s_img[4][kRows * kPitch];
    __shared__ __attribute__((aligned(16))) char s_a[2][kRows * PITCH_A];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, fr = lane & 31, kh = lane >> 5;
    // workgroups go round the eight XCDs: each gets a run of the list, in which the heads of the same rows are neighbours (they share lines of the result)
    const int total = gridDim.x, q8 = total >> 3, r8 = total & 7, xcd = blockIdx.x & 7, at = xcd * q8 + min(xcd, r8) + (int)(blockIdx.x >> 3);
    const int h = at % H, n0 = blockIdx.y * 256 + wave * 64, row0 = at / H * blocks * kRows, end = min(M, row0 + blocks * kRows);
    const bool mine = n0 < KR;  // KR is whole pieces of 64
    const float* qh = q + (size_t)h * (D + R);
    f32x4 next[LA];
    auto fetch = [&](int m0) {
#pragma unroll
        for (int i = 0; i < LA; ++i)  // (rows beyond the edge: never stored)
            next[i] = *reinterpret_cast<const f32x4*>(qh + (size_t)min(m0 + i * (256 / RPT) + tid / RPT, M - 1) * ldq + tid % RPT * 4);
    };
    fetch(row0);
    u32x4 bf[DK][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int kk = 0; kk < DK; ++kk) bf[kk][j] = *reinterpret_cast<const u32x4*>(ukT + ((size_t)h * KR + min(n0, KR - 64) + j * 32 + fr) * D + kk * 16 + kh * 8);
    char* img = s_img[wave];
    const int half = rot.dims / 2, per = R / 8;
    int buf = 0;
    for (int m0 = row0; m0 < end; m0 += kRows, buf ^= 1) {
#pragma unroll
        for (int i = 0; i < LA; ++i)
            *reinterpret_cast<u32x2*>(s_a[buf] + (i * (256 / RPT) + tid / RPT) * PITCH_A + tid % RPT * 8) = u32x2{cvt_pk_bf16(next[i].x, next[i].y), cvt_pk_bf16(next[i].z, next[i].w)};
        __syncthreads();  // (the other buffer is free: everybody has read it before writing this one)
        fetch(m0 + kRows);
        if (mine) {
            u32x4 af[DK][2];
#pragma unroll
            for (int kk = 0; kk < DK; ++kk)
#pragma unroll
                for (int i = 0; i < 2; ++i) af[kk][i] = *reinterpret_cast<const u32x4*>(s_a[buf] + (i * 32 + fr) * PITCH_A + kk * 32 + kh * 16);
            f32x16 acc[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
#pragma unroll
            for (int kk = 0; kk < DK; ++kk)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bf[kk][j]), __builtin_bit_cast(bf16x8, af[kk][i]), acc[i][j], 0, 0, 0);
            // element e of a 32 x 32 tile: column 8 (e / 4) + 4 (lane / 32) + e % 4, row lane % 32 (a wave's accesses to the LDS are in order)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<u32x2*>(img + (i * 32 + fr) * kPitch + (j * 32 + 8 * g + 4 * kh) * 2) =
                            u32x2{cvt_pk_bf16(acc[i][j][4 * g], acc[i][j][4 * g + 1]), cvt_pk_bf16(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3])};
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const int r = 8 * x + (lane >> 3), c = lane & 7, m = m0 + r;
                const u32x4 v = *reinterpret_cast<const u32x4*>(img + r * kPitch + c * 16);
                if (m < end) *reinterpret_cast<u32x4*>(qa + ((size_t)m * H + h) * (KR + R) + n0 + c * 8) = v;
            }
        }
        if (blockIdx.y == 0)  // the rotated part, eight channels a lane
            for (int i = tid; i < kRows * per; i += 256) {
                const int r = i / per, c = (i - r * per) * 8, m = m0 + r;
                if (m >= end) continue;
                const float* src = qh + (size_t)m * ldq + D;
                f32x4 v[2] = {*reinterpret_cast<const f32x4*>(src + c), *reinterpret_cast<const f32x4*>(src + c + 4)};
                if (c < rot.dims) {  // (whole pieces of eight turn)
                    const float pos = (float)row_pos[m];
                    if (rot.halves) {
                        const bool first = c < half;
                        const int p = first ? c : c - half;
                        const f32x4 o[2] = {*reinterpret_cast<const f32x4*>(src + (first ? c + half : p)), *reinterpret_cast<const f32x4*>(src + (first ? c + half : p) + 4)};
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float a = pos * rot.freq[p + e], co = cosf(a) * rot.amp, si = sinf(a) * rot.amp, x = v[e / 4][e % 4], y = o[e / 4][e % 4];
                            v[e / 4][e % 4] = first ? x * co - y * si : x * co + y * si;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const float a = pos * rot.freq[(c + e) / 2], co = cosf(a) * rot.amp, si = sinf(a) * rot.amp, x = v[e / 4][e % 4], y = v[e / 4][e % 4 + 1];
                            v[e / 4][e % 4] = x * co - y * si;
                            v[e / 4][e % 4 + 1] = y * co + x * si;
                        }
                    }
                }
                *reinterpret_cast<u32x4*>(qa + ((size_t)m * H + h) * (KR + R) + KR + c) =
                    u32x4{cvt_pk_bf16(v[0].x, v[0].y), cvt_pk_bf16(v[0].z, v[0].w), cvt_pk_bf16(v[1].x, v[1].y), cvt_pk_bf16(v[1].z, v[1].w)};
            }
    }
}

}  // namespace

int launch_latent_queries(const float* q, int ldq, const bf16_t* ukT, bf16_t* qa16, int M, int H, int D, int R, int KR, const Rotary& rot, const int* row_pos, hipStream_t s, bool* taken) {
    *taken = false;
    const uintptr_t all = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(ukT) | reinterpret_cast<uintptr_t>(qa16);
    if ((D != 64 && D != 128) || KR % 64 != 0 || R % 8 != 0 || ldq % 4 != 0 || (all & 15) != 0 || rot.dims > R || rot.dims % (rot.halves ? 16 : 8) != 0 || M <= 0) return ZG_OK;
    // 64 rows a workgroup until there are four for each compute unit
    const long long all_blocks = (long long)((M + kRows - 1) / kRows), chunks = (KR + 255) / 256;
    const int blocks = (int)std::max(1ll, std::min(all_blocks, all_blocks * H * chunks / 1024));
    const long long grid = (all_blocks + blocks - 1) / blocks * H;
    ZG_REQUIRE(grid < (1LL << 31) && chunks <= 65535, ZG_ERR_UNSUPPORTED, "latent attention: %d rows of %d heads exceed the grid", M, H);
    const dim3 g((unsigned)grid, (unsigned)chunks);
    if (D == 64) latent_queries_kernel<4><<<g, 256, 0, s>>>(q, ukT, qa16, ldq, M, H, R, KR, blocks, row_pos, rot);
    else latent_queries_kernel<8><<<g, 256, 0, s>>>(q, ukT, qa16, ldq, M, H, R, KR, blocks, row_pos, rot);
    ZG_HIP(hipGetLastError());
    note_kernel("latent_queries_kernel<%d>", D);
    *taken = true;
    return ZG_OK;
}

}  // namespace lm
}  // namespace zg
