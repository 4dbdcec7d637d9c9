// GEMM of fp32 rows with fp32 weights on the bf16 matrix cores (gfx950): the tied
// lm_head (model.py:585) over every position of a batch of token windows,
//     y[m, n] = sum_k x[m, k] w[n, k]
//
// Both operands as three bf16 planes with hi + mid + lo equal to the fp32 value
// (split3), and of the nine plane products the six of weight 2^-16 and above: what
// is dropped is below fp32 rounding of a single product, and an output is rounded
// six times per 16 columns where an fp32 chain rounds 16 times.
//
// Six products at bf16's rate are 2.6 times the fp32 matrix cores' (2.5 PFLOP/s / 6
// against 157 TFLOP/s). A workgroup of four wavefronts owns 128 rows of x and 128
// of w, each wavefront all 128 rows of x and 32 weight rows of its own, which it
// loads (lane (r, h): 16 consecutive columns of row r) and splits in registers, no
// weight split twice or passed through LDS; the planes of x are written once by
// the split kernel in operand order and shared through LDS, double buffered. Two
// workgroups a CU cover each other's waits. Workgroups that follow one another on
// an XCD share the weight rows. 50257 x 768, the platform's fp32 GEMM / this
// (us, with the split): M = 512 341 / 223, M = 100 115 / 67, M = 1024 629 / 414, at
// width 1600 M = 512 652 / 440 (1.1 PFLOP/s of bf16 products); relative error
// against 64 bits at K = 768 5.0e-7 / 4.3e-7, at K = 1600 7.2e-7 / 6.2e-7. What
// bounds it: the matrix cores at the clock they hold, and the barrier a unit.
#include <algorithm>

#include "tiq_internal.hpp"

namespace tiq {
namespace {

#include "gemm_staged_kernel.hpp"

constexpr int kFM = 128, kFN = 128;     // output tile
constexpr int kFT = kFM / 32;           // row tiles of x a workgroup
constexpr int kFX = kFT * 6;            // 1 KB operand blocks of a 32-column unit
constexpr int kFL = kFX * 64 / 256;     // their 16-byte chunks a thread

// 8 fp32 values -> three bf16x8 planes with p[0] + p[1] + p[2] == v
__device__ __forceinline__ void planes_of(const float (&v)[8], u32x4 (&p)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x0 = v[2 * i], x1 = v[2 * i + 1];
        const uint32_t hi = pk_bf16(x0, x1);
        const float r0 = x0 - bf_lo(hi), r1 = x1 - bf_hi(hi);
        const uint32_t mid = pk_bf16(r0, r1);
        p[0][i] = hi;
        p[1][i] = mid;
        p[2][i] = pk_bf16(r0 - bf_lo(mid), r1 - bf_hi(mid));
    }
}

// x (M, K) -> operand blocks: row tile t, unit u (32 columns), plane q, half e: 1 KB,
// lane l = 32 h + r holding row 32 t + r, columns 32 u + 16 h + 8 e .. + 7.
__global__ __launch_bounds__(256) void split_planes_kernel(const float* __restrict__ x, int64_t ldx, int M, int K,
                                                           uint8_t* __restrict__ x3) {
    const int K8 = K / 8, U = K / 32;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)M * K8) return;
    const int m = (int)(i / K8), c = (int)(i % K8);
    const float* xr = x + (int64_t)m * ldx + 8 * c;
    float v[8];
    *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(xr);
    *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(xr + 4);
    u32x4 p[3];
    planes_of(v, p);
    const int u = c >> 2, h = (c >> 1) & 1, e = c & 1;
#pragma unroll
    for (int q = 0; q < 3; ++q)
        *reinterpret_cast<u32x4*>(x3 + ((((int64_t)(m >> 5) * U + u) * 3 + q) * 2 + e) * 1024 +
                                  (32 * h + (m & 31)) * 16) = p[q];
}

__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const uint8_t* __restrict__ x3, const float* __restrict__ x,
                                                          int64_t ldx, const float* __restrict__ w, int64_t ldw,
                                                          float* __restrict__ y, int64_t ldy, int M, int N, int K) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2][kFX * 1024];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int U = K / 32, T = (M + 31) / 32;
    const int tiles_m = (M + kFM - 1) / kFM, tiles_n = (N + kFN - 1) / kFN;
    int tm, tn;
    staged_tile_of(blockIdx.x, tm, tn, tiles_m, tiles_n);
    const int n0 = tn * kFN + 32 * wave;
    const float* wr = w + (int64_t)min(n0 + r, N - 1) * ldw + 16 * h;  // a row past N repeats the last, unstored
    // staging chunk q of a unit: bytes 4096 q + 16 tid of its blocks; row tiles
    // past the last repeat it (not stored)
    const uint8_t* xp[kFL];
#pragma unroll
    for (int q = 0; q < kFL; ++q) {
        const int b = 4096 * q + 16 * tid, t = b / 6144;
        xp[q] = x3 + (int64_t)min(tm * kFT + t, T - 1) * U * 6144 + (b - 6144 * t);
    }
    u32x4 xs[kFL], wv[2][4];
    auto xload = [&](int u) {
#pragma unroll
        for (int q = 0; q < kFL; ++q) xs[q] = *reinterpret_cast<const u32x4*>(xp[q] + (int64_t)u * 6144);
    };
    auto xstore = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kFL; ++q) *reinterpret_cast<u32x4*>(&smem[buf][4096 * q + 16 * tid]) = xs[q];
    };
    auto wload = [&](int u, int p) {
#pragma unroll
        for (int q = 0; q < 4; ++q) wv[p][q] = *reinterpret_cast<const u32x4*>(wr + 32 * u + 4 * q);
    };
    // D[m][n]: result register q of lane (r, h) holds m = 8 (q / 4) + 4 h + q % 4, n = r
    floatx16 acc[kFT];
#pragma unroll
    for (int i = 0; i < kFT; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][q] = 0.f;
    xload(0);
    wload(0, 0);
    wload(min(1, U - 1), 1);
    xstore(0);
    xload(min(1, U - 1));
    __syncthreads();
    // unit u: its planes in buffer u % 2, its weights in set u % 2; stage u + 1 goes
    // to the other buffer (whose readers passed the last barrier). Past the last
    // unit the loads repeat it.
    auto unit = [&](int u, int p) {
        xstore(p ^ 1);
        xload(min(u + 2, U - 1));
        u32x4 wp[2][3];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(wv[p][2 * e + i / 4][i % 4]);
            planes_of(v, wp[e]);
        }
        wload(min(u + 2, U - 1), p);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            bf16x8 xf[kFT][3], wf[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                wf[q] = __builtin_bit_cast(bf16x8, wp[e][q]);
#pragma unroll
                for (int i = 0; i < kFT; ++i)
                    xf[i][q] = *reinterpret_cast<const bf16x8*>(&smem[p][((i * 3 + q) * 2 + e) * 1024 + 16 * lane]);
            }
            constexpr int kx[6] = {0, 1, 0, 2, 1, 0}, kw[6] = {0, 0, 1, 0, 1, 2};
#pragma unroll
            for (int j = 0; j < 6; ++j)
#pragma unroll
                for (int i = 0; i < kFT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[i][kx[j]], wf[kw[j]], acc[i], 0, 0, 0);
        }
        __syncthreads();
    };
    int u = 0;
    for (; u + 1 < U; u += 2) {
        unit(u, 0);
        unit(u + 1, 1);
    }
    if (u < U) unit(u, 0);
    // 32 consecutive outputs of two rows a store, written once and read by a later kernel
    const int m0 = tm * kFM + 4 * h;
    if (n0 + r >= N) return;
    float odd[kFT] = {};  // NaN where an output is not finite
#pragma unroll
    for (int i = 0; i < kFT; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int m = m0 + 32 * i + 8 * (q >> 2) + (q & 3);
            if (m < M) {
                __builtin_nontemporal_store(acc[i][q], y + (int64_t)m * ldy + n0 + r);
                odd[i] = fmaf(acc[i][q], 0.f, odd[i]);
            }
        }
    if ((odd[0] + odd[1]) + (odd[2] + odd[3]) == 0.f) return;
    // An operand that is infinite or rounds to infinity in bf16 (from 3.39e38) has a
    // NaN plane, and so has every output of it: those as plain fp32 sums, which give
    // infinities and NaN their meaning. The chain ends where it is NaN.
    uint64_t todo = 0;
#pragma unroll
    for (int i = 0; i < kFT; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q)
            todo |= (uint64_t)(acc[i][q] != acc[i][q]) << (16 * i + q);
    const float4* wn = reinterpret_cast<const float4*>(w + (int64_t)(n0 + r) * ldw);
    while (todo) {
        const int o = __builtin_ctzll(todo);
        todo &= todo - 1;
        const int m = m0 + 32 * (o >> 4) + 8 * (o >> 2 & 3) + (o & 3);
        if (m >= M) continue;
        const float4* xm = reinterpret_cast<const float4*>(x + (int64_t)m * ldx);
        float s = 0.f;
        for (int k = 0; k < K / 4 && s == s; ++k) {
            const float4 a = xm[k], b = wn[k];
            s = fmaf(a.x, b.x, s);
            s = fmaf(a.y, b.y, s);
            s = fmaf(a.z, b.z, s);
            s = fmaf(a.w, b.w, s);
        }
        y[(int64_t)m * ldy + n0 + r] = s;
    }
}

// From 65 rows: at 64 the platform's GEMM has a tile of its own (width 1024 70 us
// against 78 here, at 100 rows 125 / 79). N only has to be worth a chip of tiles.
bool f32_rows(int64_t M, int64_t K, int64_t N) {
    return M > 64 && N >= 4096 && K > 0 && K % 32 == 0 && M <= 0x7fffffff - kFM && N <= 0x7fffffff - kFN &&
           ((M + kFM - 1) / kFM) * ((N + kFN - 1) / kFN) <= 0x7fffffff && M * (K / 8) <= 0x7fffffffLL * 256;
}

}  // namespace
}  // namespace tiq

using namespace tiq;

extern "C" size_t tiq_linear_f32_workspace(int64_t M, int64_t K, int64_t N) {
    return f32_rows(M, K, N) ? (size_t)((M + 31) / 32 * 32 * K * 6) : 0;
}

extern "C" int tiq_linear_f32_ws(const float* x, int64_t M, int64_t K, int64_t ldx, const float* w, int64_t ldw,
                                 int64_t N, float* y, int64_t ldy, void* workspace, size_t workspace_bytes,
                                 void* stream) {
    if (M < 0 || N < 0 || K < 0) return TIQ_EINVAL;
    if (M == 0 || N == 0) return TIQ_OK;
    if (!x || !w || !y || K == 0 || ldx < K || ldw < K || ldy < N) return TIQ_EINVAL;
    if (!f32_rows(M, K, N)) return TIQ_EUNSUPPORTED;
    if (!aligned(x, 16) || !aligned(w, 16) || ldx % 4 != 0 || ldw % 4 != 0) return TIQ_EALIGN;
    if (!workspace || workspace_bytes < tiq_linear_f32_workspace(M, K, N) || !aligned(workspace, 16))
        return TIQ_EWORKSPACE;
    uint8_t* x3 = static_cast<uint8_t*>(workspace);
    hipLaunchKernelGGL(split_planes_kernel, dim3((unsigned)((M * (K / 8) + 255) / 256)), dim3(256), 0,
                       as_stream(stream), x, ldx, (int)M, (int)K, x3);
    const int rc = launch_status();
    if (rc != TIQ_OK) return rc;
    const int64_t tiles = ((M + kFM - 1) / kFM) * ((N + kFN - 1) / kFN);
    hipLaunchKernelGGL(gemm_f32_kernel, dim3((unsigned)tiles), dim3(256), 0, as_stream(stream), x3, x, ldx, w, ldw,
                       y, ldy, (int)M, (int)N, (int)K);
    return launch_status();
}
