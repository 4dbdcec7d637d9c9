// Causal self-attention of a prompt block on the fp32 matrix cores (gfx950):
// CausalSelfAttention.forward at T > 1 (model.py:284-309), T queries at absolute
// positions first .. first + T - 1 over the S = first + T cached keys, softmax
// (q k^T / sqrt(64)) v with an online fp32 softmax over blocks of 32 keys.
//
// A wavefront owns 32 queries of one (sequence, head) and computes transposed
// tiles with v_mfma_f32_32x32x2_f32 (full fp32 products and sums): S^T = K Q^T
// leaves lane (c, h) (c = lane % 32, h = lane / 32) with query c's scores of keys
// 8 g + 4 h + e (register 4 g + e), so the softmax over keys is a reduction over
// a lane's registers and one exchange with lane ^ 32, and the probabilities are
// already the B operand of O^T += V^T P^T: step (g, e) pairs key 8 g + e (h = 0)
// with 8 g + 4 + e (h = 1), its A operand the same key's value row. Nothing
// passes through LDS: each operand is read from memory once per wavefront, a
// key row as 32 consecutive dims a lane (dim s of one half pairs with dim 32 + s
// of the other), a value row as two consecutive dims a lane (even dims are one
// output tile, odd dims the other).
// NW wavefronts share a query tile, taking its key blocks in turn (w, w + NW,
// ...), and merge their partial (maximum, sum, output) through LDS: a few long
// prompts then still fill the chip and the longest tile is NW times shorter.
// Tiles of one head go to one XCD (its keys and values stay in that L2).
//
// Against the vector-ALU kernel it replaced (64-query tiles, keys and values in
// LDS), us: 32 sequences x 25 heads x T = 128 104 -> 44, 1 x 16 x 1001 292 -> 36,
// 8 x 16 x 500 193 -> 68, 4 x 12 x 128 39 -> 8, one query over 501 keys 147 ->
// 15; relative error against 64 bits the same or lower (T = 1001: 2.7e-7 ->
// 1.8e-7). What bounds it: v_mfma_f32_32x32x2 runs on the vector FMA units, so
// the softmax's instructions add to its time (of a block's 5500 clocks 4096 are
// MFMAs); a block's keys and values hide behind the one before.
// Tried: keys through LDS with coalesced loads (20% slower), 64-key blocks of
// one chain, eight wavefronts a tile.
#include <cmath>

#include "tiq_internal.hpp"

namespace tiq {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kPaHead = 64;   // head width
constexpr int kPaTile = 32;   // queries a tile, keys a block
constexpr int kPaXcds = 8;

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attention_kernel(
    const float* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_st, const float* __restrict__ k,
    int64_t k_sb, int64_t k_sh, int64_t k_st, const float* __restrict__ v, int64_t v_sb, int64_t v_sh, int64_t v_st,
    int H, int P, int tiles, int T, int first, float* __restrict__ y, int64_t y_sb, int64_t y_sh, int64_t y_st) {
    // Workgroup -> (sequence, head) pair p and tile: pair p on XCD p % 8; per XCD
    // the longest tiles of every pair first, every other run of 32 workgroups
    // (one a CU) backwards, so that a CU's workgroups add up to about the same
    const int xcd = blockIdx.x % kPaXcds, P8 = (P + kPaXcds - 1) / kPaXcds;
    int i = blockIdx.x / kPaXcds;
    if (i >> 5 & 1) i = (i & ~31) + min(32, tiles * P8 - (i & ~31)) - 1 - (i & 31);
    const int p = i % P8 * kPaXcds + xcd;
    if (p >= P) return;
    const int tile = tiles - 1 - i / P8;
    const int b = p / H, hd = p - b * H;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 31, h = lane >> 5;
    const int t0 = tile * kPaTile;
    const int tq = min(t0 + c, T - 1);  // past T: row T - 1 again, unstored
    const int qpos = first + tq, q_min = first + t0;
    const int s_end = first + min(T, t0 + kPaTile);  // keys this tile needs
    const int nb = (s_end + kPaTile - 1) / kPaTile;

    float qv[32];
    {
        const float* qr = q + b * q_sb + hd * q_sh + (int64_t)tq * q_st + 32 * h;
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<float4*>(qv + 4 * i) = reinterpret_cast<const float4*>(qr)[i];
    }
    const float* kb = k + b * k_sb + hd * k_sh + 32 * h;
    const float* vb = v + b * v_sb + hd * v_sh;
    const uint32_t voff = (uint32_t)(4 * h) * (uint32_t)v_st + 2 * c;
    const bool near_rows = v_st < (1 << 28);  // the lane's offset in 32 bits
    float kr[32];
    auto load_keys = [&](int j) {  // key 32 j + c (past the last: the last again, masked)
        const float4* kp = reinterpret_cast<const float4*>(kb + (int64_t)min(kPaTile * j + c, s_end - 1) * k_st);
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<float4*>(kr + 4 * i) = kp[i];
    };
    float m = -INFINITY, l = 0.f;
    floatx16 o[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) o[0][i] = 0.f, o[1][i] = 0.f;
    if (w < nb) load_keys(w);
    for (int j = w; j < nb; j += NW) {
        // value rows of keys 32 j + 8 g + 4 h + e, dims 2 c and 2 c + 1
        float2 vr[16];
        if (near_rows && kPaTile * j + kPaTile <= s_end) {  // a scalar row address and the lane's offset
            const float* vj = vb + (int64_t)(kPaTile * j) * v_st;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                vr[i] = *reinterpret_cast<const float2*>(vj + (8 * (i >> 2) + (i & 3)) * v_st + voff);
        } else {  // the last block: rows past the last key repeat it (masked)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                vr[i] = *reinterpret_cast<const float2*>(
                    vb + (int64_t)min(kPaTile * j + 8 * (i >> 2) + 4 * h + (i & 3), s_end - 1) * v_st + 2 * c);
        }
        floatx16 sc[4];  // four chains of 16 dims, summed as pairs
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const floatx16 z = {};
                sc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[8 * d + s], qv[8 * d + s], s ? sc[d] : z, 0, 0, 0);
            }
        load_keys(min(j + NW, nb - 1));  // the next block's, over the softmax and the values' products
        float pr[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            pr[i] = ((sc[0][i] + sc[1][i]) + (sc[2][i] + sc[3][i])) * 0.125f;  // 1 / sqrt(64), exact
        if (kPaTile * j + kPaTile - 1 > q_min) {  // a block not wholly before the tile's first query
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (kPaTile * j + 8 * (i >> 2) + 4 * h + (i & 3) > qpos) pr[i] = -INFINITY;
        }
        float bm = pr[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) bm = fmaxf(bm, pr[i]);
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        const float mn = fmaxf(m, bm);
        // no visible key so far (or all of them -inf): exponents of -inf, not of NaN
        const float ms = mn == -INFINITY ? 0.f : mn;
        const float alpha = expf(m - ms);
        float ps = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            pr[i] = expf(pr[i] - ms);
            ps += pr[i];
        }
        l = l * alpha + ps + __shfl_xor(ps, 32, 64);
        if (__any(mn > m)) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[0][i] *= alpha, o[1][i] *= alpha;
        }
        m = mn;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[i].x, pr[i], o[0], 0, 0, 0);
            o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[i].y, pr[i], o[1], 0, 0, 0);
        }
    }
    // register 4 g + e of o[t] is dim 2 (8 g + 4 h + e) + t of query c: unit u =
    // (g, e / 2) is the four consecutive dims 16 g + 8 h + 4 (u % 2) .. + 3
    float* yr = y + b * y_sb + hd * y_sh + (int64_t)tq * y_st + 8 * h;
    const bool store = t0 + c < T;
    if constexpr (NW == 1) {
        const float inv = 1.0f / l;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = 4 * (u >> 1) + 2 * (u & 1);
            const float4 r = make_float4(o[0][i] * inv, o[1][i] * inv, o[0][i + 1] * inv, o[1][i + 1] * inv);
            if (store) *reinterpret_cast<float4*>(yr + 16 * (u >> 1) + 4 * (u & 1)) = r;
        }
    } else {
        __shared__ float ml[NW][2][32];
        __shared__ float4 part[NW][8][64];
        if (h == 0) ml[w][0][c] = m, ml[w][1][c] = l;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = 4 * (u >> 1) + 2 * (u & 1);
            part[w][u][lane] = make_float4(o[0][i], o[1][i], o[0][i + 1], o[1][i + 1]);
        }
        __syncthreads();
        float mx = ml[0][0][c];
#pragma unroll
        for (int i = 1; i < NW; ++i) mx = fmaxf(mx, ml[i][0][c]);
        const float ms = mx == -INFINITY ? 0.f : mx;
        float wt[NW], sum = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            wt[i] = expf(ml[i][0][c] - ms);
            sum = fmaf(ml[i][1][c], wt[i], sum);
        }
        const float inv = 1.0f / sum;
#pragma unroll
        for (int u = w; u < 8; u += NW) {
            float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < NW; ++i) {  // in wavefront order
                const float4 f = part[i][u][lane];
                r.x = fmaf(f.x, wt[i], r.x);
                r.y = fmaf(f.y, wt[i], r.y);
                r.z = fmaf(f.z, wt[i], r.z);
                r.w = fmaf(f.w, wt[i], r.w);
            }
            if (store)
                *reinterpret_cast<float4*>(yr + 16 * (u >> 1) + 4 * (u & 1)) =
                    make_float4(r.x * inv, r.y * inv, r.z * inv, r.w * inv);
        }
    }
}

}  // namespace
}  // namespace tiq

using namespace tiq;

extern "C" int tiq_prefill_attention(const float* q, int64_t q_sb, int64_t q_sh, int64_t q_st, const float* k,
                                     int64_t k_sb, int64_t k_sh, int64_t k_st, const float* v, int64_t v_sb,
                                     int64_t v_sh, int64_t v_st, int64_t batch, int64_t n_head, int64_t T,
                                     int64_t first, int64_t head_dim, float* y, int64_t y_sb, int64_t y_sh,
                                     int64_t y_st, void* stream) {
    if (batch < 0 || n_head <= 0 || T < 0 || first < 0) return TIQ_EINVAL;
    if (batch == 0 || T == 0) return TIQ_OK;
    if (!q || !k || !v || !y) return TIQ_EINVAL;
    if (head_dim != kPaHead) return TIQ_EUNSUPPORTED;
    if (batch > 65535 || n_head > 65535 || T > INT32_MAX - 64 || first > INT32_MAX - 64 - T) return TIQ_EUNSUPPORTED;
    const int64_t strides[12] = {q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, y_sb, y_sh, y_st};
    for (int64_t st : strides)
        if (st < 0 || st % 4 != 0) return TIQ_EALIGN;  // 16-byte rows of 4 floats
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(y, 16)) return TIQ_EALIGN;
    const int64_t tiles = (T + kPaTile - 1) / kPaTile, P = batch * n_head;
    const int64_t grid = (P + kPaXcds - 1) / kPaXcds * kPaXcds * tiles;
    if (grid > INT32_MAX) return TIQ_EUNSUPPORTED;
    const int64_t blocks = (first + T + kPaTile - 1) / kPaTile;  // of the longest tile
    auto launch = [&](auto kernel, int nw) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * nw), 0, as_stream(stream), q, q_sb, q_sh, q_st, k,
                           k_sb, k_sh, k_st, v, v_sb, v_sh, v_st, (int)n_head, (int)P, (int)tiles, (int)T, (int)first,
                           y, y_sb, y_sh, y_st);
    };
    // Wavefronts a tile (us with 1 / 2 / 4): many tiles fill the chip by
    // themselves and pay for the merge (800 of 7 blocks 25 / 30 / 32, 3200 of up
    // to 4 44 / 45 / 54) unless their longest is long (2048 of up to 16 78 / 68 /
    // 69, 3200 of up to 32 188 / 169 / 174); with few tiles the longest one's
    // chain is the time (512 of up to 32 91 / 51 / 36, 192 of up to 4 14 / 10 /
    // 8); eight were slower than four everywhere but at equality.
    const int64_t n = tiles * P;
    const int nw = blocks <= 2 ? (int)blocks : n < 768 ? 4 : blocks >= 8 ? 2 : 1;
    if (nw == 1) launch(prefill_attention_kernel<1>, 1);
    else if (nw == 2) launch(prefill_attention_kernel<2>, 2);
    else launch(prefill_attention_kernel<4>, 4);
    return launch_status();
}
