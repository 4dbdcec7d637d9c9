// GEMM of fp32 activations with integer weights on the int8 matrix cores
// (gfx950): the quantized Linears of a prompt (model.py:254,319,352,355 with
// M = B*T rows) in a model that keeps fp32 activations:
//     y[m, n] = scale[n] * sum_k x[m, k] * q[n, k] + bias[n]
//
// A row of x becomes a fixed-point row, x[m, k] = 2^(e_m - 29) X[m, k] with
// 2^e_m <= max_k |x[m, k]| < 2^(e_m + 1) and X = rint(x 2^(29 - e_m)) a 31-bit
// integer (exact for every element within 2^-6 of the row's largest; smaller
// ones are rounded by at most 2^-30 of it), and X four signed base-256 digits, each an
// int8 plane. Every product and sum the MFMAs form is then an exact integer
// (|sum| <= K 2^14 < 2^31), four sums an output, which the epilogue combines in
// fp32: an output carries one rounding of its inputs and a handful at the end,
// where an fp32 accumulation rounds once a step. Relative 2-norm error against
// 64 bits, unit-variance rows with one column in 256 eight times larger, as
// three bf16 planes with fp32 sums before and as digits now: K = 768 1.0e-7 /
// 5.1e-8, K = 1600 5.2e-7 / 5.1e-8, K = 6400 1.0e-6 / 5.1e-8.
//
// (Exact products of sliced operands: Ozaki, Ogita, Oishi, Rump, Numerical Algorithms
// 59, 2012; on integer matrix units: Ootomo, Ozaki, Yokota, IJHPCA 38, 2024.)
//
// Rows of wide range. Where a few elements stand far above the rest, the rest's
// rounding (2^-30 of the largest) is what an output with zero codes in those few
// columns has: N(0, 1) with one element T, such outputs, K = 768: T = 1e3 3.0e-7 of
// their norm, 1e5 3.5e-5, where an fp32 chain has 5e-7 at any T. So a row whose
// largest element is more than kFar^2 sqrt(K) times the square of the mean square
// root of its other elements (of each pair of neighbours the larger) keeps its fp32
// bits, a byte a plane in the digits' place and size, and rs < 0 marks it: the product
// computes its outputs once more, by fp32 sums (wide_rows). The line lies where the
// digits' error on such outputs reaches the chain's, which grows with sqrt(K) (one
// large element among N(0, 1): T = 1400 at K = 768); the mean square root weighs a
// row's many elements and not its few: a hidden row after GELU, mostly small, stays on
// this side (rows with less than 3% of their elements above zero do not).
//
// Why four int8 planes: int8 MFMAs run at twice the bf16 rate, so four planes
// cost two bf16 passes over the product instead of three, and the codes enter
// the matrix cores as they are stored, with no widening beside the MFMAs.
// M = 4096, three planes before / digits now, the planes' pass included: 1600 x
// 4800 242 / 154 us, 1600 x 1600 82 / 64, 6400 x 1600 310 / 200; M = 512, 768 x
// 2304 25 / 15; M = 77, 768 x 3072 56 (the decode GEMV) / 11. What bounds the
// large ones: the matrix cores at the clock the chip holds under them (a loop
// of independent int8 MFMAs on random data reaches 3.0 of the nominal 5 POP/s:
// 84 us of the 143 at 1600 x 4800), then the step's LDS traffic, which does not
// hide wholly beside one wavefront's MFMAs a SIMD.
#include <algorithm>
#include <cmath>

#include "tiq_internal.hpp"

namespace tiq {
namespace {

#include "gemm_staged_kernel.hpp"

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int kDigits = 4;
// kW4G with groups of more than kPairGroup columns, whose digit sums do not join in
// int32 (256 columns: 256 (2^14 257) < 2^31); a kernel of its own, as a choice inside
// the fold costs the narrow groups 15% (1600 x 4800 M = 1024 65 -> 76 us)
constexpr int kW4GWide = 1000 + kW4G, kPairGroup = 256;

// The digit planes in MFMA operand order: for row tile t (32 rows), unit u (32
// columns) and digit d (0 lowest) a 1 KB block at ((t U + u) 4 + d) 1024, byte
// 16 l + j of it the digit of row 32 t + l % 32, column 32 u + 16 (l / 32) + j
// (NIB: the even columns of the 16 first, then the odd ones -- the order in
// which nibble weights unpack), so the product's loads and LDS accesses are
// all contiguous. One workgroup per R rows: 8 rows' chunks of a block are 128
// consecutive bytes, a whole cache line a store (4 rows where that would leave
// CUs idle). rs[m] = 2^(e_m - 29), -1 for a row held as its fp32 bits: one of wide
// range or below 2^-97 or, with fewer than kInfRows rows, one that holds an infinity or
// NaN. From kInfRows rows such a row has rs NaN (every output of it is then NaN).
// IT: 1024-column passes held in registers; 0: the row is read twice.
constexpr int kSplitThreads = 512;

// Rows from which a row that holds an infinity or NaN gives NaN in every output, as a
// split into planes does; fewer rows replace the GEMV, which gives inf there.
constexpr int kInfRows = 128;
// Rows of a row tile held as fp32 bits up to which dot products beat the MFMAs.
constexpr int kFewWide = 4;

constexpr float kFar = 7.0f;

// 2^-64 times the square root of a float, from its bits, to a constant and 6% (half
// the exponent); 0 for zero.
__device__ __forceinline__ float rough_root(uint32_t b) { return __uint_as_float(b >> 1); }

// op over the lanes of equal number modulo R (4 or 8), in every lane, by lane moves on
// the VALU (shuffles pass through the LDS crossbar).
template <int R, typename Op>
__device__ __forceinline__ uint32_t across(uint32_t v, Op op) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = op(a[0], a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = op(b[0], b[1]);
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));  // row_ror:8
    if constexpr (R == 4) v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));
    return v;
}
template <int R>
__device__ __forceinline__ float sum_across(float v) {
    return __uint_as_float(across<R>(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }));
}
template <int R>
__device__ __forceinline__ uint32_t max_across(uint32_t v) {
    return across<R>(v, [](uint32_t a, uint32_t b) { return max(a, b); });
}

__device__ __forceinline__ uint32_t digits_of(float v, float mul) {
    const int t = (int)__builtin_rintf(v * mul) + 0x00808080;
    return (uint32_t)t ^ 0x00808080u;
}

template <bool NIB>
__device__ __forceinline__ void store_digits(const float (&v)[16], float mul, bool bits, uint8_t* __restrict__ dst) {
    u32x4 pl[kDigits];
#pragma unroll
    for (int g = 0; g < 4; ++g) {  // four columns -> one dword of each plane
        uint32_t t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = 4 * g + i;
            const float e = v[NIB ? (p < 8 ? 2 * p : 2 * (p - 8) + 1) : p];
            t[i] = bits ? __float_as_uint(e) : digits_of(e, mul);
        }
        const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u);  // d0 d0 d1 d1 of t0, t1
        const uint32_t b = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u);
        const uint32_t c = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u);  // d2 d2 d3 d3
        const uint32_t d = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
        pl[0][g] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        pl[1][g] = __builtin_amdgcn_perm(b, a, 0x07060302u);
        pl[2][g] = __builtin_amdgcn_perm(d, c, 0x05040100u);
        pl[3][g] = __builtin_amdgcn_perm(d, c, 0x07060302u);
    }
#pragma unroll
    for (int q = 0; q < kDigits; ++q) *reinterpret_cast<u32x4*>(dst + 1024 * q) = pl[q];
}

// LN: the digits of LayerNorm(x) (two-pass mean and biased variance as torch;
// the row already sits in registers, so the LayerNorm's own pass -- a read and a
// write of x, 9 us at 4096 x 1600 -- costs two exchanges more here).
template <int IT, int R, bool NIB, bool LN>
__global__ __launch_bounds__(kSplitThreads) void split_digits_kernel(const float* __restrict__ x, int64_t ldx, int M,
                                                                     int K, uint8_t* __restrict__ xt,
                                                                     float* __restrict__ rs, bool gelu, float line,
                                                                     const float* __restrict__ ln_w,
                                                                     const float* __restrict__ ln_b, float ln_eps) {
    static_assert(!LN || IT > 0, "LayerNorm needs the row in registers");
    static_assert(R == 8 || R == 4, "whole quads of rows");
    constexpr int WV = kSplitThreads / 64, CT = kSplitThreads / R;  // 16-column chunks a pass
    __shared__ float2 stat[WV][R];
    __shared__ float ls[2][WV][R];
    const int tid = threadIdx.x, row = tid % R, c0 = tid / R;
    const int m = blockIdx.x * R + row;
    const int NC = K / 16, U = K / 32;
    // A quad of lanes reads 64 consecutive bytes of each of its four rows in
    // turn (16 segments a load instruction, not 64), then transposes: each lane
    // ends with the 16 columns of its own row.
    const int j4 = tid & 3;
    const float* xq[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        xq[i] = x + (int64_t)min((int)blockIdx.x * R + (row & 4) + i, M - 1) * ldx + 4 * j4;
    const bool odd = j4 & 1, high = j4 & 2;
    auto load = [&](int c, float (&v)[16]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4*>(v + 4 * i) = *reinterpret_cast<const float4*>(xq[i] + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int i = 0; i < 4; i += 2) {  // rows i, i + 1 with the neighbour lane
                const float got = dpp_move<0xB1>(odd ? v[4 * i + e] : v[4 * i + 4 + e]);
                v[4 * i + e] = odd ? got : v[4 * i + e];
                v[4 * i + 4 + e] = odd ? v[4 * i + 4 + e] : got;
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {  // rows i, i + 2 with the lane two away
                const float got = dpp_move<0x4E>(high ? v[4 * i + e] : v[4 * i + 8 + e]);
                v[4 * i + e] = high ? got : v[4 * i + e];
                v[4 * i + 8 + e] = high ? v[4 * i + 8 + e] : got;
            }
        }
        if (gelu) {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = gelu_tanh(v[i]);
        }
    };
    uint32_t mx = 0;
    // the sum, over pairs of neighbours, of their larger elements' square roots (each
    // element by itself takes twice the instructions)
    float root = 0.f;
    auto measure = [&](const float (&e)[16], bool mine) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const uint32_t b = max(abs_bits(e[i]), abs_bits(e[i + 1]));
            mx = max(mx, b);
            s += rough_root(b);
        }
        root += mine ? s : 0.f;
    };
    float v[IT ? IT : 1][16];
    if constexpr (IT > 0) {
#pragma unroll
        for (int it = 0; it < IT; ++it) load(min(c0 + CT * it, NC - 1), v[it]);  // past the row: its last chunk again
        if constexpr (LN) {
            // a row is the threads of equal tid % R: 64 / R lanes of each wavefront
            auto row_sum = [&](float s, int slot) {
                s = sum_across<R>(s);
                if ((tid & 63) < R) ls[slot][tid >> 6][row] = s;
                __syncthreads();
                float t = 0.f;
#pragma unroll
                for (int w = 0; w < WV; ++w) t += ls[slot][w][row];
                return t;
            };
            float s = 0.f;
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                float t = 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i) t += v[it][i];
                s += c0 + CT * it < NC ? t : 0.f;
            }
            const float mu = row_sum(s, 0) / (float)K;
            float d = 0.f;
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                float t = 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i) t = fmaf(v[it][i] - mu, v[it][i] - mu, t);
                d += c0 + CT * it < NC ? t : 0.f;
            }
            const float rstd = 1.0f / sqrtf(row_sum(d, 1) / (float)K + ln_eps);
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int c = 16 * min(c0 + CT * it, NC - 1);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 gw = *reinterpret_cast<const float4*>(ln_w + c + 4 * q);
                    const float4 gb = *reinterpret_cast<const float4*>(ln_b + c + 4 * q);
                    v[it][4 * q + 0] = fmaf((v[it][4 * q + 0] - mu) * rstd, gw.x, gb.x);
                    v[it][4 * q + 1] = fmaf((v[it][4 * q + 1] - mu) * rstd, gw.y, gb.y);
                    v[it][4 * q + 2] = fmaf((v[it][4 * q + 2] - mu) * rstd, gw.z, gb.z);
                    v[it][4 * q + 3] = fmaf((v[it][4 * q + 3] - mu) * rstd, gw.w, gb.w);
                }
            }
        }
#pragma unroll
        for (int it = 0; it < IT; ++it) measure(v[it], c0 + CT * it < NC);
    } else {
        for (int c = c0; c < NC; c += CT) {
            load(c, v[0]);
            measure(v[0], true);
        }
    }
    mx = max_across<R>(mx);
    root = sum_across<R>(root);
    if ((tid & 63) < R) stat[tid >> 6][row] = make_float2(__uint_as_float(mx), root);
    __syncthreads();
    root = 0.f;
#pragma unroll
    for (int w = 0; w < WV; ++w) {
        const float2 t = stat[w][row];
        mx = max(mx, __float_as_uint(t.x));
        root += t.y;
    }
    const bool finite = mx < 0x7f800000u;
    // the other pairs' sum of square roots against the largest's, whose share of it
    // is line; rows below 2^-97 would need powers of two that are not normal
    const float top = rough_root(mx);
    const int far = top > line * (root - top);
    const int tiny = (mx != 0) & (mx < (127u - 97) << 23);
    const bool wide = (finite & (far | tiny)) | (!finite & (M < kInfRows));
    const int e = max((int)(mx >> 23) - 127, -97);
    const float mul = finite ? __uint_as_float((uint32_t)(29 - e + 127) << 23) : 0.f;
    if (c0 == 0 && m < M)
        rs[m] = wide ? -1.f : finite ? __uint_as_float((uint32_t)(e - 29 + 127) << 23) : __uint_as_float(0x7fc00000u);
    uint8_t* base = xt + (int64_t)(m >> 5) * U * 4096 + (m & 31) * 16;
    if constexpr (IT > 0) {
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int c = c0 + CT * it;
            if (c < NC && m < M) store_digits<NIB>(v[it], mul, wide, base + (int64_t)(c >> 1) * 4096 + (c & 1) * 512);
        }
    } else {
        for (int c = c0; c < NC; c += CT) {
            load(c, v[0]);  // every lane of a quad: rows past M too
            if (m < M) store_digits<NIB>(v[0], mul, wide, base + (int64_t)(c >> 1) * 4096 + (c & 1) * 512);
        }
    }
}

// The product. A workgroup of four wavefronts, WMW x (4 / WMW) over its tile,
// each with TM row tiles (32 rows of x) and TN column tiles (32 rows of w): BM =
// 32 TM WMW, BN = 32 TN (4 / WMW). Per k64 step a wavefront issues 8 TM TN
// MFMAs: each of its weight fragments meets the four digits of each row tile,
// so a weight fragment is read once for four MFMAs. Digits and codes pass
// through LDS (double buffered, one barrier a step) in operand blocks; their
// loads wait in D register sets, issued D - 1 steps before their LDS store.
// Beside each MFMA goes one of the step's other operations.
// LDS blocks: the digits as they lie in memory; codes per 32-row tile 2 KB,
// chunk c (16 columns) of row r at 512 c + 16 (r ^ 2 c) -- staging stores (two
// rows' four chunks per 8 lanes) and fragment reads (8 rows of a chunk) both
// cover every bank.
// FMT kW8 (codes) or kW4 (the reference's nibbles, unpacked to 16 (n - 8) on
// the LDS store: the 16 is taken out with the scale).
// kW4G (group-wise nibbles, groups of gs k64 steps, an fp16 scale per row and
// group): a group's four sums become one fp32 value a result, which times the
// group's scale is added to fp32 sums -- the lanes of a result register share no
// column, so a scale is one load a lane and column tile; the next group starts
// from zero. A digit and a code reach 2^7 each, so a sum reaches 2^14 a column:
// two of them join in int32 (256 times one plus the other) up to 256 columns, in
// fp32 for wider groups (kW4GWide).
// gridDim.z > 1: split over K, workgroup z writes fp32 slice z of y (no bias).
// Out (fp32 output, unsplit): a residual added last, or a c_attn whose key and
// value columns go to the cache (a 32-column tile lies within one head, so its
// base address is one scalar) instead of to rows that a copy would read again.
// 32 x 128 rows of width 1600: attention with its cache 281 -> 256 us, the two
// 10 us copies gone; four windows of 128 through GPT-2 small with both LayerNorms,
// residuals and GELU inside the products 1515 -> 1374 us.
struct DigitsOut {
    const float* res;
    int64_t ldr;
    float *k, *v;
    int64_t sb, sh, st;
    uint32_t T, magic;  // magic = ceil(2^32 / T): m / T = (m magic) >> 32 for m T < 2^32; 0: T = 1
};

template <int WMW, int TM, int TN, int D, int OCC, bool PERSIST, int FMT, typename TY>
__global__ __launch_bounds__(256, OCC) void gemm_digits_kernel(
    const uint8_t* __restrict__ xt, const float* __restrict__ rs, const uint8_t* __restrict__ w, int64_t ldw,
    const float* __restrict__ scale, const float* __restrict__ bias, TY* __restrict__ y, int64_t ldy, int M, int N,
    int K, const uint16_t* __restrict__ scale16, int ngroups, int gs, DigitsOut out) {
    constexpr bool GROUPED = FMT == kW4G || FMT == kW4GWide;
    static_assert(D >= 2, "register sets");
    constexpr int WNW = 4 / WMW;
    constexpr int MT = TM * WMW, NTL = TN * WNW;  // row and column tiles of the workgroup
    constexpr int NF = TM * kDigits;              // activation fragments a k32 block
    constexpr int NRD = NF + TN, NMF = NF * TN;   // fragment reads and MFMAs a k32 block
    constexpr int XL = 2 * MT, WL = NTL / 2, NL = XL + WL;  // staging loads a thread and step
    constexpr int XS = MT * 8192, STAGE = XS + NTL * 2048;
    static_assert(NTL % 2 == 0 && NL <= 2 * NMF, "staging split");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WNW, wn = wave % WNW;
    const int r = lane & 31, h = lane >> 5;
    const int T = (M + 31) / 32, U = K / 32;
    const int tiles_m = (T + MT - 1) / MT, tiles_n = (N + 32 * NTL - 1) / (32 * NTL);
    const int NK = K / 64;
    const int s0 = (int)blockIdx.z * NK / (int)gridDim.z;
    const int nk = ((int)blockIdx.z + 1) * NK / (int)gridDim.z - s0;
    const bool split = gridDim.z > 1;

    // weight staging: rows wrow + 64 j, chunk wch (16 columns)
    constexpr int WB = FMT == kW8 ? 16 : 8;  // bytes of 16 columns
    const int wrow = tid >> 2, wch = tid & 3;
    const int ws = XS + (wrow >> 5) * 2048 + wch * 512 + (((wrow & 31) ^ (2 * wch)) * 16);
    const uint8_t* xp[MT];
    uint32_t woff[WL];
    int tm, tn;
    u32x4 st[D][NL];
    auto gload = [&](int s, int p, int q) {
        if (q < XL) {
            st[p][q] = *reinterpret_cast<const u32x4*>(xp[q >> 1] + (int64_t)s * 8192 + (q & 1) * 4096);
        } else {
            const uint8_t* src = w + (woff[q - XL] + (uint32_t)(4 * s) * WB);
            if constexpr (FMT == kW8) {
                st[p][q] = *reinterpret_cast<const u32x4*>(src);
            } else {
                const uint2 t = *reinterpret_cast<const uint2*>(src);
                st[p][q] = u32x4{t.x, t.y, 0u, 0u};
            }
        }
    };
    // a tile's addresses and its first D stages
    auto begin_tile = [&](int tile) {
        staged_tile_of(tile, tm, tn, tiles_m, tiles_n);
#pragma unroll
        for (int i = 0; i < MT; ++i)  // row tiles past the last repeat it (not stored)
            xp[i] = xt + ((int64_t)min(tm * MT + i, T - 1) * U + 2 * s0) * 4096 + tid * 16;
#pragma unroll
        for (int j = 0; j < WL; ++j)
            woff[j] = (uint32_t)min(tn * 32 * NTL + wrow + 64 * j, N - 1) * (uint32_t)ldw +
                      (uint32_t)(4 * s0 + wch) * WB;
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int q = 0; q < NL; ++q) gload(min(d, nk - 1), d, q);
    };
    auto lstore = [&](int buf, int p, int q) {
        uint8_t* base = smem + buf * STAGE;
        if (q < XL) {
            *reinterpret_cast<u32x4*>(base + q * 4096 + tid * 16) = st[p][q];
        } else {
            u32x4 v = st[p][q];
            if constexpr (FMT != kW8) {
                uint32_t e0, o0, e1, o1;
                nibbles_x16(v.x, e0, o0);
                nibbles_x16(v.y, e1, o1);
                v = u32x4{e0, e1, o0, o1};
            }
            *reinterpret_cast<u32x4*>(base + ws + (q - XL) * 4096) = v;
        }
    };
    i32x4 FX[2][NF], FW[2][TN];
    int wo[2];  // chunk 2 kk + h of row r within a code tile
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) wo[kk] = XS + wn * TN * 2048 + (2 * kk + h) * 512 + ((r ^ (2 * (2 * kk + h))) * 16);
    const int xo = wm * TM * 8192 + lane * 16;
    auto fread = [&](int buf, int kk, int set, int f) {
        const uint8_t* base = smem + buf * STAGE;
        if (f < TN)
            FW[set][f] = *reinterpret_cast<const i32x4*>(base + wo[kk] + f * 2048);
        else
            FX[set][f - TN] = *reinterpret_cast<const i32x4*>(base + xo + ((f - TN) >> 2) * 8192 + kk * 4096 +
                                                              ((f - TN) & 3) * 1024);
    };
    // D[m][n]: result register q of lane (r, h) holds m = 8 (q / 4) + 4 h + q % 4, n = r
    i32x16 acc[TN][TM][kDigits];
    auto mfma = [&](int set, int t, bool fresh) {
        const int f = t / TN, j = t % TN;
        const i32x16 z = {};
        acc[j][f >> 2][f & 3] = __builtin_amdgcn_mfma_i32_32x32x32_i8(FX[set][f], FW[set][j],
                                                                      fresh ? z : acc[j][f >> 2][f & 3], 0, 0, 0);
    };
    // Step s (register set p = s % D): the first k32 block's MFMAs (of step 0
    // from zero sums) beside the second's fragment reads and stage s + 1's LDS
    // stores; the barrier; the second block's MFMAs beside the next step's first
    // fragments and stage s + D's loads into set p. Past the last stage the
    // loads repeat it, which keeps the body one path.
    auto step = [&](int s, int p, bool fresh) {
        const int cur = s & 1, nxt = cur ^ 1, pn = (p + 1) % D;
        const int sl = min(s + D, nk - 1);
#pragma unroll
        for (int t = 0; t < NMF; ++t) {
            mfma(0, t, fresh);
#pragma unroll
            for (int f = t * NRD / NMF; f < (t + 1) * NRD / NMF; ++f) fread(cur, 1, 1, f);
#pragma unroll
            for (int q = t * NL / NMF; q < (t + 1) * NL / NMF; ++q) lstore(nxt, pn, q);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NMF; ++t) {
            mfma(1, t, false);
#pragma unroll
            for (int f = t * NRD / NMF; f < (t + 1) * NRD / NMF; ++f) fread(nxt, 0, 0, f);
#pragma unroll
            for (int q = t * NL / NMF; q < (t + 1) * NL / NMF; ++q) gload(sl, p, q);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // an output's four digit sums in fp32
    auto joined = [&](const i32x16 (&a)[kDigits], int q) -> float {
        float f = (float)a[3][q];
        f = fmaf(f, 256.f, (float)a[2][q]);
        f = fmaf(f, 256.f, (float)a[1][q]);
        return fmaf(f, 256.f, (float)a[0][q]);
    };
    // group-wise: fp32 sums, the current group's scales (fp16 bits as loaded)
    float sum[GROUPED ? TN : 1][GROUPED ? TM : 1][16];
    uint16_t sg[TN];
    auto load_scales = [&](int g) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
            sg[j] = scale16[(int64_t)min(tn * 32 * NTL + wn * 32 * TN + 32 * j + r, N - 1) * ngroups + g];
    };
    auto fold = [&]() {
        if constexpr (GROUPED) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float sc = f16_bits_to_f32(sg[j]);
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int q = 0; q < 16; ++q) {
                        float v;
                        if constexpr (FMT == kW4G) {
                            const float hi = (float)((acc[j][i][3][q] << 8) + acc[j][i][2][q]);
                            const float lo = (float)((acc[j][i][1][q] << 8) + acc[j][i][0][q]);
                            v = fmaf(hi, 65536.f, lo);
                        } else {
                            v = joined(acc[j][i], q);
                        }
                        sum[j][i][q] = fmaf(v, sc, sum[j][i][q]);
                    }
            }
        }
    };

    constexpr float unit = FMT == kW8 ? 1.f : 0.0625f;
    // The outputs of a tile's rows that are held as fp32 bits, over what the digit
    // sums gave (the same lanes' stores): few rows of a row tile by dot products, a
    // wavefront along K for one column after the other; more of them by the fp32
    // MFMAs over the whole row tile (the other rows' results are not stored). Rare rows,
    // which cost: int8, M = 4096, none / one / every 128th / every row of them, 1600 x
    // 6400 236 / 287 / 384 / 979 us, 6400 x 1600 213 / 362 / 522 / 1259 (three bf16 planes
    // with fp32 sums, which this product replaced: 310 for any row).
    auto wide_rows = [&](int tile) {
        int rm, rn;
        staged_tile_of(tile, rm, rn, tiles_m, tiles_n);
        const int n0 = rn * 32 * NTL + wn * 32 * TN, m0 = (rm * MT + wm * TM) * 32;
        const int u0 = 2 * s0, u1 = 2 * (s0 + nk);
        // a unit's codes, in the order of the digits' bytes
        auto codes = [&](const uint8_t* src) -> u32x4 {
            if constexpr (FMT == kW8) {
                return *reinterpret_cast<const u32x4*>(src);
            } else {
                const uint2 t = *reinterpret_cast<const uint2*>(src);
                uint32_t e0, o0, e1, o1;
                nibbles_x16(t.x, e0, o0);
                nibbles_x16(t.y, e1, o1);
                return u32x4{e0, e1, o0, o1};
            }
        };
        auto code = [](const u32x4& c, int p) { return (float)(int8_t)(c[p >> 2] >> 8 * (p & 3)); };
        // a unit's 16 values: byte p of the four planes
        auto values = [&](const uint8_t* src, float (&v)[16]) {
            u32x4 d[kDigits];
#pragma unroll
            for (int q = 0; q < kDigits; ++q) d[q] = *reinterpret_cast<const u32x4*>(src + 1024 * q);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t pick = e ? 0x07030602u : 0x05010400u;
                    const uint32_t lo = __builtin_amdgcn_perm(d[1][g], d[0][g], pick);
                    const uint32_t hi = __builtin_amdgcn_perm(d[3][g], d[2][g], pick);
                    v[4 * g + 2 * e] = __uint_as_float(__builtin_amdgcn_perm(hi, lo, 0x05040100u));
                    v[4 * g + 2 * e + 1] = __uint_as_float(__builtin_amdgcn_perm(hi, lo, 0x07060302u));
                }
        };
        // column tile j's outputs: where row 0 of each lane's column lies, what follows
        struct Column {
            TY* base;
            float scale, bias;
            bool in, cached;
        };
        auto column = [&](int j) {
            const int n = n0 + 32 * j + r, nc = min(n, N - 1);
            Column c = {y + (int64_t)blockIdx.z * M * ldy + n, GROUPED ? unit : scale[nc] * unit,
                        bias && !split ? bias[nc] : 0.f, n < N, false};
            if constexpr (sizeof(TY) == 4) {
                if (out.k && n0 + 32 * j >= N / 3) {  // whole tiles lie within one head
                    const int col = (n0 + 32 * j) % (N / 3);
                    c.base = (n0 + 32 * j < 2 * (N / 3) ? out.k : out.v) + (col >> 6) * out.sh + (col & 63) + r;
                    c.cached = true;
                }
            }
            return c;
        };
        auto put = [&](const Column& c, int m, float v) {
            if (!c.in) return;
            v = fmaf(v, c.scale, c.bias);
            if constexpr (sizeof(TY) == 4) {
                if (c.cached) {
                    const uint32_t b = out.magic ? __umulhi((uint32_t)m, out.magic) : (uint32_t)m;
                    c.base[(int64_t)b * out.sb + (int64_t)((uint32_t)m - b * out.T) * out.st] = v;
                } else {
                    c.base[(int64_t)m * ldy] =
                        out.res ? v + out.res[(int64_t)m * out.ldr + (c.base - y)] : v;  // unsplit with a residual
                }
            } else {
                c.base[(int64_t)m * ldy] = f32_to_bf16_bits(v);
            }
        };
#pragma unroll 1
        for (int i = 0; i < TM; ++i) {
            const int mt = m0 + 32 * i;
            uint32_t rows = (uint32_t)__ballot(mt + r < M && rs[min(mt + r, M - 1)] < 0.f);  // both halves alike
            const uint8_t* xr = xt + (int64_t)min(mt >> 5, T - 1) * U * 4096;
            if (__popc(rows) > kFewWide) {
                floatx16 a[TN][2], whole[GROUPED ? TN : 1];
                const floatx16 z = {};
                const uint8_t* wr[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) a[j][0] = a[j][1] = z, wr[j] = w + (int64_t)min(n0 + 32 * j + r, N - 1) * ldw + h * WB;
                if constexpr (GROUPED) {
                    static_assert(TN == 1, "group-wise: one column tile");
                    whole[0] = z;
                }
                for (int u = u0; u < u1; u += 2) {  // whole k64 steps
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float xv[16];
                        u32x4 c[TN];
                        values(xr + (int64_t)(u + e) * 4096 + lane * 16, xv);
#pragma unroll
                        for (int j = 0; j < TN; ++j) c[j] = codes(wr[j] + 2 * WB * (u + e));
#pragma unroll
                        for (int p = 0; p < 16; ++p)
#pragma unroll
                            for (int j = 0; j < TN; ++j)
                                a[j][e] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[p], code(c[j], p), a[j][e], 0, 0, 0);
                    }
                    if constexpr (GROUPED) {
                        if ((u + 2) % (2 * gs) == 0 || u + 2 == u1) {
                            const float sg =
                                f16_bits_to_f32(scale16[(int64_t)min(n0 + r, N - 1) * ngroups + u / (2 * gs)]);
#pragma unroll
                            for (int q = 0; q < 16; ++q)
                                whole[0][q] = fmaf(a[0][0][q] + a[0][1][q], sg, whole[0][q]);
                            a[0][0] = a[0][1] = z;
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const Column c = column(j);
#pragma unroll
                    for (int q = 0; q < 16; ++q) {
                        const int o = 8 * (q >> 2) + 4 * h + (q & 3);
                        const float v = GROUPED ? whole[0][q] : a[j][0][q] + a[j][1][q];
                        if (rows >> o & 1) put(c, mt + o, v);
                    }
                }
                continue;
            }
            while (rows) {
                const int o = __builtin_ctz(rows);
                rows &= rows - 1;
#pragma unroll 1
                for (int j = 0; j < TN; ++j) {
                    float keep = 0.f;
                    for (int ub = u0; ub < u1; ub += 32) {  // 1024 columns of x, 16 a lane
                        const int u = min(ub + (lane >> 1), u1 - 1);
                        float xv[16];
                        values(xr + (int64_t)u * 4096 + (lane & 1) * 512 + o * 16, xv);
                        const bool in = ub + (lane >> 1) < u1;
#pragma unroll
                        for (int p = 0; p < 16; ++p) xv[p] = in ? xv[p] : 0.f;
                        constexpr int kAhead = 8;  // columns in flight
#pragma unroll 1
                        for (int c = 0; c < 32; c += kAhead) {
                            u32x4 cv[kAhead];
                            float sg[GROUPED ? kAhead : 1];
#pragma unroll
                            for (int e = 0; e < kAhead; ++e) {
                                const int64_t n = min(n0 + 32 * j + c + e, N - 1);
                                cv[e] = codes(w + n * ldw + 2 * WB * u + (lane & 1) * WB);
                                if constexpr (GROUPED) sg[e] = f16_bits_to_f32(scale16[n * ngroups + u / (2 * gs)]);
                            }
                            asm volatile("" ::: "memory");
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int e = 0; e < kAhead; ++e) {
                                float s[4] = {};
#pragma unroll
                                for (int p = 0; p < 16; ++p) s[p & 3] = fmaf(xv[p], code(cv[e], p), s[p & 3]);
                                float v = (s[0] + s[1]) + (s[2] + s[3]);
                                if constexpr (GROUPED) v *= sg[e];
                                v = wave_sum_dpp(v);
                                keep = r == c + e ? keep + v : keep;
                            }
                        }
                    }
                    if (h == (o >> 2 & 1)) put(column(j), mt + o, keep);  // the half whose lanes stored this row
                }
            }
        }
    };

    const int total = tiles_m * tiles_n;
    bool wide = false;  // some row of this wavefront's tiles is held as fp32 bits
    begin_tile(blockIdx.x);
    // the workgroup's tiles: one, or every gridDim.x-th of a persistent grid,
    // where the next tile's first loads go out before the epilogue
    for (int tile = blockIdx.x;;) {
#pragma unroll
        for (int q = 0; q < NL; ++q) lstore(0, 0, q);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NRD; ++f) fread(0, 0, 0, f);
        if constexpr (GROUPED) {
            load_scales(s0 / gs);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int q = 0; q < 16; ++q) sum[j][i][q] = 0.f;
            int left = gs - s0 % gs;  // steps to the end of the current group (a split may start inside one)
            bool fresh = true;
            auto gstep = [&](int s, int p) {
                if (fresh) step(s, p, true);
                else step(s, p, false);
                fresh = --left == 0;
                if (fresh || s == nk - 1) {  // the group's (or the split's) last step
                    fold();
                    load_scales(min((s0 + s + 1) / gs, ngroups - 1));
                    left = gs;
                }
            };
            int s = 0;
            for (; s + D - 1 < nk; s += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) gstep(s + d, d);
            }
#pragma unroll
            for (int d = 0; d < D - 1; ++d)
                if (s + d < nk) gstep(s + d, d);
        } else {
            step(0, 0, true);
            int s = 1;
            for (; s + D - 1 < nk; s += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) step(s + d, (1 + d) % D, false);
            }
#pragma unroll
            for (int d = 0; d < D - 1; ++d)
                if (s + d < nk) step(s + d, (1 + d) % D, false);
        }

        // y = (((a3 256 + a2) 256 + a1) 256 + a0) 2^(e_m - 29) scale + bias; a
        // store instruction writes 32 consecutive outputs of two rows
        const int n0 = tn * 32 * NTL + wn * 32 * TN, m0 = (tm * MT + wm * TM) * 32;
        const bool full = m0 + 32 * TM <= M && n0 + 32 * TN <= N;
        float sc[TN], bi[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = min(n0 + 32 * j + r, N - 1);
            sc[j] = GROUPED ? unit : scale[n] * unit;
            bi[j] = bias && !split ? bias[n] : 0.f;
        }
        float4 rm[TM][4];  // rows past M hold whatever the buffer holds: their outputs are not stored
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                rm[i][g] = *reinterpret_cast<const float4*>(rs + min(m0 / 32 + i, T - 1) * 32 + 8 * g + 4 * h);
        // whether a row is held as fp32 bits (rows past M too: then wide_rows finds none)
        auto look = [&]() {
            uint32_t signs = 0;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    signs |= __float_as_uint(rm[i][g].x) | __float_as_uint(rm[i][g].y) |
                             __float_as_uint(rm[i][g].z) | __float_as_uint(rm[i][g].w);
            wide |= __any((int)signs < 0);
        };
        // where the registers come out better: before the stores (persistent tile, 4096 x
        // 1600 x 3200 113 -> 109 us), for the small int8 tile after them (512 x 768 11.5 -> 11.0)
        constexpr bool look_first = PERSIST || FMT != kW8;
        if constexpr (look_first) look();
        auto digit_sum = [&](int i, int j, int q) -> float {
            if constexpr (GROUPED) {
                return sum[j][i][q];
            } else {
                return joined(acc[j][i], q);
            }
        };
        tile += gridDim.x;
        const bool more = PERSIST && tile < total;
        if (more) begin_tile(tile);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            TY* yr = y + ((int64_t)blockIdx.z * M + m0 + 32 * i + 4 * h) * ldy + n0 + r;
            if constexpr (sizeof(TY) == 4) {
                if (out.res || out.k) {
                    // groups of four rows of a column tile, a group's residuals
                    // requested RD groups before its stores
                    constexpr int RD = PERSIST ? 0 : 3, NG = 4 * TN;  // persistent: the next tile's loads hold the registers
                    float rv[RD + 1][4];
                    auto request = [&](int t) {
                        const int n = min(n0 + 32 * (t >> 2) + r, N - 1);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            rv[t % (RD + 1)][e] =
                                out.res[(int64_t)min(m0 + 32 * i + 8 * (t & 3) + 4 * h + e, M - 1) * out.ldr + n];
                    };
                    if (out.res) {
#pragma unroll
                        for (int t = 0; t < RD; ++t) request(t);
                    }
                    const int C = N / 3;
#pragma unroll
                    for (int t = 0; t < NG; ++t) {
                        const int j = t >> 2, g = t & 3;
                        if (out.res && t + RD < NG) request(t + RD);
                        const int n = n0 + 32 * j;  // scalar, as is the tile's place
                        const int part = n / C, col = n - part * C;
                        const bool cached = out.k && part > 0;
                        TY* base = cached ? (part == 1 ? out.k : out.v) + (col >> 6) * out.sh + (col & 63) + r : y + n + r;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int q = 4 * g + e, m = m0 + 32 * i + 8 * g + 4 * h + e;
                            const float4 g4 = rm[i][g];
                            const float rmq = e == 0 ? g4.x : e == 1 ? g4.y : e == 2 ? g4.z : g4.w;
                            const float v = fmaf(digit_sum(i, j, q) * rmq, sc[j], bi[j]);
                            if (m < M && n + r < N) {
                                if (cached) {
                                    const uint32_t b = out.magic ? __umulhi((uint32_t)m, out.magic) : (uint32_t)m;
                                    base[(int64_t)b * out.sb + (int64_t)((uint32_t)m - b * out.T) * out.st] = v;
                                } else {
                                    base[(int64_t)m * ldy] = out.res ? v + rv[t % (RD + 1)][e] : v;
                                }
                            }
                        }
                    }
                    continue;
                }
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int q = 4 * g + e;
                    const float rmq = e == 0 ? rm[i][g].x : e == 1 ? rm[i][g].y : e == 2 ? rm[i][g].z : rm[i][g].w;
                    TY* dst = yr + (int64_t)(8 * g + e) * ldy;
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const float v = fmaf(digit_sum(i, j, q) * rmq, sc[j], bi[j]);
                        if (full || (m0 + 32 * i + 8 * g + 4 * h + e < M && n0 + 32 * j + r < N)) {
                            if constexpr (sizeof(TY) == 4) dst[32 * j] = v;
                            else dst[32 * j] = f32_to_bf16_bits(v);
                        }
                    }
                }
            }
        }
        if constexpr (!look_first) look();
        if (!more) break;
        __syncthreads();  // every wavefront's last LDS reads are done
    }
    if (wide) {
        for (int t = blockIdx.x; t < total; t += PERSIST ? (int)gridDim.x : total) wide_rows(t);
    }
}

template <int WMW, int TM, int TN, int D, int OCC, bool PERSIST, int FMT, typename TY>
int run_digits(const LinearArgs& a, const uint8_t* xt, const float* rs, TY* y, int64_t ldy, int64_t S,
               const DigitsOut& out) {
    constexpr int BM = 32 * TM * WMW, BN = 32 * TN * (4 / WMW);
    const int64_t tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
    const int64_t grid = PERSIST ? std::min<int64_t>(tiles, 256 * OCC) : tiles;
    hipLaunchKernelGGL((gemm_digits_kernel<WMW, TM, TN, D, OCC, PERSIST, FMT, TY>), dim3((unsigned)grid, 1, (unsigned)S),
                       dim3(256), 0, a.stream, xt, rs, a.w, a.ldw, a.scale, a.bias, y, ldy, (int)a.M, (int)a.N,
                       (int)a.K, a.scale16, a.fmt == kW4G ? (int)((a.K + a.group - 1) / a.group) : 0,
                       a.fmt == kW4G ? a.group / 64 : 1, out);
    return launch_status();
}

// Tiles, measured on MI355X (graph-timed products, fp32 out; us):
//   32 x 128, two or more workgroups a CU: ahead while the 64 x 128 tiles are
//     fewer than the 512 that run at once (M = 1001, 1024 x 3072: 18.9 against
//     20.2; M = 77, 768 x 3072: 7.5 against 9.6);
//   64 x 128, two a CU, persistent: the larger products (M = 4096: 1600 x 4800
//     143 against 146 at 64 x 256 and 166 at 32 x 128; 1600 x 1600 53 / 55 / 60);
//   64 x 256, one a CU: a long K, where its fewer LDS bytes a MFMA weigh more
//     than its tile's fixed cost (M = 4096, 6400 x 1600: 171 against 187).
enum DigitTile : int { kTile32x128 = 0, kTile64x128 = 1, kTile64x256 = 2 };

DigitTile digits_tile(int64_t M, int64_t N, int64_t K) {
    const int64_t rows = (M + 63) / 64;
    if (rows * ((N + 127) / 128) < 512) return kTile32x128;
    return K >= 3200 && rows * ((N + 255) / 256) >= 256 ? kTile64x256 : kTile64x128;
}

// Splits over K: only where the 32 x 128 tiles leave half of the CUs without
// work and K is long enough for the slices' sum to cost less than it saves (M
// = 77, 3072 x 768, 18 tiles: 15.1 us unsplit, 6.9 in eight; K = 768: 7.5
// unsplit, 6.3 in two, less than the reduction's launch). At least six k64
// steps a split, at most eight splits.
int64_t digits_splits(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = (M + 31) / 32 * ((N + 127) / 128);
    if (tiles * 2 > 256 || K < 1536) return 1;
    return std::max<int64_t>(1, std::min<int64_t>({256 / tiles, K / 64 / 6, 8}));
}

size_t round256(size_t b) { return (b + 255) / 256 * 256; }

template <int FMT, typename TY>
int dispatch_digits(const LinearArgs& a, DigitTile tile, const uint8_t* xt, const float* rs, TY* y, int64_t ldy,
                    int64_t S, const DigitsOut& out = {}) {
    // group-wise: the fp32 sums beside the integer ones fit the small tile
    if constexpr (FMT == kW4G || FMT == kW4GWide) return run_digits<1, 1, 1, 3, 2, false, FMT, TY>(a, xt, rs, y, ldy, S, out);
    else switch (tile) {
        case kTile64x256: return run_digits<2, 1, 4, 2, 1, false, FMT, TY>(a, xt, rs, y, ldy, S, out);
        case kTile64x128: return run_digits<2, 1, 2, 2, 2, true, FMT, TY>(a, xt, rs, y, ldy, S, out);
        default: return run_digits<1, 1, 1, 4, 2, false, FMT, TY>(a, xt, rs, y, ldy, S, out);
    }
}

// Rows below which a split workgroup takes four rows of more than 1024 columns, not
// eight: twice the workgroups and half a thread's chain where they do not fill the
// chip (with the product, us, eight / four: 3072 x 768 M = 512 24.8 / 22.5, 6400 x
// 1600 M = 128 27.9 / 24.4, M = 1024 68.3 / 66.1; level from M = 1536, where the
// eight-row stores are whole cache lines).
constexpr int64_t kSplitWideRows = 1280;

template <bool NIB>
int launch_split_digits(const LinearArgs& a, uint8_t* xt, float* rs, bool gelu, const PrefillFusion& f) {
    const float line = kFar * sqrtf(sqrtf((float)a.K)) / (0.5f * (float)a.K);
    auto launch = [&](auto kernel, int rows) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((a.M + rows - 1) / rows)), dim3(kSplitThreads), 0, a.stream,
                           static_cast<const float*>(a.x), a.ldx, (int)a.M, (int)a.K, xt, rs, gelu, line, f.ln_w,
                           f.ln_b, f.ln_eps);
        return launch_status();
    };
    if (a.K > 1024 && a.K <= 8192 && a.M < kSplitWideRows) {
        if (f.ln_w) return launch(split_digits_kernel<1, 4, NIB, true>, 4);
        if (a.K <= 2048) return launch(split_digits_kernel<1, 4, NIB, false>, 4);
        if (a.K <= 4096) return launch(split_digits_kernel<2, 4, NIB, false>, 4);
        return launch(split_digits_kernel<4, 4, NIB, false>, 4);
    }
    if (f.ln_w) return a.K <= 1024 ? launch(split_digits_kernel<1, 8, NIB, true>, 8) : launch(split_digits_kernel<2, 8, NIB, true>, 8);
    if (a.K <= 1024) return launch(split_digits_kernel<1, 8, NIB, false>, 8);
    if (a.K <= 2048) return launch(split_digits_kernel<2, 8, NIB, false>, 8);
    if (a.K <= 4096) return launch(split_digits_kernel<4, 8, NIB, false>, 8);
    if (a.K <= 7168) return launch(split_digits_kernel<7, 8, NIB, false>, 8);
    return launch(split_digits_kernel<0, 8, NIB, false>, 8);
}

template <int FMT>
int run_digits_linear(const LinearArgs& a, uint8_t* xt, float* rs, float* part, int64_t S, bool gelu,
                      const PrefillFusion& f) {
    int rc = launch_split_digits<FMT != kW8>(a, xt, rs, gelu, f);
    if (rc != TIQ_OK) return rc;
    const DigitTile tile = S > 1 ? kTile32x128 : digits_tile(a.M, a.N, a.K);
    if (S > 1) {
        rc = dispatch_digits<FMT, float>(a, tile, xt, rs, part, a.N, S);
        return rc != TIQ_OK ? rc : launch_splitk_reduce(a, part, S, nullptr, f.res, f.ldr);
    }
    if (a.y_dtype != TIQ_F32) return dispatch_digits<FMT, uint16_t>(a, tile, xt, rs, static_cast<uint16_t*>(a.y), a.ldy, 1);
    DigitsOut out = {f.res, f.ldr, f.k, f.v, f.sb, f.sh, f.st, (uint32_t)f.T, 0};
    if (f.T > 1) out.magic = (uint32_t)(((1ull << 32) + f.T - 1) / f.T);
    return dispatch_digits<FMT, float>(a, tile, xt, rs, static_cast<float*>(a.y), a.ldy, 1, out);
}

}  // namespace

size_t digits_workspace(int64_t M, int64_t K) {
    const int64_t rows = (M + 31) / 32 * 32;
    return round256((size_t)(rows * K * kDigits + rows * 4));
}

size_t digits_split_workspace(int64_t M, int64_t N, int64_t K) {
    const int64_t S = digits_splits(M, N, K);
    return S > 1 ? round256((size_t)(S * M * N * 4)) : 0;
}

// A product that is split for want of tiles leaves its key and value columns to the caller.
bool digits_write_kv(int64_t M, int64_t K, int64_t N) { return N % 192 == 0 && digits_splits(M, N, K) == 1; }

bool digits_supported(const LinearArgs& a) {
    if (a.x_dtype != TIQ_F32 || (a.fmt != kW8 && a.fmt != kW4 && a.fmt != kW4G) || a.kw) return false;
    // group-wise: whole k64 steps a group, rows of whole nibble pairs
    if (a.fmt == kW4G && (a.group % 64 != 0 || !aligned(a.scale16, 2))) return false;
    // int32 sums: K 2^14 < 2^31
    if (a.K % 64 != 0 || a.K > 65536) return false;
    if (!aligned(a.x, 16) || a.ldx % 4 != 0 || !aligned(a.w, 16) || a.ldw % 16 != 0) return false;
    // 32-bit byte offsets into the weights, tile counts within a grid
    if (a.N * a.ldw > 0xffffffffLL) return false;
    return ((a.M + 31) / 32) * ((a.N + 127) / 128) <= 0x7fffffffLL && a.M <= 0x7fffffff - 64;
}

int launch_digits(const LinearArgs& a, void* ws, size_t ws_bytes, bool gelu, const PrefillFusion& f) {
    if (!digits_supported(a)) return TIQ_EUNSUPPORTED;
    if (f.ln_w && (a.K > kDigitsLnMaxK || !aligned(f.ln_w, 16) || !aligned(f.ln_b, 16))) return TIQ_EUNSUPPORTED;
    // rows of a sequence by multiplication: m T < 2^32
    if (f.k && (!digits_write_kv(a.M, a.K, a.N) || a.M * f.T > 0xffffffffLL)) return TIQ_EUNSUPPORTED;
    const size_t need = digits_workspace(a.M, a.K);
    if (!ws || ws_bytes < need || !aligned(ws, 16)) return TIQ_EWORKSPACE;
    uint8_t* xt = static_cast<uint8_t*>(ws);
    const int64_t rows = (a.M + 31) / 32 * 32;
    float* rs = reinterpret_cast<float*>(xt + rows * a.K * kDigits);
    float* part = reinterpret_cast<float*>(xt + need);
    // the split needs room for its slices and the reduction's 16-byte accesses
    // (N % 8 for either output type: both then sum in the same order)
    const int unit = a.y_dtype == TIQ_F32 ? 4 : 8;
    int64_t S = digits_splits(a.M, a.N, a.K);
    if (a.N % 8 != 0 || a.ldy % unit != 0 || !aligned(a.y, 16) || (a.bias && !aligned(a.bias, 16))) S = 1;
    if (f.res && (f.ldr % 4 != 0 || !aligned(f.res, 16))) S = 1;
    S = std::min<int64_t>(S, (int64_t)((ws_bytes - need) / (size_t)(a.M * a.N * 4)));
    S = std::max<int64_t>(S, 1);
    if (a.fmt == kW4G)
        return a.group <= kPairGroup ? run_digits_linear<kW4G>(a, xt, rs, part, S, gelu, f)
                                     : run_digits_linear<kW4GWide>(a, xt, rs, part, S, gelu, f);
    return a.fmt == kW4 ? run_digits_linear<kW4>(a, xt, rs, part, S, gelu, f)
                        : run_digits_linear<kW8>(a, xt, rs, part, S, gelu, f);
}

}  // namespace tiq
