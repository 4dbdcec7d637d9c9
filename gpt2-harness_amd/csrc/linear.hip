// Linear entry points of the C ABI: argument checks and the choice between
// the decode GEMV (vector ALUs) and the prefill GEMM (matrix cores).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <utility>
#include <vector>

#include "tiq_internal.hpp"

namespace tiq {

int check_linear(const LinearArgs& a) {
    if (a.x_dtype != TIQ_F32 && a.x_dtype != TIQ_BF16) return TIQ_EINVAL;
    if (a.y_dtype != TIQ_F32 && a.y_dtype != TIQ_BF16) return TIQ_EINVAL;
    if (a.M < 0 || a.N < 0 || a.K < 0) return TIQ_EINVAL;
    if (a.M == 0 || a.N == 0) return TIQ_OK;
    if (a.K == 0) return TIQ_EINVAL;
    if (!a.x || !a.w || !a.y) return TIQ_EINVAL;
    if (a.fmt == kW4G ? !a.scale16 : !a.scale) return TIQ_EINVAL;
    if (a.ldx < a.K || a.ldy < a.N) return TIQ_EINVAL;
    if (a.M > 0x7fffffff || a.N > 0x7fffffff || a.K > 0x7fffffff) return TIQ_EUNSUPPORTED;
    if (a.fmt == kW4 && (a.K % 2)) return TIQ_EINVAL;
    if (a.fmt == kW4G && (a.group < 2 || (a.group & 1))) return TIQ_EINVAL;
    return TIQ_OK;
}

// Measurement state of tiq_stamp_begin / tiq_stamp_end: the caller's stamp
// buffer, the slots handed out so far and, per stamped launch, its first
// slot and workgroup count.
namespace {
struct StampState {
    std::mutex mu;
    uint64_t* base = nullptr;
    int64_t slots = 0, used = 0;
    std::vector<std::pair<int64_t, int64_t>> log;
};
StampState& stamp_state() {
    static StampState st;
    return st;
}
}  // namespace

uint64_t* stamp_slots(int64_t workgroups) {
    StampState& st = stamp_state();
    std::lock_guard<std::mutex> lk(st.mu);
    if (!st.base || workgroups <= 0 || st.used + 4 * workgroups > st.slots) return nullptr;
    uint64_t* p = st.base + st.used;
    st.log.emplace_back(st.used, workgroups);
    st.used += 4 * workgroups;
    return p;
}

namespace {

// Rows of M at and above which the 128 x 128-tile MFMA GEMM beats the
// vector-ALU GEMV (below it the GEMM wastes most of each tile).
constexpr int64_t kGemmMinRows = 128;

// Rows below kGemmMinRows from which fp32 rows against int4 codes (either
// layout) have a workspace for digit planes: there is no batched kernel for
// int4, and the LDS-staged GEMV, four activation rows a tile, grows with M
// (graph-timed us, GEMV / planes: 768 x 3072 M = 16 18 / 10; 1280 x 5120 M = 8 17
// / 12; 6400 x 1600 M = 16 29 / 17; but 768 x 768 M = 16 7.3 / 10.3).
bool w4_planes_rows(int64_t M, int64_t K, int64_t N) {
    const int64_t work = M * N * K;
    return M >= 32 || (M >= 16 && (N >= 2048 || work >= 100000000)) || (M >= 8 && N >= 2048 && work >= 25000000);
}

// bf16 rows below kGemmMinRows that the MFMA GEMM takes when neither the
// 16-row GEMV nor the batched kernel does (int8 past 64 rows or K past their
// reach; int4): the alternative is the decode GEMV, four activation rows a
// tile (us, GEMV / GEMM: int8 1600 x 4800 M = 100 166 / 17, 6400 x 1600 M = 24
// 35 / 14; int4 768 x 2304 M = 8 12.0 / 9.7, 1024 x 4096 M = 64 85 / 11). Up to 16 rows on
// matrices under 2048 rows the GEMV's direct kernel is ahead (3072 x 768 M = 16
// 6.8 / 12) until the product is large (6400 x 1600 M = 16 30 / 16). Up to four rows
// its one pass over the weights is ahead at every size (1600 x 6400, M = 4: int4 6.8 / 16.6,
// group-wise 12.7 / 18.4; M = 2: int8 4.5 / 14.3).
bool bf16_gemm_rows(int64_t M, int64_t K, int64_t N) {
    const int64_t work = M * N * K;
    return M > 64 || (M > 4 && (M > 16 || N >= 2048 ? work >= 14000000 : work >= 100000000));
}

LinearArgs make_args(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const uint8_t* w, int64_t ldw,
                     const float* scale, const uint16_t* scale16, int group, const float* bias, int64_t N, void* y,
                     int y_dtype, int64_t ldy, void* stream, WFormat fmt) {
    LinearArgs a;
    a.x = x;
    a.x_dtype = x_dtype;
    a.M = M;
    a.K = K;
    a.ldx = ldx;
    a.w = w;
    a.ldw = ldw;
    a.scale = scale;
    a.scale16 = scale16;
    a.group = group;
    a.bias = bias;
    a.N = N;
    a.y = y;
    a.y_dtype = y_dtype;
    a.ldy = ldy;
    a.stream = as_stream(stream);
    a.fmt = fmt;
    return a;
}

// x (M, K) fp32 -> x3 (M, 3K) bf16: [hi | lo | lo2] with hi = rne(x),
// lo = rne(x - hi), lo2 = rne(x - hi - lo). Both differences are exact in fp32
// and lo2 holds the last 8 significant bits, so hi + lo + lo2 == x; an int8
// weight is exact in bf16, so every product the MFMA forms is exact and the
// GEMM over the three planes is as accurate as an fp32 GEMM. gelu: the planes
// of gelu_tanh(x) (the same function as tiq_gelu_tanh's), x read once.
__global__ void split_bf16x3_kernel(const float* __restrict__ x, int64_t ldx, int M, int K,
                                    uint16_t* __restrict__ x3, bool gelu) {
    const int k4 = K / 4;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)M * k4) return;
    const int m = (int)(i / k4), k = (int)(i % k4) * 4;
    float4 v = *reinterpret_cast<const float4*>(x + (int64_t)m * ldx + k);
    if (gelu) {
        v.x = gelu_tanh(v.x);
        v.y = gelu_tanh(v.y);
        v.z = gelu_tanh(v.z);
        v.w = gelu_tanh(v.w);
    }
    // pairs through v_cvt_pk_bf16_f32 (round to nearest even)
    uint32_t p[3][2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float x0 = e ? v.z : v.x, x1 = e ? v.w : v.y;
        const uint32_t hi = pk_bf16(x0, x1);
        const float r0 = x0 - bf_lo(hi), r1 = x1 - bf_hi(hi);
        const uint32_t lo = pk_bf16(r0, r1);
        p[0][e] = hi;
        p[1][e] = lo;
        p[2][e] = pk_bf16(r0 - bf_lo(lo), r1 - bf_hi(lo));
    }
    uint16_t* row = x3 + (int64_t)m * 3 * K + k;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(row + (int64_t)q * K) = make_uint2(p[q][0], p[q][1]);
}

size_t split_workspace(int64_t M, int64_t K) { return (size_t)(M * 3 * K * 2 + 255) / 256 * 256; }

// fp32 rows that take the int8 matrix cores as digit planes, given a workspace.
// int8 has the batched kernel up to 64 rows, which holds a wavefront's whole
// share of K and reads every activation plane for each 32-row tile: past 32
// rows of a long K the planes win (us, batched / planes: 1600 x 4800 M = 64 21 /
// 15, 6400 x 1600 M = 32 32 / 20, 3072 x 768 M = 48 17.2 / 12.5; 768 x 3072 M = 64 7.5 / 10.7
// and, with few rows of weights, 1600 x 1600 M = 64 10.6 / 12.1); from 65 rows the
// only other kernel is the decode GEMV (77 rows, 768 x 3072: 56 / 11). int4 as
// w4_planes_rows, group-wise also only from the size at which its GEMV falls
// behind (768 x 768: M = 32 10.9 / 14.2, M = 48 16.4 / 14.4) and, where K is too short
// to be split and so one long chain of folds, not up to 8 rows (1024 x 4096 10.8 / 15.5,
// 1280 x 5120 15.7 / 18.0) or, between, 12 (1024 x 4096 15.8 / 16.5; 768 x 3072 15.2 / 13.7,
// 1280 x 5120 20.7 / 18.7).
bool digits_rows(WFormat fmt, int64_t M, int64_t K, int64_t N) {
    if (M >= kGemmMinRows) return true;
    if (fmt == kW8) return M > 64 || (M > 32 && K >= 1536 && (K >= 2048 || N >= 2048)) || (M == 32 && K >= 3072);
    if (!w4_planes_rows(M, K, N)) return false;
    if (fmt == kW4) return true;
    if (K < 1536 && M <= (K >= 1024 && K < 1280 ? 12 : 8)) return false;
    return M * N * K >= 24000000;
}

// fp32 activations through the matrix cores: as exact integer products of digit
// planes (gemm_digits.hip), else (K past their int32 sums, 65536, or weights past
// 32-bit offsets) split into three bf16 planes for a GEMM that takes the
// three-plane problem; TIQ_EUNSUPPORTED otherwise (groups that are no multiple of
// 64 columns, say: the caller falls back). gelu_in: the product takes gelu_tanh(x).
int run_linear_split(const LinearArgs& a, void* ws, size_t ws_bytes, bool gelu_in = false) {
    if (a.x_dtype != TIQ_F32 || a.fmt == kF32 || a.K % 4 != 0) return TIQ_EUNSUPPORTED;
    const bool few = a.M < kGemmMinRows;  // below the documented row count: the workspace is optional
    if (!digits_rows(a.fmt, a.M, a.K, a.N)) return TIQ_EUNSUPPORTED;
    if (!aligned(a.x, 16) || a.ldx % 4 != 0 || a.M * 3 * a.K > 0x7fffffffLL) return TIQ_EUNSUPPORTED;
    if (digits_supported(a)) {
        // from kGemmMinRows the documented size covers the planes
        if (!few && (!ws || ws_bytes < split_workspace(a.M, a.K) || !aligned(ws, 16))) return TIQ_EWORKSPACE;
        const int rc = launch_digits(a, ws, ws_bytes, gelu_in);
        return few && rc == TIQ_EWORKSPACE ? TIQ_EUNSUPPORTED : rc;
    }
    if (few) return TIQ_EUNSUPPORTED;
    LinearArgs g = a;
    g.x = ws;
    g.x_dtype = TIQ_BF16;
    g.K = 3 * a.K;
    g.ldx = 3 * a.K;
    g.kw = a.K;
    const bool staged = staged_gemm_supported(g);
    if (!staged && !gemm_supported(g)) return TIQ_EUNSUPPORTED;
    if (!ws || ws_bytes < split_workspace(a.M, a.K) || !aligned(ws, 16)) return TIQ_EWORKSPACE;
    const int64_t n = a.M * (a.K / 4);
    hipLaunchKernelGGL(split_bf16x3_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, a.stream,
                       static_cast<const float*>(a.x), a.ldx, (int)a.M, (int)a.K, static_cast<uint16_t*>(ws),
                       gelu_in);
    int rc = launch_status();
    if (rc != TIQ_OK) return rc;
    if (!staged) return launch_gemm(g);
    return launch_staged_gemm(g, staged_gemm_choice(g));
}

int run_linear(const LinearArgs& a) {
    int rc = check_linear(a);
    if (rc != TIQ_OK || a.M == 0 || a.N == 0) return rc;
    if (rows16_preferred(a)) return launch_rows16(a);
    if (skinny_supported(a)) return launch_skinny(a);
    if (bf16_gemm_rows(a.M, a.K, a.N) && gemm_supported(a)) return launch_gemm(a);
    return launch_gemv(a);
}

// bf16 rows of the workspace entry points that split a GEMM over K when planned
bool bf16_split_rows(const LinearArgs& a) {
    return a.x_dtype == TIQ_BF16 && bf16_gemm_rows(a.M, a.K, a.N) && !rows16_preferred(a) && !skinny_supported(a);
}

}  // namespace
}  // namespace tiq

using namespace tiq;

extern "C" int tiq_version(void) { return 132; }

extern "C" const char* tiq_status_string(int status) {
    switch (status) {
        case TIQ_OK: return "ok";
        case TIQ_EINVAL: return "invalid argument";
        case TIQ_EBITS: return "bits must be in [2, 8]";
        case TIQ_EALIGN: return "misaligned pointer or leading dimension";
        case TIQ_EUNSUPPORTED: return "unsupported shape or layout";
        case TIQ_EWORKSPACE: return "workspace too small";
        case TIQ_ESCRATCH: return "request exceeds the fixed scratch of the allocation-free entry point";
        default: break;
    }
    if (status <= TIQ_EHIP_BASE) return hipGetErrorString((hipError_t)(TIQ_EHIP_BASE - status));
    return "unknown status";
}

extern "C" int tiq_stamp_begin(uint64_t* buf, int64_t slots) {
    if (slots < 0 || (slots > 0 && !buf)) return TIQ_EINVAL;
    StampState& st = stamp_state();
    std::lock_guard<std::mutex> lk(st.mu);
    st.base = slots ? buf : nullptr;
    st.slots = slots;
    st.used = 0;
    st.log.clear();
    return TIQ_OK;
}

extern "C" int64_t tiq_stamp_end(int64_t* first_slot, int64_t* workgroups, int64_t max_launches) {
    StampState& st = stamp_state();
    std::lock_guard<std::mutex> lk(st.mu);
    const int64_t n = (int64_t)st.log.size();
    for (int64_t i = 0; i < n && i < max_launches; ++i) {
        if (first_slot) first_slot[i] = st.log[i].first;
        if (workgroups) workgroups[i] = st.log[i].second;
    }
    st.base = nullptr;
    st.slots = st.used = 0;
    st.log.clear();
    return n;
}

extern "C" int tiq_linear_w8(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                             const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                             void* stream) {
    return run_linear(make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0,
                                bias, N, y, y_dtype, ldy, stream, kW8));
}

extern "C" size_t tiq_linear_w8_workspace(int x_dtype, int64_t M, int64_t K) {
    if (x_dtype != TIQ_F32 || M < kGemmMinRows || K <= 0 || K % 64 != 0) return 0;
    return split_workspace(M, K);
}

extern "C" int tiq_linear_w8_ws(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                                const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                                void* workspace, size_t workspace_bytes, void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0, bias,
                             N, y, y_dtype, ldy, stream, kW8);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    rc = run_linear_split(a, workspace, workspace_bytes);
    if (rc != TIQ_EUNSUPPORTED) return rc;
    if (bf16_split_rows(a)) {
        rc = launch_staged_gemm_split(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
    }
    return run_linear(a);
}

extern "C" size_t tiq_gemm_w8_workspace(int x_dtype, int64_t M, int64_t K, int64_t N) {
    if ((x_dtype != TIQ_F32 && x_dtype != TIQ_BF16) || K <= 0 || K % 64 != 0 || N <= 0) return 0;
    if (!(x_dtype == TIQ_F32 ? M >= kGemmMinRows || w4_planes_rows(M, K, N) : bf16_gemm_rows(M, K, N))) return 0;
    if (x_dtype == TIQ_F32)
        return std::max(split_workspace(M, K), digits_workspace(M, K)) + digits_split_workspace(M, N, K);
    return staged_split_workspace(M, N, K);
}

extern "C" size_t tiq_linear_workspace(int w_format, int x_dtype, int64_t M, int64_t K, int64_t N) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT4 && w_format != TIQ_WF_INT4_GROUPWISE) return 0;
    if (M <= 4 || K <= 0 || N <= 0 || K % 64 != 0) return 0;
    if (x_dtype == TIQ_F32)
        return digits_rows((WFormat)w_format, M, K, N) ? tiq_gemm_w8_workspace(TIQ_F32, M, K, N) : 0;
    if (x_dtype != TIQ_BF16 || !bf16_gemm_rows(M, K, N)) return 0;
    // int8 rows of the 16-row GEMV and the batched kernel need none; nor does a
    // product that launch_staged_gemm_split leaves whole
    if (w_format == TIQ_WF_INT8 && (M <= 16 || (M <= 64 && K <= 3072))) return 0;
    if (w_format != TIQ_WF_INT4_GROUPWISE && ((M + 127) / 128) * ((N + 127) / 128) >= 48 && K / 64 <= 32) return 0;
    return staged_split_workspace(M, N, K);
}

extern "C" int tiq_gemm_w8_ws(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                              const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                              void* workspace, size_t workspace_bytes, void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0, bias,
                             N, y, y_dtype, ldy, stream, kW8);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    if (workspace && !aligned(workspace, 16)) return TIQ_EALIGN;
    if (x_dtype == TIQ_F32) {
        rc = run_linear_split(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
    } else {
        rc = launch_staged_gemm_split(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
    }
    return launch_gemm(a);
}

extern "C" int tiq_linear_gelu_in_ws(const float* x, int64_t M, int64_t K, int64_t ldx, const void* w, int w_format,
                                     const float* scale, const uint16_t* scale_f16, int group, const float* bias,
                                     int64_t N, float* y, int64_t ldy, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT4 && w_format != TIQ_WF_INT4_GROUPWISE) return TIQ_EINVAL;
    const WFormat fmt = (WFormat)w_format;
    const int64_t ldw = fmt == kW8 ? K : fmt == kW4 ? K / 2 : (K + 1) / 2;
    LinearArgs a = make_args(x, TIQ_F32, M, K, ldx, static_cast<const uint8_t*>(w), ldw, scale, scale_f16, group,
                             bias, N, y, TIQ_F32, ldy, stream, fmt);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    if (M < kGemmMinRows || K % 64 != 0) return TIQ_EUNSUPPORTED;
    if (workspace && !aligned(workspace, 16)) return TIQ_EALIGN;
    return run_linear_split(a, workspace, workspace_bytes, true);
}

extern "C" int tiq_linear_prefill_writes_kv(int w_format, int64_t M, int64_t K, int64_t N) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT4 && w_format != TIQ_WF_INT4_GROUPWISE) return 0;
    if (M <= 0 || K <= 0 || K % 64 != 0 || N <= 0 || !digits_rows((WFormat)w_format, M, K, N)) return 0;
    return digits_write_kv(M, K, N);
}

extern "C" int tiq_linear_prefill_ws(const float* x, int64_t M, int64_t K, int64_t ldx, const void* w, int w_format,
                                     const float* scale, const uint16_t* scale_f16, int group, const float* bias,
                                     int64_t N, float* y, int64_t ldy, const float* ln_weight, const float* ln_bias,
                                     float ln_eps, int gelu_in, const float* residual, int64_t ld_residual,
                                     float* k_out, float* v_out, int64_t kv_sb, int64_t kv_sh, int64_t kv_st,
                                     int64_t T, void* workspace, size_t workspace_bytes, void* stream) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT4 && w_format != TIQ_WF_INT4_GROUPWISE) return TIQ_EINVAL;
    if ((ln_weight == nullptr) != (ln_bias == nullptr) || (k_out == nullptr) != (v_out == nullptr)) return TIQ_EINVAL;
    if ((ln_weight && gelu_in) || (residual && (k_out || ld_residual < N))) return TIQ_EINVAL;
    if (k_out && (T <= 0 || M % T != 0 || N % 3 != 0 || ldy < N / 3 || kv_sb < 0 || kv_sh < 0 || kv_st < 0))
        return TIQ_EINVAL;
    const WFormat fmt = (WFormat)w_format;
    const int64_t ldw = fmt == kW8 ? K : fmt == kW4 ? K / 2 : (K + 1) / 2;
    LinearArgs a = make_args(x, TIQ_F32, M, K, ldx, static_cast<const uint8_t*>(w), ldw, scale, scale_f16, group,
                             bias, N, y, TIQ_F32, k_out ? std::max(ldy, N) : ldy, stream, fmt);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    a.ldy = ldy;
    if (!digits_rows(fmt, M, K, N)) return TIQ_EUNSUPPORTED;
    PrefillFusion f;
    f.ln_w = ln_weight;
    f.ln_b = ln_bias;
    f.ln_eps = ln_eps;
    f.res = residual;
    f.ldr = ld_residual;
    f.k = k_out;
    f.v = v_out;
    f.sb = kv_sb;
    f.sh = kv_sh;
    f.st = kv_st;
    f.T = k_out ? T : 0;
    return launch_digits(a, workspace, workspace_bytes, gelu_in != 0, f);
}

extern "C" int tiq_gemv_w8(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                           const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                           void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0, bias,
                             N, y, y_dtype, ldy, stream, kW8);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    return launch_gemv(a);
}

extern "C" int tiq_gemm_w8(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                           const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                           void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0, bias,
                             N, y, y_dtype, ldy, stream, kW8);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    return launch_gemm(a);
}

extern "C" int tiq_gemm_w8_tile(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* q,
                                const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                                int tile, void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, reinterpret_cast<const uint8_t*>(q), K, scale, nullptr, 0, bias,
                             N, y, y_dtype, ldy, stream, kW8);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    return launch_gemm_tile(a, tile);
}

extern "C" int tiq_linear_w4(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const uint8_t* packed,
                             const float* scale, const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                             void* stream) {
    return run_linear(make_args(x, x_dtype, M, K, ldx, packed, K / 2, scale, nullptr, 0, bias, N, y, y_dtype, ldy,
                                stream, kW4));
}

static int linear_fused(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* w, int w_format,
                        const float* scale, const uint16_t* scale_f16, int group, const float* bias, int64_t N,
                        void* y, int y_dtype, int64_t ldy, const float* ln_weight, const float* ln_bias,
                        float ln_eps, int activation, const float* residual, int64_t ld_residual, void* workspace,
                        size_t workspace_bytes, void* stream) {
    if (w_format < TIQ_WF_INT8 || w_format > TIQ_WF_F32) return TIQ_EINVAL;
    if (activation != TIQ_ACT_NONE && activation != TIQ_ACT_GELU_TANH) return TIQ_EINVAL;
    if ((ln_weight == nullptr) != (ln_bias == nullptr)) return TIQ_EINVAL;
    if (residual && ld_residual < N) return TIQ_EINVAL;
    const WFormat fmt = (WFormat)w_format;
    const int64_t ldw = fmt == kW8 ? K : fmt == kW4 ? K / 2 : fmt == kW4G ? (K + 1) / 2 : K * 4;
    if (fmt == kF32 && scale == nullptr) scale = reinterpret_cast<const float*>(w);  // unused, keeps checks simple
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, static_cast<const uint8_t*>(w), ldw, scale, scale_f16, group,
                             bias, N, y, y_dtype, ldy, stream, fmt);
    a.fuse.ln_w = ln_weight;
    a.fuse.ln_b = ln_bias;
    a.fuse.ln_eps = ln_eps;
    a.fuse.act = activation;
    a.fuse.res = residual;
    a.fuse.ldr = ld_residual;
    a.ws = workspace;
    a.ws_bytes = workspace_bytes;
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    if (rows16_preferred(a)) return launch_rows16(a);
    if (skinny_supported(a)) return launch_skinny(a);
    return launch_gemv(a);
}

extern "C" int tiq_linear_fused(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* w,
                                int w_format, const float* scale, const uint16_t* scale_f16, int group,
                                const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                                const float* ln_weight, const float* ln_bias, float ln_eps, int activation,
                                const float* residual, int64_t ld_residual, void* stream) {
    return linear_fused(x, x_dtype, M, K, ldx, w, w_format, scale, scale_f16, group, bias, N, y, y_dtype, ldy,
                        ln_weight, ln_bias, ln_eps, activation, residual, ld_residual, nullptr, 0, stream);
}

extern "C" size_t tiq_linear_fused_workspace(int x_dtype, int w_format, int64_t M, int64_t K, int64_t N) {
    if (x_dtype != TIQ_F32 || (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_F32)) return 0;
    if (M < kSkinnyMinRows || M > 64 || K <= 0 || K % 32 != 0 || N <= 0) return 0;
    return skinny_workspace(M, K);
}

extern "C" int tiq_linear_fused_ws(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* w,
                                   int w_format, const float* scale, const uint16_t* scale_f16, int group,
                                   const float* bias, int64_t N, void* y, int y_dtype, int64_t ldy,
                                   const float* ln_weight, const float* ln_bias, float ln_eps, int activation,
                                   const float* residual, int64_t ld_residual, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    if (workspace && !aligned(workspace, 16)) return TIQ_EALIGN;
    return linear_fused(x, x_dtype, M, K, ldx, w, w_format, scale, scale_f16, group, bias, N, y, y_dtype, ldy,
                        ln_weight, ln_bias, ln_eps, activation, residual, ld_residual, workspace, workspace_bytes,
                        stream);
}

extern "C" int tiq_linear_w4_ws(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                const uint8_t* packed, const float* scale, const float* bias, int64_t N, void* y,
                                int y_dtype, int64_t ldy, void* workspace, size_t workspace_bytes, void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, packed, K / 2, scale, nullptr, 0, bias, N, y, y_dtype, ldy,
                             stream, kW4);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    if (workspace && !aligned(workspace, 16)) return TIQ_EALIGN;
    rc = run_linear_split(a, workspace, workspace_bytes);
    if (rc != TIQ_EUNSUPPORTED) return rc;
    if (bf16_split_rows(a)) {
        rc = launch_staged_gemm_split(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
    }
    return run_linear(a);
}

extern "C" int tiq_linear_w4g_ws(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                 const uint8_t* packed, const uint16_t* scale_f16, int group, const float* bias,
                                 int64_t N, void* y, int y_dtype, int64_t ldy, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    LinearArgs a = make_args(x, x_dtype, M, K, ldx, packed, (K + 1) / 2, nullptr, scale_f16, group, bias, N, y,
                             y_dtype, ldy, stream, kW4G);
    int rc = check_linear(a);
    if (rc != TIQ_OK || M == 0 || N == 0) return rc;
    if (workspace && !aligned(workspace, 16)) return TIQ_EALIGN;
    rc = run_linear_split(a, workspace, workspace_bytes);
    if (rc != TIQ_EUNSUPPORTED) return rc;
    if (bf16_split_rows(a)) {
        rc = launch_staged_w4g(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
        rc = launch_gemm_w4g_split(a, workspace, workspace_bytes);
        if (rc != TIQ_EUNSUPPORTED) return rc;
    }
    return run_linear(a);
}

extern "C" int tiq_linear_w4g(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const uint8_t* packed,
                              const uint16_t* scale_f16, int group, const float* bias, int64_t N, void* y,
                              int y_dtype, int64_t ldy, void* stream) {
    return run_linear(make_args(x, x_dtype, M, K, ldx, packed, (K + 1) / 2, nullptr, scale_f16, group, bias, N, y,
                                y_dtype, ldy, stream, kW4G));
}

extern "C" size_t tiq_decode_linear_workspace(int w_format, int64_t M, int64_t K, int64_t N) {
    if (w_format == TIQ_WF_F32_TILED) return 0;  // planes in only: nothing staged
    if ((w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT8_TILED && w_format != TIQ_WF_INT4_TILED &&
         w_format != TIQ_WF_F32) ||
        M < kSkinnyMinRows || M > 64 || K <= 0 ||
        K % 32 != 0 || N <= 0)
        return 0;
    return decode_linear_workspace(M, K, N);
}

extern "C" int tiq_decode_linear_takes(int w_format, int64_t M, int64_t K, int64_t N, int planes_out, int finish) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT8_TILED && w_format != TIQ_WF_INT4_TILED &&
        w_format != TIQ_WF_F32 && w_format != TIQ_WF_F32_TILED)
        return 0;
    return decode_linear_takes((WFormat)w_format, M, K, N, planes_out != 0, finish != 0);
}

extern "C" int tiq_tile_int8(const int8_t* w, int64_t N, int64_t K, int64_t ldw, int8_t* tiles, void* stream) {
    return launch_tile_int8(reinterpret_cast<const uint8_t*>(w), N, K, ldw, reinterpret_cast<uint8_t*>(tiles),
                            as_stream(stream));
}

extern "C" int tiq_tile_int4(const uint8_t* w, int64_t N, int64_t K, uint8_t* tiles, void* stream) {
    return launch_tile_int4(w, N, K, tiles, as_stream(stream));
}

extern "C" size_t tiq_tile_f32_bytes(int64_t N, int64_t K) { return tile_f32_bytes(N, K); }

extern "C" int tiq_tile_f32(const float* w, int64_t N, int64_t K, int64_t ldw, float* tiles, void* stream) {
    return launch_tile_f32(w, N, K, ldw, tiles, as_stream(stream));
}

extern "C" size_t tiq_decode_planes_bytes(int64_t M, int64_t K) {
    if (M <= 0 || K <= 0 || K % 32 != 0) return 0;
    return decode_planes_bytes(M, K);
}

// ------------------------------------------- allocation-free decode linear
// tiq_decode_linear_noalloc runs tiq_decode_linear with this fixed array as
// its workspace: TIQ_NOALLOC_SCRATCH_BYTES per GPU, held by the loaded code
// object until the process ends. In host code the array's name only names the
// symbol; its device address comes from hipGetSymbolAddress, looked up once
// per device with that device current, and only that address is passed to
// the kernels. Every call on one GPU shares the array (calls that overlap on
// one GPU race); nothing in it needs clearing between calls (the planes and
// the partial slices are written whole before they are read).
static __device__ __align__(256) uint8_t scratch[TIQ_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_addr[kMaxDevices];
std::mutex g_scratch_mu;

// The scratch address on the device that runs `stream`.
int noalloc_scratch(hipStream_t stream, void** out) {
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return status_of(e);
    int dev = cur;
    if (stream) {
        e = hipStreamGetDevice(stream, &dev);
        if (e != hipSuccess) return status_of(e);
    }
    if (dev < 0 || dev >= kMaxDevices) return TIQ_EUNSUPPORTED;
    void* p = g_scratch_addr[dev].load(std::memory_order_acquire);
    if (p) {
        *out = p;
        return TIQ_OK;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_addr[dev].load(std::memory_order_relaxed);
    if (!p) {
        if (dev != cur && (e = hipSetDevice(dev)) != hipSuccess) return status_of(e);
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        const hipError_t back = dev != cur ? hipSetDevice(cur) : hipSuccess;
        if (e != hipSuccess) return status_of(e);
        if (back != hipSuccess) return status_of(back);
        if (!p) return TIQ_EINVAL;
        g_scratch_addr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return TIQ_OK;
}

}  // namespace

extern "C" int tiq_decode_linear(const float* x, int64_t ldx, const uint16_t* x_planes, int64_t M, int64_t K,
                                 const void* w, int w_format, const float* scale, const float* bias, int64_t N,
                                 float* y, int64_t ldy, const float* ln_weight, const float* ln_bias, float ln_eps,
                                 int activation, const float* residual, int64_t ld_residual,
                                 const float* next_ln_weight, const float* next_ln_bias, float next_ln_eps,
                                 uint16_t* planes_out, void* workspace, size_t workspace_bytes, void* stream) {
    if (w_format != TIQ_WF_INT8 && w_format != TIQ_WF_INT8_TILED && w_format != TIQ_WF_INT4_TILED &&
        w_format != TIQ_WF_F32 && w_format != TIQ_WF_F32_TILED)
        return TIQ_EUNSUPPORTED;
    if (activation != TIQ_ACT_NONE && activation != TIQ_ACT_GELU_TANH) return TIQ_EINVAL;
    if ((ln_weight == nullptr) != (ln_bias == nullptr)) return TIQ_EINVAL;
    if (M < 0 || K < 0 || N < 0) return TIQ_EINVAL;
    if (M == 0 || N == 0) return TIQ_OK;
    const bool f32w = w_format == TIQ_WF_F32 || w_format == TIQ_WF_F32_TILED;
    if (!w || (!f32w && !scale)) return TIQ_EINVAL;
    if (x_planes && ln_weight) return TIQ_EINVAL;  // planes already carry their LayerNorm
    if (!x_planes && (!x || ldx < K)) return TIQ_EINVAL;
    if (y && ldy < N) return TIQ_EINVAL;
    if (residual && (!y || ld_residual < N)) return TIQ_EINVAL;
    const WFormat fmt = (WFormat)w_format;
    LinearArgs a = make_args(x, TIQ_F32, M, K, ldx, static_cast<const uint8_t*>(w), fmt == kF32 ? 4 * K : K, scale,
                             nullptr, 0, bias, N, y, TIQ_F32, ldy, stream, fmt);
    a.fuse.ln_w = ln_weight;
    a.fuse.ln_b = ln_bias;
    a.fuse.ln_eps = ln_eps;
    a.fuse.act = activation;
    a.fuse.res = residual;
    a.fuse.ldr = ld_residual;
    a.ws = workspace;
    a.ws_bytes = workspace_bytes;
    return run_decode_linear(a, x_planes, next_ln_weight, next_ln_bias, next_ln_eps, planes_out);
}

extern "C" int tiq_decode_linear_noalloc(const float* x, int64_t ldx, const uint16_t* x_planes, int64_t M,
                                         int64_t K, const void* w, int w_format, const float* scale,
                                         const float* bias, int64_t N, float* y, int64_t ldy,
                                         const float* ln_weight, const float* ln_bias, float ln_eps, int activation,
                                         const float* residual, int64_t ld_residual, const float* next_ln_weight,
                                         const float* next_ln_bias, float next_ln_eps, uint16_t* planes_out,
                                         void* stream) {
    // the workspace tiq_decode_linear may use for this shape, against the fixed
    // array (host arithmetic only: nothing is launched for a refused request)
    if (tiq_decode_linear_workspace(w_format, M, K, N) > TIQ_NOALLOC_SCRATCH_BYTES) return TIQ_ESCRATCH;
    void* ws = nullptr;
    if (M > 0 && N > 0) {
        const int rc = noalloc_scratch(as_stream(stream), &ws);
        if (rc != TIQ_OK) return rc;
    }
    return tiq_decode_linear(x, ldx, x_planes, M, K, w, w_format, scale, bias, N, y, ldy, ln_weight, ln_bias, ln_eps,
                             activation, residual, ld_residual, next_ln_weight, next_ln_bias, next_ln_eps, planes_out,
                             ws, TIQ_NOALLOC_SCRATCH_BYTES, stream);
}
