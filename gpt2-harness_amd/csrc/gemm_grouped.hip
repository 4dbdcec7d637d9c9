// Group-wise int4 prefill GEMM on the register-staged kernel (gfx950): the
// library's own group-wise format (nibbles as the reference's int4 rows,
// quantization.py:132-149, one fp16 scale per row and group of 128 columns)
// behind the reference's quantized Linears over a whole prompt
// (model.py:254,319,352,355 with M = B*T):
//     y[m, n] = sum_g s[n, g] * sum_{k in g} x[m, k] * q[n, k] + bias[n]
// Built without -amdgpu-mfma-vgpr-form: the MFMAs accumulate a group's
// partial tiles in AGPRs, and the scaled sums, which only vector instructions
// touch, stay in VGPRs.
#include <algorithm>

#include "tiq_internal.hpp"

namespace tiq {
namespace {

#include "gemm_staged_kernel.hpp"

constexpr int kGroup = 128;  // two k64 steps
constexpr int kBN = 128;

// 128 x 128 tiles, two workgroups a CU (the partial and the summed tiles fit 256
// registers), whose loads and folds hide beside each other's MFMAs: ahead of one
// 224 x 128 workgroup a CU at every GPT-2 shape and row count (us, 224 rows / 128:
// 1600 x 4800 M = 4096 90 / 78, 1600 x 6400 M = 4096 119 / 104, 1024 x 4096 M =
// 2048 42 / 23, 768 x 768 M = 1024 17 / 11).
constexpr int kBM = 128;

// One workgroup per tile (the group-wise kernel does not run persistent);
// gridDim.z = S splits of whole groups, fp32 slices without bias when S > 1.
template <typename TY>
int run_w4g(const LinearArgs& a, TY* y, int64_t ldy, const float* bias, int64_t S) {
    const int64_t tiles = ((a.M + kBM - 1) / kBM) * ((a.N + kBN - 1) / kBN);
    const int ngroups = (int)((a.K + kGroup - 1) / kGroup);
    hipLaunchKernelGGL((gemm_staged<kBM, kBN, 1, kW4G, TY, false, 2, 2>), dim3((unsigned)tiles, 1, (unsigned)S), dim3(256), 0,
                       a.stream, static_cast<const uint16_t*>(a.x), a.ldx, a.w, a.ldw, nullptr, bias, y, ldy,
                       (int)a.M, (int)a.N, (int)a.K, (int)a.K, a.scale16, ngroups, nullptr);
    return launch_status();
}

}  // namespace

bool staged_w4g_supported(const LinearArgs& a) {
    if (a.fmt != kW4G || a.x_dtype != TIQ_BF16 || a.group != kGroup || (a.kw && a.kw != a.K)) return false;
    if (a.K % BK != 0 || a.ldw != a.K / 2) return false;
    const int unit = a.y_dtype == TIQ_F32 ? 4 : 8;
    if (a.N % unit != 0 || a.ldy % unit != 0 || !aligned(a.y, 16)) return false;
    if (a.N % 32 != 0) return false;  // a 32-column tile is all inside N or all outside
    if ((a.bias && !aligned(a.bias, 16)) || !aligned(a.scale16, 2)) return false;
    if (!aligned(a.x, 16) || a.ldx % 8 != 0 || !aligned(a.w, 16) || a.ldw % 16 != 0) return false;
    // 32-bit byte offsets from the base pointers, 32-bit scale offsets
    if ((a.M - 1) * a.ldx * 2 + a.K * 2 > 0xffffffffLL || (a.N - 1) * a.ldw + a.K / 2 > 0xffffffffLL) return false;
    if (a.N * ((a.K + kGroup - 1) / kGroup) * 2 > 0xffffffffLL) return false;
    return true;
}

// Splits of whole groups (at most 8, within the workspace): the one with the least
// time by a model of the timings over GPT-2's shapes at M = 64 .. 4096: per k64
// step 0.585 us with one workgroup on a CU, 0.95 with two; 3.9 us a launch; for
// a split 3.8 us and 0.3 us a MB of slices for the sum. Its choices take 0.6% more
// than the best splits altogether (us, unsplit / chosen: 6400 x 1600 M = 1024 63 /
// 40, M = 512 63 / 27; 3072 x 768 M = 2048 33 / 26; 768 x 2304 M = 256 11.3 / none).
int64_t staged_w4g_splits(int64_t M, int64_t N, int64_t K, size_t ws_bytes) {
    const int64_t tiles = ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN);
    const int64_t groups = (K + kGroup - 1) / kGroup;
    int64_t most = std::min<int64_t>(std::min<int64_t>(512 / std::max<int64_t>(tiles, 1), groups), 8);
    most = std::min<int64_t>(most, (int64_t)(ws_bytes / (size_t)(M * N * 4)));
    int64_t best = 1;
    double best_t = 1e30;
    for (int64_t S = 1; S <= most; ++S) {
        const double steps = 2.0 * (double)((groups + S - 1) / S);
        double t = steps * (tiles * S <= 256 ? 0.585 : 0.95);
        if (S > 1) t += 3.8 + 0.3e-6 * (double)(S * M * N * 4);
        if (t < best_t) best_t = t, best = S;
    }
    return best;
}

int launch_staged_w4g(const LinearArgs& a, void* ws, size_t ws_bytes) {
    if (!staged_w4g_supported(a)) return TIQ_EUNSUPPORTED;
    const int64_t S = (ws && aligned(ws, 16)) ? staged_w4g_splits(a.M, a.N, a.K, ws_bytes) : 1;
    if (S > 1 && a.M * a.N * S <= 0x7fffffffLL) {
        float* part = static_cast<float*>(ws);
        const int rc = run_w4g<float>(a, part, a.N, nullptr, S);
        if (rc != TIQ_OK) return rc;
        return launch_splitk_reduce(a, part, S, nullptr);
    }
    if (a.y_dtype == TIQ_F32) return run_w4g<float>(a, static_cast<float*>(a.y), a.ldy, a.bias, 1);
    return run_w4g<uint16_t>(a, static_cast<uint16_t*>(a.y), a.ldy, a.bias, 1);
}

}  // namespace tiq
