// Launches of the int8-MFMA GEMM on small grids (W8A8 on I8T operands) and of
// the packed-int4 GEMM of widths that are no multiple of 128.

#include "gemm_int.h"

#include <algorithm>

namespace convrot {

hipError_t gemm_i8t_large_launch(const int8_t* X, const int8_t* W, const float* xs, const float* ws, const void* bias,
                                 int bias_dt, void* out, int M, int N, int K, int epi, hipStream_t st);

static long long up(int v, int t) { return (long long)((v + t - 1) / t); }

// Kernel of a W8A8 product: the 256 x 256 tiles (gemm.hip), the 256 x 128 ring,
// the 128 x 128 ring split nsplit ways, or the direct kernel on 64 x 64 or 32 x 32 tiles.  A
// workgroup's time is its operand bytes at the rate of one CU, so the tile
// shrinks until the grid covers the CUs; the direct tiles read more bytes per
// product and win only while k is short or the grid tiny; a split's exchange
// costs about 5 us and pays from 96 blocks of 64 k.  Measured on MI355X (bursts,
// bf16 out, us; 256 x 256 / 128 x 128 / 64 x 64 / 32 x 32): 64 x 3072 -> 3072
// - / 13.4 / 8.4 / 4.6; 256 x 3072 -> 3072 - / 13.7 / 8.0 / 9.5; 512 x 3072 ->
// 3072 - / 13.8 / 13.2 / 15.5; 512 x 3072 -> 12288 and 2048 x 3072 -> 3072 20.5 on
// 128 x 128 (384 workgroups); 512 x 12288 -> 3072 100.6 / 43.6, split in two
// 29.3, in four 27.6 (64 x 64 44.6); 300 x 12288 -> 3072 (72 tiles)
// 42.8, in two 28.3, in three 23.4, in four (288 workgroups) 28.7 - what the rule
// of one workgroup per CU follows, though it gives the 96 tiles of 512 rows two
// ways where four are 1.7 us faster; 256 x 12288 ->
// 3072 28.2 split in two, 20.7 in four, 23.4 on 64 x 64; 1024 x 12288 -> 3072 44.1, split in two 42.5; 1333 x
// 2304 -> 6912 (594 workgroups) 25.6 against about 24 on 256 x 256.  Between
// one and two 128 x 128 workgroups per CU, 256 x 128 tiles of four 128 x 64 waves
// where these fit one per CU (uniform codes, 256 x 256 / 128 x 128 / 256 x 128 of
// 64 x 64 waves / of 128 x 64 waves): 2048 x 3072 -> 3072 33.5 / 26.4 / 25.0 / 23.7,
// 2048 x 12288 -> 3072 102.5 / 90.5 / 84.2 / 77.6; above that the 256 x 256 kernel:
// 4096 x 3072 -> 3072 40.8 / 45.0 / 50.3 / 47.9.
enum : int { I8_LARGE = 0, I8_RING = 1, I8_D64 = 2, I8_D32 = 3, I8_WIDE = 4 };
static int i8t_plan(int M, int N, int K, int* nsplit) {
    const long long t32 = up(M, 32) * up(N, 32), t64 = up(M, 64) * up(N, 64), t128 = up(M, 128) * up(N, 128);
    *nsplit = 1;
    if (t32 <= 256 || (t32 <= 512 && K <= 4096)) return I8_D32;
    if (t64 <= 256 && K <= 4096) return I8_D64;
    if (t128 > 512) return I8_LARGE;
    if (t128 > 256 && up(M, 256) * up(N, 128) <= 256) return I8_WIDE;
    if (K >= 64 * 96) *nsplit = (int)std::max(1ll, std::min(4ll, 256 / t128));   // one workgroup per CU
    return I8_RING;
}

using RingTile = IntTile<2, 2, 4>;

// Split counters, then the partials; 0 for a shape that is not split.
size_t gemm_i8t_workspace(int M, int N, int K) {
    int ns = 1;
    if (i8t_plan(M, N, K, &ns) != I8_RING || ns <= 1) return 0;
    return kSplitCounterBytes + (size_t)ns * up(M, RingTile::BM) * up(N, RingTile::BN) * RingTile::BM * RingTile::BN * 4;
}

template <int EPI>
static hipError_t i8t_run(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws, const void* bias,
                          int bias_dt, void* out, int M, int N, int K, void* workspace, hipStream_t st) {
    int dev = 0, ns = 1;
    const hipError_t e = current_device(&dev);
    if (e != hipSuccess) return e;
    const LoraArgs none{nullptr, nullptr, 0, 0.0f};
    switch (i8t_plan(M, N, K, &ns)) {
        case I8_D32: return direct_launch<KIND_I8T, EPI, false, 1, 1, 1, 1, 8, 4>(A, B, xs, ws, bias, bias_dt, out, M, N, K, none, dev, st);
        case I8_D64: return direct_launch<KIND_I8T, EPI, false, 2, 2, 1, 1, 8, 2>(A, B, xs, ws, bias, bias_dt, out, M, N, K, none, dev, st);
        case I8_WIDE: return int_launch<KIND_I8T, EPI, 0, false, 4, 2, 4, 4>(A, B, xs, ws, bias, bias_dt, out, M, N, K, none, 1, nullptr, nullptr, dev, st);
        case I8_RING: break;
        default: return gemm_i8t_large_launch(reinterpret_cast<const int8_t*>(A), reinterpret_cast<const int8_t*>(B), xs, ws, bias, bias_dt, out, M, N, K, EPI, st);
    }
    if (ns > 1 && workspace != nullptr)
        return int_launch<KIND_I8T, EPI, 0, true, 2, 2, 4>(
                A, B, xs, ws, bias, bias_dt, out, M, N, K, none, ns,
                reinterpret_cast<int*>(reinterpret_cast<uint8_t*>(workspace) + kSplitCounterBytes),
                reinterpret_cast<unsigned*>(workspace), dev, st);
    return int_launch<KIND_I8T, EPI, 0, false, 2, 2, 4>(A, B, xs, ws, bias, bias_dt, out, M, N, K, none, 1, nullptr,
                                                        nullptr, dev, st);
}

// workspace: gemm_i8t_workspace bytes (its counters zero), or NULL for no split
hipError_t gemm_i8t_launch(const int8_t* X, const int8_t* W, const float* xs, const float* ws, const void* bias,
                           int bias_dt, void* out, int M, int N, int K, int epi, void* workspace, hipStream_t st) {
    if (M == 0 || N == 0) return hipSuccess;
    if (K % 64 != 0) return hipErrorInvalidValue;
    const uint8_t* a = reinterpret_cast<const uint8_t*>(X);
    const uint8_t* b = reinterpret_cast<const uint8_t*>(W);
    switch (epi) {
        case EPI_F32: return i8t_run<EPI_F32>(a, b, xs, ws, bias, bias_dt, out, M, N, K, workspace, st);
        case EPI_BF16: return i8t_run<EPI_BF16>(a, b, xs, ws, bias, bias_dt, out, M, N, K, workspace, st);
        case EPI_ACC: return i8t_run<EPI_ACC>(a, b, xs, ws, bias, bias_dt, out, M, N, K, workspace, st);
        case EPI_F16: return i8t_run<EPI_F16>(a, b, xs, ws, bias, bias_dt, out, M, N, K, workspace, st);
        default: return hipErrorInvalidValue;
    }
}

// Packed int4, K % 64 == 0: the direct kernel on 32 x 32 tiles while the grid
// is small, else the ring on 128 x 128 tiles while they cover the CUs once, else
// on 256 x 128.  Measured on MI355X (bursts, bf16 out, us; 32 x 32 / 128 x 128 /
// 256 x 128), K = 1600, N = 4800: M = 1 3.4 / 11.5 / 15.4; 256 8.6 / 12.0 / 15.6
// (1200 direct workgroups); 512 14.2 / 12.5 / 15.7; 1024 24.3 / 23.3 / 16.1 (304
// of 128 x 128); 2048 48.9 / 34.3 / 30.9; 4096 92.0 / 56.2 / 46.4.  The 256 x 256
// tiles staged through registers that these widths ran on took 42.2 at M = 1024.
// The bound of 1536 direct workgroups was measured at this K alone.
template <int EPI, bool LORA>
static hipError_t p4_run(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws, const void* bias,
                         int bias_dt, void* out, int M, int N, int K, const LoraArgs& la, hipStream_t st) {
    int dev = 0;
    const hipError_t e = current_device(&dev);
    if (e != hipSuccess) return e;
    constexpr int LR = LORA ? -1 : 0;
    if (up(M, 32) * up(N, 32) <= 1536)
        return direct_launch<KIND_P4, EPI, LORA, 1, 1, 1, 1, 8, 3>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, dev, st);
    if (up(M, 128) * up(N, 128) <= 256)
        return int_launch<KIND_P4, EPI, LR, false, 2, 2, 4>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, 1, nullptr, nullptr, dev, st);
    return int_launch<KIND_P4, EPI, LR, false, 4, 2, 4>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, 1, nullptr, nullptr, dev, st);
}

hipError_t gemm_p4_launch(const int8_t* Xp, const int8_t* Wp, const float* xs, const float* ws, const void* bias,
                          int bias_dt, void* out, int M, int N, int K, const LoraArgs& la, int epi, hipStream_t st) {
    if (M == 0 || N == 0) return hipSuccess;
    if (K % 64 != 0) return hipErrorInvalidValue;
    const uint8_t* a = reinterpret_cast<const uint8_t*>(Xp);
    const uint8_t* b = reinterpret_cast<const uint8_t*>(Wp);
    if (la.R == 0) {
        switch (epi) {
            case EPI_F32: return p4_run<EPI_F32, false>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_BF16: return p4_run<EPI_BF16, false>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_BF16_EAGER: return p4_run<EPI_BF16_EAGER, false>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_ACC: return p4_run<EPI_ACC, false>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_F16: return p4_run<EPI_F16, false>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            default: return hipErrorInvalidValue;
        }
    }
    switch (epi) {
        case EPI_F32: return p4_run<EPI_F32, true>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_BF16: return p4_run<EPI_BF16, true>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_BF16_EAGER: return p4_run<EPI_BF16_EAGER, true>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_F16: return p4_run<EPI_F16, true>(a, b, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace convrot
