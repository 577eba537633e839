// Launches of the direct (register-fed) GEMM on B6T operands: W4A4 products of
// at most 256 rows.

#include "gemm_direct.h"

namespace convrot {

// Tile of a direct launch for M x N x K, 0 x 0 where the staged kernels
// (gemm_bf6.hip) are the better choice.  The tile shrinks until the grid fills
// the CUs once: a workgroup's time is its operand bytes (28 per clock and CU)
// plus about 3 us, so the smallest tile that still fits 256 workgroups wins, and
// a second round costs a whole one.  Measured on MI355X (bursts, bf16 out, us),
// K = 3072: 1 x 3072 32x32 4.3, 32x64 4.8 (96 and 48 workgroups), 1 x 12288 5.9
// and 4.8 (384 and 192), staged 128x128 12.3 and 12.7; 128 x 3072 64x32 5.1,
// 64x64 6.5 (192, 96), staged 12.7; 256 x 3072 64x32 8.9, 64x64 6.7 (384, 192),
// staged 12.7; 256 x 6144 64x64 12.0, 128x64 10.7 (384, 192), staged 13.5; 256 x
// 9216 128x64 20.7 (288) loses to the staged tiles' 16.  At K = 12288 the 128x64
// tile (96 workgroups 32.1) loses to the staged split, 64x64 (256 x 3072: 19.2)
// does not.  All k ranges are multiplied at once by eight waves, two blocks of
// loads in flight each; four waves or more blocks in flight measured slower.
void gemm_bf6_direct_tile(int M, int N, int K, int* bm, int* bn) {
    auto up = [](int v, int t) { return (long long)((v + t - 1) / t); };
    *bm = *bn = 0;
    if (M > 256) return;
    if (M <= 32) { *bm = 32; *bn = up(N, 32) <= 256 ? 32 : 64; return; }
    if (up(M, 64) * up(N, 32) <= 256) { *bm = 64; *bn = 32; return; }
    if (up(M, 64) * up(N, 64) <= 256) { *bm = 64; *bn = 64; return; }
    if (K <= 4096 && M > 64 && up(M, 128) * up(N, 64) <= 256) { *bm = 128; *bn = 64; }
}

template <int EPI, bool LORA>
static hipError_t run(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws, const void* bias,
                      int bias_dt, void* out, int M, int N, int K, const LoraArgs& la, hipStream_t st) {
    int dev = 0, bm = 0, bn = 0;
    const hipError_t e = current_device(&dev);
    if (e != hipSuccess) return e;
    gemm_bf6_direct_tile(M, N, K, &bm, &bn);
#define RUN(FM, FN, WM, WK)                                                                                        \
    return direct_launch<KIND_B6T, EPI, LORA, FM, FN, WM, 1, WK, 2>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, dev, st)
    if (bm == 32 && bn == 32) RUN(1, 1, 1, 8);
    if (bm == 32 && bn == 64) RUN(1, 2, 1, 8);
    if (bm == 64 && bn == 32) RUN(2, 1, 1, 8);
    if (bm == 64 && bn == 64) RUN(2, 2, 1, 8);
    if (bm == 128) RUN(2, 2, 2, (LORA ? 3 : 4));      // the LoRA sums take a partial's place in LDS
#undef RUN
    return hipErrorInvalidValue;
}

hipError_t gemm_bf6_direct_launch(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws,
                                  const void* bias, int bias_dt, void* out, int M, int N, int K, const LoraArgs& la,
                                  int epi, hipStream_t st) {
    if (la.R == 0) {
        switch (epi) {
            case EPI_F32: return run<EPI_F32, false>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_BF16: return run<EPI_BF16, false>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_BF16_EAGER: return run<EPI_BF16_EAGER, false>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_ACC: return run<EPI_ACC, false>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            case EPI_F16: return run<EPI_F16, false>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
            default: return hipErrorInvalidValue;
        }
    }
    switch (epi) {
        case EPI_F32: return run<EPI_F32, true>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_BF16: return run<EPI_BF16, true>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_BF16_EAGER: return run<EPI_BF16_EAGER, true>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        case EPI_F16: return run<EPI_F16, true>(A, B, xs, ws, bias, bias_dt, out, M, N, K, la, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace convrot
