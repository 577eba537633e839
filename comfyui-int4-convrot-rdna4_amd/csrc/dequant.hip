// Dequantization of ConvRot weights back to the original basis (gfx950):
//   out[n, :] = s[n] * (q[n, :] @ H)      per rotation group of G codes
// (H is symmetric and its own inverse; _int4/eager.py:138-151,
// _int4/int8_eager.py:50-57).  The butterflies run on the integer codes, so
// the sum of a group is exact (|sum| <= 256 * 128), and the row scale times
// 1/sqrt(G) (a power of two) is multiplied in once: one fp32 rounding per value.
//
// Bound by HBM: K/2 or K bytes in, 4 K (f32) or 2 K bytes out per row.  A lane
// takes 16 consecutive codes (8 or 16 bytes); the first two base-4 digits of
// the butterfly are in its registers, the others across 4 or 16 lanes through
// an LDS transpose; the results pass through LDS once more so that every store
// instruction writes 1 KB of consecutive bytes.  A wave works alone on 1024
// consecutive codes (whole groups of one or more rows): no workgroup barrier.
// Measured (MI355X, int4 12288 x 3072 to f32, kernel trace): 27.6 us, 6.2 TB/s
// over the 170 MB; the torch composition it replaces took 0.64 ms in ten passes.

#include "common.h"

namespace convrot {

constexpr int DQ_WAVES = 4;
constexpr int DQ_STRIDE = 17;             // words per lane slot of the transpose
constexpr int DQ_PAD = 272;               // words per 256 results of the store staging
constexpr int DQ_WORDS = 64 * DQ_STRIDE;  // = 4 * DQ_PAD
static_assert(DQ_WORDS == 4 * DQ_PAD, "one buffer serves both");

// H4 over the base-4 digit of stride STRIDE of the register index:
// (S - 2d, S - 2c, S - 2b, S - 2a) with S = a + b + c + d
template <int STRIDE>
__device__ __forceinline__ void h4_int(int (&v)[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if ((i / STRIDE) % 4 != 0) continue;
        const int a = v[i], b = v[i + STRIDE], c = v[i + 2 * STRIDE], d = v[i + 3 * STRIDE];
        const int s = a + b + c + d;
        v[i] = s - 2 * d;
        v[i + STRIDE] = s - 2 * c;
        v[i + 2 * STRIDE] = s - 2 * b;
        v[i + 3 * STRIDE] = s - 2 * a;
    }
}

// ODT: DT_F32, DT_BF16 or DT_F16.  nchunks = N * K / 16.
template <int G, int BITS, int ODT>
__global__ __launch_bounds__(64 * DQ_WAVES) void dequant_kernel(const uint8_t* __restrict__ q,
                                                                const float* __restrict__ scale,
                                                                void* __restrict__ out, uint32_t nchunks,
                                                                uint32_t row_chunks) {
    constexpr int LPG = G / 16;           // lanes per rotation group
    __shared__ __attribute__((aligned(16))) int lds[DQ_WAVES][DQ_WORDS];
    const int lane = threadIdx.x & 63;
    int* buf = lds[threadIdx.x >> 6];
    const uint32_t c0 = (blockIdx.x * DQ_WAVES + (threadIdx.x >> 6)) * 64u;   // the wave's first chunk
    if (c0 >= nchunks) return;
    // lanes past the end (whole groups) repeat the last chunk and store nothing
    const uint32_t c = min(c0 + lane, nchunks - 1);
    const float s = scale[c / row_chunks];
    auto load = [&](int (&v)[16]) __attribute__((always_inline)) {
        if constexpr (BITS == 4) {
            const uint2 w = reinterpret_cast<const uint2*>(q)[c];
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = (int)((i < 8 ? w.x : w.y) << (28 - 4 * (i & 7))) >> 28;
        } else {
            const uint4 w4 = reinterpret_cast<const uint4*>(q)[c];
            const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = (int)(w[i >> 2] << (24 - 8 * (i & 3))) >> 24;
        }
    };
    const int gl = lane % LPG, gfirst = lane - gl;
    auto rotate = [&](int (&v)[16]) __attribute__((always_inline)) {
        h4_int<1>(v);
        h4_int<4>(v);
        if constexpr (G != 16) {
#pragma unroll
            for (int i = 0; i < 16; ++i) buf[lane * DQ_STRIDE + i] = v[i];
            wave_sync();
            if constexpr (G == 256) {     // lane gl takes position gl of the group's 16 lanes
#pragma unroll
                for (int m = 0; m < 16; ++m) v[m] = buf[(gfirst + m) * DQ_STRIDE + gl];
                h4_int<1>(v);
            } else {                      // lane gl takes positions 4 gl .. +3 of the group's 4 lanes
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int a = 0; a < 4; ++a) v[a + 4 * b] = buf[(gfirst + b) * DQ_STRIDE + 4 * gl + a];
            }
            h4_int<4>(v);
            wave_sync();
        }
    };
    int v[16];
    load(v);
    rotate(v);
    // A row whose scale is not finite: its products are infinities of the codes' signs
    // (NaN for a code of 0), whose sum is infinite only if every term has one sign.  The
    // rotated signs are +-G there.  In a branch of its own for the whole wave: as selects
    // in every row it cost 2.2 of 33.2 us at 12288 x 3072, as a branch ahead of the rotation
    // (which then waits for the scale) 1.3, here nothing.
    const bool wild = !(fabsf(s) < __builtin_inff());
    const bool any_wild = __builtin_amdgcn_ballot_w64(wild) != 0;
    if (any_wild) [[unlikely]] {
        int t[16];
        load(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = (t[i] > 0) - (t[i] < 0);
        rotate(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = wild ? t[i] : v[i];
    }
    // s - s: 0, and NaN for a scale that is not finite
    const float f = s * (G == 256 ? 1.0f / 16 : G == 64 ? 1.0f / 8 : 1.0f / 4), nan = s - s;
    float* res = reinterpret_cast<float*>(buf);
    auto slot = [&](int e) { return res + (e >> 8) * DQ_PAD + (e & 255); };   // element e of the wave's 1024
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int e = G == 256 ? gl + 16 * i : G == 64 ? 16 * (i >> 2) + 4 * gl + (i & 3) : i;
        *slot(gfirst * 16 + e) = (float)v[i] * f + nan;
    }
    if (any_wild) [[unlikely]] {                   // the sums of one sign
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int e = G == 256 ? gl + 16 * i : G == 64 ? 16 * (i >> 2) + 4 * gl + (i & 3) : i;
            if (wild && (v[i] == G || v[i] == -G)) *slot(gfirst * 16 + e) = v[i] == G ? s : -s;
        }
    }
    wave_sync();
    const size_t e0 = (size_t)c0 * 16;
    const int live = (int)(min(64u, nchunks - c0) * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = j * 256 + lane * 4;
        if (e >= live) continue;
        const float4 r = *reinterpret_cast<const float4*>(slot(e));
        if constexpr (ODT == DT_F32) {
            reinterpret_cast<float4*>(out)[(e0 + e) / 4] = r;
        } else if constexpr (ODT == DT_BF16) {
            reinterpret_cast<uint2*>(out)[(e0 + e) / 4] = make_uint2(pack_bf16x2(r.x, r.y), pack_bf16x2(r.z, r.w));
        } else {
            auto h = [](float a, float b) {
                return (uint32_t)__half_as_ushort(__float2half_rn(a)) |
                       ((uint32_t)__half_as_ushort(__float2half_rn(b)) << 16);
            };
            reinterpret_cast<uint2*>(out)[(e0 + e) / 4] = make_uint2(h(r.x, r.y), h(r.z, r.w));
        }
    }
}

template <int G, int BITS>
static hipError_t dequant_g(const uint8_t* q, const float* s, void* out, int odt, uint32_t nchunks, uint32_t row_chunks,
                            hipStream_t st) {
    const dim3 grid((nchunks + 64 * DQ_WAVES - 1) / (64 * DQ_WAVES)), block(64 * DQ_WAVES);
    switch (odt) {
        case DT_F32: hipLaunchKernelGGL((dequant_kernel<G, BITS, DT_F32>), grid, block, 0, st, q, s, out, nchunks, row_chunks); break;
        case DT_BF16: hipLaunchKernelGGL((dequant_kernel<G, BITS, DT_BF16>), grid, block, 0, st, q, s, out, nchunks, row_chunks); break;
        case DT_F16: hipLaunchKernelGGL((dequant_kernel<G, BITS, DT_F16>), grid, block, 0, st, q, s, out, nchunks, row_chunks); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t dequant_launch(const void* q, int bits, const float* s, void* out, int odt, int N, int K, int G,
                          hipStream_t st) {
    if (N == 0) return hipSuccess;
    const uint8_t* p = reinterpret_cast<const uint8_t*>(q);
    const uint32_t rc = (uint32_t)(K / 16), n = (uint32_t)N * rc;
#define DQ_G(GV) bits == 4 ? dequant_g<GV, 4>(p, s, out, odt, n, rc, st) : dequant_g<GV, 8>(p, s, out, odt, n, rc, st)
    switch (G) {
        case 16: return DQ_G(16);
        case 64: return DQ_G(64);
        case 256: return DQ_G(256);
        default: return hipErrorInvalidValue;
    }
#undef DQ_G
}

}  // namespace convrot
