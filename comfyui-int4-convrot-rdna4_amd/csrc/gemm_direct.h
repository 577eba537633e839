// GEMM kernel for grids too small for the staged 256 x 256 and 128 x 128 tiles:
// every wave loads its MFMA operands from global memory straight into
// registers, and the waves of a workgroup split k as well as the tile.
//
// The staged kernels copy their tiles at the rate one CU reaches (28 bytes per
// clock), so a grid of few large tiles is bound by the CUs it leaves idle, and
// each launch pays about 5 us for filling and draining its LDS ring.  Here the
// tile is WM x WN waves of 32 FM x 32 FN outputs times WK k ranges: small tiles
// give every CU some of the operand bytes, the k ranges keep W = WM WN WK waves
// of loads in flight, and nothing is staged, so the loop has no barrier.  The
// tile layouts (B6T, I8T) put a wave's fragment in whole 64-byte lines that two
// consecutive loads use up.  The partial tiles meet once in LDS (row-major,
// padded rows), where each thread adds the WK partials of four columns of a
// row (exact integers: the order is immaterial) and runs the epilogue on them.
#pragma once

#include "gemm_common.h"

#include <type_traits>

namespace convrot {

// Operand kinds.  KIND_B6T: int4 codes as bf6 (128 k per block, two steps of
// 64).  KIND_I8T: int8 codes, tile-major (64 k per block, two steps of 32).
// KIND_P4: packed int4, row-major (64 k per block, one step; 16 q operands).
enum : int { KIND_B6T = 0, KIND_I8T = 1, KIND_P4 = 2 };

template <int KIND> constexpr int direct_block_k = KIND == KIND_B6T ? 128 : 64;

typedef int v8i_d __attribute__((ext_vector_type(8)));
typedef float v16f_d __attribute__((ext_vector_type(16)));
typedef unsigned v4u_d __attribute__((ext_vector_type(4)));
typedef unsigned v2u_d __attribute__((ext_vector_type(2)));

// A wave's fragments of T 32-row tiles of one operand for one block.
template <int KIND, int T>
struct DirectFrag;

template <int T>
struct DirectFrag<KIND_B6T, T> {
    v4u_d p[T][2];
    v4u_d q2[2];     // T == 2: the Q pieces of the (even, odd) tile pair
    v2u_d q1[2];     // T == 1: this tile's half of them
    // base: the wave's tiles in the operand's chunk of the block; offP / offQ per step
    __device__ __forceinline__ void load(const uint8_t* base, const uint32_t (&offP)[2], const uint32_t (&offQ)[2]) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < T; ++i) p[i][s] = *reinterpret_cast<const v4u_d*>(base + offP[s] + i * 2048);
            if constexpr (T == 2) q2[s] = *reinterpret_cast<const v4u_d*>(base + offQ[s]);
            else q1[s] = *reinterpret_cast<const v2u_d*>(base + offQ[s]);
        }
    }
    // odd: parity of a lone tile (T == 1); a pair is (even, odd)
    __device__ __forceinline__ v8i_d operand(int i, int s, bool odd) const {
        if constexpr (T == 2) {
            const v4u_d a = p[i][s], q = q2[s];
            return i ? (v8i_d){(int)q.z, (int)q.w, (int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0}
                     : (v8i_d){(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)q.x, (int)q.y, 0, 0};
        } else {
            const v4u_d a = p[0][s];
            const v2u_d q = q1[s];
            return odd ? (v8i_d){(int)q.x, (int)q.y, (int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0}
                       : (v8i_d){(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)q.x, (int)q.y, 0, 0};
        }
    }
};

template <int T>
struct DirectFrag<KIND_I8T, T> {
    v4u_d p[T][2];
    __device__ __forceinline__ void load(const uint8_t* base, const uint32_t (&offP)[2], const uint32_t (&)[2]) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < T; ++i) p[i][s] = *reinterpret_cast<const v4u_d*>(base + offP[s] + i * 2048);
    }
};

// D blocks of loads in flight over n blocks: load(d, b) fills register set d with
// block b, mul(d) multiplies it.  The steady loop has no branch around a load (a
// conditional one makes the compiler wait for every younger load as well), and
// no block is loaded twice or past the end.
template <int D, typename L, typename F>
__device__ __forceinline__ void direct_pipeline(int n, L load, F mul) {
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < n) load(d, d);
    __builtin_amdgcn_sched_barrier(0);
    int b = 0;
    for (; b + 2 * D <= n; b += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            mul(d);
            load(d, b + d + D);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
        if (b + d < n) mul(d);
        if (b + d + D < n) load(d, b + d + D);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (b + d + D < n) mul(d);
}

// KIND, epilogue, LoRA term, wave tile (FM x FN 32 x 32 tiles), wave grid
// (WM x WN tiles, WK k ranges), D blocks of loads in flight per wave.
template <int KIND, int EPI, bool LORA, int FM, int FN, int WM, int WN, int WK, int D>
struct DirectGemm {
    static constexpr int TM = 32 * FM * WM, TN = 32 * FN * WN;
    static constexpr int WAVES = WM * WN * WK, THREADS = 64 * WAVES;
    static constexpr int RS = TN + 4;                             // padded row of a partial tile, floats
    static constexpr int PART = TM * RS;                          // floats of one partial
    static constexpr int LDS_BYTES = (WK + (LORA ? 1 : 0)) * PART * 4;
    static_assert(FM <= 2 && FN <= 2 && LDS_BYTES <= 160 * 1024, "tile");
};

// Four outputs of one row from their exact integer accumulators (and LoRA sums).
template <int EPI, bool LORA>
__device__ __forceinline__ void direct_store4(const float (&a)[4], const float (&l)[4], float xsv, const float* ws,
                                              const void* bias, int bias_dt, float lscale, void* out, size_t o, int n,
                                              int N, bool vec) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int c = min(n + e, N - 1);
        const float w = EPI == EPI_ACC ? 0.0f : ws[c];
        const float b = EPI != EPI_ACC && bias ? load_bias(bias, bias_dt, c) : -0.0f;   // x + -0 == x
        if constexpr (EPI == EPI_BF16_EAGER) {
            float t = bf16r(bf16r(a[e]) * bf16r(xsv));
            t = bf16r(t * bf16r(w));
            t = bf16r(t + bf16r(b));
            if constexpr (LORA) t = bf16r(t + bf16r(__fmul_rn(lscale, l[e])));
            v[e] = t;
        } else {
            float t = __fadd_rn(__fmul_rn(__fmul_rn(a[e], xsv), w), b);
            if constexpr (LORA) t = __fadd_rn(t, __fmul_rn(lscale, l[e]));
            v[e] = t;
        }
    }
    if constexpr (EPI == EPI_F32) {
        float* p = reinterpret_cast<float*>(out) + o;
        if (vec) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
        else for (int e = 0; e < 4; ++e) if (n + e < N) p[e] = v[e];
    } else {
        const uint2 h = make_uint2(pack_out2<EPI>(v[0], v[1]), pack_out2<EPI>(v[2], v[3]));
        uint16_t* p = reinterpret_cast<uint16_t*>(out) + o;
        if (vec) *reinterpret_cast<uint2*>(p) = h;
        else for (int e = 0; e < 4; ++e) if (n + e < N) p[e] = (uint16_t)((e < 2 ? h.x : h.y) >> (16 * (e & 1)));
    }
}

template <int KIND, int EPI, bool LORA, int FM, int FN, int WM, int WN, int WK, int D>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_direct_kernel(
        const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, const float* __restrict__ xs,
        const float* __restrict__ ws, const void* __restrict__ bias, int bias_dt, void* __restrict__ out, int M, int N,
        int K, LoraArgs lora, int gm) {
    using S = DirectGemm<KIND, EPI, LORA, FM, FN, WM, WN, WK, D>;
    extern __shared__ __attribute__((aligned(16))) float dlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    int tm, tn;
    tile_of_block(blockIdx.x, (M + S::TM - 1) / S::TM, (N + S::TN - 1) / S::TN, gm, tm, tn);
    const int m0 = tm * S::TM, n0 = tn * S::TN;
    const int nkb = K / direct_block_k<KIND>;
    const int kb0 = wk * nkb / WK, nb = (wk + 1) * nkb / WK - kb0;
    const int l32 = lane & 31, h = lane >> 5;

    // First row of the wave's tiles, clamped to the last whole tile (or pair) of
    // the padded operand: an edge wave past it repeats rows whose outputs are
    // never stored.  A lane past the last row of A reads the last one instead.
    using Acc = std::conditional_t<KIND == KIND_B6T, v16f_d, v16i>;
    Acc acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = (Acc){0};

    if constexpr (KIND == KIND_P4) {
        const int Kb = K / 2;
        const uint8_t* pa[FM];
        const uint8_t* pb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
            pa[i] = A + (size_t)min(m0 + (wm * FM + i) * 32 + l32, M - 1) * Kb + (size_t)kb0 * 32 + h * 16;
#pragma unroll
        for (int j = 0; j < FN; ++j)
            pb[j] = B + (size_t)min(n0 + (wn * FN + j) * 32 + l32, N - 1) * Kb + (size_t)kb0 * 32 + h * 16;
        v4u_d fa[D][FM], fb[D][FN];
        auto load = [&](int d, int kb) __attribute__((always_inline)) {
            const size_t o = (size_t)kb * 32;
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[d][j] = *reinterpret_cast<const v4u_d*>(pb[j] + o);
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[d][i] = *reinterpret_cast<const v4u_d*>(pa[i] + o);
        };
        auto lo = [](v4u_d x) { return (v4i){(int)((x.x << 4) & 0xF0F0F0F0u), (int)(x.x & 0xF0F0F0F0u),
                                             (int)((x.y << 4) & 0xF0F0F0F0u), (int)(x.y & 0xF0F0F0F0u)}; };
        auto hi = [](v4u_d x) { return (v4i){(int)((x.z << 4) & 0xF0F0F0F0u), (int)(x.z & 0xF0F0F0F0u),
                                             (int)((x.w << 4) & 0xF0F0F0F0u), (int)(x.w & 0xF0F0F0F0u)}; };
        auto mul = [&](int d) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo(fb[d][j]), lo(fa[d][i]), acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi(fb[d][j]), hi(fa[d][i]), acc[i][j], 0, 0, 0);
                }
        };
        direct_pipeline<D>(nb, load, mul);
    } else {
        constexpr int CHUNK = KIND == KIND_B6T ? B6_CHUNK : I8T_CHUNK;
        const int tiles_a = ((M + 255) >> 8) * 8, tiles_b = ((N + 255) >> 8) * 8;     // 32-row tiles
        const int ta = min((m0 >> 5) + wm * FM, tiles_a - FM), tb = min((n0 >> 5) + wn * FN, tiles_b - FN);
        const uint8_t* ca = A + ((size_t)(ta >> 3) * nkb + kb0) * CHUNK;
        const uint8_t* cb = B + ((size_t)(tb >> 3) * nkb + kb0) * CHUNK;
        uint32_t offPa[2], offQa[2] = {0, 0}, offPb[2], offQb[2] = {0, 0};
        // the last row of A within the wave's first tile; rows of a second tile are
        // whole (the padding holds codes of 0)
        const int ra = (ta & 7) * 32 + min(l32, max(M - 1 - ta * 32, 0)), rb = (tb & 7) * 32 + l32;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int g = 2 * s + h;
            if constexpr (KIND == KIND_B6T) {
                offPa[s] = b6_p_off(FM == 2 ? (ta & 7) * 32 + l32 : ra, g);
                offQa[s] = b6_q_off(FM == 2 ? (ta & 7) * 32 + l32 : ra, g) + (FM == 1 && (ta & 1) ? 8 : 0);
                offPb[s] = b6_p_off(rb, g);
                offQb[s] = b6_q_off(rb, g) + (FN == 1 && (tb & 1) ? 8 : 0);
            } else {
                offPa[s] = i8t_off(FM == 2 ? (ta & 7) * 32 + l32 : ra, g);
                offPb[s] = i8t_off(rb, g);
            }
        }
        const bool odda = ta & 1, oddb = tb & 1;
        DirectFrag<KIND, FM> fa[D];
        DirectFrag<KIND, FN> fb[D];
        auto load = [&](int d, int kb) __attribute__((always_inline)) {
            const size_t o = (size_t)kb * CHUNK;
            fb[d].load(cb + o, offPb, offQb);
            fa[d].load(ca + o, offPa, offQa);
        };
        auto mul = [&](int d) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        if constexpr (KIND == KIND_B6T)
                            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(   // transposed tile
                                    fb[d].operand(j, s, oddb), fa[d].operand(i, s, odda), acc[i][j], 3, 3, 0,
                                    B6_OPERAND_E8M0, 0, B6_OPERAND_E8M0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                                    __builtin_bit_cast(v4i, fb[d].p[j][s]), __builtin_bit_cast(v4i, fa[d].p[i][s]),
                                    acc[i][j], 0, 0, 0);
                    }
        };
        direct_pipeline<D>(nb, load, mul);
    }

    // partial tiles to LDS: lane l, register r holds row l % 32, column 8 (r / 4) + 4 (l / 32) + r % 4
    {
        float* dst = dlds + wk * S::PART + (wm * FM * 32 + l32) * S::RS + wn * FN * 32 + 4 * h;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const Acc& a = acc[i][j];
                    typedef std::conditional_t<KIND == KIND_B6T, float, int> E;
                    typedef E v4e __attribute__((ext_vector_type(4)));
                    *reinterpret_cast<v4e*>(dst + i * 32 * S::RS + j * 32 + 8 * q) =
                        (v4e){a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
                }
    }
    if constexpr (LORA) {        // t U^T of one 32 x 32 tile per wave, 16 ranks at a time in ascending order
        for (int tl = wave; tl < (S::TM / 32) * (S::TN / 32); tl += S::WAVES) {
            const int i = tl / (S::TN / 32), j = tl % (S::TN / 32);
            const int trow = min(m0 + i * 32 + l32, M - 1), ucol = min(n0 + j * 32 + l32, N - 1);
            f32x16_t la = (f32x16_t){0};
            for (int rk = 0; rk < lora.R; rk += 16) {
                const bf16x8_t t = *reinterpret_cast<const bf16x8_t*>(lora.t + (size_t)trow * lora.R + rk + 8 * h);
                const bf16x8_t u = *reinterpret_cast<const bf16x8_t*>(lora.U + (size_t)ucol * lora.R + rk + 8 * h);
                la = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u, t, la, 0, 0, 0);
            }
            float* dst = dlds + WK * S::PART + (i * 32 + l32) * S::RS + j * 32 + 4 * h;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4*>(dst + 8 * q) = make_float4(la[4 * q], la[4 * q + 1], la[4 * q + 2], la[4 * q + 3]);
        }
    }
    __syncthreads();
    constexpr int ES = epi_bytes<EPI>;
    const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & (4 * ES - 1)) == 0;
#pragma unroll 1
    for (int c = tid; c < S::TM * S::TN / 4; c += S::THREADS) {
        const int r = c / (S::TN / 4), n = n0 + c % (S::TN / 4) * 4, m = m0 + r;
        if (m >= M || n >= N) continue;
        const float* src = dlds + r * S::RS + (n - n0);
        float a[4], l[4] = {0.f, 0.f, 0.f, 0.f};
        int ai[4];
        if constexpr (KIND == KIND_B6T) {
            float4 s = *reinterpret_cast<const float4*>(src);
#pragma unroll
            for (int k = 1; k < WK; ++k) {
                const float4 p = *reinterpret_cast<const float4*>(src + k * S::PART);
                s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
            }
            a[0] = s.x; a[1] = s.y; a[2] = s.z; a[3] = s.w;
            if constexpr (EPI == EPI_ACC) for (int e = 0; e < 4; ++e) ai[e] = (int)a[e];
        } else {
            int4 s = *reinterpret_cast<const int4*>(src);
#pragma unroll
            for (int k = 1; k < WK; ++k) {
                const int4 p = *reinterpret_cast<const int4*>(src + k * S::PART);
                s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
            }
            constexpr int ASH = KIND == KIND_P4 ? 8 : 0;
            ai[0] = s.x >> ASH; ai[1] = s.y >> ASH; ai[2] = s.z >> ASH; ai[3] = s.w >> ASH;
            for (int e = 0; e < 4; ++e) a[e] = (float)ai[e];
        }
        if constexpr (LORA) {
            const float4 p = *reinterpret_cast<const float4*>(src + WK * S::PART);
            l[0] = p.x; l[1] = p.y; l[2] = p.z; l[3] = p.w;
        }
        const size_t o = (size_t)m * N + n;
        if constexpr (EPI == EPI_ACC) {
            for (int e = 0; e < 4; ++e) if (n + e < N) reinterpret_cast<int32_t*>(out)[o + e] = ai[e];
        } else {
            direct_store4<EPI, LORA>(a, l, xs[m], ws, bias, bias_dt, lora.scale, out, o, n, N, vec && n + 4 <= N);
        }
    }
}

template <int KIND, int EPI, bool LORA, int FM, int FN, int WM, int WN, int WK, int D>
static hipError_t direct_launch(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws, const void* bias,
                                int bias_dt, void* out, int M, int N, int K, const LoraArgs& la, int dev,
                                hipStream_t st) {
    using S = DirectGemm<KIND, EPI, LORA, FM, FN, WM, WN, WK, D>;
    auto kern = &gemm_direct_kernel<KIND, EPI, LORA, FM, FN, WM, WN, WK, D>;
    static std::atomic<bool> attr[kMaxDev];
    const hipError_t e = lds_limit_once(attr, dev, reinterpret_cast<const void*>(kern), S::LDS_BYTES);
    if (e != hipSuccess) return e;
    const int tiles_m = (M + S::TM - 1) / S::TM, tiles_n = (N + S::TN - 1) / S::TN;
    hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n), dim3(S::THREADS), S::LDS_BYTES, st, A, B, xs, ws, bias, bias_dt,
                       out, M, N, K, la, tile_group_rows(tiles_m));
    return hipGetLastError();
}

}  // namespace convrot
