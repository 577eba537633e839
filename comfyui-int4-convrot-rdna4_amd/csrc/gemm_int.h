// Int8-MFMA GEMM on 64 UA x 64 UB tiles of waves of 64 x 64 or 128 x 64 outputs:
// the W8A8 GEMM on grids the 256 x 256 kernel leaves mostly idle, and the
// packed-int4 GEMM of widths that are no multiple of 128.
//
// A stage of the LDS ring is the tile's 64-row units (4 KB: 64 operand bytes a
// row) of one 64-byte block, copied by global_load_lds_dwordx4, in the chunk
// image of I8T (b6t_layout.h: row r at 64 r, 16-byte piece c at swz(r, c)).  I8T
// units are contiguous; row-major packed int4 is swizzled on the global side.
// The two-phase schedule is that of the bf6 small-tile kernel (gemm_bf6.hip):
// phase A multiplies k step 0 of a block and reads the fragments of step 1,
// phase B the reverse for the next block; the copies of the block NST-1 ahead
// go out in three parts of each phase, and one barrier per block hands its
// stage over.  Accumulators are exact int32 (packed int4: 256 acc, operands are
// 16 q), so tiles, splits and order do not show in the outputs.
//
// SPLIT: workgroup b takes tile b % T and the blocks [s nkb / S, (s+1) nkb / S)
// of split s = b / T, stores its int32 partial in the workspace (device-scope
// accesses) and draws a ticket from the tile's counter; the last one adds the
// other partials to its own, clears the counter and runs the epilogue.  No
// workgroup waits for another.
#pragma once

#include <type_traits>

#include "gemm_direct.h"

namespace convrot {

constexpr int IN_UNIT = 4096;                            // 64 rows x 64 bytes

// FM: 32-row tiles of A per wave (2: 64 x 64 outputs, 4: 128 x 64, which reads a
// quarter fewer fragment bytes per product; packed int4 keeps 2: with one wave per
// SIMD nothing hides the unpack, 1024 x 1600 -> 4800 15.3 us against 18.5).
template <int UA, int UB, int NST_, int FM = 2>
struct IntTile {
    static constexpr int NST = NST_;
    static constexpr int BM = 64 * UA, BN = 64 * UB;
    static constexpr int WAVES = UA * UB * 2 / FM, THREADS = 64 * WAVES;
    static constexpr int STAGE = (UA + UB) * IN_UNIT;
    static constexpr int LOADS = 4 * (UA + UB) / WAVES;  // copies per wave and block
    static constexpr int RING = NST * STAGE;
    static constexpr int LDS_BYTES = RING + EPI_SCALE_FLOATS * 4 + 16;
    static_assert(4 * (UA + UB) % WAVES == 0 && (NST - 1) * LOADS <= 63 && NST >= 3, "copies");
    static_assert(THREADS >= 256 && BM <= 256 && BN <= 256, "staged scales");
    static_assert(RING / WAVES >= 32 * (64 * 4 + 16), "epilogue scratch");
};

template <int KIND, int EPI, int LR, bool SPLIT, int UA, int UB, int NST_, int FM>
__global__ __launch_bounds__(128 * UA * UB / FM) void gemm_int_kernel(
        const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, const float* __restrict__ xs,
        const float* __restrict__ ws, const void* __restrict__ bias, int bias_dt, void* __restrict__ out, int M, int N,
        int K, LoraArgs lora, int gm, int nsplit, int* __restrict__ part, unsigned* __restrict__ cnt) {
    using S = IntTile<UA, UB, NST_, FM>;
    static_assert(FM == 2 || !SPLIT, "the partial exchange is laid out for 64 x 64 waves");
    constexpr int NST = S::NST;
    extern __shared__ __attribute__((aligned(16))) uint8_t ilds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / UB, wn = wave % UB;
    const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
    const int Kb = KIND == KIND_P4 ? K / 2 : K;          // operand bytes per row
    const int nkb_all = (Kb + 63) / 64;                  // packed int4: the last block may be a half one
    int tm, tn, kb0 = 0, nkb = nkb_all, split = 0, tix = blockIdx.x;
    if constexpr (SPLIT) {
        const int T = tiles_m * tiles_n;
        split = blockIdx.x / T;
        tix = blockIdx.x - split * T;
        kb0 = (int)((long long)split * nkb_all / nsplit);
        nkb = (int)((long long)(split + 1) * nkb_all / nsplit) - kb0;
    }
    tile_of_block(tix, tiles_m, tiles_n, gm, tm, tn);
    const int m0 = tm * S::BM, n0 = tn * S::BN;

    float* sc = reinterpret_cast<float*>(ilds + S::RING);
    ScaleRegs scr;
    scr.load(xs, ws, bias, bias_dt, M, N, m0, n0, tid);

    // Copy j of this wave is KB i % 4 of unit i / 4 (A units, then B units), i =
    // wave LOADS + j.  I8T units past the padded rows repeat the last one, rows of
    // packed int4 past the last row that row: their outputs are never stored.
    const uint8_t* csrc[S::LOADS];
    uint32_t cdst[S::LOADS], ck[S::LOADS];
    const int last_a = ((M + 255) >> 8) * 4 - 1, last_b = ((N + 255) >> 8) * 4 - 1;
#pragma unroll
    for (int j = 0; j < S::LOADS; ++j) {
        const int ins = wave * S::LOADS + j, u = ins / 4, o = ins % 4;
        const bool is_a = u < UA;
        if constexpr (KIND == KIND_P4) {
            const int rl = (is_a ? u : u - UA) * 64 + o * 16 + (lane >> 2);
            const int row = is_a ? min(m0 + rl, M - 1) : min(n0 + rl, N - 1);
            csrc[j] = (is_a ? A : B) + (size_t)row * Kb;
            ck[j] = swz(rl, lane & 3) * 16;
        } else {
            const int gr = is_a ? min((m0 >> 6) + u, last_a) : min((n0 >> 6) + u - UA, last_b);
            csrc[j] = (is_a ? A : B) + ((size_t)(gr >> 2) * nkb_all + kb0) * I8T_CHUNK + (gr & 3) * IN_UNIT + o * 1024 +
                      lane * 16;
            ck[j] = 0;
        }
        cdst[j] = (uint32_t)(uintptr_t)ilds + u * IN_UNIT + o * 1024;
    }
    auto dma_one = [&](int kb, int j) __attribute__((always_inline)) {
        const uint32_t dst = cdst[j] + (kb % NST) * S::STAGE;
        if constexpr (KIND == KIND_P4)   // the pieces past the row's end (a half block) repeat its last one
            dma16(dst, csrc[j] + min((uint32_t)min(kb, nkb - 1) * 64 + ck[j], (uint32_t)Kb - 16));
        else
            dma16(dst, csrc[j] + (size_t)min(kb, nkb - 1) * I8T_CHUNK);
    };
    constexpr int LOADS_B = S::LOADS / 2, LOADS_A = S::LOADS - LOADS_B;
    auto dma_part = [&](int kb, int t, int first, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int j = n * (t - 1) / 3; j < n * t / 3; ++j) dma_one(kb, first + j);
    };

    v16i acc[FM][2];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (v16i){0};
    const int l32 = lane & 31, h = lane >> 5;
    uint32_t offa[2], offb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        offa[s] = wm * (FM / 2) * IN_UNIT + i8t_off(l32, 2 * s + h);
        offb[s] = (UA + wn) * IN_UNIT + i8t_off(l32, 2 * s + h);
    }
    struct Frags { v4u_d a[FM], b[2]; };
    auto read_one = [&](uint32_t st, int s, int r, Frags& f) __attribute__((always_inline)) {
        const uint8_t* base = ilds + st;
        if (r < FM) f.a[r] = *reinterpret_cast<const v4u_d*>(base + offa[s] + r * 2048);
        else f.b[r - FM] = *reinterpret_cast<const v4u_d*>(base + offb[s] + (r - FM) * 2048);
    };
    auto reads_after = [&](int t, uint32_t st, int s, Frags& f) __attribute__((always_inline)) {
        if (t == 0) { read_one(st, s, 0, f); read_one(st, s, FM, f); }
        if (t == 1) read_one(st, s, FM + 1, f);
        if (t >= 2 && t <= FM) read_one(st, s, t - 1, f);
    };
    // slot t of a k step: A tile (t / 2) % FM against B tile t % 2 (transposed).  Packed
    // int4 has twice as many: the first 8 bytes of every fragment, then the last 8, so that
    // four MFMAs lie between two on one accumulator (1024 x 1600 -> 4800 16.1 -> 15.5
    // us against the two halves back to back, MI355X).
    constexpr int SLOTS = KIND == KIND_P4 ? 4 * FM : 2 * FM;
    auto lo = [](v4u_d x) { return (v4i){(int)((x.x << 4) & 0xF0F0F0F0u), (int)(x.x & 0xF0F0F0F0u),
                                         (int)((x.y << 4) & 0xF0F0F0F0u), (int)(x.y & 0xF0F0F0F0u)}; };
    auto hi = [](v4u_d x) { return (v4i){(int)((x.z << 4) & 0xF0F0F0F0u), (int)(x.z & 0xF0F0F0F0u),
                                         (int)((x.w << 4) & 0xF0F0F0F0u), (int)(x.w & 0xF0F0F0F0u)}; };
    auto mfma_slot = [&](const Frags& f, int t) __attribute__((always_inline)) {
        const int i = (t >> 1) % FM, j = t & 1;
        if constexpr (KIND == KIND_P4) {
            if (t < 2 * FM) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo(f.b[j]), lo(f.a[i]), acc[i][j], 0, 0, 0);
            else acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi(f.b[j]), hi(f.a[i]), acc[i][j], 0, 0, 0);
        } else {
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(v4i, f.b[j]),
                                                             __builtin_bit_cast(v4i, f.a[i]), acc[i][j], 0, 0, 0);
        }
    };

    Frags F0, F1;
#pragma unroll
    for (int b = 0; b < NST - 1; ++b)
#pragma unroll
        for (int j = 0; j < S::LOADS; ++j) dma_one(b, j);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((NST - 2) * S::LOADS));   // block 0 landed
    __syncthreads();
#pragma unroll
    for (int j = 0; j < LOADS_B; ++j) dma_one(NST - 1, j);         // the rest in phase A of block 0
#pragma unroll
    for (int r = 0; r < FM + 2; ++r) read_one(0, 0, r, F0);
    // packed int4: the last block holds one k step only when K % 128 == 64
    const bool half = KIND == KIND_P4 && Kb % 64 != 0;
    uint32_t st_cur = 0;
    for (int kb = 0; kb < nkb; ++kb) {
        const uint32_t st_nxt = st_cur == (NST - 1) * S::STAGE ? 0u : st_cur + S::STAGE;
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            mfma_slot(F0, t);
            __builtin_amdgcn_sched_barrier(0);
            if (t >= 1 && t < 4) dma_part(kb + NST - 1, t, LOADS_B, LOADS_A);
            reads_after(t, st_cur, 1, F1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // this wave's copies of block kb+1 landed, its reads of block kb done
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((NST - 2) * S::LOADS) & 0xc07f);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (KIND == KIND_P4 && half && kb == nkb - 1) break;
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            mfma_slot(F1, t);
            __builtin_amdgcn_sched_barrier(0);
            if (t >= 1 && t < 4) dma_part(kb + NST, t, 0, LOADS_B);
            reads_after(t, st_nxt, 0, F0);
            __builtin_amdgcn_sched_barrier(0);
        }
        st_cur = st_nxt;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));                      // the copies past the end have landed
    __syncthreads();                                               // every wave is done with the stages
    if constexpr (SPLIT) {
        // Partial of split s: value q of a lane is acc[q / 32][(q / 16) % 2][q % 16], at
        // part[((s T + tile) WAVES + wave) 4096 + 64 q + lane]; stored and loaded past the
        // XCDs' L2 caches, ordered before the ticket by each wave's vmcnt(0) and the barrier.
        const int T = tiles_m * tiles_n;
        auto slot = [&](int s) { return part + ((size_t)(s * T + tix) * S::WAVES + wave) * 4096 + lane; };
        int* dst = slot(split);
#pragma unroll
        for (int q = 0; q < 64; ++q)
            __hip_atomic_store(dst + q * 64, acc[q >> 5][(q >> 4) & 1][q & 15], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __syncthreads();
        unsigned* ticket = reinterpret_cast<unsigned*>(ilds + S::RING + EPI_SCALE_FLOATS * 4);
        if (tid == 0) *ticket = __hip_atomic_fetch_add(cnt + tix, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket != (unsigned)nsplit - 1) return;               // another split finishes this tile
        if (tid == 0) __hip_atomic_store(cnt + tix, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int s = 0; s < nsplit; ++s) {
            if (s == split) continue;
            const int* src = slot(s);
            int p[64];
#pragma unroll
            for (int q = 0; q < 64; ++q) p[q] = __hip_atomic_load(src + q * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int q = 0; q < 64; ++q) acc[q >> 5][(q >> 4) & 1][q & 15] += p[q];
        }
    }
    scr.store(sc, bias, bias_dt, M, N, m0, n0, tid);
    __syncthreads();
    constexpr int SCR = S::RING / S::WAVES;
    epilogue_lds<EPI, FM, 2, LR, SCR, KIND == KIND_P4 ? 8 : 0, true>(acc, sc, out, M, N, m0, n0, m0 + wm * 32 * FM,
                                                                    n0 + wn * 64, lane, lora, ilds + wave * SCR);
}

// One launch, split nsplit ways (nsplit > 1: part holds nsplit partials per tile, cnt one counter).
template <int KIND, int EPI, int LR, bool SPLIT, int UA, int UB, int NST, int FM = 2>
static hipError_t int_launch(const uint8_t* A, const uint8_t* B, const float* xs, const float* ws, const void* bias,
                             int bias_dt, void* out, int M, int N, int K, const LoraArgs& la, int nsplit, int* part,
                             unsigned* cnt, int dev, hipStream_t st) {
    using S = IntTile<UA, UB, NST, FM>;
    auto kern = &gemm_int_kernel<KIND, EPI, LR, SPLIT, UA, UB, NST, FM>;
    static std::atomic<bool> attr[kMaxDev];
    const hipError_t e = lds_limit_once(attr, dev, reinterpret_cast<const void*>(kern), S::LDS_BYTES);
    if (e != hipSuccess) return e;
    const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
    hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n * (SPLIT ? nsplit : 1)), dim3(S::THREADS), S::LDS_BYTES, st, A, B,
                       xs, ws, bias, bias_dt, out, M, N, K, la, tile_group_rows(tiles_m), nsplit, part, cnt);
    return hipGetLastError();
}

}  // namespace convrot
