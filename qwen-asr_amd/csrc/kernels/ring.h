// ring.h - the k walk shared by the mid-M GEMMs: a BM x BN tile over bf16
// hi/lo activations and bf16 weights, operands streamed through a ring of LDS
// stages by direct global -> LDS loads (prefill.hip describes the layout).
#pragma once
#include "common.h"

#define QK_GBK 32                 // k per stage

__host__ __device__ constexpr int ring_waves(int bm, int bn) { return bm / 32 * (bn / 64) < 4 ? 4 : bm / 32 * (bn / 64); }
__device__ constexpr int vmcnt_imm(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }

// wait until at most later * LPW of this wave's loads are outstanding
// (later <= MAXL: the stages issued after the one about to be read)
template <int LPW, int MAXL>
__device__ __forceinline__ void ring_wait(int later) {
    if constexpr (MAXL > 0) {
        if (later >= MAXL) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(MAXL * LPW));
            return;
        }
        ring_wait<LPW, MAXL - 1>(later);
    } else {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
}

// 16 bytes per lane from global memory straight into LDS (lane l at byte 16 l
// of the 1 KB at l0).  Called through this helper: with the builtin written in
// the kernel on pointers held in an array, hipcc's host pass drops the
// kernel's launch stub.
__device__ __forceinline__ void lds_load16(const uint16_t *g, unsigned char *l0) {
    __builtin_amdgcn_global_load_lds(g, l0, 16, 0, 0);
}

template <int BM, int BN>
struct RingShape {
    static constexpr int NW = ring_waves(BM, BN), WGM = BM / 32, WGN = NW / WGM, WTN = BN / WGN, TM = 2,
                         TN = WTN / 16;
    static constexpr int AB = BM * 64, STAGE = 2 * AB + BN * 64;   // bytes: one A half, one stage
    static constexpr int GROUPS = (2 * BM + BN) / 16, LPW = GROUPS / NW;
    static_assert(WGM * WGN == NW && WTN % 16 == 0 && GROUPS % NW == 0, "wave grid / load split");
};

// The k walk of one BM x BN tile: nk k tiles of 32 through NST LDS stages.
// issue(kt, st) issues this wave's LPW 1 KB loads of k tile kt into the stage
// at st: A_hi rows [BM][32], A_lo [BM][32] and W [BN][32] in bf16, rows of 64
// bytes, k chunk c of row r in slot c ^ ((r / 2) % 4).  Wave (wm, wn) = (wave /
// WGN, wave % WGN) ends up with rows 32 wm + 16 i + 4 (l >> 4) + r, columns WTN
// wn + 16 j + (l & 15) of the tile (lane l, acc[i][j][r]).
// PAIRED: A rows of 128 bytes, 32 hi then 32 lo values (whole cache lines), chunk c
// of row r in slot c ^ (r % 8).
template <int BM, int BN, int NST, bool PAIRED = false, typename ISSUE>
__device__ __forceinline__ void ring_walk(int nk, unsigned char *lds, f32x4 (&acc)[2][RingShape<BM, BN>::TN],
                                          ISSUE issue) {
    using RS = RingShape<BM, BN>;
    constexpr int WGN = RS::WGN, WTN = RS::WTN, TM = RS::TM, TN = RS::TN;
    constexpr int AB = RS::AB, STAGE = RS::STAGE, LPW = RS::LPW;
    static_assert((NST - 2) * LPW <= 63 && NST * STAGE <= 160 * 1024, "vmcnt / LDS range");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;

#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int fr = lane & 15;
    const int fo = fr * 64 + 16 * ((lane >> 4) ^ ((fr >> 1) & 3));
    const int fp = fr * 128 + 16 * ((lane >> 4) ^ (fr & 7));
    for (int t = 0; t < NST - 1 && t < nk; t++) issue(t, lds + t * STAGE);
    for (int kt = 0; kt < nk; kt++) {
        ring_wait<LPW, NST - 2>(min(nk - 1 - kt, NST - 2));
        // every wave's share of stage kt is in LDS and stage kt - 1 is free (a
        // plain s_barrier: __syncthreads() would also drain the later stages)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kt + NST - 1 < nk) issue(kt + NST - 1, lds + ((kt + NST - 1) % NST) * STAGE);
        const unsigned char *st = lds + (kt % NST) * STAGE;
        bf16x8 bfr[TN];
#pragma unroll
        for (int j = 0; j < TN; j++)
            bfr[j] = *reinterpret_cast<const bf16x8 *>(st + 2 * AB + (wn * WTN + j * 16) * 64 + fo);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int ro = (wm * 32 + i * 16) * (PAIRED ? 128 : 64) + (PAIRED ? fp : fo);
            const bf16x8 ah = *reinterpret_cast<const bf16x8 *>(st + ro);
            const bf16x8 al = *reinterpret_cast<const bf16x8 *>(st + (PAIRED ? ro ^ 64 : AB + ro));
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bfr[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bfr[j], acc[i][j], 0, 0, 0);
        }
    }
}

// The walk for launches of about one block per CU and K a multiple of 64: stages
// of 64 k, rows of 128 bytes, and 2 NW waves, group kg = wave / NW multiplying k
// 32 kg .. + 32 of every stage.  With 64-byte rows a load takes half of each
// cache line and the other half is fetched again a k tile later, which bounds
// the loads of a CU (1200 cycles per 64 k of a 64 x 128 tile, 600 of them MFMAs,
// whether the data is in L2 or not); whole lines halve that, and the two waves
// of a SIMD overlap one's fragment reads with the other's MFMAs.  Measured,
// k walk of a 390 x 3584 x 896 product, one block per CU: 9.4 us plain, 8.0.
// issue(p, st): this wave's LPW2 1 KB loads (8 rows of 128 bytes) of stage p;
// chunk c of row r in slot c ^ (r % 8).  The groups' sums are added at the end
// (group 0's + group 1's), each group finishing one 16-row tile: fin[j][r] is
// row 32 wm + 16 kg + 4 (l >> 4) + r, column WTN wn + 16 j + (l & 15).
template <int BM, int BN>
struct RingShape2 : RingShape<BM, BN> {
    static constexpr int AB2 = BM * 128, STAGE2 = 2 * AB2 + BN * 128;
    static constexpr int GROUPS2 = (2 * BM + BN) / 8, LPW2 = GROUPS2 / (2 * RingShape<BM, BN>::NW);
    static_assert(GROUPS2 % (2 * RingShape<BM, BN>::NW) == 0, "load split");
};

template <int BM, int BN, int NST, typename ISSUE>
__device__ __forceinline__ void ring_walk2(int np, unsigned char *lds, f32x4 (&fin)[RingShape<BM, BN>::TN],
                                           ISSUE issue) {
    using RS = RingShape2<BM, BN>;
    constexpr int NW = RS::NW, WGN = RS::WGN, WTN = RS::WTN, TM = RS::TM, TN = RS::TN;
    constexpr int AB = RS::AB2, STAGE = RS::STAGE2, LPW = RS::LPW2;
    static_assert((NST - 2) * LPW <= 63 && NST * STAGE <= 160 * 1024, "vmcnt / LDS range");
    static_assert(2 * NW * TN * 64 * 16 <= NST * STAGE, "exchange fits the stages");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / NW, wi = wave % NW, wm = wi / WGN, wn = wi % WGN;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int fr = lane & 15;
    const int fo = fr * 128 + 16 * ((4 * kg + (lane >> 4)) ^ (fr & 7));
    for (int t = 0; t < NST - 1 && t < np; t++) issue(t, lds + t * STAGE);
    for (int p = 0; p < np; p++) {
        ring_wait<LPW, NST - 2>(min(np - 1 - p, NST - 2));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (p + NST - 1 < np) issue(p + NST - 1, lds + ((p + NST - 1) % NST) * STAGE);
        const unsigned char *st = lds + (p % NST) * STAGE;
        bf16x8 bfr[TN];
#pragma unroll
        for (int j = 0; j < TN; j++)
            bfr[j] = *reinterpret_cast<const bf16x8 *>(st + 2 * AB + (wn * WTN + j * 16) * 128 + fo);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int ro = (wm * 32 + i * 16) * 128 + fo;
            const bf16x8 ah = *reinterpret_cast<const bf16x8 *>(st + ro);
            const bf16x8 al = *reinterpret_cast<const bf16x8 *>(st + AB + ro);
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bfr[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bfr[j], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();                                           // the stages are free
    f32x4 *x = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
    for (int j = 0; j < TN; j++) {
        fin[j] = kg ? acc[1][j] : acc[0][j];
        x[(wave * TN + j) * 64 + lane] = kg ? acc[0][j] : acc[1][j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TN; j++) fin[j] += x[(((1 - kg) * NW + wi) * TN + j) * 64 + lane];
}

// The k walk of block (blockIdx.x, blockIdx.y, blockIdx.z) of a plain product
// into acc (layout of ring_walk, rows from m0, columns from n0).  lds: NST
// stages of the kernel's shared memory.
template <int BM, int BN, int NST>
__device__ __forceinline__ void ring_tile(const uint16_t *__restrict__ ahi, const uint16_t *__restrict__ alo,
                                          const uint16_t *__restrict__ W, int M, int K, int kc, unsigned char *lds,
                                          f32x4 (&acc)[2][RingShape<BM, BN>::TN]) {
    using RS = RingShape<BM, BN>;
    constexpr int NW = RS::NW, AB = RS::AB, LPW = RS::LPW;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kb = blockIdx.z * kc, ke = min(K, kb + kc);
    const int nk = (ke - kb) / QK_GBK;

    // this lane's load slots: row rr of each of the wave's 16-row groups,
    // k chunk cl (swizzled); rows past M re-read row M - 1 (results dropped)
    const int rr = lane >> 2, cl = (lane & 3) ^ ((rr >> 1) & 3);
    const uint16_t *src[LPW];
    int dst[LPW];
#pragma unroll
    for (int j = 0; j < LPW; j++) {
        const int g = wave + NW * j;
        if (g < BM / 16) {
            src[j] = ahi + (size_t)min(m0 + 16 * g + rr, M - 1) * K + kb + 8 * cl;
            dst[j] = 1024 * g;
        } else if (g < BM / 8) {
            src[j] = alo + (size_t)min(m0 + 16 * (g - BM / 16) + rr, M - 1) * K + kb + 8 * cl;
            dst[j] = AB + 1024 * (g - BM / 16);
        } else {
            src[j] = W + (size_t)(n0 + 16 * (g - BM / 8) + rr) * K + kb + 8 * cl;
            dst[j] = 2 * AB + 1024 * (g - BM / 8);
        }
    }
    ring_walk<BM, BN, NST>(nk, lds, acc, [&](int kt, unsigned char *st) {
#pragma unroll
        for (int j = 0; j < LPW; j++) lds_load16(src[j] + kt * QK_GBK, st + dst[j]);
    });
}

// ring_tile by two k groups (ring_walk2): K and kc multiples of 64
template <int BM, int BN, int NST>
__device__ __forceinline__ void ring_tile2(const uint16_t *__restrict__ ahi, const uint16_t *__restrict__ alo,
                                           const uint16_t *__restrict__ W, int M, int K, int kc, unsigned char *lds,
                                           f32x4 (&fin)[RingShape<BM, BN>::TN]) {
    using RS = RingShape2<BM, BN>;
    constexpr int NW2 = 2 * RS::NW, LPW = RS::LPW2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kb = blockIdx.z * kc, ke = min(K, kb + kc);
    const int r8 = lane >> 3, c8 = (lane & 7) ^ r8;
    const uint16_t *src[LPW];
#pragma unroll
    for (int j = 0; j < LPW; j++) {
        const int g = wave + NW2 * j;                     // A_hi, A_lo, W groups of 8 rows follow one another
        src[j] = (g < BM / 8   ? ahi + (size_t)min(m0 + 8 * g + r8, M - 1) * K
                  : g < BM / 4 ? alo + (size_t)min(m0 + 8 * (g - BM / 8) + r8, M - 1) * K
                               : W + (size_t)(n0 + 8 * (g - BM / 4) + r8) * K) + kb + 8 * c8;
    }
    ring_walk2<BM, BN, NST>((ke - kb) / 64, lds, fin, [&](int p, unsigned char *st) {
#pragma unroll
        for (int j = 0; j < LPW; j++) lds_load16(src[j] + 64 * p, st + 1024 * (wave + NW2 * j));
    });
}
