// attn_prefill.hip - causal GQA attention over many query rows (the prefill
// half of qwen_causal_attention, reference qwen_asr_kernels.c:1050-1141) on
// the bf16 matrix cores of gfx950, fp32-accurate.
//
// Every fp32 operand x is carried as hi = bf16(x) and lo = bf16(x - hi)
// (together ~16 significant bits; |x - hi - lo| <= 2^-17 |x|), and each
// product a.b is taken as hi_a.hi_b + hi_a.lo_b + lo_a.hi_b on
// v_mfma_f32_16x16x32_bf16 with fp32 accumulation: the dropped lo.lo term and
// the split error leave ~2^-16 relative per product, against 2^-24 for fp32
// products, at a fifth of the matrix-core time of v_mfma_f32_16x16x4_f32.
// Softmax statistics, exponentials and the output stay fp32.
//
// Operand layout of the 16x16x32 bf16 MFMA: lane l supplies A[l & 15][8 (l >> 4)
// + i] and B[8 (l >> 4) + i][l & 15], i = 0..7; the result D[4 (l >> 4) + r][l & 15],
// r = 0..3, lands in lane l.
//
// A block owns one kv head, 64 consecutive queries of both query heads that
// share it (4 waves: head = wave & 1, queries 32 (wave >> 1) .. + 32) and one
// split of the key range (long unsplit prefills: attn_prefill_pp below).  Per 32-key tile staged in LDS (K rows and V^T,
// split into hi / lo once per block):
//   S^T = K Q^T   A = K rows (keys), B = this wave's queries, 32 dims per
//                 k-step; Q is split once, in registers.
//   online softmax per query: a query's 32 scores live in the 4 lanes
//                 l & 15 = query (keys 16 kt + 4 (l >> 4) + r), so the row
//                 max / sum are in-lane over 8 values plus two cross-lane
//                 steps; the rescale factor is lane-local.
//   O^T += V^T P^T  B = the probabilities exactly where S^T left them: k-slot
//                 8 (l >> 4) + i of the MFMA is key 4 (l >> 4) + i (i < 4) and
//                 16 + 4 (l >> 4) + i - 4 (i >= 4), and A = V^T reads the same
//                 keys, so no value crosses lanes.  A V^T row (one dim, 64
//                 bytes) stores the 32 keys in that order, so a lane's 8 keys
//                 are one 16-byte chunk: chunk c of row d sits in slot
//                 c ^ ((d / 2) % 4), and a fragment is one 16-byte read free of
//                 bank conflicts (the swizzle of the ring GEMM's tiles).
// O^T lands as lane l: dims 16 dt + 4 (l >> 4) + r of query l & 15, written
// back as float4 per dt.
//
// Splits: the key range is cut into chunks (a multiple of 32 keys) so the
// launch fills the chip; each split writes unnormalised partials (o[128], m,
// l) and attn_prefill_merge combines them in split order.  Query tiles are
// dispatched longest first (causal tiles grow with the query index).
#include "common.h"
#include "qk_kernels.h"
#include "qwen_asr_hip.h"

#include <math.h>

#define PF_Q 64                   // queries per block (per query head)
#define PF_KT 32                  // keys per LDS tile
// K tile: four 32-dim slices of 32 keys x 64-byte rows (chunk c of key row r
// in slot c ^ ((r / 2) % 4): the fragment reads are the ring GEMM's pattern,
// free of bank conflicts), slices 64 bytes apart beyond their 2 KB so the
// four slices a store instruction touches fall in different banks
#define PF_KSL (PF_KT * 32 + 32)         // bf16 per K slice
#define PF_VLDB PF_KT                     // bf16 row stride of the V^T tiles: 64 B, swizzled chunks
#define PF_MINIT (-1.0e30f)       // running-max start, as the reference's -1e30 (:1069)

__device__ __forceinline__ void pf_split4(float4 v, uint2 &h, uint2 &l) {
    bf16_split2(v.x, v.y, h.x, l.x);
    bf16_split2(v.z, v.w, h.y, l.y);
}

__device__ __forceinline__ void pf_split8(const float *x, bf16x8 &hi, bf16x8 &lo) {
    uint4 h, l;
    bf16_split2(x[0], x[1], h.x, l.x);
    bf16_split2(x[2], x[3], h.y, l.y);
    bf16_split2(x[4], x[5], h.z, l.z);
    bf16_split2(x[6], x[7], h.w, l.w);
    hi = __builtin_bit_cast(bf16x8, h);
    lo = __builtin_bit_cast(bf16x8, l);
}

// hi.hi + hi.lo + lo.hi of one 16x16x32 block
__device__ __forceinline__ f32x4 pf_mfma3(bf16x8 ah, bf16x8 al, bf16x8 bh, bf16x8 bl, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
}

// The next K/V tile, held in registers while the current one is consumed.
// V: lane l of wave w holds dim pf_vdim(w, l, j) of keys 4 pf_vgrp(l) + e: per
// store instruction a wave covers 8 dims x 8 key groups, which the swizzled
// V^T rows take without bank conflicts (the 32 lanes of a half wave land in
// 32 distinct bank pairs).
// Four waves stage a tile: per thread 4 K float4s and 4 V groups of 4 keys.
struct PfStage {
    float4 k[4];   // K rows: float4 (tid + 256 i): key (.. >> 5), dims 4 (.. & 31)
    float v[16];    // V: dim pf_vdim(wave, lane, j), keys 4 pf_vgrp(lane) + e
};

__device__ __forceinline__ int pf_vgrp(int lane) { return (lane >> 2) & 7; }
__device__ __forceinline__ int pf_vdim(int wave, int lane, int j) {
    return 8 * (wave + 4 * j) + (lane & 3) + 4 * (lane >> 5);
}

__device__ __forceinline__ void pf_load(PfStage &st, const float *kb, const float *vb, long ps, int k0, int kend,
                                        int tid) {
    if (k0 + PF_KT <= kend) {                       // a whole tile (block-uniform): no bounds tests
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int idx = tid + 256 * i;
            st.k[i] = *reinterpret_cast<const float4 *>(kb + (size_t)(k0 + (idx >> 5)) * ps + (idx & 31) * 4);
        }
        const int wave = tid >> 6, lane = tid & 63;
        const float *vr = vb + (size_t)(k0 + 4 * pf_vgrp(lane)) * ps;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = pf_vdim(wave, lane, j);
#pragma unroll
            for (int e = 0; e < 4; e++) st.v[4 * j + e] = vr[(size_t)e * ps + d];
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int idx = tid + 256 * i, key = k0 + (idx >> 5);
        st.k[i] = key < kend ? *reinterpret_cast<const float4 *>(kb + (size_t)key * ps + (idx & 31) * 4)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const int wave = tid >> 6, lane = tid & 63, g = pf_vgrp(lane);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int d = pf_vdim(wave, lane, j);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int key = k0 + 4 * g + e;
            st.v[4 * j + e] = key < kend ? vb[(size_t)key * ps + d] : 0.0f;
        }
    }
}

__device__ __forceinline__ int pf_kslot(int key, int c) { return key * 32 + 8 * (c ^ ((key >> 1) & 3)); }

__device__ __forceinline__ void pf_store(const PfStage &st, __bf16 (*sKh)[PF_KSL], __bf16 (*sKl)[PF_KSL],
                                         __bf16 (*sVh)[PF_VLDB], __bf16 (*sVl)[PF_VLDB], int tid) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int idx = tid + 256 * i;
        uint2 h, l;
        pf_split4(st.k[i], h, l);
        // dims 4 (idx & 31) .. + 3 of key idx >> 5: slice (idx & 31) / 8, chunk (idx & 7) / 2, half idx & 1
        const int o = pf_kslot(idx >> 5, (idx & 7) >> 1) + 4 * (idx & 1);
        *reinterpret_cast<uint2 *>(&sKh[(idx & 31) >> 3][o]) = h;
        *reinterpret_cast<uint2 *>(&sKl[(idx & 31) >> 3][o]) = l;
    }
    // keys 4 g .. 4 g + 3 go to chunk g % 4, half g / 4 of the row (key order
    // of the MFMA's k slots, see the header)
    const int wave = tid >> 6, lane = tid & 63, g = pf_vgrp(lane);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int d = pf_vdim(wave, lane, j);
        const int o = 8 * ((g & 3) ^ ((d >> 1) & 3)) + 4 * (g >> 2);
        uint2 h, l;
        pf_split4(make_float4(st.v[4 * j], st.v[4 * j + 1], st.v[4 * j + 2], st.v[4 * j + 3]), h, l);
        *reinterpret_cast<uint2 *>(&sVh[d][o]) = h;
        *reinterpret_cast<uint2 *>(&sVl[d][o]) = l;
    }
}

// 8 bf16 of V^T row d: keys 4 kq .. + 3 and 16 + 4 kq .. + 3 (the keys of this
// lane's scores), chunk kq of the row
__device__ __forceinline__ bf16x8 pf_vrow(const __bf16 *row, int d, int kq) {
    return *reinterpret_cast<const bf16x8 *>(row + 8 * (kq ^ ((d >> 1) & 3)));
}

__device__ __forceinline__ void pf_write_out(const qk_attn_args &a, size_t base, float4 v) {
    if (a.out) {
        *reinterpret_cast<float4 *>(a.out + base) = v;
    } else {
        uint2 h, l;
        pf_split4(v, h, l);
        *reinterpret_cast<uint2 *>(a.out_hi + base) = h;
        *reinterpret_cast<uint2 *>(a.out_lo + base) = l;
    }
}

// 64 queries per block, two blocks per CU
__global__ __launch_bounds__(256, 2) void attn_prefill(qk_attn_args a) {
    constexpr int QT = PF_Q;
    constexpr int hd = QWEN_HIP_HEAD_DIM;
    __shared__ __attribute__((aligned(16))) __bf16 sKh[4][PF_KSL];
    __shared__ __attribute__((aligned(16))) __bf16 sKl[4][PF_KSL];
    __shared__ __attribute__((aligned(16))) __bf16 sVh[hd][PF_VLDB];
    __shared__ __attribute__((aligned(16))) __bf16 sVl[hd][PF_VLDB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ql = lane & 15, kq = lane >> 4;
    const int nq = (a.seq_q + QT - 1) / QT;
    // blocks go out in x order: query tiles longest first, all kv heads of a
    // tile next to each other, so the causal triangle's long tiles start first
    const int t = nq - 1 - (int)blockIdx.x / a.kv_heads;
    const int g = (int)blockIdx.x % a.kv_heads, split = blockIdx.z;
    const int q0 = t * QT;
    const int qn = min(QT, a.seq_q - q0);
    const int kend_tile = min(a.seq_k, a.q_offset + q0 + qn);
    const int ks0 = split * a.chunk;
    if (ks0 >= kend_tile) return;                         // block-uniform
    const int ks1 = min(kend_tile, ks0 + a.chunk);
    const int h = g * 2 + (wave & 1);
    const int qs = q0 + 32 * (wave >> 1);                 // first query of this wave
    const bool wave_on = qs < a.seq_q;
    const int qstride = a.heads * hd;
    const float *kb = a.k + (size_t)g * a.head_stride;
    const float *vb = a.v + (size_t)g * a.head_stride;

    // this lane's query rows (16 per tile qt), dims 32 s + 8 kq .. + 7, split once
    bf16x8 qh[2][4], qo[2][4];
#pragma unroll
    for (int qt = 0; qt < 2; qt++) {
        const int qi = qs + 16 * qt + ql;
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            float4 x0 = make_float4(0.f, 0.f, 0.f, 0.f), x1 = x0;
            if (qi < a.seq_q) {
                const float *qp = a.q + (size_t)qi * qstride + h * hd + 32 * s4 + 8 * kq;
                x0 = *reinterpret_cast<const float4 *>(qp);
                x1 = *reinterpret_cast<const float4 *>(qp + 4);
            }
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            pf_split8(x, qh[qt][s4], qo[qt][s4]);
        }
    }
    f32x4 o[2][8];
#pragma unroll
    for (int qt = 0; qt < 2; qt++)
#pragma unroll
        for (int dt = 0; dt < 8; dt++) o[qt][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m[2] = {PF_MINIT, PF_MINIT}, l[2] = {0.f, 0.f};

    PfStage st;
    pf_load(st, kb, vb, a.pos_stride, ks0, ks1, tid);
    for (int k0 = ks0; k0 < ks1; k0 += PF_KT) {
        __syncthreads();                                  // previous tile fully consumed
        pf_store(st, sKh, sKl, sVh, sVl, tid);
        __syncthreads();
        if (k0 + PF_KT < ks1) pf_load(st, kb, vb, a.pos_stride, k0 + PF_KT, ks1, tid);
        if (!wave_on) continue;

        // scores: s[qt][kt][r] = q(query qs + 16 qt + ql) . k(key k0 + 16 kt + 4 kq + r)
        f32x4 s[2][2];
#pragma unroll
        for (int qt = 0; qt < 2; qt++)
#pragma unroll
            for (int kt = 0; kt < 2; kt++) s[qt][kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
                const int o = pf_kslot(16 * kt + ql, kq);
                const bf16x8 kh = *reinterpret_cast<const bf16x8 *>(&sKh[s4][o]);
                const bf16x8 kl = *reinterpret_cast<const bf16x8 *>(&sKl[s4][o]);
#pragma unroll
                for (int qt = 0; qt < 2; qt++) s[qt][kt] = pf_mfma3(kh, kl, qh[qt][s4], qo[qt][s4], s[qt][kt]);
            }
        }

        // online softmax (causal mask: key <= q_offset + query; keys past ks1 belong elsewhere).
        // A tile wholly below the wave's diagonal and inside the split needs no
        // mask (wave-uniform test; the unmasked scores are the same values).
        // The statistics run in base 2: m holds max(score) * scale * log2(e) and
        // p = 2^(score * scale * log2(e) - m) = e^(score * scale - max), the
        // scale and the subtraction in one fma (the merge takes 2^(m_i - M)).
        const bool open = k0 + PF_KT - 1 <= a.q_offset + qs && k0 + PF_KT <= ks1;
        const float scale2 = a.scale * 1.44269504088896341f;
        float p[2][2][4];
#pragma unroll
        for (int qt = 0; qt < 2; qt++) {
            const int qpos = a.q_offset + qs + 16 * qt + ql;
            float sc[2][4], mx = -INFINITY;
            if (open) {
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        sc[kt][r] = s[qt][kt][r];
                        mx = fmaxf(mx, sc[kt][r]);
                    }
            } else {
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int key = k0 + 16 * kt + 4 * kq + r;
                        sc[kt][r] = (key <= qpos && key < ks1) ? s[qt][kt][r] : -INFINITY;
                        mx = fmaxf(mx, sc[kt][r]);
                    }
            }
            // scaling by a positive factor keeps the maximum where it is
            mx = xor_max16_32(mx) * scale2;
            const float mn = fmaxf(m[qt], mx);
            const float corr = __builtin_amdgcn_exp2f(m[qt] - mn);
            float sum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    p[qt][kt][r] = __builtin_amdgcn_exp2f(fmaf(sc[kt][r], scale2, -mn));
                    sum += p[qt][kt][r];
                }
            sum = xor_sum16_32(sum);
            l[qt] = fmaf(l[qt], corr, sum);
            m[qt] = mn;
            if (!__all(corr == 1.0f)) {          // the running max moved for some query of the wave
#pragma unroll
                for (int dt = 0; dt < 8; dt++) o[qt][dt] *= corr;
            }
        }

        // O^T[d][query] += V^T[d][key] P^T[key][query]; B = this lane's 8 probabilities
        bf16x8 ph[2], po[2];
#pragma unroll
        for (int qt = 0; qt < 2; qt++)
            pf_split8(&p[qt][0][0], ph[qt], po[qt]);
#pragma unroll
        for (int dt = 0; dt < 8; dt++) {
            const bf16x8 vh = pf_vrow(&sVh[16 * dt + ql][0], 16 * dt + ql, kq);
            const bf16x8 vl = pf_vrow(&sVl[16 * dt + ql][0], 16 * dt + ql, kq);
#pragma unroll
            for (int qt = 0; qt < 2; qt++) o[qt][dt] = pf_mfma3(vh, vl, ph[qt], po[qt], o[qt][dt]);
        }
    }
    if (!wave_on) return;

#pragma unroll
    for (int qt = 0; qt < 2; qt++) {
        const int qi = qs + 16 * qt + ql;
        if (qi >= a.seq_q) continue;
        if (a.nsplit == 1) {
            const float inv = l[qt] > 0.0f ? 1.0f / l[qt] : 0.0f;
#pragma unroll
            for (int dt = 0; dt < 8; dt++) {
                const f32x4 v = o[qt][dt];
                pf_write_out(a, (size_t)qi * qstride + h * hd + 16 * dt + 4 * kq,
                             make_float4(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv));
            }
        } else {
            float *pp = a.part + ((size_t)(split * a.seq_q + qi) * a.heads + h) * QK_PF_PART;
#pragma unroll
            for (int dt = 0; dt < 8; dt++) {
                const f32x4 v = o[qt][dt];
                *reinterpret_cast<float4 *>(pp + 16 * dt + 4 * kq) = make_float4(v[0], v[1], v[2], v[3]);
            }
            if (kq == 0) {
                pp[hd] = m[qt];
                pp[hd + 1] = l[qt];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Long unsplit prefills: 8 waves, 128 queries of both query heads of a kv
// head, v_mfma_f32_32x32x16_bf16.  Lane l (hl = l >> 5) of that MFMA supplies
// A[l & 31][8 hl + i] and B[8 hl + i][l & 31], i = 0..7, and holds
// D[8 (r / 4) + 4 hl + r % 4][l & 31], r = 0..15.  Wave w: head w & 1, 32
// queries; per 32-key tile S^T = K Q^T (8 k-steps of 16 dims), softmax, and
// O^T += V^T P^T (4 x 32 dims, 2 k-steps of 16 keys) with the probabilities
// where S^T left them (k-slot 8 hl + i of k-step j is key 16 j + 8 (i / 4) +
// 4 hl + i % 4; a V^T row stores its 32 keys in that order, chunk 2 j + hl
// holding a lane's 8), so a query lives in two lanes and no value crosses
// them but one half-wave swap of the maximum.
//
// A tile is 48 MFMAs (1536 matrix-core cycles) and ~230 VALU operations, which
// one wave issues in about the same time.  Waves that pass the same barriers
// reach their MFMAs together, and then the matrix cores idle while both waves
// of a SIMD run their VALU work.  So the two waves of a SIMD (w and w + 4)
// alternate: a wave's tile is a matrix part (scores of tile i + 1, V^T P^T of
// tile i) and a vector part (softmax of tile i + 1, hi / lo split and LDS stores
// of a later tile, loads of the one after), with one barrier a tile, which
// waves 0..3 (group A) pass after the vector part and waves 4..7 (group B)
// after the matrix part.  Measured, 16 heads: 4096 queries 345 -> 251 us, 8191 queries
// 801 -> 715 us against 16x16x32 MFMAs with all waves in step (0.82 and 1.15
// PFLOP/s of MFMA work; the kernel's own stamps put a tile at ~4600 cycles,
// 3280 of them MFMAs: each wave's chain of matrix and vector part is what
// remains, 1900 + 2450 cycles).
//
// Between barriers q and q + 1 both groups read K q + 1 and V q (matrix part of
// tile q) and store K q + 2 and V q + 1 (the vector part, of tile q in group A
// and of tile q - 1 in group B) into the buffers (two each) of K q and V q - 1,
// which were last read before barrier q.
//
// The scores take their cross terms (hi.lo + lo.hi, 2^-8 of the product)
// first, so the large sums round 8 times a tile and not 24.  (Letting the
// running maximum lag by up to 8 in base 2 spares most rescales of the
// accumulators, 4 % of the time, but then the largest p is no longer exactly 1
// and the error against 64 bits is 3 % larger, so it moves with every maximum.)
// ---------------------------------------------------------------------------
#define PP_QT 128                 // queries per block (per query head)

typedef float pf_f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ pf_f32x16 pf_mfma32(bf16x8 a, bf16x8 b, pf_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// LDS, in bf16: K rows of 256 bytes, 16-byte chunk c of key r in slot
// c ^ (r & 15); V^T row pairs of 128 bytes, chunk c of dim d in slot
// (4 (d & 1) + c) ^ (d / 2 & 7).  Any 8 consecutive rows of a fragment read (16
// bytes per lane over 32 rows) meet 8 different 16-byte slots of 128 bytes.
struct PpLds {
    __attribute__((aligned(16))) uint16_t k[2][2][PF_KT * QWEN_HIP_HEAD_DIM];   // [buffer][hi, lo]
    __attribute__((aligned(16))) uint16_t v[2][2][QWEN_HIP_HEAD_DIM * PF_KT];
};
#define PP_PLANE (2 * PF_KT * QWEN_HIP_HEAD_DIM)       // bytes from hi to lo
#define PP_BUF (2 * PP_PLANE)                          // bytes from a buffer to the next

// One thread's share of a tile (512 threads): K float4s of keys tid / 32 and
// + 16, dims 4 (tid & 31); V dims 2 m, 2 m + 1 of keys 4 g0 + 8 hsel + 16 g2 +
// 0..3.  m = lane bits 0..2, 4..5 and wave bit 0, hsel = lane bit 3, g0 and g2 =
// wave bits 1 and 2: a half wave loads 256 consecutive bytes of a key row, and
// 16 lanes store 8 dims x both halves of a chunk (all banks).
struct PpStage {
    uint4 k[2];
    uint2 v[4];
};
typedef __amdgpu_buffer_rsrc_t pp_rsrc;

// keys [k0, k0 + 32): rows at or past the descriptors' end read as 0 (their
// scores are masked).  The whole offset is in the vector operand: the bounds
// check compares that one with the descriptor's size.
__device__ __forceinline__ void pp_load_k(PpStage &st, pp_rsrc rk, unsigned off, unsigned ps4, int k0) {
#pragma unroll
    for (int i = 0; i < 2; i++)
        st.k[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rk, off + (k0 + 16 * i) * ps4, 0, 0));
}
__device__ __forceinline__ void pp_load_v(PpStage &st, pp_rsrc rv, unsigned off, unsigned ps4, int k0) {
#pragma unroll
    for (int e = 0; e < 4; e++)
        st.v[e] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rv, off + (k0 + e) * ps4, 0, 0));
}

// ... split and stored at this thread's place of a buffer (c)
__device__ __forceinline__ void pp_store_k(const PpStage &st, char *c) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
        uint2 h, l;
        pf_split4(__builtin_bit_cast(float4, st.k[i]), h, l);
        *reinterpret_cast<uint2 *>(c + 4096 * i) = h;
        *reinterpret_cast<uint2 *>(c + 4096 * i + PP_PLANE) = l;
    }
}
__device__ __forceinline__ void pp_store_v(const PpStage &st, char *base, unsigned a) {
#pragma unroll
    for (int par = 0; par < 2; par++) {
        const float4 x = make_float4(__uint_as_float(par ? st.v[0].y : st.v[0].x), __uint_as_float(par ? st.v[1].y : st.v[1].x),
                                     __uint_as_float(par ? st.v[2].y : st.v[2].x), __uint_as_float(par ? st.v[3].y : st.v[3].x));
        uint2 h, l;
        pf_split4(x, h, l);
        char *c = base + (a ^ (64 * par));
        *reinterpret_cast<uint2 *>(c) = h;
        *reinterpret_cast<uint2 *>(c + PP_PLANE) = l;
    }
}

// this wave's LDS stores are done and every wave is here (the loads in flight
// stay in flight: __syncthreads() would drain them); nothing is scheduled
// across
__device__ __forceinline__ void pp_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The matrix part: scores of the K tile at ck (SCORES), O^T += V^T P^T of the
// V tile at cv (PV); ak / av: this lane's place of step 0 in them.  Fragments
// are read three steps ahead of their MFMAs.
template <bool SCORES, bool PV>
__device__ __forceinline__ void pp_matrix(const char *ck, const char *cv, unsigned ak, unsigned av,
                                          const bf16x8 (&qh)[8], const bf16x8 (&qo)[8], const bf16x8 (&ph)[2],
                                          const bf16x8 (&po)[2], pf_f32x16 &s, pf_f32x16 (&o)[4]) {
    // opaque here: the compiler would otherwise keep every step's address in a
    // register across the loop (and spill)
    asm volatile("" : "+v"(ak), "+v"(av));
    // step u takes one fragment, hi (u even) or lo: u < 16 k-step u / 2 of the
    // scores, then dims 32 (u - 16 >> 2), k-step (u >> 1) & 1 of V^T P^T
    constexpr int U0 = SCORES ? 0 : 16, U1 = PV ? 32 : 16, AHEAD = 3;
    bf16x8 f[32];
    auto read = [&](int u) {
        const int t = u >> 1;
        const char *c = u < 16 ? ck + (ak ^ (32 * t)) : cv + (av ^ (32 * (t & 1))) + 2048 * ((t - 8) >> 1);
        f[u] = *reinterpret_cast<const bf16x8 *>(c + (u & 1 ? PP_PLANE : 0));
    };
    if (SCORES) s = (pf_f32x16){};
#pragma unroll
    for (int u = U0; u < U0 + AHEAD; u++) read(u);
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int u = U0; u < U1; u++) {
        if (u + AHEAD < U1) read(u + AHEAD);
        const int t = u >> 1, dt = (t - 8) >> 1, j = t & 1;
        if (u < 16) {
            s = pf_mfma32(f[u], u & 1 ? qh[t] : qo[t], s);
        } else if (u & 1) {
            o[dt] = pf_mfma32(f[u], ph[j], o[dt]);
        } else {
            o[dt] = pf_mfma32(f[u], po[j], o[dt]);
            o[dt] = pf_mfma32(f[u], ph[j], o[dt]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (u < 16 || (u & 1)) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        else __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        if (u == 15) {
#pragma unroll
            for (int w = 0; w < 16; w += 2) s = pf_mfma32(f[w], qh[w >> 1], s);
            __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
        }
    }
}

__global__ __launch_bounds__(512, 1) void attn_prefill_pp(qk_attn_args a) {
    constexpr int hd = QWEN_HIP_HEAD_DIM;
    __shared__ PpLds lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hl = lane >> 5, row = lane & 31;
    const int nq = (a.seq_q + PP_QT - 1) / PP_QT;
    // longest query tiles first, all kv heads of a tile next to each other
    const int q0 = (nq - 1 - (int)blockIdx.x / a.kv_heads) * PP_QT;
    const int g = (int)blockIdx.x % a.kv_heads;
    const int kend = min(a.seq_k, a.q_offset + min(a.seq_q, q0 + PP_QT));      // >= 1
    const int h = g * 2 + (wave & 1);
    const int qs = q0 + 32 * (wave >> 1);                 // first query of this wave
    const int qi = qs + row;                              // this lane's query
    const int qstride = a.heads * hd;
    const int nt = (kend + PF_KT - 1) / PF_KT;
    const unsigned ps4 = 4u * (unsigned)a.pos_stride;
    const unsigned kvbytes = (unsigned)(kend - 1) * ps4 + 4u * hd;             // pp_fits
    const pp_rsrc rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.k + (size_t)g * a.head_stride), 0, kvbytes, 0x00020000);
    const pp_rsrc rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.v + (size_t)g * a.head_stride), 0, kvbytes, 0x00020000);
    char *const lk = reinterpret_cast<char *>(lds.k), *const lv = reinterpret_cast<char *>(lds.v);

    // this thread's places (PpStage, PpLds)
    const int vm = (lane & 7) | ((lane >> 1) & 0x18) | ((wave & 1) << 5);
    const int vs = (lane >> 3) & 1, vg0 = (wave >> 1) & 1, vg2 = wave >> 2;
    const unsigned koff = (unsigned)(tid >> 5) * ps4 + (tid & 31) * 16u;
    const unsigned voff = (unsigned)(4 * vg0 + 8 * vs + 16 * vg2) * ps4 + vm * 8u;
    const unsigned kst = (tid >> 5) * 256 + 16 * (((tid & 31) >> 1) ^ ((tid >> 5) & 15)) + 8 * (tid & 1);
    const unsigned vst = 128 * vm + 16 * ((2 * vg2 + vg0) ^ (vm & 7)) + 8 * vs;
    const unsigned ak = 256 * row + 16 * (hl ^ (row & 15));
    const unsigned av = 128 * (row >> 1) + 16 * ((4 * (row & 1) + hl) ^ ((row >> 1) & 7));

    PpStage st;
    pp_load_k(st, rk, koff, ps4, 0);
    pp_load_v(st, rv, voff, ps4, 0);
    // this lane's query row, dims 16 t + 8 hl .. + 7, split once (rows past seq_q: 0)
    bf16x8 qh[8], qo[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        float4 x[2] = {};
        if (qi < a.seq_q) {
            const float4 *qp = reinterpret_cast<const float4 *>(a.q + (size_t)qi * qstride + h * hd + 16 * t + 8 * hl);
            x[0] = qp[0];
            x[1] = qp[1];
        }
        pf_split8(&x[0].x, qh[t], qo[t]);
    }
    pp_store_k(st, lk + kst);
    pp_store_v(st, lv, vst);
    pp_load_k(st, rk, koff, ps4, PF_KT);                  // past the end: zeros, never scored
    pp_store_k(st, lk + PP_BUF + kst);
    pp_load_k(st, rk, koff, ps4, 2 * PF_KT);
    pp_load_v(st, rv, voff, ps4, PF_KT);
    pp_barrier();

    pf_f32x16 o[4] = {}, s;
    bf16x8 ph[2], po[2];                                  // the lane's 8 probabilities of each k-step
    float m = PF_MINIT, l = 0.0f;
    // base 2 throughout: p = 2^(score * scale * log2(e) - m)
    const float scale2 = a.scale * 1.44269504088896341f;
    // softmax of the scores s of tile i: p in ph / po, m, l and o brought up to date
    auto softmax = [&](int i) {
        const int k0 = i * PF_KT;
        // a tile wholly below the wave's diagonal and the end needs no mask
        if (k0 + PF_KT - 1 > a.q_offset + qs || k0 + PF_KT > kend) {
            int ln = lane;                                // opaque: nothing of this is held across the loop
            asm volatile("" : "+v"(ln));
            const int last = min(kend - 1, a.q_offset + qs + (ln & 31)) - k0 - 4 * (ln >> 5);
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 8 * (r >> 2) + (r & 3) <= last ? s[r] : -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        {
            float x = mx, y = mx;
            swap32(x, y);
            mx = fmaxf(x, y) * scale2;                    // a positive factor keeps the maximum where it is
        }
        if (__any(mx > m)) {                              // the maximum moves for some query
            const float mn = fmaxf(m, mx), corr = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < 4; dt++) o[dt] *= corr;
        }
        float p[16], sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], scale2, -m));
            sum += p[r];
        }
        l += sum;                                         // this lane's keys; both halves are added at the end
        pf_split8(p, ph[0], po[0]);
        pf_split8(p + 8, ph[1], po[1]);
    };

    pp_matrix<true, false>(lk, lv, ak, av, qh, qo, ph, po, s, o);
    softmax(0);
    pp_barrier();                                         // K 0 is read; barrier 0
    const int e = wave >> 2;                              // group B stores one tile ahead of group A
    // K j and V j - 1 into their buffers, the next ones on their way
    auto stage = [&](int j) {
        const int b = (j & 1) * PP_BUF;
        pp_store_k(st, lk + b + kst);
        pp_store_v(st, lv + (PP_BUF - b), vst);
        pp_load_k(st, rk, koff, ps4, (j + 1) * PF_KT);
        pp_load_v(st, rv, voff, ps4, j * PF_KT);
    };
    if (e) stage(2);
    for (int i = 0; i + 1 < nt; i++) {
        const int b = (i & 1) * PP_BUF;
        pp_matrix<true, true>(lk + (PP_BUF - b), lv + b, ak, av, qh, qo, ph, po, s, o);
        if (e) pp_barrier();
        __builtin_amdgcn_sched_barrier(0);
        softmax(i + 1);
        stage(i + 2 + e);
        if (!e) pp_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    pp_matrix<false, true>(lk, lv + ((nt - 1) & 1) * PP_BUF, ak, av, qh, qo, ph, po, s, o);

    {
        float x = l, y = l;
        swap32(x, y);
        l = x + y;
    }
    if (qi >= a.seq_q) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int b = 0; b < 4; b++)
            pf_write_out(a, (size_t)qi * qstride + h * hd + 32 * dt + 8 * b + 4 * hl,
                         make_float4(o[dt][4 * b] * inv, o[dt][4 * b + 1] * inv, o[dt][4 * b + 2] * inv,
                                     o[dt][4 * b + 3] * inv));
}

// attn_prefill_pp's buffer descriptors and offsets are 32-bit: a kv head's rows,
// and the tiles read past their end, lie within 2^31 bytes
static bool pp_fits(const qk_attn_args *a) {
    const long keys = a->seq_k < (long)a->q_offset + a->seq_q ? a->seq_k : (long)a->q_offset + a->seq_q;
    return a->pos_stride > 0 && (keys + 4 * PF_KT) <= 0x7fffffffL / 4 / a->pos_stride;
}

// The splits of one (query, head) combined in split order (max, then
// rescaled sums) for the 4 dims of this lane: NB splits' loads in one round
// trip (splits at or past n read split 0, finite, and weigh 0).
template <int NB>
__device__ __forceinline__ void pf_merge_batch(const float *p0, size_t stride, int s0, int n, int sl, float &M, float &L,
                                               float4 &o, bool first_pass) {
    float mv[NB], lv[NB];
    float4 v[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const bool in = s0 + j < n;
        const float *p = p0 + (in ? s0 + j : 0) * stride;
        mv[j] = in ? p[QWEN_HIP_HEAD_DIM] : PF_MINIT;
        lv[j] = p[QWEN_HIP_HEAD_DIM + 1];
        if (!first_pass) v[j] = *reinterpret_cast<const float4 *>(p + 4 * sl);
    }
    if (first_pass) {                                     // the max over this batch only
#pragma unroll
        for (int j = 0; j < NB; j++) M = fmaxf(M, mv[j]);
        return;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const float w = s0 + j < n ? __builtin_amdgcn_exp2f(mv[j] - M) : 0.0f;
        L = fmaf(lv[j], w, L);
        o.x = fmaf(v[j].x, w, o.x);
        o.y = fmaf(v[j].y, w, o.y);
        o.z = fmaf(v[j].z, w, o.z);
        o.w = fmaf(v[j].w, w, o.w);
    }
}

// 32 lanes per (query, head), 4 dims each, eight per block: combine the splits
// of the query's tile in split order (max, then rescaled sums), normalise,
// store.  Up to 8 splits take one round trip (the max from the same loads).
__global__ __launch_bounds__(256) void attn_prefill_merge(qk_attn_args a) {
    constexpr int hd = QWEN_HIP_HEAD_DIM;
    const long u = 8L * blockIdx.x + (threadIdx.x >> 5);
    if (u >= (long)a.seq_q * a.heads) return;        // a whole half wave
    const int qi = (int)(u / a.heads), h = (int)(u % a.heads), sl = threadIdx.x & 31;
    const int t = qi / PF_Q;
    const int kend_tile = min(a.seq_k, a.q_offset + min(a.seq_q, (t + 1) * PF_Q));
    const int n = (kend_tile + a.chunk - 1) / a.chunk;
    const size_t stride = (size_t)a.seq_q * a.heads * QK_PF_PART;
    const float *p0 = a.part + ((size_t)qi * a.heads + h) * QK_PF_PART;
    float M = PF_MINIT, L = 0.0f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    if (n >= 1 && n <= 4) {
        float mv[4], lv[4];
        float4 v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool in = j < n;
            const float *p = p0 + (in ? j : 0) * stride;
            mv[j] = in ? p[hd] : PF_MINIT;
            lv[j] = p[hd + 1];
            v[j] = *reinterpret_cast<const float4 *>(p + 4 * sl);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) M = fmaxf(M, mv[j]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float w = j < n ? __builtin_amdgcn_exp2f(mv[j] - M) : 0.0f;
            L = fmaf(lv[j], w, L);
            o.x = fmaf(v[j].x, w, o.x);
            o.y = fmaf(v[j].y, w, o.y);
            o.z = fmaf(v[j].z, w, o.z);
            o.w = fmaf(v[j].w, w, o.w);
        }
    } else if (n >= 5 && n <= 8) {
        float mv[8], lv[8];
        float4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const bool in = j < n;
            const float *p = p0 + (in ? j : 0) * stride;
            mv[j] = in ? p[hd] : PF_MINIT;
            lv[j] = p[hd + 1];
            v[j] = *reinterpret_cast<const float4 *>(p + 4 * sl);
        }
#pragma unroll
        for (int j = 0; j < 8; j++) M = fmaxf(M, mv[j]);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float w = j < n ? __builtin_amdgcn_exp2f(mv[j] - M) : 0.0f;
            L = fmaf(lv[j], w, L);
            o.x = fmaf(v[j].x, w, o.x);
            o.y = fmaf(v[j].y, w, o.y);
            o.z = fmaf(v[j].z, w, o.z);
            o.w = fmaf(v[j].w, w, o.w);
        }
    } else {
        // batches of 8: the max over all splits first, then the sums
        for (int s0 = 0; s0 < n; s0 += 8) pf_merge_batch<8>(p0, stride, s0, n, sl, M, L, o, true);
        for (int s0 = 0; s0 < n; s0 += 8) pf_merge_batch<8>(p0, stride, s0, n, sl, M, L, o, false);
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    const size_t base = (size_t)qi * a.heads * hd + h * hd + 4 * sl;
    const float e[4] = {o.x * inv, o.y * inv, o.z * inv, o.w * inv};
    if (a.out) {
        *reinterpret_cast<float4 *>(a.out + base) = make_float4(e[0], e[1], e[2], e[3]);
    } else {
        uint16_t hh[4], ll[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            hh[i] = f32_to_bf16_rne(e[i]);
            ll[i] = f32_to_bf16_rne(e[i] - bf16_to_f32(hh[i]));
        }
        *reinterpret_cast<uint2 *>(a.out_hi + base) = make_uint2(hh[0] | ((unsigned)hh[1] << 16), hh[2] | ((unsigned)hh[3] << 16));
        *reinterpret_cast<uint2 *>(a.out_lo + base) = make_uint2(ll[0] | ((unsigned)ll[1] << 16), ll[2] | ((unsigned)ll[3] << 16));
    }
}

extern "C" size_t qk_attn_prefill_plan(int seq_q, int seq_k, int q_offset, int heads, int kv_heads, int *chunk,
                                       int *nsplit) {
    const int nq = (seq_q + PF_Q - 1) / PF_Q;
    long tiles = 0;
    int kmax = 0;
    for (int t = 0; t < nq; t++) {
        const int qe = (t + 1) * PF_Q < seq_q ? (t + 1) * PF_Q : seq_q;
        int ke = q_offset + qe;
        if (ke > seq_k) ke = seq_k;
        if (ke > kmax) kmax = ke;
        tiles += (ke + PF_KT - 1) / PF_KT;
    }
    // about QK_PF_TARGET blocks in flight: enough to fill 256 CUs twice over
    long per = (tiles * kv_heads + QK_PF_TARGET - 1) / QK_PF_TARGET;
    if (per < 1) per = 1;
    long c = per * PF_KT;
    // no block walks more than a sixth of the longest query tile (at least 256
    // keys): the causal triangle's longest tiles then end with the rest
    long cap = ((kmax + 5) / 6 + PF_KT - 1) / PF_KT * PF_KT;
    if (cap < 256) cap = 256;
    if (c > cap) c = cap;
    // with several query tiles and up to 2048 keys, splits of a quarter of the
    // longest key range (nearest 32) at least: every split adds partials and a
    // merge pass (7 us at 401 rows), and the tiles themselves already spread
    // the work (C1 401 rows: 96-key splits 26.1 us against 32-key 28.3; C3
    // 1515 rows: 384-key 78.5 us against 224-key ~87, attention + merge)
    if (nq >= 4 && kmax <= 2048) {
        long q4 = (kmax / 4 + PF_KT / 2) / PF_KT * PF_KT;
        if (c < q4) c = q4;
    }
    // one query tile (a short continuation prefill over a long cache): 64-key
    // splits at least, half the partials of 32-key ones for the merge (C5's
    // 31 rows after ~1000 keys: 17.3 -> 15.7 us with the merge)
    if (nq == 1 && c < 2 * PF_KT) c = 2 * PF_KT;
    // with two (query tile, kv head) blocks per CU or more, the longest-first
    // order alone balances the CUs: no split, so no partials and no merge pass
    if ((long)nq * kv_heads >= 2L * 256) c = (kmax + PF_KT - 1) / PF_KT * PF_KT;
    if (c > kmax) c = (kmax + PF_KT - 1) / PF_KT * PF_KT;
    *chunk = (int)c;
    *nsplit = (int)((kmax + c - 1) / c);
    return *nsplit > 1 ? (size_t)*nsplit * seq_q * heads * QK_PF_PART : 0;
}

extern "C" int qk_attn_prefill_launch(const qk_attn_args *a, hipStream_t s) {
    if (!a || a->seq_q <= 0 || a->seq_k <= 0 || a->kv_heads <= 0 || a->heads != 2 * a->kv_heads)
        return QWEN_HIP_EINVAL;
    if (!a->out && (!a->out_hi || !a->out_lo)) return QWEN_HIP_EINVAL;
    if (a->chunk <= 0 || a->chunk % PF_KT || a->nsplit < 1 || (a->nsplit > 1 && !a->part)) return QWEN_HIP_EINVAL;
    const int nq = (a->seq_q + PF_Q - 1) / PF_Q;
    // every key the last query tile sees must fall in some split
    const int kmax = a->seq_k < a->q_offset + a->seq_q ? a->seq_k : a->q_offset + a->seq_q;
    if ((long)a->chunk * a->nsplit < kmax) return QWEN_HIP_EINVAL;
    // unsplit prefills with 128-query tiles enough for every CU: 8-wave blocks
    // (4096 queries, 256 blocks: 251 us against 345; fewer blocks would leave CUs idle)
    const int nqp = (a->seq_q + PP_QT - 1) / PP_QT;
    if (a->nsplit == 1 && (long)nqp * a->kv_heads >= 256 && pp_fits(a))
        attn_prefill_pp<<<dim3(nqp * a->kv_heads, 1, 1), 512, 0, s>>>(*a);
    else
        attn_prefill<<<dim3(nq * a->kv_heads, 1, a->nsplit), 256, 0, s>>>(*a);
    if (a->nsplit > 1)
        attn_prefill_merge<<<(unsigned)(((long)a->seq_q * a->heads + 7) / 8), 256, 0, s>>>(*a);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}
