// encoder.hip - kernels of the audio encoder (reference qwen_asr_encoder.c:
// Conv2D stem -> conv_out projection + sinusoidal positions -> pre-LayerNorm
// transformer layers with windowed bidirectional attention -> ln_post,
// proj1 + GELU, proj2).
//
// The reference computes the encoder in fp32 on weights widened from bf16
// (load_bf16_as_f32, qwen_asr_encoder.c:43-65).  bf16-valued weights are kept in
// bf16 (exact) and the fp32 activations are carried as hi + lo bf16 on the bf16
// matrix cores; other weights, and attention, run on the fp32 matrix cores.
//
//   enc_ring     products on bf16 weights with activations kept as halves; the
//                stem convolutions and conv_out gather their rows from the
//                stem's pixels (enc_conv1_halves writes the first ones)
// The general forms (any weight values and widths):
//   enc_im2col   Conv2D(3x3, stride 2, pad 1) patches of all chunks at once:
//                row n = (chunk, oh, ow), column k = (ki, kj, ic) tap-major
//                (the reference's im2col, qwen_asr_kernels.c:566-590, with
//                the weight columns reordered to match); the stem
//                activations are channel-last [chunk][h][w][480], and with
//                bf16 weights conv2 / conv3 skip this pass: the GEMM reads
//                the same patches straight from the activations
//   enc_gemm     C[M][N] = A[M][K] . B[N][K]^T with the encoder epilogues:
//                bias along M or N, GELU, residual add, positional table add,
//                zeroing of the padded positions of a partial last chunk
//   enc_stem_rows conv3 output [chunk][16][w][480] -> token rows [t][480*16]
//                (qwen_asr_encoder.c:281-290)
//   enc_layernorm  (x - mean) * inv_std * w + b, two-pass mean / variance
//                (qwen_layer_norm, qwen_asr_kernels.c:640-748)
//   enc_attention  bidirectional attention inside fixed token windows
//                (qwen_bidirectional_attention, qwen_asr_kernels.c:1003-1048)
#include "common.h"
#include "qk_kernels.h"
#include "qwen_asr_hip.h"
#include "ring.h"

#include <math.h>

__device__ __forceinline__ f32x4 enc_mfma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// GELU, tanh form (qwen_gelu, qwen_asr_kernels.c:886-893): 0.5 v (1 + tanh u) =
// v / (1 + e^(-2u)), with no cancellation for negative u.  No error of its own but
// the hardware exponential's and the last rounding: the exponent -2u log2(e) is
// hi + lo, the quotient is corrected by the remainder of v - (1 + e) q, whose 1 + e
// counts with what its rounding lost.  Error against 64 bits (root mean square,
// relative): at most 3.0e-8 for v > 0 and 1.2e-7 on [-2, 0]; the fp32 expression with
// tanhf has 4.3e-8 and 2.2e-7, and cancels below.  Beyond 9 in size the expression is
// v or 0, infinities and NaN as there.  268 M values 161 us, with tanhf 214.
__device__ __forceinline__ float enc_gelu(float v) {
    constexpr double c = -2.0 * 0.7978845608028654 * 1.4426950408889634;
    constexpr float c_hi = (float)c, c_lo = (float)(c - (double)c_hi);
    const float w = v * fmaf(0.044715f, v * v, 1.0f), hi = w * c_hi;
    const float lo = fmaf(w, c_lo, fmaf(w, c_hi, -hi));
    float e = __builtin_amdgcn_exp2f(hi);
    e = fmaf(e, 0.693147181f * lo, e);
    const float d = 1.0f + e, lost = e - (d - 1.0f), r = __builtin_amdgcn_rcpf(d), q = v * r;
    const float y = fmaf(fmaf(-lost, q, fmaf(-d, q, v)), r, q);
    return fabsf(v) > 9.0f ? v * __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f) : y;
}

// ---------------------------------------------------------------------------
// im2col of one stem layer over every chunk.  in: conv1 the mel [128][frames]
// (chunk c covering frames [c*cw, c*cw + cw), frames past `frames` read as
// 0); conv2 / conv3 channel-last [chunks][h_in][w_in][c_in].  cols:
// [chunks*h_out*w_out][kpad], the columns past c_in*9 zero.
// ---------------------------------------------------------------------------
// conv1 (one input channel, the mel read in place): thread = (row, k), 256 / kpad
// rows per block, 32-bit index math
__global__ __launch_bounds__(256) void enc_im2col_mel(const float *mel, float *cols, int rows, int h_in, int w_in,
                                                      int h_out, int w_out, int kpad, int mel_frames) {
    const int rpb = 256 / kpad, r = threadIdx.x / kpad, k = threadIdx.x % kpad;
    for (int n0 = blockIdx.x * rpb; n0 < rows; n0 += gridDim.x * rpb) {
        const int n = n0 + r;
        if (r >= rpb || n >= rows) continue;
        const int ow = n % w_out, t = n / w_out, oh = t % h_out, c = t / h_out;
        float v = 0.0f;
        if (k < 9) {
            const int ih = 2 * oh - 1 + k / 3, iw = 2 * ow - 1 + k % 3;
            const int f = c * w_in + iw;
            if (ih >= 0 && ih < h_in && iw >= 0 && iw < w_in && f < mel_frames) v = mel[(long)ih * mel_frames + f];
        }
        cols[(long)n * kpad + k] = v;
    }
}

// conv2 / conv3 on channel-last input [chunk][h_in][w_in][c_in]: one block
// per row n = (chunk, oh, ow); k = tap * c_in + ic, so each tap is c_in
// contiguous floats of one input pixel (float4 copies, both sides coalesced)
__global__ __launch_bounds__(256) void enc_im2col(const float *in, float *cols, int c_in, int chunks, int rows,
                                                  int h_in, int w_in, int h_out, int w_out, int kpad) {
    const int q4 = c_in / 4;
    for (int n = blockIdx.x; n < rows; n += gridDim.x) {
        const int ow = n % w_out, t = n / w_out, oh = t % h_out, c = t / h_out;
        float *dst = cols + (long)n * kpad;
        for (int i = threadIdx.x; i < 9 * q4; i += 256) {
            const int tap = i / q4, q = i - tap * q4;
            const int ih = 2 * oh - 1 + tap / 3, iw = 2 * ow - 1 + tap % 3;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (ih >= 0 && ih < h_in && iw >= 0 && iw < w_in)
                v = *reinterpret_cast<const float4 *>(in + (((long)c * h_in + ih) * w_in + iw) * c_in + 4 * q);
            *reinterpret_cast<float4 *>(dst + tap * c_in + 4 * q) = v;
        }
        for (int k = 9 * c_in + threadIdx.x; k < kpad; k += 256) dst[k] = 0.0f;
    }
}

extern "C" int qk_enc_im2col_launch(const float *in, float *cols, int c_in, int chunks, int h_in, int w_in,
                                    int h_out, int w_out, int kpad, int mel_frames, hipStream_t s) {
    if (!in || !cols || c_in <= 0 || chunks <= 0 || kpad < c_in * 9 || (kpad & 15)) return QWEN_HIP_EINVAL;
    if (mel_frames <= 0 && (c_in & 3)) return QWEN_HIP_EINVAL;
    const long rows = (long)chunks * h_out * w_out;
    if (rows > 0x7fffffffL) return QWEN_HIP_EINVAL;
    if (mel_frames > 0) {
        if (c_in != 1 || kpad > 256 || 256 % kpad) return QWEN_HIP_EINVAL;
        const long rpb = 256 / kpad, blocks = (rows + rpb - 1) / rpb;
        enc_im2col_mel<<<(int)(blocks < 65536 ? blocks : 65536), 256, 0, s>>>(in, cols, (int)rows, h_in, w_in, h_out,
                                                                              w_out, kpad, mel_frames);
    } else {
        enc_im2col<<<(int)(rows < 65536 ? rows : 65536), 256, 0, s>>>(in, cols, c_in, chunks, (int)rows, h_in, w_in,
                                                                     h_out, w_out, kpad);
    }
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// ---------------------------------------------------------------------------
// fp32 GEMM on v_mfma_f32_16x16x4_f32.  Block tile 64 x 64, 4 waves of 32 x 32
// (2 x 2 MFMA tiles), K walked 16 at a time through LDS with the next tile's
// loads in flight.  Within a 16-wide k block lane l supplies k = 4 (l >> 4) + c
// at k-step c for both operands (each lane reads one float4 per row).
// ---------------------------------------------------------------------------
#define EG_T 64
#define EG_K 16
#define EG_LD (EG_K + 4)

// the encoder epilogues on element (m, n) of C (y points at it)
__device__ __forceinline__ void enc_epilogue(const qk_enc_gemm_args &a, int m, int n, float v, float *y) {
    if (a.bias_m) v += a.bias_m[m];
    if (a.bias_n) v += a.bias_n[n];
    if (a.pe) v += a.pe[(long)(m % a.pe_rows) * a.N + n];
    if (a.gelu) v = enc_gelu(v);
    if (a.col_w > 0) {
        // stem output position (chunk, oh, ow) (column n, or row m when
        // pad_rows): the last chunk's positions past its valid width are the
        // zero padding the reference's next convolution sees
        const int p = a.pad_rows ? m : n;
        const int ow = p % a.col_w, c = p / (a.col_w * a.col_h);
        if (c == a.col_chunks - 1 && ow >= a.col_valid) v = 0.0f;
    }
    if (a.add) v += *y;                    // residual (qwen_add_inplace after the projection)
    *y = v;
}

__global__ __launch_bounds__(256) void enc_gemm(qk_enc_gemm_args a) {
    __shared__ __attribute__((aligned(16))) float sA[EG_T][EG_LD];
    __shared__ __attribute__((aligned(16))) float sB[EG_T][EG_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * EG_T, n0 = blockIdx.x * EG_T;
    const int lr = tid >> 2, lk = (tid & 3) * 4;      // loader: row lr, k lk .. lk+3 of the tile

    float4 ra, rb;
    auto gload = [&](int k0) {
        const int gm = m0 + lr, gn = n0 + lr, gk = k0 + lk;
        ra = (gm < a.M && gk < a.K) ? *reinterpret_cast<const float4 *>(a.A + (long)gm * a.lda + gk)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
        rb = (gn < a.N && gk < a.K) ? *reinterpret_cast<const float4 *>(a.B + (long)gn * a.ldb + gk)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // K slice of this block: [kb, ke); kc is a multiple of EG_K, so every
    // 16-wide step but the last one of the whole product lies inside K
    const int kb = blockIdx.z * a.kc, ke = min(a.K, kb + a.kc);
    gload(kb);
    for (int k0 = kb; k0 < ke; k0 += EG_K) {
        __syncthreads();
        *reinterpret_cast<float4 *>(&sA[lr][lk]) = ra;
        *reinterpret_cast<float4 *>(&sB[lr][lk]) = rb;
        __syncthreads();
        if (k0 + EG_K < ke) gload(k0 + EG_K);
        float4 af[2], bf[2];
#pragma unroll
        for (int i = 0; i < 2; i++) af[i] = *reinterpret_cast<const float4 *>(&sA[wm * 32 + i * 16 + (lane & 15)][4 * (lane >> 4)]);
#pragma unroll
        for (int j = 0; j < 2; j++) bf[j] = *reinterpret_cast<const float4 *>(&sB[wn * 32 + j * 16 + (lane & 15)][4 * (lane >> 4)]);
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = enc_mfma((&af[i].x)[c], (&bf[j].x)[c], acc[i][j]);
    }

    // D[4 (l >> 4) + r][l & 15] of each 16 x 16 tile: rows m, column n
    float *part = a.split > 1 ? a.ws + (long)blockIdx.z * a.M * a.N : nullptr;
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = n0 + wn * 32 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm * 32 + i * 16 + 4 * (lane >> 4) + r;
                if (m >= a.M || n >= a.N) continue;
                if (part)
                    part[(long)m * a.N + n] = acc[i][j][r];
                else
                    enc_epilogue(a, m, n, acc[i][j][r], a.C + (long)m * a.ldc + n);
            }
        }
    }
}

// split-K: C = epilogue(sum of the slices' partials, slice 0 first)
__global__ __launch_bounds__(256) void enc_gemm_reduce(qk_enc_gemm_args a) {
    const long MN = (long)a.M * a.N;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < MN; e += (long)gridDim.x * 256) {
        float v = a.ws[e];
        for (int z = 1; z < a.split; z++) v += a.ws[z * MN + e];
        const int m = (int)(e / a.N), n = (int)(e % a.N);
        enc_epilogue(a, m, n, v, a.C + (long)m * a.ldc + n);
    }
}

// ---------------------------------------------------------------------------
// The same product with one operand bf16 (the weights, exact) and the other
// fp32, split on the way into LDS as hi = bf16(x), lo = bf16(x - hi):
// x.w = hi.w + lo.w on v_mfma_f32_16x16x32_bf16 (fp32 accumulation).  Block
// tile 64 x 64, 4 waves of 32 x 32, K 32 at a time (one MFMA k-step), the next
// tile's loads in flight during the MFMAs.  WA: the bf16 operand is A (rows
// M); otherwise B (rows N).  Fragments: lane l supplies row (l & 15), k
// 8 (l >> 4) .. + 7, for both operands.
// ---------------------------------------------------------------------------
#define EH_K 32
#define EH_LD (EH_K + 8)           // 80-byte rows: 16-row fragment reads conflict free
typedef float eh_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 eh_bf16x4 __attribute__((ext_vector_type(4)));

template <bool WA, int TT>        // TT x TT MFMA tiles of 16 x 16 per wave: block tile 32 TT x 32 TT
__global__ __launch_bounds__(256) void enc_gemm_hl(qk_enc_gemm_args a) {
    constexpr int BT = 32 * TT;                       // block tile edge
    constexpr int XPT = BT * EH_K / 4 / 256;          // fp32 float4 loads per thread
    constexpr int WPT = BT * EH_K / 8 / 256;          // bf16 16-byte loads per thread
    __shared__ __attribute__((aligned(16))) __bf16 sX[2][BT][EH_LD];   // fp32 operand: [hi, lo]
    __shared__ __attribute__((aligned(16))) __bf16 sW[BT][EH_LD];      // bf16 operand
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT;
    // fp32 side: rows of X = M rows of A (WA false) or N rows of B (WA true)
    const float *X = WA ? a.B : a.A;
    const uint16_t *W = WA ? a.A16 : a.B16;
    const int ldx = WA ? a.ldb : a.lda, ldw = WA ? a.lda : a.ldb;
    const int xr0 = WA ? n0 : m0, xrn = WA ? a.N : a.M;
    const int wr0 = WA ? m0 : n0, wrn = WA ? a.M : a.N;
    // loaders: X rows xr + 32 i (4 floats at xk), W rows wr + 64 i (8 bf16 at wk)
    const int xr = tid >> 3, xk = (tid & 7) * 4;
    const int wr = tid >> 2, wk = (tid & 3) * 8;

    float4 rx[XPT];
    uint4 rw[WPT];
    // implicit im2col (A side only): this thread's rows as (input plane base,
    // top-left input row / column of the 3x3 window); -1 marks rows past M
    const bool conv = !WA && a.conv_c > 0;
    int cb[XPT], ci[XPT], cj[XPT];
    if (conv) {
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int g = xr0 + xr + 32 * i;
            const int ow = g % a.col_w, t = g / a.col_w, oh = t % a.col_h, c = t / a.col_h;
            cb[i] = g < xrn ? c * a.conv_in_h * a.conv_in_w : -1;
            ci[i] = 2 * oh - 1;
            cj[i] = 2 * ow - 1;
        }
    }
    auto gload = [&](int k0) {
        if (conv) {
            // a 32-wide k tile lies in one tap: channels ic .. ic + 3 of one input pixel
            const int tap = k0 / a.conv_c, ic = k0 - tap * a.conv_c + xk;
            const int dy = tap / 3, dx = tap - 3 * dy;
#pragma unroll
            for (int i = 0; i < XPT; i++) {
                const int ih = ci[i] + dy, iw = cj[i] + dx;
                const bool ok = cb[i] >= 0 && ih >= 0 && ih < a.conv_in_h && iw >= 0 && iw < a.conv_in_w;
                rx[i] = ok ? *reinterpret_cast<const float4 *>(X + ((long)cb[i] + ih * a.conv_in_w + iw) * a.conv_c + ic)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        } else {
#pragma unroll
            for (int i = 0; i < XPT; i++) {
                const int g = xr0 + xr + 32 * i, gk = k0 + xk;
                rx[i] = (g < xrn && gk < a.K) ? *reinterpret_cast<const float4 *>(X + (long)g * ldx + gk)
                                              : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
#pragma unroll
        for (int i = 0; i < WPT; i++) {
            const int g = wr0 + wr + 64 * i, gk = k0 + wk;
            rw[i] = (g < wrn && gk < a.K) ? *reinterpret_cast<const uint4 *>(W + (long)g * ldw + gk)
                                          : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    auto lstore = [&]() {
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const eh_f32x4 x = {rx[i].x, rx[i].y, rx[i].z, rx[i].w};
            const eh_bf16x4 hi = __builtin_convertvector(x, eh_bf16x4);
            const eh_bf16x4 lo = __builtin_convertvector(x - __builtin_convertvector(hi, eh_f32x4), eh_bf16x4);
            *reinterpret_cast<eh_bf16x4 *>(&sX[0][xr + 32 * i][xk]) = hi;
            *reinterpret_cast<eh_bf16x4 *>(&sX[1][xr + 32 * i][xk]) = lo;
        }
#pragma unroll
        for (int i = 0; i < WPT; i++) *reinterpret_cast<uint4 *>(&sW[wr + 64 * i][wk]) = rw[i];
    };
    f32x4 acc[TT][TT];
#pragma unroll
    for (int i = 0; i < TT; i++)
#pragma unroll
        for (int j = 0; j < TT; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int kb = blockIdx.z * a.kc, ke = min(a.K, kb + a.kc);
    gload(kb);
    for (int k0 = kb; k0 < ke; k0 += EH_K) {
        __syncthreads();
        lstore();
        __syncthreads();
        if (k0 + EH_K < ke) gload(k0 + EH_K);
        const int kf = 8 * (lane >> 4);
        bf16x8 fm[TT][2], fn[TT][2];    // [tile][hi / lo or weight]: M-side and N-side fragments
#pragma unroll
        for (int i = 0; i < TT; i++) {
            const int rm = wm * 16 * TT + i * 16 + (lane & 15), rn = wn * 16 * TT + i * 16 + (lane & 15);
            if (WA) {
                fm[i][0] = *reinterpret_cast<const bf16x8 *>(&sW[rm][kf]);
                fn[i][0] = *reinterpret_cast<const bf16x8 *>(&sX[0][rn][kf]);
                fn[i][1] = *reinterpret_cast<const bf16x8 *>(&sX[1][rn][kf]);
            } else {
                fm[i][0] = *reinterpret_cast<const bf16x8 *>(&sX[0][rm][kf]);
                fm[i][1] = *reinterpret_cast<const bf16x8 *>(&sX[1][rm][kf]);
                fn[i][0] = *reinterpret_cast<const bf16x8 *>(&sW[rn][kf]);
            }
        }
#pragma unroll
        for (int i = 0; i < TT; i++)
#pragma unroll
            for (int j = 0; j < TT; j++) {
                if (WA) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fm[i][0], fn[j][0], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fm[i][0], fn[j][1], acc[i][j], 0, 0, 0);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fm[i][0], fn[j][0], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fm[i][1], fn[j][0], acc[i][j], 0, 0, 0);
                }
            }
    }

    float *part = a.split > 1 ? a.ws + (long)blockIdx.z * a.M * a.N : nullptr;
#pragma unroll
    for (int i = 0; i < TT; i++) {
#pragma unroll
        for (int j = 0; j < TT; j++) {
            const int n = n0 + wn * 16 * TT + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm * 16 * TT + i * 16 + 4 * (lane >> 4) + r;
                if (m >= a.M || n >= a.N) continue;
                if (part)
                    part[(long)m * a.N + n] = acc[i][j][r];
                else
                    enc_epilogue(a, m, n, acc[i][j][r], a.C + (long)m * a.ldc + n);
            }
        }
    }
}

// split-K reduce of one row (block per row, N <= 1024) that then LayerNorms
// the finished row into ln_out, with enc_layernorm's element-to-thread map and
// reduction order (so the result equals a separate LayerNorm pass)
__global__ __launch_bounds__(256) void enc_gemm_reduce_ln(qk_enc_gemm_args a) {
    __shared__ float red[4];
    const int m = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long MN = (long)a.M * a.N;
    float v[4];
    float s = 0.0f;
    float x[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {      // every slice of the row's 4 columns in one batch of loads
        const int n = min(threadIdx.x + 256 * j, a.N - 1);
        x[j] = sum_splits<8>(a.ws + (long)m * a.N + n, a.split, MN);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int n = threadIdx.x + 256 * j;
        v[j] = 0.0f;
        if (n < a.N) {
            float *y = a.C + (long)m * a.ldc + n;
            enc_epilogue(a, m, n, x[j], y);
            v[j] = *y;
            s += v[j];
        }
    }
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)a.N;
    __syncthreads();
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int n = threadIdx.x + 256 * j;
        if (n < a.N) {
            const float d = v[j] - mean;
            q = fmaf(d, d, q);
        }
    }
    q = wave_sum(q);
    if (lane == 0) red[wave] = q;
    __syncthreads();
    const float var = (red[0] + red[1] + red[2] + red[3]) / (float)a.N;
    const float inv_std = 1.0f / sqrtf(var + a.ln_eps);
    float *o = a.ln_out + (long)m * a.N;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int n = threadIdx.x + 256 * j;
        if (n < a.N) o[n] = (v[j] - mean) * inv_std * a.ln_w[n] + a.ln_b[n];
    }
}

extern "C" int qk_enc_gemm_launch(const qk_enc_gemm_args *a, hipStream_t s) {
    if (!a || (a->A16 && a->B16)) return QWEN_HIP_EINVAL;
    const bool hl = a->A16 || a->B16;
    if (!(a->A || a->A16) || !(a->B || a->B16) || !a->C || a->M <= 0 || a->N <= 0 || a->K <= 0 || (a->K & 3) ||
        (a->lda & 3) || (a->ldb & 3) || a->lda < a->K || a->ldb < a->K || a->ldc < a->N || (a->pe && a->pe_rows <= 0))
        return QWEN_HIP_EINVAL;
    if (hl && ((a->K % EH_K) || (a->A16 ? (a->lda & 7) || !a->B : (a->ldb & 7) || !a->A))) return QWEN_HIP_EINVAL;
    if (a->conv_c > 0 && (!a->B16 || a->conv_c % EH_K || a->K != 9 * a->conv_c || a->col_w <= 0 || a->col_h <= 0 ||
                          a->conv_in_h <= 0 || a->conv_in_w <= 0 || !a->pad_rows))
        return QWEN_HIP_EINVAL;
    if (a->ln_out && (!a->ln_w || !a->ln_b)) return QWEN_HIP_EINVAL;
    const int kstep = hl ? EH_K : EG_K;
    qk_enc_gemm_args g = *a;
    const long tiles = (long)((a->N + EG_T - 1) / EG_T) * ((a->M + EG_T - 1) / EG_T);
    // slices so that the grid holds ~4 blocks per CU, each slice >= 128 deep
    int split = a->ws ? (int)((1024 + tiles - 1) / tiles) : 1;
    if (split > 8) split = 8;
    if (split > a->K / 128) split = a->K / 128;
    if (split < 1) split = 1;
    g.kc = ((a->K + split - 1) / split + kstep - 1) / kstep * kstep;
    g.split = (a->K + g.kc - 1) / g.kc;
    if (g.split > 1 && (long)g.split * a->M * a->N > a->ws_elems) g.kc = a->K, g.split = 1;
    if (g.split == 1) g.kc = a->K;
    dim3 grid((a->N + EG_T - 1) / EG_T, (a->M + EG_T - 1) / EG_T, g.split);
    // large products (the stem convolutions) take 128 x 128 tiles: half the
    // operand bytes per MFMA, which the per-CU load path needs at full rate
    const bool big = hl && g.split == 1 && (long)a->M * a->N >= (1L << 22);
    dim3 grid2((a->N + 127) / 128, (a->M + 127) / 128, 1);
    if (a->A16) {
        if (big) enc_gemm_hl<true, 4><<<grid2, 256, 0, s>>>(g);
        else enc_gemm_hl<true, 2><<<grid, 256, 0, s>>>(g);
    } else if (a->B16) {
        if (big) enc_gemm_hl<false, 4><<<grid2, 256, 0, s>>>(g);
        else enc_gemm_hl<false, 2><<<grid, 256, 0, s>>>(g);
    } else {
        enc_gemm<<<grid, 256, 0, s>>>(g);
    }
    const bool ln = a->ln_out != nullptr;
    if (g.split > 1 && g.split <= 8 && ln && a->N <= 1024 && a->ldc == a->N) {
        enc_gemm_reduce_ln<<<a->M, 256, 0, s>>>(g);
        return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
    }
    if (g.split > 1) {
        long blocks = ((long)a->M * a->N + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        enc_gemm_reduce<<<(int)blocks, 256, 0, s>>>(g);
    }
    if (hipGetLastError() != hipSuccess) return QWEN_HIP_EDEVICE;
    if (ln) {
        if (a->ldc != a->N) return QWEN_HIP_EINVAL;
        return qk_enc_layernorm_launch(a->C, a->ln_w, a->ln_b, a->ln_out, a->M, a->N, a->ln_eps, s);
    }
    return 0;
}

// conv3 output [480][chunks][16][w] -> rows [token][480*16], token = chunk*w + t for
// t < the chunk's token count (qwen_asr_encoder.c:281-290: column ch*16 + f)
__global__ __launch_bounds__(256) void enc_stem_rows(const float *c3, float *rows, int chunks, int w, int h,
                                                     int ch_n, int tokens) {
    const int D = ch_n * h;
    const long total = (long)tokens * D;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
        const int tok = (int)(e / D), col = (int)(e % D);
        const int ch = col / h, f = col % h;
        const int c = tok / w, t = tok % w;
        rows[e] = c3[(((long)c * h + f) * w + t) * ch_n + ch];   // c3 channel-last [chunk][h][w][ch]
    }
}

// conv1 directly from its patches (one input channel, 9 taps in cols[pos][kpad]):
// out[pos][ch] = GELU(b[ch] + sum_tap cols[pos][tap] w[ch][tap]) for 4
// channels per thread, float4 stores, so each position's 480 outputs are one
// contiguous run (the product is 9 multiply-adds per output: the pass is
// bound by the 4 bytes it writes per output).  Positions (chunk, oh, ow) of
// the last chunk with ow >= valid are the zero padding the next layer sees.
__global__ __launch_bounds__(256) void enc_conv1(const float *cols, int kpad, const float *w, const float *b, float *out,
                                                 int rows, int ch, int h_out, int w_out, int chunks, int valid) {
    // the grid stride is a multiple of ch / 4, so a thread keeps one channel
    // quad (its 36 weights and 4 biases in registers) for every position it visits
    const int q4 = ch / 4;
    const long i0 = blockIdx.x * 256L + threadIdx.x, stride = (long)gridDim.x * 256;
    const int c0 = 4 * (int)(i0 % q4);
    float wr[4][9], br[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        br[j] = b[c0 + j];
#pragma unroll
        for (int t = 0; t < 9; t++) wr[j][t] = w[(c0 + j) * kpad + t];
    }
    for (long i = i0; i < (long)rows * q4; i += stride) {
        const int pos = (int)(i / q4);
        const int ow = pos % w_out, cc = pos / (w_out * h_out);
        const float *x = cols + (long)pos * kpad;
        float v[4] = {br[0], br[1], br[2], br[3]};
#pragma unroll
        for (int t = 0; t < 9; t++) {
            const float xt = x[t];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = fmaf(xt, wr[j][t], v[j]);
        }
        const bool pad = cc == chunks - 1 && ow >= valid;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = pad ? 0.0f : enc_gelu(v[j]);
        *reinterpret_cast<float4 *>(out + (long)pos * ch + c0) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

extern "C" int qk_enc_conv1_launch(const float *cols, int kpad, const float *w, const float *b, float *out, int rows,
                                   int ch, int h_out, int w_out, int chunks, int valid, hipStream_t s) {
    if (!cols || !w || !b || !out || rows <= 0 || (ch & 3) || kpad < 9 || h_out <= 0 || w_out <= 0 || chunks <= 0)
        return QWEN_HIP_EINVAL;
    // blocks: a multiple of q4 / gcd(q4, 256) so the grid stride is a multiple of q4
    const int q4 = ch / 4;
    int g = q4, t = 256;
    while (t) { const int r = g % t; g = t; t = r; }
    const long unit = q4 / g;
    long blocks = ((long)rows * q4 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    blocks = (blocks + unit - 1) / unit * unit;
    enc_conv1<<<(int)blocks, 256, 0, s>>>(cols, kpad, w, b, out, rows, ch, h_out, w_out, chunks, valid);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

extern "C" int qk_enc_stem_rows_launch(const float *c3, float *rows, int chunks, int w, int h, int ch_n, int tokens,
                                       hipStream_t s) {
    if (!c3 || !rows || tokens <= 0 || tokens > chunks * w) return QWEN_HIP_EINVAL;
    long blocks = ((long)tokens * ch_n * h + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    enc_stem_rows<<<(int)blocks, 256, 0, s>>>(c3, rows, chunks, w, h, ch_n, tokens);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// ---------------------------------------------------------------------------
// The bf16-weight encoder: every activation that feeds a product is kept as
// rows of two bf16 halves, [K hi | K lo] (hi = bf16(x), lo = bf16(x - hi): the
// bytes of an fp32 row), written by its producer, so the products stream both
// operands through the LDS ring of ring.h with no conversion in the k loop.  Stem
// pixels hold their 480 channels as 15 times [32 hi | 32 lo], and the weights of
// the products that gather them lie as [K / 32][N][32]: a 32-deep k tile then
// reads whole 128-byte lines (with half lines the load path bounded these
// products: conv2 of 743 frames 102 -> 75 us, conv_out of 3000 41 -> 29; on
// enc_gemm_hl they took 172 and ~45).
// Encoders with a matrix of other than bf16 values, d above 1024, an ffn that is no
// multiple of 32 or outputs that are no whole float4s run on enc_gemm_hl / enc_gemm
// above (qk_enc_ring_ok); ragged columns otherwise are the ring's.
//
// What bounds it: at 100 to 400 rows these products are a few microseconds
// each, mostly ramp, the k walk's load path and drain; a k tile staged through
// registers (one in flight) took ~2x a ring step.  390 rows, 896 wide: Q|K|V 13.7 +
// 6.6 us of reduce -> 12.8, fc1 17.7 + 7.5 -> 13.5, fc2 17.5 + 7.5 -> 14.2 + 4.4.
// ---------------------------------------------------------------------------
// four values at columns n .. n + 3 of a row of n_cols, or (PIXEL) of a stem pixel
template <bool PIXEL>
__device__ __forceinline__ void enc_store_halves(uint16_t *row, int n_cols, int n, float4 v) {
    uint2 h, l;
    bf16_split2(v.x, v.y, h.x, l.x);
    bf16_split2(v.z, v.w, h.y, l.y);
    row += PIXEL ? n + (n & ~31) : n;
    *reinterpret_cast<uint2 *>(row) = h;
    *reinterpret_cast<uint2 *>(row + (PIXEL ? 32 : n_cols)) = l;
}

// stem: row m = (chunk, oh, ow) is padding of the last chunk
__device__ __forceinline__ bool enc_ring_pad(const qk_enc_ring_args &a, int m) {
    if (a.valid <= 0) return false;
    const int ow = m % a.col_w, c = m / (a.col_w * a.col_h);
    return c == a.chunks - 1 && ow >= a.valid;
}

// Results of a product: split-K partials, fp32 + bias, or halves of the GELU.
enum { ENC_PART, ENC_F32, ENC_GELU };

// One tile of the product; GATHER: rows of A are gathered from stem pixels.  The
// epilogue is chosen at compile time: with tests between the 32 values of a lane
// their chains ran one after the other, 9.3 us of a 390 x 3584 x 896 GELU
// product's 20 against 1.9 of its 12 now.
template <int BM, int BN, int NST, bool GATHER, int EPI, int KG>
__global__ __launch_bounds__(KG *ring_waves(BM, BN) * 64) void enc_ring(qk_enc_ring_args a) {
    using RS = RingShape<BM, BN>;
    constexpr int NW = RS::NW, WGN = RS::WGN, WTN = RS::WTN, TN = RS::TN, AB = RS::AB, LPW = RS::LPW;
    constexpr int NI = KG == 2 ? 1 : 2;                // 16-row tiles this wave finishes
    __shared__ __attribute__((aligned(1024))) unsigned char lds[KG * NST * RS::STAGE];   // two groups: RingShape2's stages
    const int lane = threadIdx.x & 63, bwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = bwave / NW, wave = bwave % NW;      // k group, wave of the group
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kb = blockIdx.z * a.kc, ke = min(a.K, kb + a.kc), nk = (ke - kb) / QK_GBK;
    const int rr = lane >> 2, cl = (lane & 3) ^ ((rr >> 1) & 3);
    f32x4 acc[NI][TN];
    if constexpr (GATHER) {
        // the wave's A groups: rows m0 + 8 (2 wave + h) + lane / 8, h = 0, 1
        static_assert(BM / 16 == NW && KG == 1, "two 8-row groups per wave");
        const int r8 = lane >> 3, c8 = (lane & 7) ^ r8;
        int pix[2];
        unsigned mask[2] = {0, 0};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int m = min(m0 + 8 * (2 * wave + h) + r8, a.M - 1);
            if (a.taps == 9) {         // 3 x 3, stride 2, padding 1
                const int ow = m % a.col_w, t = m / a.col_w, oh = t % a.col_h, c = t / a.col_h;
                const int ih = 2 * oh - 1, iw = 2 * ow - 1;
                pix[h] = (c * a.in_h + ih) * a.in_w + iw;
#pragma unroll
                for (int tap = 0; tap < 9; tap++) {
                    const int y = ih + tap / 3, x = iw + tap % 3;
                    if (y >= 0 && y < a.in_h && x >= 0 && x < a.in_w) mask[h] |= 1u << tap;
                }
            } else {                   // a token's column of in_h pixels, in_w apart
                pix[h] = m / a.in_w * a.in_h * a.in_w + m % a.in_w;
                mask[h] = 0xffffffffu;
            }
        }
        // W rows (16 per group): those past N re-read row N - 1
        const uint16_t *w[LPW - 2];
#pragma unroll
        for (int j = 0; j < LPW - 2; j++)
            w[j] = a.W + (size_t)(kb / QK_GBK) * a.N * QK_GBK + (size_t)min(n0 + 16 * (wave + NW * j) + rr, a.N - 1) * QK_GBK +
                   8 * cl;
        const size_t wstep = (size_t)a.N * QK_GBK;
        ring_walk<BM, BN, NST, true>(nk, lds, acc, [&](int kt, unsigned char *st) {
            // a 32-wide k tile lies in one tap
            const int k = kb + kt * QK_GBK, tap = k / QK_ENC_CH, ic = k - tap * QK_ENC_CH;
            const int off = a.taps == 9 ? (tap / 3) * a.in_w + tap % 3 : tap * a.in_w;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint16_t *p = (mask[h] >> tap) & 1 ? a.A + (long)(pix[h] + off) * (2 * QK_ENC_CH) + 2 * ic : a.zero;
                lds_load16(p + 8 * c8, st + 1024 * (2 * wave + h));
            }
#pragma unroll
            for (int j = 0; j < LPW - 2; j++) lds_load16(w[j] + kt * wstep, st + 2 * AB + 1024 * (wave + NW * j));
        });
    } else if constexpr (KG == 2) {
        using R2 = RingShape2<BM, BN>;
        const int r8 = lane >> 3, c8 = (lane & 7) ^ r8;
        const uint16_t *src[R2::LPW2];
#pragma unroll
        for (int j = 0; j < R2::LPW2; j++) {
            const int g = bwave + 2 * NW * j, ga = g < BM / 8 ? g : g - BM / 8;
            src[j] = (g < BM / 4 ? a.A + (size_t)min(m0 + 8 * ga + r8, a.M - 1) * (2 * a.K) + (g < BM / 8 ? 0 : a.K)
                                 : a.W + (size_t)min(n0 + 8 * (g - BM / 4) + r8, a.N - 1) * a.K) + kb + 8 * c8;
        }
        ring_walk2<BM, BN, NST>(nk / 2, lds, acc[0], [&](int p, unsigned char *st) {
#pragma unroll
            for (int j = 0; j < R2::LPW2; j++) lds_load16(src[j] + 64 * p, st + 1024 * (bwave + 2 * NW * j));
        });
    } else {
        const uint16_t *src[LPW];
        int dst[LPW];
#pragma unroll
        for (int j = 0; j < LPW; j++) {
            const int g = wave + NW * j, ga = g < BM / 16 ? g : g - BM / 16;
            src[j] = (g < BM / 8 ? a.A + (size_t)min(m0 + 16 * ga + rr, a.M - 1) * (2 * a.K) + (g < BM / 16 ? 0 : a.K)
                                 : a.W + (size_t)min(n0 + 16 * (g - BM / 8) + rr, a.N - 1) * a.K) + kb + 8 * cl;
            dst[j] = 1024 * g;         // A_hi, A_lo and W groups follow one another
        }
        ring_walk<BM, BN, NST>(nk, lds, acc, [&](int kt, unsigned char *st) {
#pragma unroll
            for (int j = 0; j < LPW; j++) lds_load16(src[j] + kt * QK_GBK, st + dst[j]);
        });
    }

    const int wm = wave / WGN, wn = wave % WGN, mr = m0 + wm * 32 + 16 * kg + 4 * (lane >> 4);
    const bool odd = lane & 1;
    float bias[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + wn * WTN + j * 16 + (lane & 15);
        bias[j] = EPI != ENC_PART && a.bias ? a.bias[min(n, a.N - 1)] : 0.0f;
    }
    bool pad[NI][4];
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) pad[i][r] = GATHER && EPI == ENC_GELU && enc_ring_pad(a, mr + 16 * i + r);
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = acc[i][j][r];
                if (EPI != ENC_PART) v += bias[j];
                if (EPI == ENC_GELU) v = pad[i][r] ? 0.0f : enc_gelu(v);
                acc[i][j][r] = v;
            }
    if constexpr (EPI == ENC_PART || EPI == ENC_F32) {
        float *y = EPI == ENC_PART ? a.ws + (size_t)blockIdx.z * a.M * a.N : a.C;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int m = mr + 16 * i + r, n = n0 + wn * WTN + j * 16 + (lane & 15);
                    if (m < a.M && n < a.N) y[(size_t)m * a.N + n] = acc[i][j][r];
                }
    } else {
        // columns n and n ^ 1 lie in neighbouring lanes (N is even): the even one
        // stores both hi halves, the odd one both lo halves
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int m = mr + 16 * i + r, n = n0 + wn * WTN + j * 16 + (lane & 15);
                    const float v = acc[i][j][r], pv = dpp_read<0xB1>(v);
                    uint32_t h, l;
                    bf16_split2(odd ? pv : v, odd ? v : pv, h, l);
                    if (m < a.M && n < a.N)
                        *reinterpret_cast<uint32_t *>(a.out + (size_t)m * 2 * a.N + (GATHER ? n + (n & ~31) : n) +
                                                      (odd ? (GATHER ? 32 : a.N) - 1 : 0)) = odd ? l : h;
                }
    }
}

// Split-K partials summed in slice order, then the epilogue: 4 columns a thread.
__global__ __launch_bounds__(256) void enc_ring_reduce(qk_enc_ring_args a) {
    const long MN = (long)a.M * a.N, n4 = MN / 4;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n4; e += (long)gridDim.x * 256) {
        const float4 s = sum_splits4<QK_ENC_RING_SPLIT>(a.ws + 4 * e, a.split, MN);
        const int m = (int)(4 * e / a.N), n = (int)(4 * e % a.N);
        const float4 b = a.bias ? *reinterpret_cast<const float4 *>(a.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
        float4 v = make_float4(s.x + b.x, s.y + b.y, s.z + b.z, s.w + b.w);
        if (a.gelu) v = make_float4(enc_gelu(v.x), enc_gelu(v.y), enc_gelu(v.z), enc_gelu(v.w));
        if (enc_ring_pad(a, m)) v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (a.C) *reinterpret_cast<float4 *>(a.C + 4 * e) = v;
        else if (a.taps) enc_store_halves<true>(a.out + (size_t)m * 2 * a.N, a.N, n, v);
        else enc_store_halves<false>(a.out + (size_t)m * 2 * a.N, a.N, n, v);
    }
}

// x = (x +) sum of the partials + bias (+ the positions' table), then its
// LayerNorm as halves: one block per row, N <= 1024, 4 columns a thread.
__global__ __launch_bounds__(256) void enc_ring_reduce_ln(qk_enc_ring_args a) {
    __shared__ float red[2][4];
    const int m = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = 4 * threadIdx.x;
    const bool on = n < a.N;
    const int nc = on ? n : 0;
    float *xr = a.C + (size_t)m * a.N + nc;
    const float4 w = *reinterpret_cast<const float4 *>(a.ln_w + nc), b = *reinterpret_cast<const float4 *>(a.ln_b + nc);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f), o = v, p = v;
    if (a.bias) v = *reinterpret_cast<const float4 *>(a.bias + nc);
    if (a.pe) p = *reinterpret_cast<const float4 *>(a.pe + (size_t)(m % a.pe_rows) * a.N + nc);
    if (a.add) o = *reinterpret_cast<const float4 *>(xr);
    const float4 s = sum_splits4<QK_ENC_RING_SPLIT>(a.ws + (size_t)m * a.N + nc, a.split, (long)a.M * a.N);
    v.x = ((s.x + v.x) + p.x) + o.x;
    v.y = ((s.y + v.y) + p.y) + o.y;
    v.z = ((s.z + v.z) + p.z) + o.z;
    v.w = ((s.w + v.w) + p.w) + o.w;
    if (on) *reinterpret_cast<float4 *>(xr) = v;
    else v = make_float4(0.f, 0.f, 0.f, 0.f);
    float t = wave_sum((v.x + v.y) + (v.z + v.w));
    if (lane == 0) red[0][wave] = t;
    __syncthreads();
    const float mean = (red[0][0] + red[0][1] + red[0][2] + red[0][3]) / (float)a.N;
    const float dx = v.x - mean, dy = v.y - mean, dz = v.z - mean, dw = v.w - mean;
    t = wave_sum(on ? fmaf(dw, dw, fmaf(dz, dz, fmaf(dy, dy, dx * dx))) : 0.0f);
    if (lane == 0) red[1][wave] = t;
    __syncthreads();
    const float var = (red[1][0] + red[1][1] + red[1][2] + red[1][3]) / (float)a.N;
    const float inv = 1.0f / sqrtf(var + a.ln_eps);
    if (on)
        enc_store_halves<false>(a.out + (size_t)m * 2 * a.N, a.N, n,
                         make_float4(dx * inv * w.x + b.x, dy * inv * w.y + b.y, dz * inv * w.z + b.z,
                                     dw * inv * w.w + b.w));
}

// Products with their own epilogue over few rows: 32 x 64 tiles, unsplit, on at
// most one block per CU, whose ring of 8 stages keeps the loads in flight that a
// split's extra blocks did: no partials, no reduce pass.  Whole encoder against
// split 64 x 128 tiles: 1.7B shape, 97 rows 1364 -> 1194 us, 47 rows 1254 -> 1134,
// 156 rows 1588 -> 1466; 0.6B, 97 rows 1062 -> 899; with few blocks (8 rows, 42 of
// them; 32-row tiles before) 728 -> 714.
static bool enc_ring_narrow(int M, int N, int K) {
    const long blocks = (long)((M + 31) / 32) * ((N + 63) / 64);
    return K % 64 == 0 && K <= QK_ENC_RING_FUSED * QK_GBK && blocks >= QK_ENC_NARROW_MIN && blocks <= 256;
}

// Tile, split and k groups of an M x N x K product.  64-row tiles (32 up to 32
// rows; 128 where those alone give every CU a block).  K is split while the launch
// stays within QK_ENC_RING_TARGET blocks, one per CU (fc2 at 390 rows: 294 blocks
// in six splits 18.2 us, 245 in five 14.2), k walks of 4 k tiles at least.  A
// product whose epilogue needs no reduce pass (`fused`) and walks up to
// QK_ENC_RING_FUSED k tiles is not cut in two: that saves 3.5 us, the reduce takes
// 4.5.  Launches of at most one block per CU take 64-deep stages and two k groups.
extern "C" void qk_enc_ring_plan_for(int M, int N, int K, int fused, int gather, long ws_elems, qk_enc_ring_plan *p) {
    if (fused && !gather && enc_ring_narrow(M, N, K)) {
        *p = {.bm = 32, .bn = 64, .groups = 2, .kc = K, .split = 1};
        return;
    }
    const long nt = (N + 127) / 128;
    p->bm = M <= 32 && !gather ? 32 : (long)((M + 127) / 128) * nt >= 256 ? 128 : 64;
    p->bn = 128;
    const long tiles = (M + p->bm - 1) / p->bm * nt;
    const int kt = K / QK_GBK;
    long ns = QK_ENC_RING_TARGET / tiles;
    if (fused && ns <= 2 && kt <= QK_ENC_RING_FUSED) ns = 1;
    if (ns > QK_ENC_RING_SPLIT) ns = QK_ENC_RING_SPLIT;
    if (ns > kt / 4) ns = kt / 4;
    while (ns > 1 && ns * M * N > ws_elems) ns--;
    if (ns < 1) ns = 1;
    int per = (int)((kt + ns - 1) / ns);
    if (K % 64 == 0) per += per & 1;      // whole 64-deep stages
    p->kc = per * QK_GBK;
    p->split = (kt + per - 1) / per;
    p->groups = p->bm < 128 && !gather && K % 64 == 0 && p->kc % 64 == 0 && tiles * p->split <= 256 ? 2 : 1;
}

extern "C" int qk_enc_ring_launch(const qk_enc_ring_args *a, float *ws, long ws_elems, hipStream_t s) {
    if (!a || !a->A || !a->W || a->M <= 0 || a->N <= 0 || (a->N & 3) || a->K <= 0 || a->K % QK_GBK) return QWEN_HIP_EINVAL;
    const bool ln = a->ln_w != nullptr, gather = a->taps > 0;
    if (ln ? (!a->ln_b || !a->C || !a->out || !ws || a->N > 1024 || (long)a->M * a->N > ws_elems || (a->pe && a->pe_rows <= 0))
           : (!a->C == !a->out || a->pe || a->add || (a->gelu ? !a->out : !a->C) || (gather && a->C)))
        return QWEN_HIP_EINVAL;
    if (gather && (a->K != a->taps * QK_ENC_CH || (a->taps != 9 && a->taps != a->in_h) || a->taps > 32 || !a->zero ||
                   a->in_h <= 0 || a->in_w <= 0 || (!ln && a->N % 32) ||
                   (a->taps == 9 && (a->col_h <= 0 || a->col_w <= 0 || (long)a->chunks * a->col_h * a->col_w < a->M))))
        return QWEN_HIP_EINVAL;
    if (a->valid > 0 && (!gather || ln || a->col_h <= 0 || a->col_w <= 0)) return QWEN_HIP_EINVAL;   // stem layers only
    qk_enc_ring_plan p;
    qk_enc_ring_plan_for(a->M, a->N, a->K, !ln, gather, ws ? ws_elems : 0, &p);
    qk_enc_ring_args g = *a;
    g.kc = p.kc;
    g.split = p.split;
    g.ws = ln || p.split > 1 ? ws : nullptr;
    const dim3 grid((a->N + p.bn - 1) / p.bn, (a->M + p.bm - 1) / p.bm, p.split);
    if (p.bn == 64) {
        constexpr int threads = 2 * 64 * ring_waves(32, 64);
        if (a->C) enc_ring<32, 64, 8, false, ENC_F32, 2><<<grid, threads, 0, s>>>(g);
        else enc_ring<32, 64, 8, false, ENC_GELU, 2><<<grid, threads, 0, s>>>(g);
        return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
    }
    const int epi = g.ws ? ENC_PART : a->C ? ENC_F32 : ENC_GELU;
#define QK_ENC_RING(BM_, NST_, G_, E_, KG_)                               \
    if (p.bm == BM_ && gather == G_ && epi == E_ && p.groups == KG_)      \
        enc_ring<BM_, 128, NST_, G_, E_, KG_><<<grid, KG_ * 64 * ring_waves(BM_, 128), 0, s>>>(g);
#define QK_ENC_RING_BM(BM_, NST_, G_, KG_) \
    QK_ENC_RING(BM_, NST_, G_, ENC_PART, KG_) QK_ENC_RING(BM_, NST_, G_, ENC_GELU, KG_)
    QK_ENC_RING_BM(128, 3, true, 1) QK_ENC_RING_BM(64, 4, true, 1)
    QK_ENC_RING_BM(128, 3, false, 1) QK_ENC_RING_BM(64, 4, false, 1) QK_ENC_RING_BM(64, 4, false, 2)
    QK_ENC_RING_BM(32, 4, false, 1) QK_ENC_RING_BM(32, 4, false, 2)
    QK_ENC_RING(128, 3, false, ENC_F32, 1) QK_ENC_RING(64, 4, false, ENC_F32, 1)
    QK_ENC_RING(64, 4, false, ENC_F32, 2) QK_ENC_RING(32, 4, false, ENC_F32, 1) QK_ENC_RING(32, 4, false, ENC_F32, 2)
#undef QK_ENC_RING_BM
#undef QK_ENC_RING
    if (ln) {
        enc_ring_reduce_ln<<<a->M, 256, 0, s>>>(g);
    } else if (g.split > 1) {
        long blocks = ((long)a->M * a->N / 4 + 255) / 256;
        enc_ring_reduce<<<(int)(blocks < 4096 ? blocks : 4096), 256, 0, s>>>(g);
    }
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// conv1 (one input channel) from the mel [128][frames], as pixels of halves: a
// thread holds 4 channels' weights and walks units of C1_OW consecutive output
// positions of a row: 3 x (2 C1_OW + 1) mel values (the same for the 120 threads of
// a unit), then 36 multiply-adds, 4 GELUs and a split per position.  Bound by
// those operations and the 4 bytes written per output (46 M outputs of 30 s: 74 us;
// one position at a time, twice the index work, 94).
#define C1_OW 5
__global__ __launch_bounds__(256) void enc_conv1_halves(const float *mel, int kpad, const float *w, const float *b,
                                                        uint16_t *out, int units, int h_in, int w_in, int h_out,
                                                        int w_out, int mel_frames, int chunks, int valid) {
    constexpr int q4 = QK_ENC_CH / 4, NC = 2 * C1_OW + 1;
    // the grid stride is a multiple of q4: a thread keeps one channel quad
    const long i0 = blockIdx.x * 256L + threadIdx.x, stride = (long)gridDim.x * 256;
    const int c0 = 4 * (int)(i0 % q4), du = (int)(stride / q4), upr = (w_out + C1_OW - 1) / C1_OW;
    float wr[4][9], br[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        br[j] = b[c0 + j];
#pragma unroll
        for (int t = 0; t < 9; t++) wr[j][t] = w[(c0 + j) * kpad + t];
    }
    for (int u = (int)(i0 / q4); u < units; u += du) {
        const int ow0 = u % upr * C1_OW, t1 = u / upr, oh = t1 % h_out, c = t1 / h_out;
        float x[3][NC];
#pragma unroll
        for (int y = 0; y < 3; y++) {
            const int ih = 2 * oh - 1 + y;
            const float *row = mel + (long)min(max(ih, 0), h_in - 1) * mel_frames;
#pragma unroll
            for (int k = 0; k < NC; k++) {
                const int iw = 2 * ow0 - 1 + k, f = c * w_in + iw;
                const bool in = ih >= 0 && ih < h_in && iw >= 0 && iw < w_in && f < mel_frames;
                x[y][k] = in ? row[f] : 0.0f;
            }
        }
        uint16_t *o = out + ((size_t)t1 * w_out + ow0) * 2 * QK_ENC_CH;
        const int n = min(C1_OW, w_out - ow0), nv = c == chunks - 1 ? valid - ow0 : C1_OW;
#pragma unroll
        for (int p = 0; p < C1_OW; p++) {
            float v[4] = {br[0], br[1], br[2], br[3]};
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = fmaf(x[t / 3][2 * p + t % 3], wr[j][t], v[j]);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = p < nv ? enc_gelu(v[j]) : 0.0f;
            if (p < n) enc_store_halves<true>(o + p * 2 * QK_ENC_CH, QK_ENC_CH, c0, make_float4(v[0], v[1], v[2], v[3]));
        }
    }
}

extern "C" int qk_enc_conv1_halves_launch(const float *mel, int kpad, const float *w, const float *b, uint16_t *out,
                                          int chunks, int h_in, int w_in, int h_out, int w_out, int mel_frames,
                                          int valid, hipStream_t s) {
    const long rows = (long)chunks * h_out * ((w_out + C1_OW - 1) / C1_OW);
    if (!mel || !w || !b || !out || kpad < 9 || rows <= 0 || rows > 0x7fffffffL || mel_frames <= 0) return QWEN_HIP_EINVAL;
    constexpr int unit = 15;           // blocks: a multiple of 15, so the grid stride is one of 120 (256 * 15 = 32 * 120)
    long blocks = (rows * (QK_ENC_CH / 4) + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    blocks = (blocks + unit - 1) / unit * unit;
    enc_conv1_halves<<<(int)blocks, 256, 0, s>>>(mel, kpad, w, b, out, (int)rows, h_in, w_in, h_out, w_out, mel_frames,
                                                 chunks, valid);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// Weights [rows][ch h] (column c h + f) as the gathering products read them: k =
// f ch + c, [k / 32][row][k % 32].
__global__ __launch_bounds__(256) void enc_tile_weights(const uint16_t *in, uint16_t *out, int rows, int ch, int h, long n) {
    const long e = blockIdx.x * 256L + threadIdx.x;
    if (e >= n) return;
    const int row = (int)(e / 32 % rows), k = (int)(e / 32 / rows) * 32 + (int)(e % 32), f = k / ch, c = k % ch;
    out[e] = in[(long)row * ch * h + c * h + f];
}

extern "C" int qk_enc_tile_weights_launch(const uint16_t *in, uint16_t *out, int rows, int ch, int h, hipStream_t s) {
    const long n = (long)rows * ch * h;
    if (!in || !out || n <= 0 || (ch * h) % 32) return QWEN_HIP_EINVAL;
    enc_tile_weights<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(in, out, rows, ch, h, n);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// ---------------------------------------------------------------------------
// LayerNorm, one block per row (qwen_layer_norm: mean, then mean of squared
// deviations, then (x - mean) * inv_std * w + b).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void enc_layernorm(const float *x, const float *w, const float *b, float *out,
                                                     int D, float eps) {
    __shared__ float red[4];
    const float *xr = x + (long)blockIdx.x * D;
    float *orow = out + (long)blockIdx.x * D;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float s = 0.0f;
    for (int i = threadIdx.x; i < D; i += 256) s += xr[i];
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)D;
    __syncthreads();
    float v = 0.0f;
    for (int i = threadIdx.x; i < D; i += 256) {
        const float d = xr[i] - mean;
        v = fmaf(d, d, v);
    }
    v = wave_sum(v);
    if (lane == 0) red[wave] = v;
    __syncthreads();
    const float var = (red[0] + red[1] + red[2] + red[3]) / (float)D;
    const float inv_std = 1.0f / sqrtf(var + eps);
    for (int i = threadIdx.x; i < D; i += 256) orow[i] = (xr[i] - mean) * inv_std * w[i] + b[i];
}

extern "C" int qk_enc_layernorm_launch(const float *x, const float *w, const float *b, float *out, int rows, int D,
                                       float eps, hipStream_t s) {
    if (!x || !w || !b || !out || rows <= 0 || D <= 0) return QWEN_HIP_EINVAL;
    enc_layernorm<<<rows, 256, 0, s>>>(x, w, b, out, D, eps);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}

// ---------------------------------------------------------------------------
// Windowed bidirectional attention, head_dim 64, on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32).  Block: 16 queries of one window and one head, 4
// waves; wave w takes the keys 32 w + 128 i .. + 32 of the window, two tiles of
// 16.  S^T = K Q^T: lane l holds query l & 15 and keys 4 (l >> 4) + r of a tile,
// the layout the second product takes as its B operand; O^T += V^T P^T with row
// l & 15 of tile dt standing for dim 4 (l & 15) + dt, so a lane's V values of a
// key are one float4 and its results (dims 16 (l >> 4) + 4 r + dt) are 16
// consecutive dims.  Online softmax per wave; the waves' (m, l, o) meet in LDS.
// Bound by latency (104 keys a window: one round of 16 independent 16-byte
// loads per lane, then 64 MFMAs): a window walked by one wave in blocks of 64
// keys with 4-byte V loads took 12.6 us at 390 tokens x 14 heads, this 6.6 (97 x 16: 4.6).
// The result goes out as fp32 or, for the bf16 products, as halves.
// ---------------------------------------------------------------------------
#define EA_Q 16
#define EA_KW 32                  // keys per wave and round
#define EA_LD 68                  // floats per query of a wave's o (16-byte rows, spread over the banks)

__global__ __launch_bounds__(256) void enc_attention(const float *qkv, float *out, uint16_t *out16, int T, int H, int win,
                                                     float scale) {
    constexpr int hd = 64;
    __shared__ float sm[4][EA_Q], sl[4][EA_Q];
    __shared__ __attribute__((aligned(16))) float so[4][EA_Q][EA_LD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = blockIdx.y;
    const int lq = lane & 15, lg = lane >> 4;
    const int tpw = (win + EA_Q - 1) / EA_Q;
    const int ws = (blockIdx.x / tpw) * win, we = min(T, ws + win);
    const int q0 = ws + (blockIdx.x % tpw) * EA_Q;
    if (q0 >= we) return;                              // whole block: a short last window
    const long stride = 3L * H * hd;
    const float *qrow = qkv + (long)min(q0 + lq, T - 1) * stride + h * hd;
    const float *kbase = qkv + (long)H * hd + h * hd, *vbase = qkv + 2L * H * hd + h * hd;

    float4 q[4];                                       // Q^T operand: dims 16 kb + 4 lg + c
#pragma unroll
    for (int kb = 0; kb < 4; kb++) q[kb] = *reinterpret_cast<const float4 *>(qrow + 16 * kb + 4 * lg);
    f32x4 o[4];                                        // O^T: dims 16 lg + 4 r + dt of query lq
#pragma unroll
    for (int dt = 0; dt < 4; dt++) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -1e30f, l = 0.0f;                        // the reference's max_score start

    for (int k0 = ws + EA_KW * wave; k0 < we; k0 += 4 * EA_KW) {
        float4 kk[2][4], vv[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float *krow = kbase + (long)min(k0 + 16 * t + lq, T - 1) * stride + 4 * lg;
#pragma unroll
            for (int kb = 0; kb < 4; kb++) kk[t][kb] = *reinterpret_cast<const float4 *>(krow + 16 * kb);
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                vv[t][c] = *reinterpret_cast<const float4 *>(vbase + (long)min(k0 + 16 * t + 4 * lg + c, T - 1) * stride +
                                                             4 * lq);
        if (k0 + EA_KW > we) {                         // rows past the window weigh 0: not 0 times what they hold
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (k0 + 16 * t + 4 * lg + c >= we) vv[t][c] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float p[2][4];                                 // key k0 + 16 t + 4 lg + r
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < 4; kb++)
#pragma unroll
                for (int c = 0; c < 4; c++) acc = enc_mfma((&kk[t][kb].x)[c], (&q[kb].x)[c], acc);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[t][r] = k0 + 16 * t + 4 * lg + r < we ? acc[r] * scale : -INFINITY;
                mx = fmaxf(mx, p[t][r]);
            }
        }
        mx = xor_max16_32(mx);
        const float mn = fmaxf(m, mx);
        const float corr = __expf(m - mn);
        float sum = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[t][r] = __expf(p[t][r] - mn);
                sum += p[t][r];
            }
        l = fmaf(l, corr, sum);                        // this lane's keys; lane groups summed at the end
        m = mn;
#pragma unroll
        for (int dt = 0; dt < 4; dt++) o[dt] *= corr;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int dt = 0; dt < 4; dt++) o[dt] = enc_mfma((&vv[t][c].x)[dt], p[t][c], o[dt]);
    }
    l = xor_sum16_32(l);
    if (lg == 0) {
        sm[wave][lq] = m;
        sl[wave][lq] = l;
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4 *>(&so[wave][lq][16 * lg + 4 * r]) = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
    __syncthreads();
    // thread: query tid / 16, dims 4 (tid % 16) .. + 3; wave 0 always holds keys, so M is finite
    const int qq = threadIdx.x >> 4, d = 4 * (threadIdx.x & 15);
    const float M = fmaxf(fmaxf(sm[0][qq], sm[1][qq]), fmaxf(sm[2][qq], sm[3][qq]));
    float L = 0.0f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float e = __expf(sm[w][qq] - M);
        const float4 v = *reinterpret_cast<const float4 *>(&so[w][qq][d]);
        L = fmaf(sl[w][qq], e, L);
        acc.x = fmaf(v.x, e, acc.x);
        acc.y = fmaf(v.y, e, acc.y);
        acc.z = fmaf(v.z, e, acc.z);
        acc.w = fmaf(v.w, e, acc.w);
    }
    const int qi = q0 + qq;
    if (qi >= we) return;
    const float inv = 1.0f / L;
    const float4 v = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
    if (out16) enc_store_halves<false>(out16 + (size_t)qi * 2 * H * hd, H * hd, h * hd + d, v);
    else *reinterpret_cast<float4 *>(out + (long)qi * H * hd + h * hd + d) = v;
}

extern "C" int qk_enc_attention_launch(const float *qkv, float *out, uint16_t *out16, int T, int H, int hd, int win,
                                       float scale, hipStream_t s) {
    if (!qkv || !out == !out16 || T <= 0 || H <= 0 || hd != 64 || win <= 0) return QWEN_HIP_EINVAL;
    const long nwin = (T + win - 1) / win, tpw = (win + EA_Q - 1) / EA_Q;
    if (nwin * tpw > 0x7fffffffL) return QWEN_HIP_EINVAL;
    dim3 grid((unsigned)(nwin * tpw), H);
    enc_attention<<<grid, 256, 0, s>>>(qkv, out, out16, T, H, win, scale);
    return hipGetLastError() == hipSuccess ? 0 : QWEN_HIP_EDEVICE;
}
