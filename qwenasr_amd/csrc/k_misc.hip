// Row-wise and element-wise kernels of the prefill, the audio encoder and the
// mel front end, plus the multi-row (prefill / encoder-window) attention.
#include <climits>
#include <cfloat>
#include <cstdlib>

#include "kernels.h"
#include "gemm_common.h"

namespace qasr {

// ---------------------------------------------------------------------------
// LayerNorm rows: avx::layer_norm_row (avx.rs:420-481) in its exact order —
// mean over 2x8 lane accumulators, variance with FMA accumulators, both
// through the hsum tree, then fma((x - mean) * inv, w, b) (hidden % 16 == 0,
// so every element takes the 8-wide path).  One single-wave block per row:
// lane l holds the 16-element slots s = l + 64 c in registers, the row goes
// through LDS transposed so that lanes r < 16 run the reference's sequential
// accumulator chains.
// ---------------------------------------------------------------------------
template <int NS>
__global__ __launch_bounds__(64) void k_layer_norm_rows(float *__restrict__ out, const float *__restrict__ x,
                                                        const float *__restrict__ w, const float *__restrict__ b,
                                                        int H, float eps) {
    __shared__ float T[16 * (64 * NS + 1)];   // rows one float apart beyond nslot: conflict-free reads
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const float *xr = x + row * H;
    float *o = out + row * H;
    const int nslot = H >> 4, ts = nslot + 1;
    float4 xv[NS][4];
#pragma unroll
    for (int c = 0; c < NS; c++) {
        const int sl = lane + 64 * c, se = sl < nslot ? sl : 0;
#pragma unroll
        for (int i = 0; i < 4; i++) xv[c][i] = reinterpret_cast<const float4 *>(xr + 16 * se)[i];
    }
#pragma unroll
    for (int c = 0; c < NS; c++) {
        const int sl = lane + 64 * c;
        if (sl < nslot) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                T[(4 * i) * ts + sl] = xv[c][i].x;
                T[(4 * i + 1) * ts + sl] = xv[c][i].y;
                T[(4 * i + 2) * ts + sl] = xv[c][i].z;
                T[(4 * i + 3) * ts + sl] = xv[c][i].w;
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    const float *t = T + (lane < 16 ? lane : 0) * ts;
    float acc = 0.0f;
    if (lane < 16)
        for (int i = 0; i < nslot; i++) acc = __fadd_rn(acc, t[i]);
    const float mean = div_by_count(avx16_tree(acc), H);
    acc = 0.0f;
    if (lane < 16)
        for (int i = 0; i < nslot; i++) {
            const float d = __fsub_rn(t[i], mean);
            acc = fmaf(d, d, acc);
        }
    const float var = avx16_tree(acc);
    const float inv = __fdiv_rn(1.0f, sqrt_rn(__fadd_rn(div_by_count(var, H), eps)));
#pragma unroll
    for (int c = 0; c < NS; c++) {
        const int sl = lane + 64 * c;
        if (sl < nslot) {
            float4 *op = reinterpret_cast<float4 *>(o + 16 * sl);
            const float4 *wp = reinterpret_cast<const float4 *>(w + 16 * sl);
            const float4 *bp = reinterpret_cast<const float4 *>(b + 16 * sl);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 a = xv[c][i], ww = wp[i], bb = bp[i];
                op[i] = make_float4(fmaf(__fmul_rn(__fsub_rn(a.x, mean), inv), ww.x, bb.x),
                                    fmaf(__fmul_rn(__fsub_rn(a.y, mean), inv), ww.y, bb.y),
                                    fmaf(__fmul_rn(__fsub_rn(a.z, mean), inv), ww.z, bb.z),
                                    fmaf(__fmul_rn(__fsub_rn(a.w, mean), inv), ww.w, bb.w));
            }
        }
    }
}

hipError_t launch_layer_norm_rows(float *out, const float *x, const float *w, const float *b, int64_t seq,
                                  int hidden, float eps, hipStream_t st) {
    if (hidden % 16 != 0 || hidden > 4096 || seq <= 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)seq);
    switch ((hidden + 1023) / 1024) {
        case 1: hipLaunchKernelGGL(k_layer_norm_rows<1>, grid, dim3(64), 0, st, out, x, w, b, hidden, eps); break;
        case 2: hipLaunchKernelGGL(k_layer_norm_rows<2>, grid, dim3(64), 0, st, out, x, w, b, hidden, eps); break;
        case 3: hipLaunchKernelGGL(k_layer_norm_rows<3>, grid, dim3(64), 0, st, out, x, w, b, hidden, eps); break;
        default: hipLaunchKernelGGL(k_layer_norm_rows<4>, grid, dim3(64), 0, st, out, x, w, b, hidden, eps); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// SwiGLU over rows of interleaved gate/up (swiglu_multiply, mod.rs:1291-1341 ->
// avx::swiglu_interleaved, avx.rs:568-599): fast_exp on 8-wide blocks, libm
// expf on the tail.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_swiglu_rows(float *__restrict__ out, const float *__restrict__ gu,
                                                     int64_t seq, int inter) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= seq * inter) return;
    const int64_t s = i / inter;
    const int j = (int)(i % inter);
    const float g = gu[s * 2 * inter + 2 * j], u = gu[s * 2 * inter + 2 * j + 1];
    const int nv = inter - inter % 8;
    const float e = j < nv ? fast_exp_ref(__fsub_rn(0.0f, g)) : expf(-g);
    out[i] = __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, e)), u);
}

hipError_t launch_swiglu_rows(float *out, const float *gu, int64_t seq, int inter, hipStream_t st) {
    const int64_t n = seq * inter;
    hipLaunchKernelGGL(k_swiglu_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, out, gu, seq, inter);
    return hipGetLastError();
}

// gelu in place over a buffer of n elements (gelu, mod.rs:1250-1289)
__global__ __launch_bounds__(256) void k_gelu(float *__restrict__ x, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) x[i] = gelu_ref(x[i], i, n);
}

hipError_t launch_gelu(float *x, int64_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_gelu, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, n);
    return hipGetLastError();
}

// y[r][c] += table[r % period][c]  (add_inplace of the per-chunk sinusoidal PE)
__global__ __launch_bounds__(256) void k_add_periodic(float *__restrict__ y, const float *__restrict__ table,
                                                      int64_t rows, int cols, int period) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * cols) return;
    const int64_t r = i / cols;
    const int c = (int)(i % cols);
    y[i] = __fadd_rn(y[i], table[(r % period) * cols + c]);
}

hipError_t launch_add_periodic(float *y, const float *table, int64_t rows, int cols, int period, hipStream_t st) {
    const int64_t n = rows * cols;
    hipLaunchKernelGGL(k_add_periodic, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, table, rows, cols, period);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// im2col for a batch of independent 3x3 / stride-2 / pad-1 convolutions
// (conv2d, mod.rs:1077-1154), transposed: cols[(c * Ho + oh) * Wo + ow][p] with
// p = (ic * 3 + ki) * 3 + kj.  Input element (c, ic, ih, iw) lives at
//   in + c * cs + ic * chs + ih * rs + iw.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_im2col3x3s2(float *__restrict__ cols, const float *__restrict__ in,
                                                     int n_chunks, int C, int H, int W, int64_t cs, int64_t chs,
                                                     int64_t rs, int Ho, int Wo) {
    const int P = C * 9;
    const int64_t total = (int64_t)n_chunks * Ho * Wo * P;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int p = (int)(i % P);
        const int64_t row = i / P;
        const int ow = (int)(row % Wo);
        const int oh = (int)((row / Wo) % Ho);
        const int c = (int)(row / ((int64_t)Wo * Ho));
        const int ic = p / 9, ki = (p % 9) / 3, kj = p % 3;
        const int ih = oh * 2 + ki - 1, iw = ow * 2 + kj - 1;
        float v = 0.0f;
        if (ih >= 0 && ih < H && iw >= 0 && iw < W) v = in[c * cs + ic * chs + (int64_t)ih * rs + iw];
        cols[i] = v;
    }
}

// the same patches with one block per output position (row) and the threads
// over its C * 9 columns: the position is decoded once per block and the
// column index needs only 32-bit divisions by constants
__global__ __launch_bounds__(256) void k_im2col3x3s2_rows(float *__restrict__ cols, const float *__restrict__ in,
                                                          int C, int H, int W, int64_t cs, int64_t chs, int64_t rs,
                                                          int Ho, int Wo) {
    const int P = C * 9;
    const int row = blockIdx.x;
    const int ow = row % Wo, oh = (row / Wo) % Ho, c = row / (Wo * Ho);
    const float *src = in + c * cs;
    float *dst = cols + (int64_t)row * P;
    for (int p = threadIdx.x; p < P; p += 256) {
        const int ic = p / 9, r9 = p - 9 * ic, ki = r9 / 3, kj = r9 - 3 * ki;
        const int ih = oh * 2 + ki - 1, iw = ow * 2 + kj - 1;
        float v = 0.0f;
        if (ih >= 0 && ih < H && iw >= 0 && iw < W) v = src[ic * chs + (int64_t)ih * rs + iw];
        dst[p] = v;
    }
}

// the same patches by output row strips: a block owns the Wo positions of one
// output row (chunk c, row oh) and walks the channels 32 at a time, staging
// the three input rows 2 oh - 1 .. 2 oh + 1 of those channels in LDS (zero
// columns on both sides, zero rows outside the image), so the input is read
// in contiguous rows once per strip instead of 3-float runs per position, and
// each position's 288 columns of the channel group go out as one contiguous run
constexpr int IM2COL_ICB = 32, IM2COL_XW = 128;
__global__ __launch_bounds__(256) void k_im2col3x3s2_strip(float *__restrict__ cols, const float *__restrict__ in,
                                                           int C, int H, int W, int64_t cs, int64_t chs, int64_t rs,
                                                           int Ho, int Wo) {
    // rows padded to an odd length so that the 9 taps of consecutive columns
    // fall in different LDS banks
    __shared__ float T[IM2COL_ICB][3][IM2COL_XW + 1];
    const int P = C * 9;
    const int c = blockIdx.x / Ho, oh = blockIdx.x % Ho;
    const float *src = in + c * cs;
    float *dst = cols + (int64_t)blockIdx.x * Wo * P;
    const int XW = W + 2;
    // the Wo x nq columns of one channel group; nq is a constant for full groups
    auto emit = [&](int icb, int nq) {
        for (int i = threadIdx.x; i < Wo * nq; i += 256) {
            const int ow = i / nq, q = i - ow * nq;
            const int icl = q / 9, r9 = q - 9 * icl, ki = r9 / 3, kj = r9 - 3 * ki;
            dst[(int64_t)ow * P + icb * 9 + q] = T[icl][ki][2 * ow + kj];
        }
    };
    // grid y splits the channel groups, so that short strips still fill the chip
    const int ngrp = (C + IM2COL_ICB - 1) / IM2COL_ICB, gpy = (ngrp + gridDim.y - 1) / gridDim.y;
    const int ic_end = min(C, (int)(blockIdx.y + 1) * gpy * IM2COL_ICB);
    for (int icb = blockIdx.y * gpy * IM2COL_ICB; icb < ic_end; icb += IM2COL_ICB) {
        const int nb = min(IM2COL_ICB, C - icb);
        __syncthreads();
        // eight loads in flight per thread before their LDS stores
        const int n = nb * 3 * XW;
        for (int i0 = threadIdx.x; i0 < n; i0 += 8 * 256) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int i = i0 + u * 256, ie = i < n ? i : 0;
                const int x = ie % XW, r = ie / XW, ki = r % 3, icl = r / 3;
                const int ih = 2 * oh + ki - 1, iw = x - 1;
                const bool ok = i < n && ih >= 0 && ih < H && iw >= 0 && iw < W;
                v[u] = src[ok ? (int64_t)(icb + icl) * chs + (int64_t)ih * rs + iw : 0];
                v[u] = ok ? v[u] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int i = i0 + u * 256;
                if (i < n) {
                    const int x = i % XW, r = i / XW;
                    T[r / 3][r % 3][x] = v[u];
                }
            }
        }
        __syncthreads();
        if (nb == IM2COL_ICB) emit(icb, IM2COL_ICB * 9);
        else emit(icb, nb * 9);
    }
}

hipError_t launch_im2col3x3s2(float *cols, const float *in, int n_chunks, int C, int H, int W, int64_t cs,
                              int64_t chs, int64_t rs, int Ho, int Wo, hipStream_t st) {
    const int64_t rows = (int64_t)n_chunks * Ho * Wo;
    if (C * 9 >= 256 && W + 2 <= IM2COL_XW && Wo == (W - 1) / 2 + 1 && (int64_t)n_chunks * Ho < (1ll << 31)) {
        // about 4096 blocks: strips x channel splits
        const int strips = n_chunks * Ho, ngrp = (C + IM2COL_ICB - 1) / IM2COL_ICB;
        const int cs_split = std::max(1, std::min(ngrp, (4096 + strips - 1) / strips));
        hipLaunchKernelGGL(k_im2col3x3s2_strip, dim3((unsigned)strips, (unsigned)cs_split), dim3(256), 0, st, cols, in, C,
                           H, W, cs, chs, rs, Ho, Wo);
        return hipGetLastError();
    }
    if (C * 9 >= 256 && rows < (1ll << 31)) {
        hipLaunchKernelGGL(k_im2col3x3s2_rows, dim3((unsigned)rows), dim3(256), 0, st, cols, in, C, H, W, cs, chs, rs,
                           Ho, Wo);
        return hipGetLastError();
    }
    const int64_t total = (int64_t)n_chunks * Ho * Wo * C * 9;
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(k_im2col3x3s2, dim3(blocks), dim3(256), 0, st, cols, in, n_chunks, C, H, W, cs, chs, rs,
                       Ho, Wo);
    return hipGetLastError();
}

// First convolution of the stem (one input channel, 3x3, stride 2, pad 1) +
// bias + GELU computed directly (conv2d, mod.rs:1077-1154, then gelu): a
// block stages one chunk's padded input plane in LDS and produces CONV1_OCB
// output channels of it: a thread holds one position's 9 taps in registers
// and walks the block's channels.  Each output is the f32 FMA chain over the
// taps in im2col column order (ki, kj), plus the bias, then gelu at its index
// in the chunk's [C][Ho][Wo] output (the path choice of gelu_ref, hoisted per
// channel by GeluSpan).  Outputs go to out + c * C * Ho * Wo.
constexpr int CONV1_OCB = 16, CONV1_LDS = 13312;
__global__ __launch_bounds__(256) void k_conv1_direct(float *__restrict__ out, const float *__restrict__ in,
                                                      int64_t cs, int64_t rs, int H, int W,
                                                      const uint16_t *__restrict__ w, const float *__restrict__ bias,
                                                      int C, int Ho, int Wo) {
    __shared__ float X[CONV1_LDS];
    const int c = blockIdx.x, XW = W + 2;
    const float *src = in + c * cs;
    for (int i = threadIdx.x; i < (H + 2) * XW; i += 256) {
        const int r = i / XW, x = i - r * XW, ih = r - 1, iw = x - 1;
        X[i] = (ih >= 0 && ih < H && iw >= 0 && iw < W) ? src[(int64_t)ih * rs + iw] : 0.0f;
    }
    __syncthreads();
    const int plane = Ho * Wo;
    const int64_t n = (int64_t)C * plane;
    float *dst = out + (int64_t)c * n;
    // this block's channels: weights and gelu path choices (plane <= n / 16, C >= 16)
    const int oc0 = blockIdx.y * CONV1_OCB, noc = min(CONV1_OCB, C - oc0);
    __shared__ float wsh[CONV1_OCB][10];
    __shared__ int64_t gsh[CONV1_OCB][3];
    if (threadIdx.x < noc * 9) {
        const int o = threadIdx.x / 9, k = threadIdx.x % 9;
        wsh[o][k] = bf16_to_f32(w[(oc0 + o) * 9 + k]);
    } else if (threadIdx.x >= 160 && threadIdx.x < 160 + noc) {
        const int o = threadIdx.x - 160;
        const GeluSpan gs((int64_t)(oc0 + o) * plane, n);
        wsh[o][9] = bias[oc0 + o];
        gsh[o][0] = gs.b1; gsh[o][1] = gs.ts0; gsh[o][2] = gs.ts1;
    }
    __syncthreads();
    // each thread: one position's 9 taps in registers, then every channel of the block
    for (int sp = threadIdx.x; sp < plane; sp += 256) {
        const int oh = sp / Wo, ow = sp - oh * Wo;
        const float *xp = X + 2 * oh * XW + 2 * ow;
        float xv[9];
#pragma unroll
        for (int ki = 0; ki < 3; ki++)
#pragma unroll
            for (int kj = 0; kj < 3; kj++) xv[ki * 3 + kj] = xp[ki * XW + kj];
        auto value = [&](int o) {
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < 9; k++) acc = fmaf(xv[k], wsh[o][k], acc);
            const int64_t gi = (int64_t)(oc0 + o) * plane + sp;      // the reference's (channel-major) index
            const bool vec = gi < gsh[o][0] ? gi < gsh[o][1] : gi < gsh[o][2];
            return gelu_at(__fadd_rn(acc, wsh[o][9]), vec);
        };
        for (int o = 0; o < noc; o++) dst[(int64_t)(oc0 + o) * plane + sp] = value(o);
    }
}

// The same convolution with channels-last output (the stem's form; the same
// bits).  A block owns 8 output rows of a chunk and 32 channels: a thread keeps
// the 36 weights of 4 channels in registers and walks the positions, 8 threads
// writing one position's 32 channels as a whole 128-byte line.  Bound by the
// FMAs and the GELU, about 45 vector operations per output.  Before, a block
// staged the chunk's whole plane for 16 channels and a thread wrote its
// position's 64 bytes alone (30 chunks of 480 channels 141 us, 2 chunks 40 us a
// call with 60 blocks).
constexpr int CONV1_ROWS = 8, CONV1_XW = 104;
__global__ __launch_bounds__(256) void k_conv1_last(float *__restrict__ out, const float *__restrict__ in, int64_t cs,
                                                    int64_t rs, int H, int W, const uint16_t *__restrict__ w,
                                                    const float *__restrict__ bias, int C, int Ho, int Wo) {
    __shared__ float X[(2 * CONV1_ROWS + 1) * CONV1_XW];
    const int t = threadIdx.x, c = blockIdx.x, r0 = blockIdx.y * CONV1_ROWS;
    const int oc = blockIdx.z * 32 + (t & 7) * 4, XW = W + 2;
    const float *src = in + c * cs;
    const int nr = min(CONV1_ROWS, Ho - r0);
    for (int i = t; i < (2 * nr + 1) * XW; i += 256) {
        const int r = i / XW, x = i - r * XW, ih = 2 * r0 + r - 1, iw = x - 1;
        X[i] = (ih >= 0 && ih < H && iw >= 0 && iw < W) ? src[(int64_t)ih * rs + iw] : 0.0f;
    }
    float wr[4][9], b[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        b[e] = bias[oc + e];
#pragma unroll
        for (int k = 0; k < 9; k++) wr[e][k] = bf16_to_f32(w[(oc + e) * 9 + k]);
    }
    __syncthreads();
    const int plane = Ho * Wo;
    const int64_t n = (int64_t)C * plane;
    const GeluRule gelu(n, true);
    float *dst = out + (int64_t)c * n;
    for (int p = t >> 3; p < nr * Wo; p += 32) {
        const int oh = p / Wo, ow = p - oh * Wo, sp = (r0 + oh) * Wo + ow;
        const float *xp = X + 2 * oh * XW + 2 * ow;
        float xv[9];
#pragma unroll
        for (int ki = 0; ki < 3; ki++)
#pragma unroll
            for (int kj = 0; kj < 3; kj++) xv[ki * 3 + kj] = xp[ki * XW + kj];
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < 9; k++) acc = fmaf(xv[k], wr[e][k], acc);
            v[e] = gelu(__fadd_rn(acc, b[e]), (int64_t)(oc + e) * plane + sp);   // (the channel-major index)
        }
        *reinterpret_cast<f32x4 *>(dst + (int64_t)sp * C + oc) = v;
    }
}

hipError_t launch_conv1_direct(float *out, const float *in, int n_chunks, int64_t cs, int64_t rs, int H, int W,
                               const uint16_t *w, const float *bias, int C, int Ho, int Wo, bool nhwc,
                               hipStream_t st) {
    if ((H + 2) * (W + 2) > CONV1_LDS || Ho != (H - 1) / 2 + 1 || Wo != (W - 1) / 2 + 1 || n_chunks <= 0 || C < 16)
        return hipErrorInvalidValue;
    if (nhwc) {
        if (C % 32 != 0 || (uintptr_t)out % 16 != 0 || W + 2 > CONV1_XW) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_conv1_last,
                           dim3((unsigned)n_chunks, (unsigned)((Ho + CONV1_ROWS - 1) / CONV1_ROWS), (unsigned)(C / 32)),
                           dim3(256), 0, st, out, in, cs, rs, H, W, w, bias, C, Ho, Wo);
        return hipGetLastError();
    }
    const dim3 grid((unsigned)n_chunks, (unsigned)((C + CONV1_OCB - 1) / CONV1_OCB));
    hipLaunchKernelGGL(k_conv1_direct, grid, dim3(256), 0, st, out, in, cs, rs, H, W, w, bias, C, Ho, Wo);
    return hipGetLastError();
}

// w[o][c][t] (bf16) -> the fragment-major weights (launch_pack_frag's layout) of
// the channels-last implicit-im2col GEMM, whose K index is (tap, channel);
// rows past O (a last partial group of 16) are zeros.  Cin % 32 == 0.
__global__ __launch_bounds__(256) void k_taps_last(uint16_t *__restrict__ out, const uint16_t *__restrict__ in,
                                                   int O, int Cin, int T) {
    const int nk = Cin / 32 * T;
    const int64_t total = (int64_t)((O + 15) / 16) * nk * 512;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int e = (int)(i & 511), l = e >> 3;
        const int64_t f = i >> 9;
        const int o = (int)(f / nk) * 16 + (l & 15), k = (int)(f % nk) * 32 + (l >> 4) * 8 + (e & 7);
        const int t = k / Cin, c = k - t * Cin;
        out[i] = o < O ? in[((int64_t)o * Cin + c) * T + t] : (uint16_t)0;
    }
}

hipError_t launch_taps_last(uint16_t *out, const uint16_t *in, int O, int Cin, int T, hipStream_t st) {
    if (O <= 0 || Cin <= 0 || Cin % 32 != 0 || T <= 0) return hipErrorInvalidValue;
    const int64_t total = (int64_t)gemm_frag_rows(O) * Cin * T;
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(k_taps_last, dim3(blocks), dim3(256), 0, st, out, in, O, Cin, T);
    return hipGetLastError();
}

// [chunk][C][F][T] -> [chunk * T][C * F] with column ch * F + f (encoder.rs:265-277)
__global__ __launch_bounds__(256) void k_conv_reshape(float *__restrict__ out, const float *__restrict__ in,
                                                      int n_chunks, int C, int F, int T) {
    const int64_t total = (int64_t)n_chunks * C * F * T;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int col = (int)(i % (C * F));
        const int64_t row = i / (C * F);
        const int t = (int)(row % T);
        const int c = (int)(row / T);
        const int ch = col / F, f = col % F;
        out[i] = in[(((int64_t)c * C + ch) * F + f) * T + t];
    }
}

hipError_t launch_conv_reshape(float *out, const float *in, int n_chunks, int C, int F, int T, hipStream_t st) {
    const int64_t total = (int64_t)n_chunks * C * F * T;
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(k_conv_reshape, dim3(blocks), dim3(256), 0, st, out, in, n_chunks, C, F, T);
    return hipGetLastError();
}

// prompt rows: row r < n_tok_head: embed[tok[r]]; then n_mid rows copied from
// mid; then the remaining token rows (transcribe.rs:106-169)
__global__ __launch_bounds__(256) void k_build_prompt(float *__restrict__ out, const uint16_t *__restrict__ embed,
                                                      const int *__restrict__ toks, int n_head, const float *mid,
                                                      int n_mid, int n_tail, int H) {
    const int r = blockIdx.x;
    float *o = out + (int64_t)r * H;
    if (r < n_head || r >= n_head + n_mid) {
        const int ti = r < n_head ? r : r - n_mid;
        const uint16_t *e = embed + (int64_t)toks[ti] * H;
        for (int i = threadIdx.x; i < H; i += 256) o[i] = bf16_to_f32(e[i]);
    } else {
        const float *m = mid + (int64_t)(r - n_head) * H;
        for (int i = threadIdx.x; i < H; i += 256) o[i] = m[i];
    }
    (void)n_tail;
}

// flags[r] = 1 when rows r of a and b differ in any bit (the row-equality test
// of the streaming prefill's prefix reuse, transcribe.rs:1095-1104)
__global__ __launch_bounds__(256) void k_row_diff(const float *__restrict__ a, const float *__restrict__ b,
                                                  int64_t H, int *__restrict__ flags) {
    __shared__ int any;
    const int64_t r = blockIdx.x;
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    const uint32_t *pa = reinterpret_cast<const uint32_t *>(a + r * H), *pb = reinterpret_cast<const uint32_t *>(b + r * H);
    int d = 0;
    for (int64_t i = threadIdx.x; i < H; i += 256) d |= pa[i] != pb[i];
    if (d) any = 1;
    __syncthreads();
    if (threadIdx.x == 0) flags[r] = any;
}

hipError_t launch_row_diff(const float *a, const float *b, int64_t rows, int64_t H, int *flags, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_row_diff, dim3((unsigned)rows), dim3(256), 0, st, a, b, H, flags);
    return hipGetLastError();
}

// idx[r] = the aligner's per-row argmax of x[r] (align.rs:312-321): a left
// scan that starts at column 0 and moves on only for a strictly greater value,
// i.e. the lowest column holding the maximum of the non-NaN values, and 0 when
// column 0 is NaN (nothing compares greater than it).  A lane scans a strided
// column set in increasing order; pairs merge by value, then lowest column.
__device__ inline void argmax_pick(float &v, int &i, float ov, int oi) {
    if (oi == INT_MAX) return;
    if (i == INT_MAX || ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
}

__global__ __launch_bounds__(256) void k_argmax_f32_rows(const float *__restrict__ x, int64_t ld, int64_t cols,
                                                         int32_t *__restrict__ idx) {
    __shared__ float sv[4];
    __shared__ int si[4];
    const float *row = x + blockIdx.x * ld;
    float v = 0.0f;
    int i = INT_MAX;
    for (int64_t c = threadIdx.x; c < cols; c += 256) {
        const float y = row[c];
        if (y == y && (i == INT_MAX || y > v)) { v = y; i = (int)c; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) argmax_pick(v, i, __shfl_xor(v, o), __shfl_xor(i, o));
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sv[w] = v; si[w] = i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; k++) argmax_pick(v, i, sv[k], si[k]);
        const float c0 = row[0];
        idx[blockIdx.x] = (c0 != c0 || i == INT_MAX) ? 0 : i;
    }
}

hipError_t launch_argmax_f32_rows(const float *x, int64_t ld, int64_t rows, int64_t cols, int32_t *idx,
                                  hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_argmax_f32_rows, dim3((unsigned)rows), dim3(256), 0, st, x, ld, cols, idx);
    return hipGetLastError();
}

// dst[k] = src[rows[k]] for k < n, rows of H floats
__global__ __launch_bounds__(256) void k_gather_rows(float *__restrict__ dst, const float *__restrict__ src,
                                                     const int32_t *__restrict__ rows, int64_t H) {
    const float *s = src + (int64_t)rows[blockIdx.x] * H;
    float *d = dst + (int64_t)blockIdx.x * H;
    for (int64_t c = threadIdx.x; c < H; c += 256) d[c] = s[c];
}

hipError_t launch_gather_rows(float *dst, const float *src, const int32_t *rows, int64_t n, int64_t H,
                              hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)n), dim3(256), 0, st, dst, src, rows, H);
    return hipGetLastError();
}

hipError_t launch_build_prompt(float *out, const uint16_t *embed, const int *toks, int n_head, const float *mid,
                               int n_mid, int n_tail, int H, hipStream_t st) {
    hipLaunchKernelGGL(k_build_prompt, dim3(n_head + n_mid + n_tail), dim3(256), 0, st, out, embed, toks, n_head,
                       mid, n_mid, n_tail, H);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Multi-row attention (flash-style online softmax, f32):
//   decoder prefill: causal over the KV cache, GQA (causal_attention with
//                    seq_q > 1, mod.rs:1539-1607)
//   encoder:         full attention inside fixed windows (bidirectional_attention,
//                    mod.rs:1386-1471)
// A block owns 32 query rows (QT queries x G heads of one KV head) and walks key
// tiles of 32; 8 threads per row.
// ---------------------------------------------------------------------------
// The rows [s0, s1) of the sequence that row q belongs to: the whole call, or
// with n_seg > 0 the last sequence starting at or before q (compile-time
// indices only, so the tables stay in the kernel arguments)
__device__ __forceinline__ void attn_sequence(const AttnRowsArgs &a, int q, int &s0, int &s1) {
    s0 = 0;
    s1 = min(a.n_q, a.n_k);
    if (a.n_seg > 0) {
#pragma unroll
        for (int j = 0; j < QASR_ATTN_MAX_SEG; j++)
            if (j < a.n_seg && a.seg_lo[j] <= q) {
                s0 = a.seg_lo[j];
                s1 = a.seg_hi[j];
            }
    }
}

template <int HD>
__global__ __launch_bounds__(256) void k_attn_rows(AttnRowsArgs a) {
    constexpr int R = 32, KT = 32, DP = HD / 8;
    __shared__ float Qs[R][HD + 4];
    __shared__ float Ks[KT][HD + 4];
    __shared__ float Vs[KT][HD + 4];
    __shared__ float Ps[R][KT + 1];
    const int t = threadIdx.x, r = t >> 3, sub = t & 7;
    const int G = a.G, QT = R / G;
    const int kvh = blockIdx.x, q0 = blockIdx.y * QT;
    const int qi = q0 + r / G, h = kvh * G + r % G;
    // the block's sequence (windowed calls; blocks never straddle two)
    int s0 = 0, s1 = a.n_q;
    if (a.window > 0) attn_sequence(a, q0, s0, s1);
    const bool row_ok = qi < a.n_q && qi < s1;
    // key range of this row
    int lo = 0, hi;
    if (a.window > 0) {
        lo = s0 + ((qi - s0) / a.window) * a.window;
        hi = min(lo + a.window, min(a.n_k, s1));
    } else {
        hi = min(a.q_offset + qi + 1, a.n_k);
    }
    if (!row_ok) { lo = 0; hi = 0; }
    // key range of the block
    const int qlast = min(q0 + QT, min(a.n_q, s1)) - 1;
    int blo, bhi;
    if (a.window > 0) {
        blo = s0 + ((q0 - s0) / a.window) * a.window;
        bhi = min(s0 + ((qlast - s0) / a.window) * a.window + a.window, min(a.n_k, s1));
    } else {
        blo = 0;
        bhi = min(a.q_offset + qlast + 1, a.n_k);
    }
    for (int i = t; i < R * HD; i += 256) {
        const int rr = i / HD, d = i % HD;
        const int qq = q0 + rr / G, hh = kvh * G + rr % G;
        Qs[rr][d] = qq < a.n_q ? a.q[(int64_t)qq * a.q_rs + hh * HD + d] : 0.0f;
    }
    float m = -INFINITY, l = 0.0f, o[DP];
#pragma unroll
    for (int i = 0; i < DP; i++) o[i] = 0.0f;
    const float *kb = a.k + (int64_t)kvh * a.k_hs, *vb = a.v + (int64_t)kvh * a.k_hs;
    for (int j0 = blo; j0 < bhi; j0 += KT) {
        __syncthreads();
        for (int i = t; i < KT * HD; i += 256) {
            const int kk = i / HD, d = i % HD;
            const int j = j0 + kk;
            const bool ok = j < bhi;
            const int64_t off = (int64_t)(ok ? j : j0) * a.k_rs + d;
            const float kv = kb[off], vv = vb[off];
            Ks[kk][d] = ok ? kv : 0.0f;
            Vs[kk][d] = ok ? vv : 0.0f;
        }
        __syncthreads();
        float s[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int kk = sub * 4 + c;
            float acc = 0.0f;
#pragma unroll 8
            for (int d = 0; d < HD; d++) acc = fmaf(Qs[r][d], Ks[kk][d], acc);
            const int j = j0 + kk;
            s[c] = (j >= lo && j < hi) ? __fmul_rn(acc, a.scale) : -INFINITY;
        }
        float tm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        tm = fmaxf(tm, __shfl_xor(tm, 1, 64));
        tm = fmaxf(tm, __shfl_xor(tm, 2, 64));
        tm = fmaxf(tm, __shfl_xor(tm, 4, 64));
        const float mn = fmaxf(m, tm);
        float corr = 1.0f, ps = 0.0f;
        if (mn != -INFINITY) {
            corr = m == -INFINITY ? 0.0f : expf(__fsub_rn(m, mn));
#pragma unroll
            for (int c = 0; c < 4; c++) {
                s[c] = s[c] == -INFINITY ? 0.0f : expf(__fsub_rn(s[c], mn));
                ps = __fadd_rn(ps, s[c]);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; c++) s[c] = 0.0f;
        }
        ps = __fadd_rn(ps, __shfl_xor(ps, 1, 64));
        ps = __fadd_rn(ps, __shfl_xor(ps, 2, 64));
        ps = __fadd_rn(ps, __shfl_xor(ps, 4, 64));
        l = fmaf(l, corr, ps);
        m = mn;
#pragma unroll
        for (int c = 0; c < 4; c++) Ps[r][sub * 4 + c] = s[c];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < DP; i++) o[i] = __fmul_rn(o[i], corr);
        for (int kk = 0; kk < KT; kk++) {
            const float p = Ps[r][kk];
#pragma unroll
            for (int i = 0; i < DP; i++) o[i] = fmaf(p, Vs[kk][sub * DP + i], o[i]);
        }
    }
    if (row_ok) {
        float *op = a.out + (int64_t)qi * a.o_rs + h * HD + sub * DP;
        const float inv = l > 0.0f ? __fdiv_rn(1.0f, l) : 0.0f;
#pragma unroll
        for (int i = 0; i < DP; i++) op[i] = __fmul_rn(o[i], inv);
    }
}

// e^x for 0 >= x >= -2.36e38 (the bf16-term softmax's x - max): 2^(x log2 e) with
// the product's rounding error and log2 e's second term carried to first order,
// within 1.5 ulp, in half the operations of expf; results below 2^-126 become
// 0.  Below that range (scores 2.36e38 or more apart) it is NaN, and the caller
// forms the row again with expf; a cut-off here (fminf of the correction) cost
// 2-5% of a short call's attention.
__device__ __forceinline__ float exp_neg(float x) {
    constexpr float L = 0x1.715476p+0f, LL = 0x1.4ae0cp-26f;       // log2 e = L + LL
    const float p = __fmul_rn(x, L);
    const float r = fmaf(x, LL, fmaf(x, L, -p));
    const float e = __builtin_amdgcn_exp2f(p);
    return fmaf(e, __fmul_rn(r, 0x1.62e43p-1f), e);
}

// ---------------------------------------------------------------------------
// The same multi-row attention on f32 MFMA (v_mfma_f32_16x16x4_f32, exact f32
// products, f32 accumulation): the encoder's windowed attention.  A block owns
// 16 query rows of one head; its NW waves split the keys: wave w takes the
// 16-key sub-tiles w, w + NW, ... with an online softmax of its own, and the NW
// states are merged through LDS at the end.
//
// Every wave streams its sub-tiles alone through an LDS stage of its own: K by
// global_load_lds, refilled as soon as its fragments are in registers, and V
// the same way, so that the next K rows travel during this sub-tile's softmax
// and P V and the next V rows during the next scores; no barrier before the
// merge.  (Before, the block staged 128-key chunks through registers: load,
// LDS store, barrier, compute in turn, the matrix cores idle for half of each
// chunk.)  What bounds it: 64 MFMAs of 32 clk per sub-tile, 145 TFLOP/s over
// the chip at best, and for short prompts the longest block's chain.
//
// Per sub-tile the wave forms S^T = K Q^T (16 keys x 16 queries; lane l holds
// keys 4 (l / 16) + i of query l % 16, the dot over d split as lane group l /
// 16 covering dims [l/16 HD/4, +HD/4)), so the softmax of a query reduces over
// the lane's 4 values and two cross-group shuffles, and the probabilities
// already sit in the A-operand layout of O += P V (query l % 16, key 4 (l / 16)
// + i at step i).  Column l % 16 of the B operand's tile n is dim NT (l % 16)
// + n: a lane reads its NT values of a V row as whole 16-byte slots.  The O
// rows a lane accumulates are queries 4 (l / 16) + j, whose rescale factors
// come from the lanes owning those queries.
//
// LDS placement: slot q (16 bytes) of K row r sits at q ^ (r & 7): the 16 rows
// of a fragment read fall in different banks; V rows are read along the row.
// ---------------------------------------------------------------------------
template <int HD, int NW>
__global__ __launch_bounds__(NW * 64) void k_attn_mfma(AttnRowsArgs a) {
    constexpr int NST = HD / 4, NT = HD / 16;
    constexpr int RB = HD * 4, TB = 16 * RB;               // bytes of a K or V row, of a 16-key tile
    constexpr int LPR = RB / 16, RPL = 64 / LPR, L = 16 / RPL;   // lanes per row, rows per load, loads per tile
    __shared__ __attribute__((aligned(16))) char smem[NW * 2 * TB];
    __shared__ float Mm[NW][16], Ll[NW][16], Ff[NW][16];
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h = blockIdx.x, q0 = blockIdx.y * 16;
    const int lq = lane & 15, lg = lane >> 4;
    // key range of this lane's query (for the S^T masks) and of the block
    const int qi = q0 + lq;
    // the block's sequence (blocks never straddle two)
    int s0 = 0, s1 = a.n_q;
    attn_sequence(a, q0, s0, s1);
    int lo = 0, hi = 0;
    if (qi < a.n_q && qi < s1) {
        lo = s0 + ((qi - s0) / a.window) * a.window;
        hi = min(lo + a.window, min(a.n_k, s1));
    }
    const int qlast = min(q0 + 16, min(a.n_q, s1)) - 1;
    if (qlast < q0) return;                 // padding rows between two sequences
    const int blo = s0 + ((q0 - s0) / a.window) * a.window;
    const int bhi = min(s0 + ((qlast - s0) / a.window) * a.window + a.window, min(a.n_k, s1));
    const float *kb = a.k + (int64_t)h * a.k_hs, *vb = a.v + (int64_t)h * a.k_hs;
    char *Ks = smem + wid * 2 * TB, *Vs = Ks + TB;
    // tile c (keys blo + 16 c ...): rows past the range repeat its last one (their scores are masked)
    const int n_sub = (bhi - blo + 15) / 16, lr = lane / LPR, ls = lane % LPR;
    auto issue = [&](const float *base, char *dst, int c, bool swz) {
        const int j0 = blo + 16 * c, last = bhi - 1 - j0;
        const char *p = reinterpret_cast<const char *>(base + (int64_t)j0 * a.k_rs);
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int r = u * RPL + lr;
            const uint32_t off = (uint32_t)min(r, last) * (uint32_t)a.k_rs * 4u + 16 * (swz ? ls ^ (r & 7) : ls);
            lds_dma16_s(p, off, dst + 1024 * u);
        }
    };
    if (wid < n_sub) {
        issue(kb, Ks, wid, true);
        issue(vb, Vs, wid, false);
    }
    // this lane's slice of q: dims [lg NST, lg NST + NST) of query qi, head h
    float qv[NST];
    {
        const float *qp = a.q + (int64_t)min(qi, a.n_q - 1) * a.q_rs + h * HD + lg * NST;
#pragma unroll
        for (int s = 0; s < NST; s += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(qp + s);
            qv[s] = x.x; qv[s + 1] = x.y; qv[s + 2] = x.z; qv[s + 3] = x.w;
        }
    }
#pragma unroll
    for (int s = 0; s < NST; s++) asm volatile("" : "+v"(qv[s]));   // waited for here, not inside the loop
    f32x4 o[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) o[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;
    for (int c = wid; c < n_sub; c += NW) {
        const bool more = c + NW < n_sub;
        wait_vmcnt<L>();                        // the K tile has landed (V's loads are younger)
        float4 kf[NST / 4];
#pragma unroll
        for (int s = 0; s < NST / 4; s++)
            kf[s] = *reinterpret_cast<const float4 *>(Ks + lq * RB + (((lg * (NST / 4) + s) ^ (lq & 7)) * 16));
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(kb, Ks, c + NW, true);
        }
        // S^T[key 4 lg + i][query lq]
        f32x4 st = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < NST; s += 4) {
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s / 4].x, qv[s], st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s / 4].y, qv[s + 1], st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s / 4].z, qv[s + 2], st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s / 4].w, qv[s + 3], st, 0, 0, 0);
        }
        float sv[4], tm = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int j = blo + 16 * c + 4 * lg + i;
            sv[i] = (j >= lo && j < hi) ? __fmul_rn(st[i], a.scale) : -INFINITY;
            tm = fmaxf(tm, sv[i]);
        }
        tm = xhalf_max(xrow16_max(tm));
        const float mn = fmaxf(m, tm);
        const float corr = (m == -INFINITY) ? 0.0f : expf(__fsub_rn(m, mn));
        float ps = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sv[i] = sv[i] == -INFINITY ? 0.0f : expf(__fsub_rn(sv[i], mn));
        }
        ps = __fadd_rn(__fadd_rn(sv[0], sv[1]), __fadd_rn(sv[2], sv[3]));
        ps = xhalf_sum(xrow16_sum(ps));
        l = fmaf(l, corr, ps);
        m = mn;
        // rescale the O rows this lane holds (queries 4 lg + j) by their owners' factors
        float cj[4];
#pragma unroll
        for (int j = 0; j < 4; j++) cj[j] = __shfl(corr, 4 * lg + j, 64);
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int j = 0; j < 4; j++) o[n][j] = __fmul_rn(o[n][j], cj[j]);
        if (more) wait_vmcnt<L>();              // the V tile has landed (the next K's loads are younger)
        else wait_vmcnt<0>();
        float vf[4][NT];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int n = 0; n < NT; n += 4) {
                const float4 x = *reinterpret_cast<const float4 *>(Vs + (4 * lg + i) * RB + (lq * NT + n) * 4);
                vf[i][n] = x.x; vf[i][n + 1] = x.y; vf[i][n + 2] = x.z; vf[i][n + 3] = x.w;
            }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(vb, Vs, c + NW, false);
        }
        // O += P V: step i pairs key 4 lg + i of P (this lane's sv[i]) with V row 4 lg + i
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int n = 0; n < NT; n++) o[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[i], vf[i][n], o[n], 0, 0, 0);
    }
    // merge the NW key splits: (m, l) per query, O rows through LDS (every
    // wave's loads have landed: its last wait was for all of them)
    float *Om = reinterpret_cast<float *>(smem);           // [NW waves][16 rows][HD]
    if (lg == 0) { Mm[wid][lq] = m; Ll[wid][lq] = l; }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int n = 0; n < NT; n += 4)
            *reinterpret_cast<f32x4 *>(Om + (wid * 16 + 4 * lg + j) * HD + lq * NT + n) =
                f32x4{o[n][j], o[n + 1][j], o[n + 2][j], o[n + 3][j]};
    if (t < NW * 16) {
        const int w = t >> 4, r = t & 15;
        float M = -INFINITY;
#pragma unroll
        for (int k2 = 0; k2 < NW; k2++) M = fmaxf(M, Mm[k2][r]);
        Ff[w][r] = Mm[w][r] == -INFINITY ? 0.0f : expf(__fsub_rn(Mm[w][r], M));
    }
    __syncthreads();
    for (int i = t; i < 16 * HD / 4; i += NW * 64) {
        const int r = i / (HD / 4), d = (i % (HD / 4)) * 4;
        const int q = q0 + r;
        if (q >= a.n_q) continue;
        float Ls = 0.0f;
        f32x4 O = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float f = Ff[w][r];
            const f32x4 x = *reinterpret_cast<const f32x4 *>(Om + (w * 16 + r) * HD + d);
            Ls = fmaf(Ll[w][r], f, Ls);
#pragma unroll
            for (int e = 0; e < 4; e++) O[e] = fmaf(x[e], f, O[e]);
        }
        float *op = a.out + (int64_t)q * a.o_rs + h * HD + d;
#pragma unroll
        for (int e = 0; e < 4; e++) op[e] = Ls > 0.0f ? __fdiv_rn(O[e], Ls) : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// The decoder's prefill attention (128-dim heads, two query heads per KV head)
// on bf16 MFMA: q, k, p and v are three bf16 terms each and a product is formed
// from the six term pairs that matter (hi hi, hi mid, mid hi, mid mid, hi lo,
// lo hi; the rest is below 2^-26 of it), accumulated in f32: f32-class like the
// f32 MFMA form above, at 12 MFMAs of 16 clk for its 8 of 32.  The terms of a
// K or V tile are formed once per wave, for the GH query heads (1 or 2) that
// the block owns.
//
// Same streaming as above: 8 waves of their own 16-key sub-tiles, no barrier
// before the merge.  Scores: S^T = K Q^T over 4 steps of 32 dims (lane l: key
// or query l % 16, dims 32 s + 8 (l / 16) .. + 7).  O += P V contracts 16 keys
// with 32-deep MFMAs, so each carries two term pairs: slots 0-3 of a lane are
// its keys 4 (l / 16) + i with the first pair's terms, slots 4-7 the same keys
// with the second's.
//
// What bounds it: per tile and two heads 96 MFMAs (1536 clk) and about 550
// other vector operations (the term splits, the softmax), which fill 56% of the
// issue slots at 1337 rows (MFMA units 20% busy, 31% of the waves' time at waits).
// 1337 rows 163 us on f32 MFMA, 103 with a stage per wave, 78 so.
//
// Its range is narrower than f32's: an infinite value, or one of 3.396e38 or
// more (its bf16 rounding is infinite), has no three terms, and exp_neg has the
// range above.  Each of these leaves NaN in what it meets.  And bf16's smallest
// step is 2^-133: values of v below 2^-109 hold fewer than 24 bits.  So a row
// whose merged sum or result is not finite, or below 2^-96 (but not 0), is formed
// again in plain f32 by the wave that found it (only that row; the others keep
// their bits).  What this does not see: a q or k value below 2^-109 against one
// beyond 2^100, and weights below 2^-126 of the largest, which count as 0.
// The check costs 0.2 us a call (16 rows 6.05 -> 6.25); 1337 rows all formed again
// take 1.9 ms.  (A block's rows formed again together on f32 MFMA, behind a
// barrier for every block, cost 0.3 us a call.)
// ---------------------------------------------------------------------------
// two pairs of f32 -> (hi, mid, lo), two packed dwords each
__device__ __forceinline__ void split3_4(float x0, float x1, float x2, float x3, uint32_t (&hi)[2], uint32_t (&mi)[2],
                                         uint32_t (&lo)[2], bf16x2 e0, bf16x2 e1) {
    const float x[4] = {x0, x1, x2, x3};
#pragma unroll
    for (int e = 0; e < 2; e++) {
        hi[e] = cvt_pk_bf16(x[2 * e], x[2 * e + 1]);
        const bf16x2 h = __builtin_bit_cast(bf16x2, hi[e]);
        const float r0 = __builtin_amdgcn_fdot2_f32_bf16(h, e0, x[2 * e], false);
        const float r1 = __builtin_amdgcn_fdot2_f32_bf16(h, e1, x[2 * e + 1], false);
        mi[e] = cvt_pk_bf16(r0, r1);
        const bf16x2 m = __builtin_bit_cast(bf16x2, mi[e]);
        lo[e] = cvt_pk_bf16(__builtin_amdgcn_fdot2_f32_bf16(m, e0, r0, false),
                            __builtin_amdgcn_fdot2_f32_bf16(m, e1, r1, false));
    }
}

// query q of head h (KV head kv_head, 128 dims) in f32 by one wave: a key per lane
// for the scores, two dims per lane for the result
__device__ __forceinline__ void attn_row_f32(const AttnRowsArgs &a, int q, int h, int kv_head, int lane) {
    constexpr int HD = 128;
    const float *qp = a.q + (int64_t)q * a.q_rs + h * HD;
    const float *kb = a.k + (int64_t)kv_head * a.k_hs, *vb = a.v + (int64_t)kv_head * a.k_hs + 2 * lane;
    const int hi = min(a.q_offset + q + 1, a.n_k);
    float m = -INFINITY, l = 0.0f, o0 = 0.0f, o1 = 0.0f;
    for (int j0 = 0; j0 < hi; j0 += 64) {
        const int j = min(j0 + lane, hi - 1), n = min(64, hi - j0);
        float s = 0.0f;
        for (int d = 0; d < HD; d++) s = fmaf(qp[d], kb[(int64_t)j * a.k_rs + d], s);
        s = lane < n ? __fmul_rn(s, a.scale) : -INFINITY;
        const float mn = fmaxf(m, wave_max_f32(s));
        const float corr = m == -INFINITY ? 0.0f : expf(__fsub_rn(m, mn));
        const float p = s == -INFINITY ? 0.0f : expf(__fsub_rn(s, mn));
        l = fmaf(l, corr, wave_sum_f32(p));
        m = mn;
        o0 = __fmul_rn(o0, corr);
        o1 = __fmul_rn(o1, corr);
        for (int k = 0; k < n; k++) {
            const float pk = __shfl(p, k, 64);
            const float *vp = vb + (int64_t)(j0 + k) * a.k_rs;
            o0 = fmaf(pk, vp[0], o0);
            o1 = fmaf(pk, vp[1], o1);
        }
    }
    float *op = a.out + (int64_t)q * a.o_rs + h * HD + 2 * lane;
    op[0] = l > 0.0f ? __fdiv_rn(o0, l) : 0.0f;
    op[1] = l > 0.0f ? __fdiv_rn(o1, l) : 0.0f;
}

template <int GH>
__device__ __forceinline__ void attn_bf3_block(const AttnRowsArgs &a, int q0) {
    constexpr int HD = 128, NW = 8, NT = HD / 16;
    constexpr int RB = HD * 4, TB = 16 * RB, L = 8;
    __shared__ __attribute__((aligned(16))) char smem[NW * 2 * TB];
    __shared__ float Mm[NW][GH][16], Ll[NW][GH][16], Ff[NW][GH][16];
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h0 = blockIdx.x * GH;
    const int lq = lane & 15, lg = lane >> 4;
    const int qi = q0 + lq;
    const int hi = qi < a.n_q ? min(a.q_offset + qi + 1, a.n_k) : 0;        // this lane's query sees keys [0, hi)
    const int bhi = min(a.q_offset + min(q0 + 16, a.n_q), a.n_k);           // the block's keys
    const int all = min(a.q_offset + q0 + 1, a.n_k);                        // keys that every query of the block sees
    const bool full_rows = q0 + 16 <= a.n_q;
    const int kv_head = h0 / 2;
    const float *kb = a.k + (int64_t)kv_head * a.k_hs, *vb = a.v + (int64_t)kv_head * a.k_hs;
    char *Ks = smem + wid * 2 * TB, *Vs = Ks + TB;
    const int n_sub = (bhi + 15) / 16, lr = lane >> 5, ls = lane & 31;
    auto issue = [&](const float *base, char *dst, int c, bool swz) {
        const int j0 = 16 * c, last = bhi - 1 - j0;
        const char *p = reinterpret_cast<const char *>(base + (int64_t)j0 * a.k_rs);
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int r = 2 * u + lr;
            const uint32_t off = (uint32_t)min(r, last) * (uint32_t)a.k_rs * 4u + 16 * (swz ? ls ^ (r & 7) : ls);
            lds_dma16_s(p, off, dst + 1024 * u);
        }
    };
    if (wid < n_sub) {
        issue(kb, Ks, wid, true);
        issue(vb, Vs, wid, false);
    }
    uint32_t c0, c1;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
    const bf16x2 e0 = __builtin_bit_cast(bf16x2, c0), e1 = __builtin_bit_cast(bf16x2, c1);
    // the queries' terms: [head][step of 32 dims][term]
    bf16x8 qf[GH][4][3];
    {
        float4 x[GH][4][2];
#pragma unroll
        for (int g = 0; g < GH; g++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float *qp = a.q + (int64_t)min(qi, a.n_q - 1) * a.q_rs + (h0 + g) * HD + 32 * s + 8 * lg;
                x[g][s][0] = *reinterpret_cast<const float4 *>(qp);
                x[g][s][1] = *reinterpret_cast<const float4 *>(qp + 4);
            }
#pragma unroll
        for (int g = 0; g < GH; g++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                split3(x[g][s][0], x[g][s][1], qf[g][s]);
#pragma unroll
                for (int e = 0; e < 3; e++) asm volatile("" : "+v"(qf[g][s][e]));   // formed here, not inside the loop
            }
    }
    f32x4 o[GH][NT];
    float m[GH], l[GH];
#pragma unroll
    for (int g = 0; g < GH; g++) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int n = 0; n < NT; n++) o[g][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int c = wid; c < n_sub; c += NW) {
        const bool more = c + NW < n_sub;
        wait_vmcnt<L>();                        // the K tile has landed (V's loads are younger)
        float4 kf[4][2];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int e = 0; e < 2; e++)
                kf[s][e] = *reinterpret_cast<const float4 *>(Ks + lq * RB + (((8 * s + 2 * lg + e) ^ (lq & 7)) * 16));
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(kb, Ks, c + NW, true);
        }
        // S^T[key 4 lg + i][query lq] of each head, smallest terms first
        f32x4 st[GH];
#pragma unroll
        for (int g = 0; g < GH; g++) st[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            bf16x8 kt[3];
            split3(kf[s][0], kf[s][1], kt);
#define QK(A, B) st[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt[A], qf[g][s][B], st[g], 0, 0, 0);
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(2, 0) }
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(0, 2) }
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(1, 1) }
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(1, 0) }
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(0, 1) }
#pragma unroll
            for (int g = 0; g < GH; g++) { QK(0, 0) }
#undef QK
        }
        const bool masked = 16 * c + 16 > all || !full_rows;
        bf16x8 pa[GH][3];                       // A operands of the three MFMAs per column tile
#pragma unroll
        for (int g = 0; g < GH; g++) {
            float sv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) sv[i] = __fmul_rn(st[g][i], a.scale);
            if (masked) {
#pragma unroll
                for (int i = 0; i < 4; i++) sv[i] = 16 * c + 4 * lg + i < hi ? sv[i] : -INFINITY;
            }
            const float tm = xhalf_max(xrow16_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]))));
            const float mn = fmaxf(m[g], tm);
            const float corr = (m[g] == -INFINITY) ? 0.0f : exp_neg(__fsub_rn(m[g], mn));
#pragma unroll
            for (int i = 0; i < 4; i++) sv[i] = sv[i] == -INFINITY ? 0.0f : exp_neg(__fsub_rn(sv[i], mn));
            float ps = __fadd_rn(__fadd_rn(sv[0], sv[1]), __fadd_rn(sv[2], sv[3]));
            ps = xhalf_sum(xrow16_sum(ps));
            l[g] = fmaf(l[g], corr, ps);
            m[g] = mn;
            // rescale the O rows this lane holds (queries 4 lg + j) by their
            // owners' factors, unless no query's maximum moved (factors 1)
            if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0) {
                float cj[4];
#pragma unroll
                for (int j = 0; j < 4; j++) cj[j] = __shfl(corr, 4 * lg + j, 64);
#pragma unroll
                for (int n = 0; n < NT; n++)
#pragma unroll
                    for (int j = 0; j < 4; j++) o[g][n][j] = __fmul_rn(o[g][n][j], cj[j]);
            }
            uint32_t ph[2], pm[2], pl[2];
            split3_4(sv[0], sv[1], sv[2], sv[3], ph, pm, pl, e0, e1);
            pa[g][0] = __builtin_bit_cast(bf16x8, make_uint4(ph[0], ph[1], pl[0], pl[1]));   // with (lo, hi) of V
            pa[g][1] = __builtin_bit_cast(bf16x8, make_uint4(pm[0], pm[1], pm[0], pm[1]));   // with (hi, mid)
            pa[g][2] = __builtin_bit_cast(bf16x8, make_uint4(ph[0], ph[1], ph[0], ph[1]));   // with (hi, mid)
        }
        if (more) wait_vmcnt<L>();              // the V tile has landed (the next K's loads are younger)
        else wait_vmcnt<0>();
        // column lq of tile n is dim 8 lq + n: a lane's 8 dims of a V row are two slots
        float4 vf[4][2];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 2; e++)
                vf[i][e] = *reinterpret_cast<const float4 *>(Vs + (4 * lg + i) * RB + (2 * lq + e) * 16);
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(vb, Vs, c + NW, false);
        }
#pragma unroll
        for (int n = 0; n < NT; n++) {
            uint32_t vh[2], vm[2], vl[2];
            split3_4(vf[0][n >> 2][n & 3], vf[1][n >> 2][n & 3], vf[2][n >> 2][n & 3], vf[3][n >> 2][n & 3], vh, vm, vl,
                     e0, e1);
            const bf16x8 b0 = __builtin_bit_cast(bf16x8, make_uint4(vl[0], vl[1], vh[0], vh[1]));
            const bf16x8 b1 = __builtin_bit_cast(bf16x8, make_uint4(vh[0], vh[1], vm[0], vm[1]));
#pragma unroll
            for (int g = 0; g < GH; g++) o[g][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[g][0], b0, o[g][n], 0, 0, 0);
#pragma unroll
            for (int g = 0; g < GH; g++) o[g][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[g][1], b1, o[g][n], 0, 0, 0);
#pragma unroll
            for (int g = 0; g < GH; g++) o[g][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[g][2], b1, o[g][n], 0, 0, 0);
        }
    }
    // merge the NW key splits: (m, l) per query, O rows through LDS (every
    // wave's loads have landed: its last wait was for all of them)
    float *Om = reinterpret_cast<float *>(smem);           // [NW waves][GH][16 rows][HD]
#pragma unroll
    for (int g = 0; g < GH; g++)
        if (lg == 0) { Mm[wid][g][lq] = m[g]; Ll[wid][g][lq] = l[g]; }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < GH; g++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int n = 0; n < NT; n += 4)
                *reinterpret_cast<f32x4 *>(Om + ((wid * GH + g) * 16 + 4 * lg + j) * HD + lq * NT + n) =
                    f32x4{o[g][n][j], o[g][n + 1][j], o[g][n + 2][j], o[g][n + 3][j]};
    if (t < NW * GH * 16) {
        const int w = t / (GH * 16), g = (t >> 4) % GH, r = t & 15;
        float M = -INFINITY;
#pragma unroll
        for (int k2 = 0; k2 < NW; k2++) M = fmaxf(M, Mm[k2][g][r]);
        Ff[w][g][r] = Mm[w][g][r] == -INFINITY ? 0.0f : exp_neg(__fsub_rn(Mm[w][g][r], M));
    }
    __syncthreads();
    // half a wave per row: each wave sees two whole rows a time
    for (int i = t; i < GH * 16 * HD / 4; i += NW * 64) {
        const int g = i / (16 * HD / 4), r = (i / (HD / 4)) % 16, d = (i % (HD / 4)) * 4;
        const int q = q0 + r;
        float Ls = 0.0f;
        f32x4 O = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float f = Ff[w][g][r];
            const f32x4 x = *reinterpret_cast<const f32x4 *>(Om + ((w * GH + g) * 16 + r) * HD + d);
            Ls = fmaf(Ll[w][g][r], f, Ls);
#pragma unroll
            for (int e = 0; e < 4; e++) O[e] = fmaf(x[e], f, O[e]);
        }
        bool ok = Ls > 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            O[e] = __fdiv_rn(O[e], Ls);
            ok = ok && ((fabsf(O[e]) <= FLT_MAX && fabsf(O[e]) >= 0x1p-96f) || O[e] == 0.0f);
        }
        const uint64_t redo = __builtin_amdgcn_ballot_w64(!ok && q < a.n_q);
        if ((lane < 32 ? (uint32_t)redo : (uint32_t)(redo >> 32)) == 0 && q < a.n_q) {
            float *op = a.out + (int64_t)q * a.o_rs + (h0 + g) * HD + d;
#pragma unroll
            for (int e = 0; e < 4; e++) op[e] = O[e];
        }
        if (__builtin_expect(redo != 0, 0)) {
            const int q2 = __builtin_amdgcn_readfirstlane(q);
#pragma unroll 1
            for (int u = 0; u < 2; u++)
                if ((uint32_t)(redo >> (32 * u)) != 0) attn_row_f32(a, q2 + u, h0 + g, kv_head, lane);
        }
    }
}

template <int GH>
__global__ __launch_bounds__(512) void k_attn_bf3(AttnRowsArgs a) {
    // tiles in reverse, so that the blocks with the most keys start first
    attn_bf3_block<GH>(a, (gridDim.y - 1 - blockIdx.y) * 16);
}

// Both query heads of a KV head in one block (K and V terms formed once for the
// two) where that leaves enough blocks: us with one / two heads per block, 672
// blocks of two (1337 rows) 98.6 / 77, 208 (404 rows) 18.1 / 22.9, 40 (67
// rows after 337) 13.6 / 21.8.
static int attn_heads_per_block(int n_kv_heads, int64_t row_blocks) { return n_kv_heads * row_blocks >= 384 ? 2 : 1; }

// Causal attention of several sequences in one launch (the multi-sequence
// prefill): block row y belongs to sequence j (blk[j] <= y < blk[j + 1]) and
// is that sequence's row block of a call of its own (the same q0, in the
// same reverse order), with the sequence's query / output rows, KV cache,
// key count and query offset.
template <int GH>
__global__ __launch_bounds__(512) void k_attn_bf3_seqs(AttnSeqArgs s) {
    const int y = blockIdx.y;
    int b1 = s.blk[1];
    int64_t row = s.row[0];
    const float *k = s.k[0], *v = s.v[0];
    int nq = s.n_q[0], nk = s.n_k[0], qo = s.q_offset[0];
#pragma unroll
    for (int u = 1; u < QASR_ATTN_MAX_SEQ; u++)
        if (u < s.n && y >= s.blk[u]) {
            b1 = s.blk[u + 1];
            row = s.row[u];
            k = s.k[u];
            v = s.v[u];
            nq = s.n_q[u];
            nk = s.n_k[u];
            qo = s.q_offset[u];
        }
    AttnRowsArgs a = s.base;
    a.q += row * a.q_rs;
    a.out += row * a.o_rs;
    a.k = k;
    a.v = v;
    a.n_q = nq;
    a.n_k = nk;
    a.q_offset = qo;
    attn_bf3_block<GH>(a, (b1 - 1 - y) * 16);
}

hipError_t launch_attn_rows_seqs(const AttnSeqArgs &s0, int n_kv_heads, int head_dim, hipStream_t st) {
    const AttnRowsArgs &a = s0.base;
    if (s0.n < 1 || s0.n > QASR_ATTN_MAX_SEQ || a.window > 0 || head_dim != 128 || a.G != 2)
        return hipErrorInvalidValue;
    AttnSeqArgs s = s0;
    s.blk[0] = 0;
    for (int j = 0; j < s.n; j++) {
        if (s.n_q[j] <= 0) return hipErrorInvalidValue;
        s.blk[j + 1] = s.blk[j] + (s.n_q[j] + 15) / 16;
    }
    // launch_attn_rows' form for these heads (the same bits for either number
    // of heads per block)
    if (attn_heads_per_block(n_kv_heads, s.blk[s.n]) == 2)
        hipLaunchKernelGGL(k_attn_bf3_seqs<2>, dim3(n_kv_heads, s.blk[s.n]), dim3(512), 0, st, s);
    else hipLaunchKernelGGL(k_attn_bf3_seqs<1>, dim3(n_kv_heads * 2, s.blk[s.n]), dim3(512), 0, st, s);
    return hipGetLastError();
}

hipError_t launch_attn_rows(const AttnRowsArgs &a, int n_kv_heads, int head_dim, hipStream_t st) {
    if (a.G <= 0 || 32 % a.G != 0 || a.n_q <= 0) return hipErrorInvalidValue;
    const bool aligned = a.q_rs % 4 == 0 && a.k_rs % 4 == 0 && a.k_hs % 4 == 0 && (uintptr_t)a.q % 16 == 0 &&
                         (uintptr_t)a.k % 16 == 0 && (uintptr_t)a.v % 16 == 0;
    const unsigned row_blocks = (unsigned)((a.n_q + 15) / 16);
    if (aligned && a.k_rs < 1 << 24 && head_dim == 128 && a.G == 2 && a.window == 0) {
        if (attn_heads_per_block(n_kv_heads, row_blocks) == 2)
            hipLaunchKernelGGL(k_attn_bf3<2>, dim3(n_kv_heads, row_blocks), dim3(512), 0, st, a);
        else hipLaunchKernelGGL(k_attn_bf3<1>, dim3(n_kv_heads * 2, row_blocks), dim3(512), 0, st, a);
        return hipGetLastError();
    }
    if (aligned && a.k_rs < 1 << 24 && (head_dim == 128 || head_dim == 64) && a.G == 1 && a.window > 0) {
        // one head per block; the 128-dim heads' 8 waves are 8 key splits, the
        // 64-dim encoder heads' 4
        const dim3 grid(n_kv_heads, row_blocks);
        if (head_dim == 128) hipLaunchKernelGGL((k_attn_mfma<128, 8>), grid, dim3(512), 0, st, a);
        else hipLaunchKernelGGL((k_attn_mfma<64, 4>), grid, dim3(256), 0, st, a);
        return hipGetLastError();
    }
    const dim3 grid(n_kv_heads, (a.n_q + 32 / a.G - 1) / (32 / a.G));
    if (head_dim == 128) hipLaunchKernelGGL(k_attn_rows<128>, grid, dim3(256), 0, st, a);
    else if (head_dim == 64) hipLaunchKernelGGL(k_attn_rows<64>, grid, dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// mel pieces (audio.rs:273-372)
// ---------------------------------------------------------------------------
// frames[t][n] = padded[t * 160 + n] * window[n], reflect padding of 200
__global__ __launch_bounds__(256) void k_mel_frames(float *__restrict__ fr, const float *__restrict__ x, int64_t ns,
                                                    const float *__restrict__ window, int nf) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)nf * 400) return;
    const int n = (int)(i % 400);
    const int64_t t = i / 400;
    const int64_t p = t * 160 + n;          // index into the padded signal
    float v;
    if (p < 200) {
        const int64_t s = 200 - p;
        v = s < ns ? x[s] : 0.0f;
    } else if (p < 200 + ns) {
        v = x[p - 200];
    } else {
        const int64_t s = ns - 2 - (p - 200 - ns);
        v = s >= 0 ? x[s] : 0.0f;
    }
    fr[i] = __fmul_rn(v, window[n]);
}

// powT[t][k] = re^2 + im^2 from re/im [k][t]
__global__ __launch_bounds__(256) void k_mel_power(float *__restrict__ pT, const float *__restrict__ re,
                                                   const float *__restrict__ im, int nf) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)nf * 201) return;
    const int k = (int)(i % 201);
    const int64_t t = i / 201;
    const float r = re[k * (int64_t)nf + t], m = im[k * (int64_t)nf + t];
    pT[i] = __fadd_rn(__fmul_rn(r, r), __fmul_rn(m, m));
}

// log10(max(v, 1e-10)) in place and per-block maxima
__global__ __launch_bounds__(256) void k_mel_log(float *__restrict__ mel, int64_t n, float *__restrict__ bmax) {
    __shared__ float red[4];
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    float v = -1e30f;
    if (i < n) {
        v = log10f(fmaxf(mel[i], 1e-10f));
        mel[i] = v;
    }
    v = wave_max_f32(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) bmax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(256) void k_mel_norm(float *__restrict__ mel, int64_t n, const float *__restrict__ bmax,
                                                  int nb) {
    __shared__ float gm;
    if (threadIdx.x < 64) {
        float v = -1e30f;
        for (int b = threadIdx.x; b < nb; b += 64) v = fmaxf(v, bmax[b]);
        v = wave_max_f32(v);
        if (threadIdx.x == 0) gm = v;
    }
    __syncthreads();
    const float mn = __fsub_rn(gm, 8.0f);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        mel[i] = __fdiv_rn(__fadd_rn(fmaxf(mel[i], mn), 4.0f), 4.0f);
}

hipError_t launch_mel_frames(float *fr, const float *x, int64_t ns, const float *window, int nf, hipStream_t st) {
    const int64_t n = (int64_t)nf * 400;
    hipLaunchKernelGGL(k_mel_frames, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, fr, x, ns, window, nf);
    return hipGetLastError();
}
hipError_t launch_mel_power(float *pT, const float *re, const float *im, int nf, hipStream_t st) {
    const int64_t n = (int64_t)nf * 201;
    hipLaunchKernelGGL(k_mel_power, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, pT, re, im, nf);
    return hipGetLastError();
}
hipError_t launch_mel_log_norm(float *mel, int64_t n, float *bmax, hipStream_t st) {
    const int nb = (int)((n + 255) / 256);
    hipLaunchKernelGGL(k_mel_log, dim3(nb), dim3(256), 0, st, mel, n, bmax);
    hipLaunchKernelGGL(k_mel_norm, dim3(std::min(nb, 1024)), dim3(256), 0, st, mel, n, bmax, nb);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// timing helper: one wave that idles for `ticks` of the 100 MHz constant clock
// (s_memrealtime).  Queued in front of a timed batch of launches, it holds the
// stream until the host has enqueued the whole batch, so the batch runs back to
// back.  The loop always ends: the clock is monotonic.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_delay(int64_t ticks) {
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    while ((int64_t)(__builtin_amdgcn_s_memrealtime() - t0) < ticks) __builtin_amdgcn_s_sleep(64);
}

hipError_t launch_delay(int us, hipStream_t st) {
    if (us < 0 || us > 100000) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_delay, dim3(1), dim3(64), 0, st, (int64_t)us * 100);
    return hipGetLastError();
}

}  // namespace qasr
