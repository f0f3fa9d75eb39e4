// Dense GEMMs of the prefill, the audio encoder and the mel front end.
//
//   C[m, n] (op)= sum_k A[m, k] * B[n, k]          ("NT": both operands K-contiguous)
//
// k_gemm_mfma: CDNA4 MFMA (v_mfma_f32_16x16x32_bf16), 64x64 block tile, four
// waves of 32x32, K-step 32, LDS double buffer.  Operand sources:
//   A f32, split: A = hi + mid + lo with three bf16 terms (each the RNE rounding
//                 of the remaining residual), so A*B is formed from exact bf16
//                 products accumulated in f32 — f32-class accuracy against the
//                 reference's cblas_sgemm on bf16-valued weights (mod.rs:550-628)
//   A bf16        activations already in bf16 (the int8 x bf16 GEMM)
//   B bf16        the reference's weights (exact)
//   B int8        per-row int8 weights, dequantised exactly to bf16 in LDS; the
//                 per-row scale is applied in the epilogue
// It takes every size and alignment; the shapes of the models go to k_gemm_ks
// (f32 A: k_gemm_ks.hip) and k_gemm_lds (int8 B).
// k_gemm_f32: plain f32 FMA tiles for the small GEMMs whose operands are both
// f32 tables (mel DFT and filterbank, audio.rs:339-351).
#include <cstdlib>

#include "kernels.h"
#include "gemm_common.h"

namespace qasr {

typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

template <int ASRC, int BSRC, int EPI>
__global__ __launch_bounds__(256) void k_gemm_mfma(GemmArgs g) {
    constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;
    constexpr int NA = ASRC == A_F32_SPLIT ? 3 : 1;
    __shared__ __attribute__((aligned(16))) uint16_t As[2][NA][BM][LDK];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][BN][LDK];
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wid >> 1, wn = wid & 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int M = g.M, N = g.N, K = g.K;
    // global -> register staging: thread t covers row t/4, k-offset (t%4)*8 of the tile
    const int lr = t >> 2, lk = (t & 3) * 8;
    const int am = m0 + lr, bn = n0 + lr;
    float ar[8];
    u16x8 ab;
    u16x8 br;

    auto load_tile = [&](int k0) {
        const int kk = k0 + lk;
        if (ASRC == A_F32_SPLIT) {
            const float *ap = reinterpret_cast<const float *>(g.A) + (int64_t)am * g.lda + kk;
            if (am < M && kk + 8 <= K && g.a_vec4) {
                const float4 x0 = reinterpret_cast<const float4 *>(ap)[0];
                const float4 x1 = reinterpret_cast<const float4 *>(ap)[1];
                ar[0] = x0.x; ar[1] = x0.y; ar[2] = x0.z; ar[3] = x0.w;
                ar[4] = x1.x; ar[5] = x1.y; ar[6] = x1.z; ar[7] = x1.w;
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float *q = reinterpret_cast<const float *>(g.A) + (int64_t)min(am, M - 1) * g.lda + min(kk + i, K - 1);
                    ar[i] = (am < M && kk + i < K) ? *q : 0.0f;
                }
            }
        } else {
            const uint16_t *ap = reinterpret_cast<const uint16_t *>(g.A) + (int64_t)am * g.lda + kk;
            if (am < M && kk + 8 <= K && g.a_vec4) {
                ab = *reinterpret_cast<const u16x8 *>(ap);
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint16_t *q = reinterpret_cast<const uint16_t *>(g.A) + (int64_t)min(am, M - 1) * g.lda + min(kk + i, K - 1);
                    ab[i] = (am < M && kk + i < K) ? *q : (uint16_t)0;
                }
            }
        }
        if (BSRC == B_BF16) {
            const uint16_t *bp = reinterpret_cast<const uint16_t *>(g.B) + (int64_t)bn * g.ldb + kk;
            if (bn < N && kk + 8 <= K && g.b_vec) {
                br = *reinterpret_cast<const u16x8 *>(bp);
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint16_t *q = reinterpret_cast<const uint16_t *>(g.B) + (int64_t)min(bn, N - 1) * g.ldb + min(kk + i, K - 1);
                    br[i] = (bn < N && kk + i < K) ? *q : (uint16_t)0;
                }
            }
        } else {
            const int8_t *bp = reinterpret_cast<const int8_t *>(g.B) + (int64_t)bn * g.ldb + kk;
            int8_t q[8];
            if (bn < N && kk + 8 <= K && g.b_vec) {
                const uint2 v = *reinterpret_cast<const uint2 *>(bp);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    q[i] = (int8_t)(v.x >> (8 * i));
                    q[4 + i] = (int8_t)(v.y >> (8 * i));
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int8_t *qp = reinterpret_cast<const int8_t *>(g.B) + (int64_t)min(bn, N - 1) * g.ldb + min(kk + i, K - 1);
                    q[i] = (bn < N && kk + i < K) ? *qp : (int8_t)0;
                }
            }
#pragma unroll
            for (int i = 0; i < 8; i++) br[i] = f32_to_bf16_rne((float)q[i]);   // exact, |q| <= 128
        }
    };
    auto store_tile = [&](int buf) {
        if (ASRC == A_F32_SPLIT) {
            u16x8 hi, mi, lo;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float x = ar[i];
                const uint16_t h = f32_to_bf16_rne(x);
                const float r1 = __fsub_rn(x, __uint_as_float((uint32_t)h << 16));
                const uint16_t m = f32_to_bf16_rne(r1);
                const float r2 = __fsub_rn(r1, __uint_as_float((uint32_t)m << 16));
                hi[i] = h; mi[i] = m; lo[i] = f32_to_bf16_rne(r2);
            }
            *reinterpret_cast<u16x8 *>(&As[buf][0][lr][lk]) = hi;
            *reinterpret_cast<u16x8 *>(&As[buf][1][lr][lk]) = mi;
            *reinterpret_cast<u16x8 *>(&As[buf][2 % NA][lr][lk]) = lo;
        } else {
            *reinterpret_cast<u16x8 *>(&As[buf][0][lr][lk]) = ab;
        }
        *reinterpret_cast<u16x8 *>(&Bs[buf][lr][lk]) = br;
    };

    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int nk = (K + BK - 1) / BK;
    load_tile(0);
    store_tile(0);
    __syncthreads();
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    for (int kt = 0; kt < nk; kt++) {
        const int buf = kt & 1;
        if (kt + 1 < nk) load_tile((kt + 1) * BK);
        bf16x8 bfrag[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
            bfrag[j] = *reinterpret_cast<const bf16x8 *>(&Bs[buf][wn * 32 + j * 16 + fr][fk]);
#pragma unroll
        for (int s = NA - 1; s >= 0; s--) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const bf16x8 afrag = *reinterpret_cast<const bf16x8 *>(&As[buf][s][wm * 32 + i * 16 + fr][fk]);
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afrag, bfrag[j], acc[i][j], 0, 0, 0);
            }
        }
        if (kt + 1 < nk) store_tile(buf ^ 1);
        __syncthreads();
    }

    // epilogue: lane holds rows 4*(lane/16)+r, column lane%16 of each 16x16 tile
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm * 32 + i * 16 + (lane >> 4) * 4 + r;
                const int n = n0 + wn * 32 + j * 16 + (lane & 15);
                if (m >= M || n >= N) continue;
                float v = acc[i][j][r];
                // EPI_TRANS: rows are (chunk, spatial) of a batched conv and the
                // output keeps the reference layout [chunk][channel][spatial];
                // EPI_CHW: the same GELU index, row-major (channels-last) output
                int64_t off, gidx;
                if (EPI & EPI_TRANS) {
                    const int c = m / g.gelu_rows, sp = m % g.gelu_rows;
                    gidx = (int64_t)n * g.gelu_rows + sp;
                    off = (int64_t)c * g.gelu_n + gidx;
                } else if (EPI & EPI_CHW) {
                    gidx = (int64_t)n * g.gelu_rows + m % g.gelu_rows;
                    off = (int64_t)m * g.ldc + n;
                } else {
                    gidx = (int64_t)m * g.ldc + n;
                    off = gidx;
                }
                float *cp = g.C + off;
                if (EPI & EPI_SCALE) v = __fmul_rn(v, g.scale[n]);
                if (EPI & EPI_ACCUM) {
                    float c = *cp;
                    if (g.bias) c = __fadd_rn(c, g.bias[n]);
                    v = __fadd_rn(c, v);
                } else if (g.bias) {
                    v = __fadd_rn(v, g.bias[n]);
                }
                if (EPI & EPI_GELU) v = gelu_ref(v, gidx, g.gelu_n);
                *cp = v;
            }
}

// ---------------------------------------------------------------------------
// k_gemm_lds: bf16 A x int8 B (config-1 prefill GEMMs), fed by direct global ->
// LDS loads (global_load_lds_dwordx4) through a ring of NS stages, so NS - 1
// K-steps of 64 are in flight while one is computed.  A stage holds the
// block's A tile (BM rows x 128 bytes) and B tile (BN rows x 64 bytes).  A load
// writes lane l's 16 bytes at LDS offset 16 l, so the lane -> (row, 16-byte
// slot) map is chosen with an XOR swizzle of the slot by the row, which
// spreads a fragment read's 16 rows over the banks.  int8 B is widened to bf16
// (exact) as the fragment is read.  K-steps past the end load a zero page, so
// the wait count is the same in every iteration.  Requires K % 64 == 0 and
// 16-byte aligned rows.
//
// VEC (N a multiple of 4, 16-byte aligned C rows): the columns are the MFMA's
// rows, so a lane ends with 4 consecutive columns and stores 16 bytes; else a
// column per lane (16 consecutive floats per store).  The same bits; the
// dispatch below says where which is faster.
//
// KP > 1 splits the K loop inside the block: 4 KP waves in KP groups of 4,
// group p taking the K-steps p, p + KP, ... through a ring of its own; at the
// end groups 1 .. KP - 1 leave their partial tiles in LDS and group 0 adds
// them in group order and runs the epilogue.  At the M ~ 400 shapes of config
// 1 a 64 x 64 tile's K loop is a chain of K-steps that one wave per SIMD walks
// alone (the grid holds 96-384 tiles for 256 CUs); KP groups shorten the chain
// KP times and give each SIMD KP waves to overlap.
// ---------------------------------------------------------------------------
__device__ __attribute__((aligned(256))) int4 g_gemm_zero16[16];

// LDS placement of the ring's 16-byte slots: slot q of tile row r sits at
// slot q ^ a_swz(r) (A rows: 128 B, 8 slots) or q ^ b_swz(r) (B rows: 64 B, 4
// slots): the conflict-free forms (config-1 LM head at M = 375 184 -> 178 us
// against r & 7 and r & 3, the seven 64 x 64 shapes within 2%)
__device__ __forceinline__ int a_swz(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int b_swz(int r) { return (r & 3) ^ ((r >> 2) & 3); }

template <int NS, int BM, int BN, int KP, bool VEC>
__global__ __launch_bounds__(256 * KP, BM * BN > 64 * 64 ? 2 : 1) void k_gemm_lds(GemmArgs g) {
    constexpr int BK = 64;
    constexpr int ASZ = BM * 128, BSZ = BN * 64, STG = ASZ + BSZ;
    constexpr int LA = BM / 32, LB = BN / 64;                        // one-KiB loads per wave per stage
    // wave tiling: int8 B, which needs converting, is owned by one wave per
    // fragment (BN/4-column strips), so no fragment is converted twice.
    // (Measured and rejected for the LM head at M = 375, in loops: 2 x 2 waves of
    // (BM/2) x (BN/2), which halve the A reads from LDS but widen every B
    // fragment in two waves: 143 -> 160 us with 128 x 128 tiles, 157-167 with
    // 192 x 128 and 128 x 256; 8 waves on 128 x 256 tiles 156-162.)
    constexpr int WR = BM / 16, WC = BN / 4 / 16;
    static_assert(BM % 32 == 0 && BN % 64 == 0, "tile");
    static_assert((KP - 1) * 4 * WR * WC * 4 * 64 * 4 <= KP * NS * STG, "partials fit the rings");
    __shared__ __attribute__((aligned(16))) char smem_all[KP][NS][STG];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int grp = wave >> 2, wid = wave & 3;          // K group, wave within the group
    auto &smem = smem_all[grp];
    const int nw = (BN / 4) * wid;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int M = g.M, N = g.N, K = g.K;
    const int nk = K / BK;
    // KP groups: this group's i-th K-step is grp + KP i; nit iterations each
    const int nit = (nk + KP - 1) / KP;
    // this lane's rows and swizzled 16-byte slots in the wave's loads: A load j
    // covers tile rows 8 j .. 8 j + 7 (8 slots each), B load j rows 16 j .. 16 j + 15 (4 slots)
    const char *A = reinterpret_cast<const char *>(g.A), *B = reinterpret_cast<const char *>(g.B);
    const char *a_src[LA], *b_src[LB];
#pragma unroll
    for (int u = 0; u < LA; u++) {
        const int r = 8 * (wid * LA + u) + (lane >> 3), p = (lane & 7) ^ a_swz(r);
        a_src[u] = A + ((int64_t)min(m0 + r, M - 1) * g.lda) * 2 + 16 * p;
    }
#pragma unroll
    for (int u = 0; u < LB; u++) {
        const int r = 16 * (wid * LB + u) + (lane >> 2), p = (lane & 3) ^ b_swz(r);
        b_src[u] = B + (int64_t)min(n0 + r, N - 1) * g.ldb + 16 * p;
    }
    const char *zero = reinterpret_cast<const char *>(g_gemm_zero16);
    auto issue = [&](int buf, int kt) {
        char *st = smem[buf];
        const int kg = grp + KP * kt;       // the group's kt-th K-step
        const bool live = kt < nit && kg < nk;
        const int64_t ka = live ? (int64_t)kg * BK * 2 : 0, kb = live ? (int64_t)kg * BK : 0;
#pragma unroll
        for (int u = 0; u < LA; u++) lds_dma16(live ? a_src[u] + ka : zero, st + 1024 * (wid * LA + u));
#pragma unroll
        for (int u = 0; u < LB; u++) lds_dma16(live ? b_src[u] + kb : zero, st + ASZ + 1024 * (wid * LB + u));
    };

    f32x4 acc[WR][WC];
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // The column scales do not depend on the products: loaded before the
    // ring's first stage, so that no load is left after the K loop.  Being
    // older than every ring load, they are complete by the first wait.  (By every
    // group, though group 0 alone uses them: under a test of the group the
    // pointer's argument load falls behind the others, a round trip more before
    // the first stage: 33 x 10001 x 1024 in 64 x 64 tiles 7.7 -> 7.3 us.)
    const int fr = lane & 15, fg = lane >> 4;
    f32x4 pre_s[WC];
    const bool sv = ((uintptr_t)g.scale & 15) == 0;
#pragma unroll
    for (int j = 0; j < WC; j++) {
        if constexpr (VEC) {
            pre_s[j] = gemm_load4(g.scale, min(n0 + nw + j * 16 + 4 * fg, N - 1), N, sv);
        } else {
            const float x = g.scale[min(n0 + nw + j * 16 + fr, N - 1)];
            pre_s[j] = f32x4{x, x, x, x};
        }
    }

#pragma unroll
    for (int s = 0; s < NS - 1; s++) issue(s, s);
    for (int kt = 0; kt < nit; kt++) {
        wait_vmcnt<(LA + LB) * (NS - 2)>();   // this wave's loads of stage kt have landed
        __syncthreads();                      // ... and every wave's; stage kt - 1 is free
        issue((kt + NS - 1) % NS, kt + NS - 1);
        const char *st = smem[kt % NS];
        if (BN == 128) __builtin_amdgcn_iglp_opt(1);   // LDS reads spread between the MFMAs
#pragma unroll
        for (int s = 0; s < BK / 32; s++) {
            bf16x8 bfrag[WC];
#pragma unroll
            for (int j = 0; j < WC; j++) {
                const int n = nw + j * 16 + fr;
                // 8 int8 weights -> bf16 (exact: |q| <= 128 has 8 significant bits)
                const int p = (2 * s + (fg >> 1)) ^ b_swz(n);
                const uint2 v = *reinterpret_cast<const uint2 *>(st + ASZ + n * 64 + p * 16 + (fg & 1) * 8);
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const uint32_t x = e ? v.y : v.x;
                    w[2 * e] = cvt_pk_bf16((float)(int8_t)(x & 0xFF), (float)(int8_t)((x >> 8) & 0xFF));
                    w[2 * e + 1] = cvt_pk_bf16((float)(int8_t)((x >> 16) & 0xFF), (float)(int8_t)(x >> 24));
                }
                bfrag[j] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
            }
#pragma unroll
            for (int i = 0; i < WR; i++) {
                const int r = i * 16 + fr;
                const bf16x8 af = *reinterpret_cast<const bf16x8 *>(st + r * 128 + ((4 * s + fg) ^ a_swz(r)) * 16);
#pragma unroll
                for (int j = 0; j < WC; j++)
                    acc[i][j] = VEC ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfrag[j], af, acc[i][j], 0, 0, 0)
                                    : __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfrag[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    wait_vmcnt<0>();                          // no load may land in LDS after the block ends
    if constexpr (KP > 1) {
        // groups 1 .. KP - 1 hand their partial tiles to group 0 through the
        // rings' LDS (every wave is past its last ring read at the barrier)
        constexpr int EW = WR * WC * 4;      // accumulator values per lane
        float *red = reinterpret_cast<float *>(&smem_all[0][0][0]);
        __syncthreads();
        if (grp > 0) {
            float *dst = red + ((grp - 1) * 4 + wid) * EW * 64 + lane;
#pragma unroll
            for (int i = 0; i < WR; i++)
#pragma unroll
                for (int j = 0; j < WC; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) dst[((i * WC + j) * 4 + r) * 64] = acc[i][j][r];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int p = 1; p < KP; p++) {
            const float *src = red + ((p - 1) * 4 + wid) * EW * 64 + lane;
#pragma unroll
            for (int i = 0; i < WR; i++)
#pragma unroll
                for (int j = 0; j < WC; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[i][j][r] = __fadd_rn(acc[i][j][r], src[((i * WC + j) * 4 + r) * 64]);
        }
    }

    // epilogue: a lane holds 4 consecutive columns of one row of each 16 x 16
    // tile (VEC), else 4 consecutive rows of one column; every value first,
    // then only stores under the bounds tests: an operand use inside a store's
    // branch would make the compiler wait for all vector memory there, the
    // previous stores included
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = __fmul_rn(acc[i][j][r], pre_s[j][r]);
                asm volatile("" : "+v"(v));
                acc[i][j][r] = v;
            }
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) {
            if constexpr (VEC) {                 // N % 4 == 0: whole runs
                const int m = m0 + i * 16 + fr, n = n0 + nw + j * 16 + 4 * fg;
                if (m < M && n < N) *reinterpret_cast<f32x4 *>(g.C + (int64_t)m * g.ldc + n) = acc[i][j];
            } else {
                const int n = n0 + nw + j * 16 + fr;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + i * 16 + fg * 4 + r;
                    if (m < M && n < N) g.C[(int64_t)m * g.ldc + n] = acc[i][j][r];
                }
            }
        }
}

// ---------------------------------------------------------------------------
// f32 SIMT GEMM (NT), 64x64 tile, 4x4 outputs per thread, K-step 16
// ---------------------------------------------------------------------------
// T x T output tile per block of 16 x 16 threads, (T / 16)^2 outputs per
// thread; each output's sum runs over k in order in one thread (fmaf), so the
// tile size does not change a bit
template <int T>
__global__ __launch_bounds__(256) void k_gemm_f32(GemmArgs g) {
    constexpr int R = T / 16;
    __shared__ float As[16][T + 1], Bs[16][T + 1];
    const int t = threadIdx.x, tx = t & 15, ty = t >> 4;
    const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    const float *A = reinterpret_cast<const float *>(g.A), *B = reinterpret_cast<const float *>(g.B);
    float acc[R][R] = {};
    for (int k0 = 0; k0 < g.K; k0 += 16) {
        for (int i = t; i < T * 16; i += 256) {
            const int r = i >> 4, k = i & 15;
            const int m = m0 + r, n = n0 + r, kk = k0 + k;
            const float av = A[(int64_t)min(m, g.M - 1) * g.lda + min(kk, g.K - 1)];
            const float bv = B[(int64_t)min(n, g.N - 1) * g.ldb + min(kk, g.K - 1)];
            As[k][r] = (m < g.M && kk < g.K) ? av : 0.0f;
            Bs[k][r] = (n < g.N && kk < g.K) ? bv : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; k++) {
            float a[R], b[R];
#pragma unroll
            for (int i = 0; i < R; i++) { a[i] = As[k][ty * R + i]; b[i] = Bs[k][tx * R + i]; }
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int j = 0; j < R; j++) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int m = m0 + ty * R + i, n = n0 + tx * R + j;
            if (m < g.M && n < g.N) g.C[(int64_t)m * g.ldc + n] = acc[i][j];
        }
}

template <int ASRC, int BSRC>
static hipError_t go_gemm(const GemmArgs &g, int epi, hipStream_t st) {
    const dim3 grid((g.N + 63) / 64, (g.M + 63) / 64);
    switch (epi) {
#define QE(E) case E: hipLaunchKernelGGL((k_gemm_mfma<ASRC, BSRC, E>), grid, dim3(256), 0, st, g); break;
        QE(EPI_NONE) QE(EPI_ACCUM) QE(EPI_SCALE) QE(EPI_GELU) QE(EPI_TRANS) QE(EPI_TRANS | EPI_GELU)
        QE(EPI_GELU | EPI_CHW)
#undef QE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// bf16 A x int8 B.  K groups: 64 x 64 tiles in at most 32 columns, with at
// least 16 K-steps of 64, run 4 groups per block of 3 stages each (config 1 at M
// = 375, us per launch, KP 1 -> 4: k / v 7.7 -> 6.6, q 8.5 -> 7.5, o 12.4 -> 9.2,
// down 17.1 -> 11.9; gate / up, 48 tile columns: 10.2 -> 12.2).
//
// Otherwise the tile is free (an element's sum runs over the same K-steps in
// the same order in every form) and the call takes the form with the least
// estimated time: `one` for a CU's first tile, `more` for each further round
// of tiles over the 256 CUs, halfway between the whole and the fractional
// count of rounds (several blocks share a CU).  The figures are fits, in 0.1 us
// at K = 1024, to a sweep over M = 16 ... 404 and N = 4096 ... 151936; one (64 x
// 128) is raised for K = 2048 and 3072, where two 64 x 64 tiles are faster.  K <
// 512, where a tile's fixed part weighs more, has figures of its own (256 x 20000
// x 192 11.2 -> 9.2 us).  Rows fitted to more shapes gained 0.5% on those and lost
// 0.3% (up to 15%) on 172 others; they were not taken.  us per launch with 64 x 64 tiles below 2048 of them and 128 x 128 beyond, then by
// this rule: M = 16, N = 60001 17.2 -> 14.0, N = 151936 42.2 -> 27.0; M = 64, N
// = 151936 46.6 -> 37.0; M = 90, N = 60001 36.6 -> 27.6; M = 140, N = 151936
// 88.6 -> 65.4; M = 375, N = 20000 32.2 -> 24.0; M = 404, N = 151936 182 -> 170.
// The 128-column forms keep a ring of 2 stages, so that more blocks share a CU
// (LM head at M = 375, 128 x 128, 3 stages -> 2: 174 -> 155 us).  Measured and
// rejected there: the M tiles of one column strip grouped on one XCD (162 us,
// against 155); each block walking every M tile of its strip (205); non-temporal
// stores of C (143 -> 147); the activations split into three int8 planes on the
// int8 MFMA (273-282: three bytes per activation through the ring).
//
// 16-byte stores (VEC), on buffers that are not in the cache: 64 x 64 tiles always
// (375 x 4096 x 1024 10.5 -> 10.25 us), 32 x 64 in more than one round of tiles
// (90 x 6144 7.7 -> 7.5; in one round 5.8 -> 6.0), 128 columns in one round (375 x
// 10000 16.3 -> 15.6; in more, where a tile's stores run beside the next tile's
// K loop, the longer runs of single rows are better: LM head at M = 375 159 ->
// 152, 190 x 60000 39.9 -> 37.8).
struct W8Form { int bm, bn, one, more; };

template <int NS, int BM, int BN, int KP>
static void go_w8(const GemmArgs &g, bool vec, hipStream_t st) {
    const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM);
    if (vec) hipLaunchKernelGGL((k_gemm_lds<NS, BM, BN, KP, true>), grid, dim3(256 * KP), 0, st, g);
    else hipLaunchKernelGGL((k_gemm_lds<NS, BM, BN, KP, false>), grid, dim3(256 * KP), 0, st, g);
}

static hipError_t go_gemm_lds(const GemmArgs &g, hipStream_t st) {
    const bool vec = g.N % 4 == 0 && g.ldc % 4 == 0 && (uintptr_t)g.C % 16 == 0;
    const int64_t small_blocks = (int64_t)((g.N + 63) / 64) * ((g.M + 63) / 64);
    if (small_blocks < 2048 && g.K / 64 >= 16 && (g.N + 63) / 64 <= 32) {
        go_w8<3, 64, 64, 4>(g, vec, st);
        return hipGetLastError();
    }
    static const W8Form longk[] = {{32, 64, 64, 26}, {64, 64, 80, 37}, {64, 128, 125, 68},
                                   {96, 128, 118, 80}, {128, 128, 132, 96}, {160, 128, 147, 119}};
    static const W8Form shortk[] = {{32, 64, 66, 27}, {64, 64, 94, 30}, {64, 128, 123, 59},
                                    {96, 128, 143, 71}, {128, 128, 169, 88}, {160, 128, 176, 172}};
    const W8Form *f = g.K < 512 ? shortk : longk;
    int best = 5;
    int64_t best_cost = INT64_MAX;
    for (int i = 0; i < 6; i++) {
        const int64_t rows = (g.M + f[i].bm - 1) / f[i].bm, tiles = rows * ((g.N + f[i].bn - 1) / f[i].bn);
        if (rows > 65535) continue;                  // the grid's y limit
        const int64_t rounds = (tiles + 255) / 256;
        const int64_t c = 512 * (int64_t)f[i].one + (rounds > 1 ? f[i].more * (tiles + 256 * rounds - 512) : 0);
        if (c < best_cost) { best_cost = c; best = i; }
    }
    const int64_t tiles = (int64_t)((g.M + f[best].bm - 1) / f[best].bm) * ((g.N + f[best].bn - 1) / f[best].bn);
    const bool one_round = tiles <= 256;
    switch (best) {
        case 0: go_w8<4, 32, 64, 1>(g, vec && !one_round, st); break;
        case 1: go_w8<4, 64, 64, 1>(g, vec, st); break;
        case 2: go_w8<2, 64, 128, 1>(g, vec && one_round, st); break;
        case 3: go_w8<2, 96, 128, 1>(g, vec && one_round, st); break;
        case 4: go_w8<2, 128, 128, 1>(g, vec && one_round, st); break;
        default: go_w8<2, 160, 128, 1>(g, vec && one_round, st); break;
    }
    return hipGetLastError();
}

hipError_t launch_gemm(const GemmArgs &g0, int asrc, int bsrc, int epi, hipStream_t st) {
    GemmArgs g = g0;
    if (g.M <= 0 || g.N <= 0 || g.K <= 0) return hipErrorInvalidValue;
    g.a_vec4 = (g.lda % 8 == 0) && ((uintptr_t)g.A % 16 == 0);
    g.b_vec = (g.ldb % 8 == 0) && ((uintptr_t)g.B % 16 == 0);
    if ((epi & (EPI_TRANS | EPI_CHW)) && g.gelu_rows <= 0) return hipErrorInvalidValue;
    if (asrc == A_CONV) {
        // implicit im2col: whole 32-channel runs, every K-step inside one tap
        const bool ok = bsrc == B_BF16_FRAG && g.conv_c > 0 && g.conv_c % 32 == 0 && g.conv_kh > 0 && g.conv_kw > 0 &&
                        g.K == g.conv_c * g.conv_kh * g.conv_kw && g.conv_hout > 0 && g.conv_wout > 0 &&
                        g.conv_hin > 0 && g.conv_win > 0 && g.M % (g.conv_hout * g.conv_wout) == 0;
        if (!ok || g.K >= (1 << 22)) return hipErrorInvalidValue;
        g.conv_rc = 1.0f / (float)g.conv_c;
        g.conv_rkw = 1.0f / (float)g.conv_kw;
        return launch_gemm_ks(g, asrc, bsrc, epi, st);
    }
    if (bsrc == B_BF16_FRAG) return launch_gemm_ks(g, asrc, bsrc, epi, st);
    if (asrc == A_F32_SPLIT && bsrc == B_BF16)
        return gemm_ks_ok(g, asrc, bsrc, epi) ? launch_gemm_ks(g, asrc, bsrc, epi, st)
                                              : go_gemm<A_F32_SPLIT, B_BF16>(g, epi, st);
    if (asrc == A_BF16 && bsrc == B_I8) {
        // the LDS ring takes whole stages and 16-byte aligned rows
        const bool ring = epi == EPI_SCALE && !g.bias && g.K % 64 == 0 && (g.lda * 2) % 16 == 0 && g.ldb % 16 == 0 &&
                          (uintptr_t)g.A % 16 == 0 && (uintptr_t)g.B % 16 == 0;
        if (!ring) return go_gemm<A_BF16, B_I8>(g, epi, st);
        return go_gemm_lds(g, st);
    }
    if (asrc == A_BF16 && bsrc == B_BF16) return go_gemm<A_BF16, B_BF16>(g, epi, st);
    return hipErrorInvalidValue;
}

hipError_t launch_gemm_f32(const GemmArgs &g, hipStream_t st) {
    if (g.M <= 0 || g.N <= 0 || g.K <= 0) return hipErrorInvalidValue;
    // 32 x 32 tiles while 64 x 64 ones would leave CUs idle (the mel DFT and
    // filterbank: 94-188 blocks of 64 x 64)
    const int64_t tiles64 = (int64_t)((g.N + 63) / 64) * ((g.M + 63) / 64);
    if (tiles64 < 512) {
        hipLaunchKernelGGL(k_gemm_f32<32>, dim3((g.N + 31) / 32, (g.M + 31) / 32), dim3(256), 0, st, g);
    } else {
        hipLaunchKernelGGL(k_gemm_f32<64>, dim3((g.N + 63) / 64, (g.M + 63) / 64), dim3(256), 0, st, g);
    }
    return hipGetLastError();
}

}  // namespace qasr
