// f32-class GEMM of the prefill, the audio encoder and its convolutions
//
//   C[m, n] (op)= sum_k A[m, k] * B[n, k]
//
// A f32: rows, or (CONV) the im2col rows of a channels-last convolution read in
// place, each K-step one kernel tap's run of 32 channels (zero past the
// borders).  B bf16: fragment-major weights (BP, laid out once at load by
// launch_pack_frag) or plain rows.  A is split into three bf16 terms in
// registers and multiplied by v_mfma_f32_16x16x32_bf16: exact products, f32
// accumulation.
//
// Split of the work: each of the block's S waves owns the K-steps w, w + S, ...
// of the whole TM x TN tile and walks them alone: A through a stage of LDS of
// its own (global_load_lds, refilled as soon as its fragments are in
// registers), fragment-major B straight into registers (1 KiB contiguous
// loads), no barrier until the S partial tiles are summed in slice order.
// What bounds it, by count: per 64 x 64 x 32 step the matrix cores need 192 clk
// of a CU, the vector memory path 192 (12 KiB at 64 B per clk), and data that
// passes through LDS 1 clk per 64 B written and per 128 B read; B rows through
// LDS (plain weights) add half to that, which is why the weights are laid out
// fragment-major.  By the counters: the convolutions of 30 s the vector
// instructions (60% of the issue slots: split and row addresses; MFMA units
// 44% busy, waits for memory 17% of the waves' time); 404 rows no resource (MFMA
// 12-25%, waits for memory 20-40%: one K chain per wave, one or two blocks per
// CU); 67 rows the launch, the first load and the reduction.  Before, four
// waves shared each K-step of a 64 x 64 tile (24 KiB read from LDS per step, a
// block barrier per step).  us per launch, cold weights, before -> now
// (fragment-major):
//   M = 404: 4096 x 1024  19.3 -> 13.7,  1024 x 2048  16 -> 8.5,
//            6144 x 1024  28.7 -> 18.4,  1024 x 3072  24 -> 11.9
//   M = 67:  4096 x 1024  15.1 -> 6.3,   1024 x 2048  17 -> 5.0,
//            6144 x 1024  17.1 -> 8.0,   1024 x 3072  23 -> 6.1
//   conv2 of 30 s (24000 x 480 x 4320) 379 -> 307, conv3 175 -> 88,
//   the stem's projection (390 x 896 x 7680) 63 -> 32
// Measured and rejected: the waves side by side over the columns with the A
// rows in LDS once (a barrier per K-step: 19.0 and 26.2 us for the first and
// third M = 404 shapes); 64 x 128 tiles (over 256 registers: one wave per
// SIMD, 19.2 and 25.9); fragments of plain rows loaded straight into registers
// (16 rows x 16 bytes per quarter wave: 38 B per ns and CU against 140).
#include <algorithm>

#include "kernels.h"
#include "gemm_common.h"

namespace qasr {

__device__ __attribute__((aligned(256))) int4 g_ks_zero[16];    // A_CONV's rows past the borders

// the fewest row groups (a divisor of the wr fragments) whose partials, at
// row_bytes per tile row, fit the ring; one fragment each if none does
constexpr int ks_phases(int wr, int row_bytes, int ring) {
    for (int p = 1; p < wr; p++)
        if (wr % p == 0 && wr / p * 16 * row_bytes <= ring) return p;
    return wr;
}

template <bool CONV, bool BP, int EPI, int TM, int TN, int S, int KU>
__global__ __launch_bounds__(64 * S, 2) void k_gemm_ks(GemmArgs g) {
    constexpr int WR = TM / 16, WC = TN / 16;
    constexpr int ASZ = TM * 128, BSZ = BP ? 0 : TN * 64, STG = ASZ + BSZ;   // one K-step: f32 A rows, bf16 B rows
    constexpr int LA = TM / 8, LB = BP ? 0 : TN / 16;                        // its one-KiB loads
    constexpr int LD = TN + 4;                                       // partial rows in LDS
    constexpr int RING = S * KU * STG;
    constexpr int PH = ks_phases(WR, S * LD * 4, RING);              // the tile is reduced PH row groups at a time
    constexpr int PR = TM / PH;
    constexpr int SM = RING > S * PR * LD * 4 ? RING : S * PR * LD * 4;
    static_assert(TM % 16 == 0 && TN % 16 == 0 && WR % PH == 0, "tile");
    __shared__ __attribute__((aligned(16))) char smem[SM];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int M = g.M, N = g.N;
    // tile of this block: XCD x (blocks x, x + 8, ...) takes a contiguous run of
    // tiles, ordered so that neighbours share the larger operand's strip
    int m0, n0;
    {
        const int gx = (N + TN - 1) / TN, gy = (M + TM - 1) / TM, total = gx * gy;
        const int x = blockIdx.x & 7, k = blockIdx.x >> 3, q = total >> 3, rem = total & 7;
        const int tile = x * q + min(x, rem) + k;
        if (g.m_major) { m0 = tile / gx; n0 = tile - m0 * gx; }
        else { n0 = tile / gy; m0 = tile - n0 * gy; }
        m0 *= TM;
        n0 *= TN;
    }
    char *ring = smem + wave * (KU * STG);
    const int nk = g.K / 32;
    // this lane's source of every load: A load u covers tile rows 8 u .. 8 u + 7
    // (8 slots of 16 bytes each), B load u rows 16 u .. 16 u + 15 (4 slots)
    const char *A = reinterpret_cast<const char *>(g.A) + (CONV ? 0 : (int64_t)m0 * g.lda * 4);
    const char *B = reinterpret_cast<const char *>(g.B) + (BP ? 0 : (int64_t)n0 * g.ldb * 2);
    uint32_t a_off[CONV ? 1 : LA], b_off[BP ? 1 : LB];
    const char *a_src[CONV ? LA : 1];
    int a_iy[CONV ? LA : 1], a_ix[CONV ? LA : 1];
#pragma unroll
    for (int u = 0; u < LA; u++) {
        const int r = 8 * u + (lane >> 3), p = (lane & 7) ^ (r & 7);
        const int m = min(r, M - 1 - m0);
        if constexpr (CONV) {
            const int plane = g.conv_hout * g.conv_wout, mm = m0 + m, ch = mm / plane, rem = mm - ch * plane;
            const int oy = rem / g.conv_wout, ox = rem - oy * g.conv_wout;
            a_iy[u] = oy * g.conv_sy - g.conv_py;
            a_ix[u] = ox * g.conv_sx - g.conv_px;
            a_src[u] = A + (int64_t)ch * g.conv_hin * g.conv_win * g.conv_c * 4 + 16 * p;
        } else {
            a_off[u] = (uint32_t)m * (uint32_t)g.lda * 4u + 16 * p;
        }
    }
    // packed B: fragment (column group c, K-step s) is the KiB at (c nk + s), lane l's 16 bytes at 16 l
    int64_t b_frag[BP ? WC : 1];
    if constexpr (BP) {
        const int last = (N + 15) / 16 - 1;
#pragma unroll
        for (int j = 0; j < WC; j++) b_frag[j] = (int64_t)min(n0 / 16 + j, last) * nk * 1024;
    } else {
#pragma unroll
        for (int u = 0; u < LB; u++) {
            const int r = 16 * u + (lane >> 2), p = (lane & 3) ^ ((r >> 1) & 3);
            b_off[u] = (uint32_t)min(r, N - 1 - n0) * (uint32_t)g.ldb * 2u + 16 * p;
        }
    }
    const int nst = wave < nk ? (nk - wave + S - 1) / S : 0;         // this wave's K-steps: wave, wave + S, ...
    bf16x8 xn[BP ? KU : 1][BP ? WC : 1];                             // packed B of the stage in flight
    // K-steps st .. st + KU - 1 of this wave into the stage
    auto issue = [&](int st0) {
#pragma unroll
        for (int ku = 0; ku < KU; ku++) {
            if (KU > 1 && st0 + ku >= nst) break;
            char *st = ring + ku * STG;
            const int kg = wave + S * (st0 + ku);
            if constexpr (CONV) {
                const int k0 = kg * 32;
                const int tp = (int)(((float)k0 + 16.0f) * g.conv_rc), c0 = k0 - tp * g.conv_c;
                const int ky = (int)(((float)tp + 0.5f) * g.conv_rkw), kx = tp - ky * g.conv_kw;
#pragma unroll
                for (int u = 0; u < LA; u++) {
                    const int iy = a_iy[u] + ky, ix = a_ix[u] + kx;
                    const bool in = iy >= 0 && iy < g.conv_hin && ix >= 0 && ix < g.conv_win;
                    const int64_t off = ((int64_t)iy * g.conv_win + ix) * g.conv_c + c0;
                    lds_dma16(in ? a_src[u] + off * 4 : reinterpret_cast<const char *>(g_ks_zero), st + 1024 * u);
                }
            } else {
                const char *ak = A + (int64_t)kg * 128;
#pragma unroll
                for (int u = 0; u < LA; u++) lds_dma16_s(ak, a_off[u], st + 1024 * u);
            }
            if constexpr (BP) {
#pragma unroll
                for (int j = 0; j < WC; j++)
                    xn[ku][j] = *reinterpret_cast<const bf16x8 *>(B + b_frag[j] + (int64_t)kg * 1024 + 16 * lane);
            } else {
                const char *bk = B + (int64_t)kg * 64;
#pragma unroll
                for (int u = 0; u < LB; u++) lds_dma16_s(bk, b_off[u], st + ASZ + 1024 * u);
            }
        }
    };

    f32x4 acc[WR][WC];
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int fr = lane & 15, fg = lane >> 4;
    if (nst > 0) issue(0);
    // The epilogue's operands (bias, the old C of +=) of this thread's runs of
    // 4 columns are loaded ahead of the K loop: loaded behind it, every row
    // group would wait for them and for the previous group's stores.
    constexpr int Q = PR * (TN / 4), NQ = (Q + 64 * S - 1) / (64 * S);
    const bool vec = (g.ldc & 3) == 0 && ((uintptr_t)g.C & 15) == 0;
    constexpr bool HAS_B = (EPI & EPI_SWIGLU) == 0, HAS_C = (EPI & EPI_ACCUM) != 0;
    // (run u of a thread keeps its column over the row groups; one column for all u when 64 S is a multiple of TN / 4)
    constexpr int NB = 64 * S % (TN / 4) == 0 ? 1 : NQ;
    f32x4 eb[NB], ec[HAS_C ? PH : 1][HAS_C ? NQ : 1];
    auto ecol = [&](int u) { return min(n0 + ((t + u * 64 * S) % (TN / 4)) * 4, N - 1); };
#pragma unroll
    for (int u = 0; u < NB; u++) {
        eb[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (HAS_B && g.bias) eb[u] = gemm_load4(g.bias, ecol(u), N, ((uintptr_t)g.bias & 15) == 0);
    }
    if constexpr (HAS_C) {
#pragma unroll
        for (int ph = 0; ph < PH; ph++)
#pragma unroll
            for (int u = 0; u < NQ; u++) {
                const int m = min(m0 + ph * PR + (t + u * 64 * S) / (TN / 4), M - 1);
                ec[ph][u] = gemm_load4(g.C + (int64_t)m * g.ldc, ecol(u), N, vec);
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    for (int it = 0; it < nst; it += KU) {
        wait_vmcnt<0>();
        bf16x8 xb[KU][WC];
        float4 xa[KU][WR][2];
#pragma unroll
        for (int ku = 0; ku < KU; ku++) {
            const char *st = ring + ku * STG;
#pragma unroll
            for (int j = 0; j < WC; j++) {
                const int n = j * 16 + fr;
                if constexpr (BP) {
                    // (a use of the loaded value here: the compiler's own wait for
                    // it falls before the next stage's loads, not behind them)
                    asm volatile("" : "+v"(xn[ku][j]));
                    xb[ku][j] = xn[ku][j];
                } else {
                    xb[ku][j] = *reinterpret_cast<const bf16x8 *>(st + ASZ + n * 64 + ((fg ^ ((n >> 1) & 3)) * 16));
                }
            }
#pragma unroll
            for (int i = 0; i < WR; i++) {
                const int r = i * 16 + fr;
                xa[ku][i][0] = *reinterpret_cast<const float4 *>(st + r * 128 + (((2 * fg) ^ (r & 7)) * 16));
                xa[ku][i][1] = *reinterpret_cast<const float4 *>(st + r * 128 + (((2 * fg + 1) ^ (r & 7)) * 16));
            }
        }
        if (it + KU < nst) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the stage is in registers: refill it
            issue(it + KU);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ku = 0; ku < KU; ku++) {
            if (KU > 1 && ku > 0 && it + ku >= nst) break;
#pragma unroll
            for (int i = 0; i < WR; i++) {
                bf16x8 af[3];
                split3(xa[ku][i][0], xa[ku][i][1], af);
#pragma unroll
                for (int a = 2; a >= 0; a--)
#pragma unroll
                    for (int j = 0; j < WC; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], xb[ku][j], acc[i][j], 0, 0, 0);
            }
        }
    }

    // the S partial tiles meet in LDS, PR rows at a time; every thread then sums
    // the slices (in slice order) of its runs of 4 columns and finishes them
    float *P = reinterpret_cast<float *>(smem);
    const GeluRule gr(g.gelu_n, (EPI & EPI_GELU) != 0);
#pragma unroll
    for (int ph = 0; ph < PH; ph++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < WR / PH; i++)
#pragma unroll
            for (int j = 0; j < WC; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    P[(wave * PR + i * 16 + fg * 4 + r) * LD + j * 16 + fr] = acc[ph * (WR / PH) + i][j][r];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int idx = t + u * 64 * S;
            if (Q % (64 * S) != 0 && idx >= Q) break;
            const int row = idx / (TN / 4), c4 = (idx % (TN / 4)) * 4;
            f32x4 v = *reinterpret_cast<const f32x4 *>(P + row * LD + c4);
#pragma unroll
            for (int s = 1; s < S; s++) {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(P + (s * PR + row) * LD + c4);
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = __fadd_rn(v[e], x[e]);
            }
            const int m = m0 + ph * PR + row, n = n0 + c4;
            if (m < M && n < N) gemm_store4<EPI>(g, gr, m, n, v, eb[NB > 1 ? u : 0],
                                                ec[HAS_C ? ph : 0][HAS_C ? u : 0], vec);
        }
    }
}

// ---------------------------------------------------------------------------
// Plain rows of B with many tiles: a 128 x 128 tile per block whose four waves
// share every K-step (32 rows of A each, all columns) through a ring of three
// LDS stages, two in flight while one is computed, a block barrier per step.
// Per product it moves half the bytes of the 64 x 64 tiles above, whose waves
// each take whole K-steps; with few tiles those are faster, since they split
// the K chain.  Past the last K-step the ring is filled with that step again,
// so that the wait count is the same in every iteration.  VEC (16-byte aligned
// C rows): the columns are the MFMA's rows, so a lane ends with 4 consecutive
// columns; else a column per lane (16 consecutive floats per store).
// ---------------------------------------------------------------------------
template <int EPI, bool VEC>
__global__ __launch_bounds__(256, 2) void k_gemm_ring(GemmArgs g) {
    constexpr int T = 128, NS = 3, ASZ = T * 128, STG = ASZ + T * 64;
    constexpr int LA = 4, LB = 2, WR = 2, WC = 8;                    // one-KiB loads per wave and stage; fragments
    __shared__ __attribute__((aligned(16))) char smem[NS][STG];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int M = g.M, N = g.N, m0 = blockIdx.y * T, n0 = blockIdx.x * T, nk = g.K / 32;
    const char *A = reinterpret_cast<const char *>(g.A) + (int64_t)m0 * g.lda * 4;
    const char *B = reinterpret_cast<const char *>(g.B) + (int64_t)n0 * g.ldb * 2;
    uint32_t a_off[LA], b_off[LB];
#pragma unroll
    for (int u = 0; u < LA; u++) {
        const int r = 8 * (wave * LA + u) + (lane >> 3), p = (lane & 7) ^ (r & 7);
        a_off[u] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)g.lda * 4u + 16 * p;
    }
#pragma unroll
    for (int u = 0; u < LB; u++) {
        const int r = 16 * (wave * LB + u) + (lane >> 2), p = (lane & 3) ^ ((r >> 1) & 3);
        b_off[u] = (uint32_t)min(r, N - 1 - n0) * (uint32_t)g.ldb * 2u + 16 * p;
    }
    auto issue = [&](int buf, int kt) {
        char *st = smem[buf];
        const int kg = min(kt, nk - 1);
        const char *ak = A + (int64_t)kg * 128, *bk = B + (int64_t)kg * 64;
#pragma unroll
        for (int u = 0; u < LA; u++) lds_dma16_s(ak, a_off[u], st + 1024 * (wave * LA + u));
#pragma unroll
        for (int u = 0; u < LB; u++) lds_dma16_s(bk, b_off[u], st + ASZ + 1024 * (wave * LB + u));
    };
    f32x4 acc[WR][WC];
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int fr = lane & 15, fg = lane >> 4, mw = m0 + 32 * wave;
#pragma unroll
    for (int s = 0; s < NS - 1; s++) issue(s, s);
    for (int kt = 0; kt < nk; kt++) {
        wait_vmcnt<(LA + LB) * (NS - 2)>();   // this wave's loads of stage kt have landed
        __syncthreads();                      // ... and every wave's; stage kt - 1 is free
        issue((kt + NS - 1) % NS, kt + NS - 1);
        const char *st = smem[kt % NS];
        bf16x8 xb[WC];
#pragma unroll
        for (int j = 0; j < WC; j++) {
            const int n = j * 16 + fr;
            xb[j] = *reinterpret_cast<const bf16x8 *>(st + ASZ + n * 64 + ((fg ^ ((n >> 1) & 3)) * 16));
        }
#pragma unroll
        for (int i = 0; i < WR; i++) {
            const int r = wave * 32 + i * 16 + fr;
            bf16x8 af[3];
            split3(*reinterpret_cast<const float4 *>(st + r * 128 + (((2 * fg) ^ (r & 7)) * 16)),
                   *reinterpret_cast<const float4 *>(st + r * 128 + (((2 * fg + 1) ^ (r & 7)) * 16)), af);
#pragma unroll
            for (int a = 2; a >= 0; a--)
#pragma unroll
                for (int j = 0; j < WC; j++)
                    acc[i][j] = VEC ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(xb[j], af[a], acc[i][j], 0, 0, 0)
                                    : __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], xb[j], acc[i][j], 0, 0, 0);
        }
    }
    wait_vmcnt<0>();                          // no load may land in LDS after the block ends
    // the epilogue's operands (bias, the old C of +=), all of them ahead of the
    // first store, behind which a load would wait for it
    constexpr bool HAS_C = (EPI & EPI_ACCUM) != 0;
    f32x4 eb[WC], ec[HAS_C ? WR : 1][HAS_C ? WC : 1];
    const bool bv = ((uintptr_t)g.bias & 15) == 0;
#pragma unroll
    for (int j = 0; j < WC; j++) {
        const int n = min(n0 + 16 * j + (VEC ? 4 * fg : fr), N - 1);
        eb[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (g.bias) {
            if (VEC) eb[j] = gemm_load4(g.bias, n, N, bv);
            else eb[j][0] = g.bias[n];
        }
        if constexpr (HAS_C) {
#pragma unroll
            for (int i = 0; i < WR; i++) {
                if (VEC) {
                    ec[i][j] = gemm_load4(g.C + (int64_t)min(mw + 16 * i + fr, M - 1) * g.ldc, n, N, true);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        ec[i][j][r] = g.C[(int64_t)min(mw + 16 * i + 4 * fg + r, M - 1) * g.ldc + n];
                }
            }
        }
    }
    const GeluRule gr(0, false);
#pragma unroll
    for (int i = 0; i < WR; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) {
            if constexpr (VEC) {
                const int m = mw + 16 * i + fr, n = n0 + 16 * j + 4 * fg;
                if (m < M && n < N)
                    gemm_store4<EPI>(g, gr, m, n, acc[i][j], eb[j], ec[HAS_C ? i : 0][HAS_C ? j : 0], true);
            } else {
                const int n = n0 + 16 * j + fr;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = mw + 16 * i + 4 * fg + r;
                    float v = acc[i][j][r], c = ec[HAS_C ? i : 0][HAS_C ? j : 0][r];
                    if (HAS_C) v = __fadd_rn(g.bias ? __fadd_rn(c, eb[j][0]) : c, v);
                    else if (g.bias) v = __fadd_rn(v, eb[j][0]);
                    asm volatile("" : "+v"(v));              // formed here, not inside the store's branch
                    if (m < M && n < N) g.C[(int64_t)m * g.ldc + n] = v;
                }
            }
        }
}

// ---------------------------------------------------------------------------
// B [N][K] bf16 rows -> fragment-major, in place: column group c (16 rows of
// B) and K-step s (32 of K) are one KiB at (c K / 32 + s), in the order the
// lanes of the MFMA's B operand hold it: lane l holds row l % 16, K 8 (l / 16)
// .. + 7.  A block owns one column group (the same bytes before and after),
// read into registers whole; rows past N (a last partial group; the buffer
// holds whole groups) become zeros.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_pack_frag(uint16_t *b, int N, int K) {
    constexpr int U = GEMM_FRAG_MAX_K * 2 / 1024;                // 16-byte pieces per thread
    uint4 *g = reinterpret_cast<uint4 *>(b) + (int64_t)blockIdx.x * 2 * K;
    const int t = threadIdx.x, kp = K / 8, n = 16 * kp, rows = N - 16 * blockIdx.x;
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int p = t + 1024 * u;
        if (1024 * u >= n) break;
        v[u] = p < n && p / kp < rows ? g[p] : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (1024 * u >= n) break;
        const int p = t + 1024 * u, r = p / kp, c = p - r * kp;
        if (p < n) g[(c >> 2) * 64 + (c & 3) * 16 + r] = v[u];
    }
}

hipError_t launch_pack_frag(uint16_t *b, int64_t N, int64_t K, hipStream_t st) {
    if (N <= 0 || !gemm_frag_ok(K) || (uintptr_t)b % 16 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_pack_frag, dim3((unsigned)((N + 15) / 16)), dim3(1024), 0, st, b, (int)N, (int)K);
    return hipGetLastError();
}

// A tile form: its cost is the time of one tile per CU in units of one round
// of the cheapest form, so a call takes the form with the least rounds x cost.
struct KsForm { int tm, tn, cost; };

template <int NF>
static int ks_pick(const KsForm (&f)[NF], int M, int N, int64_t &best_cost) {
    int best = 0;
    best_cost = INT64_MAX;
    for (int i = 0; i < NF; i++) {
        const int64_t tiles = (int64_t)((M + f[i].tm - 1) / f[i].tm) * ((N + f[i].tn - 1) / f[i].tn);
        const int64_t c = (tiles + 255) / 256 * f[i].cost;
        if (c < best_cost) { best_cost = c; best = i; }
    }
    return best;
}

template <bool CONV, bool BP, int EPI, int TM, int TN, int S, int KU>
static void go_ks(GemmArgs g, hipStream_t st) {
    const unsigned tiles = (unsigned)((g.M + TM - 1) / TM) * (unsigned)((g.N + TN - 1) / TN);
    hipLaunchKernelGGL((k_gemm_ks<CONV, BP, EPI, TM, TN, S, KU>), dim3(tiles), dim3(64 * S), 0, st, g);
}

// the ring's cost in ks_pick's units; a CU holds two of its tiles at a time
static int64_t ring_cost(int M, int N) {
    const int64_t rounds = ((int64_t)((M + 127) / 128) * ((N + 127) / 128) + 255) / 256;
    return rounds / 2 * 380 + rounds % 2 * 320;
}

template <int EPI>
static void go_ring(const GemmArgs &g, hipStream_t st) {
    const dim3 grid((unsigned)((g.N + 127) / 128), (unsigned)((g.M + 127) / 128));
    if (g.N % 4 == 0 && g.ldc % 4 == 0 && (uintptr_t)g.C % 16 == 0)
        hipLaunchKernelGGL((k_gemm_ring<EPI, true>), grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL((k_gemm_ring<EPI, false>), grid, dim3(256), 0, st, g);
}

// Rows of f32.  The number of K slices depends on N and K alone, so that a row's
// result does not depend on how many rows share the call: 8 for N < 2048 (few
// tiles: the K chain is what shortens) from K = 512 on, else 4 (8 partial tiles
// cost more than they shorten: M = 404, N = 4096 15.5 against 12.8 us; plain
// rows, N = 1000, M = 1337, 8 -> 4 slices: K = 256 7.1 -> 6.1, K = 1024 13.3 ->
// 13.5, and M = 16 there 3.6 -> 4.4).  The tile is
// free (each element's sum runs over the same K-steps in the same order):
// costs from sweeps over M = 15 ... 1300 and the shapes of both models; e.g.
// N = 1024, K = 2048: 16 x 32 tiles 4.9-5.0 us up to 256 of them (M = 67; 32 x
// 64 7.9), 32 x 64 8.5 at M = 404 (32 x 32 11.0), 32 x 128 14.4 at M = 800
// (32 x 64 17.3), 48 x 128 20.6 at M = 1300 (32 x 128 25.5); N = 6144, K = 1024
// at M = 404 32 x 160 18.4 (32 x 64 20.8), N = 2688, K = 896 48 x 96 10.1 (10.9):
// larger tiles move fewer bytes per product where they leave no last round
// nearly empty.  Plain rows prefer 64 x 64 tiles to 32 x 128: half the B rows
// through LDS.
//
// Plain rows take the ring where its estimate is less, unless the caller wants
// rows alike (the ring adds the K-steps in one chain, so a row's bits would go
// with the number of rows).  us, these forms / the ring: M = 2048, N = 12288,
// K = 2048 432 / 243; M = 8192, N = 1024, K = 2048 131 / 88; M = 1600, N = 4096,
// K = 1024 52 / 40; M = 1337, N = 4096 43 / 38 (taken from there on); M = 1337,
// N = 6144 58 / 68; M = 404, N = 6144 22 / 29.
template <bool BP, int EPI>
static void go_ks_rows(const GemmArgs &g, hipStream_t st) {
    int64_t cost;
    const bool ring = !BP && !g.rows_alike && (g.M + 127) / 128 <= 65535;
    if (g.N < 2048 && g.K >= 512) {
        static const KsForm f[] = {{16, 32, 30}, {32, 32, 45}, {32, 64, 65}, {48, 64, 85}, {32, 128, 105}, {48, 128, 165}};
        const int best = ks_pick(f, g.M, g.N, cost);
        if constexpr (!BP)
            if (ring && ring_cost(g.M, g.N) <= cost) return go_ring<EPI>(g, st);
        switch (best) {
            case 0: go_ks<false, BP, EPI, 16, 32, 8, 2>(g, st); break;
            case 1: go_ks<false, BP, EPI, 32, 32, 8, 1>(g, st); break;
            case 2: go_ks<false, BP, EPI, 32, 64, 8, 1>(g, st); break;
            case 3: go_ks<false, BP, EPI, 48, 64, 8, 1>(g, st); break;
            case 4: go_ks<false, BP, EPI, 32, 128, 8, 1>(g, st); break;
            default: go_ks<false, BP, EPI, 48, 128, 8, 1>(g, st); break;
        }
        return;
    }
    if constexpr (BP) {
        static const KsForm f[] = {{16, 64, 26}, {32, 64, 40}, {48, 64, 54}, {32, 128, 70},
                                   {48, 96, 78}, {32, 160, 85}, {48, 128, 95}};
        switch (ks_pick(f, g.M, g.N, cost)) {
            case 0: go_ks<false, BP, EPI, 16, 64, 4, 2>(g, st); break;
            case 1: go_ks<false, BP, EPI, 32, 64, 4, 1>(g, st); break;
            case 2: go_ks<false, BP, EPI, 48, 64, 4, 1>(g, st); break;
            case 3: go_ks<false, BP, EPI, 32, 128, 4, 1>(g, st); break;
            case 4: go_ks<false, BP, EPI, 48, 96, 4, 1>(g, st); break;
            case 5: go_ks<false, BP, EPI, 32, 160, 4, 1>(g, st); break;
            default: go_ks<false, BP, EPI, 48, 128, 4, 1>(g, st); break;
        }
    } else {
        static const KsForm f[] = {{16, 64, 28}, {32, 64, 43}, {64, 64, 70}};
        const int best = ks_pick(f, g.M, g.N, cost);
        if (ring && ring_cost(g.M, g.N) <= cost) return go_ring<EPI>(g, st);
        switch (best) {
            case 0: go_ks<false, BP, EPI, 16, 64, 4, 2>(g, st); break;
            case 1: go_ks<false, BP, EPI, 32, 64, 4, 1>(g, st); break;
            default: go_ks<false, BP, EPI, 64, 64, 4, 1>(g, st); break;
        }
    }
}

// Convolutions: the number of slices goes with the form (a chunk's rows always
// come with their sequence's).  us per tile and CU at K = 4320 from sweeps: 16
// x 32 8, 32 x 32 13.8, 32 x 64 17.5, 32 x 96 25.5 (8 slices), 64 x 96 44, 32 x
// 160 33 (4 slices; the stem's 480 channels are 3 columns of 160, 5 of 96).
template <int EPI>
static void go_ks_conv(const GemmArgs &g, hipStream_t st) {
    static const KsForm f[] = {{16, 32, 80}, {32, 32, 138}, {32, 64, 175}, {32, 96, 255}, {64, 96, 440}, {32, 160, 330}};
    int64_t cost;
    switch (ks_pick(f, g.M, g.N, cost)) {
        case 0: go_ks<true, true, EPI, 16, 32, 8, 2>(g, st); break;
        case 1: go_ks<true, true, EPI, 32, 32, 8, 1>(g, st); break;
        case 2: go_ks<true, true, EPI, 32, 64, 8, 1>(g, st); break;
        case 3: go_ks<true, true, EPI, 32, 96, 8, 1>(g, st); break;
        case 4: go_ks<true, true, EPI, 64, 96, 4, 1>(g, st); break;
        default: go_ks<true, true, EPI, 32, 160, 4, 1>(g, st); break;
    }
}

// whole K-steps, 16-byte aligned rows, 32-bit offsets inside a tile (at most
// 128 rows of A, 160 of B), a tile count that fits the grid
bool gemm_ks_ok(const GemmArgs &g, int asrc, int bsrc, int epi) {
    const int64_t tiles = (int64_t)((g.M + 15) / 16) * ((g.N + 31) / 32);
    if (g.K % 32 != 0 || (uintptr_t)g.A % 16 != 0 || (uintptr_t)g.B % 16 != 0 || tiles >= 1ll << 31) return false;
    if (asrc == A_CONV) return bsrc == B_BF16_FRAG && (epi == EPI_NONE || epi == (EPI_GELU | EPI_CHW));
    if (asrc != A_F32_SPLIT || g.lda % 4 != 0 || g.lda >= 1 << 23) return false;
    if (bsrc == B_BF16) return g.ldb % 8 == 0 && g.ldb < 1 << 23 && (epi == EPI_NONE || epi == EPI_ACCUM);
    return bsrc == B_BF16_FRAG &&
           (epi == EPI_NONE || epi == EPI_ACCUM || epi == EPI_GELU || (epi == EPI_SWIGLU && g.N % 2 == 0));
}

hipError_t launch_gemm_ks(const GemmArgs &g0, int asrc, int bsrc, int epi, hipStream_t st) {
    GemmArgs g = g0;
    if (!gemm_ks_ok(g, asrc, bsrc, epi)) return hipErrorInvalidValue;
    // neighbouring tiles share the strip of the operand with more bytes
    g.m_major = asrc == A_CONV || 2 * (int64_t)g.M > g.N;
    if (asrc == A_CONV) {
        if (epi == EPI_NONE) go_ks_conv<EPI_NONE>(g, st);
        else go_ks_conv<EPI_GELU | EPI_CHW>(g, st);
    } else if (bsrc == B_BF16) {
        if (epi == EPI_NONE) go_ks_rows<false, EPI_NONE>(g, st);
        else go_ks_rows<false, EPI_ACCUM>(g, st);
    } else {
        switch (epi) {
            case EPI_NONE: go_ks_rows<true, EPI_NONE>(g, st); break;
            case EPI_ACCUM: go_ks_rows<true, EPI_ACCUM>(g, st); break;
            case EPI_GELU: go_ks_rows<true, EPI_GELU>(g, st); break;
            default: go_ks_rows<true, EPI_SWIGLU>(g, st); break;
        }
    }
    return hipGetLastError();
}

}  // namespace qasr
