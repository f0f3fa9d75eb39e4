// Device pieces shared by the GEMM translation units.
#pragma once
#include "kernels.h"

namespace qasr {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// One global_load_lds_dwordx4: lane l's 16 bytes from g land at LDS byte
// lds + 16 l.  Written as inline assembly, with the waits below, because the
// compiler otherwise treats every LDS read as possibly aliasing any load in
// flight and waits for all of them (vmcnt(0)) before it, which would drain
// the stages every step.  The compiler does not see these loads.  Vector-memory
// loads complete in the order in which a wave issued them, so
//   - the compiler's own waits, which count only the loads it sees, are at
//     least as strict as they need to be: a hidden load that is younger than
//     the one waited for makes vmcnt(n) wait for more, never for less;
//   - wait_vmcnt<N> here is right where at least N loads of the wave are younger
//     than the ones it waits for.  k_gemm_lds and k_gemm_ring: the loads of the
//     NS - 2 stages behind (their other loads come before the first stage or
//     after the last wait).  k_gemm_ks: N = 0.  k_attn_mfma and k_attn_bf3: the
//     L loads of the next K tile or of the V tile; q is loaded behind the first
//     two tiles and waited for ahead of the loop.
// The compiler makes no use of M0 in the kernels of the files that include this
// header (every mention of it in their generated code is one of these lines).
// The s_nop is the wait state GFX9 asks for between a scalar write of M0 and
// an LDS load that reads it.
__device__ __forceinline__ void lds_dma16(const void *g, const void *lds) {
    const uint32_t la = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)lds;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(la) : "memory");
}
// the same from a wave-uniform base plus a 32-bit byte offset per lane
__device__ __forceinline__ void lds_dma16_s(const void *base, uint32_t off, const void *lds) {
    const uint32_t la = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)lds;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(la) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// float pair -> bf16 pair, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// 8 f32 = hi + mid + lo, each term the RNE bf16 of the remaining residual.  A
// residual x - (float)h is v_dot2_f32_bf16 of the packed pair with (-1, 0) or
// (0, -1) plus x: one instruction per value where a shift or mask and a
// subtraction are two, and exact, since the difference is representable
// (bit-identical to the subtraction over 2^20 random values of 200 binades;
// the GEMM 3-8% faster).  The constants stay in registers: as literals the
// compiler folds -1.0 into an f32 inline constant, another value here.
__device__ __forceinline__ void split3(const float4 x0, const float4 x1, bf16x8 *af) {
    uint32_t c0, c1;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
    const bf16x2 e0 = __builtin_bit_cast(bf16x2, c0), e1 = __builtin_bit_cast(bf16x2, c1);
    const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    uint32_t hi[4], mi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        hi[e] = cvt_pk_bf16(xv[2 * e], xv[2 * e + 1]);
        const bf16x2 h = __builtin_bit_cast(bf16x2, hi[e]);
        const float r0 = __builtin_amdgcn_fdot2_f32_bf16(h, e0, xv[2 * e], false);
        const float r1 = __builtin_amdgcn_fdot2_f32_bf16(h, e1, xv[2 * e + 1], false);
        mi[e] = cvt_pk_bf16(r0, r1);
        const bf16x2 m = __builtin_bit_cast(bf16x2, mi[e]);
        lo[e] = cvt_pk_bf16(__builtin_amdgcn_fdot2_f32_bf16(m, e0, r0, false),
                            __builtin_amdgcn_fdot2_f32_bf16(m, e1, r1, false));
    }
    af[0] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
    af[1] = __builtin_bit_cast(bf16x8, make_uint4(mi[0], mi[1], mi[2], mi[3]));
    af[2] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
}

// gelu_ref's path choice over a buffer of n elements: when none of gelu()'s
// 16 per-thread chunks has a scalar tail every element takes the vector form,
// and the per-element index arithmetic is left out
struct GeluRule {
    int64_t n;
    bool all_vec;
    __device__ __forceinline__ GeluRule(int64_t n_, bool used) : n(n_), all_vec(false) {
        if (used && n > 4096 && n < (int64_t)1 << 31) all_vec = (n & 127) == 0;   // 16 equal chunks, each a multiple of 8
    }
    __device__ __forceinline__ float operator()(float v, int64_t idx) const {
        return all_vec ? gelu_at(v, true) : gelu_ref(v, idx, n);
    }
};

// 4 consecutive floats p[n .. n + 3] of a row of N (n < N; repeats past the end)
__device__ __forceinline__ f32x4 gemm_load4(const float *p, int n, int N, bool vec) {
    if (vec && n + 3 < N) return *reinterpret_cast<const f32x4 *>(p + n);
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = p[min(n + e, N - 1)];
    return v;
}

// the epilogue of 4 consecutive columns n .. n + 3 of row m (n % 4 == 0): b
// holds their bias, c the old C (EPI_ACCUM); vec: C rows are 16-byte aligned
template <int EPI>
__device__ __forceinline__ void gemm_store4(const GemmArgs &g, const GeluRule &gr, int m, int n, f32x4 v, f32x4 b,
                                            f32x4 c, bool vec) {
    if constexpr ((EPI & EPI_SWIGLU) != 0) {
        // columns (n, n + 1) are a (gate, up) pair: outputs n / 2, n / 2 + 1
        const int half = g.N >> 1, nv = half - half % 8;
        float *cp = g.C + (int64_t)m * g.ldc + (n >> 1);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int jj = (n >> 1) + e;
            if (jj >= half) break;
            const float gt = v[2 * e], up = v[2 * e + 1];
            const float x = jj < nv ? fast_exp_ref(__fsub_rn(0.0f, gt)) : expf(-gt);
            cp[e] = __fmul_rn(__fdiv_rn(gt, __fadd_rn(1.0f, x)), up);
        }
        return;
    }
    float *cp = g.C + (int64_t)m * g.ldc + n;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (EPI & EPI_ACCUM) {
            if (g.bias) c[e] = __fadd_rn(c[e], b[e]);
            v[e] = __fadd_rn(c[e], v[e]);
        } else if (g.bias) {
            v[e] = __fadd_rn(v[e], b[e]);
        }
        if (EPI & EPI_GELU) {
            const int64_t gidx = (EPI & EPI_CHW) ? (int64_t)(n + e) * g.gelu_rows + m % g.gelu_rows
                                                 : (int64_t)m * g.ldc + n + e;
            v[e] = gr(v[e], gidx);
        }
    }
    if (vec && n + 3 < g.N) {
        *reinterpret_cast<f32x4 *>(cp) = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < g.N) cp[e] = v[e];
    }
}

}  // namespace qasr
