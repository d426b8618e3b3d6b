// rh_gemm_epi.h -- what the prefill GEMM kernels do with four consecutive
// output features of one token (rh_gemm.hip, rh_skinny.hip).
#pragma once
#include "rh_device.h"
#include "rh_kernels.h"

namespace rh {
namespace {

// SiLU-gate backward (layer.rs:7083-7104) of the gate gradient g = (v0..v3)
// of token m, features n..n+3, and the saved a1 = h1, a3 = h3 there:
// dh3 = g silu(h1), dh1 = g h3 silu'(h1), fp16 in fragment order [M][2N]
// (dh1 in columns 0..N-1, dh3 in N..2N-1).
__device__ __forceinline__ void silu_bwd4(const GemmArgs& a, int m, int n, float v0, float v1, float v2, float v3,
                                          f16x4 a1, f16x4 a3) {
    const float g[4] = {v0, v1, v2, v3};
    f16x4 o1, o3;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float h1 = (float)a1[e], h3 = (float)a3[e];
        const float sig = 1.0f / (1.0f + __expf(-h1));
        o3[e] = (f16)(g[e] * (h1 * sig));
        o1[e] = (f16)(g[e] * h3 * (sig * (1.0f + h1 * (1.0f - sig))));
    }
    *(f16x4*)(a.out_f16 + frag_off(m, n, 2 * a.ldo)) = o1;
    *(f16x4*)(a.out_f16 + frag_off(m, a.ldo + n, 2 * a.ldo)) = o3;
}

// The fp32 output that holds feature n; n becomes the feature's column in it.
// (The pointers are read before the choice: a choice between fields would put
// the argument copies of the split kernels in scratch memory.)
__device__ __forceinline__ float* out_part(const GemmArgs& a, int& n) {
    float *p0 = a.out_f32, *p1 = a.out_part1, *p2 = a.out_part2;
    const int c = a.part_cols;
    if (c == 0) return p0;
    const int k = (n >= c) + (n >= 2 * c);
    n -= k * c;
    return k == 0 ? p0 : k == 1 ? p1 : p2;
}

// Stores four consecutive output features n..n+3 of token m (every epilogue
// but SwiGLU, whose lanes hold W1 and W3 rows and store gate features).
template <int EPI>
__device__ __forceinline__ void store4(const GemmArgs& a, int m, int n, float v0, float v1, float v2, float v3) {
    if constexpr (EPI == EPI_F32) {
        if (a.alpha != 0.f) {  // optional output scale (0 = none)
            v0 *= a.alpha; v1 *= a.alpha; v2 *= a.alpha; v3 *= a.alpha;
        }
        if (a.softcap > 0.f) {
            const float c = a.softcap, ic = 1.0f / c;
            v0 = tanhf(v0 * ic) * c; v1 = tanhf(v1 * ic) * c;
            v2 = tanhf(v2 * ic) * c; v3 = tanhf(v3 * ic) * c;
        }
        f32x4* po = (f32x4*)(out_part(a, n) + (size_t)m * a.ldo + n);
        if (a.nt_out) __builtin_nontemporal_store(f32x4{v0, v1, v2, v3}, po);
        else *po = f32x4{v0, v1, v2, v3};
    } else if constexpr (EPI == EPI_RESID) {
        float* out = out_part(a, n);
        const size_t o = (size_t)m * a.ldo + n;
        f32x4* px = (f32x4*)(out + o);
        f32x4 x = *(const f32x4*)((a.resid_in ? a.resid_in : out) + o);
        x[0] = v0 * a.alpha + x[0]; x[1] = v1 * a.alpha + x[1];
        x[2] = v2 * a.alpha + x[2]; x[3] = v3 * a.alpha + x[3];
        if (a.nt_out) __builtin_nontemporal_store(x, px);
        else *px = x;
    } else if constexpr (EPI == EPI_QKV) {
        // no integer divisions by run-time values here but the per-row m / S
        // (hoisted out of the feature loop): n < 3D, hd a power of two
        const int sec = (n >= a.D) + (n >= 2 * a.D), c = n - sec * a.D;
        const int h = c >> __builtin_ctz(a.hd), d = c & (a.hd - 1);
        const int b = m / a.S, s = m - b * a.S, pos = a.pos0 + s;
        if (sec < 2) {
            const float2 cs0 = a.rope[(size_t)pos * (a.hd / 2) + d / 2];
            const float2 cs1 = a.rope[(size_t)pos * (a.hd / 2) + d / 2 + 1];
            const float r0 = v0 * cs0.x + (-v1) * cs0.y, r1 = v1 * cs0.x + v0 * cs0.y;
            const float r2 = v2 * cs1.x + (-v3) * cs1.y, r3 = v3 * cs1.x + v2 * cs1.y;
            v0 = r0; v1 = r1; v2 = r2; v3 = r3;
        }
        f16* dst;
        if (sec == 0)
            dst = a.q + (((size_t)b * a.H + h) * a.S + s) * a.hd + d;
        else
            dst = (sec == 1 ? a.kc : a.vc) + (((size_t)b * a.H + h) * a.ctx + pos) * a.hd + d;
        *(f16x4*)dst = f16x4{(f16)v0, (f16)v1, (f16)v2, (f16)v3};
    } else if constexpr (EPI == EPI_SILU_BWD) {
        const size_t o = (size_t)m * a.ldo + n, plane = (size_t)a.M * a.ldo;
        silu_bwd4(a, m, n, v0, v1, v2, v3, *(const f16x4*)(a.h13 + o), *(const f16x4*)(a.h13 + plane + o));
    }
}

// SwiGLU output of token m, gate features f..f+3 from h1 (W1 rows) and h3
// (the matching W3 rows); EPI_SWIGLU_SAVE also keeps h1, h3 for the backward.
template <int EPI>
__device__ __forceinline__ void store_swiglu(const GemmArgs& a, int m, int f, const float (&h1)[4],
                                             const float (&h3)[4]) {
    f16x4 g;
#pragma unroll
    for (int r = 0; r < 4; ++r) g[r] = (f16)(silu_f(h1[r]) * h3[r]);
    *(f16x4*)(a.out_f16 + frag_off(m, f, a.ldo)) = g;
    if constexpr (EPI == EPI_SWIGLU_SAVE) {
        // the pre-activations for the backward pass: h1 | h3 planes [M][F]
        const size_t o = (size_t)m * a.ldo + f, plane = (size_t)a.M * a.ldo;
        *(f16x4*)(a.h13 + o) = f16x4{(f16)h1[0], (f16)h1[1], (f16)h1[2], (f16)h1[3]};
        *(f16x4*)(a.h13 + plane + o) = f16x4{(f16)h3[0], (f16)h3[1], (f16)h3[2], (f16)h3[3]};
    }
}

}  // namespace
}  // namespace rh
