/*
 * gemm_device.h - what the GEMM kernels share (gemm.hip, gemm_rs.hip,
 * gemm_sw.hip): the tile of a workgroup, the split of fp32 rows into bf16
 * hi + lo, and the fused operations at a tile's end.
 */
#ifndef SMOL_GEMM_DEVICE_H
#define SMOL_GEMM_DEVICE_H

#include "attn_device.h"
#include "smol_linear.h"

#define GEMM_XCD 8

namespace {

/* the tile (row block tm, output block tn) of workgroup b; workgroups b and
 * b + 8 run on one XCD; false: the workgroup has none */
__device__ __forceinline__ bool gemm_tile_of(const GemmParams &p, int b, int &tm, int &tn) {
    const int xcd = b % GEMM_XCD, idx = b / GEMM_XCD;
    if (p.rm > 0) {
        /* XCD x: region (x / rn, x % rn) of the tile grid, so the rows of x
         * and of W that its tiles share stay in its own L2 */
        const int tiles_n = p.tiles / p.tiles_m;
        const int ri = xcd / p.rn, rj = xcd % p.rn;
        const int m_lo = ri * p.tiles_m / p.rm, m_hi = (ri + 1) * p.tiles_m / p.rm;
        const int n_lo = rj * tiles_n / p.rn, n_hi = (rj + 1) * tiles_n / p.rn;
        if (idx >= (m_hi - m_lo) * (n_hi - n_lo)) return false;
        tm = m_lo + idx % (m_hi - m_lo);
        tn = n_lo + idx / (m_hi - m_lo);
    } else {
        const int t = xcd * p.per_xcd + idx;
        if (idx >= p.per_xcd || t >= p.tiles) return false;
        tm = t % p.tiles_m;
        tn = t / p.tiles_m;
    }
    return true;
}

/* the output that column n of the joint column space belongs to: its
 * segment's weight rows, y, width, and n within it (a tile never straddles
 * two segments) */
struct GemmOut {
    const uint16_t *w;
    void *y;
    int n0, n;
};
__device__ __forceinline__ GemmOut gemm_out_of(const GemmParams &p, int n) {
    GemmOut o{p.w, p.y, n, p.N};
    if (p.nseg > 0) {
        const int sg = (n >= p.seg_c[1] ? 1 : 0) + (p.nseg > 2 && n >= p.seg_c[2] ? 1 : 0);
        const int c0 = sg == 0 ? 0 : sg == 1 ? p.seg_c[1] : p.seg_c[2];
        o.n = (sg == 0 ? p.seg_c[1] : sg == 1 ? p.seg_c[2] : p.seg_c[3]) - c0;
        o.w = sg == 0 ? p.seg_w[0] : sg == 1 ? p.seg_w[1] : p.seg_w[2];
        o.y = sg == 0 ? p.seg_y[0] : sg == 1 ? p.seg_y[1] : p.seg_y[2];
        o.n0 -= c0;
    }
    return o;
}

__device__ __forceinline__ float act_fn(float g, int act) {
    if (act == SMOL_LINEAR_ACT_SWIGLU) return g / (1.0f + expf(-g));
    const float x3 = g * g * g;
    const float inner = 0.7978845608028654f * (g + 0.044715f * x3);
    return 0.5f * g * (1.0f + tanhf(inner));
}

/* x_hi = bf16_rne(x), x_lo = bf16_rne(xc - bf16_rne(xc)) of 8 floats, xc =
 * x clamped to bf16's largest finite magnitude (about 3.39e38): the same
 * x_lo for every |x| up to that bound, 0 for an infinite x (which goes to
 * x_hi whole and so reaches y as it would in fp32), never an infinite or
 * NaN lo part beside a finite one. Per pair: one packed conversion for the
 * hi pair, two clamps, two conversions over a zero low half (which are
 * bf16(xc) as floats), two differences, one packed conversion for the lo
 * pair. */
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float fl2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_frag(const float *v, b8 &hi, b8 &lo) {
    constexpr float BF16_MAX = 3.3895313892515355e38f;
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x0 = v[2 * i], x1 = v[2 * i + 1];
        hw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((fl2){x0, x1}, bf2));
        const float c0 = __builtin_amdgcn_fmed3f(x0, -BF16_MAX, BF16_MAX);
        const float c1 = __builtin_amdgcn_fmed3f(x1, -BF16_MAX, BF16_MAX);
        const float h0 = __builtin_bit_cast(float, __builtin_convertvector((fl2){0.0f, c0}, bf2));
        const float h1 = __builtin_bit_cast(float, __builtin_convertvector((fl2){0.0f, c1}, bf2));
        lw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((fl2){c0 - h0, c1 - h1}, bf2));
    }
    hi = as_b8(make_uint4(hw[0], hw[1], hw[2], hw[3]));
    lo = as_b8(make_uint4(lw[0], lw[1], lw[2], lw[3]));
}

/* A row's sum of squares over 64-wide steps, eight lanes a row (lane lq holds
 * chunk lq, eight values), in k_gemm's order: four running sums, of chunks q and
 * then q + 4, which rest in lanes lq < 4, go to lanes lq + 4 and come back; at
 * the end they are added as row_sum4 does (every lane lq < 4 gets the row's) */
__device__ __forceinline__ float gemm_squares64(const float *v, float ss) {
    auto squares = [&](float t) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 8; b++) t = fmaf(v[b], v[b], t);
        return t;
    };
    const float up = __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(squares(ss)),
                                                                 0x114 /* row_shr:4 */, 0xf, 0xf, true));
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(squares(up)), 0x104 /* row_shl:4 */, 0xf,
                                                       0xf, true));
}
__device__ __forceinline__ float gemm_squares64_sum(float t) {
    t += __shfl_xor(t, 2, 64);
    return t + __shfl_xor(t, 1, 64);
}

/* v truncated to bf16, and the bf16 decoder's GeGLU of a truncated (gate, up)
 * pair before its own truncation: every step rounded as written
 * (qkn_bf16_decoder.c:235-251) */
__device__ __forceinline__ float bf16_trunc(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }
__device__ __forceinline__ float bf16_geglu(float g, float u) {
    const float x3 = __fmul_rn(__fmul_rn(g, g), g);
    const float inner = __fmul_rn(0.7978845608028654f, __fadd_rn(g, __fmul_rn(0.044715f, x3)));
    return __fmul_rn(__fmul_rn(__fmul_rn(0.5f, g), __fadd_rn(1.0f, tanhf(inner))), u);
}

/* Outputs n .. n + 3 (n < NN, a multiple of 4) of row m from their sums v:
 * row scale r (NORM), bias, activation, residual, store (a bf16 y truncates;
 * its activation is the bf16 decoder's GeGLU) */
template <bool YBF, bool NORM>
__device__ __forceinline__ void gemm_store4(const GemmParams &p, void *Yt, int m, int n, int NN, float (&v)[4],
                                            float r) {
    const bool has_act = p.act != SMOL_LINEAR_ACT_NONE;
    const int ycols = has_act ? NN / 2 : NN;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (NORM) v[e] *= r;
        if (p.bias) v[e] += n + e < NN ? p.bias[n + e] : 0.0f;
    }
    if (has_act) {
        const int col = n / 2;
        float o[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            if constexpr (YBF) o[e] = bf16_geglu(bf16_trunc(v[2 * e]), bf16_trunc(v[2 * e + 1]));
            else o[e] = act_fn(v[2 * e], p.act) * v[2 * e + 1];
        }
        const long long yi = (long long)m * ycols + col;
        const int nv = min(2, ycols - col);
        if (p.res) {
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (e < nv) o[e] += p.res[yi + e];
        }
        if constexpr (YBF) {
            uint16_t *y = static_cast<uint16_t *>(Yt) + yi;
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (e < nv) y[e] = (uint16_t)(__float_as_uint(o[e]) >> 16);
        } else {
            float *y = static_cast<float *>(Yt) + yi;
            if (nv == 2 && ((yi & 1) == 0)) *reinterpret_cast<float2 *>(y) = make_float2(o[0], o[1]);
            else
                for (int e = 0; e < nv; e++) y[e] = o[e];
        }
    } else {
        const long long yi = (long long)m * ycols + n;
        const int nv = min(4, NN - n);
        if (p.res) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (e < nv) v[e] += p.res[yi + e];
        }
        if constexpr (YBF) {
            uint16_t *y = static_cast<uint16_t *>(Yt) + yi;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (e < nv) y[e] = (uint16_t)(__float_as_uint(v[e]) >> 16);
        } else {
            float *y = static_cast<float *>(Yt) + yi;
            if (nv == 4 && ((yi & 3) == 0)) *reinterpret_cast<float4 *>(y) = make_float4(v[0], v[1], v[2], v[3]);
            else
                for (int e = 0; e < nv; e++) y[e] = v[e];
        }
    }
}

} // namespace

#endif
