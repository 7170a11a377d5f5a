/*
 * gemm_kw.hip - k_gemm_kw: the projections of k_gemm (gemm.hip: the same
 * operands, products and fused operations) for launches whose k_gemm tiles
 * would leave the device idle or waiting: a few to a few hundred rows.
 *
 * What bounds those launches is latency, not a rate: k_gemm stages each
 * 64-wide K step through LDS behind a barrier, so a step costs about a
 * memory round trip. Here the KW waves of a workgroup split K instead of
 * the tile: each forms the whole BM x BN tile (rows x outputs) over its own
 * KC-wide steps, w, w + KW, ..., and meets the others only at the end, when
 * the waves' sums are added in wave order. A wave loads a step as whole row
 * pieces (16 bytes a lane, neighbouring lanes along a row) into registers,
 * DEPTH steps ahead, splits an fp32 x as k_gemm does, and passes it through
 * its own LDS region into the MFMA operand layout: no barrier, and the
 * waits are the compiler's counted ones. (Loading the operand layout
 * straight from memory, where sixteen neighbouring lanes hold sixteen rows,
 * needs no LDS but reaches a quarter of the 64 bytes a clock that a compute
 * unit can load: one cache line per lane.)
 *
 * Measured, k_gemm before and this kernel now: 26 fp32 rows, 6144 -> 2048:
 * 49 -> 11.3 us (25 MB of weights: 2.2 TB/s); 2048 -> 2048: 18.2 -> 7.7 us;
 * 2048 -> 12288 with the norm and SwiGLU: 22.4 -> 14.6 us (50 MB: 3.4 TB/s);
 * 333 bf16 rows, 3072 -> 1024: 24.3 -> 13.4 us; 1024 -> 1024: 11.7 -> 7.8 us.
 * From about 700 rows on the tile kernel is the faster one: its tile is
 * loaded once for all its waves (1536 fp32 rows, 1024 -> 6144: 51 us, here
 * 76). The host chooses by a fitted cost of each (gemm_cfg, linear.hip).
 */
#include "gemm_device.h"

template <int MT, int NT, int KW, bool XBF, bool YBF, bool NORM>
__global__ __launch_bounds__(64 * KW) __attribute__((amdgpu_waves_per_eu(2, 4)))
void k_gemm_kw(const GemmParams p) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    constexpr int KC = MT * NT >= 8 ? 32 : 64; /* K of a step */
    constexpr int CPR = KC / 8;                /* 16-byte bf16 chunks of a row */
    constexpr int WL = BN * CPR / 64, XL = BM * CPR / 64; /* chunks a lane loads of W and x */
    constexpr int STEP_REGS = 4 * WL + (XBF ? 4 : 8) * XL + (NORM ? 8 : 0);
    constexpr int DEPTH = STEP_REGS > 40 ? 2 : STEP_REGS > 24 ? 3 : 4;
    constexpr int STAGE = (BN + (XBF ? 1 : 2) * BM) * KC * 2; /* W, x hi, x lo of one step */
    constexpr int QN = BN / 4; /* 16-byte chunks of a partial's row */
    constexpr int LDS = KW * (STAGE > BM * BN * 4 ? STAGE : BM * BN * 4);
    /* a step per wave; at the end a partial tile [BM][BN] per wave */
    __shared__ __attribute__((aligned(16))) unsigned char smem[LDS];
    __shared__ float s_ss[NORM ? KW * BM : 1];
    /* both with their 16-byte chunks XOR-swizzled by the row, so that the
     * eight lanes that an LDS access serves at a time hit distinct banks */
    auto part = [&](int w, int row, int q) __attribute__((always_inline)) {
        const int sw = QN == 4 ? (row >> 1) & 3 : row & 7;
        return reinterpret_cast<f4 *>(smem + ((w * BM + row) * BN + 4 * (q ^ sw)) * 4);
    };

    int tm, tn;
    if (!gemm_tile_of(p, blockIdx.x, tm, tn)) return;
    const int m0 = tm * BM, K = p.K;
    const GemmOut out = gemm_out_of(p, tn * BN);
    const int n0 = out.n0, NN = out.n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, j = lane >> 4;
    unsigned char *const st = smem + wave * STAGE;
    auto stage = [&](int base, int row, int q) __attribute__((always_inline)) {
        const int sw = CPR == 4 ? (row >> 1) & 3 : row & 7;
        return reinterpret_cast<uint4 *>(st + base + row * (KC * 2) + ((q ^ sw) << 4));
    };
    constexpr int XH = BN * KC * 2, XLO = XH + BM * KC * 2;

    /* lane: chunk lq (8 elements) of rows lr + (64 / CPR) e. Rows past the
     * operands read zero by the buffer's range; the step's offset goes in
     * the scalar offset, which the range check leaves out */
    constexpr int xes = XBF ? 2 : 4;
    const rsrc_t rw = make_rsrc(out.w + (long long)n0 * K, (long long)min(BN, NN - n0) * K * 2);
    const rsrc_t rx = make_rsrc(static_cast<const char *>(p.x) + (long long)m0 * K * xes,
                                (long long)min(BM, p.M - m0) * K * xes);
    const rsrc_t rg = make_rsrc(NORM ? (const void *)p.g : (const void *)out.w, NORM ? (long long)K * 4 : 0);
    const int lr = lane / CPR, lq = lane % CPR;
    unsigned w_off[WL], x_off[XL], g_off = (unsigned)(32 * lq);
#pragma unroll
    for (int e = 0; e < WL; e++) w_off[e] = (unsigned)(((lr + 64 / CPR * e) * K + 8 * lq) * 2);
#pragma unroll
    for (int e = 0; e < XL; e++) x_off[e] = (unsigned)(((lr + 64 / CPR * e) * K + 8 * lq) * xes);

    struct Raw {
        uint4 w[WL], x[XL][XBF ? 1 : 2], g[NORM ? 2 : 1];
    };
    const int n_steps = (K + KC - 1) / KC;
    const int mine = wave < n_steps ? (n_steps - wave + KW - 1) / KW : 0;
    int next = wave; /* the step the next issue loads */
    auto issue = [&](Raw &r) __attribute__((always_inline)) {
        const int k0 = KC * next;
        if (k0 + KC > K && k0 + 8 * lq >= K) {
            /* K's end inside the step, or steps past it: these lanes load zeros from here on */
#pragma unroll
            for (int e = 0; e < WL; e++) w_off[e] = OOB_OFF;
#pragma unroll
            for (int e = 0; e < XL; e++) x_off[e] = OOB_OFF;
            g_off = OOB_OFF;
        }
        if constexpr (NORM) {
            r.g[0] = bload(rg, g_off, (unsigned)(k0 * 4));
            r.g[1] = bload(rg, g_off + 16u, (unsigned)(k0 * 4));
        }
#pragma unroll
        for (int e = 0; e < XL; e++) {
            r.x[e][0] = bload(rx, x_off[e], (unsigned)(k0 * xes));
            if constexpr (!XBF) r.x[e][1] = bload(rx, x_off[e] + 16u, (unsigned)(k0 * xes));
        }
#pragma unroll
        for (int e = 0; e < WL; e++) r.w[e] = bload(rw, w_off[e], (unsigned)(k0 * 2));
        next += KW;
    };

    f4 acc[NT][MT];
    float ss[XL];
#pragma unroll
    for (int e = 0; e < XL; e++) ss[e] = 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t][mt] = f4{0.f, 0.f, 0.f, 0.f};
    Raw raw[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; d++) issue(raw[d]);
    for (int i = 0; i < mine; i += DEPTH)
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
        if (i + d >= mine) break;
        Raw &r = raw[d];
        /* this step into the wave's region (a wave's LDS accesses execute in
         * order: the fences only hold the compiler to it) */
#pragma unroll
        for (int e = 0; e < XL; e++) {
            const int row = lr + 64 / CPR * e;
            if constexpr (XBF) {
                *stage(XH, row, lq) = r.x[e][0];
            } else {
                const uint4 u = r.x[e][0], w = r.x[e][1];
                float v[8] = {__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w),
                              __uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w)};
                if constexpr (NORM) {
                    const uint4 g0 = r.g[0], g1 = r.g[1];
                    const uint32_t g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
                    for (int b = 0; b < 8; b++) {
                        ss[e] = fmaf(v[b], v[b], ss[e]);
                        v[b] *= __uint_as_float(g[b]);
                    }
                }
                b8 h, l;
                split_frag(v, h, l);
                *reinterpret_cast<b8 *>(stage(XH, row, lq)) = h;
                *reinterpret_cast<b8 *>(stage(XLO, row, lq)) = l;
            }
        }
#pragma unroll
        for (int e = 0; e < WL; e++) *stage(0, lr + 64 / CPR * e, lq) = r.w[e];
        issue(r);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int ks = 0; ks < KC / 32; ks++) {
            b8 a[NT], h[MT], l[XBF ? 1 : MT];
#pragma unroll
            for (int t = 0; t < NT; t++) a[t] = as_b8(*stage(0, 16 * t + c, 4 * ks + j));
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                h[mt] = as_b8(*stage(XH, 16 * mt + c, 4 * ks + j));
                if constexpr (!XBF) l[mt] = as_b8(*stage(XLO, 16 * mt + c, 4 * ks + j));
            }
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], h[mt], acc[t][mt], 0, 0, 0);
            if constexpr (!XBF) {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], l[mt], acc[t][mt], 0, 0, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    /* the waves' partial tiles, over the staging once every wave is done
     * with it: lane (c, j) holds outputs 4 j + e of row c of each 16 x 16
     * product */
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) *part(wave, 16 * mt + c, 4 * t + j) = acc[t][mt];
    if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < XL; e++) {
            float s = ss[e];
#pragma unroll
            for (int m = 1; m < CPR; m <<= 1) s += __shfl_xor(s, m, 64);
            if (lq == 0) s_ss[wave * BM + lr + 64 / CPR * e] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (BM * QN + 64 * KW - 1) / (64 * KW); i++) {
        const int idx = tid + 64 * KW * i;
        const int row = idx / QN, q = idx % QN;
        const int m = m0 + row, n = n0 + 4 * q;
        if (idx >= BM * QN || m >= p.M || n >= NN) continue;
        f4 s = *part(0, row, q);
#pragma unroll
        for (int w = 1; w < KW; w++) s += *part(w, row, q);
        float r = 1.0f;
        if constexpr (NORM) {
            float t = s_ss[row];
#pragma unroll
            for (int w = 1; w < KW; w++) t += s_ss[w * BM + row];
            r = 1.0f / sqrtf(t / (float)K + p.eps);
        }
        float v[4] = {s[0], s[1], s[2], s[3]};
        gemm_store4<YBF, NORM>(p, out.y, m, n, NN, v, r);
    }
}

/* ------------------------------------------------------------------ launch */

template <int MT, int NT, int KW>
static int launch_kw(const GemmParams &p, bool xbf, bool ybf, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const dim3 grid((unsigned)(GEMM_XCD * p.per_xcd)), block(64 * KW);
    if (xbf) {
        if (ybf) hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, true, true, false>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, true, false, false>), grid, block, 0, st, e0, e1, 0, p);
    } else if (p.g) {
        if (ybf) hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, false, true, true>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, false, false, true>), grid, block, 0, st, e0, e1, 0, p);
    } else {
        if (ybf) hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, false, true, false>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_kw<MT, NT, KW, false, false, false>), grid, block, 0, st, e0, e1, 0, p);
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

/* cfg as in smol_gemm_tile (gemm.hip) */
extern "C" int smol_launch_gemm_kw(const GemmParams *p, int cfg, bool xbf, bool ybf, hipStream_t st, hipEvent_t e0,
                                   hipEvent_t e1) {
    switch (cfg) {
    case 3: return launch_kw<4, 4, 8>(*p, xbf, ybf, st, e0, e1);
    case 4: return launch_kw<4, 4, 4>(*p, xbf, ybf, st, e0, e1);
    case 5: return launch_kw<2, 4, 8>(*p, xbf, ybf, st, e0, e1);
    case 6: return launch_kw<2, 2, 4>(*p, xbf, ybf, st, e0, e1);
    case 7: return launch_kw<1, 2, 8>(*p, xbf, ybf, st, e0, e1);
    case 8: return launch_kw<1, 1, 8>(*p, xbf, ybf, st, e0, e1);
    default: return -1;
    }
}
