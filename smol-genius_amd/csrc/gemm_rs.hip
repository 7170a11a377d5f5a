/*
 * gemm_rs.hip - k_gemm_rs: k_gemm's product (gemm.hip: the same operands and
 * fused operations) for an fp32 x on 192 x 192 tiles, the large prompts.
 *
 * What bounds them is the matrix cores: W.x_hi + W.x_lo of 1536 rows, 1024 ->
 * 6144, is 38.7 GFLOP, 33 us at the 1.17 PFLOP/s that a large bf16 product
 * reaches here. k_gemm holds an fp32 x in LDS as loaded, so both waves that
 * share a fragment read 32 bytes an element pair more and split it again, in
 * the way of their MFMAs. Here the stages come through registers and are split
 * once, on the way into LDS, by the thread that loaded them: 51.2 -> 47.5 us
 * there, 180 -> 162 us for 2048 -> 12288. (The norm's squares in eight parts a
 * row take 46.4 and 159 us, but leave the scale other last bits than the other
 * tiles' four.) (128 x 128 and a bf16 x gain nothing: 25.3 / 25.4 us, bf16
 * 192 x 192 37.2 / 39.9; k_gemm's direct transfers stay there. A third LDS stage, with the next step's
 * fragments read during the products, spilled registers: 58 us.)
 */
#include "gemm_device.h"

#define GEMM_BK 64

template <int BM, int BN, int WN, int WM, bool YBF, bool NORM>
__global__ __launch_bounds__(64 * WN * WM) __attribute__((amdgpu_waves_per_eu(WN * WM / 4, WN * WM / 4)))
void k_gemm_rs(const GemmParams p) {
    constexpr int NW = WN * WM, TPB = 64 * NW;
    constexpr int TN = BN / WN, TM = BM / WM, NT = TN / 16, MT = TM / 16; /* wave tile */
    constexpr int ROWB = GEMM_BK * 2; /* bytes of an LDS row: 64 bf16 */
    constexpr int XH = BN * ROWB, XLO = XH + BM * ROWB;
    constexpr int STAGE = XLO + BM * ROWB; /* W, x hi, x lo of one step */
    constexpr int WL = BN * 8 / TPB, XL = BM * 8 / TPB; /* 16-byte bf16 chunks a thread stages of W and x */
    static_assert(2 * STAGE <= 160 * 1024 - 1024, "LDS");
    static_assert(WL * TPB == BN * 8 && XL * TPB == BM * 8, "staging shape");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * STAGE];
    __shared__ float s_rinv[NORM ? BM : 1];

    int tm, tn;
    if (!gemm_tile_of(p, blockIdx.x, tm, tn)) return;
    const int m0 = tm * BM, K = p.K;
    const GemmOut out = gemm_out_of(p, tn * BN);
    const int n0 = out.n0, NN = out.n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int c = lane & 15, j = lane >> 4;

    /* thread: chunk lq (8 elements) of rows lr + TPB / 8 e. Rows past the
     * operands read zero by the buffer's range; the step's offset goes in
     * the scalar offset, which the range check leaves out */
    constexpr int xes = 4;
    const rsrc_t rw = make_rsrc(out.w + (long long)n0 * K, (long long)min(BN, NN - n0) * K * 2);
    const rsrc_t rx = make_rsrc(static_cast<const char *>(p.x) + (long long)m0 * K * xes,
                                (long long)min(BM, p.M - m0) * K * xes);
    const rsrc_t rg = make_rsrc(NORM ? (const void *)p.g : (const void *)out.w, NORM ? (long long)K * 4 : 0);
    const int lr = tid >> 3, lq = tid & 7;
    unsigned w_off[WL], x_off[XL], g_off = (unsigned)(32 * lq);
#pragma unroll
    for (int e = 0; e < WL; e++) w_off[e] = (unsigned)(((lr + TPB / 8 * e) * K + 8 * lq) * 2);
#pragma unroll
    for (int e = 0; e < XL; e++) x_off[e] = (unsigned)(((lr + TPB / 8 * e) * K + 8 * lq) * xes);
    /* every row a thread stages has the same low 3 bits (TPB / 8 is a
     * multiple of 8), so one swizzled position serves them all */
    const unsigned pos = (unsigned)(lr * ROWB + ((lq ^ (lr & 7)) << 4));
    static_assert(TPB / 8 % 8 == 0, "one swizzle per thread");

    struct Raw {
        uint4 w[WL], x[XL][2], g[NORM ? 2 : 1];
    };
    const int n_steps = (K + GEMM_BK - 1) / GEMM_BK;
    auto issue = [&](int s, Raw &r) __attribute__((always_inline)) {
        const int k0 = s * GEMM_BK;
        if (k0 + GEMM_BK > K && k0 + 8 * lq >= K) {
            /* K's end inside the step, or a step past it: these lanes load zeros from here on */
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
            r.x[e][1] = bload(rx, x_off[e] + 16u, (unsigned)(k0 * xes));
        }
#pragma unroll
        for (int e = 0; e < WL; e++) r.w[e] = bload(rw, w_off[e], (unsigned)(k0 * 2));
    };
    float ss[XL];
#pragma unroll
    for (int e = 0; e < XL; e++) ss[e] = 0.0f;
    auto store = [&](const Raw &r, unsigned char *st) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < WL; e++) *reinterpret_cast<uint4 *>(st + pos + TPB / 8 * e * ROWB) = r.w[e];
#pragma unroll
        for (int e = 0; e < XL; e++) {
            unsigned char *const xp = st + XH + pos + TPB / 8 * e * ROWB;
            const uint4 u = r.x[e][0], w = r.x[e][1];
            float v[8] = {__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w),
                          __uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w)};
            if constexpr (NORM) {
                ss[e] = gemm_squares64(v, ss[e]);
                const uint4 g0 = r.g[0], g1 = r.g[1];
                const uint32_t g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
                for (int b = 0; b < 8; b++) v[b] *= __uint_as_float(g[b]);
            }
            b8 h, l;
            split_frag(v, h, l);
            *reinterpret_cast<b8 *>(xp) = h;
            *reinterpret_cast<b8 *>(xp + (XLO - XH)) = l;
        }
    };

    f4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = f4{0.f, 0.f, 0.f, 0.f};
    auto frag = [&](const unsigned char *base, int row, int ks) __attribute__((always_inline)) {
        return as_b8(*reinterpret_cast<const uint4 *>(base + row * ROWB + (((4 * ks + j) ^ (row & 7)) << 4)));
    };
    auto multiply = [&](const unsigned char *st, int ks) __attribute__((always_inline)) {
        b8 a[NT], h[MT], l[MT];
#pragma unroll
        for (int t = 0; t < NT; t++) a[t] = frag(st, wn * TN + 16 * t + c, ks);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            h[mt] = frag(st + XH, wm * TM + 16 * mt + c, ks);
            l[mt] = frag(st + XLO, wm * TM + 16 * mt + c, ks);
        }
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], h[mt], acc[t][mt], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], l[mt], acc[t][mt], 0, 0, 0);
    };

    /* Step s multiplies LDS stage s % 2 while stage s + 1 is written from
     * registers (loaded two steps before) and step s + 3 is loaded into the
     * same registers. The one barrier a step orders the writes of a stage
     * before its reads and its reads before the next writes. Steps past the
     * end load and write zeros. */
    Raw raw[2];
    issue(0, raw[0]);
    issue(1, raw[1]);
    store(raw[0], smem);
    issue(2, raw[0]);
    __syncthreads();
    for (int s0 = 0; s0 < n_steps; s0 += 2)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int s = s0 + u;
            if (s >= n_steps) break;
            const unsigned char *st = smem + u * STAGE;
            store(raw[1 - u], smem + (1 - u) * STAGE);
            issue(s + 3, raw[1 - u]);
            multiply(st, 0);
            multiply(st, 1);
            __syncthreads();
        }

    /* the rows' scale */
    if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < XL; e++) {
            const float t = gemm_squares64_sum(ss[e]);
            if (lq == 0) s_rinv[lr + TPB / 8 * e] = 1.0f / sqrtf(t / (float)K + p.eps);
        }
        __syncthreads();
    }

    /* epilogue: lane (c, j) holds outputs n = 4 j + e of row m = c of each
     * 16 x 16 product tile */
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int ml = wm * TM + 16 * mt + c;
        const int m = m0 + ml;
        if (m >= p.M) continue;
        const float r = NORM ? s_rinv[ml] : 1.0f;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int n = n0 + wn * TN + 16 * t + 4 * j;
            if (n >= NN) continue;
            float v[4] = {acc[t][mt][0], acc[t][mt][1], acc[t][mt][2], acc[t][mt][3]};
            gemm_store4<YBF, NORM>(p, out.y, m, n, NN, v, r);
        }
    }
}

extern "C" int smol_launch_gemm_rs(const GemmParams *p, bool ybf, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const dim3 grid((unsigned)(GEMM_XCD * p->per_xcd)), block(512);
    if (p->g) {
        if (ybf) hipExtLaunchKernelGGL((k_gemm_rs<192, 192, 2, 4, true, true>), grid, block, 0, st, e0, e1, 0, *p);
        else hipExtLaunchKernelGGL((k_gemm_rs<192, 192, 2, 4, false, true>), grid, block, 0, st, e0, e1, 0, *p);
    } else {
        if (ybf) hipExtLaunchKernelGGL((k_gemm_rs<192, 192, 2, 4, true, false>), grid, block, 0, st, e0, e1, 0, *p);
        else hipExtLaunchKernelGGL((k_gemm_rs<192, 192, 2, 4, false, false>), grid, block, 0, st, e0, e1, 0, *p);
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}
