/*
 * gemm_sw.hip - k_gemm_sw: k_gemm's product (gemm.hip: the same operands,
 * products and fused operations) for launches whose k_gemm tiles would leave
 * the device idle or waiting: a few to a few hundred rows.
 *
 * Every output's sum over K is formed by one wave in k_gemm's order (32-wide
 * steps ascending, an fp32 x its hi product before its lo one), and the norm's
 * sum of squares as k_gemm's lanes form it, so a row's results are the same
 * bits in every tile of gemm.hip, gemm_rs.hip and here, however many rows are
 * beside it. (K split over a workgroup's waves, their sums added at the end,
 * was about as fast, but tied a row's bits to the tile that the number of rows
 * chose, which a bf16 output's truncation then makes a whole bf16 step.)
 *
 * What bounds those launches is latency, not a rate: k_gemm stages each
 * 64-wide K step through LDS behind a barrier, so a step costs about a memory
 * round trip. Here a workgroup's waves have roles. SW waves stage: each slab of
 * KC columns of W and x comes as whole row pieces (16 bytes a lane,
 * neighbouring lanes along a row) into registers, DEPTH slabs ahead, an fp32
 * x is split (and scaled) there, and goes into one of two LDS stages. WN x WM
 * waves multiply the other stage meanwhile, and with the norm BM / 16 more sum
 * the rows' squares (in 64-wide slabs the staging threads: x as loaded in LDS
 * too makes 64 x 64 21.2 us of 20.2, 64 rows, 2048 -> 12288, and 96 of 77, 1536
 * rows, 1024 -> 6144). One barrier a slab. (With every wave doing both, the
 * multiplying waves' own staging delayed every slab: 26 fp32 rows, 6144 ->
 * 2048, 15.7 us.)
 *
 * Measured, weights not in L2, k_gemm's 64 x 64 tile / K split over the waves
 * / this kernel (us): 26 fp32 rows, 6144 -> 2048 49.5 / 12.5 / 13.2 (25 MB of
 * weights: 1.9 TB/s); 2048 -> 2048 18.1 / 6.2 / 6.5; 2048 -> 12288 with the norm
 * and SwiGLU 22.9 / 15.1 / 14.6 (50 MB: 3.4 TB/s); 333 bf16 rows, 3072 -> 1024
 * 24.4 / 12.6 / 12.8; 5 bf16 rows, 6144 -> 2048 44 / 9.4 / 11.2. Chunks
 * swizzled by four row bits where a row has 16 or more: 15% of the LDS cycles
 * were conflicts with three, and those tiles took 2 to 12% longer. The host
 * chooses by a fitted cost of each tile
 * (gemm_cfg, linear.hip); without k_gemm's own 64 x 64 tile that choice is
 * 0.03% worse on average over 484 products, so that tile is gone.
 */
#include "gemm_device.h"

/* waves that sum squares: none with 64-wide slabs, where the staging threads do */
constexpr int sw_square_waves(int bm, int kc, bool norm) { return norm && kc > 64 ? bm / 16 : 0; }

template <int BM, int BN, int WN, int WM, int SW, int KC, int DEPTH, bool XBF, bool YBF, bool NORM>
__global__ __launch_bounds__(64 * (SW + WN * WM + sw_square_waves(BM, KC, NORM))) void k_gemm_sw(const GemmParams p) {
    constexpr int TPB = 64 * SW, MW = WN * WM;
    constexpr int TN = BN / WN, TM = BM / WM, NT = TN / 16, MT = TM / 16; /* a multiplying wave's tile */
    constexpr int KS = KC / 32;   /* 32-wide steps of a slab */
    constexpr int CPR = KC / 8;   /* 16-byte bf16 chunks of a row of a slab */
    constexpr int ROWB = KC * 2;  /* bytes of an LDS row */
    constexpr int RS = TPB / CPR; /* rows between two chunks of a staging thread */
    constexpr int SWZ = CPR < 16 ? 7 : 15; /* row bits that swizzle a chunk: a fragment's rows then span every bank */
    /* a stage: W, x (hi), x lo, and for waves that sum squares x as loaded (the
     * first four values of each chunk, then the last four) */
    constexpr bool RAW = sw_square_waves(BM, KC, NORM) > 0;
    constexpr int XH = BN * ROWB, XLO = XH + BM * ROWB, XR = XLO + (XBF ? 0 : BM * ROWB);
    constexpr int STAGE = XR + (RAW ? 2 * BM * ROWB : 0);
    constexpr int WL = BN * CPR / TPB, XL = BM * CPR / TPB; /* chunks a thread stages of W and x */
    static_assert(2 * STAGE <= 160 * 1024, "LDS");
    static_assert(WL * TPB == BN * CPR && XL * TPB == BM * CPR, "staging shape");
    static_assert(RS % (SWZ + 1) == 0, "every row of a thread has one swizzle");
    static_assert(KS % 2 == 0, "fragments are read two steps at a time");
    static_assert(!(XBF && NORM), "the norm takes an fp32 x");
    static_assert(!NORM || RAW || KC == 64, "two 32-wide halves a slab");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * STAGE];
    float *const s_rinv = reinterpret_cast<float *>(smem); /* after the last slab */

    int tm, tn;
    if (!gemm_tile_of(p, blockIdx.x, tm, tn)) return;
    const int m0 = tm * BM, K = p.K;
    const GemmOut out = gemm_out_of(p, tn * BN);
    const int n0 = out.n0, NN = out.n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, j = lane >> 4;
    const int n_slabs = (K + KC - 1) / KC;

    /* One barrier a slab, in every role: it orders the writes of a stage before
     * its reads and its reads before the next writes. */
    if (wave < SW) {
        /* thread: chunk lq (8 elements) of rows lr + RS e. Rows past the
         * operands read zero by the buffer's range; the slab's offset goes in
         * the scalar offset, which the range check leaves out */
        constexpr int xes = XBF ? 2 : 4, XP = XBF ? 1 : 2;
        const rsrc_t rw = make_rsrc(out.w + (long long)n0 * K, (long long)min(BN, NN - n0) * K * 2);
        const rsrc_t rx = make_rsrc(static_cast<const char *>(p.x) + (long long)m0 * K * xes,
                                    (long long)min(BM, p.M - m0) * K * xes);
        const rsrc_t rg = make_rsrc(NORM ? (const void *)p.g : (const void *)out.w, NORM ? (long long)K * 4 : 0);
        const int lr = tid / CPR, lq = tid % CPR;
        unsigned w_off[WL], x_off[XL], g_off = (unsigned)(32 * lq);
#pragma unroll
        for (int e = 0; e < WL; e++) w_off[e] = (unsigned)(((lr + RS * e) * K + 8 * lq) * 2);
#pragma unroll
        for (int e = 0; e < XL; e++) x_off[e] = (unsigned)(((lr + RS * e) * K + 8 * lq) * xes);
        const unsigned pos = (unsigned)(lr * ROWB + ((lq ^ (lr & SWZ)) << 4));

        struct Raw {
            uint4 w[WL], x[XL][XP], g[NORM ? 2 : 1];
        };
        auto issue = [&](int s, Raw &r) __attribute__((always_inline)) {
            const int k0 = s * KC;
            if (k0 + KC > K && k0 + 8 * lq >= K) {
                /* K's end inside the slab, or a slab past it: these lanes load zeros from here on */
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
            for (int e = 0; e < XL; e++)
#pragma unroll
                for (int h = 0; h < XP; h++) r.x[e][h] = bload(rx, x_off[e] + 16u * h, (unsigned)(k0 * xes));
#pragma unroll
            for (int e = 0; e < WL; e++) r.w[e] = bload(rw, w_off[e], (unsigned)(k0 * 2));
        };
        float ss[XL];
#pragma unroll
        for (int e = 0; e < XL; e++) ss[e] = 0.0f;
        auto store = [&](const Raw &r, unsigned char *st) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < WL; e++) *reinterpret_cast<uint4 *>(st + pos + RS * e * ROWB) = r.w[e];
#pragma unroll
            for (int e = 0; e < XL; e++) {
                unsigned char *const xp = st + pos + RS * e * ROWB;
                if constexpr (XBF) {
                    *reinterpret_cast<uint4 *>(xp + XH) = r.x[e][0];
                } else {
                    const uint4 u = r.x[e][0], w = r.x[e][XP - 1];
                    float v[8] = {__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z),
                                  __uint_as_float(u.w), __uint_as_float(w.x), __uint_as_float(w.y),
                                  __uint_as_float(w.z), __uint_as_float(w.w)};
                    if constexpr (RAW) {
                        *reinterpret_cast<uint4 *>(xp + XR) = u;
                        *reinterpret_cast<uint4 *>(xp + XR + BM * ROWB) = w;
                    } else if constexpr (NORM) {
                        ss[e] = gemm_squares64(v, ss[e]);
                    }
                    if constexpr (NORM) {
                        const uint4 g0 = r.g[0], g1 = r.g[1];
                        const uint32_t g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
                        for (int b = 0; b < 8; b++) v[b] *= __uint_as_float(g[b]);
                    }
                    b8 h, l;
                    split_frag(v, h, l);
                    *reinterpret_cast<b8 *>(xp + XH) = h;
                    *reinterpret_cast<b8 *>(xp + XLO) = l;
                }
            }
        };
        /* slabs past the end load and write zeros */
        Raw raw[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH; d++) issue(d, raw[d]);
        store(raw[0], smem);
        issue(DEPTH, raw[0]);
        __syncthreads();
        constexpr int U = DEPTH % 2 == 0 ? DEPTH : 2 * DEPTH;
        for (int s0 = 0; s0 < n_slabs; s0 += U)
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (s0 + u >= n_slabs) break;
                store(raw[(u + 1) % DEPTH], smem + (1 - u % 2) * STAGE);
                issue(s0 + u + 1 + DEPTH, raw[(u + 1) % DEPTH]);
                __syncthreads();
            }
        if constexpr (NORM && !RAW) {
#pragma unroll
            for (int e = 0; e < XL; e++) {
                const float t = gemm_squares64_sum(ss[e]);
                if (lq == 0) s_rinv[lr + RS * e] = 1.0f / sqrtf(t / (float)K + p.eps);
            }
        }
        if constexpr (NORM) __syncthreads();
        return;
    }

    /* lane (c, j): chunk 4 ks + j of a row, step ks of the slab */
    auto frag = [&](const unsigned char *base, int row, int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<const uint4 *>(base + row * ROWB + (((4 * ks + j) ^ (row & SWZ)) << 4));
    };
    if (RAW && wave >= SW + MW) {
        const int row = 16 * (wave - SW - MW) + c;
        float t = 0.0f;
        __syncthreads();
        for (int s = 0; s < n_slabs; s++) {
            const unsigned char *st = smem + (s & 1) * STAGE + XR;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const uint4 u = frag(st, row, ks), w = frag(st + BM * ROWB, row, ks);
                const uint32_t v[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
                for (int b = 0; b < 8; b++) t = fmaf(__uint_as_float(v[b]), __uint_as_float(v[b]), t);
            }
            __syncthreads();
        }
        t = row_sum4(t);
        if (j == 0) s_rinv[row] = 1.0f / sqrtf(t / (float)K + p.eps);
        __syncthreads();
        return;
    }

    const int mw = wave - SW, wn = mw % WN, wm = mw / WN;
    f4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = f4{0.f, 0.f, 0.f, 0.f};
    struct Frag {
        b8 a[NT], h[MT], l[XBF ? 1 : MT];
    };
    auto read = [&](const unsigned char *st, int ks, Frag &f) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) f.a[t] = as_b8(frag(st, wn * TN + 16 * t + c, ks));
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            f.h[mt] = as_b8(frag(st + XH, wm * TM + 16 * mt + c, ks));
            if constexpr (!XBF) f.l[mt] = as_b8(frag(st + XLO, wm * TM + 16 * mt + c, ks));
        }
    };
    auto multiply = [&](const Frag &f) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[t], f.h[mt], acc[t][mt], 0, 0, 0);
        if constexpr (!XBF) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[t], f.l[mt], acc[t][mt], 0, 0, 0);
        }
    };
    __syncthreads();
    for (int s = 0; s < n_slabs; s++) {
        const unsigned char *st = smem + (s & 1) * STAGE;
        Frag f[2][2];
        read(st, 0, f[0][0]);
        read(st, 1, f[0][1]);
#pragma unroll
        for (int g = 0; g < KS / 2; g++) {
            if (g + 1 < KS / 2) {
                read(st, 2 * g + 2, f[(g + 1) & 1][0]);
                read(st, 2 * g + 3, f[(g + 1) & 1][1]);
            }
            __builtin_amdgcn_sched_barrier(0);
            multiply(f[g & 1][0]);
            multiply(f[g & 1][1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }
    if constexpr (NORM) __syncthreads(); /* the rows' scale */

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

/* ------------------------------------------------------------------ launch */

/* staging waves, slab width and depth for an fp32 x, with the norm, and for a bf16 x */
template <int BM, int BN, int WN, int WM, int SWF, int KF, int DF, int KN, int DN, int SWB, int KB, int DB>
static int launch_sw(const GemmParams &p, bool xbf, bool ybf, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const dim3 grid((unsigned)(GEMM_XCD * p.per_xcd));
    constexpr int MW = WN * WM;
    if (xbf) {
        const dim3 block(64 * (SWB + MW));
        if (ybf) hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWB, KB, DB, true, true, false>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWB, KB, DB, true, false, false>), grid, block, 0, st, e0, e1, 0, p);
    } else if (p.g) {
        const dim3 block(64 * (SWF + MW + sw_square_waves(BM, KN, true)));
        if (ybf) hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWF, KN, DN, false, true, true>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWF, KN, DN, false, false, true>), grid, block, 0, st, e0, e1, 0, p);
    } else {
        const dim3 block(64 * (SWF + MW));
        if (ybf) hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWF, KF, DF, false, true, false>), grid, block, 0, st, e0, e1, 0, p);
        else hipExtLaunchKernelGGL((k_gemm_sw<BM, BN, WN, WM, SWF, KF, DF, false, false, false>), grid, block, 0, st, e0, e1, 0, p);
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

/* cfg as in smol_gemm_tile (gemm.hip) */
extern "C" int smol_launch_gemm_sw(const GemmParams *p, int cfg, bool xbf, bool ybf, hipStream_t st, hipEvent_t e0,
                                   hipEvent_t e1) {
    switch (cfg) {
    case 2: return launch_sw<64, 64, 2, 2, 8, 64, 4, 64, 3, 4, 64, 3>(*p, xbf, ybf, st, e0, e1);
    case 3: return launch_sw<64, 128, 2, 2, 8, 64, 2, 64, 3, 8, 64, 3>(*p, xbf, ybf, st, e0, e1);
    case 4: return launch_sw<32, 64, 2, 2, 8, 128, 3, 128, 3, 8, 128, 3>(*p, xbf, ybf, st, e0, e1);
    case 5: return launch_sw<32, 32, 2, 2, 8, 256, 2, 128, 3, 8, 256, 2>(*p, xbf, ybf, st, e0, e1);
    case 6: return launch_sw<16, 32, 2, 1, 8, 256, 3, 256, 3, 8, 256, 3>(*p, xbf, ybf, st, e0, e1);
    case 7: return launch_sw<16, 16, 1, 1, 8, 256, 3, 256, 3, 8, 256, 3>(*p, xbf, ybf, st, e0, e1);
    default: return -1;
    }
}
