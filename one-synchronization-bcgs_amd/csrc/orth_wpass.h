// The FP64 fused pass for block widths 17 to 32 and slabs of up to 512
// columns: double-buffered tiles streamed straight into LDS.
//
// What bounds it: the FP64 MFMA work.  At 512 columns a tile of 16 rows takes
// 512 MFMA of 64 cycles each for step 1 and for the projection, 16400 cycles
// of a CU, against 7700 cycles of HBM time for its 64 KB.  The projection's
// accumulators (512 x 64) and the coefficients of step 1 (512 x 64) would
// fill the CU's register file by themselves, so each wave keeps its first UR
// units (16 columns) of coefficients in registers and reads the others from
// L2 in every tile, one unit behind each register unit; 8 waves with 256
// registers per CU above 256 columns, two workgroups of 4 waves below, where
// each covers the other's barriers and triangular solve.
//
// Tiles, loads and the LDS layout are the tile pass's (orth_tpass.h).  A wave
// owns one 16-column tile of Z (16 zn) for ZI 16-row chunks, over one of KS
// slices of the inner dimension.  A group's 32 columns are two Z tiles; the
// wave of the first one (slice 0) collects both, subtracts them and runs the
// blocked triangular solve (8 blocks of 4 columns, one MFMA per block and
// tile), while the other waves issue the next tile's loads and start on the
// part of the projection that no group takes part in.  Z and the solve are
// transposed, as in the tile pass.
//
// 2^22 x 512, s = 32, P-1S: 112 ms, 110 of them in 20 passes (F = 4 m n^2 at
// 39 TFLOP/s), where separate projection and update kernels took 178.
#pragma once

#include "orth_tpass.h"

namespace orth {

constexpr int kWpN1 = kWpassN1;   // columns of Z: two groups of 32
constexpr int kWpMaxCols4 = 256;  // columns of a buffer of the 4-wave form

// NW waves, TS rows, ZN used 16-column tiles of Z (2: one group, 4: two).
template <int NW, int TS, int ZN>
struct WpZ {
    static constexpr int ZT = TS / 16 * ZN;
    static constexpr int ZI = ZT > NW ? ZT / NW : 1;  // 16-row chunks per wave, ST apart
    static constexpr int ST = NW / ZN;
    static constexpr int KS = ZT < NW ? NW / ZT : 1;
    static constexpr int MaxU = (NW == 8 ? kWpassMaxCols : kWpMaxCols4 * 16 / TS) / 16;
    static constexpr int UQ = (MaxU + KS - 1) / KS;  // units per wave
    static constexpr int UR = UQ > 8 ? 2 : UQ;       // of them in registers
    // Partial Z tiles in LDS: every slice's but the collecting waves' own.
    static constexpr int Zs = KS > 1 ? ((KS - 1) * ZN + ZN / 2) * 256 : 0;
    static_assert(KS == 1 || TS == 16, "partial Z tiles are indexed by zn");
};

template <int NW, int TS, int NB, int ZN, int MT, bool SEQ>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_wpass(
    PassArgs a)
{
    using ZP = WpZ<NW, TS, ZN>;
    constexpr int kD = 64 * NW, N1 = kWpN1, ZI = ZP::ZI, ST = ZP::ST, KS = ZP::KS, UR = ZP::UR,
                  US = ZP::UQ - ZP::UR;
    static_assert(!SEQ || ZN == 4, "the sequential form has two groups");
    static_assert(NB == 2 || NB == 4, "N-tiles");
    extern __shared__ double sm[];
    const uint64_t kst = kernarg_stash();
    const int tid = threadIdx.x, lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tsz = a.wl * TS;
    double *const zs = sm + 2 * tsz;
    double *const wf = zs + ZP::Zs, *const sfl = wf + 1024;

    // Padding columns [ncols, wl) of both buffers are never loaded: zero.
    for (int e = tid; e < (a.wl - a.ncols) * TS; e += kD) {
        sm[a.ncols * TS + e] = 0.0;
        sm[tsz + a.ncols * TS + e] = 0.0;
    }

    // This wave's Z tile and its group.
    const int item = wave % ZP::ZT, ksp = wave / ZP::ZT;
    const int zn = item % ZN, zm0 = item / ZN, gi = zn >> 1, half = zn & 1;
    const int gw = gi < a.ngrp ? ORTH_G(a, min(gi, 1), w) : 0;
    const int gt = gi < a.ngrp ? ORTH_G(a, min(gi, 1), t0) : 0;
    const double *const gT = gi < a.ngrp ? ORTH_G(a, min(gi, 1), T) : nullptr;
    const bool zany = 16 * half < gw;
    const int zc = 16 * zn + li;
    const int cfin = SEQ ? a.g[0].t0 : 0;  // first finished column of the sequential form
    const int k1 = SEQ ? min(cfin, a.k1) : a.k1;
    // Units [ulo, ulo + nun) of 16 columns.  The slice that holds the last
    // unit, which may reach past k1, takes it first, from column addresses
    // clamped below k1 (zero coefficients).
    const int nu = zany ? (k1 + 15) >> 4 : 0;
    const int ulo = nu * ksp / KS, nun = nu * (ksp + 1) / KS - ulo;
    const int uf = ulo + nun == nu ? nu - 1 : ulo;  // the first unit taken
    const int ur = uf == ulo ? ulo + 1 : ulo;       // start of the others
    double cf[UR][4];
#pragma unroll
    for (int u = 0; u < UR; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = 16 * (u == 0 ? uf : ur + u - 1) + 4 * v + lk;
            cf[u][v] = u < nun && k < k1 ? a.C[wpass_cidx(k, zc)] : 0.0;
        }
    const int kc = 16 * uf + 16 > k1 ? k1 - 1 : 1 << 20;  // column clamp of unit uf
    // Units UR .. nun - 1 are whole ones, from L2: the first at row ks0 of C.
    const int nst = max(nun - UR, 0);
    const int ks0 = 16 * (ur + UR - 1);

    // Solve operands: the row blocks of each group's factor, in LDS (the
    // second group of the sequential form has no factor).
    const bool solver = ksp == 0 && half == 0 && gw > 0;
    for (int g = 0; g < (SEQ ? 1 : min(a.ngrp, ZN / 2)); g++) {
        const double *T = ORTH_G(a, g, T);
        if (T)
            for (int e = tid; e < 1024; e += kD) wf[1024 * g + e] = T[kSlotW + e];
    }
    // Good columns of this wave's group: those before a bad pivot.
    int gx = gw;
    if (gT && solver) {
        const int c = lane & (kLdT - 1);
        const uint32_t bad = (uint32_t)__ballot(
            c < gw && is_nan(gT[kSlotW + slot_last(c, gw) * kLdT + c]));
        if (bad) gx = __builtin_ctz(bad);
    }
    // Sequential form: the second group's coefficients on the first group's
    // columns.
    if constexpr (SEQ) {
        const int w0 = a.g[0].w, w1 = a.ngrp > 1 ? a.g[1].w : 0;
        for (int e = tid; e < 32 * 32; e += kD) {
            const int k = e >> 5, c = e & 31;
            sfl[e] = k < w0 && c < w1 ? a.C[wpass_cidx(cfin + k, 32 + c)] : 0.0;
        }
    }
    // Make the compiler wait for these loads here, once.
#pragma unroll
    for (int u = 0; u < UR; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) asm volatile("" ::"v"(cf[u][v]));

    // Projection: M-tiles m0 + NW i, all NB N-tiles; the waves on the solving
    // waves' SIMDs (the even ones), then those themselves, get the last ones.
    const int Ma = (a.na + 15) >> 4;
    const int m0 = wave & 1 ? wave >> 1 : NW / 2 + (NW == 8 ? (wave >> 1) ^ 2 : wave >> 1);
    const bool proj = a.na > 0 && m0 < Ma;
    // The N-tiles end with the buffer where they would leave it.
    const int b0 = a.b0 - a.bsh;
    const int pab = tpos<TS>(a.a0 + 16 * m0 + li, lk), pbb = tpos<TS>(b0 + li, lk);
    dbl4 acc[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NB; t++) acc[i][t] = dbl4{0.0, 0.0, 0.0, 0.0};
    const bool hasg = a.ngrp > 0;
    // The next tile's loads are issued at the tile's start when no solve or
    // no projection follows; otherwise after step 1 (whose L2 reads would wait
    // behind them), kEB before each M-tile during the solve and kFB before each
    // after it: a CU takes about 9 bytes per cycle, and a wave that finds the
    // path full stands still.  2^22 x 512, kEB / kFB: 1/1 116.2 ms, 1/2 118.1,
    // 2/1 123.5, 3/0 121.1, 0/1 and the rest at the end 129.0.
    const bool late = hasg && a.na > 0;
    constexpr int kEB = 1, kFB = 1;
    // M-tiles (bit i) whose product with the N-tiles from 2 on touches no
    // group's columns: the waves that do not solve take it during the solve.
    auto clean = [&](int c0, int c1) {
        bool r = true;
        for (int g = 0; g < a.ngrp; g++) {
            const int t0 = ORTH_G(a, g, t0), t1 = t0 + ORTH_G(a, g, w);
            r = r && (c1 <= t0 || c0 >= t1);
        }
        return r;
    };
    int early = 0;
    if (NB == 4 && hasg && proj && !solver && clean(b0 + 32, b0 + 64)) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int c0 = a.a0 + 16 * (m0 + NW * i);
            if (m0 + NW * i < Ma && clean(c0, c0 + 16)) early |= 1 << i;
        }
    }
    early = __builtin_amdgcn_readfirstlane(early);
    // One slice: are columns of a group's second Z tile step-1 operands (the
    // folded form's second group multiplies the first group's columns)?  Then
    // a barrier separates step 1 from the subtraction in place (a slot in LDS
    // does not fit beside two full buffers and two groups' solve operands).
    bool hand = false;
    if (KS == 1)
        for (int g = 0; g < a.ngrp; g++)
            hand = hand || (ORTH_G(a, g, w) > 16 && ORTH_G(a, g, t0) + 16 < k1);

    const int64_t rb = (int64_t)blockIdx.x * a.rows_per;
    const int64_t re = min(a.m, rb + a.rows_per);
    const int nt = re > rb ? (int)((re - rb + TS - 1) / TS) : 0;
    const int nfull = re > rb ? (int)((re - rb) / TS) : 0;

    // Loads (as in the tile pass): span i covers 64 consecutive 16-byte slots,
    // CS columns; the spans go round the waves.
    constexpr int CS = 128 / TS;
    const bool st16 = a.ldX % 2 == 0 && (uintptr_t)a.X % 16 == 0;
    const int nspan = (a.ncols + CS - 1) / CS;
    const int nsp = nspan > wave ? (nspan - wave + NW - 1) / NW : 0;  // this wave's spans
    const int ldc = CS * wave + lane / (TS / 2), ls = lane & (TS / 2 - 1);
    const char *gb = (const char *)(a.X + rb + (int64_t)ldc * a.ldX);
    const int64_t gs = (int64_t)CS * NW * a.ldX * 8;
    const int ncols = a.ncols;
    // This wave's spans [j0, j1) of tile t into buf.
    auto issue = [&](int t, double *buf, int j0, int j1) {
        if (t >= nfull) return;
        j1 = min(j1, nsp);
        if (st16) {
            const char *g = gb + (int64_t)t * (TS * 8) + j0 * gs;
            int c = ldc + j0 * CS * NW, i = wave + j0 * NW;
            for (int j = j0; j < j1; j++, g += gs, c += CS * NW, i += NW)
                if (c < ncols)
                    __builtin_amdgcn_global_load_lds((tp_glb_t *)(g + 16 * (ls ^ tswz<TS>(c))),
                                                     (tp_lds_t *)(buf + i * 128), 16, 0, 0);
        } else {
            const int ln = tp_opaque(lane);
            const double *Xr = a.X + rb + (int64_t)t * TS;
            for (int j = j0; j < j1; j++)
                for (int q = 0; q < 4; q++) {
                    const int i = wave + j * NW;
                    const int e = 16 * q + (ln >> 2), s = e & (TS / 2 - 1);
                    const int c = i * CS + e / (TS / 2);
                    if (c < ncols)
                        __builtin_amdgcn_global_load_lds(
                            (tp_glb_t *)((const float *)(Xr + 2 * (s ^ tswz<TS>(c)) +
                                                         (int64_t)c * a.ldX) + (ln & 3)),
                            (tp_lds_t *)(buf + i * 128 + 32 * q), 4, 0, 0);
                }
        }
    };
    issue(0, sm, 0, nsp);

    for (int t = 0; t < nt; t++) {
        double *cur = sm + (t & 1) * tsz;
        double *nxt = sm + ((t + 1) & 1) * tsz;
        // Tile t has landed, and every wave is done with the other buffer.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int lq = tp_opaque(lane), liq = lq & 15, lkq = lq >> 4;
        if (t >= nfull) {
            // The matrix's last rows: element by element, zeros past them.
            const int64_t r0 = rb + (int64_t)t * TS;
            for (int e = tp_opaque(tid); e < ncols * TS; e += kD) {
                const int c = e / TS, r = e % TS;
                cur[tpos<TS>(c, r)] = r0 + r < re ? a.X[r0 + r + (int64_t)c * a.ldX] : 0.0;
            }
            tp_barrier();
        }
        if (!late) issue(t + 1, nxt, 0, nsp);

        // Step 2, M-tile i of this wave with N-tiles [q0, q0 + 2).
        const int pa = tp_opaque(pab), pb = tp_opaque(pbb);
        auto project = [&](dbl4 *c, int i, int q0) {
#pragma unroll
            for (int ks = 0; ks < TS / 4; ks++) {
                const int o = 32 * (ks >> 3);
                const double av = cur[(pa ^ (4 * (ks & 7))) + o + 16 * TS * NW * i];
#pragma unroll
                for (int q = q0; q < q0 + 2; q++)
                    c[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        av, cur[(pb ^ (4 * (ks & 7))) + o + 16 * TS * q], c[q], 0, 0, 0);
            }
        };

        if (hasg) {
            dbl4 z[ZI];
#pragma unroll
            for (int i = 0; i < ZI; i++) z[i] = dbl4{0.0, 0.0, 0.0, 0.0};
            // Streamed coefficients: the next pair of units in flight during a
            // pair's products (past the last unit the loads repeat it).
            const uint32_t cl = 32 * lq;
            double c0[4], c1[4], c2[4], c3[4];
            auto cload = [&](double (&c)[4], int u) {
                // Wave-uniform base, 32-bit lane offset.
                const int k = ks0 + 16 * min(u, nst - 1);
                const char *cu = (const char *)(a.C + k * N1 + 256 * zn) + cl;
                const dbl2t x = ((const dbl2t *)cu)[0], y = ((const dbl2t *)cu)[1];
                c[0] = x.x, c[1] = x.y, c[2] = y.x, c[3] = y.y;
            };
            if (US > 0 && nst > 0) {
                cload(c0, 0);
                cload(c1, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            // B operand of a k-step: row 16 zm + li of its column lk.
            auto mma = [&](const double (&av)[ZI][4], const double (&cv)[4]) {
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int i = 0; i < ZI; i++)
                        z[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(cv[v], av[i][v], z[i], 0, 0, 0);
            };
            // The upper half of the waves would finish last, alone on its SIMDs
            // (the older wave goes first); this way round measured 0.5 % less.
            if (NW == 8 && wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
            if (nun > 0) {
                double av[ZI][4];
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int i = 0; i < ZI; i++)
                        av[i][v] = cur[tpos<TS>(min(16 * uf + 4 * v + lkq, kc), 16 * (zm0 + ST * i) + liq)];
                const int zq = tpos<TS>(16 * ur + lkq, 16 * zm0 + liq);
                auto load = [&](double (&d)[ZI][4], int o) {
#pragma unroll
                    for (int v = 0; v < 4; v++)
#pragma unroll
                        for (int i = 0; i < ZI; i++)
                            d[i][v] = cur[(zq ^ (4 * v) ^ (16 * ST * i)) + 4 * v * TS + o];
                };
                if constexpr (US > 0) {
                    // Operands one unit ahead (past the last unit: it again).
                    static_assert(UR == 2, "two register units before the streamed ones");
                    const int om = 16 * TS * max(nun - 2, 0);
                    double aw[ZI][4];
                    load(aw, 0);
                    mma(av, cf[0]);
                    load(av, min(16 * TS, om));
                    if (nun > 1) mma(aw, cf[1]);
                    int o = 16 * TS;
#pragma unroll 1
                    for (int u = 0; u < nst; u += 4, o += 64 * TS) {
                        cload(c2, u + 2);
                        cload(c3, u + 3);
                        load(aw, min(o + 16 * TS, om));
                        __builtin_amdgcn_sched_barrier(0);
                        mma(av, c0);
                        load(av, min(o + 32 * TS, om));
                        __builtin_amdgcn_sched_barrier(0);
                        if (u + 1 < nst) mma(aw, c1);
                        cload(c0, u + 4);
                        cload(c1, u + 5);
                        load(aw, min(o + 48 * TS, om));
                        __builtin_amdgcn_sched_barrier(0);
                        if (u + 2 < nst) mma(av, c2);
                        load(av, min(o + 64 * TS, om));
                        __builtin_amdgcn_sched_barrier(0);
                        if (u + 3 < nst) mma(aw, c3);
                    }
                } else {
                    mma(av, cf[0]);
#pragma unroll
                    for (int u = 1; u < UR; u++)
                        if (u < nun) {
                            load(av, 16 * TS * (u - 1));
                            if (ZI == 1) __builtin_amdgcn_sched_barrier(0);
                            mma(av, cf[u]);
                        }
                }
            }
            if (NW == 8) __builtin_amdgcn_s_setprio(0);
            // Hand the Z tiles to the collecting waves: partials through LDS,
            // or (one slice) a group's second tile by subtracting it in place,
            // after every wave's last read of those columns (hand).
            if (KS == 1 && hand) tp_barrier();
            if constexpr (KS > 1) {
                if (ksp > 0 || half == 1) {
                    const int slot = ksp > 0 ? (ksp - 1) * ZN + zn : (KS - 1) * ZN + gi;
#pragma unroll
                    for (int v = 0; v < 4; v++) zs[slot * 256 + v * 64 + lq] = z[0][v];
                }
            } else if (half == 1) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int c = 16 + 4 * v + lkq;
                    const int xi = tpos<TS>(gt + c, 16 * zm0 + liq);
#pragma unroll
                    for (int i = 0; i < ZI; i++)
                        if (c < gw) cur[xi ^ (16 * ST * i)] -= z[i][v];
                }
            }
            tp_barrier();
            if (solver) {
                __builtin_amdgcn_s_setprio(3);
                // Chunk zm of the group, transposed (lane: row li, columns
                // lk + 4 v), which is the accumulator layout of Z^T and makes
                // value b the B operand of block b of the blocked solve: the
                // chain of a solve is its MFMAs alone.
                dbl4 x0[ZI], x1[ZI];
                int xi[8];
#pragma unroll
                for (int v = 0; v < 8; v++)
                    xi[v] = tpos<TS>(gt + min(4 * v + lkq, gw - 1), 16 * zm0 + liq);
#pragma unroll
                for (int i = 0; i < ZI; i++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        x0[i][v] = cur[xi[v] ^ (16 * ST * i)];
                        x1[i][v] = cur[xi[4 + v] ^ (16 * ST * i)];
                    }
                    if constexpr (KS > 1) {
                        dbl4 y;
#pragma unroll
                        for (int v = 0; v < 4; v++) y[v] = zs[((KS - 1) * ZN + gi) * 256 + v * 64 + lq];
#pragma unroll
                        for (int k = 1; k < KS; k++)
#pragma unroll
                            for (int v = 0; v < 4; v++) {
                                z[i][v] += zs[((k - 1) * ZN + zn) * 256 + v * 64 + lq];
                                y[v] += zs[((k - 1) * ZN + zn + 1) * 256 + v * 64 + lq];
                            }
#pragma unroll
                        for (int v = 0; v < 4; v++) x1[i][v] -= y[v];
                    }
#pragma unroll
                    for (int v = 0; v < 4; v++) x0[i][v] -= z[i][v];
                }
                if constexpr (SEQ) {
                    if (gi == 1) {
                        // Wait for the first group, subtract its product.
                        tp_barrier();
#pragma unroll
                        for (int i = 0; i < ZI; i++) {
                            dbl4 y0 = dbl4{0.0, 0.0, 0.0, 0.0}, y1 = y0;
#pragma unroll
                            for (int b = 0; b < 8; b++) {
                                const double av =
                                    cur[tpos<TS>(cfin + min(4 * b + lkq, a.g[0].w - 1),
                                                 16 * (zm0 + ST * i) + liq)];
                                const double *s = sfl + 32 * (4 * b + lkq) + liq;
                                y0 = __builtin_amdgcn_mfma_f64_16x16x4f64(s[0], av, y0, 0, 0, 0);
                                y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(s[16], av, y1, 0, 0, 0);
                            }
#pragma unroll
                            for (int v = 0; v < 4; v++) {
                                x0[i][v] -= y0[v];
                                x1[i][v] -= y1[v];
                            }
                        }
                    }
                }
                // Columns past the good ones: zero, with zero rows of W.
#pragma unroll
                for (int i = 0; i < ZI; i++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        if (4 * v + lkq >= gx) x0[i][v] = 0.0;
                        if (16 + 4 * v + lkq >= gx) x1[i][v] = 0.0;
                    }
                if (gT) {
                    // (Rows of W past the group are zero.)
                    const double *W = wf + 1024 * gi + 32 * lkq + liq;
                    double w0[4], w1[8];
#pragma unroll
                    for (int b = 0; b < 8; b++) {
                        if (b < 4) w0[b] = W[128 * b];
                        w1[b] = W[128 * b + 16];
                    }
#pragma unroll
                    for (int b = 0; b < 8; b++)
#pragma unroll
                        for (int i = 0; i < ZI; i++) {
                            const double x = b < 4 ? x0[i][b & 3] : x1[i][b & 3];
                            if (b < 4) {
                                x0[i][b & 3] = 0.0;
                                x0[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(w0[b & 3], x, x0[i],
                                                                             0, 0, 0);
                            } else {
                                x1[i][b & 3] = 0.0;
                            }
                            x1[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(w1[b], x, x1[i], 0, 0, 0);
                        }
                }
#pragma unroll
                for (int i = 0; i < ZI; i++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        if (4 * v + lkq < gw) cur[xi[v] ^ (16 * ST * i)] = x0[i][v];
                        if (16 + 4 * v + lkq < gw) cur[xi[4 + v] ^ (16 * ST * i)] = x1[i][v];
                    }
                __builtin_amdgcn_s_setprio(0);
                // (Every wave meets this barrier once, the second group's
                // solver before its subtraction.)
                if (SEQ && gi == 0) tp_barrier();
            } else if (SEQ) {
                tp_barrier();
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                if (late) issue(t + 1, nxt, kEB * i, kEB * (i + 1));
                if (NB == 4 && (early >> i & 1)) project(acc[i], i, NB - 2);
            }
            tp_barrier();
            // The updated groups back to X: TS / 2 row pairs of a column by
            // consecutive threads.
            const int tq = tp_opaque(tid);
#pragma unroll
            for (int e0 = 0; e0 < 16 * ZN * (TS / 2); e0 += kD) {
                const int e = e0 + tq, col = e / (TS / 2), sq = e % (TS / 2);
                const int g = col >> 5, off = col & 31;
                if (e < 16 * ZN * (TS / 2) && g < a.ngrp && off < ORTH_G(a, g, w)) {
                    const int c = ORTH_G(a, g, t0) + off;
                    const dbl2t d = *(const dbl2t *)(cur + c * TS + 2 * (sq ^ tswz<TS>(c)));
                    const int64_t r = (int64_t)t * TS + 2 * sq;
                    double *gp = a.X + rb + r + (int64_t)c * a.ldX;
                    if (t < nfull && st16) {
                        __builtin_nontemporal_store(d, (dbl2t *)gp);
                    } else {
                        const int64_t left = re - rb - r;
                        if (left > 0) __builtin_nontemporal_store(d.x, gp);
                        if (left > 1) __builtin_nontemporal_store(d.y, gp + 1);
                    }
                }
            }
        }

        if (a.na > 0) {
#pragma unroll
            for (int i = 0; i < MT; i++) {
                if (late) issue(t + 1, nxt, kEB * MT + kFB * i, i + 1 < MT ? kEB * MT + kFB * (i + 1) : nsp);
                if (m0 + NW * i < Ma) project(acc[i], i, 0);
                if (NB == 4 && m0 + NW * i < Ma && !(early >> i & 1)) project(acc[i], i, NB - 2);
            }
        }
    }

    if (proj) {
        double *out = a.part + (int64_t)blockIdx.x * a.na * a.nb;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int q = 0; q < NB; q++) {
                const int col = q * 16 + li - a.bsh;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int row = (m0 + NW * i) * 16 + lk + 4 * v;
                    if (row < a.na && col >= 0 && col < a.nb) out[row + (int64_t)col * a.na] = acc[i][q][v];
                }
            }
    }
    pass_tail(a, sm, kst, kD);
}

}  // namespace orth
