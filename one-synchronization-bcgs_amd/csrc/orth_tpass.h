// The FP64 fused pass for block widths up to 16: double-buffered tiles of TS
// rows streamed straight into LDS, 512 threads, two workgroups per CU.
//
// What bounds it: on wide slabs the FP64 MFMA work (at 256 columns 31 MFMA of
// 64 cycles per wave and 16 rows, 3970 cycles per CU, against 4500 cycles of
// HBM time for the tile), on narrow ones HBM; what a pass loses beside that
// are the phases in which a workgroup cannot multiply: the opening of a tile,
// the triangular solve (a serial chain in a few waves) and the barriers.  Two
// independent workgroups per CU cover each other's, so a tile takes as few
// rows as that needs: TS wl <= 4096 doubles per buffer.
//
// Right after the barrier that opens tile i the waves issue
// global_load_lds_dwordx4 for tile i+1 into the other buffer.  Vector-memory
// loads complete in issue order and share one counter, so the tile body
// issues no other load: the step-1 coefficient fragments and the
// triangular-solve operands are held in registers for the whole pass, and
// the only vector-memory wait is the one that opens a tile.
//
// LDS layout of a buffer (see tpos): column c at c * TS doubles, its 16-byte
// slots (row pairs) permuted by XOR with swz(c), so that an operand read by
// itself spreads over all 64 banks: 16 columns x 2 rows (projection) and 16
// rows x 2 columns (step 1).  Measured in conflict cycles per LDS cycle: none
// in 16-row tiles with one N-tile, 0 to 14 % in 128-row ones, 23 to 39 % with
// two N-tiles, whose operands sit on the same banks as each other.  No
// padding: a load instruction moves 64 slots of data.
//
// Per tile: step 1 (Z = tile(:, 0:k1) C, 16 x 16 tiles of Z over the waves,
// the inner dimension split KS ways when there are fewer tiles than waves);
// the wave that sums a Z tile subtracts it from the columns of the groups
// that own its 16 columns (two groups of at most 8 columns share one tile,
// ZN = 1) and runs their blocked triangular solve on MFMA (one MFMA per
// 4-column block with the row blocks [D_b | -D_b T] beside the factor), at
// raised priority.  Z and the solve are transposed, so that a block's columns
// are the next MFMA's operand as they stand; through LDS, at equal priority,
// 2^20 x 256 (s = 16, A-1S) took 9.38 ms instead of 9.16, 2^24 x 256 135.6
// instead of 130.4 (with a 13 ms copy).  The
// groups go back to X; step 2 accumulates tile(:, a0:a0+na)^T
// tile(:, b0:b0+nb), M-tile m by wave NW - 1 - m (mod NW), away from the
// solving waves.
#pragma once

#include "orth_device.h"
#include "orth_tail.h"

namespace orth {

constexpr int kTpBuf = 4096;      // doubles per tile buffer with more than 16 rows

// Step-1 split for TS rows and ZN 16-column tiles of Z.  The inner dimension
// goes to the waves in units of 16 columns; WIDE: slabs of more than 256.
template <int NW, int TS, int ZN, bool WIDE>
struct TpZ {
    static constexpr int ZT = TS / 16 * ZN;                 // Z tiles
    static constexpr int ZI = ZT > NW ? ZT / NW : 1;        // tiles per wave
    static constexpr int KS = ZT < NW ? NW / ZT : 1;        // inner-dimension split
    static constexpr int MaxU =
        (WIDE ? kTpassMaxCols : NW == 16 || TS == 16 ? 256 : kTpBuf / TS) / 16;
    static constexpr int UQ = (MaxU + KS - 1) / KS;  // units per wave
    static constexpr int Zs = (KS - 1) * ZT * 256;   // doubles of partial Z tiles
};

template <int TS>
__device__ __forceinline__ int tswz(int c)
{
    return ((c >> 1) & 7) | (TS > 16 ? (c & 1) << 3 : 0);
}

// Index (in doubles) of row r of column c in a buffer.
template <int TS>
__device__ __forceinline__ int tpos(int c, int r)
{
    return c * TS + (((r >> 1) ^ tswz<TS>(c)) << 1) + (r & 1);
}

typedef __attribute__((address_space(3))) void tp_lds_t;
typedef __attribute__((address_space(1))) const void tp_glb_t;
typedef double dbl2t __attribute__((ext_vector_type(2)));
typedef float flt4t __attribute__((ext_vector_type(4)));

// A copy of v the optimizer cannot see through, so that addresses derived
// from it inside the row loop are not hoisted into registers.
__device__ __forceinline__ int tp_opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Workgroup barrier over LDS that leaves vector-memory operations in flight
// (__syncthreads() would wait for the next tile's loads).
__device__ __forceinline__ void tp_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Orders the wave's own LDS accesses for the compiler (the hardware executes
// them in order).
__device__ __forceinline__ void tp_wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// SEQ: the second group's product uses the first group's finished columns:
// step 1 ends before them, and the second group subtracts their product after
// the first group's solve.
// NW waves: 8 (two workgroups per CU) or 16 (one).  WIDE: over 256 columns.
// MIX: the mixed form with FP64 products.  Columns from raw0 on (at most 32,
// never step-1 operands) have not been written yet and come from the FP32
// input: a thread loads four rows of a column into registers beside the next
// tile's LDS loads and widens them into the tile when it opens.
template <int NW, int TS, int NB, int ZN, int MT, bool WIDE, bool SEQ, bool MIX = false>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_tpass(
    PassArgs a)
{
    using ZP = TpZ<NW, TS, ZN, WIDE>;
    constexpr int kD = 64 * NW, N1 = 16 * ZN, ZT = ZP::ZT, ZI = ZP::ZI, KS = ZP::KS,
                  UQ = ZP::UQ;
    extern __shared__ double sm[];
    const uint64_t kst = kernarg_stash();
    const int tid = threadIdx.x, lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tsz = a.wl * TS;
    double *const zs = sm + 2 * tsz;

    // Padding columns [ncols, wl) of both buffers are never loaded: zero.
    for (int e = tid; e < (a.wl - a.ncols) * TS; e += kD) {
        sm[a.ncols * TS + e] = 0.0;
        sm[tsz + a.ncols * TS + e] = 0.0;
    }

    // Step-1 items of this wave: Z tiles (zm = zm0 + NW / ZN i, zn) over the
    // units [ulo, uhi) of the inner dimension.  The slice that holds the last
    // unit, which may reach past k1, takes it first, from per-lane column
    // addresses clamped below k1 (zero coefficients); the other units sit at
    // compile-time offsets.
    const int item = wave % ZT, ksp = wave / ZT;
    const int zn = item % ZN, zm0 = item / ZN;
    const bool zany = ztile_used(a, zn);
    const int cfin = SEQ ? a.g[0].t0 : 0;  // first finished column of the sequential form
    const int k1 = SEQ ? min(a.k1, cfin) : a.k1;
    const int nu = zany ? (k1 + 15) >> 4 : 0;
    const int ulo = nu * ksp / KS, nun = nu * (ksp + 1) / KS - ulo;
    const int uf = ulo + nun == nu ? nu - 1 : ulo;  // the first unit taken
    const int ur = uf == ulo ? ulo + 1 : ulo;       // start of the others
    // This lane's Z column as an operand row, and its group (lv: any).
    const int zc = 16 * zn + li;
    const int gl = a.ngrp == 2 && zc >= a.g[1].zoff ? 1 : 0;
    const int goff = zc - ORTH_G(a, gl, zoff);
    const bool lv = gl < a.ngrp && goff >= 0 && goff < ORTH_G(a, gl, w);
    double cf[UQ][4];
#pragma unroll
    for (int u = 0; u < UQ; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = 16 * (u == 0 ? uf : ur + u - 1) + 4 * v + lk;
            cf[u][v] = u < nun && k < k1 ? a.C[k * N1 + zc] : 0.0;
        }
    // Index of k-step 0 of units uf and ur; k-step v is this XOR 4 v, plus
    // 4 v TS.
    const int zf = tpos<TS>(16 * uf + lk, 16 * zm0 + li);
    const int zr = tpos<TS>(16 * ur + lk, 16 * zm0 + li);
    const int kc = 16 * uf + 16 > k1 ? k1 - 1 : 1 << 20;  // column clamp of unit uf
    // The Z tile is computed transposed (lane: row li of the chunk, columns
    // lk + 4 v), so that value v of the chunk is the operand of block v of the
    // blocked solve.  xi: the index of column lk + 4 v, or -1 past its group.
    // Solve operands, held for the pass: A fragments (lane: column li, row
    // lk) of the row blocks of the four 4-column blocks, each of one group;
    // zero in the other group's lanes.  smask: blocks to solve, group 0 in
    // bits 0-3, group 1 in bits 4-7.
    const bool solver = ksp == 0 && zany;
    double bw[4];
    int xi[4], smask = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int zb = 16 * zn + 4 * b;
        const int gb = a.ngrp == 2 && zb >= a.g[1].zoff ? 1 : 0;
        const int ob = zb - ORTH_G(a, gb, zoff), gw = gb < a.ngrp ? ORTH_G(a, gb, w) : 0;
        const double *T = ob < gw ? ORTH_G(a, gb, T) : nullptr;
        if (T) smask |= 1 << (b + 4 * gb);
        bw[b] = T && gl == gb && goff >= 0 ? T[kSlotW + 32 * ob + lk * kLdT + goff] : 0.0;
        xi[b] = ob + lk < gw ? tpos<TS>(ORTH_G(a, gb, t0) + ob + lk, 16 * zm0 + li) : -1;
    }
    // Sequential form: the second group's coefficients on the first group's
    // columns, row k at sfl + 16 k (lane: its Z column).
    double *const sfl = zs + ZP::Zs;
    if constexpr (SEQ) {
        if (solver && zm0 == 0 && 16 * zn + 16 > a.g[1].zoff) {
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int k = 4 * b + lk;
                sfl[16 * k + li] = lv && gl == 1 && k < a.g[0].w ? a.C[(cfin + k) * N1 + zc] : 0.0;
            }
        }
    }
    // Z columns past a bad pivot, which the solve must not see: bits 8 to 23 of
    // smask (one scalar for both: the kernel has none to spare).
    const bool badl = is_nan(bw[0]) || is_nan(bw[1]) || is_nan(bw[2]) || is_nan(bw[3]);
    smask |= ((int)__ballot(badl) & 0xffff) << 8;
    smask = __builtin_amdgcn_readfirstlane(smask);
    const int gsplit = a.ngrp == 2 ? a.g[1].zoff / 4 - 4 * zn : 4;  // first block of group 1
    // Make the compiler wait for these loads here, once.
#pragma unroll
    for (int u = 0; u < UQ; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) asm volatile("" ::"v"(cf[u][v]));
#pragma unroll
    for (int b = 0; b < 4; b++) asm volatile("" ::"v"(bw[b]));

    // Projection: M-tiles m0 + NW i, all NB N-tiles.  Operand of k-step ks:
    // row 4 ks + lk, i.e. the base index XOR 4 (ks & 7), plus 32 (ks >> 3).
    const int Ma = (a.na + 15) >> 4, m0 = NW - 1 - wave;
    const bool proj = a.na > 0 && m0 < Ma;
    const int pab = tpos<TS>(a.a0 + 16 * m0 + li, lk), pbb = tpos<TS>(a.b0 - a.bsh + li, lk);
    dbl4 acc[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NB; t++) acc[i][t] = dbl4{0.0, 0.0, 0.0, 0.0};

    const int64_t rb = (int64_t)blockIdx.x * a.rows_per;
    const int64_t re = min(a.m, rb + a.rows_per);
    const int nt = re > rb ? (int)((re - rb + TS - 1) / TS) : 0;
    // Tiles [0, nfull) end inside the matrix; at most the last one does not.
    const int nfull = re > rb ? (int)((re - rb) / TS) : 0;

    // Loads: span i covers 64 consecutive 16-byte slots of the buffer
    // (128 / TS columns); the spans go round the waves.  The lane's address
    // of span wave + NW j is gb + j gs; the swizzle repeats every 16 columns,
    // so only at TS = 128 (NW j columns apart) the odd j differ, by gx.  A
    // slab without 16-byte aligned row pairs (odd leading dimension or base)
    // moves four bytes per lane, a span in four loads.
    constexpr int CS = 128 / TS;  // columns per span
    const bool st16 = a.ldX % 2 == 0 && (uintptr_t)a.X % 16 == 0;
    const int nspan = ((MIX ? min(a.ncols, a.raw0) : a.ncols) + CS - 1) / CS;
    const int lc0 = CS * wave + lane / (TS / 2), ls = lane & (TS / 2 - 1);
    const char *gb = (const char *)(a.X + rb + (int64_t)lc0 * a.ldX + 2 * (ls ^ tswz<TS>(lc0)));
    const int gx = TS == 128 ? 16 * ((ls ^ tswz<TS>(lc0 + NW)) - (ls ^ tswz<TS>(lc0))) : 0;
    const int64_t gs = (int64_t)CS * NW * a.ldX * 8;
    const int ncols = MIX ? min(a.ncols, a.raw0) : a.ncols;  // columns loaded into LDS
    auto issue = [&](int t, double *buf) {
        if (t >= nfull) return;
        const char *g = gb + (int64_t)t * (TS * 8);
        if (st16) {
            int c = lc0;
            for (int i = wave, j = 0; i < nspan; i += NW, j++, g += gs, c += CS * NW)
                if (c < ncols)
                    __builtin_amdgcn_global_load_lds(
                        (tp_glb_t *)(TS == 128 && (j & 1) ? g + gx : g),
                        (tp_lds_t *)(buf + i * 128), 16, 0, 0);
        } else {
            const int ln = tp_opaque(lane);
            const double *Xr = a.X + rb + (int64_t)t * TS;
            for (int i = wave; i < nspan; i += NW)
                for (int q = 0; q < 4; q++) {
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
    // Raw columns: chunk e = tid + kD q is rows 4 (e % (TS / 4)) .. + 3 of
    // column ncols + e / (TS / 4); one 16-byte load where the input allows it.
    constexpr int NRV = 8 * TS > kD ? 8 * TS / kD : 1;
    const int nraw = a.ncols - ncols;
    const bool rv4 = MIX && a.ldX32 % 4 == 0 && (uintptr_t)a.X32 % 16 == 0;
    flt4t rv[MIX ? NRV : 1];
    auto raw_load = [&](int t) {
        if constexpr (MIX) {
            if (t >= nfull) return;
#pragma unroll
            for (int q = 0; q < NRV; q++) {
                const int e = tp_opaque(tid) + kD * q, c = e / (TS / 4);
                if (c >= nraw) continue;
                const float *p = a.X32 + rb + (int64_t)t * TS + 4 * (e % (TS / 4)) +
                                 (int64_t)(ncols + c) * a.ldX32;
                if (rv4) {
                    rv[q] = __builtin_nontemporal_load((const flt4t *)p);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++) rv[q][k] = __builtin_nontemporal_load(p + k);
                }
            }
        }
    };
    auto raw_store = [&](double *buf) {
        if constexpr (MIX) {
#pragma unroll
            for (int q = 0; q < NRV; q++) {
                const int e = tp_opaque(tid) + kD * q, c = e / (TS / 4), r = 4 * (e % (TS / 4));
                if (c >= nraw) continue;
                *(dbl2t *)(buf + tpos<TS>(ncols + c, r)) = dbl2t{(double)rv[q][0], (double)rv[q][1]};
                *(dbl2t *)(buf + tpos<TS>(ncols + c, r + 2)) = dbl2t{(double)rv[q][2], (double)rv[q][3]};
            }
        }
    };
    raw_load(0);
    issue(0, sm);

    // Write-back: LP threads per column, row pairs sq + LP i.
    constexpr int LP = TS / 2 < 16 ? TS / 2 : 16;
    const int sg = tid / (16 * LP), sc = (tid / LP) % 16, sq = tid % LP;
    const bool sv = sg < a.ngrp && sc < ORTH_G(a, min(sg, 1), w);
    const int scol = sv ? ORTH_G(a, min(sg, 1), t0) + sc : 0;
    const int sidx = scol * TS + 2 * (sq ^ tswz<TS>(scol));
    double *sp = a.X + rb + 2 * sq + (int64_t)scol * a.ldX;
    const bool hasg = a.ngrp > 0;
    constexpr int SN = TS / 2 / LP;  // store instructions per thread and full tile
    const bool wst = __builtin_amdgcn_readfirstlane((int)(__ballot(sv) != 0)) && st16;
    // The next tile's loads are issued at the tile's start by the waves that
    // solve in it (and by all when no solve or no projection follows), else
    // while the groups are solved.
    const bool late = hasg && a.na > 0 && !solver;

    for (int t = 0; t < nt; t++, sp += TS) {
        double *cur = sm + (t & 1) * tsz;
        double *nxt = sm + ((t + 1) & 1) * tsz;
        // Tile t has landed (every wave waits for its own loads; the barrier
        // makes all of them visible), and every wave is done with the other
        // buffer.  Memory operations complete in issue order, so a wave that
        // stored in the previous tile, after issuing these loads, leaves its
        // SN stores in flight: their acknowledgement takes longer than the
        // projection.
        if (t > 0 && wst)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(SN) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int lq = tp_opaque(lane), liq = lq & 15;
        if (MIX && t < nfull) raw_store(cur);
        if (t >= nfull) {
            // The matrix's last rows: element by element, zeros past them.
            const int64_t r0 = rb + (int64_t)t * TS;
            for (int e = tp_opaque(tid); e < a.ncols * TS; e += kD) {
                const int c = e / TS, r = e % TS;
                double x = 0.0;
                if (r0 + r < re)
                    x = MIX && c >= ncols ? (double)a.X32[r0 + r + (int64_t)c * a.ldX32]
                                          : a.X[r0 + r + (int64_t)c * a.ldX];
                cur[tpos<TS>(c, r)] = x;
            }
            tp_barrier();
        } else if (MIX && !hasg) {
            tp_barrier();  // (with groups the raw columns' readers wait in step 1)
        }
        if (MIX) raw_load(t + 1);
        if (!late) issue(t + 1, nxt);

        if (hasg) {
            dbl4 z[ZI];
#pragma unroll
            for (int i = 0; i < ZI; i++) z[i] = dbl4{0.0, 0.0, 0.0, 0.0};
            // B operand of a k-step: row 16 zm + li of its column lk.
            auto unit = [&](int u, const double *const (&p)[4], int o) {
                double av[ZI][4];
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int i = 0; i < ZI; i++)
                        av[i][v] = p[v][o + 16 * (NW / ZN) * i];
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int i = 0; i < ZI; i++)
                        z[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(cf[u][v], av[i][v], z[i], 0, 0,
                                                                   0);
            };
            if (nun > 0) {
                if (kc < 1 << 20) {
                    const double *p[4];
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        p[v] = cur + tpos<TS>(min(16 * uf + 4 * v + (lq >> 4), kc), 16 * zm0 + liq);
                    unit(0, p, 0);
                } else {
                    const int zq = tp_opaque(zf);
                    const double *const p[4] = {cur + zq, cur + (zq ^ 4) + 4 * TS,
                                                cur + (zq ^ 8) + 8 * TS, cur + (zq ^ 12) + 12 * TS};
                    unit(0, p, 0);
                }
                const int zq = tp_opaque(zr);
                const double *const p[4] = {cur + zq, cur + (zq ^ 4) + 4 * TS,
                                            cur + (zq ^ 8) + 8 * TS, cur + (zq ^ 12) + 12 * TS};
#pragma unroll
                for (int u = 1; u < UQ; u++)
                    if (u < nun) unit(u, p, 16 * TS * (u - 1));
            }
            if (KS > 1 && ksp > 0) {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    zs[((ksp - 1) * ZT + item) * 256 + v * 64 + lq] = z[0][v];
            }
            tp_barrier();
            if (late) issue(t + 1, nxt);
            // Chunk zm of the groups of tile zn, minus the fixed-order sum of
            // the partial Z tiles; then the blocked triangular solve, whose
            // chain is its MFMAs alone.
            auto blocks = [&](dbl4 &x, int mask) {
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    if (!(mask >> b & 1)) continue;
                    const dbl4 x0 = x;
                    x[b] = 0.0;
                    x = __builtin_amdgcn_mfma_f64_16x16x4f64(bw[b], x0[b], x, 0, 0, 0);
                    // Two groups in one tile: the other group's columns keep
                    // their values (0 times a NaN of this group is NaN).
                    if (ZN == 1) {
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            if ((v >= gsplit) != (b >= gsplit)) x[v] = x0[v];
                    }
                }
            };
            dbl4 x[ZI];
            auto contain = [&] {
                if (smask >> 8) {
#pragma unroll
                    for (int i = 0; i < ZI; i++)
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            if (smask >> (8 + 4 * v + (lq >> 4)) & 1) x[i][v] = 0.0;
                }
            };
            if (solver) {
                __builtin_amdgcn_s_setprio(3);
#pragma unroll
                for (int i = 0; i < ZI; i++) {
                    const int o = 16 * (NW / ZN) * i;
#pragma unroll
                    for (int v = 0; v < 4; v++) x[i][v] = xi[v] >= 0 ? cur[xi[v] + o] : 0.0;
#pragma unroll
                    for (int k = 1; k < KS; k++)
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            z[i][v] += zs[((k - 1) * ZT + item) * 256 + v * 64 + lq];
#pragma unroll
                    for (int v = 0; v < 4; v++) x[i][v] -= z[i][v];
                }
                contain();
#pragma unroll
                for (int i = 0; i < ZI; i++) {
                    const int o = 16 * (NW / ZN) * i;
                    blocks(x[i], SEQ ? smask & 15 : smask | smask >> 4);
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (xi[v] >= 0 && !(SEQ && v >= gsplit)) cur[xi[v] + o] = x[i][v];
                }
            }
            if (solver) __builtin_amdgcn_s_setprio(0);
            if constexpr (SEQ) {
                tp_barrier();
                if (solver && a.ngrp == 2 && 16 * zn + 16 > a.g[1].zoff) {
#pragma unroll
                    for (int i = 0; i < ZI; i++) {
                        const int o = 16 * (NW / ZN) * i;
                        dbl4 y = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int b = 0; b < 4; b++) {
                            const double av =
                                cur[tpos<TS>(cfin + min(4 * b + (lq >> 4), a.g[0].w - 1), 16 * zm0 + liq) + o];
                            const double sv = sfl[64 * b + lq];
                            y = __builtin_amdgcn_mfma_f64_16x16x4f64(sv, av, y, 0, 0, 0);
                        }
#pragma unroll
                        for (int v = 0; v < 4; v++) x[i][v] -= y[v];
                    }
                    contain();
#pragma unroll
                    for (int i = 0; i < ZI; i++) {
                        const int o = 16 * (NW / ZN) * i;
                        blocks(x[i], smask >> 4);
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            if (xi[v] >= 0 && v >= gsplit) cur[xi[v] + o] = x[i][v];
                    }
                }
            }
            tp_barrier();
            // The updated groups back to X.
            if (sv) {
#pragma unroll
                for (int i = 0; i < SN; i++) {
                    const dbl2t d = *(const dbl2t *)(cur + sidx + 2 * LP * i);
                    double *g = sp + 2 * LP * i;
                    if (t < nfull && st16) {
                        __builtin_nontemporal_store(d, (dbl2t *)g);
                    } else {
                        const int64_t left = re - rb - (int64_t)t * TS - 2 * (sq + LP * i);
                        if (left > 0) __builtin_nontemporal_store(d.x, g);
                        if (left > 1) __builtin_nontemporal_store(d.y, g + 1);
                    }
                }
            }
        }

        // Step 2: projection partial over this tile's rows.
        if (proj) {
            const int pa = tp_opaque(pab), pb = tp_opaque(pbb);
#pragma unroll
            for (int ks = 0; ks < TS / 4; ks++) {
                const double *ca = cur + (pa ^ (4 * (ks & 7))) + 32 * (ks >> 3);
                const double *cb = cur + (pb ^ (4 * (ks & 7))) + 32 * (ks >> 3);
                double bv[NB];
#pragma unroll
                for (int q = 0; q < NB; q++) bv[q] = cb[16 * TS * q];
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    if (i > 0 && m0 + NW * i >= Ma) continue;
                    const double av = ca[16 * TS * NW * i];
#pragma unroll
                    for (int q = 0; q < NB; q++)
                        acc[i][q] =
                            __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[q], acc[i][q], 0, 0, 0);
                }
                if ((ks & 1) == 1) __builtin_amdgcn_sched_barrier(0);
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
