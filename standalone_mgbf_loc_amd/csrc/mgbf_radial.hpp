// Radial 2-D beta filter kernel (template), instantiated per half-width H and
// kind of taps in mgbf_radial_inst.hip.
#pragma once

#include "mgbf_device.hpp"
#include "mgbf_launch.hpp"

namespace mgbf {

template <int H>
__host__ __device__ constexpr int disc_extent(int b) {
    int a = H;
    while (a >= 0 && a * a + b * b >= (H + 1) * (H + 1)) --a;
    return a;
}

typedef const __attribute__((address_space(4))) float* ConstF;
typedef const __attribute__((address_space(4))) int* ConstI;

// A buffer over 2 GiB from `base` (rows are below that size): accesses at
// kDropped and beyond are out of its range, which the hardware turns into
// loads of zero and no store.
constexpr int kDropped = (int)0x80000000;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc_2g(const float* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)0x80000000, 0x00020000);
}

// Row buffers of the input pipeline (one being combined, the others in
// flight): 4 where the registers of the ring and its epilogues leave room. A
// narrow filter has too little arithmetic a row to be worth them: memory bounds
// it on a large field, and more waves a SIMD use that better (the line procedure
// at half-width 3, 80 x 768 x 768 x 64: 16.4 ms with 1 buffer, 16.8 with 2, 17.5
// with 4 and the matrix cores beside; 1440 x 960 x 65 at half-width 1: 789, 798
// and 801 us).
// With the band beside 4 columns, the disc of half-width 10 has registers for one
// only (256 registers and one wave a SIMD with 2: 512 x 512 x 1024, whole
// application, 4.29 ms against 3.73).
__host__ __device__ constexpr int radial_bufs(int H, int TI, bool disc, int VHB) {
    if (H > 9 && TI == 4 && disc && VHB > 0) return 1;
    return H <= 3 ? 1 : H <= 6 ? 4 : (H <= 8 ? 3 : 2);
}

// One step per ring row S, S+1, .. NR-1 of a turn; the first step past the
// tile ends it (nested, so that no path rejoins another between two steps and
// the waits for the row buffers stay exact).
template <int S, int NR, class F>
__device__ __forceinline__ void radial_turn(F& step, int rb, int nsteps) {
    if constexpr (S < NR) {
        if (rb + S < nsteps) {
            step(rb + S, std::integral_constant<int, S>{});
            radial_turn<S + 1, NR>(step, rb, nsteps);
        }
    }
}

// ---------------------------------------------------------------------------
// Radial 2-D beta filter F (gather form, half-sample mirror halo) with the
// epilogue of its generation:
//   s(k,i,j) = scale(k,i,j) * sum_{a,b} w(|a|,|b|) in(k, mx(i+a), my(j+b))
//              [+ (P coarse)(k,i,j)]                       (PRO)
//   out(k,i,j) = sum_d c(L,d) s(k+d,i,j) over the column    (VHB > 0)
// scale = wfield (per point, not with PRO) or wconst. One wave computes
// TI x TJ outputs for each of its 64 lanes' k: input rows stream through
// registers; for every input row the x-pair sums P_a = v(i+a)+v(i-a) give the
// per-row partial sums Z_b = sum_a w(a,b) P_a, which are added to the output
// rows j = r-b and r+b held in a ring of accumulator rows.
// TAPS: the box of w(a,b), the lattice disc a^2 + b^2 < (H+1)^2 with
// w(a,b) = w(b,a) (one kernel argument each), or the product fx(a) fy(b) (one
// x-sum per row, fy(b) into rows r+-b).
// PRO adds the prolongation of the next coarser generation (direct1 on the
// 2-point mirrored coarse field): a window of 4 x-interpolated coarse rows
// slides down with the output rows, one new coarse row every other row.
// VHB applies a vertical band of half-width VHB across the lanes of the wave.
// RES restricts the input field to the next generation on the way (R = P^T
// with the folded edges): every loaded fine row is restricted in x over the
// tile's 2 coarse columns (interior columns 2I-3 .. 2I+4 with kW8, or
// 2I-2 .. 2I+3 with the quadratic weights under QP; the 2 columns at each
// domain edge with the edge table) and added into a shift register of the
// coarse rows whose windows are open (4 or 3 in the interior, up to 6 next
// to an edge, with weights from a per-fine-row table there); a coarse row
// is stored when its window closes. The wave owns coarse rows j0/2 ..
// (j0+TJ)/2 - 1, whose windows lie inside the rows it loads (checked on the
// host).
// QP selects the quadratic transfer (direct2 / adjoint2) for PRO or RES.
//
// Lanes. Where the stack's Kc = K - klo values fill their last 64-k chunk
// badly (radial_flattened), the values of all column tiles of a tile row are
// laid end to end and cut into waves of 64: lane l of wave w works on
// f = 64 w + l, k = klo + f % Kc of column tile f / Kc. K = 32 fills a wave
// with two tiles, K = 65 loses nothing where chunks of 64 lose half, and the
// 2 or 3 two-dimensional variables behind the 3-D ones take 32 or 21 tiles a
// wave. Column offsets, tile edges and mirrors are per lane (VGPRs) in either
// layout. The band takes stacks of whole 64-k chunks (with lm dividing 64 a
// wave then holds whole columns).
//
// Input rows are loaded NB - 1 steps ahead into NB register buffers (none ahead
// up to half-width 3, see radial_bufs): the VALU
// is what bounds this kernel (62 operations an output for the H = 6 disc), and
// with the loads in flight two waves a SIMD keep it busy: 89 % (with RES) and all
// of the time (PRO and the band) on 768 x 768 x 5120, 66 and 79 % in the one round
// of 384 x 384 x 320; at H = 8 on 1024 x 1024 x 127, 63 % (RES) and 79 % (PRO); at
// H = 1, where memory bounds it, 21 and 23 %. The ring has
// the next multiple of NB above 2H rows, so that ring row and buffer of a step
// are compile-time constants; the spare rows cost TI registers each.
// 512 x 512 x 1024 at H = 6: 0.54 ms plain, 0.60 with PRO, 0.70 with PRO and
// the band of half-width 6, 0.70 with RES (0.60, 0.72, 0.91 and 0.72 when rows
// were loaded as they were needed, at 3 to 5 waves a SIMD).
//
// Partial sums Z_b that reach no output row of the tile are left out: a tile
// of TJ rows reads TJ + 2H, and of the first and last 2H of them only some b
// are needed (all of them: 7/3 of the needed work at TJ = 4, H = 6). That
// makes the short tiles cheap that give a small grid enough waves.
// ---------------------------------------------------------------------------
enum { kTapsBox = 0, kTapsDisc = 1, kTapsSep = 2 };

template <int H, int TI, int TAPS, bool PRO, int VHB, bool RES, bool QP>
__global__ void __launch_bounds__(kBlock) radial_kernel(RadialParams p) {
    static_assert(!QP || PRO || (RES && VHB == 0), "the quadratic transfer rides in PRO or RES");
    static_assert(!RES || (TI == 4 && !PRO && VHB == 0), "restriction epilogue shape");
    constexpr bool DISC = TAPS == kTapsDisc;
    constexpr int NB = radial_bufs(H, TI, DISC, VHB);
    constexpr int NR = (2 * H + 1 + NB - 1) / NB * NB;
    // columns and rows loaded on each side: H for the filter, 4 columns and 3
    // rows for the restriction's 8-point stencils; the D extra rows feed the
    // restriction only
    constexpr int HL = (RES && H < 4) ? 4 : H;
    constexpr int HR = (RES && H < 3) ? 3 : H;
    constexpr int D = HR - H;
    constexpr int NC = TI + 2 * HL;
    constexpr int NCC = TI / 2 + 4;   // coarse columns of the tile (TI even)
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = (int)xcd_block(blockIdx.x, gridDim.x) * p.wpb + wv;
    if (item >= p.nitems) return;
    const int K = p.K, n = p.n, m = p.m;
    int tj, k, ti;
    bool valid = true;
    if (p.kc > 0) {   // the stack end to end over the column tiles
        const int w = item % p.nfw;
        tj = item / p.nfw;
        int f = w * kWave + lane;
        const int last = p.ntile_i * p.kc - 1;
        valid = f <= last;
        f = valid ? f : last;
        ti = f / p.kc;
        k = p.klo + f - ti * p.kc;
    } else {          // 64-k chunks: tiles fastest, chunks slowest
        ti = item % p.ntile_i;
        const int rest = item / p.ntile_i;
        tj = rest % p.ntile_j;
        k = p.klo + rest / p.ntile_j * kWave + lane;
        valid = k < K;
        k = valid ? k : K - 1;
    }
    const int i0 = ti * TI, j0 = tj * p.TJ;
    const size_t rowstride = (size_t)n * K;

    // byte offsets inside a row, per lane
    int voff[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) voff[c] = (mirror_half(i0 - HL + c, n) * K + k) * 4;
    // a lane past the last tile, and columns past the domain, store at an
    // offset past the buffer's end, which the hardware drops: a branch on a
    // lane's own condition would cost more than the offsets
    int vst[TI];
#pragma unroll
    for (int t = 0; t < TI; ++t) vst[t] = valid && i0 + t < n ? ((i0 + t) * K + k) * 4 : kDropped;

    float acc[NR][TI];
#pragma unroll
    for (int s = 0; s < NR; ++s)
#pragma unroll
        for (int t = 0; t < TI; ++t) acc[s][t] = 0.f;

    // prolongation window: 4 x-interpolated coarse rows, and the raw values
    // of the row that enters next, loaded one window step ahead
    float XV[4][TI];
    float cvn[NCC];
    int csoff[NCC];
    int cbase = 0;
    const int nc = n / 2, mc = m / 2;
    const size_t crow = (size_t)nc * K;
    auto load_craw = [&](int r, float* dst) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rc = buf_rsrc(p.coarse + (size_t)mirror_half(r, mc) * crow);
#pragma unroll
        for (int c = 0; c < NCC; ++c) dst[c] = buf_ld(rc, csoff[c], 0);
    };
    using PS = Stencil<QP>;
    auto wbase = [&](int j) { return QP ? (j >> 1) - 1 : ((j + 1) >> 1) - 2; };
    auto xinterp = [&](const float* cv, float* dst) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TI; ++t) {
            if constexpr (QP)
                dst[t] = PS::C[t & 1][0] * cv[t / 2 + 1] + PS::C[t & 1][1] * cv[t / 2 + 2] +
                         PS::C[t & 1][2] * cv[t / 2 + 3];
            else if ((t & 1) == 0)
                dst[t] = kQc[0] * cv[t / 2] + kQc[1] * cv[t / 2 + 1] + kQc[2] * cv[t / 2 + 2] +
                         kQc[3] * cv[t / 2 + 3];
            else
                dst[t] = kPc[0] * cv[(t + 1) / 2] + kPc[1] * cv[(t + 1) / 2 + 1] +
                         kPc[2] * cv[(t + 1) / 2 + 2] + kPc[3] * cv[(t + 1) / 2 + 3];
        }
    };
    if constexpr (PRO) {
#pragma unroll
        for (int c = 0; c < NCC; ++c) csoff[c] = (mirror_half(i0 / 2 - 2 + c, nc) * K + k) * 4;
        cbase = wbase(j0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            load_craw(cbase + u, cvn);
            xinterp(cvn, XV[u]);
        }
        load_craw(cbase + 4, cvn);
    }

    // vertical band coefficients of this lane's level (identity past nfilt)
    constexpr int NVB = VHB > 0 ? 2 * VHB + 1 : 1;
    float vc[NVB];
    if constexpr (VHB > 0) {
        if (k < p.nfilt) {
            const float* row = p.band + (k % p.lm) * NVB;
#pragma unroll
            for (int d = 0; d < NVB; ++d) vc[d] = row[d];
        } else {
#pragma unroll
            for (int d = 0; d < NVB; ++d) vc[d] = d == VHB ? 1.f : 0.f;
        }
#pragma unroll
        for (int d = 0; d < NVB; ++d) settle(vc[d]);
    }

    const int tj_eff = p.TJ < m - j0 ? p.TJ : m - j0;
    const int nsteps = tj_eff + 2 * HR;

    // fused restriction state; whether the tile lies at the low or the high
    // edge is per lane
    constexpr int NRC = RES ? TI / 2 : 1;
    constexpr int NQ = 6;
    float racc[NQ][NRC];
    const int Jlo = j0 / 2, Jhi = (j0 + tj_eff) / 2;
    const bool xlow = i0 == 0, xhigh = i0 + TI >= n;
    int vco[NRC];   // where the coarse columns are stored
    if constexpr (RES) {
#pragma unroll
        for (int c = 0; c < NRC; ++c)
            vco[c] = valid && i0 / 2 + c < nc ? ((i0 / 2 + c) * K + k) * 4 : kDropped;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int c = 0; c < NRC; ++c) racc[q][c] = 0.f;
    }
    auto store_coarse = [&](int J, const float* val) __attribute__((always_inline)) {
        if (J < Jlo || J >= Jhi) return;
        const __amdgpu_buffer_rsrc_t ro = buf_rsrc_2g(p.rout + (size_t)J * crow);
#pragma unroll
        for (int c = 0; c < NRC; ++c) buf_st(val[c], ro, vco[c], 0);
    };

    // what step rr needs from memory goes into buffer rr % NB: input row rr
    // and, with a weight field, the weights of the output row it completes.
    // Always issued (past the tile's end the last row again), so that the
    // number of loads behind the ones a step waits for is known.
    float vb[NB][NC];
    float wb[RES || !PRO ? NB : 1][TI];
    auto load_row = [&](int rr, float* v, float* w) __attribute__((always_inline)) {
        rr = rr < nsteps ? rr : nsteps - 1;
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(p.in + (size_t)mirror_half(j0 - HR + rr, m) * rowstride);
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = buf_ld(rs, voff[c], 0);
        if constexpr (!PRO) {
            if (p.wfield) {
                int jr = rr - D - 2 * H;
                jr = jr < 0 ? 0 : (jr < tj_eff ? jr : tj_eff - 1);
                const __amdgpu_buffer_rsrc_t rw = buf_rsrc_2g(p.wfield + (size_t)(j0 + jr) * rowstride);
#pragma unroll
                for (int t = 0; t < TI; ++t) w[t] = buf_ld(rw, vst[t], 0);   // a dropped column reads zero
            }
        }
    };
#pragma unroll
    for (int e = 0; e < NB - 1; ++e) load_row(e, vb[e], wb[PRO ? 0 : e]);

    auto step = [&](const int rr, auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        float* const v = vb[s % NB];
        load_row(rr + NB - 1, vb[(s + NB - 1) % NB], wb[PRO ? 0 : (s + NB - 1) % NB]);
        if constexpr (RES) {
            const int vr = j0 - HR + rr;   // fine row, before mirroring
            if (vr >= 0 && vr < m) {
                using RS = Stencil<QP>;
                float xr[NRC];
#pragma unroll
                for (int c = 0; c < NRC; ++c) {   // fine columns 2I+ROFF .. 2I+ROFF+NR-1
                    float a = 0.f;
#pragma unroll
                    for (int t = 0; t < RS::NR; ++t) a = __builtin_fmaf(RS::R[t], v[HL + RS::ROFF + 2 * c + t], a);
                    xr[c] = a;
                }
                if (__any(xlow || xhigh)) {   // fine columns 0 .. 7, n-8 .. n-1
#pragma unroll
                    for (int c = 0; c < NRC; ++c) {
                        float lo = 0.f, hi = 0.f;
#pragma unroll
                        for (int t = 0; t < 8; ++t) {
                            lo = __builtin_fmaf(QP ? kEdgeRWQ.w[c][t] : kEdgeRW.w[c][t], v[HL + t], lo);
                            hi = __builtin_fmaf(QP ? kEdgeRWQ.w[NRC - 1 - c][7 - t] : kEdgeRW.w[NRC - 1 - c][7 - t],
                                                v[HL - 4 + t], hi);
                        }
                        xr[c] = xlow ? lo : (xhigh ? hi : xr[c]);
                    }
                }
                // the row enters the open coarse rows: inside, NO of them,
                // with the stencil's odd or even taps, and a row of parity CP
                // closes the oldest; in the 8 rows next to an edge up to 6,
                // with weights and closing rows from the table (constant
                // address space: scalar loads, which leave the count of row
                // loads in flight alone)
                constexpr int NO = RS::NR / 2;
                constexpr int CP = (RS::ROFF + RS::NR - 1) & 1;
                const bool edge = vr < 8 || vr > m - 9;
                float yw[NQ];
                int J, nclose;
                if (edge) {
                    const ConstF ry = (ConstF)(size_t)p.rytab + 8 * vr;
                    const ConstI rm = (ConstI)(size_t)p.rymeta + 2 * vr;
#pragma unroll
                    for (int q = 0; q < NQ; ++q) yw[q] = ry[q];
                    J = rm[0];
                    nclose = rm[1];
                } else {
                    const bool closes = (vr & 1) == CP;
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                        yw[q] = q >= NO ? 0.f : (closes ? RS::R[RS::NR - 1 - 2 * (q % NO)] : RS::R[RS::NR - 2 - 2 * (q % NO)]);
                    J = (vr - RS::ROFF - RS::NR + 1) >> 1;
                    nclose = closes ? 1 : 0;
                }
#pragma unroll
                for (int q = 0; q < NO; ++q)
#pragma unroll
                    for (int c = 0; c < NRC; ++c) racc[q][c] = __builtin_fmaf(yw[q], xr[c], racc[q][c]);
                if (edge) {
#pragma unroll
                    for (int q = NO; q < NQ; ++q)
#pragma unroll
                        for (int c = 0; c < NRC; ++c) racc[q][c] = __builtin_fmaf(yw[q], xr[c], racc[q][c]);
                }
#pragma unroll 1
                for (; nclose > 0; --nclose, ++J) {
                    store_coarse(J, racc[0]);
#pragma unroll
                    for (int q = 0; q + 1 < NQ; ++q)
#pragma unroll
                        for (int c = 0; c < NRC; ++c) racc[q][c] = racc[q + 1][c];
#pragma unroll
                    for (int c = 0; c < NRC; ++c) racc[NQ - 1][c] = 0.f;
                }
            }
        }
        // filter row f, the centre of output row c = f - H: Z_b reaches output
        // rows c - b and c + b, one of which must lie in the tile
        const int f = rr - D;
        if (D > 0 && (f < 0 || f >= tj_eff + 2 * H)) return;
        const int ctr = f - H;
        const int blo = ctr < 0 ? -ctr : (ctr >= tj_eff ? ctr - tj_eff + 1 : 0);
        const int up = tj_eff - 1 - ctr;
        int bhi = ctr < 0 ? up : (ctr >= tj_eff ? ctr : (ctr > up ? ctr : up));
        bhi = bhi < H ? bhi : H;
        const unsigned need = (2u << bhi) - (1u << blo);   // bit b: Z_b is needed
        constexpr int sf = s + 2 * NR - D;   // ring row of f, modulo NR
        if constexpr (TAPS == kTapsSep) {
            // w(a,b) = fx(a) fy(b): one x-sum per row, fy(b) into rows f+-b
            float q[TI];
#pragma unroll
            for (int t = 0; t < TI; ++t) {
                q[t] = p.W.w[0][0] * v[t + HL];
#pragma unroll
                for (int a = 1; a <= H; ++a)
                    q[t] = __builtin_fmaf(p.W.w[0][a], v[t + HL + a] + v[t + HL - a], q[t]);
            }
#pragma unroll
            for (int b = 0; b <= H; ++b) {
                if (!(need >> b & 1)) continue;
#pragma unroll
                for (int t = 0; t < TI; ++t) {
                    acc[(sf + b) % NR][t] = __builtin_fmaf(p.W.w[1][b], q[t], acc[(sf + b) % NR][t]);
                    if (b > 0) acc[(sf - b) % NR][t] = __builtin_fmaf(p.W.w[1][b], q[t], acc[(sf - b) % NR][t]);
                }
            }
        } else {
            float P[TI][H + 1];
#pragma unroll
            for (int t = 0; t < TI; ++t) {
                P[t][0] = v[t + HL];
#pragma unroll
                for (int a = 1; a <= H; ++a) P[t][a] = v[t + HL + a] + v[t + HL - a];
            }
#pragma unroll
            for (int b = 0; b <= H; ++b) {
                if (!(need >> b & 1)) continue;
                const int A = DISC ? disc_extent<H>(b) : H;
#pragma unroll
                for (int t = 0; t < TI; ++t) {
                    // on the disc w(a,b) = w(b,a): one kernel argument each
                    float z = p.W.w[DISC ? 0 : b][DISC ? b : 0] * P[t][0];
#pragma unroll
                    for (int a = 1; a <= H; ++a)
                        if (a <= A)
                            z = __builtin_fmaf(p.W.w[DISC && a < b ? a : b][DISC && a < b ? b : a], P[t][a], z);
                    acc[(sf + b) % NR][t] += z;
                    if (b > 0) acc[(sf - b) % NR][t] += z;
                }
            }
        }
        // output row j = j0 + f - 2H is complete
        const int jrel = f - 2 * H;
        constexpr int os = (sf - H) % NR;
        if (jrel >= 0 && jrel < tj_eff) {
            const int j = j0 + jrel;
            float o[TI];
#pragma unroll
            for (int t = 0; t < TI; ++t) o[t] = (!PRO && p.wfield ? wb[PRO ? 0 : s % NB][t] : p.wconst) * acc[os][t];
            if constexpr (PRO) {
                const int nb = wbase(j);
                if (nb != cbase) {   // the window moves down one coarse row
#pragma unroll
                    for (int u = 0; u < 3; ++u)
#pragma unroll
                        for (int t = 0; t < TI; ++t) XV[u][t] = XV[u + 1][t];
                    xinterp(cvn, XV[3]);
                    load_craw(nb + 4, cvn);
                    cbase = nb;
                }
                const bool oj = (j & 1) != 0;
                constexpr int NP = PS::NP;
                float y[NP];
#pragma unroll
                for (int u = 0; u < NP; ++u) y[u] = oj ? PS::C[1][u] : PS::C[0][u];
#pragma unroll
                for (int t = 0; t < TI; ++t) {
                    if constexpr (QP)
                        o[t] += y[0] * XV[0][t] + y[1] * XV[1][t] + y[2] * XV[2][t];
                    else
                        o[t] += y[0] * XV[0][t] + y[1] * XV[1][t] + y[2] * XV[2][t] + y[NP - 1] * XV[3][t];
                }
            }
            if constexpr (VHB > 0) {
                // the band over the lanes: level k+d sits in lane lane+d,
                // reached by d single-lane wave shifts (DPP); lanes shifted in
                // from outside the wave read 0 and meet a zero band
                // coefficient, as do lanes of the neighbouring column
#pragma unroll
                for (int t = 0; t < TI; ++t) {
                    float lu = o[t], ld = o[t];
                    float rsum = vc[VHB] * o[t];
#pragma unroll
                    for (int d = 1; d <= VHB; ++d) {
                        lu = lane_from_above(lu);
                        ld = lane_from_below(ld);
                        rsum = __builtin_fmaf(vc[VHB + d], lu, rsum);
                        rsum = __builtin_fmaf(vc[VHB - d], ld, rsum);
                    }
                    o[t] = rsum;
                }
            }
            const __amdgpu_buffer_rsrc_t ro = buf_rsrc_2g(p.out + (size_t)j * rowstride);
#pragma unroll
            for (int t = 0; t < TI; ++t) buf_st(o[t], ro, vst[t], 0);
        }
#pragma unroll
        for (int t = 0; t < TI; ++t) acc[os][t] = 0.f;
    };
    for (int rb = 0; rb < nsteps; rb += NR) radial_turn<0, NR>(step, rb, nsteps);
}

template <int H, int TI, int TAPS, bool PRO, int VHB, bool RES, bool QP>
hipError_t launch_radial_variant(const RadialArgs& a, hipStream_t st) {
    RadialParams p{};
    p.in = a.in;
    p.out = a.out;
    p.wfield = a.wfield;
    p.wconst = a.wconst;
    p.coarse = a.coarse;
    p.band = a.band;
    p.K = a.K;
    p.klo = a.klo;
    p.n = a.n;
    p.m = a.m;
    p.TJ = a.TJ;
    p.lm = a.lm;
    p.nfilt = a.nfilt;
    p.W = a.coef;
    p.rout = a.rout;
    p.rytab = a.rytab;
    p.rymeta = a.rymeta;
    p.ntile_i = (a.n + TI - 1) / TI;
    p.ntile_j = (a.m + a.TJ - 1) / a.TJ;
    const int kc = a.K - a.klo;
    p.kc = radial_flattened(kc) ? kc : 0;
    const long long row = radial_row_waves(kc, a.n, TI);
    p.nfw = (int)row;
    const long long nitems = row * p.ntile_j;
    if (nitems >= (1ll << 31) || (long long)p.ntile_i * kc >= (1ll << 31)) return hipErrorInvalidValue;
    p.nitems = (int)nitems;
    // Few waves go out one a block, so that they reach all CUs: 288 of them, 2
    // values a column 1032 bytes apart, in 24 us against 37 on 72 CUs (1152:
    // 91 against 105; 1152 of 192 x 192 x 32 with the restriction: 21 against
    // 24). From 1872 waves on neighbours of a block share more than that
    // gains: 14.4 us against 13.5.
    p.wpb = nitems <= 1536 ? 1 : kWavesPerBlock;
    const unsigned nblocks = (unsigned)((nitems + p.wpb - 1) / p.wpb);
    hipLaunchKernelGGL((radial_kernel<H, TI, TAPS, PRO, VHB, RES, QP>), dim3(nblocks), dim3(p.wpb * kWave), 0, st, p);
    return hipGetLastError();
}

// The pass kinds; radial_built, checked here, lists what is built.
template <int H, int TI, int TAPS, int VHB>
hipError_t launch_radial_band(const RadialArgs& a, hipStream_t st) {
    if constexpr (TAPS != kTapsBox)
        return a.quad ? launch_radial_variant<H, TI, TAPS, true, VHB, false, true>(a, st)
                      : launch_radial_variant<H, TI, TAPS, true, VHB, false, false>(a, st);
    else
        return hipErrorInvalidValue;
}

template <int H, int TI, int TAPS>
hipError_t launch_radial_ti(const RadialArgs& a, hipStream_t st) {
    if (a.band) {
        switch (a.vhb) {
            case 3: return launch_radial_band<H, TI, TAPS, 3>(a, st);
            case 4: return launch_radial_band<H, TI, TAPS, 4>(a, st);
            case 6: return launch_radial_band<H, TI, TAPS, 6>(a, st);
            case 8: return launch_radial_band<H, TI, TAPS, 8>(a, st);
            default: return hipErrorInvalidValue;
        }
    }
    if (!a.coarse) return launch_radial_variant<H, TI, TAPS, false, 0, false, false>(a, st);
    return a.quad ? launch_radial_variant<H, TI, TAPS, true, 0, false, true>(a, st)
                  : launch_radial_variant<H, TI, TAPS, true, 0, false, false>(a, st);
}

// Passes of 4 columns a lane, and those with the restriction
template <int H, int TAPS>
hipError_t launch_radial_taps(const RadialArgs& a, hipStream_t st) {
    if (!radial_built(a) || a.TJ < 1 || (TAPS == kTapsDisc) != a.exact_disc || (TAPS == kTapsSep) != a.separable)
        return hipErrorInvalidValue;
    if (a.rout)
        return a.quad ? launch_radial_variant<H, 4, TAPS, false, 0, true, true>(a, st)
                      : launch_radial_variant<H, 4, TAPS, false, 0, true, false>(a, st);
    return launch_radial_ti<H, 4, TAPS>(a, st);
}

// Passes of 2 columns a lane
template <int H, int TAPS>
hipError_t launch_radial_taps2(const RadialArgs& a, hipStream_t st) {
    if (!radial_built(a) || a.rout || a.TJ < 1 || (TAPS == kTapsDisc) != a.exact_disc || (TAPS == kTapsSep) != a.separable)
        return hipErrorInvalidValue;
    return launch_radial_ti<H, 2, TAPS>(a, st);
}

}  // namespace mgbf
