// HIP kernels of the MGBF operator for CDNA4 (gfx950): vertical band,
// restriction, prolongation, scaling and reductions; the radial filter kernel
// is in mgbf_radial.hpp (one translation unit per half-width).
//
// Field layout: k fastest, then x (i), then y (j); element (k,i,j) at
// k + K*(i + n*j). One wavefront (64 lanes) owns 64 consecutive k; every
// stage acts on each k independently except the vertical filter, which mixes
// levels of one column. Halo fills of the reference (boco_2d, half-sample
// mirror at the domain edge) become wave-uniform index remapping, so no
// padded copies are stored; adjoint folds are never formed because the
// radial filter is symmetric under that mirror (F^T = F) and the restriction
// uses precomputed transposed tables.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mgbf_device.hpp"
#include "mgbf_launch.hpp"

namespace mgbf {
namespace {

// ---------------------------------------------------------------------------
// Banded vertical operator along the stack (Vf, Vf^T or the product Vf Vf^T):
// out(k) = sum_{t=-HB..HB} c(L,t) in(k+t) for k < nfilt, L = k mod lm, with the
// whole-sample mirror folded into the band; entries k >= nfilt pass through.
// Rows ilo <= L < ihi (clear of the mirror folds) share the uniform interior
// weights; the rows near the ends of a column read their row of the table. A block stages a
// contiguous span of up to kVSpan elements (one chunk of a point's column, or
// several whole points) plus the halo in LDS, so HBM is streamed contiguously.
// ---------------------------------------------------------------------------
constexpr int kVPer = 8;                    // elements per thread
constexpr int kVSpan = kBlock * kVPer;      // elements per block

template <int HB, bool FIXL>
__global__ void __launch_bounds__(kBlock)
vband_kernel(const float* __restrict__ in, float* __restrict__ out,
             const float* __restrict__ band, VBandW wint, int ilo, int ihi, int K, int lm,
             int nfilt, long long N, int chunks_per_point, int pspan) {
    constexpr int NB = 2 * HB + 1;
    __shared__ float s[kVSpan + 2 * HB];
    long long e0;
    int kbase, span;
    if (chunks_per_point > 0) {            // K > kVSpan: one chunk of one point
        const long long pt = blockIdx.x / chunks_per_point;
        kbase = (int)(blockIdx.x % chunks_per_point) * kVSpan;
        e0 = pt * K + kbase;
        span = K - kbase < kVSpan ? K - kbase : kVSpan;
    } else {                               // whole points, pspan = ppb * K elements
        kbase = 0;
        e0 = (long long)blockIdx.x * pspan;
        span = (int)(N - e0 < pspan ? N - e0 : pspan);
    }
    const int tid = threadIdx.x;
    float tmp[kVPer];
#pragma unroll
    for (int r = 0; r < kVPer; ++r) {
        const int i = tid + r * kBlock;
        const long long e = e0 - HB + i;
        tmp[r] = (i < span + 2 * HB && e >= 0 && e < N) ? in[e] : 0.f;
    }
    float tail = 0.f;
    if (tid < 2 * HB) {
        const int i = kVSpan + tid;
        const long long e = e0 - HB + i;
        tail = (i < span + 2 * HB && e >= 0 && e < N) ? in[e] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < kVPer; ++r) s[tid + r * kBlock] = tmp[r];
    if (tid < 2 * HB) s[kVSpan + tid] = tail;
    __syncthreads();
    if constexpr (FIXL) {
        // every column is filtered and lm divides the block: the level of
        // each element of this thread is tid mod lm, its band row is fixed
        float vc[NB];
        const float* c = band + (tid % lm) * NB;
#pragma unroll
        for (int t = 0; t < NB; ++t) vc[t] = c[t];
#pragma unroll
        for (int r = 0; r < kVPer; ++r) {
            const int l = tid + r * kBlock;
            if (l < span) {
                const float* row = s + l + HB;
                float v = 0.f;
#pragma unroll
                for (int t = 0; t < NB; ++t) v = __builtin_fmaf(vc[t], row[t - HB], v);
                out[e0 + l] = v;
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < kVPer; ++r) {
        const int l = tid + r * kBlock;
        if (l < span) {
            const int k = chunks_per_point > 0 ? kbase + l : l % K;
            const float* row = s + l + HB;
            float v;
            if (k < nfilt) {
                const int L = k % lm;
                v = 0.f;
                if (L >= ilo && L < ihi) {
#pragma unroll
                    for (int t = 0; t < NB; ++t) v = __builtin_fmaf(wint.w[t], row[t - HB], v);
                } else {
                    const float* c = band + L * NB;
#pragma unroll
                    for (int t = 0; t < NB; ++t) v = __builtin_fmaf(c[t], row[t - HB], v);
                }
            } else {
                v = row[0];
            }
            out[e0 + l] = v;
        }
    }
}

// The same operator where every column is filtered but no column fits the
// block (lm = 65, 127). A block takes 64 whole columns, lane l of its 4 waves
// column l, each wave a quarter of the levels: the level, and with it the band
// row, is the same in all lanes (scalar coefficients, read from memory only
// next to the column ends). The columns' contiguous span passes LDS in 16-byte
// pieces; a wave walks down its levels with the window in registers and leaves
// the results in place, past a copy of the HB levels below its quarter, which
// the next wave overwrites. An element passes LDS 4 times where the block
// above reads it 2 HB + 1 times and finds its level by two divisions. A pitch
// of lm keeps the lanes in different banks for odd lm, in pairs for
// lm = 2 mod 4. HBM is the bound, and LDS (lm x 256 bytes a block) limits the
// blocks that hide its latency: 1440 x 960 x 65 at HB = 6, 0.72 GB, in 139 us
// against 278 with the block above; 1024 x 1024 x 127 at HB = 3, 1.07 GB, in
// 193 against 268 (one wave a column block, without the quarters, took 396).
// ---------------------------------------------------------------------------
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
constexpr int kVColMaxHB = 8;     // hz <= 8 for Vf and Vf^T, <= 4 for their product
// Shorter columns give a block too few values beside its two waits, which tells
// on large fields: 1024 x 1024 points at HB = 1, 5 levels in 20 us against 13 with
// the block above, 7 in 22 against 18; at HB = 3, 9 in 26 against 23 and 11 in 27.8
// against 27.1. On small ones its launch is the shorter: 256 x 256 x 5 in 4.1 us
// against 5.5, even at 512 x 512 (7.5 against 7.0; 7 levels 8.1 against 7.9).
constexpr int kVColMinLm = 11;
constexpr long long kVColSmall = 1 << 18;   // columns
constexpr int kVColMaxLm = 128;   // 32 KB of columns: 4 blocks, 16 waves a CU
constexpr int kVColWaves = kBlock / kWave;
constexpr int kVColStep = 8;      // levels between shifts of the window

template <int HB, bool VEC>
__global__ void __launch_bounds__(kBlock)
vcol_kernel(const float* __restrict__ in, float* __restrict__ out, const float* __restrict__ band, VBandW wint,
            int ilo, int ihi, int lm, long long ncol) {
    constexpr int NB = 2 * HB + 1;
    extern __shared__ __align__(16) float s_mem[];
    float* const s_halo = s_mem;                                // [wave][HB][64]
    float* const s_col = s_mem + kVColWaves * HB * kWave;       // [64][lm]
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const long long c0 = (long long)blockIdx.x * kWave;
    const int cols = (int)(ncol - c0 < kWave ? ncol - c0 : kWave);
    const int span = cols * lm;
    const float* src = in + c0 * lm;
    float* dst = out + c0 * lm;
    // 8 loads in flight; those past the span's last 16 bytes read nothing
    const int n4 = span >> 2;
    constexpr int kStep = 8;
    if constexpr (VEC) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), (short)0, n4 * 16, 0x00020000);
        for (int e0 = 0; e0 < n4; e0 += kStep * kBlock) {
            u4 v[kStep];
#pragma unroll
            for (int q = 0; q < kStep; ++q)
                v[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, (e0 + q * kBlock + tid) * 16, 0, 0);
#pragma unroll
            for (int q = 0; q < kStep; ++q) {
                const int e = e0 + q * kBlock + tid;
                if (e < n4) reinterpret_cast<f4*>(s_col)[e] = __builtin_bit_cast(f4, v[q]);
            }
        }
        if (4 * n4 + tid < span) s_col[4 * n4 + tid] = src[4 * n4 + tid];
    } else {
        for (int e = tid; e < span; e += kBlock) s_col[e] = src[e];
    }
    __syncthreads();
    // levels l0 .. l1 - 1 are this wave's; lanes past the last column work on
    // their unused places
    const int q4 = (lm + kVColWaves - 1) / kVColWaves;
    const int l0 = wave * q4 < lm ? wave * q4 : lm, l1 = l0 + q4 < lm ? l0 + q4 : lm;
    float* const col = s_col + lane * lm;
    float* const halo = s_halo + wave * HB * kWave + lane;
    // w[t]: level L0 + t - HB; levels outside the column read as zero
    float w[2 * HB + kVColStep];
#pragma unroll
    for (int t = 0; t < 2 * HB; ++t) w[t] = 0.f;
    if (l0 < l1) {
#pragma unroll
        for (int t = 0; t < 2 * HB; ++t) {
            const int L = l0 + t - HB;
            if (L >= 0 && L < lm) w[t] = col[L];
        }
#pragma unroll
        for (int t = 0; t < HB; ++t) halo[t * kWave] = l1 + t < lm ? col[l1 + t] : 0.f;
    }
    __syncthreads();
    for (int L0 = l0; L0 < l1; L0 += kVColStep) {
#pragma unroll
        for (int t = 0; t < kVColStep; ++t) {
            const int L = L0 + HB + t;
            w[2 * HB + t] = L < l1 ? col[L] : halo[(L - l1 < HB ? L - l1 : HB - 1) * kWave];
        }
        if (L0 >= ilo && L0 + kVColStep <= ihi && L0 + kVColStep <= l1) {
#pragma unroll
            for (int q = 0; q < kVColStep; ++q) {
                float v = 0.f;
#pragma unroll
                for (int t = 0; t < NB; ++t) v = __builtin_fmaf(wint.w[t], w[q + t], v);
                col[L0 + q] = v;
            }
        } else {
#pragma unroll
            for (int q = 0; q < kVColStep; ++q) {
                const int L = L0 + q;
                if (L >= l1) break;
                float v = 0.f;
                const float* c = band + L * NB;
#pragma unroll
                for (int t = 0; t < NB; ++t) v = __builtin_fmaf(c[t], w[q + t], v);
                col[L] = v;
            }
        }
#pragma unroll
        for (int t = 0; t < 2 * HB; ++t) w[t] = w[t + kVColStep];
    }
    __syncthreads();
    if constexpr (VEC) {
        for (int e = tid; e < n4; e += kBlock) reinterpret_cast<f4*>(dst)[e] = reinterpret_cast<const f4*>(s_col)[e];
        if (4 * n4 + tid < span) dst[4 * n4 + tid] = s_col[4 * n4 + tid];
    } else {
        for (int e = tid; e < span; e += kBlock) dst[e] = s_col[e];
    }
}

// ---------------------------------------------------------------------------
// Prolongation P (coarse -> fine), optionally accumulated: the coarse field is
// read through the half-sample mirror (boco_2d) and interpolated with the
// stencil S, x then y (direct1, or direct2 for the quadratic stencil). One
// lane computes TJ fine rows of one fine column for its k; the NR
// x-interpolated coarse rows they need stay in registers.
// ---------------------------------------------------------------------------
template <int TJ, bool Q>
__global__ void __launch_bounds__(kBlock)
prolong2_kernel(const float* __restrict__ coarse, const float* addend, float* out, int K, int nf,
                int mf, int nkc, int nstrip, int nitems) {
    using S = Stencil<Q>;
    constexpr int NP = S::NP;
    constexpr int CO = S::OFF[0] < S::OFF[1] ? S::OFF[0] : S::OFF[1];  // lowest coarse offset
    constexpr int NR = TJ / 2 + NP - 1 + (S::OFF[1] - CO);
    const int lane = threadIdx.x & (kWave - 1);
    const int item = (int)xcd_block(blockIdx.x, gridDim.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (item >= nitems) return;
    const int kc = item % nkc;
    const int rest = item / nkc;
    const int i = rest % nf;
    const int js = rest / nf;
    const int k = kc * kWave + lane;
    const bool kvalid = k < K;
    const int kk = kvalid ? k : K - 1;
    const int nc = nf / 2, mc = mf / 2;
    const int u = i >> 1;
    const int par = i & 1;
    const int cs = u + (par ? S::OFF[1] : S::OFF[0]);
    float cw[NP];
    int xo[NP];
#pragma unroll
    for (int t = 0; t < NP; ++t) {
        cw[t] = par ? S::C[1][t] : S::C[0][t];
        xo[t] = mirror_half(cs + t, nc) * K;
    }
    const int j0 = js * TJ;
    const int u0 = j0 >> 1;
    const size_t crow = (size_t)nc * K;
    float xv[NR];   // coarse rows u0 + CO .. u0 + CO + NR - 1, interpolated along x
#pragma unroll
    for (int t = 0; t < NR; ++t) {
        const int r = mirror_half(u0 + CO + t, mc);
        const float* row = coarse + kk + (size_t)r * crow;
        float a = 0.f;
#pragma unroll
        for (int c = 0; c < NP; ++c) a = __builtin_fmaf(cw[c], row[xo[c]], a);
        xv[t] = a;
    }
    if (!kvalid) return;
    const size_t frow = (size_t)nf * K;
#pragma unroll
    for (int q = 0; q < TJ; ++q) {
        const int j = j0 + q;
        if (j < mf) {
            const int pq = q & 1;
            const int b = (q >> 1) + (pq ? S::OFF[1] : S::OFF[0]) - CO;
            float a = 0.f;
#pragma unroll
            for (int t = 0; t < NP; ++t) a = __builtin_fmaf(pq ? S::C[1][t] : S::C[0][t], xv[b + t], a);
            const size_t e = kk + (size_t)j * frow + (size_t)i * K;
            out[e] = (addend ? addend[e] : 0.f) + a;
        }
    }
}


// ---------------------------------------------------------------------------
// Restriction R = Fold o P^T (fine -> coarse). One lane computes TI2 coarse
// columns x TJ2 coarse rows for its k, coarse row by coarse row. An interior
// coarse row J is the NR-point stencil S::R over the x-restricted fine rows
// 2J+ROFF .. 2J+ROFF+NR-1 (2J-3 .. 2J+4 for the 4-point stencil, 2J-2 ..
// 2J+3 for the quadratic one), which a sliding window keeps in registers: the
// next row needs two new fine rows. Rows and columns within S::EDGE of an
// edge carry the folded mirror contributions and use the window tables.
// ---------------------------------------------------------------------------
// A wave whose columns lie within S::EDGE of a domain edge reads each coarse
// column's own 8-column window with the weights of the x table (wave-uniform
// scalar loads); everything else is the same for both, so an edge tile takes
// about as long as an interior one: 256^2 x 64 in 18 us, 1440 x 960 x 65 and
// its next two generations in 105 us each on average for the first two and
// 27 us (162 us and 303, 203 and 172 us when an edge tile worked through one
// coarse point at a time, 64 dependent loads each, in strips of 16 rows).
// What bounds it is the latency of the two new fine rows of a coarse row.
// The rows per wave tj2 are a launch parameter: launch_restrict.
template <int TI2, bool Q>
__global__ void __launch_bounds__(kBlock)
restrict3_kernel(const float* __restrict__ fine, float* __restrict__ coarse, int K, int nf,
                 int mf, const int* __restrict__ rxs, const float* __restrict__ rxw,
                 const int* __restrict__ rys, const float* __restrict__ ryw, int tj2, int nkc, int ntile_i,
                 int nstrip, int nitems) {
    constexpr int WR = kRWidthDev;
    using S = Stencil<Q>;
    constexpr int NRW = S::NR, E = S::EDGE;
    constexpr int NCF = 2 * TI2 + NRW - 2;
    const int lane = threadIdx.x & (kWave - 1);
    const int item = (int)xcd_block(blockIdx.x, gridDim.x) * kWavesPerBlock +
                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= nitems) return;
    // k chunks fastest: consecutive waves read the whole k extent of a column
    // (K x 4 contiguous bytes) together, which keeps DRAM pages open; the
    // halo columns this re-reads mostly hit the caches
    const int kc = item % nkc;
    const int rest = item / nkc;
    const int ti = rest % ntile_i;
    const int js = rest / ntile_i;
    const int k = kc * kWave + lane;
    const bool kvalid = k < K;
    const int kk = kvalid ? k : K - 1;
    const int nc = nf / 2, mc = mf / 2;
    const int I0 = ti * TI2, J0 = js * tj2;
    const int J1 = J0 + tj2 < mc ? J0 + tj2 : mc;
    const bool xedge = !(I0 >= E && I0 + TI2 <= nc - E);
    const size_t frow = (size_t)nf * K;
    // interior columns: fine columns 2*I0+ROFF .. 2*I0+ROFF+NCF-1, addressed
    // as the row's buffer + lane k + wave-uniform column offset
    const float* base = fine + (xedge ? (size_t)0 : (size_t)(2 * I0 + S::ROFF) * K);
    const int vk = kk * 4;
    auto xrow = [&](int fr, float* out) {
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(base + (size_t)fr * frow);
        if (xedge) {
            float v[TI2][WR];
#pragma unroll
            for (int c = 0; c < TI2; ++c) {
                const int s0 = rxs[I0 + c < nc ? I0 + c : nc - 1];
#pragma unroll
                for (int t = 0; t < WR; ++t) v[c][t] = buf_ld(rs, vk, (s0 + t < nf ? s0 + t : nf - 1) * K * 4);
            }
#pragma unroll
            for (int c = 0; c < TI2; ++c) {
                const int I = I0 + c < nc ? I0 + c : nc - 1;
                const int s0 = rxs[I];
                float a = 0.f;
#pragma unroll
                for (int t = 0; t < WR; ++t) {
                    const float w = s0 + t < nf ? rxw[I * WR + t] : 0.f;
                    a = __builtin_fmaf(w, v[c][t], a);
                }
                out[c] = a;
            }
            return;
        }
        float v[NCF];
#pragma unroll
        for (int c = 0; c < NCF; ++c) v[c] = buf_ld(rs, vk, c * K * 4);
#pragma unroll
        for (int c = 0; c < TI2; ++c) {
            float a = 0.f;
#pragma unroll
            for (int t = 0; t < NRW; ++t) a = __builtin_fmaf(S::R[t], v[2 * c + t], a);
            out[c] = a;
        }
    };
    float win[NRW][TI2];   // x-restricted fine rows 2J+ROFF .. 2J+ROFF+NRW-1
    int wbase = -1000;     // fine row held in win[0]
    for (int J = J0; J < J1; ++J) {
        float acc[TI2];
        if (J >= E && J <= mc - 1 - E) {
            const int fb = 2 * J + S::ROFF;
            if (fb == wbase + 2) {
#pragma unroll
                for (int t = 0; t < NRW - 2; ++t)
#pragma unroll
                    for (int c = 0; c < TI2; ++c) win[t][c] = win[t + 2][c];
                xrow(fb + NRW - 2, win[NRW - 2]);
                xrow(fb + NRW - 1, win[NRW - 1]);
            } else {
#pragma unroll
                for (int t = 0; t < NRW; ++t) xrow(fb + t, win[t]);
            }
            wbase = fb;
#pragma unroll
            for (int c = 0; c < TI2; ++c) {
                float a = 0.f;
#pragma unroll
                for (int t = 0; t < NRW; ++t) a = __builtin_fmaf(S::R[t], win[t][c], a);
                acc[c] = a;
            }
        } else {
            // fold rows: the y window table of coarse row J
            const int ys = rys[J];
#pragma unroll
            for (int c = 0; c < TI2; ++c) acc[c] = 0.f;
#pragma unroll
            for (int t = 0; t < WR; ++t) {
                const int jj = ys + t < mf ? ys + t : mf - 1;
                const float wy = ys + t < mf ? ryw[J * WR + t] : 0.f;
                float xv[TI2];
                xrow(jj, xv);
#pragma unroll
                for (int c = 0; c < TI2; ++c) acc[c] = __builtin_fmaf(wy, xv[c], acc[c]);
            }
            wbase = -1000;
        }
        if (kvalid) {
            const __amdgpu_buffer_rsrc_t ro = buf_rsrc(coarse + (size_t)K * ((size_t)I0 + (size_t)nc * J));
#pragma unroll
            for (int c = 0; c < TI2; ++c)
                if (I0 + c < nc) buf_st(acc[c], ro, vk, c * K * 4);
        }
    }
}

// out = in * (wfield ? f(wfield) : f(wconst)), f = identity or sqrt
__global__ void __launch_bounds__(kBlock)
scale_kernel(const float* __restrict__ in, float* __restrict__ out,
             const float* __restrict__ wfield, float wconst, int use_sqrt, long long count) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += stride) {
        float w = wfield ? wfield[e] : wconst;
        if (use_sqrt) w = __builtin_sqrtf(w);
        out[e] = w * in[e];
    }
}

__global__ void __launch_bounds__(kBlock)
copy_kernel(const float* __restrict__ in, float* __restrict__ out, long long count) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += stride)
        out[e] = in[e];
}

// FP64-accumulated inner product in two launches with a fixed order (so
// the result does not depend on scheduling): each of kDotBlocks blocks sums
// its grid-stride share into partial[block], 16-byte loads when both arrays
// are 16-byte aligned; one block then sums the partials.
__device__ __forceinline__ double block_sum(double s) {
    __shared__ double ws[kWavesPerBlock];
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & (kWave - 1)) == 0) ws[threadIdx.x / kWave] = s;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kWavesPerBlock; ++w) t += ws[w];
    return t;
}

template <bool VEC>
__global__ void __launch_bounds__(kBlock)
dot_partial_kernel(const float* __restrict__ a, const float* __restrict__ b, long long count,
                   double* __restrict__ partial) {
    double s = 0.0;
    const long long tid = (long long)blockIdx.x * kBlock + threadIdx.x;
    const long long stride = (long long)gridDim.x * kBlock;
    long long head = 0;
    if constexpr (VEC) {
        const long long n4 = count >> 2;
        const float4* a4 = reinterpret_cast<const float4*>(a);
        const float4* b4 = reinterpret_cast<const float4*>(b);
        for (long long e = tid; e < n4; e += stride) {
            const float4 x = a4[e], y = b4[e];
            s = __builtin_fma((double)x.x, (double)y.x, s);
            s = __builtin_fma((double)x.y, (double)y.y, s);
            s = __builtin_fma((double)x.z, (double)y.z, s);
            s = __builtin_fma((double)x.w, (double)y.w, s);
        }
        head = n4 << 2;
    }
    for (long long e = head + tid; e < count; e += stride) s = __builtin_fma((double)a[e], (double)b[e], s);
    const double t = block_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kBlock) dot_final_kernel(const double* __restrict__ partial, int n,
                                                           double* __restrict__ acc) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += kBlock) s += partial[i];
    const double t = block_sum(s);
    if (threadIdx.x == 0) *acc = t;
}

__global__ void __launch_bounds__(kBlock) fill_kernel(float* p, float v, long long count) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += stride)
        p[e] = v;
}

unsigned grid_for(long long count) {
    long long g = (count + kBlock - 1) / kBlock;
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (unsigned)g;
}

}  // namespace

// The band runs only over whole columns (lm divides the wave, the wave the
// stack) after a prolongation, with the half-widths launch_radial_band lists; a
// weight field or a restriction does not go with a prolongation.
bool radial_built(const RadialArgs& a) {
    if (a.mfma || (a.exact_disc && a.separable) || (a.coarse && (a.wfield || a.rout))) return false;
    if (a.TI != 2 && a.TI != 4) return false;
    if (!a.band) return true;
    const bool hb = a.vhb == 3 || a.vhb == 4 || a.vhb == 6 || a.vhb == 8;
    return hb && (a.exact_disc || a.separable) && a.coarse && !a.klo && a.lm >= 1 && kWave % a.lm == 0 && a.K % kWave == 0;
}

hipError_t launch_radial(const RadialArgs& a, hipStream_t st) {
    // a k offset takes no band (whole columns are not in the wave) and no
    // matrix-core engine
    if (a.klo < 0 || a.klo >= a.K || (a.klo && (a.mfma || a.band))) return hipErrorInvalidValue;
    const bool two = a.TI == 2 && !a.rout;
#define MGBF_RADIAL_CASE(h)                                                                       \
    case h:                                                                                       \
        if (a.mfma) return launch_radial_mx_H##h(a, st);                                          \
        if (a.exact_disc) return two ? launch_radial_disc2_H##h(a, st) : launch_radial_disc_H##h(a, st); \
        if (a.separable) return two ? launch_radial_sep2_H##h(a, st) : launch_radial_sep_H##h(a, st);   \
        return two ? launch_radial_box2_H##h(a, st) : launch_radial_box_H##h(a, st);
    switch (a.H) {
        MGBF_RADIAL_CASE(1) MGBF_RADIAL_CASE(2) MGBF_RADIAL_CASE(3) MGBF_RADIAL_CASE(4) MGBF_RADIAL_CASE(5)
        MGBF_RADIAL_CASE(6) MGBF_RADIAL_CASE(7) MGBF_RADIAL_CASE(8) MGBF_RADIAL_CASE(9) MGBF_RADIAL_CASE(10)
        default: return hipErrorInvalidValue;
    }
#undef MGBF_RADIAL_CASE
}

hipError_t launch_ball3(const Ball3Args& a, hipStream_t st) {
    if (a.HZ < 0 || a.HZ > kBall3MaxHZ || a.lm < 2 * a.HZ + 2 || kWave % a.lm != 0 || a.TJ < 1 ||
        a.K3 > a.K || a.K3 < 1)
        return hipErrorInvalidValue;
    switch (a.H) {
        case 1: return launch_ball3_H1(a, st);
        case 2: return launch_ball3_H2(a, st);
        case 3: return launch_ball3_H3(a, st);
        case 4: return launch_ball3_H4(a, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_restrict(const TransferArgs& a, hipStream_t st) {
    constexpr int TI2 = 4;
    const int nc = a.nf / 2, mc = a.mf / 2;
    const int ntile_i = (nc + TI2 - 1) / TI2;
    const int nkc = (a.K + kWave - 1) / kWave;
    // Coarse rows per wave: 16 read 38 fine rows (2.4 a row) where 4 read 14
    // (3.5 a row), so shorter strips pay only while the launch leaves SIMDs
    // without a wave to hide the loads of the others.
    int tj2 = 16;
    while (tj2 > 2 && (long long)ntile_i * nkc * ((mc + tj2 - 1) / tj2) < 8192) tj2 /= 2;
    const int nstrip = (mc + tj2 - 1) / tj2;
    const long long nitems = (long long)ntile_i * nstrip * nkc;
    if (nitems >= (1ll << 31)) return hipErrorInvalidValue;
    const unsigned nblocks = (unsigned)((nitems + kWavesPerBlock - 1) / kWavesPerBlock);
    if (a.quad)
        hipLaunchKernelGGL((restrict3_kernel<TI2, true>), dim3(nblocks), dim3(kBlock), 0, st,
                           a.src, a.dst, a.K, a.nf, a.mf, a.xs, a.xw, a.ys, a.yw, tj2, nkc,
                           ntile_i, nstrip, (int)nitems);
    else
        hipLaunchKernelGGL((restrict3_kernel<TI2, false>), dim3(nblocks), dim3(kBlock), 0, st,
                           a.src, a.dst, a.K, a.nf, a.mf, a.xs, a.xw, a.ys, a.yw, tj2, nkc,
                           ntile_i, nstrip, (int)nitems);
    return hipGetLastError();
}

hipError_t launch_prolong(const TransferArgs& a, const float* addend, hipStream_t st) {
    constexpr int TJ = 16;
    const int nstrip = (a.mf + TJ - 1) / TJ;
    const int nkc = (a.K + kWave - 1) / kWave;
    const long long nitems = (long long)a.nf * nstrip * nkc;
    const unsigned nblocks = (unsigned)((nitems + kWavesPerBlock - 1) / kWavesPerBlock);
    if (a.quad)
        hipLaunchKernelGGL((prolong2_kernel<TJ, true>), dim3(nblocks), dim3(kBlock), 0, st, a.src,
                           addend, a.dst, a.K, a.nf, a.mf, nkc, nstrip, (int)nitems);
    else
        hipLaunchKernelGGL((prolong2_kernel<TJ, false>), dim3(nblocks), dim3(kBlock), 0, st, a.src,
                           addend, a.dst, a.K, a.nf, a.mf, nkc, nstrip, (int)nitems);
    return hipGetLastError();
}

template <int HB>
hipError_t launch_vband_h(const VBandArgs& a, hipStream_t st) {
    const bool fixl = a.nfilt == a.K && kBlock % a.lm == 0 && a.K % a.lm == 0;
    const long long N = (long long)a.K * a.npts;
    // whole columns of a length that spreads them over the LDS banks
    const long long ncol = a.nfilt == a.K && a.K % a.lm == 0 ? N / a.lm : 0;
    if constexpr (HB <= kVColMaxHB) if (!fixl && ncol && a.lm % 4 && (a.lm >= kVColMinLm || ncol < kVColSmall) && a.lm <= kVColMaxLm && ncol <= (1ll << 30) - kWave) {   // 4 threads a column, below 2^32
        const dim3 g((unsigned)((ncol + kWave - 1) / kWave));
        const size_t lds = sizeof(float) * kWave * (a.lm + kVColWaves * HB);
        // 64 columns start at a multiple of 256 bytes from the base
        if (((reinterpret_cast<size_t>(a.in) | reinterpret_cast<size_t>(a.out)) & 15) == 0)
            hipLaunchKernelGGL((vcol_kernel<HB, true>), g, dim3(kBlock), lds, st, a.in, a.out, a.band, a.wint, a.ilo,
                               a.ihi, a.lm, ncol);
        else
            hipLaunchKernelGGL((vcol_kernel<HB, false>), g, dim3(kBlock), lds, st, a.in, a.out, a.band, a.wint, a.ilo,
                               a.ihi, a.lm, ncol);
        return hipGetLastError();
    }
    int cpp = 0, pspan = 0;
    long long nblocks;
    if (a.K > kVSpan) {
        cpp = (a.K + kVSpan - 1) / kVSpan;
        nblocks = a.npts * cpp;
    } else {
        const int ppb = kVSpan / a.K;
        pspan = ppb * a.K;
        nblocks = (N + pspan - 1) / pspan;
    }
    if (fixl)
        hipLaunchKernelGGL((vband_kernel<HB, true>), dim3((unsigned)nblocks), dim3(kBlock), 0, st,
                           a.in, a.out, a.band, a.wint, a.ilo, a.ihi, a.K, a.lm, a.nfilt, N, cpp,
                           pspan);
    else
        hipLaunchKernelGGL((vband_kernel<HB, false>), dim3((unsigned)nblocks), dim3(kBlock), 0, st,
                           a.in, a.out, a.band, a.wint, a.ilo, a.ihi, a.K, a.lm, a.nfilt, N, cpp,
                           pspan);
    return hipGetLastError();
}

hipError_t launch_vband(const VBandArgs& a, hipStream_t st) {
    switch (a.HB) {
#define MGBF_VB(h) case h: return launch_vband_h<h>(a, st);
        MGBF_VB(1) MGBF_VB(2) MGBF_VB(3) MGBF_VB(4) MGBF_VB(5) MGBF_VB(6) MGBF_VB(7)
        MGBF_VB(8) MGBF_VB(9) MGBF_VB(10) MGBF_VB(11) MGBF_VB(12) MGBF_VB(13) MGBF_VB(14)
        MGBF_VB(15) MGBF_VB(16) MGBF_VB(17) MGBF_VB(18) MGBF_VB(19) MGBF_VB(20)
#undef MGBF_VB
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_scale(const float* in, float* out, const float* wfield, float wconst,
                        int use_sqrt, long long count, hipStream_t st) {
    hipLaunchKernelGGL(scale_kernel, dim3(grid_for(count)), dim3(kBlock), 0, st, in, out, wfield,
                       wconst, use_sqrt, count);
    return hipGetLastError();
}

hipError_t launch_copy(const float* in, float* out, long long count, hipStream_t st) {
    hipLaunchKernelGGL(copy_kernel, dim3(grid_for(count)), dim3(kBlock), 0, st, in, out, count);
    return hipGetLastError();
}

// One wave per output point and 64 consecutive k: the window weights are
// wave-uniform (scalar loads), every tap a 256-byte coalesced read.
__global__ void __launch_bounds__(kBlock) xfer2d_kernel(XferArgs a, long long nitems) {
    const long long item = (long long)blockIdx.x * kWavesPerBlock +
                           __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= nitems) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int nkc = (a.K + kWave - 1) / kWave;
    const int kc = (int)(item % nkc);
    const long long pt = item / nkc;
    const int i = (int)(pt % a.nout_x), j = (int)(pt / a.nout_x);
    const int k = kc * kWave + lane;
    if (k >= a.K) return;
    const int x0 = a.xs[i], y0 = a.ys[j];
    float acc = 0.f;
    for (int ty = 0; ty < a.wy; ++ty) {
        const float wyv = a.yw[(size_t)j * a.wy + ty];
        const float* row = a.in + k + (size_t)a.K * ((size_t)a.nin_x * (y0 + ty) + x0);
        float r = 0.f;
        for (int tx = 0; tx < a.wx; ++tx) r = __builtin_fmaf(a.xw[(size_t)i * a.wx + tx], row[(size_t)tx * a.K], r);
        acc = __builtin_fmaf(wyv, r, acc);
    }
    a.out[k + (size_t)a.K * ((size_t)a.nout_x * j + i)] = acc;
}

// One wave per 8 x 8 output points and 64 consecutive k: the input block of
// the tile streams through registers row by row; each row is interpolated in
// x for the 8 output columns (dense tile weights, wave-uniform) and added
// into the 8 output rows with their y weights.
// MODE 1 (direct transfer with its vertical map): the 64 k are filter
// levels; each finished output row goes through a per-wave LDS tile, and
// each lane forms up to two analysis levels of every point from a window
// of 4 of the chunk's levels. MODE 2 (adjoint transfer): every input point
// brings the chunk's analysis levels (up to 128, two coalesced loads per
// lane) through a per-wave LDS tile, and each lane maps its window of 4 to
// its filter level before the horizontal pass.
template <int SX, int MODE>
__global__ void __launch_bounds__(kBlock) xfer_tile_kernel(XferTileArgs a, XferVArgs v, int ntx, int nty,
                                                         long long nitems) {
    constexpr int TB = 8;
    constexpr int DP = kWave + 4;        // LDS pitch of an output point's levels (MODE 1)
    constexpr int AP = 2 * kWave + 4;    // LDS pitch of an input point's levels (MODE 2)
    constexpr int LDSW = MODE == 1 ? TB * DP : (MODE == 2 ? SX * AP : 1);
    __shared__ float lds_v[kWavesPerBlock][LDSW];
    // the tile's x weights, read by every lane at the same address (held in
    // scalar registers they spill: TB x SX of them beside the column offsets)
    __shared__ __align__(16) float lds_wx[kWavesPerBlock][TB * SX];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long item = (long long)xcd_block(blockIdx.x, gridDim.x) * kWavesPerBlock + wv;
    if (item >= nitems) return;
    const int lane = threadIdx.x & (kWave - 1);
    // With a vertical map the chunks of one tile are neighbours in the
    // launch: their level runs on the analysis grid (lm_a levels a column)
    // share cache lines at the chunk boundaries. The adjoint, which reads
    // the analysis grid, takes the tiles in strips of kStrip columns from
    // top to bottom: a row of tiles starts as the row above it finishes and
    // finds the input rows they share still cached.
    int p, q, kc;
    if constexpr (MODE == 0) {
        p = (int)(item % ntx);
        const long long rest = item / ntx;
        q = (int)(rest % nty);
        kc = (int)(rest / nty);
    } else if constexpr (MODE == 1) {
        const int nkc = (a.K + kWave - 1) / kWave;
        kc = (int)(item % nkc);
        const long long rest = item / nkc;
        p = (int)(rest % ntx);
        q = (int)(rest / ntx);
    } else {
        constexpr int kStrip = 16;
        const int nkc = (a.K + kWave - 1) / kWave;
        kc = (int)(item % nkc);
        const long long t = item / nkc;
        const int nfull = ntx / kStrip;
        const long long fullsz = (long long)kStrip * nty;
        if (t < nfull * fullsz) {
            const long long r = t % fullsz;
            q = (int)(r / kStrip);
            p = (int)(t / fullsz) * kStrip + (int)(r % kStrip);
        } else {
            const long long r = t - nfull * fullsz;
            const int wl = ntx - nfull * kStrip;
            q = (int)(r / wl);
            p = nfull * kStrip + (int)(r % wl);
        }
    }
    const int k = kc * kWave + lane;
    const bool kvalid = k < a.K;
    const int vk = (kvalid ? k : a.K - 1) * 4;
    const int x0 = a.x0[p], y0 = a.y0[q];
    const float* WX = a.wx + (size_t)p * TB * SX;
    for (int e = lane; e < TB * SX; e += kWave) lds_wx[wv][e] = WX[e];
    const float* WXL = lds_wx[wv];
    const float* WY = a.wy + (size_t)q * TB * a.SY;
    float* const col = lds_v[wv];
    // levels per input point: the filter stack, or (MODE 2) the analysis one
    const int kin = MODE == 2 ? v.kv : a.K;
    int soff[SX];
#pragma unroll
    for (int c = 0; c < SX; ++c) soff[c] = (x0 + c) * kin * 4;
    // MODE 2: the chunk's analysis levels lo .. lo+cnt-1, loaded as lo + lane
    // and lo + 64 + lane (clamped into the span, zero beyond it), and the
    // lane's window r0 .. r0+3 of them
    int voff[2] = {vk, vk};
    bool vin[2] = {true, true};
    int r0 = 0;
    float vw[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE == 2) {
        const int lo = v.lo[kc], cnt = v.cnt[kc];
        const int last = cnt > 0 ? cnt - 1 : 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = lane + h * kWave;
            vin[h] = e < cnt;
            voff[h] = (lo + (e < last ? e : last)) * 4;
        }
        const int kk = kvalid ? k : a.K - 1;
        r0 = v.r0[kk];
#pragma unroll
        for (int u = 0; u < 4; ++u) vw[u] = v.w[(size_t)kk * 4 + u];
        settle(r0);
#pragma unroll
        for (int u = 0; u < 4; ++u) settle(vw[u]);
        // the pads past the last level: read by zero taps only
        for (int e = lane; e < 4 * SX; e += kWave) col[(e >> 2) * AP + 2 * kWave + (e & 3)] = 0.f;
    }
    float acc[TB][TB];
#pragma unroll
    for (int u = 0; u < TB; ++u)
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[u][t] = 0.f;
    const size_t rowstride = (size_t)a.nin_x * kin;
    constexpr int NH = MODE == 2 ? 2 : 1;
    // the next input row is loaded while the current one is combined
    float vn[SX][NH];
    auto load_row = [&](int y) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(a.in + (size_t)y * rowstride);
#pragma unroll
        for (int c = 0; c < SX; ++c)
#pragma unroll
            for (int h = 0; h < NH; ++h) vn[c][h] = buf_ld(rs, voff[h], soff[c]);
    };
    load_row(y0);
    for (int r = 0; r < a.SY; ++r) {
        float vc[SX];
        if constexpr (MODE == 2) {
            // the row's points through LDS, then each lane's window
#pragma unroll
            for (int c = 0; c < SX; ++c) {
                col[c * AP + lane] = vin[0] ? vn[c][0] : 0.f;
                col[c * AP + kWave + lane] = vin[1] ? vn[c][1] : 0.f;
            }
            if (r + 1 < a.SY) load_row(y0 + r + 1);
#pragma unroll
            for (int c = 0; c < SX; ++c) {
                const float* cv = col + c * AP + r0;
                vc[c] = __builtin_fmaf(vw[0], cv[0],
                                       __builtin_fmaf(vw[1], cv[1], __builtin_fmaf(vw[2], cv[2], vw[3] * cv[3])));
            }
        } else {
#pragma unroll
            for (int c = 0; c < SX; ++c) vc[c] = vn[c][0];
            if (r + 1 < a.SY) load_row(y0 + r + 1);
        }
        float xr[TB];
        // the x weights again at every row (an offset the compiler cannot
        // hoist): held in registers across the loop they would take TB x SX
        // VGPRs
        int wo = 0;
        asm("" : "+s"(wo) : "s"(r));
        const float* wl = WXL + wo;
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            float z = 0.f;
#pragma unroll
            for (int c = 0; c < SX; ++c) z = __builtin_fmaf(wl[t * SX + c], vc[c], z);
            xr[t] = z;
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const float wy = WY[u * a.SY + r];
#pragma unroll
            for (int t = 0; t < TB; ++t) acc[u][t] = __builtin_fmaf(wy, xr[t], acc[u][t]);
        }
    }
    if constexpr (MODE == 1) {
        // every lane (also those past K, whose levels no window reads)
        // writes its level of each point; a lane forms analysis levels
        // lo + lane and lo + 64 + lane of the chunk
        const int lo = v.lo[kc], cnt = v.cnt[kc];
        int o0[2];
        bool ov[2];
        float ow[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int o = s * kWave + lane;
            ov[s] = o < cnt;
            // a lane past cnt reads output lo's entry and drops its result
            const int ko = lo + (ov[s] ? o : 0);
            o0[s] = v.r0[ko];
#pragma unroll
            for (int u = 0; u < 4; ++u) ow[s][u] = v.w[(size_t)ko * 4 + u];
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            settle(o0[s]);
#pragma unroll
            for (int u = 0; u < 4; ++u) settle(ow[s][u]);
        }
        if (lane < 4 * TB) col[(lane >> 2) * DP + kWave + (lane & 3)] = 0.f;
        const size_t orow = (size_t)a.nout_x * v.kv;
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const int j = q * TB + u;
            if (j >= a.nout_y) break;
#pragma unroll
            for (int t = 0; t < TB; ++t) col[t * DP + lane] = acc[u][t];
            const __amdgpu_buffer_rsrc_t ro = buf_rsrc(a.out + (size_t)j * orow);
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                const int i = p * TB + t;
                if (i >= a.nout_x) break;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const float* cv = col + t * DP + o0[s];
                    const float y = __builtin_fmaf(
                        ow[s][0], cv[0], __builtin_fmaf(ow[s][1], cv[1], __builtin_fmaf(ow[s][2], cv[2], ow[s][3] * cv[3])));
                    if (ov[s]) buf_st(y, ro, (lo + s * kWave + lane) * 4, i * v.kv * 4);
                }
            }
        }
        return;
    }
    if (!kvalid) return;
#pragma unroll
    for (int u = 0; u < TB; ++u) {
        const int j = q * TB + u;
        if (j < a.nout_y) {
            const __amdgpu_buffer_rsrc_t ro = buf_rsrc(a.out + (size_t)j * a.nout_x * a.K + (size_t)p * TB * a.K);
#pragma unroll
            for (int t = 0; t < TB; ++t)
                if (p * TB + t < a.nout_x) buf_st(acc[u][t], ro, vk, t * a.K * 4);
        }
    }
}

// One wave per 64 consecutive output k and kWinPoints consecutive points:
// each lane reads its window (start and weights) once and applies it to
// every point of the run.
constexpr int kWinPoints = 8;
constexpr int kWinMaxWidth = 8;

template <int W>
__global__ void __launch_bounds__(kBlock)
kwin_kernel(const float* __restrict__ in, float* __restrict__ out, int kin, int kout, long long npts,
            const int* __restrict__ ks, const float* __restrict__ kw, int w, int nkc, long long nitems) {
    const long long item = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (item >= nitems) return;
    const int kc = (int)(item % nkc);
    const long long p0 = (item / nkc) * kWinPoints;
    const int ko = kc * kWave + (threadIdx.x & (kWave - 1));
    if (ko >= kout) return;
    const int s0 = ks[ko];
    if constexpr (W == 0) {   // any width: the weights are read per point
        for (int q = 0; q < kWinPoints; ++q) {
            const long long p = p0 + q;
            if (p < npts) {
                const float* col = in + p * kin + s0;
                float acc = 0.f;
                for (int u = 0; u < w; ++u) acc = __builtin_fmaf(kw[(size_t)ko * w + u], col[u], acc);
                out[p * kout + ko] = acc;
            }
        }
    } else {
        float c[W];
#pragma unroll
        for (int u = 0; u < W; ++u) c[u] = u < w ? kw[(size_t)ko * w + u] : 0.f;
        // every load of the run is issued before the first store
        float x[kWinPoints][W];
#pragma unroll
        for (int q = 0; q < kWinPoints; ++q) {
            const long long p = p0 + q < npts ? p0 + q : npts - 1;
            const float* col = in + p * kin + s0;
#pragma unroll
            for (int u = 0; u < W; ++u) x[q][u] = u < w ? col[u] : 0.f;
        }
#pragma unroll
        for (int q = 0; q < kWinPoints; ++q) {
            float acc = 0.f;
#pragma unroll
            for (int u = 0; u < W; ++u) acc = __builtin_fmaf(c[u], x[q][u], acc);
            if (p0 + q < npts) out[(p0 + q) * kout + ko] = acc;
        }
    }
}

// 3-D filter of procedures 4 and 5 (vrbeta3 / vrbeta3T with sup_vrbeta3's
// level mirror; the hexad lines with zeros beyond the column ends) and the
// 2-D filter of the 2-D variables, as a gather: one
// lane per stacked k, one wave per 64 k of a grid point, taps wave-uniform.
// The transpose gathers every level L whose mirrored shift L + c lands on
// the output level (at most one direct and one mirrored preimage).
template <bool T>
__global__ void __launch_bounds__(kBlock) ball_kernel(BallArgs a, int nkc, long long nitems) {
    const long long item = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (item >= nitems) return;
    const int kc = (int)(item % nkc) + a.klo / kWave;
    const long long rest = item / nkc;
    const int i = (int)(rest % a.n), j = (int)(rest / a.n);
    const int k = kc * kWave + (threadIdx.x & (kWave - 1));
    if (k >= a.K || k < a.klo) return;
    const int lm = a.lm;
    float acc = 0.f;
    if (k < a.K3) {
        const int v0 = (k / lm) * lm, L = k - v0;
        for (int t = 0; t < a.n3; ++t) {
            const int4 g = a.t3[t];
            const int ii = mirror_half(i + g.x, a.n), jj = mirror_half(j + g.y, a.m);
            const float* col = a.in + (size_t)a.K * ((size_t)ii + (size_t)a.n * jj) + v0;
            float s;
            if (!T) {
                const int Ls = L + g.z;
                s = (a.zero_levels && (Ls < 0 || Ls >= lm)) ? 0.f : col[mirror_whole(Ls, lm)];
            } else {
                const int L1 = L - g.z, L2 = -L - g.z, L3 = 2 * (lm - 1) - L - g.z;
                s = (L1 >= 0 && L1 < lm) ? col[L1] : 0.f;
                if (!a.zero_levels) {
                    if (L > 0 && L2 >= 0 && L2 < lm) s += col[L2];
                    if (L < lm - 1 && L3 >= 0 && L3 < lm) s += col[L3];
                }
            }
            acc = __builtin_fmaf(a.w3[t], s, acc);
        }
    } else {
        for (int t = 0; t < a.n2; ++t) {
            const int4 g = a.t2[t];
            const int ii = mirror_half(i + g.x, a.n), jj = mirror_half(j + g.y, a.m);
            acc = __builtin_fmaf(a.w2[t], a.in[k + (size_t)a.K * ((size_t)ii + (size_t)a.n * jj)], acc);
        }
    }
    a.out[k + (size_t)a.K * ((size_t)i + (size_t)a.n * j)] = acc;
}

hipError_t launch_ball(const BallArgs& a, hipStream_t st) {
    if (a.klo < 0 || a.klo >= a.K) return hipErrorInvalidValue;
    const int nkc = (a.K + kWave - 1) / kWave - a.klo / kWave;
    const long long nitems = (long long)nkc * a.n * a.m;
    const long long nblocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock;
    if (nblocks >= (1ll << 31)) return hipErrorInvalidValue;
    if (a.transpose)
        hipLaunchKernelGGL(ball_kernel<true>, dim3((unsigned)nblocks), dim3(kBlock), 0, st, a, nkc, nitems);
    else
        hipLaunchKernelGGL(ball_kernel<false>, dim3((unsigned)nblocks), dim3(kBlock), 0, st, a, nkc, nitems);
    return hipGetLastError();
}

// The radial filter of a generation whose aspect tensor varies per point
// (vrbeta2 / vrbeta2T with el(:,:,ix,iy) and ss(ix,iy), jp_pbfil.f90:
// 888-928, 1011-1050) as a gather: point p = i + n j carries its weights over
// the box |gx|, |gy| <= H, w[p][t] with t = (gy+H)(2H+1) + gx+H.
//   F   (T = false): out(p) = sum_t w[p][t] in(mirror(p + g_t)), the gather of
//                    vrbeta2 over the mirrored halo of boco_2d (ss included,
//                    zero off the point's ellipse);
//   F^T (T = true):  out(p) = sum_t w[p][t] in(p + g_t) over the points of the
//                    domain, with the rows of the transposed matrix (the
//                    scatter of vrbeta2T and the fold of bocoT_2d, collected
//                    per output point when the tensors are set; zero where
//                    p + g_t lies outside).
//
// A wave computes TI x TJ outputs for its 64 k: each input row of the tile's
// halo enters the TJ output rows with every output's own weights. A row of an
// output's weights is one load that puts weight gx into lane gx of every 16
// lanes (two loads from half-width 8 on), and the FMAs take it from there by
// a DPP row broadcast, so a weight costs no instruction of its own. Inputs and
// weights of two rows are in flight while a third is combined: what bounds it
// is the (2H+1)^2 FMAs of an output (a third of their rate at 256 x 256 x 64,
// H = 6: 36 us for F and for F^T), and on a small grid the latency of the
// rows (20 us at 64 x 64 x 64). One tap at a time, behind a scalar load, a
// vector load and a branch on the weight, took 438 us (F) and 746 us (F^T);
// the weights as scalar operands 80 us, waiting on the scalar loads.
// Zero weights are multiplied like the others, which differs from leaving
// the tap out only where an input is infinite or NaN: an output of the tile
// that is not finite sends the wave through aspect_point, which leaves them
// out.
//
// One output point by its taps one after the other, zero weights left out.
template <bool T>
__device__ float aspect_point(const AspectArgs& a, int i, int j, int kk) {
    const int H = a.H, NB = 2 * H + 1, n = a.n, m = a.m;
    const size_t K = (size_t)a.K;
    const float* wp = a.w + ((size_t)i + (size_t)n * j) * NB * NB;
    float acc = 0.f;
    for (int gy = -H; gy <= H; ++gy)
        for (int gx = -H; gx <= H; ++gx) {
            const float wv = wp[(gy + H) * NB + gx + H];
            if (wv == 0.f) continue;
            // F^T has no weight on a point outside the domain
            const int ii = T ? i + gx : mirror_half(i + gx, n), jj = T ? j + gy : mirror_half(j + gy, m);
            acc = __builtin_fmaf(wv, a.in[kk + K * ((size_t)ii + (size_t)n * jj)], acc);
        }
    return acc;
}

template <int H, bool T>
__global__ void __launch_bounds__(kBlock) aspect_kernel(AspectArgs a, int nkc, int ntile_i, int nitems) {
    constexpr int TI = 4, TJ = 4, NB = 2 * H + 1, NT = NB * NB, NC = TI + 2 * H;
    const int item = (int)xcd_block(blockIdx.x, gridDim.x) * kWavesPerBlock +
                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= nitems) return;
    const int kc = item % nkc;
    const int rest = item / nkc;
    const int i0 = (rest % ntile_i) * TI, j0 = (rest / ntile_i) * TJ;
    const int k = kc * kWave + (threadIdx.x & (kWave - 1));
    const int K = a.K, n = a.n, m = a.m;
    const bool kvalid = k < K;
    const int vk = (kvalid ? k : K - 1) * 4;
    const size_t rowstride = (size_t)n * K;
    // a point outside the domain: its mirror image for F, any point for F^T
    // (its weight is zero)
    auto at = [](int q, int len) { return T ? (q < 0 ? 0 : (q < len ? q : len - 1)) : mirror_half(q, len); };
    int voff[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) voff[c] = vk + at(i0 - H + c, n) * K * 4;
    constexpr int NW = NB > 16 ? 2 : 1;
    int wl[NW];   // this lane's weight of a row of weights, in bytes
#pragma unroll
    for (int e = 0; e < NW; ++e) {
        const int gx = (threadIdx.x & 15) + 16 * e;
        wl[e] = (gx < NB ? gx : NB - 1) * 4;
    }
    float acc[TJ][TI];
#pragma unroll
    for (int q = 0; q < TJ; ++q)
#pragma unroll
        for (int t = 0; t < TI; ++t) acc[q][t] = 0.f;
    struct Row {
        float v[NC];
        float w[TJ][TI][NW];
    };
    auto used = [&](int r, int q) {   // does input row r enter output row j0 + q?
        const int gy = r - (j0 + q);
        return j0 + q < m && gy >= -H && gy <= H;
    };
    auto load = [&](int r, Row& d) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(a.in + (size_t)at(r, m) * rowstride);
#pragma unroll
        for (int c = 0; c < NC; ++c) d.v[c] = buf_ld(rs, voff[c], 0);
#pragma unroll
        for (int q = 0; q < TJ; ++q) {
            if (!used(r, q)) continue;
            const __amdgpu_buffer_rsrc_t rw =
                buf_rsrc(a.w + ((size_t)i0 + (size_t)n * (j0 + q)) * NT + (r - (j0 + q) + H) * NB);
            // a column past the domain takes the last one's weights; its output is dropped
#pragma unroll
            for (int t = 0; t < TI; ++t)
#pragma unroll
                for (int e = 0; e < NW; ++e)
                    d.w[q][t][e] = buf_ld(rw, wl[e], (i0 + t < n ? t : n - 1 - i0) * NT * 4);
        }
    };
    auto combine = [&](int r, const Row& d) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < TJ; ++q) {
            if (!used(r, q)) continue;
#pragma unroll
            for (int t = 0; t < TI; ++t) {
                fmac_row<(NB < 16 ? NB : 16)>(acc[q][t], d.w[q][t][0], d.v + t);
                if constexpr (NB > 16) fmac_row<NB - 16>(acc[q][t], d.w[q][t][1], d.v + t + 16);
            }
        }
    };
    static_assert((TJ + 2 * H) % 2 == 0, "rows come in pairs");
    Row A, B;
    load(j0 - H, A);
    load(j0 - H + 1, B);
    for (int r = j0 - H; r < j0 + TJ + H; r += 2) {
        combine(r, A);
        if (r + 2 < j0 + TJ + H) load(r + 2, A);
        combine(r + 1, B);
        if (r + 2 < j0 + TJ + H) load(r + 3, B);
    }
    bool odd = false;
#pragma unroll
    for (int q = 0; q < TJ; ++q)
#pragma unroll
        for (int t = 0; t < TI; ++t) odd = odd || !(__builtin_fabsf(acc[q][t]) < __builtin_inff());
    if (__any(odd)) {
        for (int q = 0; q < TJ; ++q)
            for (int t = 0; t < TI; ++t)
                if (j0 + q < m && i0 + t < n) {
                    const float x = aspect_point<T>(a, i0 + t, j0 + q, vk / 4);
#pragma unroll
                    for (int e = 0; e < TJ * TI; ++e)
                        if (e == q * TI + t) acc[e / TI][e % TI] = x;
                }
    }
    if (!kvalid) return;
#pragma unroll
    for (int q = 0; q < TJ; ++q) {
        const int j = j0 + q;
        if (j >= m) break;
        const size_t off = (size_t)j * rowstride + (size_t)i0 * K;
        const __amdgpu_buffer_rsrc_t ro = buf_rsrc(a.out + off);
        const __amdgpu_buffer_rsrc_t rw = buf_rsrc((a.wfield ? a.wfield : a.out) + off);
#pragma unroll
        for (int t = 0; t < TI; ++t)
            if (i0 + t < n) {
                const float s = a.wfield ? buf_ld(rw, vk, t * K * 4) : a.wconst;
                buf_st(s * acc[q][t], ro, vk, t * K * 4);
            }
    }
}

// The rows of the transposed matrix from those of F: point p takes the weight
// of every tap of p + g that reaches p, directly or through a mirror image of
// p (the box holds all of them: folding moves a point towards the tap's
// origin). The threads stride over the weights: a launch of one thread each
// would pass 2^32 threads, which HIP refuses, at 3120 x 3136 points of
// half-width 10.
__global__ void __launch_bounds__(kBlock) aspect_transpose_kernel(const float* __restrict__ w, float* __restrict__ wt,
                                                                int n, int m, int H, long long count) {
    const int NB = 2 * H + 1, nt = NB * NB;
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x; e < count; e += stride) {
        const int t = (int)(e % nt);
        const long long p = e / nt;
        const int i = (int)(p % n), j = (int)(p / n);
        const int sx = i + t % NB - H, sy = j + t / NB - H;
        float acc = 0.f;
        if (sx >= 0 && sx < n && sy >= 0 && sy < m) {
            const float* ws = w + ((size_t)sx + (size_t)n * sy) * nt;
            for (int b = 0; b < 3; ++b) {
                const int gy = (b == 0 ? j : (b == 1 ? -1 - j : 2 * m - 1 - j)) - sy;
                if (gy < -H || gy > H) continue;
                for (int c = 0; c < 3; ++c) {
                    const int gx = (c == 0 ? i : (c == 1 ? -1 - i : 2 * n - 1 - i)) - sx;
                    if (gx >= -H && gx <= H) acc += ws[(gy + H) * NB + gx + H];
                }
            }
        }
        wt[e] = acc;
    }
}

hipError_t launch_aspect_transpose(const float* w, float* wt, int n, int m, int H, hipStream_t st) {
    const long long count = (long long)n * m * (2 * H + 1) * (2 * H + 1);
    if (H < 1 || n < H || m < H) return hipErrorInvalidValue;
    hipLaunchKernelGGL(aspect_transpose_kernel, dim3(grid_for(count)), dim3(kBlock), 0, st, w, wt, n, m, H, count);
    return hipGetLastError();
}

// F^T without the rows of the transposed matrix, for a device that has no room
// for them: one wave per point and 64 k collects, over the mirror preimages e of
// the point (per axis -1-q within H of the low edge, 2n-1-q within H of the high
// one) and the taps t whose source e - g_t lies in the domain, that source's
// weight times its value. Each tap is a scalar load, a branch and a vector load:
// 850 us on 256 x 256 x 64 at H = 6, where the rows take 37.
__global__ void __launch_bounds__(kBlock) aspect_scatter_kernel(AspectArgs a) {
    const int H = a.H, NB = 2 * H + 1, n = a.n, m = a.m;
    const size_t K = (size_t)a.K;
    const int k = blockIdx.y * kWave + (threadIdx.x & (kWave - 1));
    const bool kvalid = k < a.K;
    const int kk = kvalid ? k : a.K - 1;
    const long long npts = (long long)n * m;
    for (long long pt = (long long)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
         pt < npts; pt += (long long)gridDim.x * kWavesPerBlock) {
        const int i = (int)(pt % n), j = (int)(pt / n);
        float acc = 0.f;
        for (int b = 0; b < 3; ++b) {
            if ((b == 1 && j > H - 1) || (b == 2 && j < m - H)) continue;
            const int ey = b == 0 ? j : (b == 1 ? -1 - j : 2 * m - 1 - j);
            for (int gy = -H; gy <= H; ++gy) {
                const int sy = ey - gy;
                if (sy < 0 || sy >= m) continue;
                for (int c = 0; c < 3; ++c) {
                    if ((c == 1 && i > H - 1) || (c == 2 && i < n - H)) continue;
                    const int ex = c == 0 ? i : (c == 1 ? -1 - i : 2 * n - 1 - i);
                    for (int gx = -H; gx <= H; ++gx) {
                        const int sx = ex - gx;
                        if (sx < 0 || sx >= n) continue;
                        const size_t sp = (size_t)sx + (size_t)n * sy;
                        const float wv = a.w[sp * NB * NB + (gy + H) * NB + gx + H];
                        if (wv != 0.f) acc = __builtin_fmaf(wv, a.in[kk + K * sp], acc);
                    }
                }
            }
        }
        const size_t o = kk + K * (size_t)pt;
        if (kvalid) a.out[o] = (a.wfield ? a.wfield[o] : a.wconst) * acc;
    }
}

hipError_t launch_aspect_scatter(const AspectArgs& a, hipStream_t st) {
    if (a.H < 1 || a.n < a.H || a.m < a.H || a.K < 1) return hipErrorInvalidValue;
    const long long nkc = (a.K + kWave - 1) / kWave, nb = ((long long)a.n * a.m + kWavesPerBlock - 1) / kWavesPerBlock;
    if (nkc > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(aspect_scatter_kernel, dim3((unsigned)std::min(nb, 1ll << 20), (unsigned)nkc), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int H>
hipError_t launch_aspect_h(const AspectArgs& a, bool transpose, hipStream_t st) {
    const int nkc = (a.K + kWave - 1) / kWave, ntile_i = (a.n + 3) / 4, ntile_j = (a.m + 3) / 4;
    const long long nitems = (long long)nkc * ntile_i * ntile_j;
    const long long nblocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock;
    // 32-bit offsets inside a row
    if (nitems >= (1ll << 31) || (long long)(a.n + 16) * a.K * 4 >= (1ll << 31)) return hipErrorInvalidValue;
    if (transpose)
        hipLaunchKernelGGL((aspect_kernel<H, true>), dim3((unsigned)nblocks), dim3(kBlock), 0, st, a, nkc, ntile_i,
                           (int)nitems);
    else
        hipLaunchKernelGGL((aspect_kernel<H, false>), dim3((unsigned)nblocks), dim3(kBlock), 0, st, a, nkc, ntile_i,
                           (int)nitems);
    return hipGetLastError();
}

hipError_t launch_aspect(const AspectArgs& a, bool transpose, hipStream_t st) {
    if (a.H < 1 || a.n < a.H || a.m < a.H || a.K < 1) return hipErrorInvalidValue;
    switch (a.H) {
        case 1: return launch_aspect_h<1>(a, transpose, st);
        case 2: return launch_aspect_h<2>(a, transpose, st);
        case 3: return launch_aspect_h<3>(a, transpose, st);
        case 4: return launch_aspect_h<4>(a, transpose, st);
        case 5: return launch_aspect_h<5>(a, transpose, st);
        case 6: return launch_aspect_h<6>(a, transpose, st);
        case 7: return launch_aspect_h<7>(a, transpose, st);
        case 8: return launch_aspect_h<8>(a, transpose, st);
        case 9: return launch_aspect_h<9>(a, transpose, st);
        case 10: return launch_aspect_h<10>(a, transpose, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_xfer2d(const XferArgs& a, hipStream_t st) {
    const long long nkc = (a.K + kWave - 1) / kWave;
    const long long nitems = nkc * a.nout_x * a.nout_y;
    const long long nblocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock;
    hipLaunchKernelGGL(xfer2d_kernel, dim3((unsigned)nblocks), dim3(kBlock), 0, st, a, nitems);
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_xfer_tile_mode(const XferTileArgs& a, const XferVArgs& v, hipStream_t st) {
    const int ntx = (a.nout_x + 7) / 8, nty = (a.nout_y + 7) / 8;
    const long long nkc = (a.K + kWave - 1) / kWave;
    const long long nitems = nkc * ntx * nty;
    const long long nblocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock;
    if (nblocks >= (1ll << 31) || a.SY < 1 || a.SY > a.nin_y || a.SX > a.nin_x) return hipErrorInvalidValue;
    const dim3 g((unsigned)nblocks), b(kBlock);
    switch (a.SX) {
        case 8: hipLaunchKernelGGL((xfer_tile_kernel<8, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        case 12: hipLaunchKernelGGL((xfer_tile_kernel<12, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        case 16: hipLaunchKernelGGL((xfer_tile_kernel<16, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        case 20: hipLaunchKernelGGL((xfer_tile_kernel<20, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        case 24: hipLaunchKernelGGL((xfer_tile_kernel<24, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        case 32: hipLaunchKernelGGL((xfer_tile_kernel<32, MODE>), g, b, 0, st, a, v, ntx, nty, nitems); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_xfer_tile(const XferTileArgs& a, hipStream_t st) {
    return launch_xfer_tile_mode<0>(a, XferVArgs{}, st);
}

hipError_t launch_xfer_tile_v(const XferTileArgs& a, const XferVArgs& v, bool adjoint, hipStream_t st) {
    if (!v.lo || !v.cnt || !v.r0 || !v.w || v.kv < 1) return hipErrorInvalidValue;
    // 32-bit offsets inside a row of analysis points
    const long long npts = adjoint ? a.nin_x : a.nout_x;
    if (npts * v.kv * 4 >= (1ll << 31)) return hipErrorInvalidValue;
    return adjoint ? launch_xfer_tile_mode<2>(a, v, st) : launch_xfer_tile_mode<1>(a, v, st);
}

hipError_t launch_kwin(const float* in, float* out, int kin, int kout, long long npts, const int* ks,
                       const float* kw, int w, hipStream_t st) {
    if (w < 1) return hipErrorInvalidValue;
    const int nkc = (kout + kWave - 1) / kWave;
    const long long nitems = (long long)nkc * ((npts + kWinPoints - 1) / kWinPoints);
    const long long nblocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock;
    if (nblocks >= (1ll << 31)) return hipErrorInvalidValue;
    const dim3 g((unsigned)nblocks), b(kBlock);
    if (w <= 4)
        hipLaunchKernelGGL(kwin_kernel<4>, g, b, 0, st, in, out, kin, kout, npts, ks, kw, w, nkc, nitems);
    else if (w <= kWinMaxWidth)
        hipLaunchKernelGGL(kwin_kernel<kWinMaxWidth>, g, b, 0, st, in, out, kin, kout, npts, ks, kw, w, nkc,
                           nitems);
    else
        hipLaunchKernelGGL(kwin_kernel<0>, g, b, 0, st, in, out, kin, kout, npts, ks, kw, w, nkc, nitems);
    return hipGetLastError();
}

hipError_t launch_fill(float* p, float v, long long count, hipStream_t st) {
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for(count)), dim3(kBlock), 0, st, p, v, count);
    return hipGetLastError();
}

hipError_t launch_dot(const float* a, const float* b, long long count, double* acc,
                      hipStream_t st) {
    double* partial = acc + 1;
    const bool vec = ((reinterpret_cast<size_t>(a) | reinterpret_cast<size_t>(b)) & 15) == 0;
    if (vec)
        hipLaunchKernelGGL(dot_partial_kernel<true>, dim3(kDotBlocks), dim3(kBlock), 0, st, a, b, count, partial);
    else
        hipLaunchKernelGGL(dot_partial_kernel<false>, dim3(kDotBlocks), dim3(kBlock), 0, st, a, b, count, partial);
    hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kBlock), 0, st, partial, kDotBlocks, acc);
    return hipGetLastError();
}

}  // namespace mgbf
