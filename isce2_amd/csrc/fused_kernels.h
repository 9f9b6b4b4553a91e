// Building blocks of the fused per-window kernels (fused.hip): one workgroup
// of NT threads per window keeps the window's chips, spectra and surfaces in
// LDS; every FFT transforms all rows (or columns) of a chip at once in place.
//
// Correlations use row FFTs of length L >= search width plus a direct sum over
// template rows per frequency bin:
//   c[u,v] = (1/L) IFFT_L( sum_i conj(T_i) S_{i+u} )[v]
// which equals the reference's zero-padded 2-D FFT correlation
// (cuCorrFrequency.cu:63-79) at every valid lag.
#pragma once
#include <cfloat>
#include "cx.h"
#include "fft_inplace.h"

namespace ampcor {
namespace fused {

constexpr int NT = 512;   // threads per workgroup (8 wave64)

using cf = cx<float>;

// one pixel as loaded (real images: (value, 0)), and its amplitude
__device__ __forceinline__ float2 pixel_raw(const void *img, int mode, int64_t off) {
    if (mode == 2) return {static_cast<const float *>(img)[off], 0.f};
    return static_cast<const float2 *>(img)[off];
}

__device__ __forceinline__ float raw_amp(float2 z, int mode) {
    return mode == 2 ? fabsf(z.x) : fast_sqrt(z.x * z.x + z.y * z.y);
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
// b % 8), each with its own L2. Giving every XCD a contiguous run of windows
// keeps neighbouring windows, whose chips overlap in the image, in one L2.
__device__ __forceinline__ int xcd_window(int b, int n) {
    const int x = b & 7, j = b >> 3;
    const int q = n >> 3, r = n & 7;     // XCD x runs q + (x < r) of the n blocks
    return x * q + min(x, r) + j;
}

// FP64 workgroup sum over NTH threads; `sh` holds NTH/64 doubles
template <int NTH = NT>
__device__ __forceinline__ double block_sum(double v, double *sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NTH / 64; ++i) s += sh[i];
    __syncthreads();
    return s;
}

// ---------------------------------------------------------------------------
// Normalization factors 1/sqrt(x) of n lags in LDS, and the normalized value of a lag sum
// c / L. The cancellation in x is resolved in FP64 either way.
// Norms32: the hardware's reciprocal square root (within 1 ulp) of the FP32 value.
// Norms48: the FP64 one, held as a float and the upper half of the float that is left over
// (2^-32 of the factor), and one rounding of an FP64 product, for the surfaces whose calls
// in automatic mode had been the staged pipeline's, which divides in FP64: x, two sums of
// squares multiplied, leaves FP32's range where amplitudes reach about 1e7. Six bytes a
// factor keep two workgroups a CU at window 64, half search 20 (81.6 KB each): 3,844 windows
// at factor 32 take 1.13 ms, with FP64 factors (84.9 KB) 1.37 ms, with Norms32 1.12 ms.
// ---------------------------------------------------------------------------
struct Norms32 {
    static constexpr int BYTES = 4;
    static constexpr bool WIDE = false;
    float *p;
    __device__ Norms32(void *lds, int) : p(static_cast<float *>(lds)) {}
    __device__ __forceinline__ void put(int i, double x) const { p[i] = __builtin_amdgcn_rsqf(float(x)); }
    template <int L> __device__ __forceinline__ float normalized(float c, int i) const { return c * (1.0f / float(L)) * p[i]; }
};
struct Norms48 {
    static constexpr int BYTES = 6;
    static constexpr bool WIDE = true;       // the kernel's other FP64 steps come with it
    float *hi;
    uint16_t *lo;
    __device__ Norms48(void *lds, int n) : hi(static_cast<float *>(lds)), lo(reinterpret_cast<uint16_t *>(hi + n)) {}
    __device__ __forceinline__ void put(int i, double x) const {
        double r = __builtin_amdgcn_rsq(x);              // one Newton step to FP64
        r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
        const float h = float(r);
        hi[i] = h;
        lo[i] = uint16_t(__float_as_uint(float((r - double(h)) * 0x1p24)) >> 16);   // scaled: normal wherever h is
    }
    template <int L> __device__ __forceinline__ float normalized(float c, int i) const {
        const double r = fma(double(__uint_as_float(uint32_t(lo[i]) << 16)), 0x1p-24, double(hi[i]));
        return float(double(c) * r * (1.0 / L));
    }
};

// ---------------------------------------------------------------------------
// FP64 window sums -> nrm[u][v] = 1/sqrt((s2 - s1^2/n) t2 + FLT_EPSILON)
// (cuCorrNormalization.cu:230-314, cuCorrNormalizationSAT.cu:237-240).
// Vertical sums of s and s^2 over the first TH rows of every column come from
// NB row blocks summed by all threads at once (`part`: 2*NB*SW doubles of
// scratch); each wave then slides them down to its first lag row, and walks
// its contiguous lag rows with the horizontal window sums taken as differences
// of wave prefix scans (lanes own columns, CPL per lane; the scans run on DPP
// row shifts and row broadcasts, so they are VALU work with no LDS round trip).
// One barrier, which every thread of the workgroup must reach.
// ---------------------------------------------------------------------------
constexpr int NORM_BLOCKS = 4;

// Lag-row phase of window_norms: part holds, for NB row blocks, the column sums
// of s ([b][SW]) then of s^2 ([NB + b][SW]). With blk = 0 the blocks cover rows
// [0, TH) and every wave slides its window down from row 0; with blk > 0 they
// are blocks of blk rows from row 0 down the whole search (TH a multiple of
// blk), and a wave starts from the TH / blk blocks at or above its first lag
// row, sliding at most blk - 1 rows. amp(r, c) is read for the slides only.
//
// Horizontal window sums of the column sums g (lane l holds columns l + 64m):
// * TWB = 0 (any TW): differences of the wave prefix over all SW columns,
//   read across lanes;
// * TWB = TW / 64 > 0: window(v) = sum_{c<TW} g[c] + sum_{j<v} (g[j+TW] - g[j]),
//   and column j + TW sits in the same lane as column j, so each 64-column
//   block of lag columns costs one wave scan of the differences plus one wave
//   sum of the first TW columns per lag row, with no value read across lanes.
template <int CPL, int NTH, int TWB = 0, class Amp, class Norms>
__device__ __forceinline__ void window_norms_rows(Amp amp, const double *part, int NB, int SW, int TH, int TW,
                                                  int NLh, int NLw, double t2, Norms nrm, int blk = 0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int NW = NTH / 64;
    const int per = (NLh + NW - 1) / NW;
    const int u_beg = wave * per, u_end = min(NLh, u_beg + per);
    if (u_beg >= u_end) return;
    const int b_lo = blk ? u_beg / blk : 0, nb = blk ? TH / blk : NB;
    double g1[CPL], g2[CPL];
#pragma unroll
    for (int m = 0; m < CPL; ++m) {
        g1[m] = 0.0; g2[m] = 0.0;
        const int c = lane + 64 * m;
        if (c < SW) {
            for (int b = b_lo; b < b_lo + nb; ++b) {
                g1[m] += part[b * SW + c];
                g2[m] += part[(NB + b) * SW + c];
            }
            // slide down to u_beg (two independent chains)
            double d1 = 0.0, d2 = 0.0, e1 = 0.0, e2 = 0.0;
            int u = b_lo * blk;
#pragma unroll 2
            for (; u + 1 < u_beg; u += 2) {
                const double vn = amp(u + TH, c), vo = amp(u, c);
                const double wn = amp(u + 1 + TH, c), wo = amp(u + 1, c);
                d1 += vn - vo; d2 += vn * vn - vo * vo;
                e1 += wn - wo; e2 += wn * wn - wo * wo;
            }
            if (u < u_beg) {
                const double vn = amp(u + TH, c), vo = amp(u, c);
                d1 += vn - vo; d2 += vn * vn - vo * vo;
            }
            g1[m] += d1 + e1;
            g2[m] += d2 + e2;
        }
    }
    const double inv_n = 1.0 / double(TH * TW);
    #pragma unroll 1
    for (int u = u_beg; u < u_end; ++u) {
        if constexpr (TWB > 0) {
            static_assert(TWB < CPL, "lanes hold a column beyond the first TW");
            double e1 = g1[0], e2 = g2[0];
#pragma unroll
            for (int m = 1; m < TWB; ++m) { e1 += g1[m]; e2 += g2[m]; }
            double c1 = lane63_f64(wave_scan_f64(e1)), c2 = lane63_f64(wave_scan_f64(e2));
#pragma unroll
            for (int k = 0; k + TWB <= CPL; ++k) {
                if (64 * k >= NLw) break;
                const double h1 = k + TWB < CPL ? g1[k + TWB] : 0.0, h2 = k + TWB < CPL ? g2[k + TWB] : 0.0;
                const double d1 = h1 - g1[k], d2 = h2 - g2[k];
                const double x1 = wave_scan_f64(d1), x2 = wave_scan_f64(d2);
                const int v = lane + 64 * k;
                if (v < NLw) {
                    const double s1 = c1 + (x1 - d1), s2 = c2 + (x2 - d2);
                    const double norm2 = (s2 - s1 * s1 * inv_n) * t2;
                    nrm.put(u * NLw + v, norm2 + double(FLT_EPSILON));
                }
                c1 += lane63_f64(x1);
                c2 += lane63_f64(x2);
            }
        } else {
        double p1[CPL], p2[CPL];
        double c1 = 0.0, c2 = 0.0;
#pragma unroll
        for (int m = 0; m < CPL; ++m) {
            const double x1 = wave_scan_f64(g1[m]) + c1, x2 = wave_scan_f64(g2[m]) + c2;
            p1[m] = x1; p2[m] = x2;
            c1 = lane63_f64(x1);
            c2 = lane63_f64(x2);
        }
        #pragma unroll 1
        for (int k = 0; k * 64 < NLw; ++k) {
            const int v = lane + 64 * k;
            const int hi = min(v + TW - 1, SW - 1), lo = v - 1;
            double ph1 = 0, ph2 = 0, pl1 = 0, pl2 = 0;
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                const double a1 = __shfl(p1[m], hi & 63), a2 = __shfl(p2[m], hi & 63);
                const double b1 = __shfl(p1[m], lo & 63), b2 = __shfl(p2[m], lo & 63);
                if ((hi >> 6) == m) { ph1 = a1; ph2 = a2; }
                if (lo >= 0 && (lo >> 6) == m) { pl1 = b1; pl2 = b2; }
            }
            if (v < NLw) {
                const double s1 = ph1 - pl1, s2 = ph2 - pl2;
                const double norm2 = (s2 - s1 * s1 * inv_n) * t2;
                nrm.put(u * NLw + v, norm2 + double(FLT_EPSILON));
            }
        }
        }
        if (u + 1 < u_end) {
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                const int c = lane + 64 * m;
                if (c < SW) {
                    const double vn = amp(u + TH, c), vo = amp(u, c);
                    g1[m] += vn - vo;
                    g2[m] += vn * vn - vo * vo;
                }
            }
        }
    }
}

// Window sums from column sums of row blocks covering the whole search height
// (SH rows, blocks of NORM_BLK rows; part holds 2 * ceil(SH / NORM_BLK) * SW
// doubles), so that no wave slides far to its first lag row. TH must be a
// multiple of NORM_BLK.
constexpr int NORM_BLK = 16;
template <int CPL, int NTH = NT, int TWB = 0, class Amp, class Norms>
__device__ __forceinline__ void window_norms_blk(Amp amp, int SH, int SW, int TH, int TW, int NLh, int NLw,
                                                 double t2, Norms nrm, double *part) {
    const int NB = (SH + NORM_BLK - 1) / NORM_BLK;
    #pragma unroll 1
    for (int t = threadIdx.x; t < NB * SW; t += NTH) {
        const int b = t / SW, c = t - b * SW;
        const int r0 = b * NORM_BLK, r1 = min(SH, r0 + NORM_BLK);
        double a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
        int r = r0;
        for (; r + 1 < r1; r += 2) {
            const double x = amp(r, c), y = amp(r + 1, c);
            a1 += x; a2 += x * x;
            b1 += y; b2 += y * y;
        }
        if (r < r1) {
            const double x = amp(r, c);
            a1 += x; a2 += x * x;
        }
        part[b * SW + c] = a1 + b1;
        part[(NB + b) * SW + c] = a2 + b2;
    }
    __syncthreads();
    window_norms_rows<CPL, NTH, TWB>(amp, part, NB, SW, TH, TW, NLh, NLw, t2, nrm, NORM_BLK);
}

template <int CPL, int NTH = NT, int TWB = 0, class Amp, class Norms>
__device__ __forceinline__ void window_norms(Amp amp, int SW, int TH, int TW, int NLh, int NLw, double t2, Norms nrm,
                             double *part) {
    constexpr int NB = NORM_BLOCKS;
    const int rows_per = (TH + NB - 1) / NB;
    #pragma unroll 1
    for (int t = threadIdx.x; t < NB * SW; t += NTH) {
        const int b = t / SW, c = t - b * SW;
        const int r0 = b * rows_per, r1 = min(TH, r0 + rows_per);
        double a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
        int r = r0;
        for (; r + 1 < r1; r += 2) {
            const double x = amp(r, c), y = amp(r + 1, c);
            a1 += x; a2 += x * x;
            b1 += y; b2 += y * y;
        }
        if (r < r1) {
            const double x = amp(r, c);
            a1 += x; a2 += x * x;
        }
        part[b * SW + c] = a1 + b1;
        part[(NB + b) * SW + c] = a2 + b2;
    }
    __syncthreads();
    window_norms_rows<CPL, NTH, TWB>(amp, part, NB, SW, TH, TW, NLh, NLw, t2, nrm);
}

// ---------------------------------------------------------------------------
// In-place split of packed real-pair spectra. Signal j (pitch P) holds
// Z = FFT(a + i b) in digit-reversed order (fft_nat2dr); afterwards slots
// [0, H) hold A_k (row 2j) and [H, 2H) hold B_k (row 2j+1), k < H = L/2, with
// slot 0 = (DC, Nyquist) of that row. A round covers whole signals only: the
// reads of signal j (bins k and L-k) must all happen before any write to j.
// ---------------------------------------------------------------------------
template <int R1, int R2, int NTH = NT, int U = 4>
__device__ __forceinline__ void split_pairs_inplace(cf *buf, int nsig, int P) {
    constexpr int L = R1 * R2, H = L / 2;
    // each thread keeps one bin for the whole call (its storage indices computed
    // once): bins 1..H-1 on the first SPR (H-1) threads, bin 0 on the next SPR,
    // so only the wave that holds the bin-0 threads takes both paths; a round
    // covers U SPR whole signals
    constexpr int SPR = NTH / H, NG = SPR * (H - 1);
    static_assert(SPR >= 1, "a pass must hold at least one signal");
    const int t = threadIdx.x;
    const bool gen = t < NG, act = t < NG + SPR;
    const int jj = gen ? t / (H - 1) : t - NG;
    const int k = gen ? 1 + t % (H - 1) : 0;
    const int pk = dr_pos<R1, R2>(k), pc = dr_pos<R1, R2>(gen ? L - k : H);
    #pragma unroll 1
    for (int j0 = 0; j0 < nsig; j0 += U * SPR) {
        cf av[U], bv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = j0 + jj + u * SPR;
            if (act && j < nsig) {
                const cf *z = buf + j * P;
                const cf zk = z[pk], zp = z[pc];
                if (gen) {
                    const cf zc = conj(zp);
                    av[u] = (zk + zc) * 0.5f;
                    const cf d = (zk - zc) * 0.5f;
                    bv[u] = {d.y, -d.x};
                } else {
                    av[u] = {zk.x, zp.x};
                    bv[u] = {zk.y, zp.y};
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = j0 + jj + u * SPR;
            if (act && j < nsig) {
                buf[j * P + k] = av[u];
                buf[j * P + H + k] = bv[u];
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// MAC over template rows [i_beg, i_end): q[k] += conj(T_i[f]) S_{i+u0+k}[f]
// (slot 0 packs two real bins: (DC, Nyquist) multiply component-wise). Rows sit in pairs (row r at slot (r >> 1) P +
// (r & 1) H); i_beg and t_off are even and the range a multiple of 8, so a
// thread's search rows keep the parity of u0 and every load of a block is a
// fixed offset from one of two addresses. Template row i meets search row
// i + u0 + k, so a search row at or past SH meets only lags u0 + k >=
// SH - (i_end - 1), past the last lag the callers keep (SH - template height + 1
// lags), and the callers' LDS continues past their search rows: such rows are
// read without a bound check and only reach sums that are discarded.
// ---------------------------------------------------------------------------
template <int H, int K>
__device__ __forceinline__ void mac_rows(cf (&q)[K], const cf *S, int Sp, const cf *Tsp, int Tp, int t_off,
                                         int i_beg, int i_end, int u0, int SH, int f) {
    const bool dc = f == 0;
    const int p = u0 & 1;
    const int e0 = p ? H : 0, e1 = p ? Sp : H;      // slot offset of even / odd block rows
    (void)SH;
    #pragma unroll 1
    for (int i0 = i_beg; i0 < i_end; i0 += 8) {
        const cf *sb = S + ((i0 + u0) >> 1) * Sp + f;
        const cf *tb = Tsp + ((i0 - t_off) >> 1) * Tp + f;
        cf sw[K + 7];
#pragma unroll
        for (int m = 0; m < K + 7; ++m) sw[m] = sb[(m >> 1) * Sp + ((m & 1) ? e1 : e0)];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const cf tv = tb[(i >> 1) * Tp + (i & 1) * H];
            // one branch-free form for every lane: conj(t) s, or for slot 0 the
            // component-wise product (t.x s.x, t.y s.y)
            const float c0 = tv.x, c1 = dc ? 0.f : tv.y, c2 = dc ? tv.y : tv.x, c3 = dc ? 0.f : -tv.y;
            // two chained FMAs per component (the accumulator is the addend)
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const cf s = sw[i + k];
                q[k].x = fmaf(c1, s.y, fmaf(c0, s.x, q[k].x));
                q[k].y = fmaf(c3, s.x, fmaf(c2, s.y, q[k].y));
            }
        }
    }
}

// mac_rows in parts of 16 template rows that are summed apart (PARTS), as the staged
// pipeline's sums are by its waves: chains of 16 and W / 16 additions for one of W (windows of
// 32, rms error of the refined offset: 1.13 times the staged pipeline's before, 0.97 now).
template <int H, int K, bool PARTS>
__device__ __forceinline__ void mac_row_parts(cf (&q)[K], const cf *S, int Sp, const cf *Tsp, int Tp, int t_off,
                                              int i_beg, int i_end, int u0, int SH, int f) {
    if constexpr (!PARTS) {
        mac_rows<H, K>(q, S, Sp, Tsp, Tp, t_off, i_beg, i_end, u0, SH, f);
    } else {
        #pragma unroll 1
        for (int i = i_beg; i < i_end; i += 16) {
            cf part[K];
#pragma unroll
            for (int k = 0; k < K; ++k) part[k] = {0.f, 0.f};
            mac_rows<H, K>(part, S, Sp, Tsp, Tp, t_off, i, i + 16, u0, SH, f);
#pragma unroll
            for (int k = 0; k < K; ++k) q[k] = q[k] + part[k];
        }
    }
}

// ---------------------------------------------------------------------------
// Lag sums on the matrix cores, for up to 17 lags and row transforms of R1 x 16 points:
// Q[u][f] = sum_i conj(T_i[f]) S_{i+u}[f]. v_mfma_f32_4x4x1_16b multiplies, in each of 16
// blocks of 4 lanes, a column of 4 values by a row of 4: here a block is one bin f, the
// column 4 template rows 4 m + a, the row 4 search rows 4 (m + d) + b, so accumulator d
// holds, for a in its registers and b in its lanes, sums for the lag 4 d + b - a. All 16
// products of a block are wanted (17 of the 20 lags of d = 0..4 for each a), a lane loads
// one template row and one search row for 20 instructions, and each of those does four
// times the work of a v_fma_f32 in 2.1 times its issue time.
// The spectra come straight from the transform of packed row pairs, Z = FFT(row 2j + i
// row 2j+1) in digit-reversed order: row 2j + p enters as w = Z_k +- conj(Z_{L-k}), which
// is 2 A for the even row and 2i B for the odd one; the factors (1/4, and +-i where the
// two rows' parities differ) are applied to the finished sums.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int LAG_D = 5;                    // blocks of 4 lags met by 4 template rows: 17 + 3 <= 20

struct LagSums {
    f32x4 re[LAG_D], im[LAG_D];
    __device__ LagSums() {
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) re[d] = im[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
};

// v, of which the compiler knows nothing: what is computed from it is computed in place
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// What a lane of R1 - 1 waves works on. Bins R1 q + c, q < 8, sit next to each other in
// digit-reversed order (storage 16 c + q; their mirrors L - k also, reversed), so a group
// of 8 bins shares c: waves 1.. take group c = wave over the two halves of a chunk's
// template rows, wave 0 the groups 0 and R1 - 1, each over both halves.
template <int R1>
struct LagLane {
    int wave, bin, pk, pc, part, halves, pair;
    float sign;
    __device__ LagLane(int w, int lane) {
        wave = __builtin_amdgcn_readfirstlane(w);
        const int blk = lane >> 2, q = blk & 7, hi = blk >> 3;
        const int c = wave ? wave : hi * (R1 - 1);
        bin = R1 * q + c;
        pk = 16 * c + q;
        pc = c ? 16 * (R1 - c) + 15 - q : (16 - q) & 15;
        part = wave ? hi : 0;
        halves = wave ? 1 : 2;
        pair = (lane >> 1) & 1;             // row a = lane & 3 of a group of 4: its pair and parity
        sign = (lane & 1) ? -1.f : 1.f;
    }
};

// acc += 4 M template rows (T; M > 0) against 4 (M + 4) search rows (S), both at the lane's first pair
template <int R1>
__device__ __forceinline__ void lag_sums(LagSums &acc, const cf *S, const cf *T, int P, int M, const LagLane<R1> &ll) {
    // pointers to bins k and L - k; the next group's values are loaded ahead of the products
    const cf *sk = S + ll.pk, *sc = S + ll.pc, *tk = T + ll.pk, *tc = T + ll.pc;
    auto row = [&](cf zk, cf zc) { return cf{fmaf(ll.sign, zc.x, zk.x), fmaf(-ll.sign, zc.y, zk.y)}; };
    cf s[LAG_D];
#pragma unroll
    for (int g = 0; g < 4; ++g) s[g] = row(sk[2 * g * P], sc[2 * g * P]);
    cf ak = sk[8 * P], ac = sc[8 * P], bk = *tk, bc = *tc;
    #pragma unroll 4
    for (int m = 0; m < M; ++m) {
        s[4] = row(ak, ac);
        const cf t = row(bk, bc);
        const float nty = -t.y;
        sk += 2 * P; sc += 2 * P; tk += 2 * P; tc += 2 * P;
        if (m + 1 < M) {
            ak = sk[8 * P]; ac = sc[8 * P]; bk = *tk; bc = *tc;
        }
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            acc.re[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(t.x, s[d].x, acc.re[d], 0, 0, 0);
            acc.im[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(t.x, s[d].y, acc.im[d], 0, 0, 0);
        }
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            acc.re[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(t.y, s[d].y, acc.re[d], 0, 0, 0);
            acc.im[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(nty, s[d].x, acc.im[d], 0, 0, 0);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) s[d] = s[d + 1];
    }
}

// Nyquist bin (real, row 2j + p in component p of S/T's pair j) of TC template rows: lane
// u + NL k sums lag u over the k-th third of the rows
template <int TC, int NL>
__device__ __forceinline__ float nyquist_sums(float acc, const cf *S, const cf *T, int P, int lane) {
    static_assert(3 * NL <= 64, "three lanes a lag");
    constexpr int TH = (TC + 2) / 3;
    auto at = [&](const cf *z, int r) { return reinterpret_cast<const float *>(z + (r >> 1) * P)[r & 1]; };
    const int k = lane / NL, u = lane - k * NL;
    if (k < 3) {
#pragma unroll
        for (int i = 0; i < TH; ++i) {
            const int r = k * TH + i;
            if (r < TC) acc = fmaf(at(T, r), at(S, r + u), acc);
        }
    }
    return acc;
}

template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// finished sums -> Qs[u][f] (slot 0: DC and Nyquist): lag 4 d + b of a bin sits in lane b
// of its four after the sums of template row a have moved a lanes down
template <int H, int NL, int R1>
__device__ __forceinline__ void store_lag_sums(const LagSums &acc, float nyq, cf *Qs, const LagLane<R1> &ll, bool nyquist) {
    const int lane = threadIdx.x & 63, b = lane & 3;
    cf out[LAG_D];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        cf v[LAG_D + 1];
        const bool mixed = ((a ^ b) & 1) != 0;           // rows of different parity: times i or -i
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            const float re = acc.re[d][a], im = acc.im[d][a];
            v[d] = {mixed ? ((a & 1) ? -im : im) : re, mixed ? ((a & 1) ? re : -re) : im};
        }
        v[LAG_D] = {0.f, 0.f};
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            if (a == 0) {
                out[d] = v[d];
                continue;
            }
            const cf s = b >= a ? v[d] : v[d + 1];
            constexpr int rot[4] = {0xe4, 0x39, 0x4e, 0x93};
            out[d].x += a == 1 ? quad_perm<rot[1]>(s.x) : a == 2 ? quad_perm<rot[2]>(s.x) : quad_perm<rot[3]>(s.x);
            out[d].y += a == 1 ? quad_perm<rot[1]>(s.y) : a == 2 ? quad_perm<rot[2]>(s.y) : quad_perm<rot[3]>(s.y);
        }
    }
    if (ll.halves == 1) {                                // the other half of the rows, 32 lanes up
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            out[d].x += __shfl_xor(out[d].x, 32);
            out[d].y += __shfl_xor(out[d].y, 32);
        }
    }
    if (ll.part == 0) {
#pragma unroll
        for (int d = 0; d < LAG_D; ++d) {
            const int u = 4 * d + b;
            if (u < NL) {
                cf *q = Qs + u * H + ll.bin;
                q->x = 0.25f * out[d].x;
                if (ll.bin) q->y = 0.25f * out[d].y;
            }
        }
    }
    if (nyquist) {
        const float sum = nyq + __shfl(nyq, lane + NL) + __shfl(nyq, lane + 2 * NL);
        if (lane < NL) Qs[lane * H].y = sum;
    }
}

// Inverse of the accumulated Q[u][f] (Qs: [NLh][H]), times nrm[u][v], into corr[u][v]
// for v < NLw: lag pairs (2p, 2p+1) share one complex transform placed in Y
// (npair signals, pitch P, digit-reversed input order).
template <int R1, int R2, int NTH = NT, class Norms>
__device__ __forceinline__ void inverse_lags(const cf *Qs, int NLh, int NLw, cf *Y, int P, const cx<float> *tw, Norms nrm,
                             float *corr) {
    constexpr int L = R1 * R2, H = L / 2;
    const int npair = (NLh + 1) / 2;
    for (int i = threadIdx.x; i < npair * L; i += NTH) {
        const int p = i / L, k = i - p * L;
        const int ua = 2 * p, ub = ua + 1;
        const cf *qa = Qs + ua * H;
        const bool hb = ub < NLh;
        const cf *qb = Qs + (hb ? ub : ua) * H;
        cf y;
        if (k == 0) y = {qa[0].x, hb ? qb[0].x : 0.f};
        else if (k == H) y = {qa[0].y, hb ? qb[0].y : 0.f};
        else if (k < H) {
            const cf a = qa[k], b = hb ? qb[k] : cf{0.f, 0.f};
            y = {a.x - b.y, a.y + b.x};
        } else {
            const cf a = qa[L - k], b = hb ? qb[L - k] : cf{0.f, 0.f};
            y = {a.x + b.y, b.x - a.y};
        }
        Y[p * P + dr_pos<R1, R2>(k)] = y;
    }
    __syncthreads();
    fft_dr2nat<float, +1, R1, R2, NTH>(Y, npair, P, 1, tw);
    for (int i = threadIdx.x; i < NLh * NLw; i += NTH) {
        const int u = i / NLw, v = i - u * NLw;
        const cf y = Y[(u >> 1) * P + v];
        corr[i] = nrm.template normalized<L>((u & 1) ? y.y : y.x, i);
    }
    __syncthreads();
}

// argmax over n values in LDS with the reference tie rule
__device__ __forceinline__ Top2<float> block_argmax(const float *v, int n, double *red) {
    Top2<float> t;
    for (int i = threadIdx.x; i < n; i += NT) t.add(v[i], maxloc_key(uint32_t(i)));
    float *shv = reinterpret_cast<float *>(red + 8);
    float *shv2 = shv + 8;
    uint64_t *shk = reinterpret_cast<uint64_t *>(red + 16);
    t.reduce<NT>(shv, shv2, shk);
    return t;
}

}  // namespace fused
}  // namespace ampcor
