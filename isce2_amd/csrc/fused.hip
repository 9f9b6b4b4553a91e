// Fused per-window pipeline: the fast path for square windows of 32 or 64
// pixels with 2x raw oversampling, a 16x16 zoom surface (the reference's
// defaults) and surface oversampling by 2 to 32, by the FFT or the windowed sinc.
// Three kernels per chunk of windows: k_coarse -> k_oversample (reference chip; search
// zoom chip) -> k_fine.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>
#include "engine.h"
#include "fused_kernels.h"
#include "stage_kernels.h"

namespace ampcor {
namespace fused {

__host__ __device__ inline int al16(int x) { return (x + 15) & ~15; }

// ---------------------------------------------------------------------------
// coarse stage (cuAmpcorChunk.cpp:18-106), one workgroup per window
// ---------------------------------------------------------------------------
// template rows per spectrum chunk of the coarse stage: the window-64 layout
// then fits two workgroups per CU (77 KB of LDS each)
__host__ __device__ constexpr int coarse_tc(int W) { return W > 32 ? 32 : W; }

struct CoarseLds {
    int spec, nrm, red, tw, total, y_off, corr_off;   // bytes (spec, nrm, red, tw, total); cf units (y_off, corr_off)
    // nb: bytes of a normalization factor
    __host__ __device__ CoarseLds(int W, int L, int SH, int NLh, int NLw, int nb) {
        const int P = L + 1, H = L / 2;
        const int nS = (SH + 1) / 2, nTc = coarse_tc(W) / 2;
        y_off = (NLh * H + 1) & ~1;                   // lag spectra Q, then the inverse pairs Y
        const int npair = (NLh + 1) / 2;
        corr_off = y_off + npair * P;                 // then the normalized surface
        int cf_units = (nS + nTc) * P;                // search + one template chunk
        const int need = corr_off + (NLh * NLw + 1) / 2;
        if (need > cf_units) cf_units = need;
        spec = 0;
        nrm = al16(spec + cf_units * 8);
        red = al16(nrm + NLh * NLw * nb);
        tw = red + 32 * 8;                            // the row transform's twiddles
        total = tw + L * 8;
    }
};

struct CoarseArgs {
    const void *ref; int64_t ref_pitch;
    const void *sec; int64_t sec_pitch;
    int mode;                      // 0 complex, 1 |z| chips, 2 real image
    const int32_t *ref_d, *ref_a, *sec_d, *sec_a;
    int hs_d, hs_a, hz, patch_h, patch_w;
    int32_t *maxloc; float *maxval; int32_t *start, *shift; float *snr, *cov;
    float *margin;                 // [n] top-1 minus top-2 of the normalized surface, or null
};

struct OsArgs;
template <int R1, int R2, bool MEAN, int NTH, bool WIDE>
__device__ __forceinline__ void oversample_window(const OsArgs &a, int win);

// With an OsArgs as `os` the launch has a second workgroup a window (from n = gridDim.x / 2
// on) that oversamples its reference chip: neither reads what the other writes. For calls
// of few windows, where each stage's latency is the other's idle chip (MERGE_MAX).
template <int W, int R1, int R2, int K, class Norms, class... Os>
__global__ void __launch_bounds__(NT, (K >= 9 ? 2 : 4)) k_coarse(CoarseArgs a, const cf *tw_g, int w0, Os... os) {
    if constexpr (sizeof...(Os) > 0) {
        const int n = int(gridDim.x >> 1);
        if (int(blockIdx.x) >= n) {
            oversample_window<8, W / 8, true, NT, Norms::WIDE>(os..., w0 + int(blockIdx.x) - n);
            return;
        }
    }
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int L = R1 * R2, H = L / 2, P = L + 1, TC = coarse_tc(W), nTc = TC / 2;
    static_assert(W % TC == 0, "template chunks cover the window");
    // mac_rows reads up to K - 2 rows past the search (only discarded lags use them):
    // they land in the template chunk right after the search pairs
    static_assert(nTc >= K / 2 + 1, "the template chunk follows the search rows");
    static_assert(2 * NORM_BLOCKS * L <= nTc * P, "window-sum scratch fits the template chunk region");
    const int SH = W + 2 * a.hs_d, SW = W + 2 * a.hs_a;
    const int NLh = SH - W + 1, NLw = SW - W + 1;
    const int nS = (SH + 1) / 2;
    const CoarseLds lay(W, L, SH, NLh, NLw, Norms::BYTES);
    cf *S = reinterpret_cast<cf *>(smem + lay.spec);
    cf *Tb = S + nS * P;
    const Norms nrm(smem + lay.nrm, NLh * NLw);
    float *corr = reinterpret_cast<float *>(S + lay.corr_off);
    double *red = reinterpret_cast<double *>(smem + lay.red);
    const int win = w0 + (sizeof...(Os) > 0 ? int(blockIdx.x) : xcd_window(blockIdx.x, gridDim.x));
    // twiddles read from LDS (the transforms' table loads wait one at a time)
    cf *twl = reinterpret_cast<cf *>(smem + lay.tw);
    for (int i = threadIdx.x; i < L; i += NT) twl[i] = tw_g[i];
    const cf *tw = twl;

    // search amplitudes, row pairs packed as (row 2j, row 2j+1), and the
    // template's FP64 sum and sum of squares, gathers unrolled for memory parallelism
    const int64_t rd = a.ref_d[win], ra = a.ref_a[win];
    const int64_t sd = a.sec_d[win], sa = a.sec_a[win];
    // template pixels are requested first and held raw in registers, so that
    // their loads overlap the search chip's
    constexpr int TI = W * W / NT;
    static_assert(W * W % NT == 0, "template pixels divide evenly over the workgroup");
    static_assert(NT % L == 0 && NT % W == 0, "fixed column per thread in the gathers");
    float2 traw[TI];
#pragma unroll
    for (int k = 0; k < TI; ++k) {
        const int i = threadIdx.x + k * NT, r = i / W, x = i - r * W;
        traw[k] = pixel_raw(a.ref, a.mode, (rd + r) * a.ref_pitch + ra + x);
    }
    {
        // every thread keeps one column x of the search chip and walks its row
        // pairs with a running pointer
        const int x = threadIdx.x % L;
        const int j0 = threadIdx.x / L;
        constexpr int JS = NT / L;
        const bool in = x < SW;
        const int64_t step = int64_t(2 * JS) * a.sec_pitch;
        int64_t off = (sd + 2 * j0) * a.sec_pitch + sa + (in ? x : 0);
        auto put = [&](auto amp_at) {
#pragma unroll 4
            for (int j = j0; j < nS; j += JS, off += step) {
                cf v = {0.f, 0.f};
                if (in) {
                    v.x = amp_at(off);
                    if (2 * j + 1 < SH) v.y = amp_at(off + a.sec_pitch);
                }
                S[j * P + x] = v;
            }
        };
        if (a.mode == 2) {
            const float *img = static_cast<const float *>(a.sec);
            put([&](int64_t o) { return fabsf(img[o]); });
        } else {
            const float2 *img = static_cast<const float2 *>(a.sec);
            put([&](int64_t o) {
                const float2 z = img[o];
                return fast_sqrt(z.x * z.x + z.y * z.y);
            });
        }
    }
    // template amplitudes, held for the chunk loads below
    float tamp[TI];
    double sum = 0.0, sum2 = 0.0;
#pragma unroll
    for (int k = 0; k < TI; ++k) {
        tamp[k] = raw_amp(traw[k], a.mode);
        const double v = tamp[k];
        sum += v;
        sum2 += v * v;
    }
    sum = block_sum(sum, red);
    sum2 = block_sum(sum2, red);
    const double mean = sum / double(W * W);
    const double t2 = fmax(sum2 - sum * sum / double(W * W), 0.0);   // sum of squared deviations
    // window sums from 16-row block sums down the whole search (the template
    // chunk's region, not loaded yet, holds them: 2 * ceil(SH/16) * SW doubles)
    static_assert(W % NORM_BLK == 0, "template height a multiple of the norm block");
    static_assert(2 * ((L + NORM_BLK - 1) / NORM_BLK) * L <= nTc * P, "block sums fit the template chunk region");
    window_norms_blk<(L + 63) / 64, NT, W % 64 == 0 ? W / 64 : 0>(
        [&](int r, int c) -> double { return reinterpret_cast<const float *>(S)[2 * ((r >> 1) * P + c) + (r & 1)]; },
        SH, SW, W, W, NLh, NLw, t2, nrm, reinterpret_cast<double *>(Tb));
    __syncthreads();

    const int f = threadIdx.x % H, blk = threadIdx.x / H, u0 = blk * K;
    const bool active = (blk < NT / H) && (u0 < NLh);
    cf q[K];
#pragma unroll
    for (int k = 0; k < K; ++k) q[k] = {0.f, 0.f};
    #pragma unroll 1
    for (int c0 = 0; c0 < W; c0 += TC) {
        // template rows [c0, c0 + TC) minus the FP64 mean, packed in pairs, from
        // the amplitudes held in registers; zero beyond column W
#pragma unroll
        for (int k = 0; k < TI; ++k) {
            const int i = threadIdx.x + k * NT, r = i / W, x = i - r * W;
            if (r >= c0 && r < c0 + TC) {
                float *slot = reinterpret_cast<float *>(Tb + ((r - c0) >> 1) * P + x) + (r & 1);
                *slot = float(double(tamp[k]) - mean);
            }
        }
        for (int i = threadIdx.x; i < nTc * (L - W); i += NT) {
            const int j = i / (L - W), x = W + i - j * (L - W);
            Tb[j * P + x] = cf{0.f, 0.f};
        }
        __syncthreads();
        if (c0 == 0) {
            // row spectra of the search and of the first template chunk in one pass
            fft_nat2dr<float, -1, R1, R2, NT>(S, nS + nTc, P, 1, tw);
            split_pairs_inplace<R1, R2>(S, nS + nTc, P);
        } else {
            fft_nat2dr<float, -1, R1, R2, NT>(Tb, nTc, P, 1, tw);
            split_pairs_inplace<R1, R2>(Tb, nTc, P);
        }
        if (active) mac_row_parts<H, K, Norms::WIDE>(q, S, P, Tb, P, c0, c0, c0 + TC, u0, SH, f);
        __syncthreads();
    }
    cf *Qs = S;
    if (active) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (u0 + k < NLh) Qs[(u0 + k) * H + f] = q[k];
    }
    __syncthreads();
    inverse_lags<R1, R2>(Qs, NLh, NLw, S + lay.y_off, P, tw, nrm, corr);

    const Top2<float> top = block_argmax(corr, NLh * NLw, red);
    const int idx = top.index();
    const float val = top.v1;
    const int px = idx / NLw, py = idx - px * NLw;
    if (threadIdx.x < 64)      // wave 0: SNR patch sum over its lanes, covariance on lane 0
        window_stats(corr, NLh, NLw, px, py, double(val), W * W, a.patch_h, a.patch_w, a.cov + 3 * win,
                     a.snr + win);
    if (threadIdx.x == 0) {
        if (a.margin) a.margin[win] = top.margin();
        int s0, h0, s1, h1;
        adjust_axis(px, a.hs_d, a.hz, s0, h0);
        adjust_axis(py, a.hs_a, a.hz, s1, h1);
        a.maxloc[2 * win] = px; a.maxloc[2 * win + 1] = py;
        a.maxval[win] = val;
        a.start[2 * win] = s0; a.start[2 * win + 1] = s1;
        a.shift[2 * win] = h0; a.shift[2 * win + 1] = h1;
    }
}

// ---------------------------------------------------------------------------
// Covariance of the coarse peak from the images: the normalized correlation at the peak
// and its eight neighbours, as FP64 sums over the window (the formula divides second
// differences of the surface, whose FP32 rounding it can magnify tenfold and more, by
// another rounding in each pipeline). Run for the surfaces that reach the fused kernels
// in automatic mode only, where the staged pipeline's rounding had been the result's.
// One 128-thread workgroup per window; a thread keeps a column and walks its rows, three
// columns and rows of the neighbourhood in registers, the next row's loads in flight.
// Bound by its FP64 sums (17 a pixel; more waves a window would repeat the reductions).
// ---------------------------------------------------------------------------
constexpr int COV_NT = 128;
template <int W>
__global__ void __launch_bounds__(COV_NT) k_peak_cov(CoarseArgs a, int w0) {
    constexpr int RP = W * W / COV_NT, NW = COV_NT / 64, NV = 29;   // rows per thread; t, t^2, then s, s^2, t s per lag
    __shared__ double part[NW][NV];
    const int win = w0 + blockIdx.x;
    const int px = a.maxloc[2 * win], py = a.maxloc[2 * win + 1];
    const int NLh = 2 * a.hs_d + 1, NLw = 2 * a.hs_a + 1;
    if (px < 1 || py < 1 || px + 1 >= NLh || py + 1 >= NLw) return;     // the coarse kernel's sentinel stands
    const int c = threadIdx.x % W, r0 = (threadIdx.x / W) * RP;
    const int64_t t0 = (int64_t(a.ref_d[win]) + r0) * a.ref_pitch + a.ref_a[win] + c;
    const int64_t s0 = (int64_t(a.sec_d[win]) + px - 1 + r0) * a.sec_pitch + a.sec_a[win] + py - 1 + c;
    double st = 0.0, stt = 0.0, ts[3][3], s1[3], s2[3], s[3][3], head[2][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        s1[j] = s2[j] = 0.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) ts[i][j] = 0.0;
    }
    auto walk = [&](auto load) {
        auto amp = [&](float2 z) { return double(raw_amp(z, a.mode)); };
        float2 nt, ns[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            s[0][j] = head[0][j] = amp(load(a.sec, s0 + j));
            s[1][j] = head[1][j] = amp(load(a.sec, s0 + a.sec_pitch + j));
            ns[j] = load(a.sec, s0 + 2 * a.sec_pitch + j);
        }
        nt = load(a.ref, t0);
        #pragma unroll 2
        for (int r = 0; r < RP; ++r) {
            const double t = amp(nt);
#pragma unroll
            for (int j = 0; j < 3; ++j) s[2][j] = amp(ns[j]);
            if (r + 1 < RP) {
                nt = load(a.ref, t0 + (r + 1) * a.ref_pitch);
#pragma unroll
                for (int j = 0; j < 3; ++j) ns[j] = load(a.sec, s0 + (r + 3) * a.sec_pitch + j);
            }
            st += t;
            stt = fma(t, t, stt);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                s1[j] += s[0][j];
                s2[j] = fma(s[0][j], s[0][j], s2[j]);
#pragma unroll
                for (int i = 0; i < 3; ++i) ts[i][j] = fma(t, s[i][j], ts[i][j]);
                s[0][j] = s[1][j];
                s[1][j] = s[2][j];
            }
        }
    };
    if (a.mode == 2) walk([](const void *img, int64_t o) { return float2{static_cast<const float *>(img)[o], 0.f}; });
    else walk([](const void *img, int64_t o) { return static_cast<const float2 *>(img)[o]; });
    auto put = [&](int i, double v) {
        v = wave_scan_f64(v);
        if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6][i] = v;
    };
    put(0, st);
    put(1, stt);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        // sums of the rows one and two further down, from the first two rows and the last
        // two, which are left in s[0] and s[1]
        double a1 = s1[j], a2 = s2[j];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            put(2 + 3 * (3 * i + j), a1);
            put(3 + 3 * (3 * i + j), a2);
            put(4 + 3 * (3 * i + j), ts[i][j]);
            if (i < 2) {
                a1 += s[i][j] - head[i][j];
                a2 += s[i][j] * s[i][j] - head[i][j] * head[i][j];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x >= 9) return;
    auto total = [&](int i) {
        double v = 0.0;
        for (int w = 0; w < NW; ++w) v += part[w][i];
        return v;
    };
    const int k = threadIdx.x;
    const double n = double(W * W), tt = total(0), t2 = fmax(total(1) - tt * tt / n, 0.0);
    const double q1 = total(2 + 3 * k), q2 = total(3 + 3 * k), qt = total(4 + 3 * k);
    const double ncc = (qt - tt * q1 / n) / sqrt((q2 - q1 * q1 / n) * t2 + double(FLT_EPSILON));
    double v[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) v[i] = __shfl(ncc, i);
    if (k == 0)
        peak_covariance([&](int dx, int dy) { return v[3 * (dx + 1) + dy + 1]; }, true, v[4], W * W, a.cov + 3 * win);
}

// ---------------------------------------------------------------------------
// x2 chip oversampling (cuOverSampler.cpp:72-78, cuArraysPadding.cu:59-103,
// cuDeramp.cu:67-148): per axis, odd samples = (1/N) FFT_-(FFT_+(x) e^{-i pi k_s/N}),
// even samples = x. Output pixel (2r+p, 2c+q) comes from:
//   p=0,q=0: X;  p=1,q=0: columns of X interpolated;
//   p=0,q=1: Y = rows of X interpolated;  p=1,q=1: columns of Y interpolated.
// One N x N complex chip lives in LDS (so several workgroups share a CU) and each
// thread keeps its pixels of X in registers, from which X is written a second time
// after its columns have been interpolated in place. |.| goes to HBM from the
// registers that hold each value on its way: X's as it is loaded, Y's as its columns
// are first read, the others' as their last pass ends.
// Bound by vector instructions (about 12.2k a window at N = 64, 17k at N = 72, deramped)
// and LDS round trips, three an interpolation (fft_half_sample). 31,248 windows of 64:
// reference chips (N = 64) 1516 -> 822 us, search chips (N = 72) 1661 -> 1118 us against
// the form with four passes, two gathers and separate amplitude passes; the same
// interpolations as products with the half-sample matrix on v_mfma_f32_16x16x4_f32,
// which shares the vector ALU's throughput here: 902 and 1596 us.
// ---------------------------------------------------------------------------
struct OsArgs {
    const void *img; int64_t pitch; int mode;
    const int32_t *sd, *sa, *start;   // start may be null
    int deramp;
    const cf *tw, *shift;             // [N] e^{-2 pi i k/N}, e^{-i pi k_s/N} / N
    float *out;                       // [n][4][N][N]: pixel (2r+p, 2c+q) in plane 2p+q at (r, c)
    double *mean;                     // [n][2]: mean and sum of squared deviations of |.| (MEAN kernels)
};

// chip (pitch N+1), deramp row/column rotation factors, reduction scratch, twiddles, shifts
__host__ __device__ inline int os_lds_bytes(int N, bool wide) {
    return al16(N * (N + 1) * 8) + 2 * N * (wide ? 16 : 8) + 32 * 8 + 2 * N * 8;
}

// threads per workgroup, and waves per SIMD to fit its registers to: as many as the LDS
// of the workgroups that share a CU leaves room for (four of N = 64, three of N = 72)
__host__ __device__ constexpr int os_threads(int N) { return N >= 64 ? 512 : N == 40 ? 320 : 256; }

// WIDE: the deramp's factors and rotation in FP64 (deramp_apply), as the staged pipeline has
// them, for the surfaces whose calls in automatic mode had been its (Norms48)
template <int R1, int R2, bool MEAN, int NTH, bool WIDE>
__device__ __forceinline__ void oversample_window(const OsArgs &a, int win) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int N = R1 * R2, PC = N + 1, NW = NTH / 64;
    static_assert(2 * N <= NTH, "one thread per deramp row and column factor");
    static_assert(4 * NW <= 32, "wave sums fit the reduction scratch");
    cf *C = reinterpret_cast<cf *>(smem);
    using F = std::conditional_t<WIDE, double, float>;
    cx<F> *rowf = reinterpret_cast<cx<F> *>(smem + al16(N * PC * 8));     // e^{i r phy}
    cx<F> *colf = rowf + N;                                               // e^{i c phx}
    double *red = reinterpret_cast<double *>(colf + N);
    cf *twl = reinterpret_cast<cf *>(red + 32), *shl = twl + N;           // twiddles and shifts, read from LDS
    if (threadIdx.x < N) {
        twl[threadIdx.x] = a.tw[threadIdx.x];
        shl[threadIdx.x] = a.shift[threadIdx.x];
    }
    int64_t r0 = a.sd[win], c0 = a.sa[win];
    if (a.start) { r0 += a.start[2 * win]; c0 += a.start[2 * win + 1]; }
    // a thread keeps one chip column and RP consecutive rows of it in registers; where the
    // workgroup is not whole columns of RP pixels, its last threads repeat rows of others
    // (the same values to the same places: no access needs a condition), and only the
    // phase sums leave the repeated rows out (k < first)
    constexpr int GR = NTH / N, RP = (N + GR - 1) / GR;
    constexpr bool EXACT = GR * N == NTH && GR * RP == N;
    static_assert(EXACT || !MEAN, "the amplitude sums count every row once");
    const int c = threadIdx.x % N, grp = threadIdx.x / N, rb = EXACT ? grp * RP : min(grp * RP, N - RP);
    const int first = EXACT ? 0 : (grp < GR ? grp * RP - rb : RP);
    cf z[RP];
    {
        auto load = [&](auto pixel) {
            const int64_t off = (r0 + rb) * a.pitch + c0 + c;
#pragma unroll
            for (int k = 0; k < RP; ++k) z[k] = pixel(off + k * a.pitch);
        };
        if (a.mode == 2) load([&](int64_t o) { return cf{static_cast<const float *>(a.img)[o], 0.f}; });
        else load([&](int64_t o) { return static_cast<const cf *>(a.img)[o]; });
        if (a.mode == 1)
#pragma unroll
            for (int k = 0; k < RP; ++k) z[k] = {fast_sqrt(z[k].x * z[k].x + z[k].y * z[k].y), 0.f};
    }
    float *out = a.out + size_t(win) * 4 * N * N;
    double s1 = 0.0, s2 = 0.0;           // FP64 sums of |.| and |.|^2 (MEAN)
    auto add = [&](float v) {
        if (MEAN) {
            s1 += v;
            s2 += double(v) * v;
        }
    };
    cf *own = C + rb * PC + c;
    if (a.deramp == 1) {
#pragma unroll
        for (int k = 0; k < RP; ++k) own[k * PC] = z[k];
        __syncthreads();
        // FP64 sums of z conj(right neighbour) and z conj(neighbour below): the one to the
        // right comes from LDS, the one below is the thread's own next pixel
        double t[4] = {0.0, 0.0, 0.0, 0.0};
        // (neighbours past the last column or row count as zero)
        const bool right = c < N - 1, below = rb + RP < N;
        double zr = z[0].x, zi = z[0].y;
#pragma unroll
        for (int k = 0; k < RP; ++k) {
            const bool once = EXACT || k >= first;
            const cf w = own[k * PC + 1], d = k + 1 < RP ? z[(k + 1) % RP] : own[(below ? k + 1 : k) * PC];
            const double br = right && once ? w.x : 0.f, bi = right && once ? w.y : 0.f;
            t[0] += zr * br + zi * bi; t[1] += zi * br - zr * bi;
            const bool dn = once && (k + 1 < RP || below);
            const double dr = dn ? d.x : 0.f, di = dn ? d.y : 0.f;
            t[2] += zr * dr + zi * di; t[3] += zi * dr - zr * di;
            if (EXACT) { zr = dr; zi = di; }
            else { zr = d.x; zi = d.y; }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = wave_scan_f64(t[j]);
        if ((threadIdx.x & 63) == 63)
#pragma unroll
            for (int j = 0; j < 4; ++j) red[4 * (threadIdx.x >> 6) + j] = t[j];
        __syncthreads();
        // the phase c*phx + r*phy is separable: one FP64 sincos per row (phy, from the sums to
        // the right) and per column (phx, from the sums below)
        if (threadIdx.x < 2 * N) {
            const bool row = threadIdx.x < N;
            double ar = 0.0, ai = 0.0;
#pragma unroll
            for (int w = 0; w < NTH / 64; ++w) {
                ar += red[4 * w + (row ? 0 : 2)];
                ai += red[4 * w + (row ? 1 : 3)];
            }
            const int k = row ? threadIdx.x : threadIdx.x - N;
            double sn, cs;
            sincos(double(k) * atan2(ai, ar), &sn, &cs);
            (row ? rowf : colf)[k] = {F(cs), F(sn)};
        }
        __syncthreads();
        // rotation through float2's operator*= (float2.h:71-75: the imaginary part uses the new
        // real part); the phases and their sines and cosines are FP64, the factors and the
        // rotation FP32 unless WIDE
        const cx<F> fc = colf[c];
#pragma unroll
        for (int k = 0; k < RP; ++k) {
            // read again from LDS: held through the FP64 sines, the pixels spill
            z[k] = own[k * PC];
            if constexpr (WIDE) {
                z[k] = deramp_apply(z[k], rowf[rb + k], fc);
            } else {
                const cf f = cmul(fc, rowf[rb + k]);
                const float nx = z[k].x * f.x - z[k].y * f.y;
                z[k] = {nx, z[k].y * f.x + nx * f.y};
            }
        }
    }
    // X: even rows, even columns
#pragma unroll
    for (int k = 0; k < RP; ++k) {
        const float v = fast_sqrt(z[k].x * z[k].x + z[k].y * z[k].y);
        add(v);
        out[(rb + k) * N + c] = v;
    }
    if (!EXACT && a.deramp == 1) __syncthreads();     // a repeated row has two readers above
#pragma unroll
    for (int k = 0; k < RP; ++k) own[k * PC] = z[k];
    __syncthreads();
    auto emit = [&](int plane, int r, int col, cf v) {
        const float m = fast_sqrt(v.x * v.x + v.y * v.y);
        add(m);
        out[plane * N * N + r * N + col] = m;
    };
    auto skip = [](int, int, cf) {};
    // columns of X (the registers keep X), then X again and its rows in place, then the columns of those
    fft_half_sample<float, R1, R2, NTH>(C, N, 1, PC, twl, shl, skip, [&](int s, int m, cf v) { emit(2, m, s, v); });
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RP; ++k) own[k * PC] = z[k];
    __syncthreads();
    fft_half_sample<float, R1, R2, NTH>(C, N, PC, 1, twl, shl, skip, [&](int s, int m, cf v) { C[s * PC + m] = v; });
    __syncthreads();
    fft_half_sample<float, R1, R2, NTH>(C, N, 1, PC, twl, shl, [&](int s, int m, cf v) { emit(1, m, s, v); },
                                        [&](int s, int m, cf v) { emit(3, m, s, v); });
    if (MEAN) {
        // FP64 mean and sum of squared deviations (sum2 - sum^2 / count)
        const double sum = block_sum<NTH>(s1, red), sum2 = block_sum<NTH>(s2, red);
        const double cnt = double(4 * N * N);
        if (threadIdx.x == 0) {
            a.mean[2 * win] = sum / cnt;
            a.mean[2 * win + 1] = fmax(sum2 - sum * sum / cnt, 0.0);
        }
    }
}

template <int R1, int R2, bool MEAN, bool WIDE, int NTH = os_threads(R1 * R2)>
__global__ void __launch_bounds__(NTH, R1 * R2 == 72 ? 6 : 8) k_oversample(OsArgs a, int w0) {
    oversample_window<R1, R2, MEAN, NTH, WIDE>(a, w0 + xcd_window(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------------------
// fine stage (cuAmpcorChunk.cpp:148-207): oversampled correlation, normalization,
// trim to 16x16, 16x surface interpolation (16-sparse spectrum evaluated with
// 16-point DFTs), argmax with the reference tie rule, sub-pixel offset. The
// whole template's row spectra sit in LDS next to the search's (for window 64:
// 72 + 64 packed signals of 144 bins, 158 KB), so both are transformed and
// split together and the per-bin sums run over all template rows in one pass.
// ---------------------------------------------------------------------------

// normalization factors by surface stage (fine_finish)
template <int SURF> using NormsOf = std::conditional_t<SURF == 16, Norms32, Norms48>;
// bytes of the factors of NL x NL lags, whose place the surface's column list of SO ints takes after them
__host__ __device__ constexpr int norm_bytes(int NL, int SO, int nb) { return NL * NL * nb > SO * 4 ? NL * NL * nb : SO * 4; }

// complex values the surface stage holds: G[16][SO], the 16 x 16 spectrum, e^{-2 pi i k/SO}
__host__ __device__ constexpr int surface_units(int SO) { return 16 * SO + 256 + SO; }

struct FineLds {
    int spec, tchunk, nrm, corr, red, total, y_off;
    // SO: surface side (16 x the surface oversampling factor); nb: bytes of a normalization factor
    __host__ __device__ FineLds(int P, int NL, int T, int SO, int nb) {
        const int L = P, PP = L + 1, H = L / 2;
        const int nS = P / 2;
        y_off = (NL * H + 1) & ~1;
        int s_units = nS * PP;
        const int npair = (NL + 1) / 2;
        if (y_off + npair * PP > s_units) s_units = y_off + npair * PP;
        const int t_units = (T / 2) * PP;                     // template row spectra
        spec = 0;
        tchunk = al16(s_units * 8);
        // the surface's G[16][SO], 16x16 spectrum and twiddles reuse both regions
        const int chips = tchunk + t_units * 8, surf = surface_units(SO) * 8;
        nrm = al16(chips > surf ? chips : surf);
        corr = al16(nrm + norm_bytes(NL, SO, nb));
        red = al16(corr + NL * NL * 4);
        total = red + 64 * 8;          // block sums + workgroup argmax scratch (up to 1024 threads)
    }
};

struct FineArgs {
    const float *tamp; const double *tmean;   // [n][4][T/2][T/2] planar, [n][2] (mean, sum of squared deviations)
    const float *samp;                         // [n][4][P/2][P/2] planar (k_oversample's layout)
    const int32_t *start;
    int hs_d, hs_a;
    float ratio;                               // 1/(surf_ovs*raw_ovs)
    int ovs;                                   // surface oversampling factor
    const cf *tws;                             // e^{-2 pi i k/(16 ovs)} (FFT surface)
    SincTable sinc;                            // windowed-sinc surface
    const int32_t *shift;
    int32_t *zoom_idx; float *offset;
    float *margin;                             // [n] top-1 minus top-2 of the surface, or null
    float *surf;                               // [n][16][16] trimmed surface for the FP64 refinement, or null
};

// the surface's argmax over the workgroup -> zoom index, offset, margin
template <int NTH>
__device__ __forceinline__ void fine_peak(const FineArgs &a, Top2<float> &top, int SO, double *red, int win) {
    // red: [0, 16) block sums, then NTH/64 top-1 values, runner-up values and keys
    top.reduce<NTH>(reinterpret_cast<float *>(red + 16), reinterpret_cast<float *>(red + 16) + 16,
                    reinterpret_cast<uint64_t *>(red + 32));
    if (threadIdx.x == 0) {
        const int idx = top.index();
        const int px = idx / SO, py = idx % SO;
        a.zoom_idx[2 * win] = px;
        a.zoom_idx[2 * win + 1] = py;
        a.offset[2 * win] = a.ratio * float(px) + float(a.start[2 * win]) - float(a.hs_d);
        a.offset[2 * win + 1] = a.ratio * float(py) + float(a.start[2 * win + 1]) - float(a.hs_a);
        if (a.margin) a.margin[win] = top.margin();
    }
}

// ---------------------------------------------------------------------------
// Surface stage of the fine kernels: trimmed 16x16 normalized surface (corr,
// row pitch NL) -> 16x16 +i DFT -> 16-sparse spectrum G[16][SO] -> column
// bounds -> evaluation of the kept columns with 16-point DFTs -> argmax with the
// reference tie rule -> zoom index, offset, margin. SO = 16 M for a surface
// oversampling factor M; with p = M a + b, q = M c + d and signed bins ks,
//   G[k1][M c + d]  = DFT16_k2( A[k1][k2] e^{-2 pi i d ks2/SO} )[c]
//   out[M a + b][q] = Re DFT16_k1( G[k1][q] e^{-2 pi i b ks1/SO} )[a].
// OVS: M when known at compile time, 0 to take it from the arguments (2..32).
// LDS: G (16*SO cf), abuf (256 + SO cf: the 16x16 spectrum and the twiddles),
// cols (SO ints), red (64 doubles).
// ---------------------------------------------------------------------------
template <int NTH, int OVS>
__device__ __forceinline__ void fine_surface(const FineArgs &a, const float *corr, int NL, cf *G, cf *abuf, int *cols,
                                             double *red, int win) {
    constexpr int Z = 16;
    const int M = OVS ? OVS : a.ovs, SO = 16 * M;
    // trimmed 16x16 surface -> 2-D +i DFT / 256 (cuOverSampler.cpp:141-145)
    cf *a16 = abuf;          // [16][16]
    cf *tws = abuf + 256;    // e^{-2 pi i k/SO}
    for (int i = threadIdx.x; i < Z * Z; i += NTH) {
        const int r = i / Z, c = i - r * Z;
        a16[i] = {corr[r * NL + c] * (1.0f / 256.0f), 0.f};
        if (a.surf) a.surf[size_t(win) * Z * Z + i] = corr[r * NL + c];
    }
    for (int i = threadIdx.x; i < SO; i += NTH) tws[i] = a.tws[i];
    __syncthreads();
    if (threadIdx.x < 16) {
        cf x[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) x[c] = a16[threadIdx.x * 16 + c];
        dft16<float, +1>(x);
#pragma unroll
        for (int c = 0; c < 16; ++c) a16[threadIdx.x * 16 + c] = x[c];
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        cf x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = a16[r * 16 + threadIdx.x];
        dft16<float, +1>(x);
#pragma unroll
        for (int r = 0; r < 16; ++r) a16[r * 16 + threadIdx.x] = x[r];
    }
    __syncthreads();
    // G[k1][Mc+dd] = DFT16_c( A[k1][k2] e^{-2 pi i dd ks2/SO} ), ks2 = signed k2 (|dd ks2| < SO / 2)
    if (threadIdx.x < 16 * M) {
        const int k1 = threadIdx.x / M, dd = threadIdx.x - k1 * M;
        cf x[16];
#pragma unroll
        for (int k2 = 0; k2 < 16; ++k2) {
            const int t = dd * (k2 < 8 ? k2 : k2 - 16);
            x[k2] = cmul(a16[k1 * 16 + k2], tws[t < 0 ? t + SO : t]);
        }
        dft16<float, -1>(x);
#pragma unroll
        for (int c = 0; c < 16; ++c) G[k1 * SO + M * c + dd] = x[c];
    }
    __syncthreads();
    // Column pruning. Every value of surface column q is at most
    // B_q = sum_k1 |G[k1][q]|, and the surface passes through the trimmed
    // samples, so its maximum is at least their largest value amax. A column with
    // B_q (1 + 2^-10) + 2^-11 |a|max < amax can hold neither the argmax nor any
    // value within 2^-12 |a|max of it (the slack covers FP32 rounding many times
    // over): it is skipped, which leaves the argmax, the tie rule and every
    // margin below 2^-12 |a|max unchanged. NaN bounds keep their column.
    static_assert(NTH >= 512 && OVS <= 32, "one thread per surface column for the bounds");
    constexpr int NBW = OVS ? (16 * OVS + 63) / 64 : 8;         // waves that hold columns
    float amax = -FLT_MAX, amag = 0.f;
    for (int i = threadIdx.x & 63; i < Z * Z; i += 64) {
        const float v = corr[(i / Z) * NL + (i % Z)];
        amax = fmaxf(amax, v);
        amag = fmaxf(amag, fabsf(v));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        amax = fmaxf(amax, __shfl_xor(amax, o));
        amag = fmaxf(amag, __shfl_xor(amag, o));
    }
    uint64_t *masks = reinterpret_cast<uint64_t *>(red + 48);   // ballots of the bound waves
    bool keep = false;
    if (threadIdx.x < SO) {
        float bq = 0.f;
#pragma unroll
        for (int k1 = 0; k1 < 16; ++k1) {
            const cf g = G[k1 * SO + threadIdx.x];
            bq += fast_sqrt(g.x * g.x + g.y * g.y);
        }
        keep = !(bq * (1.0f + 0x1p-10f) + 0x1p-11f * amag < amax);
    }
    const uint64_t wm = __ballot(keep);
    if (threadIdx.x < 64 * NBW && (threadIdx.x & 63) == 0) masks[threadIdx.x >> 6] = wm;
    __syncthreads();
    int ncols = 0, before = 0;
#pragma unroll
    for (int w = 0; w < NBW; ++w) {
        const int c = __popcll(masks[w]);
        if (w < (threadIdx.x >> 6)) before += c;
        ncols += c;
    }
    if (keep) cols[before + __popcll(wm & ((uint64_t(1) << (threadIdx.x & 63)) - 1))] = threadIdx.x;
    __syncthreads();
    // out[Maa+b][q] = Re DFT16_aa( G[k1][q] e^{-2 pi i b ks1/SO} ) over the kept
    // columns q; task t = (b, column list entry); running argmax
    Top2<float> top;
    #pragma unroll 1
    for (int t = threadIdx.x; t < M * ncols; t += NTH) {
        const int b = t / ncols, qq = cols[t - b * ncols];
        // times e^{-2 pi i b k/SO} for k = 1..8, its conjugate for the negative bins
        cf x[16];
        x[0] = G[qq];
#pragma unroll
        for (int k = 1; k <= 8; ++k) {
            const cf w = tws[b * k];
            if (k < 8) x[k] = cmul(G[k * SO + qq], w);
            x[16 - k] = cmul(G[(16 - k) * SO + qq], conj(w));
        }
        dft16<float, -1>(x);
#pragma unroll
        for (int aa = 0; aa < 16; ++aa) top.add_idx(x[aa].x, uint32_t((M * aa + b) * SO + qq));
    }
    fine_peak<NTH>(a, top, SO, red, win);
}

// Windowed-sinc surface (cuSincOverSampler.cu:84-195) and its peak: the values of
// the interpolated patch around the (shifted) centre, zero elsewhere, are never
// stored. LDS: R (size * 16 doubles, size = 4 ovs + 1), corr as in fine_surface.
template <int NTH>
__device__ __forceinline__ void fine_sinc(const FineArgs &a, const float *corr, int NL, double *R, double *red, int win) {
    constexpr int Z = 16;
    const int SO = Z * a.ovs;
    if (a.surf)
        for (int i = threadIdx.x; i < Z * Z; i += NTH) a.surf[size_t(win) * Z * Z + i] = corr[(i / Z) * NL + i % Z];
    Top2<float> top;
    sinc_patch_peak<NTH>([&](int x, int y) { return corr[x * NL + y]; }, Z, SO, a.shift[2 * win], a.shift[2 * win + 1], a.sinc,
                         a.ovs, 2 * a.ovs, R, 4 * a.ovs + 1, top);
    fine_peak<NTH>(a, top, SO, red, win);
}

// the surface stage by kind: SURF = 16 (FFT, factor 16), 0 (FFT, any factor of 2..32), -1 (windowed sinc)
template <int NTH, int SURF>
__device__ __forceinline__ void fine_finish(const FineArgs &a, const float *corr, int NL, cf *work, int *cols, double *red,
                                            int win) {
    if constexpr (SURF < 0) fine_sinc<NTH>(a, corr, NL, reinterpret_cast<double *>(work), red, win);
    else fine_surface<NTH, SURF>(a, corr, NL, work, work + 256 * (SURF ? SURF : a.ovs), cols, red, win);
}

// Windows of 32 (T = 64): 49.5 KB of LDS lets three workgroups share a CU, so registers
// are held to 84 (about 20 spilled around the surface's evaluation); the radix-16 pass is
// the one without twiddles, and a split round takes 36 of the 72 signals (U = 3). 15,625
// windows: 780 -> 680 us against two workgroups a CU and radices 16, 5.
template <int T, int R1, int R2, int K, int NTH, int SURF>
__global__ void __launch_bounds__(NTH, T == 64 ? 6 : 2) k_fine(FineArgs a, const cf *tw, int w0) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int P = R1 * R2, L = P, PP = L + 1, H = L / 2, nS = P / 2;
    constexpr int NL = P - T + 1;      // 17
    constexpr int Z = NL - 1;          // 16 (trimmed surface)
    static_assert(Z == 16, "fused surface stage assumes a 16x16 zoom surface");
    // mac_rows reads up to K - 2 rows past the search; the template spectra follow it
    static_assert(T / 2 >= K / 2 + 1, "the template region follows the search rows");
    constexpr int U = T == 64 ? 3 : 4;      // signals a thread splits at a time: two rounds either way
    const FineLds lay(P, NL, T, SURF > 0 ? 16 * SURF : 16 * a.ovs, NormsOf<SURF>::BYTES);
    cf *S = reinterpret_cast<cf *>(smem + lay.spec);
    cf *Tb = reinterpret_cast<cf *>(smem + lay.tchunk);
    const NormsOf<SURF> nrm(smem + lay.nrm, NL * NL);
    float *corr = reinterpret_cast<float *>(smem + lay.corr);
    double *red = reinterpret_cast<double *>(smem + lay.red);
    const int win = w0 + xcd_window(blockIdx.x, gridDim.x);
    const float *tp = a.tamp + size_t(win) * T * T;
    const float *sg = a.samp + size_t(win) * P * P;
    const double mean = a.tmean[2 * win], t2 = a.tmean[2 * win + 1];
    // the search chip's loads are all issued before any of its values is stored
    constexpr int SN = nS * L, SI = (SN + NTH - 1) / NTH;
    constexpr int TN = (T / 2) * L, TI = (TN + NTH - 1) / NTH;
    cf sv[SI], tv[TI];
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        const int i = threadIdx.x + k * NTH, j = i / L, x = i - j * L;
        // planar oversampled chip: row 2j + p, column x -> plane 2p + (x & 1), (j, x >> 1)
        const float *s0 = sg + size_t(x & 1) * (P / 2) * (P / 2) + j * (P / 2) + (x >> 1);
        if (SN % NTH == 0 || i < SN) sv[k] = {s0[0], s0[size_t(2) * (P / 2) * (P / 2)]};
    }
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        const int i = threadIdx.x + k * NTH, j = i / L, x = i - j * L;
        if (SN % NTH == 0 || i < SN) S[j * PP + x] = sv[k];
    }
    __syncthreads();
    // the template's loads go out once the search chip has arrived (they would
    // only delay it) and stay in flight through the window sums
#pragma unroll
    for (int k = 0; k < TI; ++k) {
        const int i = threadIdx.x + k * NTH, j = i / L, x = i - j * L;
        const float *t0 = tp + size_t(x & 1) * (T / 2) * (T / 2) + j * (T / 2) + (x >> 1);
        tv[k] = {0.f, 0.f};
        if ((TN % NTH == 0 || i < TN) && x < T) tv[k] = {t0[0], t0[size_t(2) * (T / 2) * (T / 2)]};
    }
    window_norms<(P + 63) / 64, NTH, T % 64 == 0 ? T / 64 : 0>(
        [&](int r, int c) -> double { return reinterpret_cast<const float *>(S)[2 * ((r >> 1) * PP + c) + (r & 1)]; },
        P, T, T, NL, NL, t2, nrm, reinterpret_cast<double *>(Tb));   // template not loaded yet
    __syncthreads();
    // template rows minus the FP64 mean, row pairs packed, zero beyond column T
#pragma unroll
    for (int k = 0; k < TI; ++k) {
        const int i = threadIdx.x + k * NTH, j = i / L, x = i - j * L;
        if (TN % NTH == 0 || i < TN)
            Tb[j * PP + x] = x < T ? cf{float(double(tv[k].x) - mean), float(double(tv[k].y) - mean)} : cf{0.f, 0.f};
    }
    __syncthreads();
    if (lay.tchunk == nS * PP * 8) {
        // search and template spectra are one evenly spaced set of signals
        fft_nat2dr<float, -1, R1, R2, NTH>(S, nS + T / 2, PP, 1, tw);
        split_pairs_inplace<R1, R2, NTH, U>(S, nS + T / 2, PP);
    } else {
        fft_nat2dr<float, -1, R1, R2, NTH>(S, nS, PP, 1, tw);
        fft_nat2dr<float, -1, R1, R2, NTH>(Tb, T / 2, PP, 1, tw);
        split_pairs_inplace<R1, R2, NTH>(S, nS, PP);
        split_pairs_inplace<R1, R2, NTH>(Tb, T / 2, PP);
    }

    const int f = threadIdx.x % H, blk = threadIdx.x / H, u0 = blk * K;
    const bool active = (blk < NTH / H) && (u0 < NL);
    cf q[K];
#pragma unroll
    for (int k = 0; k < K; ++k) q[k] = {0.f, 0.f};
    if (active) mac_row_parts<H, K, SURF != 16>(q, S, PP, Tb, PP, 0, 0, T, u0, P, f);
    __syncthreads();
    cf *Qs = S;
    if (active) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (u0 + k < NL) Qs[(u0 + k) * H + f] = q[k];
    }
    __syncthreads();
    inverse_lags<R1, R2, NTH>(Qs, NL, NL, S + lay.y_off, PP, tw, nrm, corr);

    fine_finish<NTH, SURF>(a, corr, NL, S, reinterpret_cast<int *>(smem + lay.nrm), red, win);
}

// ---------------------------------------------------------------------------
// Fine stage, streamed over template rows: the computation of k_fine with the
// template taken TC rows at a time and only the search rows those rows meet in
// LDS (TC + NL - 1 rows; the last NL - 1 carry over to the next chunk), so a
// workgroup needs ~68 KB of LDS and two share a CU. The window sums of the
// normalization come from FP64 column sums accumulated as the search rows
// arrive, with the first and last NL - 1 rows kept for the slides. The lag sums run on
// the matrix cores from the transforms of packed row pairs (lag_sums), without the pass
// that splits the pairs.
// Bound by vector and matrix issue (about 30.9k + 2.9k instructions a window, 70% of its
// time) and, with two workgroups a CU, by the waits between its short phases: of 3.1 ms
// for 31,248 windows the chip loads take 0.8, the row transforms 0.5, the lag sums 0.6,
// the normalization 0.25, the inverse 0.1 and the surface 0.45 ms. With split spectra and
// v_fma_f32 sums (40.8k instructions, 1.0 ms for split and sums): 3.4 ms.
// ---------------------------------------------------------------------------
struct Fine2Lds {
    int sr, tb, save, nrm, corr, red, tw, total;   // bytes
    __host__ __device__ Fine2Lds(int P, int NL, int TC, int SO, int nb) {
        const int PP = P + 1;
        const int srp = (TC + NL - 1 + 1) / 2, tcp = TC / 2;
        sr = 0;
        tb = sr + srp * PP * 8;                    // template pairs directly after the search pairs
        save = tb + tcp * PP * 8;
        // the surface stage reuses everything below nrm, and its column list nrm itself
        const int chips = save + 2 * (NL - 1) * P * 4, surf = surface_units(SO) * 8;
        nrm = al16(chips > surf ? chips : surf);
        corr = al16(nrm + norm_bytes(NL, SO, nb));
        red = al16(corr + NL * NL * 4);
        tw = red + 64 * 8;                         // the row transform's twiddles
        total = tw + P * 8;
    }
};

template <int T, int R1, int R2, int NTH, int TC, int SURF>
__global__ void __launch_bounds__(NTH, 4) k_fine2(FineArgs a, const cf *tw_g, int w0) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int P = R1 * R2, L = P, PP = L + 1, H = L / 2;
    constexpr int NL = P - T + 1;            // lags per axis (17)
    constexpr int NCH = T / TC;              // template chunks
    constexpr int SROWS = TC + NL - 1;       // search rows a chunk meets
    constexpr int SRP = (SROWS + 1) / 2;     // as row pairs
    constexpr int KEEP = (NL - 1) / 2;       // pairs carried to the next chunk
    constexpr int TCP = TC / 2;
    constexpr int NS = NL - 1;               // rows kept at each end for the slides
    constexpr int Q = P / 2, TQ = T / 2;     // polyphase plane sides
    static_assert(T % TC == 0 && TC % 2 == 0 && NS % 2 == 0 && NS == 16, "even chunks, 16x16 zoom surface");
    static_assert(NCH > 1 && NS <= 2 * SRP && TC + NS <= 2 * SRP, "the kept rows lie in the first and last chunks");
    static_assert(R2 == 16 && R1 == NTH / 64 + 1 && TC == 32 && NL <= 17, "LagLane's and lag_sums' shapes");
    static_assert(3 * P <= NTH, "one thread per column and row-pair phase");
    static_assert(6 * P * 8 <= (TC / 2) * (P + 1) * 8, "column-sum partials fit the template chunk region");
    const Fine2Lds lay(P, NL, TC, SURF > 0 ? 16 * SURF : 16 * a.ovs, NormsOf<SURF>::BYTES);
    cf *SR = reinterpret_cast<cf *>(smem + lay.sr);
    cf *TB = reinterpret_cast<cf *>(smem + lay.tb);
    float *save = reinterpret_cast<float *>(smem + lay.save);   // rows [0, NS) then [T, T + NS), pitch P
    const NormsOf<SURF> nrm(smem + lay.nrm, NL * NL);
    float *corr = reinterpret_cast<float *>(smem + lay.corr);
    double *red = reinterpret_cast<double *>(smem + lay.red);
    // twiddles read from LDS (the transforms' table loads wait one at a time)
    cf *twl = reinterpret_cast<cf *>(smem + lay.tw);
    for (int i = threadIdx.x; i < P; i += NTH) twl[i] = tw_g[i];
    const cf *tw = twl;
    const int win = w0 + xcd_window(blockIdx.x, gridDim.x);
    const float *tp = a.tamp + size_t(win) * T * T;
    const float *sg = a.samp + size_t(win) * P * P;
    const double mean = a.tmean[2 * win], t2 = a.tmean[2 * win + 1];
    // FP64 column sums of s and s^2 over rows [0, T): thread (column, phase)
    // takes the row pairs whose index is phase mod 3, both rows of a pair from
    // one load; the three partials are added in phase order by the window sums
    const int cs_c = threadIdx.x % P, cs_ph = threadIdx.x / P;
    double cs1 = 0.0, cs2 = 0.0;

    // bins by wave (LagLane): wave 0 keeps two groups of 8 over all the chunk's template rows, the
    // other waves one group over each half of them; the last wave adds the Nyquist sums
    LagSums lag;
    float nyq = 0.f;

    // Chip loads: search rows [c0 + 2 first, c0 + SROWS) and template rows [c0, c0 + TC) of
    // the planar chips (pixel (2j + p, 2c + q) in plane 2p + q at (j, c)), four columns of
    // one parity per work item, from 16-byte loads of both rows of a pair, all of a chunk's
    // in flight at once. Neighbouring lanes take the even and the odd columns, which halves
    // the LDS bank conflicts of the stores against eight columns a lane. (Asked for a chunk
    // ahead, the values spill: 3.5 ms, and 3.2 ms between the lag sums and the next chunk,
    // against 3.1 ms for 31,248 windows.)
    constexpr int LI = L / 4, TI = T / 4;    // work items a row pair
    static_assert(TCP * TI == NTH && (SRP - KEEP) * LI >= NTH && SRP * LI <= 2 * NTH, "items of a chunk by thread");
    struct Quad { float4 e0, e1; };
    auto fetch = [&](const float *plane, int side, int row, int x) {
        const float *b = plane + (x & 1) * side * side + row * side + 2 * (x & ~1);
        return Quad{*reinterpret_cast<const float4 *>(b), *reinterpret_cast<const float4 *>(b + 2 * side * side)};
    };
    auto put = [&](cf *pair, int x, const Quad &v) {
        cf *d = pair + 4 * (x & ~1) + (x & 1);
        d[0] = {v.e0.x, v.e1.x}; d[2] = {v.e0.y, v.e1.y}; d[4] = {v.e0.z, v.e1.z}; d[6] = {v.e0.w, v.e1.w};
    };
    #pragma unroll 1
    for (int ch = 0; ch < NCH; ++ch) {
        const int c0 = ch * TC;
        const int first = ch ? KEEP : 0;     // first pair slot loaded in this chunk
        // positions worked out in place: kept over the loop, they would be spilled
        const int tid = opaque(threadIdx.x), si1 = tid + NTH, row = ch * TCP + first;
        Quad qs1 = {};
        const Quad qs0 = fetch(sg, Q, row + tid / LI, tid % LI);
        if (si1 < (SRP - first) * LI) qs1 = fetch(sg, Q, row + si1 / LI, si1 % LI);
        const Quad qt = fetch(tp, TQ, ch * TCP + tid / TI, tid % TI);
        put(SR + (first + tid / LI) * PP, tid % LI, qs0);
        if (si1 < (SRP - first) * LI) put(SR + (first + si1 / LI) * PP, si1 % LI, qs1);
        // template rows minus the FP64 mean, zero beyond column T
        auto m = [&](float v) { return float(double(v) - mean); };
        put(TB + tid / TI * PP, tid % TI, Quad{{m(qt.e0.x), m(qt.e0.y), m(qt.e0.z), m(qt.e0.w)},
                                   {m(qt.e1.x), m(qt.e1.y), m(qt.e1.z), m(qt.e1.w)}});
        for (int i = threadIdx.x; i < TCP * (L - T); i += NTH) TB[i / (L - T) * PP + T + i % (L - T)] = cf{0.f, 0.f};
        __syncthreads();
        // column sums of the new row pairs below T (T is even: no pair straddles it)
        if (cs_ph < 3) {
            const int g0 = (c0 >> 1) + first, g1 = min((c0 >> 1) + SRP, T / 2);
            int gp = g0 + (cs_ph - g0 % 3 + 3) % 3;
            const cf *src = SR + (gp - (c0 >> 1)) * PP + cs_c;
            #pragma unroll 2
            for (; gp < g1; gp += 3, src += 3 * PP) {
                const cf pv = *src;
                const double x = pv.x, y = pv.y;
                cs1 += x + y;
                cs2 += fma(x, x, y * y);
            }
        }
        // the first NS rows (chunk 0's first NS/2 pairs) and the last NS (rows
        // [T, P), the last chunk's) kept for the slides
        if (ch == 0 || ch == NCH - 1) {
            const int pr0 = ch == 0 ? 0 : T / 2 - (c0 >> 1), sr0 = ch == 0 ? 0 : NS;
            for (int i = threadIdx.x; i < (NS / 2) * P; i += NTH) {
                const int j = i / P, c = i - j * P;
                const cf pv = SR[(pr0 + j) * PP + c];
                save[(sr0 + 2 * j) * P + c] = pv.x;
                save[(sr0 + 2 * j + 1) * P + c] = pv.y;
            }
        }
        __syncthreads();
        // row spectra of the new search pairs and the template pairs (contiguous in LDS)
        fft_nat2dr<float, -1, R1, R2, NTH>(SR + first * PP, SRP - first + TCP, PP, 1, tw);
        const LagLane<R1> ll(tid >> 6, tid & 63);
        // half `part` of the chunk is template rows [16 part, 16 part + 16)
        lag_sums(lag, SR + (8 * ll.part + ll.pair) * PP, TB + (8 * ll.part + ll.pair) * PP, PP, 4 * ll.halves, ll);
        if (ll.wave == NTH / 64 - 1) nyq = nyquist_sums<TC, NL>(nyq, SR + R2 / 2, TB + R2 / 2, PP, tid & 63);
        __syncthreads();
        if (ch + 1 < NCH) {
            // the last KEEP pairs are the next chunk's first
            for (int i = threadIdx.x; i < KEEP * PP; i += NTH) SR[i] = SR[(SRP - KEEP) * PP + i];
            __syncthreads();
        }
    }
    // the template region is free once the last chunk's sums are done
    double *part = reinterpret_cast<double *>(TB);
    if (cs_ph < 3) {
        part[cs_ph * P + cs_c] = cs1;
        part[(3 + cs_ph) * P + cs_c] = cs2;
    }
    cf *Qs = SR;
    const LagLane<R1> ll(threadIdx.x >> 6, threadIdx.x & 63);
    store_lag_sums<H, NL>(lag, nyq, Qs, ll, ll.wave == NTH / 64 - 1);
    __syncthreads();
    window_norms_rows<(P + 63) / 64, NTH, T % 64 == 0 ? T / 64 : 0>(
        [&](int r, int c) -> double { return double(r < NS ? save[r * P + c] : save[(NS + r - T) * P + c]); },
        part, 3, P, T, T, NL, NL, t2, nrm);
    inverse_lags<R1, R2, NTH>(Qs, NL, NL, SR + ((NL * H + 1) & ~1), PP, tw, nrm, corr);
    fine_finish<NTH, SURF>(a, corr, NL, SR, reinterpret_cast<int *>(smem + lay.nrm), red, win);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
int coarse_L(int SW) { return SW <= 64 ? 64 : (SW <= 128 ? 128 : 0); }
const int kK[] = {2, 3, 5, 6, 9};

int pick_k(int nl, int blocks) {
    for (int k : kK)
        if (k * blocks >= nl) return k;
    return 0;
}

// Windows up to which the reference chips' oversampling shares the coarse stage's launch:
// one window of either stage a CU. One window of 64: 121 -> 109 us a call; 14 x 14
// windows: 272 -> 255 us. (Past it the coarse stage alone fills the chip.)
constexpr int MERGE_MAX = 256;

// o: the reference chips' oversampling in the same launch, or null
template <int W, int R1, int R2, class Norms>
void launch_coarse(int K, const CoarseArgs &a, const cf *tw, const OsArgs *o, int n, int w0, size_t lds, hipStream_t st) {
    auto go = [&](auto k) {
        constexpr int KK = decltype(k)::value;
        if (o) hipLaunchKernelGGL((k_coarse<W, R1, R2, KK, Norms, OsArgs>), dim3(2 * n), dim3(NT), lds, st, a, tw, w0, *o);
        else hipLaunchKernelGGL((k_coarse<W, R1, R2, KK, Norms>), dim3(n), dim3(NT), lds, st, a, tw, w0);
    };
    switch (K) {
        case 2: go(std::integral_constant<int, 2>()); break;
        case 3: go(std::integral_constant<int, 3>()); break;
        case 5: go(std::integral_constant<int, 5>()); break;
        case 6: go(std::integral_constant<int, 6>()); break;
        default: go(std::integral_constant<int, 9>()); break;
    }
}

template <class Norms>
void launch_coarse(int W, int L, int K, const CoarseArgs &a, const cf *tw, const OsArgs *o, int n, int w0, size_t lds,
                   hipStream_t st) {
    if (W == 64) launch_coarse<64, 8, 16, Norms>(K, a, tw, o, n, w0, lds, st);
    else if (L == 128) launch_coarse<32, 8, 16, Norms>(K, a, tw, o, n, w0, lds, st);
    else launch_coarse<32, 8, 8, Norms>(K, a, tw, o, n, w0, lds, st);
}

// N x N chips of n windows
template <int R1, int R2, bool MEAN>
void launch_oversample(bool wide, const OsArgs &a, int n, int w0, hipStream_t st) {
    constexpr int N = R1 * R2;
    const int lds = os_lds_bytes(N, wide);
    if (wide) hipLaunchKernelGGL((k_oversample<R1, R2, MEAN, true>), dim3(n), dim3(os_threads(N)), lds, st, a, w0);
    else hipLaunchKernelGGL((k_oversample<R1, R2, MEAN, false>), dim3(n), dim3(os_threads(N)), lds, st, a, w0);
}

// bytes of a normalization factor (NormsOf)
int norm_size(const ampcor_params &p) { return p.surf_ovs == 16 && p.surf_method == 0 ? Norms32::BYTES : Norms48::BYTES; }

// k_fine2 for the surfaces other than factor 16 by the FFT
void launch_fine2(int surf, const FineArgs &a, const cf *tw, int n, int w0, size_t lds, hipStream_t st) {
    if (surf == 0) hipLaunchKernelGGL((k_fine2<128, 9, 16, NT, 32, 0>), dim3(n), dim3(NT), lds, st, a, tw, w0);
    else hipLaunchKernelGGL((k_fine2<128, 9, 16, NT, 32, -1>), dim3(n), dim3(NT), lds, st, a, tw, w0);
}

}  // namespace fused

// Surface oversampling factors the fused kernels evaluate: 2..32 (FFT: one thread
// per surface column of a 512-thread workgroup; sinc: the patch's rows fit in LDS).
// Factor 1 and above 32 stay with the staged pipeline. 3,844 windows of 64, half
// search 20, factor 32: staged 2.66 ms, fused 1.18 ms; 900 with the sinc surface:
// staged 0.76 ms, fused 0.39 ms.
bool fused_fits(const ampcor_params &p, const ampcor_sizes &s) {
    using namespace fused;
    if (p.window_h != p.window_w || (p.window_h != 32 && p.window_h != 64)) return false;
    if (p.raw_ovs != 2 || s.zoom != 16 || p.surf_ovs < 2 || p.surf_ovs > 32) return false;
    const int L = coarse_L(s.search_w);
    if (L == 0) return false;
    if (pick_k(s.raw_corr_h, NT / (L / 2)) == 0) return false;
    const int nb = norm_size(p);
    if (CoarseLds(p.window_w, L, s.search_h, s.raw_corr_h, s.raw_corr_w, nb).total > 160 * 1024) return false;
    // the window sums' block sums (doubles) live in the template chunk's region (cf)
    if (2 * ((s.search_h + NORM_BLK - 1) / NORM_BLK) * s.search_w > coarse_tc(p.window_w) / 2 * (L + 1)) return false;
    const int P = 2 * s.zoom_in_w;
    if (FineLds(P, P - 2 * p.window_w + 1, 2 * p.window_w, s.surf_out, nb).total > 160 * 1024) return false;
    return true;
}

bool fused_supported(const ampcor_params &p, const ampcor_sizes &s) {
    return p.surf_ovs == 16 && p.surf_method == 0 && fused_fits(p, s);
}

// Tables the fused kernels read (twiddles, half-sample shifts). Built on first
// use; Engine::setup builds them for fused configurations, so that the
// allocation-free entry finds them in place.
FusedTables Engine::fused_tables() {
    using namespace fused;
    const int W = p.window_w, Zc = sz.zoom_in_w;
    auto tw = [&](int n) { return static_cast<const void *>(plan(n).tw32.ptr); };
    FusedTables t;
    t.tw_ref = tw(W);
    t.shift_ref = half_shifts<float>(W);
    t.tw_zoom = tw(Zc);
    t.shift_zoom = half_shifts<float>(Zc);
    t.tw1 = tw(coarse_L(sz.search_w));
    t.tw2 = tw(2 * Zc);
    t.tws = tw(sz.surf_out);
    t.tws_64 = plan(sz.surf_out).tw64.ptr;
    if (p.surf_method) ensure_sinc_table();
    return t;
}

// One launch of each fused kernel over windows [w0, w0 + n) of the arrays in c
// (starts, stage outputs and final outputs indexed by absolute window; the
// oversampled-chip intermediates hold this launch's n windows only).
void Engine::launch_fused(const FusedTables &tb, const FusedLaunch &c, int n, int w0, hipStream_t st) {
    using namespace fused;
    const int W = p.window_w, Zc = sz.zoom_in_w;          // 64 -> 72, 32 -> 40
    const int T2 = 2 * W, P = 2 * Zc;
    const int L1 = coarse_L(sz.search_w);
    const int K1 = pick_k(sz.raw_corr_h, NT / (L1 / 2));
    const int mode = p.image_complex ? (p.deramp == 0 ? 1 : 0) : 2;
    const int surf = p.surf_method ? -1 : (p.surf_ovs == 16 ? 16 : 0);   // surface stage (fine_finish)
    const cf *tw1 = static_cast<const cf *>(tb.tw1), *tw2 = static_cast<const cf *>(tb.tw2);
    const cf *tw_ref = static_cast<const cf *>(tb.tw_ref), *shift_ref = static_cast<const cf *>(tb.shift_ref);
    const cf *tw_zoom = static_cast<const cf *>(tb.tw_zoom), *shift_zoom = static_cast<const cf *>(tb.shift_zoom);
    float *tamp = c.tamp - size_t(w0) * T2 * T2;          // indexed by absolute window inside the kernels
    double *tmean = c.tmean - 2 * size_t(w0);
    float *samp = c.samp - size_t(w0) * P * P;

    CoarseArgs ca{c.ref, c.ref_pitch, c.sec, c.sec_pitch, mode, c.ref_d, c.ref_a, c.sec_d, c.sec_a,
                  p.hs_down, p.hs_across, sz.half_zoom, sz.corr_raw_zoom_h, sz.corr_raw_zoom_w,
                  c.loc, c.val, c.start, c.shift, c.snr, c.cov, c.mc};
    const int nb = norm_size(p);
    const size_t lds_c = CoarseLds(W, L1, sz.search_h, sz.raw_corr_h, sz.raw_corr_w, nb).total;
    const bool wide = surf != 16;
    const size_t lds_or = os_lds_bytes(W, wide);
    const size_t lds_f = FineLds(P, P - T2 + 1, T2, sz.surf_out, nb).total;
    const size_t lds_f2 = Fine2Lds(P, P - T2 + 1, 32, sz.surf_out, nb).total;
    {
        OsArgs oref{c.ref, c.ref_pitch, mode, c.ref_d, c.ref_a, nullptr, p.deramp, tw_ref, shift_ref, tamp, tmean};
        // (a profile times the stages one by one)
        const bool merged = n <= MERGE_MAX && !profiling;
        const OsArgs *o = merged ? &oref : nullptr;
        const size_t lds_m = merged ? std::max(lds_c, lds_or) : lds_c;
        timed("k_coarse", n, st, [&] {
            if (wide) launch_coarse<Norms48>(W, L1, K1, ca, tw1, o, n, w0, lds_m, st);
            else launch_coarse<Norms32>(W, L1, K1, ca, tw1, o, n, w0, lds_m, st);
        });
        if (wide) {
            if (W == 64) hipLaunchKernelGGL(k_peak_cov<64>, dim3(n), dim3(COV_NT), 0, st, ca, w0);
            else hipLaunchKernelGGL(k_peak_cov<32>, dim3(n), dim3(COV_NT), 0, st, ca, w0);
        }
        OsArgs osec{c.sec, c.sec_pitch, mode, c.sec_d, c.sec_a, c.start, p.deramp, tw_zoom, shift_zoom, samp, nullptr};
        FineArgs fa{tamp, tmean, samp, c.start, p.hs_down, p.hs_across, 1.0f / float(p.surf_ovs * p.raw_ovs),
                    p.surf_ovs, static_cast<const cf *>(tb.tws), SincTable{sinc_table.as<float>(), sinc_dec}, c.shift,
                    c.zidx, c.offset, c.mf, c.surf ? c.surf - size_t(w0) * 256 : nullptr};
        if (W == 64) {
            if (!merged) timed("k_oversample_ref", n, st, [&] {
                launch_oversample<8, 8, true>(wide, oref, n, w0, st);
            });
            timed("k_oversample_search", n, st, [&] {
                launch_oversample<9, 8, false>(wide, osec, n, w0, st);
            });
            timed("k_fine", n, st, [&] {
                // the whole-template kernel is built for the surfaces AMPCOR_MODE_FUSED accepts
                if (surf != 16)
                    launch_fine2(surf, fa, tw2, n, w0, lds_f2, st);
                else if (fine_kernel == 2)
                    hipLaunchKernelGGL((k_fine2<128, 9, 16, NT, 32, 16>), dim3(n), dim3(NT), lds_f2, st, fa, tw2, w0);
                else if (fine_threads == 1024)
                    hipLaunchKernelGGL((k_fine<128, 9, 16, 2, 1024, 16>), dim3(n), dim3(1024), lds_f, st, fa, tw2, w0);
                else
                    hipLaunchKernelGGL((k_fine<128, 16, 9, 3, NT, 16>), dim3(n), dim3(NT), lds_f, st, fa, tw2, w0);
            });
        } else {
            if (!merged) timed("k_oversample_ref", n, st, [&] {
                launch_oversample<8, 4, true>(wide, oref, n, w0, st);
            });
            timed("k_oversample_search", n, st, [&] {
                launch_oversample<5, 8, false>(wide, osec, n, w0, st);
            });
            timed("k_fine", n, st, [&] {
                if (surf == 16)
                    hipLaunchKernelGGL((k_fine<64, 5, 16, 2, NT, 16>), dim3(n), dim3(NT), lds_f, st, fa, tw2, w0);
                else if (surf == 0)
                    hipLaunchKernelGGL((k_fine<64, 5, 16, 2, NT, 0>), dim3(n), dim3(NT), lds_f, st, fa, tw2, w0);
                else
                    hipLaunchKernelGGL((k_fine<64, 5, 16, 2, NT, -1>), dim3(n), dim3(NT), lds_f, st, fa, tw2, w0);
            });
        }
        if (c.refined)
            hipLaunchKernelGGL(k_refine<float>, dim3(n), dim3(64), refine_lds(16), st, c.surf, 16, 16, 16,
                               p.surf_ovs, 1.0 / double(p.surf_ovs * p.raw_ovs), c.zidx + 2 * size_t(w0),
                               c.start + 2 * size_t(w0), p.hs_down, p.hs_across,
                               static_cast<const cx<double> *>(tb.tws_64), c.refined + 2 * size_t(w0));
        HIP_OK(hipGetLastError());
    }
}

void Engine::run_fused(const RunArgs &a) {
    const int W = p.window_w, Zc = sz.zoom_in_w;
    const int T2 = 2 * W, P = 2 * Zc;
    const int chunk = std::min(a.chunk > 0 ? a.chunk : 32768, 65535);
    const int nb = std::min(chunk, a.n);
    const FusedTables tb = fused_tables();
    FusedLaunch c{};
    c.ref = a.ref; c.ref_pitch = a.ref_pitch; c.sec = a.sec; c.sec_pitch = a.sec_pitch;
    c.ref_d = a.ref_d; c.ref_a = a.ref_a; c.sec_d = a.sec_d; c.sec_a = a.sec_a;
    c.loc = a.maxloc ? a.maxloc : buf<int32_t>("f_loc", size_t(a.n) * 2);
    c.val = a.maxval ? a.maxval : buf<float>("f_val", a.n);
    c.start = a.start ? a.start : buf<int32_t>("f_start", size_t(a.n) * 2);
    c.shift = a.shift ? a.shift : buf<int32_t>("f_shift", size_t(a.n) * 2);
    c.zidx = a.zoom_idx ? a.zoom_idx : buf<int32_t>("f_zidx", size_t(a.n) * 2);
    c.tamp = buf<float>("f_tamp", size_t(nb) * T2 * T2);
    c.tmean = buf<double>("f_tmean", 2 * size_t(nb));
    c.samp = buf<float>("f_samp", size_t(nb) * P * P);
    const bool want_margin = precision == 1 || a.margin_coarse || a.margin_fine;
    c.mc = a.margin_coarse ? a.margin_coarse : (want_margin ? buf<float>("f_mc", a.n) : nullptr);
    c.mf = a.margin_fine ? a.margin_fine : (want_margin ? buf<float>("f_mf", a.n) : nullptr);
    c.offset = a.offset; c.snr = a.snr; c.cov = a.cov;
    if (a.refined) {
        c.surf = buf<float>("f_surf", size_t(nb) * 256);
        c.refined = a.refined;
    }
    for (int w0 = 0; w0 < a.n; w0 += nb) launch_fused(tb, c, std::min(nb, a.n - w0), w0, a.stream);
    if (precision == 1 && !a.nosync) rerun_fp64(a, c.mc, c.mf, c.start, c.shift);
}

// ---------------------------------------------------------------------------
// Allocation-free entry (ampcor_run_windows_noalloc). Every intermediate of the
// fused kernels lives in one file-scope device array; each GPU holds its own
// copy until the process ends, and every call on that GPU shares it (calls that
// overlap on one GPU race). Its address on each device is taken once, at context
// creation, with that device current.
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = size_t(256) << 20;   // 256 MiB per GPU
// In host code `scratch` names a host-side stand-in, never the device array:
// host code uses the address hipGetSymbolAddress returns for each device.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mu;
std::map<int, void *> g_scratch;                      // device -> address of that device's copy

size_t al256(size_t x) { return (x + 255) & ~size_t(255); }
}  // namespace

void *noalloc_scratch_init(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    auto it = g_scratch.find(device);
    if (it != g_scratch.end()) return it->second;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        (void)hipGetLastError();
        throw Error(AMPCOR_E_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    }
    g_scratch[device] = ptr;
    return ptr;
}

// Per-window bytes of the carve-up below: sanitized starts, bad flags, stage
// outputs, margins, template mean, oversampled template and search amplitudes.
static size_t noalloc_window_bytes(int T2, int P) {
    return 16 + 4 + 8 * 4 + 4 + 8 + 16 + size_t(T2) * T2 * 4 + size_t(P) * P * 4;
}

void Engine::run_fused_noalloc(const RunArgs &a) {
    if (!scratch_ptr) throw Error(AMPCOR_E_DEVICE, "the no-alloc scratch of this device is not set up");
    const int W = p.window_w, Zc = sz.zoom_in_w;
    const int T2 = 2 * W, P = 2 * Zc;
    const size_t per = noalloc_window_bytes(T2, P);
    // 11 arrays, each padded to 256 bytes
    const size_t cap = (kScratchBytes - 11 * 256) / per;
    if (cap < 1)
        throw Error(AMPCOR_E_UNSUPPORTED, "one window needs " + std::to_string(per) + " bytes, more than the " +
                                              std::to_string(kScratchBytes) + "-byte no-alloc scratch");
    const int m = int(std::min<size_t>({cap, size_t(a.n), 65535}));
    const FusedTables tb = fused_tables();                 // built by ampcor_setup; never allocates here
    unsigned char *s = static_cast<unsigned char *>(scratch_ptr);
    auto take = [&](size_t bytes) {
        void *q = s;
        s += al256(bytes);
        return q;
    };
    int32_t *st4 = static_cast<int32_t *>(take(16 * size_t(m)));
    int32_t *bad = static_cast<int32_t *>(take(4 * size_t(m)));
    FusedLaunch c{};
    c.ref = a.ref; c.ref_pitch = a.ref_pitch; c.sec = a.sec; c.sec_pitch = a.sec_pitch;
    c.ref_d = st4; c.ref_a = st4 + m; c.sec_d = st4 + 2 * m; c.sec_a = st4 + 3 * m;
    c.loc = static_cast<int32_t *>(take(8 * size_t(m)));
    c.start = static_cast<int32_t *>(take(8 * size_t(m)));
    c.shift = static_cast<int32_t *>(take(8 * size_t(m)));
    c.zidx = static_cast<int32_t *>(take(8 * size_t(m)));
    c.val = static_cast<float *>(take(4 * size_t(m)));
    c.mc = static_cast<float *>(take(4 * size_t(m)));
    c.mf = static_cast<float *>(take(4 * size_t(m)));
    c.tmean = static_cast<double *>(take(16 * size_t(m)));
    c.tamp = static_cast<float *>(take(size_t(m) * T2 * T2 * 4));
    c.samp = static_cast<float *>(take(size_t(m) * P * P * 4));
    if (size_t(s - static_cast<unsigned char *>(scratch_ptr)) > kScratchBytes)
        throw Error(AMPCOR_E_UNSUPPORTED, "no-alloc scratch carve-up exceeds the array");
    for (int w0 = 0; w0 < a.n; w0 += m) {
        const int n = std::min(m, a.n - w0);
        // this chunk's starts, bounds-checked on the device (out-of-image windows get NaN outputs)
        hipLaunchKernelGGL(k_sanitize_starts<int32_t>, dim3(idivup(n, 256)), dim3(256), 0, a.stream, a.ref_d + w0,
                           a.ref_a + w0, a.sec_d + w0, a.sec_a + w0, n, a.ref_h, a.ref_w, a.sec_h, a.sec_w,
                           p.window_h, p.window_w, sz.search_h, sz.search_w, st4, bad);
        if (n < m) {            // the sanitized arrays of a short last chunk start at the same offsets
            c.ref_a = st4 + n; c.sec_d = st4 + 2 * n; c.sec_a = st4 + 3 * n;
        }
        c.offset = a.offset + 2 * size_t(w0);
        c.snr = a.snr + w0;
        c.cov = a.cov + 3 * size_t(w0);
        launch_fused(tb, c, n, 0, a.stream);
        hipLaunchKernelGGL(k_mark_bad<float>, dim3(idivup(n, 256)), dim3(256), 0, a.stream, bad, n, c.offset, c.snr,
                           c.cov);
        HIP_OK(hipGetLastError());
    }
}

}  // namespace ampcor
