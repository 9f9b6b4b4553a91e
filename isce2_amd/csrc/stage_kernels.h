// Batched per-stage kernels of the staged pipeline (one launch per stage over a
// chunk of windows, intermediates in HBM). Each kernel names the reference
// function whose arithmetic it performs (paths under contrib/PyCuAmpcor/src/).
#pragma once
#include <cfloat>
#include <type_traits>
#include "cx.h"
#include "fft_inplace.h"
#include "fft_lds.h"

namespace ampcor {

// ---------------------------------------------------------------------------
// 1D FFTs over rows / columns of batched row-major images in HBM
// ---------------------------------------------------------------------------
// rows: `nrows` contiguous rows of length d.n (row pitch d.n), `g` rows per block
template <class T, int DIR>
__global__ void __launch_bounds__(256) k_fft_rows(cx<T> *data, int nrows, int g, FftDesc d) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + g * d.n;
    const int r0 = blockIdx.x * g;
    const int nr = min(g, nrows - r0);
    const int tot = nr * d.n;
    cx<T> *base = data + size_t(r0) * d.n;
    for (int i = threadIdx.x; i < tot; i += blockDim.x) a[i] = base[i];
    __syncthreads();
    cx<T> *res = fft_lds<T, DIR>(a, b, d, nr, 1, d.n);
    for (int i = threadIdx.x; i < tot; i += blockDim.x) base[i] = res[i];
}

// columns: images [nimg][h][w] with h = d.n; `c` columns per block
template <class T, int DIR>
__global__ void __launch_bounds__(512) k_fft_cols(cx<T> *data, int w, int c, FftDesc d) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + c * d.n;
    const int h = d.n;
    const int col0 = blockIdx.x * c;
    const int nc = min(c, w - col0);
    cx<T> *img = data + size_t(blockIdx.y) * h * w + col0;
    const int tot = h * nc;
    for (int i = threadIdx.x; i < tot; i += blockDim.x) {
        const int r = i / nc, cc = i - r * nc;
        a[r * c + cc] = img[size_t(r) * w + cc];
    }
    __syncthreads();
    cx<T> *res = fft_lds<T, DIR>(a, b, d, nc, c, 1);
    for (int i = threadIdx.x; i < tot; i += blockDim.x) {
        const int r = i / nc, cc = i - r * nc;
        img[size_t(r) * w + cc] = res[r * c + cc];
    }
}

// Inverse 2-D FFT of the quadrant padding of h x w spectra into H x W
// (cuArraysPadding.cu:59-103 followed by the oversampler's second transform,
// cuOverSampler.cpp:72-78 and :141-148), in two passes that never store the
// padding. Row pass: each of the 2*(h/2) non-zero padded rows is built in LDS
// from the small spectrum (scaled by 1/(h*w), zeros between the quadrants) and
// transformed; it lands at its padded row of `out` ([nimg][H][d.n]), whose
// all-zero rows are left unwritten. `g` rows per block.
template <class T, int DIR>
__global__ void __launch_bounds__(256) k_fft_rows_quad(const cx<T> *in, int nimg, int h, int w, cx<T> *out, int H,
                                                       int g, FftDesc d) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + g * d.n;
    const int W = d.n, h2 = h / 2, w2 = w / 2, sel = 2 * h2;
    const T f = T(1) / T(h * w);
    const int t0 = blockIdx.x * g;
    const int nr = min(g, nimg * sel - t0);
    for (int i = threadIdx.x; i < nr * W; i += blockDim.x) {
        const int k = i / W, q = i - k * W;
        const int t = t0 + k, img = t / sel, s = t - img * sel;
        const int sr = s < h2 ? s : h - sel + s;   // rows [0, h2) and [h - h2, h) of the spectrum
        const int sc = q < w2 ? q : (q >= W - w2 ? q - W + w : -1);
        a[i] = sc >= 0 ? in[(size_t(img) * h + sr) * w + sc] * f : cx<T>{T(0), T(0)};
    }
    __syncthreads();
    cx<T> *res = fft_lds<T, DIR>(a, b, d, nr, 1, W);
    for (int i = threadIdx.x; i < nr * W; i += blockDim.x) {
        const int k = i / W, q = i - k * W;
        const int t = t0 + k, img = t / sel, s = t - img * sel;
        const int p = s < h2 ? s : H - sel + s;    // padded rows [0, h2) and [H - h2, H)
        out[(size_t(img) * H + p) * W + q] = res[i];
    }
}

// Column pass of the same inverse over [nimg][d.n][w] images whose rows
// [h2, d.n - h2) are zero and not read. Only a real image is kept: |z| (OUT 1,
// the oversampled chips' amplitude, cuArraysCopy.cu:510-529) or Re z (OUT 2,
// the oversampled surface, cuArraysCopy.cu:326-339), written to `out`
// ([nimg][d.n][w]). `c` columns per block.
template <class T, int DIR, int OUT>
__global__ void __launch_bounds__(512) k_fft_cols_quad(const cx<T> *data, int w, int c, int h2, FftDesc d, T *out) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + c * d.n;
    const int h = d.n;
    const int col0 = blockIdx.x * c;
    const int nc = min(c, w - col0);
    const cx<T> *img = data + size_t(blockIdx.y) * h * w + col0;
    const int tot = h * nc;
    for (int i = threadIdx.x; i < tot; i += blockDim.x) {
        const int r = i / nc, cc = i - r * nc;
        a[r * c + cc] = (r < h2 || r >= h - h2) ? img[size_t(r) * w + cc] : cx<T>{T(0), T(0)};
    }
    __syncthreads();
    const cx<T> *res = fft_lds<T, DIR>(a, b, d, nc, c, 1);
    T *o = out + size_t(blockIdx.y) * h * w + col0;
    for (int i = threadIdx.x; i < tot; i += blockDim.x) {
        const int r = i / nc, cc = i - r * nc;
        const cx<T> v = res[r * c + cc];
        o[size_t(r) * w + cc] = OUT == 1 ? amag(v) : v.x;
    }
}

// ---------------------------------------------------------------------------
// chips read straight from the images: window w's chip starts at row d[w], column
// a[w] (plus the zoom chip's origin start[w] when given); mode as k_gather's
// ---------------------------------------------------------------------------
struct ChipSrc {
    const void *img;
    int64_t pitch;
    const int32_t *d, *a, *start;
    int mode;
};

// image offset of the chip's first pixel
__device__ __forceinline__ int64_t chip_origin(const ChipSrc &s, int w) {
    int64_t r = s.d[w], c = s.a[w];
    if (s.start) { r += s.start[2 * w]; c += s.start[2 * w + 1]; }
    return r * s.pitch + c;
}

// A chip's pixel in two steps, so that the loads of several pixels can be in flight
// before the first is converted: the raw value at image offset `off` (REAL: (x, 0)),
// and the pixel as the pipeline's chips hold it. with_kind(src, f) calls f with
// std::true_type for real images, so that the choice is made once and not per load.
template <bool REAL>
__device__ __forceinline__ float2 chip_raw(const ChipSrc &s, int64_t off) {
    if constexpr (REAL) return {static_cast<const float *>(s.img)[off], 0.f};
    else return static_cast<const float2 *>(s.img)[off];
}
template <class T>
__device__ __forceinline__ cx<T> chip_value(const ChipSrc &s, float2 z) {
    if (s.mode == 1) return {T(fast_abs(z.x, z.y)), T(0)};
    return {T(z.x), T(z.y)};
}
template <class F>
__device__ __forceinline__ void with_kind(const ChipSrc &s, F f) {
    if (s.mode == 2) f(std::true_type{});
    else f(std::false_type{});
}

template <class T>
__global__ void k_gather(ChipSrc src, int h, int w, cx<T> *out, T *amp) {
    const int win = blockIdx.y;
    const int tot = h * w;
    const int64_t o0 = chip_origin(src, win);
    cx<T> *o = out + size_t(win) * tot;
    with_kind(src, [&](auto real) {
        #pragma unroll 2
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += gridDim.x * blockDim.x) {
            const int r = i / w, c = i - r * w;
            const cx<T> v = chip_value<T>(src, chip_raw<decltype(real)::value>(src, o0 + r * src.pitch + c));
            o[i] = v;
            if (amp) amp[size_t(win) * tot + i] = amag(v);
        }
    });
}

// No-sync bounds check: copy the start arrays ([4][n] out), replacing every
// window whose chips leave their image by window (0, 0) and flagging it
template <class I>
__global__ void k_sanitize_starts(const I *rd, const I *ra, const I *sd, const I *sa, int n, int64_t ref_h,
                                  int64_t ref_w, int64_t sec_h, int64_t sec_w, int wh, int ww, int sh, int sw,
                                  I *out, int32_t *bad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t r0 = rd[i], a0 = ra[i], s0 = sd[i], t0 = sa[i];
    const bool ok = r0 >= 0 && a0 >= 0 && r0 + wh <= ref_h && a0 + ww <= ref_w && s0 >= 0 && t0 >= 0 &&
                    s0 + sh <= sec_h && t0 + sw <= sec_w && ref_h >= wh && ref_w >= ww && sec_h >= sh && sec_w >= sw;
    out[i] = ok ? I(r0) : I(0);
    out[n + i] = ok ? I(a0) : I(0);
    out[2 * n + i] = ok ? I(s0) : I(0);
    out[3 * n + i] = ok ? I(t0) : I(0);
    bad[i] = ok ? 0 : 1;
}

// NaN outputs for the windows k_sanitize_starts flagged
template <class T>
__global__ void k_mark_bad(const int32_t *bad, int n, T *offset, T *snr, T *cov) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !bad[i]) return;
    const T q = T(__builtin_nanf(""));
    offset[2 * i] = q; offset[2 * i + 1] = q;
    snr[i] = q;
    cov[3 * i] = q; cov[3 * i + 1] = q; cov[3 * i + 2] = q;
}

// block-wide FP64 sum (256 threads)
// block sum for blocks of up to 64 * (size of sh) threads
__device__ __forceinline__ double block_sum256(double v, double *sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wv] = v;
    __syncthreads();
    double s = 0.0;
    const int nw = (blockDim.x + 63) >> 6;
    for (int i = 0; i < nw; ++i) s += sh[i];
    __syncthreads();
    return s;
}

// mean subtraction per image, FP64 sum (cuCorrNormalization.cu:98-139)
template <class T>
__global__ void __launch_bounds__(1024) k_sub_mean(T *data, int size, double *ssd) {
    __shared__ double sh[16];
    T *img = data + size_t(blockIdx.x) * size;
    double s1 = 0.0, s2 = 0.0;
    for (int i = threadIdx.x; i < size; i += blockDim.x) {
        const double v = double(img[i]);
        s1 += v;
        s2 += v * v;
    }
    s1 = block_sum256(s1, sh);
    const T mean = T(s1 / size);
    for (int i = threadIdx.x; i < size; i += blockDim.x) img[i] -= mean;
    if (ssd) {
        // sum of squares of the mean-subtracted image (the normalization's template term)
        s2 = block_sum256(s2, sh);
        if (threadIdx.x == 0) ssd[blockIdx.x] = fmax(s2 - s1 * s1 / size, 0.0);
    }
}

// f(r, c) for the pixels of an h x w chip that fall to this thread of the block, U at a
// time so that their loads are in flight together; past the last pixel f gets ok = false
// (and the last pixel again)
template <int U, class F>
__device__ __forceinline__ void chip_pixels(int h, int w, F f) {
    const int n = h * w, nt = blockDim.x, dr = nt / w, dc = nt - dr * w;
    int r = threadIdx.x / w, c = threadIdx.x - r * w;
    for (int i = threadIdx.x; i < n; i += U * nt) {
        int rr[U], cc[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ok[u] = r < h;
            rr[u] = ok[u] ? r : h - 1;
            cc[u] = ok[u] ? c : w - 1;
            r += dr;
            c += dc;
            if (c >= w) { c -= w; ++r; }
        }
        f(rr, cc, ok);
    }
}

// FP64 mean and sum of squared deviations of [nimg][size] images, which are left as
// they are (their consumer subtracts the mean as it loads them); one block per image
template <class T>
__global__ void __launch_bounds__(1024) k_array_mean(const T *data, int size, double *mean, double *ssd) {
    __shared__ double sh[16];
    const T *img = data + size_t(blockIdx.x) * size;
    double s1 = 0.0, s2 = 0.0;
    #pragma unroll 8
    for (int i = threadIdx.x; i < size; i += blockDim.x) {
        const double v = double(img[i]);
        s1 += v;
        s2 += v * v;
    }
    s1 = block_sum256(s1, sh);
    s2 = block_sum256(s2, sh);
    if (threadIdx.x == 0) {
        mean[blockIdx.x] = s1 / size;
        ssd[blockIdx.x] = fmax(s2 - s1 * s1 / size, 0.0);
    }
}

// FP64 sums of chips' amplitudes and of their squares, read from the image, over
// gridDim.y row ranges of each chip: part[(w * ranges + range) * 2 + (0, 1)] (k_mean_parts)
template <class T>
__global__ void __launch_bounds__(256) k_chip_sums(ChipSrc src, int h, int w, double *part) {
    __shared__ double sh[16];
    const int per = (h + gridDim.y - 1) / gridDim.y, r0 = blockIdx.y * per, rows = max(0, min(h, r0 + per) - r0);
    const int64_t o0 = chip_origin(src, blockIdx.x) + r0 * src.pitch;
    double s1 = 0.0, s2 = 0.0;
    constexpr int U = 8;
    with_kind(src, [&](auto real) {
        chip_pixels<U>(rows, w, [&](const int (&r)[U], const int (&c)[U], const bool (&ok)[U]) {
            float2 z[U];
#pragma unroll
            for (int u = 0; u < U; ++u) z[u] = chip_raw<decltype(real)::value>(src, o0 + r[u] * src.pitch + c[u]);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double v = ok[u] ? double(amag(chip_value<T>(src, z[u]))) : 0.0;
                s1 += v;
                s2 += v * v;
            }
        });
    });
    s1 = block_sum256(s1, sh);
    s2 = block_sum256(s2, sh);
    if (threadIdx.x == 0) {
        double *o = part + (size_t(blockIdx.x) * gridDim.y + blockIdx.y) * 2;
        o[0] = s1;
        o[1] = s2;
    }
}

// ---------------------------------------------------------------------------
// Row-spectrum correlation over NL lag rows:
//   c[u][v] = (1/L) IFFT_L( sum_t conj(T_t) S_{t+u} )[v],   0 <= u < NL,
// equal to the zero-padded 2-D correlation (cuCorrFrequency.cu:63-79) at every
// valid lag for any row length L >= the search width. Row half spectra come
// from k_rowspec, are summed over template rows per bin and lag (k_mac_lags),
// and only the NL lag rows go back through a row IFFT (k_lagrows_real).
// ---------------------------------------------------------------------------

// Half spectra of the rows of real images ([nimg][h][L/2+1]): rows 2j and 2j+1 are
// loaded as one complex row z = r_2j + i r_2j+1 of length L (zero beyond w and h),
// transformed in LDS, and split with A = (Z[k] + conj Z[-k]) / 2, B = (Z[k] -
// conj Z[-k]) / (2i). One launch does the template rows and the search rows: a RowJob
// each, the first `blocks` workgroups the first. The rows come from an array
// ([nimg][h][w]) or are the amplitudes of chips read in place (img null), which also go
// to `amp` when given; `mean`: per-image mean subtracted on load when given.
template <class T>
struct RowJob {
    const T *img;
    ChipSrc chip;
    int h, w;
    const double *mean;
    cx<T> *spec;
    T *amp;
    int blocks;
};

// row pairs [t0, t0 + nr) of the job into z(k, x); org and mu hold a value per pair in LDS
// (short rows come by more pairs than the workgroup has threads)
template <class T, class Z>
__device__ __forceinline__ void load_row_pairs(const RowJob<T> &j, int t0, int nr, int L, int64_t *org, T *mu, Z z) {
    const int np = (j.h + 1) / 2;
    for (int k = threadIdx.x; k < nr; k += blockDim.x) {
        const int t = t0 + k, win = t / np, r = 2 * (t - win * np);
        org[k] = j.img ? (int64_t(win) * j.h + r) * j.w : chip_origin(j.chip, win) + r * j.chip.pitch;
        mu[k] = j.mean ? T(j.mean[win]) : T(0);
    }
    __syncthreads();
    auto rows = [&](auto pixels) {
        #pragma unroll 4
        for (int i = threadIdx.x; i < nr * L; i += blockDim.x) {
            const int k = i / L, x = i - k * L;
            const int t = t0 + k, win = t / np, r = 2 * (t - win * np);
            const bool in = x < j.w, two = in && r + 1 < j.h;
            cx<T> v = {T(0), T(0)};
            if (in) v = pixels(k, x, win, r, two);
            if (in) v.x -= mu[k];
            if (two) v.y -= mu[k];
            z(k, x, v);
        }
    };
    if (j.img)
        rows([&](int k, int x, int, int, bool two) {
            const T *p = j.img + org[k] + x;
            return cx<T>{p[0], two ? p[j.w] : T(0)};
        });
    else
        with_kind(j.chip, [&](auto real) {
            rows([&](int k, int x, int win, int r, bool two) {
                constexpr bool R = decltype(real)::value;
                const float2 a = chip_raw<R>(j.chip, org[k] + x);
                const float2 b = two ? chip_raw<R>(j.chip, org[k] + j.chip.pitch + x) : float2{0.f, 0.f};
                const cx<T> v = {amag(chip_value<T>(j.chip, a)), amag(chip_value<T>(j.chip, b))};
                if (j.amp) {
                    T *o = j.amp + (size_t(win) * j.h + r) * j.w + x;
                    o[0] = v.x;
                    if (two) o[j.w] = v.y;
                }
                return v;
            });
        });
    __syncthreads();
}

// the split half spectra of pairs [t0, t0 + nr) to memory; z(k, bin) reads the transform
template <class T, class Z>
__device__ __forceinline__ void store_row_spectra(const RowJob<T> &j, int t0, int nr, int L, Z z) {
    const int np = (j.h + 1) / 2, H1 = L / 2 + 1;
    for (int i = threadIdx.x; i < nr * H1; i += blockDim.x) {
        const int k = i / H1, kk = i - k * H1;
        const int t = t0 + k, win = t / np, p = t - win * np;
        const cx<T> za = z(k, kk), bc = conj(z(k, kk ? L - kk : 0));
        cx<T> *sp = j.spec + (size_t(win) * j.h + 2 * p) * H1 + kk;
        sp[0] = (za + bc) * T(0.5);
        if (2 * p + 1 < j.h) {
            const cx<T> dd = (za - bc) * T(0.5);
            sp[H1] = {dd.y, -dd.x};
        }
    }
}

// general lengths (Stockham), `g` row pairs per block; LDS: 2 g L cx<T>, then g of (int64, T)
template <class T>
__global__ void __launch_bounds__(256) k_rowspec(RowJob<T> a, RowJob<T> b, int nimg, int g, FftDesc d) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *p = reinterpret_cast<cx<T> *>(smem_raw), *q = p + g * d.n;
    int64_t *org = reinterpret_cast<int64_t *>(q + g * d.n);
    T *mu = reinterpret_cast<T *>(org + g);
    const bool first = int(blockIdx.x) < a.blocks;
    const RowJob<T> &j = first ? a : b;
    const int t0 = (blockIdx.x - (first ? 0 : a.blocks)) * g, nr = min(g, nimg * ((j.h + 1) / 2) - t0);
    load_row_pairs(j, t0, nr, d.n, org, mu, [&](int k, int x, cx<T> v) { p[k * d.n + x] = v; });
    const cx<T> *Z = fft_lds<T, -1>(p, q, d, nr, 1, d.n);
    store_row_spectra(j, t0, nr, d.n, [&](int k, int bin) { return Z[k * d.n + bin]; });
}

// in-place transforms (fft_nat2dr, length L = R1 * R2, read back from digit-reversed
// order), G row pairs per block of odd LDS pitch
template <class T, int R1, int R2, int G, int NTH = 256>
__global__ void __launch_bounds__(NTH) k_rowspec_f(RowJob<T> a, RowJob<T> b, int nimg, const cx<T> *tw) {
    constexpr int L = R1 * R2, PR = L + 1;
    __shared__ cx<T> C[G * PR];
    __shared__ int64_t org[G];
    __shared__ T mu[G];
    __shared__ cx<T> twl[L];                           // twiddles, read from LDS
    for (int i = threadIdx.x; i < L; i += NTH) twl[i] = tw[i];
    const bool first = int(blockIdx.x) < a.blocks;
    const RowJob<T> &j = first ? a : b;
    const int t0 = (blockIdx.x - (first ? 0 : a.blocks)) * G, nr = min(G, nimg * ((j.h + 1) / 2) - t0);
    load_row_pairs(j, t0, nr, L, org, mu, [&](int k, int x, cx<T> v) { C[k * PR + x] = v; });
    fft_nat2dr<T, -1, R1, R2, NTH>(C, nr, PR, 1, twl);
    store_row_spectra(j, t0, nr, L, [&](int k, int bin) { return C[k * PR + dr_pos<R1, R2>(bin)]; });
}

// the inverse row FFT of the lag rows and its real part: rows t of
// length d.n (t = window * nl + lag) -> out[t][v] = Re, v < nlw; `g` rows per block
template <class T>
__global__ void __launch_bounds__(256) k_lagrows_real(const cx<T> *q, int nrows, int g, FftDesc d, int nlw, T *out) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + g * d.n;
    const int r0 = blockIdx.x * g;
    const int nr = min(g, nrows - r0);
    const cx<T> *base = q + size_t(r0) * d.n;
    for (int i = threadIdx.x; i < nr * d.n; i += blockDim.x) a[i] = base[i];
    __syncthreads();
    const cx<T> *res = fft_lds<T, 1>(a, b, d, nr, 1, d.n);
    for (int i = threadIdx.x; i < nr * nlw; i += blockDim.x) {
        const int k = i / nlw, v = i - k * nlw;
        out[size_t(r0 + k) * nlw + v] = res[k * d.n + v].x;
    }
}

// q[u][k] = scale * sum_t conj(T_t[k]) S_{t+u}[k] for lags u0 <= u < u0 + K (u < nl),
// written as full Hermitian rows of length L for the inverse row FFT. A workgroup
// of NQ waves per (64 bins, lag group, window): wave w walks the w-th contiguous
// part of the search rows, keeping the template rows of its K lags in a sliding
// register window, so each thread's chain of row loads is 1/NQ of the whole;
// the NQ partial sums are added in wave order through LDS.
template <class T, int K, int NQ>
__global__ void __launch_bounds__(64 * NQ) k_mac_lags(const cx<T> *tspec, int th, const cx<T> *sspec, int sh, int nl,
                                                      int L, cx<T> *q, T scale) {
    __shared__ cx<T> part[NQ > 1 ? NQ - 1 : 1][K][64];
    const int H1 = L / 2 + 1, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane, u0 = blockIdx.y * K, win = blockIdx.z;
    const int r_end = min(sh, u0 + K - 1 + th), per = (r_end - u0 + NQ - 1) / NQ;
    const int ra = u0 + w * per, rb = min(r_end, ra + per);
    cx<T> acc[K], tw[K];
#pragma unroll
    for (int j = 0; j < K; ++j) acc[j] = tw[j] = cx<T>{T(0), T(0)};
    if (k < H1) {
        const cx<T> *ts = tspec + size_t(win) * th * H1 + k;
        const cx<T> *ss = sspec + size_t(win) * sh * H1 + k;
        // the template rows the lags meet just before row ra: tw[m] = T_{ra - u0 - 1 - m}
#pragma unroll
        for (int m = 0; m + 1 < K; ++m) {
            const int t = ra - u0 - 1 - m;
            if (t >= 0 && t < th) tw[m] = ts[size_t(t) * H1];
        }
        #pragma unroll 2
        for (int r = ra; r < rb; ++r) {
#pragma unroll
            for (int j = K - 1; j > 0; --j) tw[j] = tw[j - 1];     // tw[j] = T_{r - u0 - j}
            tw[0] = r - u0 < th ? ts[size_t(r - u0) * H1] : cx<T>{T(0), T(0)};
            const cx<T> sv = ss[size_t(r) * H1];
#pragma unroll
            for (int j = 0; j < K; ++j) acc[j] = cmac_conj(acc[j], tw[j], sv);
        }
    }
    if (NQ > 1) {
        if (w > 0) {
#pragma unroll
            for (int j = 0; j < K; ++j) part[w - 1][j][lane] = acc[j];
        }
        __syncthreads();
        if (w > 0) return;
#pragma unroll
        for (int p = 0; p + 1 < NQ; ++p)
#pragma unroll
            for (int j = 0; j < K; ++j) acc[j] = acc[j] + part[p][j][lane];
    }
    if (k >= H1) return;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (u0 + j < nl) {   // no early exit: the unrolled loop keeps acc[] in registers
            cx<T> *row = q + (size_t(win) * nl + u0 + j) * L;
            const cx<T> v = acc[j] * scale;
            row[k] = v;
            if (k && L - k != k) row[L - k] = conj(v);
        }
    }
}

// ---------------------------------------------------------------------------
// Window sums for the normalization (formula of cuCorrNormalization.cu:230-314 and
// cuCorrNormalizationSAT.cu:237-240), FP64, by lag rows: the sums of s and s^2 over SUM_BLK
// rows of every search column (k_block_sums) give a lag row's column sums from th / SUM_BLK
// blocks and a few rows at the ends; the next lag rows slide down from it; a wave prefix
// scan over the columns then leaves every horizontal window sum as a difference.
// ---------------------------------------------------------------------------
constexpr int SUM_BLK = 16;

// sums[w][b][0 and 1][c]: s and s^2 over rows [SUM_BLK b, SUM_BLK (b + 1)) of column c of
// [n][sh][sw] images; a wave per 64 columns and row block (task), 4 tasks a workgroup
__host__ __device__ inline int block_sum_tasks(int sh, int sw) { return ((sh + SUM_BLK - 1) / SUM_BLK) * ((sw + 63) / 64); }

template <class T>
__device__ __forceinline__ void block_sums_task(const T *img, int sh, int sw, int task, int win, double *sums) {
    const int cols = (sw + 63) / 64, b = task / cols, c = 64 * (task - b * cols) + (threadIdx.x & 63);
    if (task >= block_sum_tasks(sh, sw) || c >= sw) return;
    const int nblk = (sh + SUM_BLK - 1) / SUM_BLK, r0 = b * SUM_BLK;
    const T *p = img + (size_t(win) * sh + r0) * sw + c;
    T v[SUM_BLK];
#pragma unroll
    for (int r = 0; r < SUM_BLK; ++r) v[r] = r0 + r < sh ? p[size_t(r) * sw] : T(0);
    double a = 0.0, q = 0.0;
#pragma unroll
    for (int r = 0; r < SUM_BLK; ++r) {
        a += double(v[r]);
        q += double(v[r]) * double(v[r]);
    }
    double *o = sums + ((size_t(win) * nblk + b) * 2) * sw + c;
    o[0] = a;
    o[sw] = q;
}

template <class T>
__global__ void __launch_bounds__(256) k_block_sums(const T *img, int sh, int sw, double *sums) {
    block_sums_task(img, sh, sw, blockIdx.x * 4 + (threadIdx.x >> 6), blockIdx.y, sums);
}

// prefix sums over the columns of the window sums of lag rows [u0, u0 + kl): V[2 j] of s,
// V[2 j + 1] of s^2 (rows of sw doubles in LDS); every thread of the NTH calls it
template <int NTH, class T>
__device__ __forceinline__ void lag_row_prefixes(const T *im, const double *sums, int sh, int sw, int th, int u0, int kl,
                                                 double *V) {
    const int lo = min((u0 + SUM_BLK - 1) / SUM_BLK, (u0 + th) / SUM_BLK), hi = (u0 + th) / SUM_BLK;
    for (int c = threadIdx.x; c < sw; c += NTH) {
        double a = 0.0, b = 0.0;
        auto row = [&](int r, double sign) {
            const double v = double(im[size_t(r) * sw + c]);
            a = fma(sign, v, a);
            b = fma(sign * v, v, b);
        };
        #pragma unroll 4
        for (int k = lo; k < hi; ++k) {
            a += sums[size_t(2 * k) * sw + c];
            b += sums[size_t(2 * k + 1) * sw + c];
        }
        #pragma unroll 4
        for (int r = u0; r < min(lo * SUM_BLK, u0 + th); ++r) row(r, 1.0);
        #pragma unroll 4
        for (int r = max(hi * SUM_BLK, u0); r < u0 + th; ++r) row(r, 1.0);
        for (int j = 0; j < kl; ++j) {
            V[size_t(2 * j) * sw + c] = a;
            V[size_t(2 * j + 1) * sw + c] = b;
            if (j + 1 < kl) {
                row(u0 + j + th, 1.0);
                row(u0 + j, -1.0);
            }
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int i = threadIdx.x >> 6; i < 2 * kl; i += NTH / 64) {
        double *v = V + size_t(i) * sw, carry = 0.0;
        for (int c0 = 0; c0 < sw; c0 += 64) {
            const double x = wave_scan_f64(c0 + lane < sw ? v[c0 + lane] : 0.0) + carry;
            if (c0 + lane < sw) v[c0 + lane] = x;
            carry = lane63_f64(x);
        }
    }
    __syncthreads();
}

// 1 / the correlation's norm squared is norm2 + FLT_EPSILON at lag (row j of V, v)
__device__ __forceinline__ double lag_norm2(const double *V, int j, int sw, int v, int tw, double inv, double t2) {
    const double *p1 = V + size_t(2 * j) * sw, *p2 = p1 + sw;
    const double s1 = p1[v + tw - 1] - (v ? p1[v - 1] : 0.0), s2 = p2[v + tw - 1] - (v ? p2[v - 1] : 0.0);
    return (s2 - s1 * s1 * inv) * t2;
}

// corr[w][u][v] /= norm for K lag rows of one window per workgroup; LDS: 2 K sw doubles.
// (841 windows of 128, half search 32, both correlations: 316 us with column sums of every
// lag row through HBM, 252 us with the block sums' pass.)
template <class T>
__global__ void __launch_bounds__(256) k_norm_lags(T *corr, int nl, int nlw, int th, int tw, const T *sr, int sh, int sw,
                                                   const double *sums, const double *ssd, int K) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *V = reinterpret_cast<double *>(smem_raw);
    const int win = blockIdx.y, u0 = blockIdx.x * K, kl = min(K, nl - u0), nblk = (sh + SUM_BLK - 1) / SUM_BLK;
    lag_row_prefixes<256>(sr + size_t(win) * sh * sw, sums + size_t(win) * nblk * 2 * sw, sh, sw, th, u0, kl, V);
    const double t2 = ssd[win], inv = 1.0 / (double(th) * tw);
    T *c = corr + (size_t(win) * nl + u0) * nlw;
    for (int o = threadIdx.x; o < kl * nlw; o += 256) {
        const int j = o / nlw, v = o - j * nlw;
        c[o] = T(double(c[o]) / sqrt(lag_norm2(V, j, sw, v, tw, inv, t2) + double(FLT_EPSILON)));
    }
}

// ---------------------------------------------------------------------------
// Normalized correlation of few windows (the FP64 pipeline: re-runs of near ties, and
// precision 2 up to direct_lags' line), from the row half spectra in two launches instead of four (k_mac_lags,
// k_lagrows_real and the normalization). With few windows those are bound by latency (a
// thread walks a quarter of the search rows, or a whole column), so here
//   k_lag_parts: partial lag sums over template rows [t0, t0 + per): a wave per 64 bins,
//     K lag rows and row part, a sliding window of K search rows in registers; and, in the
//     same launch, the block sums of the search amplitudes;
//   k_corr_lags: one lag row per workgroup (K when there are many windows) sums the parts,
//     evaluates c[v] = (1/L) sum_k Q[k] e^{2 pi i k v / L} at the wanted lags only (8 threads
//     a value) and divides by the norm.
// Windows of 64, half search 20: both correlations of 64 windows 91 -> 62 us, the
// oversampled one of a single window 40 -> 16 us.
// ---------------------------------------------------------------------------
// q[w][part][u][k] = sum over the part's template rows t of conj(T_t[k]) S_{t+u}[k]
template <class T, int K>
__global__ void __launch_bounds__(256) k_lag_parts(const cx<T> *tspec, int th, const cx<T> *sspec, int sh, int nl, int H1,
                                                   int parts, cx<T> *q, int lag_blocks, const T *sr, int sw, double *sums) {
    const int win = blockIdx.y, lane = threadIdx.x & 63;
    if (int(blockIdx.x) >= lag_blocks) {
        block_sums_task(sr, sh, sw, (blockIdx.x - lag_blocks) * 4 + (threadIdx.x >> 6), win, sums);
        return;
    }
    const int bins = (H1 + 63) / 64, task = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int part = task % parts, g = task / parts, k = 64 * (g % bins) + lane, u0 = (g / bins) * K;
    if (k >= H1 || u0 >= nl) return;
    const int per = (th + parts - 1) / parts, t0 = part * per, t1 = min(th, t0 + per);
    const cx<T> *ts = tspec + size_t(win) * th * H1 + k, *ss = sspec + (size_t(win) * sh + u0) * H1 + k;
    const int last = sh - 1 - u0;               // search rows past the end meet only lags past nl
    cx<T> acc[K], s[K];
#pragma unroll
    for (int j = 0; j < K; ++j) acc[j] = cx<T>{T(0), T(0)};
#pragma unroll
    for (int j = 0; j + 1 < K; ++j) s[j] = ss[size_t(min(t0 + j, last)) * H1];
    #pragma unroll 4
    for (int t = t0; t < t1; ++t) {
        const cx<T> tv = ts[size_t(t) * H1];
        s[K - 1] = ss[size_t(min(t + K - 1, last)) * H1];
#pragma unroll
        for (int j = 0; j < K; ++j) acc[j] = cmac_conj(acc[j], tv, s[j]);
#pragma unroll
        for (int j = 0; j + 1 < K; ++j) s[j] = s[j + 1];
    }
    cx<T> *o = q + ((size_t(win) * parts + part) * nl + u0) * H1 + k;
#pragma unroll
    for (int j = 0; j < K; ++j)
        if (u0 + j < nl) o[size_t(j) * H1] = acc[j];
}

// bytes of LDS: Q [K][H1], V [K][2][sw], twiddles [L]
template <class T>
__host__ __device__ inline size_t corr_lags_lds(int K, int L, int sw) {
    return (size_t(K) * (L / 2 + 1) + L) * sizeof(cx<T>) + size_t(2) * K * sw * sizeof(double);
}

template <class T>
__global__ void __launch_bounds__(256) k_corr_lags(const cx<T> *q, int parts, int L, int nl, int nlw, int th, int tw,
                                                   const T *sr, int sh, int sw, const double *sums, const double *ssd,
                                                   const cx<T> *twid, T *out, int K) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int H1 = L / 2 + 1, win = blockIdx.y, u0 = blockIdx.x * K, kl = min(K, nl - u0);
    const int nblk = (sh + SUM_BLK - 1) / SUM_BLK;
    cx<T> *Q = reinterpret_cast<cx<T> *>(smem_raw), *twl = Q + size_t(K) * H1;
    double *V = reinterpret_cast<double *>(twl + L);
    for (int i = threadIdx.x; i < L; i += 256) twl[i] = twid[i];
    const cx<T> *qw = q + (size_t(win) * parts * nl + u0) * H1;
    for (int i = threadIdx.x; i < kl * H1; i += 256) {
        cx<T> v = qw[i];
        #pragma unroll 4
        for (int p = 1; p < parts; ++p) v = v + qw[size_t(p) * nl * H1 + i];
        Q[i] = v;
    }
    lag_row_prefixes<256>(sr + size_t(win) * sh * sw, sums + size_t(win) * nblk * 2 * sw, sh, sw, th, u0, kl, V);
    const double t2 = ssd[win], inv = 1.0 / (double(th) * tw);
    const int slice = threadIdx.x & 7, nyq = L % 2 ? -1 : L / 2;           // an even L's Nyquist bin counts once
    for (int o = threadIdx.x >> 3; o < kl * nlw; o += 32) {
        const int j = o / nlw, v = o - j * nlw;
        const cx<T> *qj = Q + j * H1;
        T acc = T(0);
        int m = int((int64_t(slice) * v) % L);
        const int step = int((int64_t(8) * v) % L);
        for (int k = slice; k < H1; k += 8) {
            const cx<T> w = twl[m];                                        // e^{-2 pi i k v / L}
            const T re = fma(qj[k].x, w.x, qj[k].y * w.y);
            acc += k == 0 || k == nyq ? re : T(2) * re;
            m += step;
            if (m >= L) m -= L;
        }
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) acc += __shfl_xor(acc, d);
        if (slice == 0)
            out[(size_t(win) * nl + u0 + j) * nlw + v] =
                T(double(acc) / double(L) / sqrt(lag_norm2(V, j, sw, v, tw, inv, t2) + double(FLT_EPSILON)));
    }
}

// ---------------------------------------------------------------------------
// normalization (formula of cuCorrNormalization.cu:230-314 and
// cuCorrNormalizationSAT.cu:237-240) with FP64 window sums computed directly:
// per-column vertical sums over the template height, slid down one lag row at
// a time, and horizontal window sums from a block prefix scan of them. One
// 256-thread block per window; dynamic LDS 4*sw + 2 doubles. Used for search
// chips wider than the lag-row form above handles (1024 columns).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void block_scan256(double &x1, double &x2, double *sh4) {
    // inclusive scan of (x1, x2) over the 256 threads; sh4 holds 8 doubles
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const double y1 = __shfl_up(x1, d), y2 = __shfl_up(x2, d);
        if (lane >= d) { x1 += y1; x2 += y2; }
    }
    __syncthreads();
    if (lane == 63) { sh4[wv] = x1; sh4[4 + wv] = x2; }
    __syncthreads();
    for (int k = 0; k < wv; ++k) { x1 += sh4[k]; x2 += sh4[4 + k]; }
}

template <class T>
__global__ void __launch_bounds__(256) k_normalize(T *corr, int ch, int cw, const T *tmpl, int th, int tw,
                                                   const T *srch, int sh, int sw) {
    __shared__ double sh_red[8];
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *V1 = reinterpret_cast<double *>(smem_raw);
    double *V2 = V1 + sw;
    double *P1 = V2 + sw;            // [sw + 1] prefix sums
    double *P2 = P1 + sw + 1;
    const int win = blockIdx.x;
    const T *t = tmpl + size_t(win) * th * tw;
    const T *s = srch + size_t(win) * sh * sw;
    double t2 = 0.0;
    for (int i = threadIdx.x; i < th * tw; i += blockDim.x) {
        const double v = double(t[i]);
        t2 += v * v;
    }
    t2 = block_sum256(t2, sh_red);
    for (int c = threadIdx.x; c < sw; c += blockDim.x) {
        double a1 = 0.0, a2 = 0.0;
        for (int r = 0; r < th; ++r) {
            const double v = double(s[size_t(r) * sw + c]);
            a1 += v;
            a2 += v * v;
        }
        V1[c] = a1;
        V2[c] = a2;
    }
    if (threadIdx.x == 0) { P1[0] = 0.0; P2[0] = 0.0; }
    __syncthreads();
    const int per = (sw + blockDim.x - 1) / blockDim.x;     // columns per thread, contiguous
    const int c0 = threadIdx.x * per, c1 = min(sw, c0 + per);
    const double inv = 1.0 / double(th * tw);
    T *cc = corr + size_t(win) * ch * cw;
    for (int u = 0; u < ch; ++u) {
        double x1 = 0.0, x2 = 0.0;
        for (int c = c0; c < c1; ++c) { x1 += V1[c]; x2 += V2[c]; }
        block_scan256(x1, x2, sh_red);
        double e1 = x1, e2 = x2;                              // inclusive end of this thread's segment
        for (int c = c1 - 1; c >= c0; --c) {
            P1[c + 1] = e1; P2[c + 1] = e2;
            e1 -= V1[c]; e2 -= V2[c];
        }
        __syncthreads();
        for (int v = threadIdx.x; v < cw; v += blockDim.x) {
            const double s1 = P1[v + tw] - P1[v], s2 = P2[v + tw] - P2[v];
            const double norm2 = (s2 - s1 * s1 * inv) * t2;
            cc[u * cw + v] = T(double(cc[u * cw + v]) / sqrt(norm2 + double(FLT_EPSILON)));
        }
        if (u + 1 < ch) {
            for (int c = threadIdx.x; c < sw; c += blockDim.x) {
                const double vn = double(s[size_t(u + th) * sw + c]), vo = double(s[size_t(u) * sw + c]);
                V1[c] += vn - vo;
                V2[c] += vn * vn - vo * vo;
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// argmax with the reference tie rule (cuOffset.cu:23-84), one block per surface
// ---------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(256) k_maxloc(const T *surf, int h, int w, int32_t *loc, T *val, float *margin) {
    __shared__ T shv[4], shv2[4];
    __shared__ uint64_t shk[4];
    const T *s = surf + size_t(blockIdx.x) * h * w;
    Top2<T> top;
    for (int i = threadIdx.x; i < h * w; i += blockDim.x) top.add(s[i], maxloc_key(uint32_t(i)));
    top.template reduce<256>(shv, shv2, shk);
    if (threadIdx.x == 0) {
        const int idx = top.index();
        loc[2 * blockIdx.x] = idx / w;
        loc[2 * blockIdx.x + 1] = idx % w;
        if (val) val[blockIdx.x] = top.v1;
        if (margin) margin[blockIdx.x] = top.margin();
    }
}

// ---------------------------------------------------------------------------
// covariance, SNR, zoom start/shift; one thread per window
// (cuEstimateStats.cu:20-110, cuArraysCopy.cu:249-284, cuCorrNormalization.cu:143-192,
//  cuOffset.cu:190-241)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void adjust_axis(int maxloc, int old_range, int new_range, int &start, int &shift) {
    start = maxloc - new_range;
    shift = 0;
    const int rbound = 2 * (old_range - new_range);
    if (start < 0) { shift = -start; start = 0; }
    else if (start > rbound) { shift = start - rbound; start = rbound; }
}

// covariance from the peak's curvature (cuEstimateStats.cu:49-110); g(dx, dy): the
// normalized surface around the peak, read only when `inner` (the peak has neighbours)
template <class G>
__device__ __forceinline__ void peak_covariance(G g, bool inner, double peak, int template_size, float *cov3) {
    double cxx = 99.0, cyy = 99.0, cxy = 0.0;
    if (inner) {
        double dxx = -(g(1, 0) + g(-1, 0) - 2.0 * g(0, 0)) * template_size;
        double dyy = -(g(0, 1) + g(0, -1) - 2.0 * g(0, 0)) * template_size;
        double dxy = (g(1, 1) + g(-1, -1) - g(1, -1) - g(-1, 1)) * 0.25 * template_size;
        double n2 = fmax(1.0 - peak, 0.0);
        const double n4 = n2 * n2 * 0.5 * template_size;
        n2 *= 2.0;
        const double u = dxy * dxy - dxx * dyy;
        const double u2 = u * u;
        if (fabs(u) >= 1e-2) {
            cxx = (-n2 * u * dyy + n4 * (dyy * dyy + dxy * dxy)) / u2;
            cyy = (-n2 * u * dxx + n4 * (dxx * dxx + dxy * dxy)) / u2;
            cxy = (n2 * u * dxy - n4 * (dxx + dyy) * dxy) / u2;
        }
    }
    cov3[0] = float(cxx); cov3[1] = float(cyy); cov3[2] = float(cxy);
}

// Covariance and SNR of one window's normalized surface, computed by one wave:
// lanes share the SNR patch sum, lane 0 writes both results.
template <class T>
__device__ void window_stats(const T *c, int nx, int ny, int px, int py, double peak, int template_size,
                             int patch_h, int patch_w, float *cov3, float *snr) {
    const int lane = threadIdx.x & 63;
    // SNR over the patch centred on the peak (offset -size/2), zero outside
    double sum = 0.0;
    int count = 0;
    for (int k = lane; k < patch_h * patch_w; k += 64) {
        const int i = k / patch_w, j = k - i * patch_w;
        const int x = px + i - patch_h / 2, y = py + j - patch_w / 2;
        if (x >= 0 && x < nx && y >= 0 && y < ny) {
            const double v = double(c[x * ny + y]);
            sum += v * v;
            ++count;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o);
        count += __shfl_xor(count, o);
    }
    if (lane != 0) return;
    peak_covariance([&](int dx, int dy) { return double(c[(px + dx) * ny + py + dy]); },
                    !(px - 1 < 0 || py - 1 < 0 || px + 1 >= nx || py + 1 >= ny), peak, template_size, cov3);
    const double mean = (sum - peak * peak) / double(count - 1);
    *snr = float(peak * peak / mean);
}

// argmax (k_maxloc), then covariance, SNR and the zoom start/shift of one surface per
// 256-thread block
template <class T>
__global__ void __launch_bounds__(256) k_peak(const T *corr, int nx, int ny, int template_size, int patch_h, int patch_w,
                                              int hs_down, int hs_across, int hz, int32_t *loc, T *val, float *margin,
                                              float *cov, float *snr, int32_t *start, int32_t *shift) {
    __shared__ T shv[4], shv2[4];
    __shared__ uint64_t shk[4];
    const int w = blockIdx.x;
    const T *s = corr + size_t(w) * nx * ny;
    Top2<T> top;
    for (int i = threadIdx.x; i < nx * ny; i += 256) top.add(s[i], maxloc_key(uint32_t(i)));
    top.template reduce<256>(shv, shv2, shk);
    if (threadIdx.x >= 64) return;
    const int idx = top.index(), px = idx / ny, py = idx - px * ny;
    window_stats(s, nx, ny, px, py, double(top.v1), template_size, patch_h, patch_w, cov + 3 * w, snr + w);
    if (threadIdx.x == 0) {
        loc[2 * w] = px; loc[2 * w + 1] = py;
        val[w] = top.v1;
        if (margin) margin[w] = top.margin();
        int s0, h0, s1, h1;
        adjust_axis(px, hs_down, hz, s0, h0);
        adjust_axis(py, hs_across, hz, s1, h1);
        start[2 * w] = s0; start[2 * w + 1] = s1;
        shift[2 * w] = h0; shift[2 * w + 1] = h1;
    }
}

// ---------------------------------------------------------------------------
// deramp method 1 (cuDeramp.cu:67-148) with float2.h's operator*= (imaginary
// part reuses the updated real part); sums, phases and rotation in FP64. The
// phase is separable, c*phx + r*phy: k_deramp_phase writes one FP64 table per
// chip, e^{i r phy} for its h rows then e^{i c phx} for its w columns, and the
// forward row FFT applies the rotation as it loads the chip (deramp_apply).
// ---------------------------------------------------------------------------
// chip win of [nimg][ih][iw] images, cropped at `start` (row, column) when given
template <class T>
__device__ __forceinline__ const cx<T> *crop_origin(const cx<T> *src, int ih, int iw, const int32_t *start, int win) {
    const cx<T> *o = src + size_t(win) * ih * iw;
    return start ? o + start[2 * win] * iw + start[2 * win + 1] : o;
}

// two kinds of chips in one launch: blockIdx.y picks the job
struct PhaseJob {
    ChipSrc chip;
    int h, w;
    cx<double> *tab;
};

static __global__ void __launch_bounds__(1024) k_deramp_phase(PhaseJob a, PhaseJob b) {
    __shared__ double sh[4][16];
    const PhaseJob &j = blockIdx.y ? b : a;
    const int h = j.h, w = j.w, lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int64_t o0 = chip_origin(j.chip, blockIdx.x);
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    // pixels as stored: deramped chips are complex or real images (mode 1 is derampMethod 0)
    constexpr int U = 4;
    with_kind(j.chip, [&](auto real) {
        constexpr bool R = decltype(real)::value;
        chip_pixels<U>(h, w, [&](const int (&r)[U], const int (&c)[U], const bool (&ok)[U]) {
            float2 z[U], x[U], y[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // neighbours past the last column or row count as zero (the pixel itself is read instead)
                const int64_t o = o0 + r[u] * j.chip.pitch + c[u];
                z[u] = chip_raw<R>(j.chip, o);
                x[u] = chip_raw<R>(j.chip, c[u] < w - 1 ? o + 1 : o);
                y[u] = chip_raw<R>(j.chip, r[u] < h - 1 ? o + j.chip.pitch : o);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool right = ok[u] && c[u] < w - 1, below = ok[u] && r[u] < h - 1;
                const double zr = z[u].x, zi = z[u].y;
                const double xr = right ? x[u].x : 0.f, xi = right ? x[u].y : 0.f;
                const double yr = below ? y[u].x : 0.f, yi = below ? y[u].y : 0.f;
                t[0] += zr * xr + zi * xi;      // z * conj(z_right)
                t[1] += zi * xr - zr * xi;
                t[2] += zr * yr + zi * yi;      // z * conj(z_below)
                t[3] += zi * yr - zr * yi;
            }
        });
    });
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        t[k] = wave_scan_f64(t[k]);
        if (lane == 63) sh[k][wv] = t[k];
    }
    __syncthreads();
    cx<double> *rowf = j.tab + size_t(blockIdx.x) * (h + w);
    for (int i = threadIdx.x; i < h + w; i += blockDim.x) {
        const bool row = i < h;
        double re = 0.0, im = 0.0;
        for (int k = 0; k < nw; ++k) {
            re += sh[row ? 0 : 2][k];
            im += sh[row ? 1 : 3][k];
        }
        const double phase = atan2(im, re);
        sincos(double(row ? i : i - h) * phase, &rowf[i].y, &rowf[i].x);
    }
}

template <class T>
__device__ __forceinline__ cx<T> deramp_apply(cx<T> v, cx<double> rf, cx<double> cf) {
    const cx<double> f = cmul(cf, rf);
    const double x = double(v.x), y = double(v.y);
    const double nx = x * f.x - y * f.y;
    const double ny = y * f.x + nx * f.y;
    return {T(nx), T(ny)};
}

// forward row FFT of h x d.n chips read from [nimg][ih][iw] sources (cropped at
// `start` when given: the secondary zoom-in window, cuArraysCopy.cu:209-224),
// deramped on load when `tab` is given, written to dst [nimg][h][d.n] (dst may
// be the source itself when there is no crop); `g` rows per block
template <class T, int DIR>
__global__ void __launch_bounds__(256) k_fft_rows_chip(const cx<T> *src, int ih, int iw, const int32_t *start,
                                                       const cx<double> *tab, cx<T> *dst, int nimg, int h, int g,
                                                       FftDesc d) {
    extern __shared__ unsigned char smem_raw[];
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + g * d.n;
    const int w = d.n, r0 = blockIdx.x * g;
    const int nr = min(g, nimg * h - r0);
    for (int i = threadIdx.x; i < nr * w; i += blockDim.x) {
        const int k = i / w, c = i - k * w;
        const int t = r0 + k, win = t / h, r = t - win * h;
        cx<T> v = crop_origin(src, ih, iw, start, win)[r * iw + c];
        if (tab) {
            const cx<double> *rowf = tab + size_t(win) * (h + w);
            v = deramp_apply(v, rowf[r], rowf[h + c]);
        }
        a[i] = v;
    }
    __syncthreads();
    const cx<T> *res = fft_lds<T, DIR>(a, b, d, nr, 1, w);
    cx<T> *base = dst + size_t(r0) * w;
    for (int i = threadIdx.x; i < nr * w; i += blockDim.x) base[i] = res[i];
}

// ---------------------------------------------------------------------------
// x2 chip oversampling, separable form. The quadrant-padded inverse 2-D FFT of
// the reference's oversampler (cuOverSampler.cpp:72-78 with
// cuArraysPadding.cu:59-103) is the tensor product of one 1-D interpolation
// per axis, because the padding and both transforms factor by axis. Along an
// axis of N samples, output sample 2m is input sample m, and output sample
// 2m+1 is (1/N) FFT_-(FFT_+(x) e^{-i pi k_s/N})[m] with k_s = k for k < N/2 and
// k - N otherwise (the padding puts bin N/2 among the negative frequencies).
// Column pass (k_os2_cols): the odd output rows Y of each chip. Row pass
// (k_os2_rows): every output row (chip row m or Y row m), |.| at even columns
// and |.| of its interpolation at odd columns. Chips are read from
// [nimg][ih][iw] sources, cropped at `start` when given and deramped with
// `tab` when given, as in k_fft_rows_chip.
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ cx<T> half_shift(int k, int n) {
    const int ks = k < n / 2 ? k : k - n;
    double s, c;
    sincospi(-double(ks) / double(n), &s, &c);
    return {T(c / n), T(s / n)};
}

// pixel (r, c) of window win's h x w chip, whose first pixel is at image offset `org`,
// deramped with `tab` when given
template <class T, bool REAL>
__device__ __forceinline__ cx<T> chip_pixel(const ChipSrc &src, int64_t org, const cx<double> *tab, int win, int h, int w,
                                            int r, int c) {
    cx<T> v = chip_value<T>(src, chip_raw<REAL>(src, org + r * src.pitch + c));
    if (tab) {
        const cx<double> *rowf = tab + size_t(win) * (h + w);
        v = deramp_apply(v, rowf[r], rowf[h + c]);
    }
    return v;
}

// `cb` chip columns per block (blockIdx.x), one chip per blockIdx.y; d.n = h;
// Y: [nimg][h][w]
template <class T>
__global__ void __launch_bounds__(256) k_os2_cols(ChipSrc src, const cx<double> *tab, int w, int cb, FftDesc d,
                                                  cx<T> *Y) {
    extern __shared__ unsigned char smem_raw[];
    const int h = d.n;
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + cb * h;
    cx<T> *sh = b + cb * h;
    const int win = blockIdx.y, c0 = blockIdx.x * cb, nc = min(cb, w - c0);
    const int64_t org = chip_origin(src, win);
    with_kind(src, [&](auto real) {
        #pragma unroll 4
        for (int i = threadIdx.x; i < h * nc; i += blockDim.x) {
            const int r = i / nc, c = i - r * nc;
            a[r * cb + c] = chip_pixel<T, decltype(real)::value>(src, org, tab, win, h, w, r, c0 + c);
        }
    });
    for (int k = threadIdx.x; k < h; k += blockDim.x) sh[k] = half_shift<T>(k, h);
    __syncthreads();
    cx<T> *X = fft_lds<T, +1>(a, b, d, nc, cb, 1);
    cx<T> *other = X == a ? b : a;
    for (int i = threadIdx.x; i < h * nc; i += blockDim.x) {
        const int k = i / nc, c = i - k * nc;
        X[k * cb + c] = cmul(X[k * cb + c], sh[k]);
    }
    __syncthreads();
    const cx<T> *res = fft_lds<T, -1>(X, other, d, nc, cb, 1);
    cx<T> *y = Y + size_t(win) * h * w + c0;
    for (int i = threadIdx.x; i < h * nc; i += blockDim.x) {
        const int r = i / nc, c = i - r * nc;
        y[size_t(r) * w + c] = res[r * cb + c];
    }
}

// `g` output rows per block over the nimg * 2h rows; d.n = w; out: [nimg][2h][2w]
// real, |.| (OUT 1) of the oversampled chip. LDS: os2_rows_lds
template <class T>
__host__ __device__ inline size_t os2_rows_lds(int g, int w) {
    return (2 * size_t(g) + 1) * w * sizeof(cx<T>) + size_t(g) * w * sizeof(T) + 8 + size_t(g) * sizeof(int64_t);
}
template <class T>
__global__ void __launch_bounds__(256) k_os2_rows(ChipSrc src, const cx<double> *tab, const cx<T> *Y, int nimg, int h, int g,
                                                  FftDesc d, T *out) {
    extern __shared__ unsigned char smem_raw[];
    const int w = d.n;
    cx<T> *a = reinterpret_cast<cx<T> *>(smem_raw);
    cx<T> *b = a + g * w;
    cx<T> *sh = b + g * w;
    T *amp = reinterpret_cast<T *>(sh + w);
    int64_t *org = reinterpret_cast<int64_t *>((reinterpret_cast<uintptr_t>(amp + size_t(g) * w) + 7) & ~uintptr_t(7));
    const int t0 = blockIdx.x * g;
    const int nr = min(g, nimg * 2 * h - t0);
    for (int k = threadIdx.x; k < nr; k += blockDim.x) org[k] = chip_origin(src, (t0 + k) / (2 * h));
    __syncthreads();
    with_kind(src, [&](auto real) {
        for (int i = threadIdx.x; i < nr * w; i += blockDim.x) {
            const int k = i / w, c = i - k * w;
            const int t = t0 + k, win = t / (2 * h), tr = t - win * 2 * h, m = tr >> 1;
            const cx<T> v = (tr & 1) ? Y[(size_t(win) * h + m) * w + c]
                                     : chip_pixel<T, decltype(real)::value>(src, org[k], tab, win, h, w, m, c);
            a[i] = v;
            amp[i] = amag(v);
        }
    });
    for (int k = threadIdx.x; k < w; k += blockDim.x) sh[k] = half_shift<T>(k, w);
    __syncthreads();
    cx<T> *X = fft_lds<T, +1>(a, b, d, nr, 1, w);
    cx<T> *other = X == a ? b : a;
    for (int i = threadIdx.x; i < nr * w; i += blockDim.x) {
        const int c = i % w;
        X[i] = cmul(X[i], sh[c]);
    }
    __syncthreads();
    const cx<T> *res = fft_lds<T, -1>(X, other, d, nr, 1, w);
    T *o = out + size_t(t0) * 2 * w;
    for (int i = threadIdx.x; i < nr * w; i += blockDim.x) {
        const int k = i / w, c = i - k * w;
        *reinterpret_cast<cx<T> *>(o + size_t(k) * 2 * w + 2 * c) = cx<T>{amp[i], amag(res[i])};
    }
}

// The same two passes for chip sides N = R1 * R2 with the interpolation in place
// (fft_half_sample: three LDS passes), one chip line per LDS row of odd pitch.
// `tw`, `shift`: e^{-2 pi i k/N} and the half-sample shifts, copied into LDS.

// One kind of chips: h x w pixels, Y [nimg][h][w] (odd rows), out [nimg][2h][2w]; twiddles
// and shifts of the column (h) and the row (w) transforms. The first `blocks` workgroups (of a window in the column
// pass, of the launch in the row pass) take the first job of a launch with two.
template <class T>
struct OsJob {
    ChipSrc chip;
    const cx<double> *tab;
    int h, w;
    const cx<T> *tw_h, *shift_h, *tw_w, *shift_w;
    cx<T> *Y;
    T *out;
    double *part;
    int blocks;
};

// CB chip columns of window win (block bx); chip height R1 * R2; LDS: os2_cols_lds
template <class T>
__host__ __device__ constexpr size_t os2_cols_lds(int N, int CB) { return (size_t(N) * (CB + 1) + 2 * N) * sizeof(cx<T>); }
template <class T, int R1, int R2, int CB, int NTH>
__device__ __forceinline__ void os2_cols_body(const OsJob<T> &j, int bx, int win, unsigned char *smem_raw) {
    constexpr int N = R1 * R2, PC = CB + 1;
    cx<T> *C = reinterpret_cast<cx<T> *>(smem_raw);   // [N][PC]: column c at C[c + r * PC]
    cx<T> *twl = C + N * PC, *sh = twl + N;
    const int c0 = bx * CB, nc = min(CB, j.w - c0);
    const int64_t org = chip_origin(j.chip, win);
    with_kind(j.chip, [&](auto real) {
        #pragma unroll 4
        for (int i = threadIdx.x; i < N * CB; i += NTH) {
            const int r = i / CB, c = i - r * CB;
            if (c < nc) C[r * PC + c] = chip_pixel<T, decltype(real)::value>(j.chip, org, j.tab, win, N, j.w, r, c0 + c);
        }
    });
    for (int k = threadIdx.x; k < N; k += NTH) {
        sh[k] = j.shift_h[k];
        twl[k] = j.tw_h[k];
    }
    __syncthreads();
    // consecutive work items hold consecutive columns: the results go out as they are made
    cx<T> *y = j.Y + size_t(win) * N * j.w + c0;
    fft_half_sample<T, R1, R2, NTH>(C, nc, 1, PC, twl, sh, [](int, int, cx<T>) {},
                                    [&](int c, int r, cx<T> v) { y[size_t(r) * j.w + c] = v; });
}

// G output rows (block bx) over the nimg * 2h rows; chip width R1 * R2. With `part`
// (G dividing 2h, so that a block holds rows of one chip only), the block also writes
// the FP64 sums of its amplitudes and of their squares to part[2 bx], part[2 bx + 1].
template <class T>
__host__ __device__ constexpr size_t os2_rows_f_lds(int N, int G) {
    return (size_t(G) * (N + 1) + 2 * N) * sizeof(cx<T>) + size_t(G) * N * sizeof(T);
}
template <class T, int R1, int R2, int G, int NTH>
__device__ __forceinline__ void os2_rows_body(const OsJob<T> &j, int bx, int nimg, unsigned char *smem_raw, int64_t *org,
                                              double *red) {
    constexpr int N = R1 * R2, PR = N + 1;
    cx<T> *C = reinterpret_cast<cx<T> *>(smem_raw);   // [G][PR]
    cx<T> *twl = C + G * PR, *sh = twl + N;
    T *amp = reinterpret_cast<T *>(sh + N);            // [G][N]
    const int h = j.h, t0 = bx * G;
    const int nr = min(G, nimg * 2 * h - t0);
    if (threadIdx.x < nr) org[threadIdx.x] = chip_origin(j.chip, (t0 + threadIdx.x) / (2 * h));
    for (int k = threadIdx.x; k < N; k += NTH) {
        sh[k] = j.shift_w[k];
        twl[k] = j.tw_w[k];
    }
    __syncthreads();
    with_kind(j.chip, [&](auto real) {
        #pragma unroll 2
        for (int i = threadIdx.x; i < nr * N; i += NTH) {
            const int k = i / N, c = i - k * N;
            const int t = t0 + k, win = t / (2 * h), tr = t - win * 2 * h, m = tr >> 1;
            const cx<T> v = (tr & 1) ? j.Y[(size_t(win) * h + m) * N + c]
                                     : chip_pixel<T, decltype(real)::value>(j.chip, org[k], j.tab, win, h, N, m, c);
            C[k * PR + c] = v;
            amp[i] = amag(v);
        }
    });
    __syncthreads();
    fft_half_sample<T, R1, R2, NTH>(C, nr, PR, 1, twl, sh, [](int, int, cx<T>) {},
                                    [&](int k, int c, cx<T> v) { C[k * PR + c] = v; });
    __syncthreads();
    T *o = j.out + size_t(t0) * 2 * N;
    double s1 = 0.0, s2 = 0.0;
    for (int i = threadIdx.x; i < nr * N; i += NTH) {
        const int k = i / N, c = i - k * N;
        const T a0 = amp[i], a1 = amag(C[k * PR + c]);
        *reinterpret_cast<cx<T> *>(o + size_t(k) * 2 * N + 2 * c) = cx<T>{a0, a1};
        s1 += double(a0) + double(a1);
        s2 += double(a0) * double(a0) + double(a1) * double(a1);
    }
    if (j.part) {
        s1 = block_sum256(s1, red);
        s2 = block_sum256(s2, red);
        if (threadIdx.x == 0) {
            j.part[2 * bx] = s1;
            j.part[2 * bx + 1] = s2;
        }
    }
}

// one kind of chips per launch (many windows: each kind keeps its own registers and threads)
template <class T, int R1, int R2, int CB, int NTH = 256>
__global__ void __launch_bounds__(NTH) k_os2_cols_f(OsJob<T> j) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    os2_cols_body<T, R1, R2, CB, NTH>(j, blockIdx.x, blockIdx.y, smem_raw);
}
template <class T, int R1, int R2, int G, int NTH = 256>
__global__ void __launch_bounds__(NTH) k_os2_rows_f(OsJob<T> j, int nimg) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int64_t org[G];
    __shared__ double red[16];
    os2_rows_body<T, R1, R2, G, NTH>(j, blockIdx.x, nimg, smem_raw, org, red);
}

// reference and search chips in one launch (the FP64 pipeline's few windows, where a
// launch more costs what a kernel does): sides A1 * A2 and B1 * B2
template <class T, int A1, int A2, int B1, int B2, int CB>
__global__ void __launch_bounds__(256) k_os2_cols_pair(OsJob<T> a, OsJob<T> b) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if (int(blockIdx.x) < a.blocks) os2_cols_body<T, A1, A2, CB, 256>(a, blockIdx.x, blockIdx.y, smem_raw);
    else os2_cols_body<T, B1, B2, CB, 256>(b, blockIdx.x - a.blocks, blockIdx.y, smem_raw);
}
template <class T, int A1, int A2, int B1, int B2, int G>
__global__ void __launch_bounds__(256) k_os2_rows_pair(OsJob<T> a, OsJob<T> b, int nimg) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int64_t org[G];
    __shared__ double red[16];
    if (int(blockIdx.x) < a.blocks) os2_rows_body<T, A1, A2, G, 256>(a, blockIdx.x, nimg, smem_raw, org, red);
    else os2_rows_body<T, B1, B2, G, 256>(b, blockIdx.x - a.blocks, nimg, smem_raw, org, red);
}

// idx[0..cap) = the first cap windows (in order) whose margins are below the
// thresholds (NaN counts as below), then the first windows that are not, for
// cap <= n. One workgroup of 1024 threads: per 1024-window slice, a ballot
// per wave and the wave totals give each flagged window its slot.
static __global__ void __launch_bounds__(1024) k_select_near(const float *mc, const float *mf, int n, float tc,
                                                             float tf, int cap, int32_t *idx) {
    __shared__ int wtot[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int filled = 0;                     // slots taken so far (the same in every thread)
    for (int pass = 0; pass < 2 && filled < cap; ++pass) {
        for (int c0 = 0; c0 < n && filled < cap; c0 += blockDim.x) {
            const int i = c0 + threadIdx.x;
            bool flag = false;
            if (i < n) {
                const bool near = !(mc[i] >= tc) || !(mf[i] >= tf);
                flag = pass == 0 ? near : !near;
            }
            const unsigned long long m = __ballot(flag);
            const int before = __popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) wtot[wv] = __popcll(m);
            __syncthreads();
            int off = 0, tot = 0;
            for (int k = 0; k < nw; ++k) {
                const int t = wtot[k];
                if (k < wv) off += t;
                tot += t;
            }
            const int slot = filled + off + before;
            if (flag && slot < cap) idx[slot] = i;
            filled += tot;
            __syncthreads();
        }
        if (filled > cap) filled = cap;
    }
}

// mean and sum of squared deviations of each [size] image from nb block sums
// (os2_rows_body's `part`), for the consumer to subtract the mean as it loads the
// image; one wave per image, four a block
static __global__ void __launch_bounds__(256) k_mean_parts(const double *part, int nb, int size, int nimg, double *mean,
                                                           double *ssd) {
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= nimg) return;
    double s1 = 0.0, s2 = 0.0;
    for (int j = lane; j < nb; j += 64) {
        s1 += part[2 * (size_t(w) * nb + j)];
        s2 += part[2 * (size_t(w) * nb + j) + 1];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        s1 += __shfl_xor(s1, o);
        s2 += __shfl_xor(s2, o);
    }
    if (lane == 0) {
        mean[w] = s1 / size;
        ssd[w] = fmax(s2 - s1 * s1 / size, 0.0);
    }
}

template <class T>
__global__ void k_trim_complex(const T *in, int ih, int iw, cx<T> *out, int z) {
    const int win = blockIdx.y;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < z * z; i += gridDim.x * blockDim.x) {
        const int r = i / z, c = i - r * z;
        out[size_t(win) * z * z + i] = {in[size_t(win) * ih * iw + r * iw + c], T(0)};
    }
}

// table of the windowed-sinc surface interpolation: taps * dec coefficients
// (cuSincOverSampler.cu:21-80), TAPS taps of dec phases each
struct SincTable {
    static constexpr int TAPS = 8;
    const float *coef;
    int dec;
};

// Windowed-sinc surface oversampling (cuSincOverSampler.cu:84-195) and its argmax.
// The reference writes a (2*2*covs+1)^2 patch around out/2 + shift*factor into a
// zeroed nout x nout surface and searches all of it; here only the patch is
// evaluated (the weights separate: R[i][y] interpolates along x for `cap` patch
// rows at a time, then each thread keeps one patch column's weights and walks the
// rows) and the zeros enter the argmax as one candidate, the zero that the tie
// rule prefers, and one runner-up. Sums in FP64. a(x, y): the nin x nin trimmed
// surface. Every thread of the workgroup calls it; the caller reduces `top`.
template <int NTH, class T, class A>
__device__ __forceinline__ void sinc_patch_peak(A a, int nin, int nout, int shift0, int shift1, SincTable tb, int covs,
                                                int factor, double *R, int cap, Top2<T> &top) {
    constexpr int TAPS = SincTable::TAPS;
    const int rng = 2 * covs;
    const int x0 = nout / 2 - rng + shift0 * factor, y0 = nout / 2 - rng + shift1 * factor;
    const int size = min(2 * rng + 1, nout);           // distinct positions per axis
    // from [-nout, 2 nout): the patch of the smallest surface (nin = 2) starts before it
    auto wrap = [&](int o) { return o < 0 ? o + nout : o >= nout ? o - nout : o; };
    // integer part and phase of an output position, as the reference computes them
    auto split = [&](int o, int &i, int &f) {
        i = o / covs;
        f = int((float(o) / covs - i) * tb.dec);
    };
    auto tap = [&](int i, int p) {
        int x = i - p + TAPS / 2;
        if (nin == 2) return x & 1;                    // fewer samples than half the taps wrap twice
        if (x < 0) x += nin;
        if (x >= nin) x -= nin;
        return x;
    };
    const int lanes = min(size, NTH), groups = NTH / lanes;
    const int jt = threadIdx.x % lanes, g = threadIdx.x / lanes;
    for (int i0 = 0; i0 < size; i0 += cap) {
        const int ni = min(cap, size - i0);
        for (int t = threadIdx.x; t < ni * nin; t += NTH) {
            const int i = t / nin, y = t - i * nin;
            int xi, xf;
            split(wrap(x0 + i0 + i), xi, xf);
            double acc = 0.0, ws = 0.0;
#pragma unroll
            for (int p = 0; p < TAPS; ++p) {
                const double w = tb.coef[p * tb.dec + xf];
                ws += w;
                acc += w * double(a(tap(xi, p), y));
            }
            R[t] = acc / ws;
        }
        __syncthreads();
        for (int j = jt; j < size && g < groups; j += lanes) {
            const int oy = wrap(y0 + j);
            int yi, yf, yy[TAPS];
            double w[TAPS], ws = 0.0;
            split(oy, yi, yf);
#pragma unroll
            for (int q = 0; q < TAPS; ++q) {
                w[q] = tb.coef[q * tb.dec + yf];
                ws += w[q];
                yy[q] = tap(yi, q);
            }
#pragma unroll
            for (int q = 0; q < TAPS; ++q) w[q] /= ws;
            for (int i = g; i < ni; i += groups) {
                double acc = 0.0;
#pragma unroll
                for (int q = 0; q < TAPS; ++q) acc += w[q] * R[i * nin + yy[q]];
                top.add(T(acc), maxloc_key(uint32_t(wrap(x0 + i0 + i) * nout + oy)));
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && size < nout) {
        // the zeros outside the patch: the first in the tie rule's order, and another
        auto inside = [&](int o, int s) { return (o - s + nout) % nout < size; };
        const int n = nout * nout, s0 = wrap(x0), s1 = wrap(y0);
        for (uint32_t r = 0; r < 512; ++r) {
            int idx = int(bitrev9(r));
            while (idx < n && inside(idx / nout, s0) && inside(idx % nout, s1)) idx += 512;
            if (idx < n) {
                top.add(T(0), maxloc_key(uint32_t(idx)));
                top.add(T(0), (uint64_t(511) << 32) | 0xffffffffu);
                break;
            }
        }
    }
}

// windowed-sinc surface, argmax and sub-pixel offset of the top-left nin x nin of
// corr ([n][ch][cw]); one 256-thread block per window; LDS: cap * nin doubles
template <class T>
__global__ void __launch_bounds__(256) k_sinc_peak(const T *corr, int ch, int cw, int nin, int nout, const int32_t *start,
                                                   const int32_t *shift, SincTable tb, int covs, int factor, int cap,
                                                   int hs_down, int hs_across, float ratio, int32_t *zidx, float *margin,
                                                   float *offset) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ T shv[4], shv2[4];
    __shared__ uint64_t shk[4];
    const int win = blockIdx.x;
    const T *c = corr + size_t(win) * ch * cw;
    Top2<T> top;
    sinc_patch_peak<256>([&](int x, int y) { return c[x * cw + y]; }, nin, nout, shift[2 * win], shift[2 * win + 1], tb, covs,
                         factor, reinterpret_cast<double *>(smem_raw), cap, top);
    top.template reduce<256>(shv, shv2, shk);
    if (threadIdx.x == 0) {
        const int idx = top.index(), px = idx / nout, py = idx - px * nout;
        zidx[2 * win] = px;
        zidx[2 * win + 1] = py;
        offset[2 * win] = ratio * float(px) + float(start[2 * win]) - float(hs_down);
        offset[2 * win + 1] = ratio * float(py) + float(start[2 * win + 1]) - float(hs_across);
        if (margin) margin[win] = top.margin();
    }
}

// final offset (cuOffset.cu:137-146)
// ---------------------------------------------------------------------------
// 16x16 -> SO x SO surface oversampling, SO = 16 M (cuOverSampler.cpp:141-148, real
// part cuArraysCopy.cu:326-339), argmax (cuOffset.cu:23-84) and sub-pixel offset
// (cuOffset.cu:137-187) in one kernel, one NTH-thread block per window. The
// padded SO x SO spectrum has only 16x16 non-zero bins, so with p = M a + b,
// q = M c + d and signed bins ks:
//   G[k1][Mc+d]   = DFT16_k2( A[k1][k2] e^{-2 pi i d ks2/SO} )[c]
//   out[Ma+b][q]  = Re DFT16_k1( G[k1][q] e^{-2 pi i b ks1/SO} )[a]
// where A = (+i 2-D DFT of the trimmed patch) / 256. Needs zoom = 16 and
// 16 M <= NTH, M >= 2 (one thread per surface column). LDS: surface_cx(M) cx<T>.
// ---------------------------------------------------------------------------
// cx<T> values: G[16][SO], the twiddles (tws below), the 16x16 spectrum
__host__ __device__ constexpr int surface_cx(int M) { return 256 + 16 * M + 256 * M; }

template <class T, int NTH>
__global__ void __launch_bounds__(NTH) k_surface(const T *corr, int ch, int cw, int M, const int32_t *start, int hs_down,
                                                 int hs_across, float ratio, const cx<T> *tw, int32_t *zidx,
                                                 float *margin, float *offset) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *a16 = reinterpret_cast<cx<T> *>(smem_raw);
    const int SO = 16 * M;
    cx<T> *tws = a16 + 256;
    cx<T> *G = tws + SO;
    constexpr int NW = NTH / 64;
    __shared__ T shv[NW], shv2[NW];
    __shared__ uint64_t shk[NW];
    const int win = blockIdx.x;
    const T *c = corr + size_t(win) * ch * cw;
    if (threadIdx.x < 256) {
        const int r = threadIdx.x >> 4, q = threadIdx.x & 15;
        a16[threadIdx.x] = {c[r * cw + q] * T(1.0 / 256.0), T(0)};
    }
    if (threadIdx.x < SO) tws[threadIdx.x] = tw[threadIdx.x];
    __syncthreads();
    if (threadIdx.x < 16) {
        cx<T> x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = a16[threadIdx.x * 16 + q];
        dft16<T, +1>(x);
#pragma unroll
        for (int q = 0; q < 16; ++q) a16[threadIdx.x * 16 + q] = x[q];
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        cx<T> x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = a16[r * 16 + threadIdx.x];
        dft16<T, +1>(x);
#pragma unroll
        for (int r = 0; r < 16; ++r) a16[r * 16 + threadIdx.x] = x[r];
    }
    __syncthreads();
    if (threadIdx.x < SO) {
        const int k1 = threadIdx.x / M, dd = threadIdx.x - k1 * M;
        cx<T> x[16];
#pragma unroll
        for (int k2 = 0; k2 < 16; ++k2) {
            const int t = dd * (k2 < 8 ? k2 : k2 - 16);         // |t| < SO / 2
            x[k2] = cmul(a16[k1 * 16 + k2], tws[t < 0 ? t + SO : t]);
        }
        dft16<T, -1>(x);
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) G[k1 * SO + M * cc + dd] = x[cc];
    }
    __syncthreads();
    // Column pruning: every value of column q is at most B_q = sum_k1 |G[k1][q]|
    // and the surface passes through the 16x16 samples, so its maximum is at
    // least their largest value amax. Columns with B_q (1 + 2^-10) + 2^-11 |a|max
    // < amax hold neither the argmax nor any value within 2^-12 |a|max of it, and
    // are skipped (argmax, tie rule and margins below that are unchanged; NaN
    // bounds keep their column).
    __shared__ uint64_t masks[NW];
    __shared__ int cols[NTH];
    T amax = -INFINITY, amag = T(0);
    for (int i = threadIdx.x & 63; i < 256; i += 64) {
        const T v = c[(i >> 4) * cw + (i & 15)];
        amax = fmax(amax, v);
        amag = fmax(amag, fabs(v));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        amax = fmax(amax, __shfl_xor(amax, o));
        amag = fmax(amag, __shfl_xor(amag, o));
    }
    bool keep = false;
    if (threadIdx.x < SO) {
        T bq = T(0);
#pragma unroll
        for (int k1 = 0; k1 < 16; ++k1) {
            const cx<T> g = G[k1 * SO + threadIdx.x];
            if constexpr (sizeof(T) == 8) {
                // max + min / 2 is never below the modulus (and at most 12% above), and
                // costs a tenth of an FP64 square root
                const T x = fabs(g.x), y = fabs(g.y);
                bq += fma(T(0.5), fmin(x, y), fmax(x, y));
            } else {
                bq += ampcor::amag(g);
            }
        }
        keep = !(bq * T(1.0 + 0x1p-10) + T(0x1p-11) * amag < amax);
    }
    const uint64_t wm = __ballot(keep);
    if ((threadIdx.x & 63) == 0) masks[threadIdx.x >> 6] = wm;
    __syncthreads();
    int ncols = 0, before = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int n = __popcll(masks[w]);
        if (w < (threadIdx.x >> 6)) before += n;
        ncols += n;
    }
    if (keep) cols[before + __popcll(wm & ((uint64_t(1) << (threadIdx.x & 63)) - 1))] = threadIdx.x;
    __syncthreads();
    Top2<T> top;
    #pragma unroll 1
    for (int t = threadIdx.x; t < M * ncols; t += NTH) {
        const int b = t / ncols, qq = cols[t - b * ncols];
        cx<T> x[16];
#pragma unroll
        for (int k1 = 0; k1 < 16; ++k1) {
            const int k = b * (k1 < 8 ? k1 : k1 - 16);
            x[k1] = cmul(G[k1 * SO + qq], tws[k < 0 ? k + SO : k]);
        }
        dft16<T, -1>(x);
#pragma unroll
        for (int aa = 0; aa < 16; ++aa) top.add_idx(x[aa].x, uint32_t((M * aa + b) * SO + qq));
    }
    top.template reduce<NTH>(shv, shv2, shk);
    if (threadIdx.x == 0) {
        const int idx = top.index();
        const int px = idx / SO, py = idx - px * SO;
        zidx[2 * win] = px;
        zidx[2 * win + 1] = py;
        offset[2 * win] = ratio * float(px) + float(start[2 * win]) - float(hs_down);
        offset[2 * win + 1] = ratio * float(py) + float(start[2 * win + 1]) - float(hs_across);
        if (margin) margin[win] = top.margin();
    }
}

static __global__ void k_subpixel(const int32_t *start, const int32_t *zidx, int n, float ratio, int hs_down,
                           int hs_across, float *offset) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n) return;
    offset[2 * w] = ratio * float(zidx[2 * w]) + float(start[2 * w]) - float(hs_down);
    offset[2 * w + 1] = ratio * float(zidx[2 * w + 1]) + float(start[2 * w + 1]) - float(hs_across);
}

// ---------------------------------------------------------------------------
// FP64 sub-pixel refinement of the oversampled-surface peak. No counterpart in
// the reference, whose offset is the bare argmax on the 1/(surf_ovs*raw_ovs)
// grid (cuOffset.cu:137-187). The surface is the FFT interpolation of the
// trimmed Z x Z surface a (spectrum zero-padded to N = Z*ovs with the Nyquist
// bin on the negative side, real part; cuOverSampler.cpp:141-148), so at any
// integer (X, Y) of the N x N grid
//   s(X, Y) = Re (1/Z^2) sum_{r,c} a[r][c] D(r, X) D(c, Y),
//   D(r, X) = sum_{f=-Z/2}^{Z/2-1} e^{2 pi i f (r ovs - X)/N},
// which is evaluated in FP64 at the peak (px, py) and its four axis neighbours
// (wrapping, as the interpolation is periodic); a parabola through each axis'
// three values gives the vertex d in [-1/2, 1/2], and the refined offset is
// (p + d)/(ovs * raw_ovs) + start - hs. One wave per window; the trimmed
// surface is the top-left Z x Z of surf ([n][ch][cw]); LDS: refine_lds(Z).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double parabola_vertex(double fm, double f0, double fp) {
    const double den = fm - 2.0 * f0 + fp;
    const double d = den < 0.0 ? 0.5 * (fm - fp) / den : 0.0;
    return fmin(0.5, fmax(-0.5, d));
}

__host__ __device__ inline size_t refine_lds(int Z) { return sizeof(double) * (size_t(Z) * Z + 5) + 16 * 9 * size_t(Z); }

template <class T>
__global__ void __launch_bounds__(64) k_refine(const T *surf, int ch, int cw, int Z, int ovs, double ratio,
                                               const int32_t *zidx, const int32_t *start, int hs_d, int hs_a,
                                               const cx<double> *tw, double *out) {
    extern __shared__ __align__(16) unsigned char smem[];
    cx<double> *D = reinterpret_cast<cx<double> *>(smem);    // [2 axes][3][Z]
    cx<double> *B = D + 6 * Z;                                 // [3][Z]
    double *a = reinterpret_cast<double *>(B + 3 * Z);         // [Z][Z]
    double *s5 = a + Z * Z;
    const int w = blockIdx.x, lane = threadIdx.x;
    const int N = Z * ovs;
    const T *src = surf + size_t(w) * ch * cw;
    for (int i = lane; i < Z * Z; i += 64) a[i] = double(src[(i / Z) * cw + i % Z]);
    const int px = zidx[2 * w], py = zidx[2 * w + 1];
    // D(r, p - 1 + t) for both axes (e^{+2 pi i k/N} = conj(tw[k])); the table
    // index f*m mod N advances by m from f = -Z/2 on
    for (int i = lane; i < 6 * Z; i += 64) {
        const int axis = i / (3 * Z), j = i - axis * 3 * Z, t = j / Z, r = j - t * Z;
        const int X = (axis ? py : px) - 1 + t;
        const int m = ((r * ovs - X) % N + N) % N;
        int k = int((int64_t(N - Z / 2) * m) % N);
        cx<double> acc{0.0, 0.0};
        for (int f = 0; f < Z; ++f) {
            acc.x += tw[k].x;
            acc.y -= tw[k].y;
            k += m;
            if (k >= N) k -= N;
        }
        D[i] = acc;
    }
    __syncthreads();
    // B[t][r] = sum_c a[r][c] D(c, py - 1 + t)
    for (int i = lane; i < 3 * Z; i += 64) {
        const int t = i / Z, r = i - t * Z;
        const cx<double> *dy = D + (3 + t) * Z;
        cx<double> acc{0.0, 0.0};
        for (int c = 0; c < Z; ++c) {
            acc.x += a[r * Z + c] * dy[c].x;
            acc.y += a[r * Z + c] * dy[c].y;
        }
        B[i] = acc;
    }
    __syncthreads();
    // the centre and its four axis neighbours: (tx, ty) = (1,1) (0,1) (2,1) (1,0) (1,2)
    if (lane < 5) {
        const int tx = lane == 1 ? 0 : (lane == 2 ? 2 : 1);
        const int ty = lane == 3 ? 0 : (lane == 4 ? 2 : 1);
        double acc = 0.0;
        for (int r = 0; r < Z; ++r) {
            const cx<double> d = D[tx * Z + r], b = B[ty * Z + r];
            acc += d.x * b.x - d.y * b.y;
        }
        s5[lane] = acc / (double(Z) * Z);
    }
    __syncthreads();
    if (lane == 0) {
        const double dx = parabola_vertex(s5[1], s5[0], s5[2]);
        const double dy = parabola_vertex(s5[3], s5[0], s5[4]);
        out[2 * w] = (double(px) + dx) * ratio + double(start[2 * w]) - double(hs_d);
        out[2 * w + 1] = (double(py) + dy) * ratio + double(start[2 * w + 1]) - double(hs_a);
    }
}

}  // namespace ampcor
