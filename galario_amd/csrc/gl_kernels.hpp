// Pipeline kernels: profile/image -> shifted R2C spectrum -> sampled visibilities -> chi2.
//
// Data layout in HBM (one evaluation):
//   Tm  : row-transformed image, only the 2*Rs rows that can be non-zero,
//         row-major [2*Rs][ldT] complex (ldT >= N/2+1).  Compact row kk maps
//         to quadrant-shifted image row kk (kk < Rs) or N-2*Rs+kk (kk >= Rs).
//   S   : shifted spectrum, column-major [N/2+1][ldS] complex: element
//         (v-row r, u-column l) at l*ldS + r, r = (k + N/2) mod N for FFT row
//         k (the reference's fftshift_axis0 folded into the stores).
//         The four interpolation corners are then two 32-byte pairs.
//
// The stages that restate galario arithmetic (sweep, central pixel, and on
// the complex spectrum and in float interpolation, phase and chi2 terms) are
// compiled without FMA contraction so they round exactly as the reference's
// -std=c++11 x86-64 build.  In double on the real spectrum the sample point
// has a shorter order with explicit fused operations (sym_position and below).
#pragma once

#include <type_traits>

#include "gl_common.hpp"
#include "gl_fft.hpp"

namespace gl {

enum { SRC_SWEEP = 0, SRC_IMAGE_SHIFT = 1, SRC_IMAGE_PLAIN = 2 };
enum { OUT_COLMAJOR_SHIFT = 0, OUT_ROWMAJOR_PLAIN = 1 };
enum { MODE_VIS = 0, MODE_CHI2 = 1 };

// ---------------------------------------------------------------------------
// sweep (galario.cpp:1048-1071) and central pixel (galario.cpp:1214-1232)
// ---------------------------------------------------------------------------
template <typename T>
struct SweepPrm {
    const T* I;        // radial profile, nr values (device)
    int nr;
    T Rmin, dR, dxy, cos_inc, sr_to_px;
    int iIN;           // floor((dxy/2 - Rmin)/dR), validated on the host
    int rmax;          // half side of the swept box (0: only the central pixel)
};

// Pixel value at x = xi*dxy, y = yi*dxy (xi = N/2 - column, yi = N/2 - row).
template <typename T>
__device__ __forceinline__ T sweep_pixel(int xi, int yi, const SweepPrm<T>& p) {
    const T x = T(xi) * p.dxy;
    const T y = T(yi) * p.dxy;
    T r;
    if constexpr (std::is_same<T, double>::value) {
        const double xs = x / p.cos_inc;
        r = sqrt(xs * xs + y * y);
    } else {
        // pow(float, 2) and the sum are double in the reference; r is stored as float
        const double xs = double(x / p.cos_inc);
        r = float(sqrt(xs * xs + double(y) * double(y)));
    }
    T fi = floor((r - p.Rmin) / p.dR);
    fi = fi > T(0) ? fi : T(0);
    if (!(fi <= T(p.nr - 2))) return T(0);
    const int iR = int(fi);
    const T I0 = p.I[iR], I1 = p.I[iR + 1];
    return p.sr_to_px * (I0 + (r - T(iR) * p.dR - p.Rmin) * (I1 - I0) / p.dR);
}

// Central pixel (create_image_d's central value, galario.cpp:1135-1154): the
// profile's flux inside the pixel's inscribed disc over its area.  I(i)
// returns profile value i; it is read for i = 0..iIN+1.
template <typename T, class Prof>
__device__ __forceinline__ T central_value_of(const SweepPrm<T>& p, Prof I) {
    const int iIN = p.iIN;
    const T Rmin = p.Rmin, dR = p.dR;
    T flux = T(0);
    for (int i = 1; i < iIN; ++i) flux += (Rmin + dR * T(i)) * I(i);
    flux = T(double(flux) * 2.0);
    flux += Rmin * I(0) + (Rmin + T(iIN) * dR) * I(iIN);
    flux *= dR;
    const double half = double(p.dxy) / 2.0;
    if constexpr (std::is_same<T, double>::value) {
        const double I_interp = (I(iIN + 1) - I(iIN)) / dR * (half - (Rmin + dR * iIN)) + I(iIN);
        flux += ((Rmin + iIN * dR) * I(iIN) + half * I_interp) * (half - (Rmin + iIN * dR));
        const double area = half * half - Rmin * Rmin;
        return p.sr_to_px * flux / area;
    } else {
        const float edge = Rmin + dR * float(iIN);
        const float I_interp = float(double((I(iIN + 1) - I(iIN)) / dR) * (half - double(edge)) + double(I(iIN)));
        const double term = (double(edge * I(iIN)) + half * double(I_interp)) * (half - double(edge));
        flux = float(double(flux) + term);
        const float area = float(half * half - double(Rmin) * double(Rmin));
        return p.sr_to_px * flux / area;
    }
}

template <typename T>
__device__ __noinline__ T central_value(const SweepPrm<T>& p) {
    return central_value_of(p, [&](int i) { return p.I[i]; });
}

// Value of quadrant-shifted image pixel (row k, column n) built from a profile.
template <typename T>
__device__ __forceinline__ T sweep_shifted(int k, int n, int N, const SweepPrm<T>& p) {
    if (k == 0 && n == 0) return central_value(p);
    if (p.rmax == 0) return T(0);
    const int xi = n < N / 2 ? -n : N - n;
    const int yi = k < N / 2 ? -k : N - k;
    return sweep_pixel(xi, yi, p);
}

// ---------------------------------------------------------------------------
// row pass: 2 real rows per workgroup packed as one complex N-point FFT
// ---------------------------------------------------------------------------
template <typename T>
struct RowArgs {
    SweepPrm<T> sw;              // SRC_SWEEP
    const T* img;                // SRC_IMAGE_*: N rows of ldimg reals (image in the first N)
    int ldimg;
    int N, Rs, ldT;
    const cpx<T>* tw;            // W_N^e table
    cpx<T>* Tm;                  // out: [2*Rs][ldT]
};

__device__ __forceinline__ int compact_to_row(int kk, int Rs, int N) { return kk < Rs ? kk : kk + N - 2 * Rs; }

template <typename T, int SRC>
__device__ __forceinline__ T row_source(const RowArgs<T>& a, int k, int n) {
    const int N = a.N;
    if constexpr (SRC == SRC_SWEEP) {
        return sweep_shifted(k, n, N, a.sw);
    } else if constexpr (SRC == SRC_IMAGE_SHIFT) {
        const int i = k + N / 2 < N ? k + N / 2 : k - N / 2;
        const int j = n + N / 2 < N ? n + N / 2 : n - N / 2;
        return a.img[size_t(i) * a.ldimg + j];
    } else {
        return a.img[size_t(k) * a.ldimg + n];
    }
}

template <typename T, int LOG2N, int SRC>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_rowpass(RowArgs<T> a) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    __shared__ T lds[S::LDS_ELEMS];
    const int tid = threadIdx.x;
    const int kk_a = 2 * blockIdx.x, kk_b = kk_a + 1;
    const int ka = compact_to_row(kk_a, a.Rs, N), kb = compact_to_row(kk_b, a.Rs, N);
    cpx<T> v[E];
    F::run(v, lds, tid, a.Rs, a.tw, [&](int n) -> cpx<T> {
        return cpx<T>{row_source<T, SRC>(a, ka, n), row_source<T, SRC>(a, kb, n)};
    });
    // X_a[l] = (Z[l] + conj Z[N-l]) / 2, X_b[l] = (Z[l] - conj Z[N-l]) / 2i, one component at a time
    const int C = N / 2 + 1;
    cpx<T>* outa = a.Tm + size_t(kk_a) * a.ldT;
    cpx<T>* outb = a.Tm + size_t(kk_b) * a.ldT;
#pragma unroll
    for (int r = 0; r < E; ++r) lds[lpad(tid + r * NT)] = v[r].re;
    __syncthreads();
    for (int l = tid; l < C; l += NT) {
        const T zr = lds[lpad(l)], wr = lds[lpad((N - l) & (N - 1))];
        outa[l].re = T(0.5) * (zr + wr);
        outb[l].im = T(0.5) * (wr - zr);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) lds[lpad(tid + r * NT)] = v[r].im;
    __syncthreads();
    for (int l = tid; l < C; l += NT) {
        const T zi = lds[lpad(l)], wi = lds[lpad((N - l) & (N - 1))];
        outa[l].im = T(0.5) * (zi - wi);
        outb[l].re = T(0.5) * (zi + wi);
    }
}

// ---------------------------------------------------------------------------
// column pass: one column of the row-transformed image per workgroup
// ---------------------------------------------------------------------------
template <typename T>
struct ColArgs {
    const cpx<T>* Tm;
    int N, Rs, ldT;
    const cpx<T>* tw;
    cpx<T>* S;
    size_t ldS;      // OUT_COLMAJOR_SHIFT: column stride; OUT_ROWMAJOR_PLAIN: unused (row stride C)
};

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous run of columns so that the strided reads of Tm share L2 lines.
__device__ __forceinline__ int xcd_column(int b, int nblocks) {
    const int per = nblocks >> 3;
    return (b & 7) * per + (b >> 3);
}

template <typename T, int LOG2N, int OUT>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_colpass(ColArgs<T> a) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    constexpr int C = N / 2 + 1;
    __shared__ T lds[S::LDS_ELEMS];
    const int col = xcd_column(blockIdx.x, gridDim.x);
    if (col >= C) return;
    const int tid = threadIdx.x;
    const int Rs = a.Rs;
    const cpx<T>* src = a.Tm + col;
    const size_t ldT = a.ldT;
    cpx<T> v[E];
    F::run(v, lds, tid, Rs, a.tw, [&](int n) -> cpx<T> {
        const int kk = n < Rs ? n : n - N + 2 * Rs;
        return src[size_t(kk) * ldT];
    });
    if constexpr (OUT == OUT_COLMAJOR_SHIFT) {
        cpx<T>* dst = a.S + size_t(col) * a.ldS;
#pragma unroll
        for (int r = 0; r < E; ++r) dst[(tid + r * NT + N / 2) & (N - 1)] = v[r];
    } else {
#pragma unroll
        for (int r = 0; r < E; ++r) a.S[size_t(tid + r * NT) * C + col] = v[r];
    }
}

// ---------------------------------------------------------------------------
// other even N: direct DFT with exact twiddle indices, each output one chain of fused multiply-adds over n.
// (A fast transform of such a size, Bluestein's with two power-of-two transforms, errs 4 to 6 times as much in the weak
// cells, the long baselines: its errors follow the strongest cell, a chain's its own largest partial sum. 400 x 400
// pixels of a compact source in double, median error of the cells below 1e-3 of the peak: 4.3e-15 against 6.7e-16.)
// A thread sums 2 frequencies (256 apart) of 4 rows or columns, so that a twiddle, gathered from the table
// in LDS, serves 4 sums and its index arithmetic 8 or 16 multiply-adds.  What bounds it: those, and the LDS reads (a
// gathered table padded against bank conflicts costs more than it saves: in float 76 + 104 us against 71 + 98).
// 1000 x 1000 pixels: with one sum per thread and a twiddle from memory for each term 900 us in float and a sampleImage call of
// 1400 us in double; 158 us (double: 86 + 126) and a call of 480 us now.
// ---------------------------------------------------------------------------
constexpr int DFT_LINES = 4, DFT_FREQS = 512, DFT_STAGE = 256;
constexpr size_t DFT_TABLE_BYTES = 65536;   // largest table: two workgroups per CU

// W_N^(n f) for n = 0, 1, ...: byte offset of the table's entry, B n f mod B N for entries of B bytes
template <typename T>
struct TwiddleWalk {
    static constexpr unsigned B = sizeof(cpx<T>);
    unsigned at, step, end;
    __device__ __forceinline__ void start(int f, int N, int n) {
        end = B * unsigned(N);
        step = B * unsigned(f);
        at = B * unsigned((long long)n * f % N);
    }
    __device__ __forceinline__ cpx<T> next(const unsigned char* tw) {
        const cpx<T> w = *reinterpret_cast<const cpx<T>*>(tw + at);
        const unsigned t = at + step;
        at = min(t, t - end);                      // (t < end: t - end wraps beyond it)
        return w;
    }
};

template <typename T>
__device__ __forceinline__ void load_twiddles(unsigned char* lds, const cpx<T>* tw, int N, int tid) {
    for (int e = tid; e < N; e += 256) reinterpret_cast<cpx<T>*>(lds)[e] = tw[e];
}

// acc + y w: y real (rows) or complex (columns)
template <typename T>
__device__ __forceinline__ void dft_term(cpx<T>& acc, T y, cpx<T> w) {
    acc.re = ffma(y, w.re, acc.re);
    acc.im = ffma(y, w.im, acc.im);
}
template <typename T>
__device__ __forceinline__ void dft_term(cpx<T>& acc, cpx<T> y, cpx<T> w) {
    acc.re = ffma(y.re, w.re, ffma(-y.im, w.im, acc.re));
    acc.im = ffma(y.re, w.im, ffma(y.im, w.re, acc.im));
}

// Terms from .. to - 1 of a stage (x in LDS) added to the sums; a group of dft_ahead terms is read ahead
// (1000 x 1000 pixels leave one wave per SIMD: in float rows and columns 66 + 92 us with 8, 71 + 98 with 4, 95 + 115 with
// 2; in double a sampleImage call takes 481 us with 4, 490 with 2, and at 2000 x 2000, 2.46 and 2.27 ms).
template <typename T>
constexpr int dft_ahead() { return sizeof(T) == 4 ? 8 : 4; }

template <typename T, typename X>
struct DftTerms {
    cpx<T> p, q;
    X y[DFT_LINES];
};
template <typename T, typename X>
__device__ __forceinline__ void dft_terms(const X (*x)[DFT_LINES], const unsigned char* tw, TwiddleWalk<T>& wa,
                                          TwiddleWalk<T>& wb, int from, int to, cpx<T> (&A)[DFT_LINES],
                                          cpx<T> (&B)[DFT_LINES]) {
    using Term = DftTerms<T, X>;
    const auto read = [&](Term& t, int s) {
        t.p = wa.next(tw);
        t.q = wb.next(tw);
#pragma unroll
        for (int r = 0; r < DFT_LINES; ++r) t.y[r] = x[s][r];
    };
    const auto add = [&](const Term& t) {
#pragma unroll
        for (int r = 0; r < DFT_LINES; ++r) {
            dft_term(A[r], t.y[r], t.p);
            dft_term(B[r], t.y[r], t.q);
        }
    };
    constexpr int G = dft_ahead<T>();
    int s = from;
    if (to - from >= G) {
        Term cur[G];
#pragma unroll
        for (int g = 0; g < G; ++g) read(cur[g], s + g);
#pragma unroll 2
        for (; s + 2 * G <= to; s += G) {
            Term nxt[G];
#pragma unroll
            for (int g = 0; g < G; ++g) read(nxt[g], s + G + g);
#pragma unroll
            for (int g = 0; g < G; ++g) add(cur[g]);
#pragma unroll
            for (int g = 0; g < G; ++g) cur[g] = nxt[g];
        }
#pragma unroll
        for (int g = 0; g < G; ++g) add(cur[g]);
        s += G;
    }
    for (; s < to; ++s) {
        Term t;
        read(t, s);
        add(t);
    }
}

// All 2 Rs terms of DFT_LINES lines at frequencies fa and fb; load(s, x) fills a term's values.
template <typename T, typename X, typename Load>
__device__ __forceinline__ void dft_tile(X (*x)[DFT_LINES], const unsigned char* tw, int N, int Rs, int fa, int fb,
                                         cpx<T> (&A)[DFT_LINES], cpx<T> (&B)[DFT_LINES], Load&& load) {
    const int tid = threadIdx.x;
    TwiddleWalk<T> wa, wb;
    wa.start(fa, N, 0);
    wb.start(fb, N, 0);
    X y[DFT_LINES];
    if (tid < 2 * Rs) load(tid, y);
    for (int s0 = 0; s0 < 2 * Rs; s0 += DFT_STAGE) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < DFT_LINES; ++r) x[tid][r] = y[r];
        __syncthreads();
        if (s0 + DFT_STAGE + tid < 2 * Rs) load(s0 + DFT_STAGE + tid, y);
        const int end = min(DFT_STAGE, 2 * Rs - s0), cut = min(max(Rs - s0, 0), end);
        dft_terms(x, tw, wa, wb, 0, cut, A, B);
        if (s0 <= Rs && Rs < s0 + end) {           // (the support goes on at n = N - Rs)
            wa.start(fa, N, N - Rs);
            wb.start(fb, N, N - Rs);
        }
        dft_terms(x, tw, wa, wb, cut, end, A, B);
    }
}

template <typename T, int SRC>
__global__ __launch_bounds__(256) void k_rowdft_tiled(RowArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];    // twiddle table
    __shared__ __align__(16) T x[DFT_STAGE][DFT_LINES];
    const int N = a.N, Rs = a.Rs, C = N / 2 + 1, tid = threadIdx.x;
    const int kk0 = DFT_LINES * blockIdx.x, l0 = DFT_FREQS * blockIdx.y + tid;
    load_twiddles(smem_raw, a.tw, N, tid);
    int k[DFT_LINES];
#pragma unroll
    for (int r = 0; r < DFT_LINES; ++r) k[r] = compact_to_row(min(kk0 + r, 2 * Rs - 1), Rs, N);
    cpx<T> A[DFT_LINES] = {}, B[DFT_LINES] = {};
    dft_tile(x, smem_raw, N, Rs, min(l0, C - 1), min(l0 + 256, C - 1), A, B, [&](int s, T (&y)[DFT_LINES]) {
        const int n = s < Rs ? s : s + N - 2 * Rs;
#pragma unroll
        for (int r = 0; r < DFT_LINES; ++r) y[r] = row_source<T, SRC>(a, k[r], n);
    });
#pragma unroll
    for (int r = 0; r < DFT_LINES; ++r) {
        if (kk0 + r >= 2 * Rs) break;
        cpx<T>* out = a.Tm + size_t(kk0 + r) * a.ldT;
        if (l0 < C) out[l0] = A[r];
        if (l0 + 256 < C) out[l0 + 256] = B[r];
    }
}

// (the row spectra are padded to whole groups of four columns)
template <typename T, int OUT>
__global__ __launch_bounds__(256) void k_coldft_tiled(ColArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];    // twiddle table
    __shared__ __align__(16) cpx<T> x[DFT_STAGE][DFT_LINES];
    const int N = a.N, Rs = a.Rs, C = N / 2 + 1, tid = threadIdx.x;
    const int c0 = DFT_LINES * blockIdx.x, k0 = DFT_FREQS * blockIdx.y + tid;
    load_twiddles(smem_raw, a.tw, N, tid);
    cpx<T> A[DFT_LINES] = {}, B[DFT_LINES] = {};
    dft_tile(x, smem_raw, N, Rs, min(k0, N - 1), min(k0 + 256, N - 1), A, B, [&](int s, cpx<T> (&y)[DFT_LINES]) {
        const cpx<T>* src = a.Tm + size_t(s) * a.ldT + c0;
#pragma unroll
        for (int c = 0; c < DFT_LINES; ++c) y[c] = src[c];
    });
    const auto store = [&](int col, int k, cpx<T> X) {
        if (col >= C || k >= N) return;
        if constexpr (OUT == OUT_COLMAJOR_SHIFT) a.S[size_t(col) * a.ldS + (k < N / 2 ? k + N / 2 : k - N / 2)] = X;
        else a.S[size_t(k) * C + col] = X;
    };
#pragma unroll
    for (int c = 0; c < DFT_LINES; ++c) {
        store(c0 + c, k0, A[c]);
        store(c0 + c, k0 + 256, B[c]);
    }
}

// ---------------------------------------------------------------------------
// even N whose twiddle table is too large for that (in double beyond 4096, in float beyond 8192): as above, one output
// at a time.
// ---------------------------------------------------------------------------
template <typename T, int SRC>
__global__ __launch_bounds__(256) void k_rowdft_generic(RowArgs<T> a) {
    extern __shared__ unsigned char smem_raw[];
    T* x = reinterpret_cast<T*>(smem_raw);           // 2*Rs support values
    const int N = a.N, Rs = a.Rs, C = N / 2 + 1;
    const int kk = blockIdx.x;
    const int k = compact_to_row(kk, Rs, N);
    for (int s = threadIdx.x; s < 2 * Rs; s += blockDim.x) {
        const int n = s < Rs ? s : s + N - 2 * Rs;
        x[s] = row_source<T, SRC>(a, k, n);
    }
    __syncthreads();
    cpx<T>* out = a.Tm + size_t(kk) * a.ldT;
    for (int l = threadIdx.x; l < C; l += blockDim.x) {
        T re = 0, im = 0;
        int e = 0;                                     // (n*l) mod N for n = 0, 1, ...
        for (int s = 0; s < Rs; ++s) {
            const cpx<T> w = a.tw[e];
            re = ffma(x[s], w.re, re);
            im = ffma(x[s], w.im, im);
            e += l; if (e >= N) e -= N;
        }
        e = int((long long)(N - Rs) * l % N);
        for (int s = Rs; s < 2 * Rs; ++s) {
            const cpx<T> w = a.tw[e];
            re = ffma(x[s], w.re, re);
            im = ffma(x[s], w.im, im);
            e += l; if (e >= N) e -= N;
        }
        out[l] = cpx<T>{re, im};
    }
}

template <typename T, int OUT>
__global__ __launch_bounds__(256) void k_coldft_generic(ColArgs<T> a) {
    extern __shared__ unsigned char smem_raw[];
    cpx<T>* x = reinterpret_cast<cpx<T>*>(smem_raw);  // 2*Rs support values
    const int N = a.N, Rs = a.Rs, C = N / 2 + 1;
    const int col = blockIdx.x;
    for (int s = threadIdx.x; s < 2 * Rs; s += blockDim.x) x[s] = a.Tm[size_t(s) * a.ldT + col];
    __syncthreads();
    for (int k = threadIdx.x; k < N; k += blockDim.x) {
        T re = 0, im = 0;
        int e = 0;
        for (int s = 0; s < Rs; ++s) {
            const cpx<T> w = a.tw[e];
            re = ffma(x[s].re, w.re, ffma(-x[s].im, w.im, re));
            im = ffma(x[s].re, w.im, ffma(x[s].im, w.re, im));
            e += k; if (e >= N) e -= N;
        }
        e = int((long long)(N - Rs) * k % N);
        for (int s = Rs; s < 2 * Rs; ++s) {
            const cpx<T> w = a.tw[e];
            re = ffma(x[s].re, w.re, ffma(-x[s].im, w.im, re));
            im = ffma(x[s].re, w.im, ffma(x[s].im, w.re, im));
            e += k; if (e >= N) e -= N;
        }
        if constexpr (OUT == OUT_COLMAJOR_SHIFT) {
            int r = k + N / 2; if (r >= N) r -= N;
            a.S[size_t(col) * a.ldS + r] = cpx<T>{re, im};
        } else {
            a.S[size_t(k) * C + col] = cpx<T>{re, im};
        }
    }
}

// ---------------------------------------------------------------------------
// profile path with the image symmetry: a swept radial profile depends on
// x^2 and y^2 only, and the quadrant-shifted image z[k][n] is exactly even in
// both indices (z[N-k][n] = z[k][n] = z[k][N-n]; the box rows/columns that
// have no mirror inside the box are zero, since there r >= rmax*dxy puts the
// radial index at nr-1 or beyond).  Its DFT is therefore real and even in both
// frequencies: the row pass packs rows m_a, m_b as one complex FFT and reads
// the two real results off the real and imaginary parts; the column pass does
// the same for two columns and stores frequencies 0..N/2 only.
//   Ts : real, row transform of image row m = |y| pixel index (m = 0..Rs') at
//        u-frequency l (l < C), in 64-byte blocks of 2 rows x 4 frequencies
//        (ts_index): a row pass workgroup (two rows) writes whole lines, and a
//        column pair reads 16 bytes per row, two rows per line.
//   H  : real, S at u-column l and |v-frequency| m (S at shifted row r is
//        m = |r - N/2|), columns interleaved in pairs (h_index): column pair
//        {2p, 2p+1} is a run of ldH (m, 2p), (m, 2p+1) pairs, so the column pass
//        stores one 16-byte pair per row and a sample's four corners (columns
//        c, c+1, rows m0, m1) share one 32-byte run when c is even.
// ---------------------------------------------------------------------------
// Offset of H element (column l, row m); ldH (>= N/2 + 1) rows per column.
__device__ __forceinline__ size_t h_index(int l, int m, int ldH) {
    return (size_t(l >> 1) * size_t(ldH) + size_t(m)) * 2 + size_t(l & 1);
}

// Offset of Ts element (row m, frequency l); ldT (>= C, a multiple of 8) reals per row.
__device__ __forceinline__ size_t ts_index(int m, int l, int ldT) {
    return (size_t(m >> 1) * size_t(ldT) + size_t(l >> 2) * 4) * 2 + size_t(((m & 1) << 2) + (l & 3));
}

template <typename T>
struct SymRowArgs {
    SweepPrm<T> sw;
    int N, Rs;            // symmetric support half-width Rs' (columns [0,Rs') U [N-Rs',N))
    int nrows;            // Rs' + 1 rows m = 0..Rs'
    int ldT;              // reals per row of Ts (>= C, a multiple of 8; see ts_index)
    const cpx<T>* tw;
    T* Ts;
    double* zero;         // optional: workgroup 0 clears zero[0..nzero) and *zero1 (gradient accumulators)
    int nzero;
    double* zero1;
    int ncol;             // frequencies stored: 0..ncol-1 (<= C; those the column pass reads)
};

// SPLIT: the half-LDS exchange (more workgroups per CU: the batched form's many
// walkers); otherwise both parts per round trip (lower latency: one call's
// ~Rs'/2 workgroups).
template <typename T, int LOG2N, bool SPLIT = false>
__device__ __forceinline__ void rowpass_sym_body(const SymRowArgs<T>& a, int blk) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false, SPLIT>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    static_assert(F::LDS_REALS >= N + 2, "the transform's LDS holds N/2 + 1 swept pixels of both rows");
    __shared__ __align__(16) T lds[F::LDS_REALS];
    __shared__ T Ic[NT];
    const int tid = threadIdx.x;
    const int ma = 2 * blk, mb = ma + 1;
    const bool hb = mb < a.nrows;
    const bool cen = ma == 0;     // this workgroup's row ma = 0 holds the central pixel
    if (blk == 0) {
        if (a.zero)
            for (int k = tid; k < a.nzero; k += NT) a.zero[k] = 0.0;
        if (a.zero1 && tid == 0) *a.zero1 = 0.0;
    }
    // The central pixel is row 0's input n = 0: a constant that adds its value
    // to every output frequency.  The transform runs without it and the value
    // is added at the store, so its profile reads (issued here, beside the
    // sweep's) and its serial arithmetic stay off the transform's path.
    T ipre = T(0);
    if (cen && tid < a.sw.nr) ipre = a.sw.I[tid];
    cpx<T> v[E];
    // a pixel's value serves x and -x: swept once into LDS, read from there as positions n and N - n
    // (Rs' = 803 at nxy = 4096: 14.8 -> 13.8 us; Rs' = 202: the call 33.65 -> 33.35 us)
    cpx<T>* px = reinterpret_cast<cpx<T>*>(lds);
    for (int x = tid; x <= a.Rs; x += NT) {
        const T za = (ma == 0 && x == 0) ? T(0) : sweep_pixel(x, ma, a.sw);
        const T zb = hb ? sweep_pixel(x, mb, a.sw) : T(0);
        px[x] = cpx<T>{za, zb};
    }
    __syncthreads();
    F::template run<true>(v, lds, tid, a.Rs, a.tw, [&](int n) -> cpx<T> { return px[n < N / 2 ? n : N - n]; });
    T c = T(0);
    if (cen) {
        Ic[tid] = ipre;
        __syncthreads();
        c = central_value_of(a.sw, [&](int i) { return i < NT ? Ic[i] : a.sw.I[i]; });
    }
    // rows ma, mb of Ts (mb = nrows is a padding row): four consecutive lanes fill one line
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int k = tid + r * NT;
        if (r * NT <= N / 2 && k < a.ncol) {
            T* o = a.Ts + ts_index(ma, k, a.ldT);
            o[0] = cen ? v[r].re + c : v[r].re;
            o[4] = v[r].im;
        }
    }
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_rowpass_sym(SymRowArgs<T> a) {
    rowpass_sym_body<T, LOG2N>(a, blockIdx.x);
}

template <typename T>
struct SymColArgs {
    const T* Ts;
    int N, Rs, ldT;
    const cpx<T>* tw;
    T* H;
    int ldH;
    double rc2;                  // > 0: store only cells within sqrt(rc2) (cells) of the origin (stored_rows)
    const cpx<T>* tw512;         // W_512^e table (k_colpass_sub)
};

// Highest row of column l of a half spectrum that a sample within the store
// radius sqrt(rc2) can read (-1: none); N/2 when there is no radius (rc2 <= 0).
__device__ __forceinline__ int stored_rows(double rc2, int l, int N) {
    if (!(rc2 > 0.0)) return N / 2;
    const double r = rc2 - double(l) * double(l);
    if (r < 0.0) return -1;
    const int k = int(sqrt(r));
    return k < N / 2 ? k : N / 2;
}

// Column N/2 of H (the one column without a partner among the N/2 + 1):
// H[N/2][k] = sum over the loaded rows n of Ts[|n|][N/2] cos(2 pi n k / N), i.e.
// Ts[0] + 2 sum_{0<m<Rs} Ts[m] cos(2 pi m k/N) + Ts[Rs] cos(2 pi Rs k/N), as a
// direct sum (FP64 accumulation) by one wave per output k = blk + q N/4.
template <typename T, int LOG2N, int NW = (FftShape<LOG2N>::NT / 64 > 0 ? FftShape<LOG2N>::NT / 64 : 1)>
__device__ __forceinline__ void colpass_nyquist(const SymColArgs<T>& a, int blk) {
    constexpr int N = 1 << LOG2N;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int kmax = stored_rows(a.rc2, N / 2, N);
    for (int q = wv; q < 3; q += NW) {
        const int k = blk + q * (N / 4);
        if (k > kmax) break;
        double acc = 0.0;
        for (int m = lane; m <= a.Rs; m += 64) {
            const double wm = (m == 0 || m == a.Rs) ? 1.0 : 2.0;
            acc += wm * double(a.Ts[ts_index(m, N / 2, a.ldT)]) * double(a.tw[(m * k) & (N - 1)].re);
        }
        acc = wave_sum(acc);
        if (lane == 0) a.H[h_index(N / 2, k, a.ldH)] = T(acc);
    }
}

template <typename T, int LOG2N, bool SPLIT = true>
__device__ __forceinline__ void colpass_sym_body(const SymColArgs<T>& a, int blk, int nblk) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false, SPLIT>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    constexpr int NPAIR = N / 4;                  // pairs of columns 0..N/2-1; column N/2 separately
    __shared__ T lds[F::LDS_REALS];
    const int pair = xcd_column(blk, nblk);
    if (pair >= NPAIR) return;
    const int la = 2 * pair;
    const int tid = threadIdx.x;
    const int kc = stored_rows(a.rc2, la, N);   // rows a sample can read (column la + 1: no more)
    if (kc >= 0) {                              // (else no sample reaches these columns)
        // columns la, la + 1 of Ts: one aligned 16-byte pair per row m (la even)
        cpx<T> v[E];
        F::run(v, lds, tid, a.Rs, a.tw, [&](int n) -> cpx<T> {
            const int m = n < N / 2 ? n : N - n;
            return *reinterpret_cast<const cpx<T>*>(a.Ts + ts_index(m, la, a.ldT));
        });
        cpx<T>* hab = reinterpret_cast<cpx<T>*>(a.H + h_index(la, 0, a.ldH));   // columns la, la + 1
#pragma unroll
        for (int r = 0; r <= E / 2; ++r) {
            const int k = tid + r * NT;
            if (k <= kc) hab[k] = v[r];
        }
    }
    colpass_nyquist<T, LOG2N>(a, pair);
}

// Pruned column transforms.  Column pair (la, la + 1) of Ts is nonzero only
// for signed positions |n'| < Rs (row |n'| of Ts; rows rmax = Rs - 1 and Rs lie
// beyond the swept profile and hold zeros, unless Rs = N/2).  With Rs <= 256
// that support fits in the window n' in [-256, 256) of 512 positions, so
// output k = k0 + P K (P = N / 512) of the N-point transform is the 512-point
// transform, at K, of z[m] = x[m'] W_N^(m' k0), m' = m or m - 512 the signed
// position of window slot m.  The input is even, so X[N - k] = X[k]: residues
// k0 = 0..P/2 give every row 0..N/2 (residue P - k0 as the mirror of residue
// k0).  One wave per residue (NK = P/2 + 1 waves per workgroup, one workgroup
// per column pair): 40% fewer FP64 operations per column pair than the full
// transform and a shorter path per workgroup (no barrier inside the
// transform), for about the same LDS traffic (each residue wave reads the
// whole window, and the outputs, rows P apart per wave, are transposed
// through LDS into contiguous row stores).
template <int LOG2N>
struct ResidueShape {
    static constexpr int N = 1 << LOG2N, P = N / 512, NK = P / 2 + 1, NT = 64 * NK;
    static_assert(LOG2N >= 9 && LOG2N <= 13, "residue transforms for 512 <= N <= 8192");
};
constexpr int RESIDUE_MAX_RS = 256;

template <typename T, int LOG2N, bool SPLITROW = false>
__device__ __forceinline__ void colpass_sub_body(const SymColArgs<T>& a, int pair) {
    using CS = ResidueShape<LOG2N>;
    using F = ResidueFft<T, true>;
    constexpr int N = CS::N, P = CS::P;
    // LDS: the window (read once per workgroup) and the waves' exchange regions, then the output
    // rows 0..N/2 (row i at i + i/8: the residue waves write rows P apart, which the padding spreads
    // over the banks), read back in row order for contiguous stores.  SPLITROW (the batched form, bound
    // by throughput): the rows pass through LDS real parts first, then imaginary parts, in half the
    // space, so more workgroups fit on a CU
    constexpr size_t FFT_BYTES = 512 * sizeof(cpx<T>) + CS::NK * F::LDS_REALS * sizeof(T);
    constexpr size_t ROW_BYTES = (N / 2 + N / 16 + 1) * (SPLITROW ? sizeof(T) : sizeof(cpx<T>));
    __shared__ __align__(16) unsigned char smem[FFT_BYTES > ROW_BYTES ? FFT_BYTES : ROW_BYTES];
    cpx<T>* xin = reinterpret_cast<cpx<T>*>(smem);
    T* lds = reinterpret_cast<T*>(smem + 512 * sizeof(cpx<T>));
    cpx<T>* rows = reinterpret_cast<cpx<T>*>(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int k0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int la = 2 * pair;
    const int kc = stored_rows(a.rc2, la, N);   // rows a sample can read (column la + 1: no more)
    if (kc >= 0) {
        // window slot m holds signed position m' = m (m < 256) or m - 512; P = 1: the whole
        // column, position -256 = N/2 included
#pragma unroll
        for (int q = 0; q < (512 + CS::NT - 1) / CS::NT; ++q) {
            const int m = tid + q * CS::NT;
            if (m < 512) {
                const int mp = m < 256 ? m : m - 512;
                const bool in = mp >= 0 ? mp < a.Rs : (P == 1 ? -mp <= a.Rs : -mp < a.Rs);
                const T* src = a.Ts + ts_index(in ? (mp >= 0 ? mp : -mp) : 0, la, a.ldT);
                const T re = src[0], im = src[1];
                xin[m] = in ? cpx<T>{re, im} : cpx<T>{T(0), T(0)};
            }
        }
        __syncthreads();
        // y[m] = x[m'] W_N^(-512 k0 [m' < 0]) with pass 0's W_N^(64 k0 r): one factor per r
        cpx<T> v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            v[r] = xin[lane + 64 * r];
            if (r != 0 && k0 != 0) v[r] = cmul(v[r], a.tw[(64 * k0 * (r < 4 ? r : r - 8)) & (N - 1)]);
        }
        F::run(v, lds + k0 * F::LDS_REALS, lane, a.tw, a.tw512, P, k0);
        __syncthreads();                             // every wave is done with the window and its region
        const bool mirror = k0 != 0 && 2 * k0 != P;
        cpx<T>* hab = reinterpret_cast<cpx<T>*>(a.H + h_index(la, 0, a.ldH));   // columns la, la + 1
        if constexpr (SPLITROW) {
            constexpr int PER = (N / 2 + 1 + CS::NT - 1) / CS::NT;
            T* rr = reinterpret_cast<T*>(smem);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int k = k0 + P * (lane + 64 * r);
                const int row = k <= N / 2 ? k : (mirror ? N - k : -1);
                if (row >= 0 && row <= kc) rr[row + (row >> 3)] = v[r].re;
            }
            __syncthreads();
            T keep[PER];
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int row = tid + q * CS::NT;
                keep[q] = row <= kc ? rr[row + (row >> 3)] : T(0);
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int k = k0 + P * (lane + 64 * r);
                const int row = k <= N / 2 ? k : (mirror ? N - k : -1);
                if (row >= 0 && row <= kc) rr[row + (row >> 3)] = v[r].im;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int row = tid + q * CS::NT;
                if (row <= kc) hab[row] = cpx<T>{keep[q], rr[row + (row >> 3)]};
            }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int k = k0 + P * (lane + 64 * r);
                const int row = k <= N / 2 ? k : (mirror ? N - k : -1);
                if (row >= 0 && row <= kc) rows[row + (row >> 3)] = v[r];
            }
            __syncthreads();
            for (int row = tid; row <= kc; row += CS::NT) hab[row] = rows[row + (row >> 3)];
        }
    }
    colpass_nyquist<T, LOG2N, CS::NK>(a, pair);
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(ResidueShape<LOG2N>::NT) void k_colpass_sub(SymColArgs<T> a) {
    // rows of more than 64 KB (nxy = 8192 in double) pass through LDS in halves: 74 KB would leave two workgroups
    // per CU (67.0 -> 60.6 us per forward call, 1e6 points; at 4096 the halves cost 0.8 us)
    constexpr bool HALVES = size_t(ResidueShape<LOG2N>::N / 2) * sizeof(cpx<T>) >= 65536;
    colpass_sub_body<T, LOG2N, HALVES>(a, xcd_column(blockIdx.x, gridDim.x));
}

// At most 128 VGPRs (4 waves per SIMD): one call's N/4 workgroups then all fit
// on the chip at once (at 130 VGPRs a quarter of them waited for a second
// round); the cap costs a 20-byte spill at N=4096 FP64 and still saves ~6%.
// The batched kernel, whose many walkers fill the chip regardless, keeps the
// compiler's choice.
template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) __attribute__((amdgpu_waves_per_eu(4))) void k_colpass_sym(
    SymColArgs<T> a) {
    colpass_sym_body<T, LOG2N>(a, blockIdx.x, gridDim.x);
}

// Few workgroups: both parts per LDS round trip (half the barriers, twice the LDS), no register cap.
template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_colpass_sym_few(SymColArgs<T> a) {
    colpass_sym_body<T, LOG2N, false>(a, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// rotate -> interpolate -> phase -> (visibilities | chi2)
// interpolate_core galario.cpp:749-815, apply_phase_sampled_core 877-884,
// uv_rotate_core 955-960, diff_weighted_core 1453-1461.
// ---------------------------------------------------------------------------
template <typename T>
struct SampleArgs {
    const cpx<T>* S;             // complex spectrum (general path)
    long long rs, cs;            // element (row, col) at row*rs + col*cs
    const T* H;                  // real half spectrum (symmetric path), h_index layout
    int ldH;
    int nrow, ncol;
    T v_origin, duv;
    int rotate;  T cosPA, sinPA;
    int phase;   T dRA2, dDec2;  // 2*pi*dRArot, 2*pi*dDecrot
    T dRAt, dDect;               // dRArot, dDecrot: the phase in turns (double: sincos_turns)
    T inv_duv;                   // 1/duv (double: the grid position multiplies by it)
    int nd;
    const T* u; const T* v;
    cpx<T>* vis;                 // MODE_VIS
    const int* perm;             // MODE_VIS: point i is written to vis[perm[i]] (null: vis[i])
    const T* re; const T* im; const T* w;
    double* partials;            // MODE_CHI2: one per workgroup
    unsigned* flag;              // bit 0: a point fell outside the grid
    double ext2;                 // squared uv extent in uv units, points beyond it count as outside (infinite: none)
    double duv_d, inv_duv_d;     // duv and 1/duv in double (the FP32-bulk form's FP64 per-point arithmetic)
};

// Grid coordinates of a (rotated) point; oob when it is not inside the grid
// (or on its last row/column, where the weight beyond is zero).  The general
// complex path's form, in galario's order of operations.
template <typename T>
struct GridPos {
    int fl_u, fl_v, fu1, fv1;
    T q, t, sign_u, urot, vrot;
    bool oob;
};

template <typename T>
__device__ __forceinline__ GridPos<T> grid_pos(const SampleArgs<T>& a, T u0, T v0) {
    GridPos<T> g;
    g.urot = u0;
    g.vrot = v0;
    if (a.rotate) {
        g.urot = u0 * a.cosPA - v0 * a.sinPA;
        g.vrot = u0 * a.sinPA + v0 * a.cosPA;
    }
    g.sign_u = copysign(T(1), g.urot);
    const T indu = fabs(g.urot) / a.duv;
    const T indv = T(a.nrow / 2) + a.v_origin * g.sign_u * g.vrot / a.duv;
    g.oob = !(indu <= T(a.ncol - 1) && indv >= T(0) && indv <= T(a.nrow - 1));
    g.fl_u = g.oob ? 0 : int(floor(indu));
    g.fl_v = g.oob ? 0 : int(floor(indv));
    g.q = indu - T(g.fl_u);
    g.t = indv - T(g.fl_v);
    g.fu1 = g.fl_u + 1 < a.ncol ? g.fl_u + 1 : g.fl_u;   // weight q == 0 there
    g.fv1 = g.fl_v + 1 < a.nrow ? g.fl_v + 1 : g.fl_v;   // weight t == 0 there
    return g;
}

// a b + c d and a b - c d: in double one product is fused into the sum (an ulp of the grid position is
// 4e-13 cells at most); in float each operation rounds, as the reference's do.
template <typename P>
__device__ __forceinline__ P dot2(P a, P b, P c, P d) {
    if constexpr (std::is_same<P, double>::value) return ffma(a, b, c * d);
    else return a * b + c * d;
}
template <typename P>
__device__ __forceinline__ P det2(P a, P b, P c, P d) {
    if constexpr (std::is_same<P, double>::value) return ffma(a, b, -(c * d));
    else return a * b - c * d;
}

// a b + c with the constant c in scalar registers: a vector constant would be rebuilt by two register
// moves in front of every term of a polynomial.
__device__ __forceinline__ double fma_const(double a, double b, double c) {
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
}

// sin and cos of 2 pi x, x in turns.  f = x - (nearest integer) and then g = f - n / 4, |g| <= 1/8, n the
// integer nearest to 4 f (rounded by the addition of 1.5 2^52, whose low word then holds n); both
// differences are exact.  Minimax polynomials in z = g^2 (Remez; truncation error of the sine 3e-18
// relative, of the cosine 3e-20): sin(2 pi g) = 2 pi g + g z S(z), cos(2 pi g) = 1 + z C(z).  Each result is
// within 1.03 ulp over 2e7 arguments up to 1e3 turns, in 35 vector instructions and no branch; the
// library's sincospi takes 72.
__device__ __forceinline__ void sincos_turns(double x, double* s, double* c) {
    const double big = 6755399441055744.0;   // 1.5 * 2^52
    const double f = x - rint(x);
    const double sh = ffma(f, 4.0, big);
    const unsigned n = unsigned(__double2loint(sh));
    const double g = ffma(-0.25, sh - big, f);
    const double z = g * g;
    double ps = ffma(z, 0.0004615925796822367 * 8192.0, -0.00737003384915244 * 2048.0);
    ps = fma_const(ps, z, 0.08214587013039897 * 512.0);
    ps = fma_const(ps, z, -0.5992645289748814 * 128.0);
    ps = fma_const(ps, z, 2.5501640398740073 * 32.0);
    ps = fma_const(ps, z, -5.16771278004996 * 8.0);
    const double S = ffma(g, 6.28318530717958647692, (g * z) * ps);
    double pc = ffma(z, -0.00010357788609251752 * 16384.0, 0.0019294681734144596 * 4096.0);
    pc = fma_const(pc, z, -0.025806885879331866 * 1024.0);
    pc = fma_const(pc, z, 0.23533063020160833 * 256.0);
    pc = fma_const(pc, z, -1.3352627688521883 * 64.0);
    pc = fma_const(pc, z, 4.058712126416751 * 16.0);
    pc = fma_const(pc, z, -4.934802200544679 * 4.0);
    const double C = ffma(z, pc, 1.0);
    const bool odd = n & 1;
    const double s0 = odd ? C : S, c0 = odd ? S : C;
    const unsigned fs = (n << 30) & 0x80000000u, fc = ((n + 1) << 30) & 0x80000000u;
    *s = __hiloint2double(int(unsigned(__double2hiint(s0)) ^ fs), __double2loint(s0));
    *c = __hiloint2double(int(unsigned(__double2hiint(c0)) ^ fc), __double2loint(c0));
}

// e^{i theta}, theta = 2 pi (urot dRArot + vrot dDecrot).  In double from theta / 2 pi.
template <typename T>
__device__ __forceinline__ void phase_factor(const SampleArgs<T>& a, T urot, T vrot, T* s, T* c) {
    if constexpr (std::is_same<T, double>::value) {
        sincos_turns(dot2(urot, a.dRAt, vrot, a.dDect), s, c);
    } else {
        fsincos(urot * a.dRA2 + vrot * a.dDec2, s, c);
    }
}

template <typename T>
__device__ __forceinline__ cpx<T> apply_phase_pt(const SampleArgs<T>& a, const GridPos<T>& g, cpx<T> V) {
    if (a.phase) {
        T s, c;
        phase_factor(a, g.urot, g.vrot, &s, &c);
        V = cpx<T>{V.re * c - V.im * s, V.re * s + V.im * c};
    }
    return V;
}

template <typename T>
__device__ __forceinline__ cpx<T> sample_point(const SampleArgs<T>& a, T u0, T v0, bool& oob) {
    const GridPos<T> g = grid_pos(a, u0, v0);
    oob = g.oob;
    const T q = g.q, t = g.t;
    const cpx<T> y0 = a.S[g.fl_v * a.rs + g.fl_u * a.cs];
    const cpx<T> y1 = a.S[g.fv1 * a.rs + g.fl_u * a.cs];
    const cpx<T> y2 = a.S[g.fv1 * a.rs + g.fu1 * a.cs];
    const cpx<T> y3 = a.S[g.fl_v * a.rs + g.fu1 * a.cs];
    // Z = t*(q*((y0+y2)-(y1+y3))) + (t*(y1-y0) + q*(y3-y0)) + y0
    const T df_re = (y0.re + y2.re) - (y1.re + y3.re), df_im = (y0.im + y2.im) - (y1.im + y3.im);
    const T t1_re = t * (q * df_re), t1_im = t * (q * df_im);
    const T t2_re = t * (y1.re - y0.re), t2_im = t * (y1.im - y0.im);
    const T t3_re = q * (y3.re - y0.re), t3_im = q * (y3.im - y0.im);
    const T z_re = (t1_re + (t2_re + t3_re)) + y0.re;
    const T z_im = (t1_im + (t2_im + t3_im)) + y0.im;
    const T ph = atan2(z_im, z_re) * g.sign_u;
    const T a0 = hypot(y0.re, y0.im), a1 = hypot(y1.re, y1.im);
    const T a2 = hypot(y2.re, y2.im), a3 = hypot(y3.re, y3.im);
    T amp = a0;
    amp += (a3 - a0) * q;
    amp += (a1 - a0) * t;
    amp += (((a0 - a1) + a2) - a3) * t * q;
    T sp, cp;
    fsincos(ph, &sp, &cp);
    cpx<T> V = apply_phase_pt(a, g, cpx<T>{amp * cp, amp * sp});
    if (oob) V = cpx<T>{T(NAN), T(NAN)};
    return V;
}

// The same on the real, even spectrum H: the corners are real, Z is real, the
// phase of galario's amplitude/phase interpolation is 0 or pi, so
// V = (copysign(A, Z), 0) before the phase shift.
//
// Storage and arithmetic may differ: the spectrum H is read from `a` (type T)
// while the position, interpolation and phase use the scalars of `sc` and
// arithmetic in P.  P = T (sc = a) is that precision throughout (float: galario's order);
// T = float, P = double is the FP32-bulk form with FP64 per-point arithmetic.
//
// The batched sample kernels issue vector instructions at 60 to 85% of the rate the chip can (nxy = 4096 and
// 2048; 130 instructions per walker and 64 points became 106: 256 walkers x 3 datasets 2.58 to 2.11 ms), so the
// forms below are the ones with few instructions and no branches (a branch also keeps the loads of one point
// behind the arithmetic of another): without a rotation the scalars are cos = 1, sin = 0 (no selection per
// point), without offsets the phase factor of 0 is computed; the real path's v_origin is 1; the extent is checked on the unrotated radius, once per point for all
// walkers; the fraction of the position comes from one instruction; corners are 32-bit byte
// offsets from H (H holds less than 2^29 bytes); in double the bilinear forms are nested fused products.
// Every kernel samples through these functions, so one point gives the same bits in all of them.
template <typename P>
struct SymPoint {
    int iu, d;           // cell: column, signed row (the folded rows of its corners: |d| and |d + 1|)
    P q, t;              // position inside it
    P urot, vrot;
    bool in;             // inside the grid
};

// Point beyond the extent declared for the dataset (or not a number).
template <typename P>
__device__ __forceinline__ bool beyond_extent(double ext2, P u0, P v0) {
    const double u = double(u0), v = double(v0);
    return !(ffma(u, u, v * v) <= ext2);
}

// The integer part of x >= 0; 0 for x < 0 and NaN, the largest integer for x beyond it (the
// instruction's own limits, which a C++ conversion would leave undefined).
__device__ __forceinline__ unsigned to_u32(double x) {
    unsigned r;
    asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ unsigned to_u32(float x) {
    unsigned r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// A point outside the grid gets some cell inside it.
template <typename P>
__device__ __forceinline__ SymPoint<P> sym_position(const SampleArgs<P>& sc, P u0, P v0) {
    SymPoint<P> p;
    p.urot = det2(u0, sc.cosPA, v0, sc.sinPA);
    p.vrot = dot2(u0, sc.sinPA, v0, sc.cosPA);
    const int half = sc.nrow / 2;
    P indu, indv;
    if constexpr (std::is_same<P, double>::value) {
        const double vs = __hiloint2double(
            __double2hiint(p.vrot) ^ (__double2hiint(p.urot) & int(0x80000000u)), __double2loint(p.vrot));
        indu = fabs(p.urot) * sc.inv_duv;
        // (rounded twice: a fused one puts points on the first row a last bit outside the grid)
        indv = vs * sc.inv_duv + P(half);
        p.t = __builtin_amdgcn_fract(indv);
    } else {
        indu = fabs(p.urot) / sc.duv;
        indv = P(half) + (signbit(p.urot) ? -p.vrot : p.vrot) / sc.duv;
        p.t = __builtin_amdgcn_fractf(indv);
    }
    p.in = (indu <= P(sc.ncol - 1)) & (indv >= P(0)) & (indv <= P(sc.nrow - 1));
    // (inside, both are >= 0: truncation is the floor)
    p.iu = int(min(to_u32(indu), unsigned(half - 1)));   // (the last column: position 1 in the cell before it)
    p.q = indu - P(p.iu);
    p.d = int(min(to_u32(indv), unsigned(sc.nrow - 1))) - half;
    return p;
}

// The folded rows of a cell's corners.
__device__ __forceinline__ int row_lo(int d) { return max(d, -d); }        // |d|
__device__ __forceinline__ int row_hi(int d) { return max(d + 1, ~d); }    // |d + 1|

// H element at a byte offset (uniform base, 32-bit offset: one address register per corner)
template <typename T>
__device__ __forceinline__ T h_at(const T* H, unsigned bytes) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(H) + size_t(bytes));
}

// Corner values y0 = (iu, |d|), y1 = (iu, |d + 1|), y3 = (iu + 1, |d|), y2 = (iu + 1, |d + 1|) in P.
template <typename P>
struct SymValues {
    P y0, y1, y2, y3;
};
template <typename P, typename T>
__device__ __forceinline__ SymValues<P> sym_values(const T* H, int ldH, int iu, int d) {
    constexpr unsigned B = sizeof(T);
    const unsigned ld2 = 2u * B * unsigned(ldH);                  // bytes per column pair (< 2^24)
    const unsigned odd = unsigned(iu) & 1u;
    const unsigned b0 = __umul24(unsigned(iu) >> 1, ld2) + odd * B;
    const unsigned dc = odd ? ld2 - B : B;
    const unsigned o0 = b0 + 2u * B * unsigned(row_lo(d)), o1 = b0 + 2u * B * unsigned(row_hi(d));
    SymValues<P> y;
    y.y0 = P(h_at(H, o0));
    y.y1 = P(h_at(H, o1));
    y.y3 = P(h_at(H, o0 + dc));
    y.y2 = P(h_at(H, o1 + dc));
    return y;
}

// copysign(A, Z): the interpolated real visibility.
template <typename P>
__device__ __forceinline__ P sym_amplitude(const SymValues<P>& y, P q, P t) {
    const P a0 = fabs(y.y0), a1 = fabs(y.y1), a2 = fabs(y.y2), a3 = fabs(y.y3);
    if constexpr (std::is_same<P, double>::value) {
        const P z10 = y.y3 - y.y0, z01 = y.y1 - y.y0, z11 = (y.y2 - y.y3) - z01;
        const P z = ffma(q, ffma(t, z11, z10), ffma(t, z01, y.y0));
        const P e10 = a3 - a0, e01 = a1 - a0, e11 = (a2 - a3) - e01;
        return copysign(ffma(q, ffma(t, e11, e10), ffma(t, e01, a0)), z);
    } else {
        const P z = (t * (q * ((y.y0 + y.y2) - (y.y1 + y.y3))) + (t * (y.y1 - y.y0) + q * (y.y3 - y.y0))) + y.y0;
        P amp = a0;
        amp += (a3 - a0) * q;
        amp += (a1 - a0) * t;
        amp += (((a0 - a1) + a2) - a3) * t * q;
        return copysign(amp, z);
    }
}

// Visibility of a point (of some cell's values where p.in is false).
template <typename T, typename P>
__device__ __forceinline__ cpx<P> sample_point_sym2(const SampleArgs<T>& a, const SampleArgs<P>& sc,
                                                    const SymPoint<P>& p) {
    const SymValues<P> y = sym_values<P>(a.H, a.ldH, p.iu, p.d);
    P s = P(0), c = P(1);
    if (std::is_same<P, double>::value || sc.phase) phase_factor(sc, p.urot, p.vrot, &s, &c);
    const P V0 = sym_amplitude(y, p.q, p.t);
    // (plus zero: without an offset the imaginary part of a negative V0 is +0, its angle +pi)
    return cpx<P>{V0 * c, ffma(V0, s, P(0))};
}

// Visibility of a point on the real path; NaN and oob outside the grid or the extent.
template <typename T>
__device__ __forceinline__ cpx<T> sample_point_sym(const SampleArgs<T>& a, T u0, T v0, bool& oob) {
    const SymPoint<T> p = sym_position(a, u0, v0);
    oob = !p.in | beyond_extent(a.ext2, u0, v0);
    const cpx<T> V = sample_point_sym2<T, T>(a, a, p);
    return oob ? cpx<T>{T(NAN), T(NAN)} : V;
}

// chi2 term w |V - O|^2 of a point.  In double from w itself (galario multiplies the residual by sqrt(w),
// src/galario.cpp:1453-1461: NaN for a negative weight, which is kept), one factor of the residual at a time: no step
// leaves the range of a double where the term itself is within it.  In float in galario's order.
template <typename P>
__device__ __forceinline__ P weight_factor(P w) {
    if constexpr (std::is_same<P, double>::value) return w < P(0) ? P(NAN) : w;
    else return sqrt(w);
}
template <typename P>
__device__ __forceinline__ double chi2_term(P wf, P dre, P dim) {
    if constexpr (std::is_same<P, double>::value) {
        return ffma(wf * dre, dre, (wf * dim) * dim);
    } else {
        const P cr = dre * wf, ci = dim * wf;
        return double(cr) * cr + double(ci) * ci;
    }
}

// Deterministic sum over a workgroup of any size <= 1024 (red: 16 doubles);
// every thread gets the result.
__device__ __forceinline__ double block_sum_any(double acc, double* red16) {
    acc = wave_sum(acc);
    const int nw = int((blockDim.x + 63) >> 6);
    if ((threadIdx.x & 63) == 0) red16[threadIdx.x >> 6] = acc;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < nw; ++k) s += red16[k];
    return s;
}

// Read-rate reference: the workgroups read n2 16-byte elements in a
// grid-stride loop and write one sum each.  A plain stream of the same bytes
// as a kernel bounds the rate that kernel's own reads can reach.
__global__ __launch_bounds__(256) void k_read_probe(const cpx<double>* __restrict__ p, size_t n2, double* out);

// Deterministic block sum of `acc` (blockDim 256) into *out on thread 0.
__device__ __forceinline__ double block_sum256(double acc, double* red4) {
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = acc;
    __syncthreads();
    return (red4[0] + red4[1]) + (red4[2] + red4[3]);
}

// acc + p[i0] + p[i0 + 1024] + ... (terms below n), added in that order; the
// loads of eight terms are issued together, one memory round trip per eight.
__device__ __forceinline__ double sum_stride1024(const double* __restrict__ p, int i0, int n, double acc) {
    for (; i0 < n; i0 += 8 * 1024) {
        double x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = i0 + q * 1024 < n ? p[i0 + q * 1024] : 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (i0 + q * 1024 < n) acc += x[q];
    }
    return acc;
}

__global__ __launch_bounds__(256) void k_read_probe(const cpx<double>* __restrict__ p, size_t n2, double* out) {
    __shared__ double red[16];
    double s = 0.0;
    const size_t stride = size_t(gridDim.x) * 256;
    for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < n2; i += stride) {
        const cpx<double> x = p[i];
        s += x.re + x.im;
    }
    s = block_sum_any(s, red);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// Deterministic final sum of n per-workgroup partials (one workgroup of 1024
// threads, fixed order).  A separate launch: publishing partials across the
// 8 XCDs from inside one kernel would need a device-scope release per
// workgroup, which on gfx950 writes back the whole L2 each time.
template <typename T>
__global__ __launch_bounds__(1024) void k_sum_partials(const double* __restrict__ p, int n, double* out_d, T* out_t) {
    __shared__ double red[16];
    double acc = sum_stride1024(p, threadIdx.x, n, 0.0);
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int k = 0; k < 16; ++k) s += red[k];
        if (out_d) out_d[0] = s;
        if (out_t) out_t[0] = T(s);
    }
}

template <typename T, int MODE, bool SYM>
__device__ __forceinline__ void sample_body(const SampleArgs<T>& a, int blk) {
    __shared__ double red[4];
    const int i = blk * 256 + threadIdx.x;
    double acc = 0.0;
    bool oob = false;
    if (i < a.nd) {
        const cpx<T> V = SYM ? sample_point_sym(a, a.u[i], a.v[i], oob) : sample_point(a, a.u[i], a.v[i], oob);
        if constexpr (MODE == MODE_VIS) {
            a.vis[a.perm ? a.perm[i] : i] = V;
        } else {
            acc = chi2_term(weight_factor(a.w[i]), V.re - a.re[i], V.im - a.im[i]);
        }
    }
    if (oob && a.flag) raise_flag(a.flag);
    if constexpr (MODE == MODE_CHI2) {
        const double b = block_sum256(acc, red);
        if (threadIdx.x == 0) a.partials[blk] = b;
    }
}

template <typename T, int MODE, bool SYM>
__global__ __launch_bounds__(256) void k_sample(SampleArgs<T> a) {
    sample_body<T, MODE, SYM>(a, blockIdx.x);
}

// Several sources with the same profile, inclination and PA at different
// offsets (galario's multi-source recipe: the visibilities of each source,
// phase-shifted by its own offset, summed; docs/tech-specs.rst:45-57).  They
// share the spectrum and the interpolated value V0 at each point, so
// V = sum_k flux_k * apply_phase(V0, dRA_k, dDec_k), k in order.
// src: nsrc x 3 (flux, dRA, dDec) in the caller's (unrotated) frame.
template <typename T>
__device__ __forceinline__ cpx<T> multisrc_point(const SampleArgs<T>& a, int i, int nsrc, const T* __restrict__ src,
                                                 bool& oob) {
    SampleArgs<T> b = a;
    b.phase = 0;
    cpx<T> V0;
    if (a.H) {
        const SymPoint<T> p = sym_position(a, a.u[i], a.v[i]);
        oob = !p.in | beyond_extent(a.ext2, a.u[i], a.v[i]);
        V0 = cpx<T>{sym_amplitude(sym_values<T>(a.H, a.ldH, p.iu, p.d), p.q, p.t), T(0)};
    } else {
        V0 = sample_point(b, a.u[i], a.v[i], oob);
    }
    T ur = a.u[i], vr = a.v[i];
    if (a.H) {                     // the real path's rotation (sym_position)
        ur = det2(a.u[i], a.cosPA, a.v[i], a.sinPA);
        vr = dot2(a.u[i], a.sinPA, a.v[i], a.cosPA);
    } else if (a.rotate) {
        ur = a.u[i] * a.cosPA - a.v[i] * a.sinPA;
        vr = a.u[i] * a.sinPA + a.v[i] * a.cosPA;
    }
    cpx<T> V{T(0), T(0)};
    for (int k = 0; k < nsrc; ++k) {
        const T f = src[3 * k], dRA = src[3 * k + 1], dDec = src[3 * k + 2];
        T dRAr = dRA, dDecr = dDec;
        if (a.rotate) {
            dRAr = dRA * a.cosPA - dDec * a.sinPA;
            dDecr = dRA * a.sinPA + dDec * a.cosPA;
        }
        cpx<T> Vk = V0;
        if (!(dRAr == T(0) && dDecr == T(0))) {
            SampleArgs<T> ak;          // this source's phase scalars, as setup_sample forms them
            ak.dRA2 = T(double(dRAr) * (2. * double(T(M_PI))));
            ak.dDec2 = T(double(dDecr) * (2. * double(T(M_PI))));
            ak.dRAt = dRAr;
            ak.dDect = dDecr;
            T sn, cs;
            phase_factor(ak, ur, vr, &sn, &cs);
            if (a.H) Vk = cpx<T>{V0.re * cs, V0.re * sn};
            else Vk = cpx<T>{V0.re * cs - V0.im * sn, V0.re * sn + V0.im * cs};
        }
        V.re += f * Vk.re;
        V.im += f * Vk.im;
    }
    if (oob) V = cpx<T>{T(NAN), T(NAN)};
    return V;
}

// PPT blocks of 256 points per workgroup (more loads in flight per wave);
// block q's chi2 partial is the same fixed-order sum as in k_sample.
template <typename T, int MODE, int PPT>
__global__ __launch_bounds__(256) void k_sample_multisrc(SampleArgs<T> a, int nsrc, const T* __restrict__ src,
                                                         int nblocks) {
    __shared__ double red[PPT][4];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double acc[PPT];
    bool oob_any = false;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        acc[q] = 0.0;
        const int i = (blockIdx.x * PPT + q) * 256 + tid;
        if (i < a.nd) {
            bool oob = false;
            const cpx<T> V = multisrc_point(a, i, nsrc, src, oob);
            oob_any |= oob;
            if constexpr (MODE == MODE_VIS) {
                a.vis[a.perm ? a.perm[i] : i] = V;
            } else {
                acc[q] = chi2_term(weight_factor(a.w[i]), V.re - a.re[i], V.im - a.im[i]);
            }
        }
    }
    if (oob_any && a.flag) raise_flag(a.flag);
    if constexpr (MODE == MODE_CHI2) {
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
            const double x = wave_sum(acc[q]);
            if (lane == 0) red[q][wv] = x;
        }
        __syncthreads();
        if (tid < PPT) {
            const int b = blockIdx.x * PPT + tid;
            if (b < nblocks) a.partials[b] = (red[tid][0] + red[tid][1]) + (red[tid][2] + red[tid][3]);
        }
    }
}

// chi2 with PPT blocks of 256 points per workgroup (more loads in flight per
// wave); block q's partial is the same fixed-order sum as in k_sample.
// PPT = 2 from more than SAMPLE_ONE_ROUND blocks on (1e6 points at nxy = 4096: 11.0 us against 11.6 with 1 and 13 with 4),
// 1 up to there, where all workgroups of one block each are resident at once and half as many longer
// ones would leave CUs idle (3e5 points: 0.7 us less per call).
constexpr int SAMPLE_PPT = 2;
constexpr int SAMPLE_ONE_ROUND = 2048;   // 256 CUs x 8 workgroups of 4 waves

template <typename T, bool SYM, int PPT>
__global__ __launch_bounds__(256) void k_sample_chi2_n(SampleArgs<T> a, int nblocks) {
    __shared__ double red[PPT][4];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double acc[PPT];
    bool oob_any = false;
    // (lanes beyond the data take the last point and count nothing: no branch, so the loads of the PPT
    // points are all in flight together)
    const int base = blockIdx.x * (256 * PPT);
    T u0[PPT], v0[PPT], re[PPT], im[PPT], w[PPT];
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const unsigned i = unsigned(min(q * 256 + tid, a.nd - 1 - base)) * unsigned(sizeof(T));
        u0[q] = h_at(a.u + base, i);
        v0[q] = h_at(a.v + base, i);
        re[q] = h_at(a.re + base, i);
        im[q] = h_at(a.im + base, i);
        w[q] = h_at(a.w + base, i);
    }
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const bool valid = base + q * 256 + tid < a.nd;
        bool oob = false;
        const cpx<T> V = SYM ? sample_point_sym(a, u0[q], v0[q], oob) : sample_point(a, u0[q], v0[q], oob);
        oob_any |= oob & valid;
        const double x = chi2_term(weight_factor(w[q]), V.re - re[q], V.im - im[q]);
        acc[q] = valid ? x : 0.0;
    }
    if (oob_any && a.flag) raise_flag(a.flag);
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const double x = wave_sum(acc[q]);
        if (lane == 0) red[q][wv] = x;
    }
    __syncthreads();
    if (tid < PPT) {
        const int b = blockIdx.x * PPT + tid;
        if (b < nblocks) a.partials[b] = (red[tid][0] + red[tid][1]) + (red[tid][2] + red[tid][3]);
    }
}

// ---------------------------------------------------------------------------
// expert stages
// ---------------------------------------------------------------------------
// Full nxy x nxy image of a profile (create_image_h without the padding columns).
template <typename T>
__global__ __launch_bounds__(256) void k_sweep_image(SweepPrm<T> p, int N, int ld, T* img) {
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= size_t(N) * ld) return;
    const int i = int(idx / ld), j = int(idx % ld);
    T val = T(0);
    const int lo = N / 2 - p.rmax, hi = N / 2 + p.rmax;
    if (i == N / 2 && j == N / 2) {
        val = central_value(p);
    } else if (i >= lo && i < hi && j >= lo && j < hi) {
        val = sweep_pixel(N / 2 - j, N / 2 - i, p);
    }
    img[idx] = val;
}

// uv_rotate_core (galario.cpp:955-960) over arrays.
template <typename T>
__global__ __launch_bounds__(256) void k_rotate(int nd, T c, T s, const T* u, const T* v, T* ur, T* vr) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nd) return;
    const T u0 = u[i], v0 = v[i];
    ur[i] = u0 * c - v0 * s;
    vr[i] = u0 * s + v0 * c;
}

// apply_phase_sampled_core (galario.cpp:877-884), in place; dRA2/dDec2 include 2*pi.
template <typename T>
__global__ __launch_bounds__(256) void k_apply_phase(int nd, T dRA2, T dDec2, const T* u, const T* v, cpx<T>* vis) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nd) return;
    const T ang = u[i] * dRA2 + v[i] * dDec2;
    T s, c;
    fsincos(ang, &s, &c);
    const cpx<T> V = vis[i];
    vis[i] = cpx<T>{V.re * c - V.im * s, V.re * s + V.im * c};
}

// chi2 terms of given visibilities (reduce_chi2, galario.cpp:1506-1538);
// `a` carries only the reduction field (partials).
template <typename T>
__global__ __launch_bounds__(256) void k_chi2_terms(int nd, const T* re, const T* im, const cpx<T>* vis, const T* w,
                                                    SampleArgs<T> a) {
    __shared__ double red[4];
    const int i = blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    if (i < nd) {
        const cpx<T> V = vis[i];
        acc = chi2_term(weight_factor(w[i]), V.re - re[i], V.im - im[i]);
    }
    const double b = block_sum256(acc, red);
    if (threadIdx.x == 0) a.partials[blockIdx.x] = b;
}

// Clears n doubles (a kernel rather than a memset, so that it may sit in a captured graph).
__global__ __launch_bounds__(256) void k_fill_zero(double* p, size_t n) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Copies n2 16-byte words (the host-array calls' packed inputs, read over the bus from pinned memory).
__global__ __launch_bounds__(256) void k_copy16(const cpx<double>* __restrict__ in, cpx<double>* __restrict__ out,
                                                unsigned n2) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < n2) out[i] = in[i];
}

// Quadrant swap of the N x N real image held in rows of ld reals
// (shift_core, galario.cpp:565-589); the padding columns are copied through.
template <typename T>
__global__ __launch_bounds__(256) void k_fftshift_padded(int N, int ld, const T* in, T* out) {
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= size_t(N) * ld) return;
    const int i = int(idx / ld), j = int(idx % ld);
    out[idx] = j < N ? in[size_t((i + N / 2) % N) * ld + (j + N / 2) % N] : in[idx];
}

// Swap of the upper and lower row halves of an nrow x ncol complex matrix
// (shift_axis0_core, galario.cpp:657-668).
template <typename T>
__global__ __launch_bounds__(256) void k_fftshift_axis0(int nrow, int ncol, cpx<T>* m) {
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    const size_t half = size_t(nrow / 2) * ncol;
    if (idx >= half) return;
    const cpx<T> a = m[idx];
    m[idx] = m[idx + half];
    m[idx + half] = a;
}

}  // namespace gl
