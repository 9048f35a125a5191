// FFTs of the oversampled grid, pruned to the zero-padded image and fused
// with the deapodization.
//
// The forward transform of the table1 NUFFT is fftn(x * sn, Kd): only the
// first N_d entries of every axis are non-zero before the FFT.  The adjoint
// keeps only the first N_d entries of every axis after the inverse FFT.
// Transforming axis 0 first (forward) and last (adjoint), every pass works on
// the lines whose higher axes index the image (n_e < N_e) and whose lower
// axes are already (forward) or still (adjoint) full length:
//   forward axis d: lines (k_0..k_{d-1} < K, n_{d+1}.. < N), read t < N_d
//                   (the rest is zero), write t < K_d;
//   adjoint axis d: the same lines, read t < K_d, write t < N_d.
// Axis 0 reads the image (times sn) in the forward and writes the image
// (times scale * sn) in the adjoint, so deapod_pad and crop_deapod vanish
// into the FFT passes, and rows and planes outside the image are never
// read or written.
//
// A workgroup transforms lpw lines, TL threads per line, with a Stockham
// auto-sort FFT.  Thread t0 of a line holds the points t0 + e step (FftSpan)
// in registers: they are at once what it loads from memory, the inputs of its
// first butterflies and, after the last pass, what it stores.  The LDS only
// carries the exchanges between passes (one for two-pass lengths, two for
// three-pass ones).  With power-of-two lengths all radices and strides are
// compile-time constants (K > 0 below); other lengths whose prime factors
// are 2, 3, 5 and 7 run the same kernels with a radix list from the host
// (K = 0), one butterfly per thread and pass.
// Twiddles come from a table rounded once from double, one section per pass,
// ordered by butterfly (FftAxis), copied into LDS.
#pragma once

#include "device_common.hpp"
#include "kernels_grid.hpp"

namespace mi355 {

constexpr int kFftMinK = 16;
constexpr int kFftMaxK = 2048;
constexpr int kFftMaxPasses = 6;
constexpr int kFftMaxRadix = 10;  // of the mixed lengths

// Points per thread of a power-of-two line: 16 where that saves a pass.
__host__ __device__ constexpr int fft_points(int K) {
    return (K == 1024 || K == 2048) ? 16 : 8;
}
// Radix of the pass of sub-transform size ns of a power-of-two line:
// 16 = 8.2, 32 = 8.4, 64 = 8.8, 128 = 8.8.2, 256 = 8.8.4, 512 = 8.8.8,
// 1024 = 16.8.8, 2048 = 16.16.8.
__host__ __device__ constexpr int fft_radix(int K, int ns) {
    const int rest = K / ns;
    if (fft_points(K) == 16 && rest >= 16 && rest != 64) return 16;
    return rest >= 8 ? 8 : rest;
}
// Entries of the twiddle table before the pass of sub-transform size ns
// (the passes with ns > 1, in order): the pass stores w^(k r K / (ns R)),
// 1 <= r < R, k < ns, at offset + (r - 1) ns + k.
__host__ __device__ constexpr int fft_tw_offset(int K, int ns) {
    int off = 0;
    for (int s = fft_radix(K, 1); s < ns; s *= fft_radix(K, s)) off += (fft_radix(K, s) - 1) * s;
    return off;
}

// One axis of a fused FFT, made on the host (fft_axis_init).
struct FftAxis {
    int K;
    int TL;    // threads per line
    int ntw;   // entries of the twiddle table
    int np;    // passes
    int R[kFftMaxPasses];        // radix of each pass
    int off[kFftMaxPasses];      // its section of the twiddle table
    float inv_ns[kFftMaxPasses]; // 1 / sub-transform size
};

// LDS position of point t of a line: one unused slot per eight points
// spreads the strided writes of the passes over the banks.
__host__ __device__ constexpr int fft_pad(int t) { return t + (t >> 3); }

// Stride of lpw lines in LDS: 32 / lpw (16 / lpw for complex128) modulo 32 (16)
// slots, so that the lanes of lpw neighbouring lines and consecutive points
// fall on different banks.  Lines of the mixed lengths have no unused slots:
// their first radix is odd where one is, so their first writes have an odd
// stride.
__host__ __device__ constexpr int fft_line_stride(int K, int lpw, int cxs) {
    const int unit = 256 / cxs;
    const int want = lpw < unit ? unit / lpw : 1;
    const int base = (K & (K - 1)) ? K : fft_pad(K - 1) + 1;
    return base + ((want - base) % unit + unit) % unit;
}

// Small DFTs: X[k] = sum_n x[n] exp(SIGN * 2 pi i n k / R)
template <typename T, int SIGN>
__device__ __forceinline__ cx<T> mul_i(cx<T> a) {  // a * (SIGN i)
    return SIGN < 0 ? mkcx<T>(a.y, -a.x) : mkcx<T>(-a.y, a.x);
}

template <typename T>
__device__ __forceinline__ cx<T> cadd(cx<T> a, cx<T> b) { return mkcx<T>(a.x + b.x, a.y + b.y); }
template <typename T>
__device__ __forceinline__ cx<T> csub(cx<T> a, cx<T> b) { return mkcx<T>(a.x - b.x, a.y - b.y); }
template <typename T>
__device__ __forceinline__ cx<T> cmulc(cx<T> a, cx<T> w) {
#pragma clang fp contract(on)  // one rounding less per component
    return mkcx<T>(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
}

// cos(2 pi m / n) at compile time: folded to an angle of at most pi / 4,
// then the Taylor series of cos or sin
constexpr double fft_taylor(double x, bool sine) {
    double term = sine ? x : 1.0, sum = 0.0;
    for (int k = 0; k < 14; ++k) {
        sum += term;
        const int a = 2 * k + (sine ? 2 : 1);
        term *= -x * x / ((double)a * (a + 1));
    }
    return sum;
}
constexpr double fft_cos(int m, int n) {
    m = ((m % n) + n) % n;
    if (2 * m > n) m = n - m;
    double sign = 1.0;
    if (4 * m > n) {  // cos(pi - a) = -cos(a)
        m = n - 2 * m;
        n = 2 * n;
        sign = -1.0;
    }
    constexpr double tau = 6.283185307179586476925;
    if (8 * m > n) return sign * fft_taylor(tau * (double)(n - 4 * m) / (double)(4 * n), true);
    return sign * fft_taylor(tau * (double)m / (double)n, false);
}
constexpr double fft_sin(int m, int n) { return fft_cos(4 * m - n, 4 * n); }

// a * exp(SIGN 2 pi i M / N)
template <typename T, int SIGN, int M, int N>
__device__ __forceinline__ cx<T> mul_root(cx<T> a) {
    constexpr int m = ((SIGN * M) % N + N) % N;
    if constexpr (m == 0) return a;
    else if constexpr (4 * m == N) return mul_i<T, 1>(a);
    else if constexpr (2 * m == N) return mkcx<T>(-a.x, -a.y);
    else if constexpr (4 * m == 3 * N) return mul_i<T, -1>(a);
    else {
        constexpr double c = fft_cos(m, N), s = fft_sin(m, N);
        return cmulc<T>(a, mkcx<T>((T)c, (T)s));
    }
}

template <typename T, int SIGN>
__device__ __forceinline__ void dft2(cx<T>* v) {
    const cx<T> a = v[0], b = v[1];
    v[0] = cadd<T>(a, b);
    v[1] = csub<T>(a, b);
}

template <typename T, int SIGN>
__device__ __forceinline__ void dft4(cx<T>* v) {
    const cx<T> c0 = cadd<T>(v[0], v[2]), c1 = csub<T>(v[0], v[2]);
    const cx<T> d0 = cadd<T>(v[1], v[3]), d1 = mul_i<T, SIGN>(csub<T>(v[1], v[3]));
    v[0] = cadd<T>(c0, d0);
    v[1] = cadd<T>(c1, d1);
    v[2] = csub<T>(c0, d0);
    v[3] = csub<T>(c1, d1);
}

// radix 8 as two radix-4 DFTs of the even and odd halves after one radix-2
// step with the twiddles exp(SIGN 2 pi i n / 8), n = 0..3
template <typename T, int SIGN>
__device__ __forceinline__ void dft8(cx<T>* v) {
    const T h = (T)0.70710678118654752440;
    cx<T> a[4], b[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        a[n] = cadd<T>(v[n], v[n + 4]);
        b[n] = csub<T>(v[n], v[n + 4]);
    }
    // b1 *= (h, SIGN h); b2 *= SIGN i; b3 *= (-h, SIGN h)
    b[1] = mkcx<T>(h * (b[1].x - (T)SIGN * b[1].y), h * (b[1].y + (T)SIGN * b[1].x));
    b[2] = mul_i<T, SIGN>(b[2]);
    b[3] = mkcx<T>(-h * (b[3].x + (T)SIGN * b[3].y), h * ((T)SIGN * b[3].x - b[3].y));
    dft4<T, SIGN>(a);
    dft4<T, SIGN>(b);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[2 * k] = a[k];
        v[2 * k + 1] = b[k];
    }
}

// odd prime lengths through the even and odd parts of the conjugate pairs:
// X[k], X[R - k] = (x0 + sum_p cos(2 pi p k / R) (x_p + x_{R-p}))
//                  +- SIGN i sum_p sin(2 pi p k / R) (x_p - x_{R-p})
template <typename T, int R, int SIGN, int P, int KK>
__device__ __forceinline__ void dft_odd_term(const cx<T>* s, const cx<T>* d, cx<T>& re, cx<T>& im) {
#pragma clang fp contract(on)
    if constexpr (2 * P < R) {
        constexpr double c = fft_cos(P * KK, R), w = fft_sin(P * KK, R);
        re.x += (T)c * s[P].x;
        re.y += (T)c * s[P].y;
        im.x += (T)w * d[P].x;
        im.y += (T)w * d[P].y;
        dft_odd_term<T, R, SIGN, P + 1, KK>(s, d, re, im);
    }
}
template <typename T, int R, int SIGN, int KK>
__device__ __forceinline__ void dft_odd_out(cx<T> x0, const cx<T>* s, const cx<T>* d, cx<T>* v) {
    if constexpr (2 * KK < R) {
        cx<T> re = x0, im = mkcx<T>((T)0, (T)0);
        dft_odd_term<T, R, SIGN, 1, KK>(s, d, re, im);
        const cx<T> q = mul_i<T, SIGN>(im);
        v[KK] = cadd<T>(re, q);
        v[R - KK] = csub<T>(re, q);
        dft_odd_out<T, R, SIGN, KK + 1>(x0, s, d, v);
    }
}
template <typename T, int R, int SIGN>
__device__ __forceinline__ void dft_odd(cx<T>* v) {
    constexpr int H = (R + 1) / 2;
    cx<T> s[H], d[H];
    const cx<T> x0 = v[0];
    cx<T> t = x0;
#pragma unroll
    for (int p = 1; p < H; ++p) {
        s[p] = cadd<T>(v[p], v[R - p]);
        d[p] = csub<T>(v[p], v[R - p]);
        t = cadd<T>(t, s[p]);
    }
    dft_odd_out<T, R, SIGN, 1>(x0, s, d, v);
    v[0] = t;
}

template <typename T, int R, int SIGN>
__device__ __forceinline__ void dft_r(cx<T>* v);

// A * B points: DFTs of length A over n1 (n = B n1 + n2), twiddles
// exp(SIGN 2 pi i n2 k1 / (A B)), DFTs of length B over n2 (k = k1 + A k2)
template <typename T, int A, int B, int SIGN, int N2, int K1>
__device__ __forceinline__ void dft_ab_twiddle(cx<T>* y) {
    if constexpr (N2 < B) {
        y[N2 * A + K1] = mul_root<T, SIGN, N2 * K1, A * B>(y[N2 * A + K1]);
        if constexpr (K1 + 1 < A) dft_ab_twiddle<T, A, B, SIGN, N2, K1 + 1>(y);
        else dft_ab_twiddle<T, A, B, SIGN, N2 + 1, 1>(y);
    }
}
template <typename T, int A, int B, int SIGN>
__device__ __forceinline__ void dft_ab(cx<T>* v) {
    cx<T> y[A * B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n2 * A + n1] = v[B * n1 + n2];
        dft_r<T, A, SIGN>(y + n2 * A);
    }
    dft_ab_twiddle<T, A, B, SIGN, 1, 1>(y);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        cx<T> z[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) z[n2] = y[n2 * A + k1];
        dft_r<T, B, SIGN>(z);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = z[k2];
    }
}

template <typename T, int R, int SIGN>
__device__ __forceinline__ void dft_r(cx<T>* v) {
    if constexpr (R == 2) dft2<T, SIGN>(v);
    else if constexpr (R == 4) dft4<T, SIGN>(v);
    else if constexpr (R == 8) dft8<T, SIGN>(v);
    else if constexpr (R == 16) dft_ab<T, 4, 4, SIGN>(v);
    else if constexpr (R == 6) dft_ab<T, 3, 2, SIGN>(v);
    else if constexpr (R == 9) dft_ab<T, 3, 3, SIGN>(v);
    else if constexpr (R == 10) dft_ab<T, 5, 2, SIGN>(v);
    else dft_odd<T, R, SIGN>(v);
}

// Orders the LDS accesses of one wave (its LDS operations execute in order;
// this keeps the compiler from moving one lane's reads above its writes).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Butterflies of one pass on the registers of thread t0: butterfly j = t0 +
// q TL takes the points j + r K / R, which are v[q + r NB], times
// w^(k r K / (NS R)), k = j mod NS.
template <typename T, int K, int R, int NS, int SIGN>
__device__ __forceinline__ void fft_butterflies(cx<T> (&v)[fft_points(K)], int t0, const cx<T>* tw) {
    constexpr int E = fft_points(K), TL = K / E, NB = E / R;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        cx<T> w[R];
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = v[q + r * NB];
        if constexpr (NS > 1) {
            const cx<T>* t = tw + fft_tw_offset(K, NS) + (t0 + q * TL) % NS;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                cx<T> f = t[(r - 1) * NS];
                if (SIGN > 0) f.y = -f.y;
                w[r] = cmulc<T>(w[r], f);
            }
        }
        dft_r<T, R, SIGN>(w);
#pragma unroll
        for (int r = 0; r < R; ++r) v[q + r * NB] = w[r];
    }
}

// Their outputs in auto-sort order: (j / NS) NS R + k + r NS.  NS (or R for
// the first pass) is a multiple of 8, so the padded offset of r is a constant.
template <typename T, int K, int R, int NS>
__device__ __forceinline__ void fft_put(const cx<T> (&v)[fft_points(K)], int t0, cx<T>* line) {
    constexpr int E = fft_points(K), TL = K / E, NB = E / R;
    static_assert(NS == 1 ? R % 8 == 0 : NS % 8 == 0, "padding of a pass's outputs");
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int j = t0 + q * TL;
        cx<T>* o = line + fft_pad((j / NS) * NS * R + j % NS);
#pragma unroll
        for (int r = 0; r < R; ++r) o[fft_pad(r * NS)] = v[q + r * NB];
    }
}

template <typename T, int K>
__device__ __forceinline__ void fft_get(cx<T> (&v)[fft_points(K)], int t0, const cx<T>* line) {
    constexpr int E = fft_points(K), TL = K / E;
    if constexpr (TL % 8 == 0) {
        const cx<T>* o = line + fft_pad(t0);
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = o[fft_pad(e * TL)];
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = line[fft_pad(t0 + e * TL)];
    }
}

// One pass of run-time size (mixed radices): thread j of a line takes the
// points j + r K / R, from registers in the first pass and from LDS after
// it, and leaves its outputs in LDS, or in registers after the last pass.
// Every thread of the workgroup calls it (it holds the barriers).
template <typename T, int R, int SIGN>
__device__ __forceinline__ void fft_mixed_pass(cx<T> (&v)[kFftMaxRadix], cx<T>* line, int j, bool act, int K, int ns,
                                               float inv_ns, const cx<T>* tw, bool first, bool last) {
    const int nbf = K / R;  // uniform
    const bool on = act && j < nbf;
    const int b = (int)(((float)j + 0.5f) * inv_ns);  // j / ns, exact below 2^22
    const int k = j - b * ns;
    if (on) {
        if (!first) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = line[j + r * nbf];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                cx<T> f = tw[(r - 1) * ns + k];
                if (SIGN > 0) f.y = -f.y;
                v[r] = cmulc<T>(v[r], f);
            }
        }
        dft_r<T, R, SIGN>(v);
    }
    if (last) return;  // uniform
    if (!first) __syncthreads();
    if (on) {
        cx<T>* o = line + b * ns * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) o[r * ns] = v[r];
    }
    __syncthreads();
}

// points per thread of the kernels' registers (K = 0: mixed, at most the
// largest radix)
template <int K>
constexpr int kFftE = K > 0 ? fft_points(K > 0 ? K : 16) : kFftMaxRadix;

// Where thread t0 of a line finds its registers' points: point e is
// t0 + e step, for t0 < step and e < n (step = K / n).  The mixed lengths
// load by their first radix and store by their last one.
struct FftSpan {
    int step, n;
};
template <int K>
__device__ __forceinline__ FftSpan fft_span(const FftAxis& ax, bool store) {
    FftSpan s;
    s.n = K > 0 ? kFftE<K> : ax.R[store ? ax.np - 1 : 0];
    s.step = K > 0 ? K / kFftE<K> : ax.K / s.n;
    return s;
}

// whether thread t0 holds a point e
template <int K>
__device__ __forceinline__ bool fft_has(const FftSpan& s, int t0, int e) {
    return K > 0 || (e < s.n && t0 < s.step);
}

// FFT of the workgroup's lines.  On entry v holds the points of thread ta of
// line la, on return those of thread ts of line ls (FftSpan); the passes
// between run on line lm with thread index tm.  PRIV: in the (lm, tm) mapping
// a line's threads belong to one wave, so its exchanges need no workgroup
// barrier (cross: the (ls, ts) mapping differs, the last exchange needs one).
// The first barrier also publishes the twiddles.
template <typename T, int K, int SIGN, bool PRIV>
__device__ __forceinline__ void fft_lines(cx<T> (&v)[kFftE<K>], cx<T>* lds, int stride, int la, int ta, int lm,
                                          int tm, int ls, int ts, bool act, bool cross, const FftAxis& ax,
                                          const cx<T>* tw) {
    if constexpr (K > 0) {
        constexpr int R0 = fft_radix(K, 1), R1 = fft_radix(K, R0);
        static_assert(K <= R0 * R1 * 16, "two or three passes");
        fft_butterflies<T, K, R0, 1, SIGN>(v, ta, tw);
        fft_put<T, K, R0, 1>(v, ta, lds + la * stride);
        __syncthreads();
        if constexpr (R0 * R1 == K) {
            fft_get<T, K>(v, ts, lds + ls * stride);
            fft_butterflies<T, K, R1, R0, SIGN>(v, ts, tw);
        } else {
            fft_get<T, K>(v, tm, lds + lm * stride);
            fft_butterflies<T, K, R1, R0, SIGN>(v, tm, tw);
            if (PRIV) wave_fence();
            else __syncthreads();
            fft_put<T, K, R1, R0>(v, tm, lds + lm * stride);
            if (PRIV && !cross) wave_fence();
            else __syncthreads();
            fft_get<T, K>(v, ts, lds + ls * stride);
            fft_butterflies<T, K, K / (R0 * R1), R0 * R1, SIGN>(v, ts, tw);
        }
    } else {
        int ns = 1;
        for (int p = 0; p < ax.np; ++p) {
            const int R = ax.R[p];
            const bool first = p == 0, last = p == ax.np - 1;
            int l = first ? la : last ? ls : lm;
            int j = first ? ta : last ? ts : tm;
            // keeps the addresses of every radix from being formed before
            // the loop (column pass 108 -> 66 VGPRs)
            asm volatile("" : "+v"(l), "+v"(j));
            switch (R) {
#define MI355_MIXED(RR)                                                                                      \
    case RR:                                                                                                  \
        fft_mixed_pass<T, RR, SIGN>(v, lds + l * stride, j, act, ax.K, ns, ax.inv_ns[p], tw + ax.off[p], first, last); \
        break;
                MI355_MIXED(2) MI355_MIXED(3) MI355_MIXED(4) MI355_MIXED(5) MI355_MIXED(6) MI355_MIXED(7)
                MI355_MIXED(8) MI355_MIXED(9) MI355_MIXED(10)
#undef MI355_MIXED
            }
            ns *= R;
        }
    }
}

// the twiddle table, copied to LDS behind the lines
template <typename T>
__device__ __forceinline__ cx<T>* stage_twiddles(cx<T>* lds, int lpw, int stride, int ntw,
                                                 const cx<T>* __restrict__ tw) {
    cx<T>* tws = lds + lpw * stride;
    for (int i = threadIdx.x; i < ntw; i += blockDim.x) tws[i] = tw[i];
    return tws;
}

struct FftRowGeom {
    int N[3];          // image size
    int K[3];          // grid size
    int64_t nk;        // prod K
    int64_t xs[4];     // image strides: axes 0..2, repetition
    int64_t nlines;    // N1 * N2 * nimg
    int lpw;           // lines per workgroup
    int stride;        // LDS line stride
    const void* mult;  // adjoint: complex T grid (one image) multiplying the loaded rows, or null
    int across;        // image side read / written with lanes across neighbouring lines (image axis 1
                       // or 2 is the contiguous one, as for C-ordered images), else along each line
    int swap;          // neighbouring lines step along image axis 2 instead of axis 1
    FftAxis ax;
};

// image indices (m2, m3, repetition) of a line
__device__ __forceinline__ void row_of_line(int64_t line, const FftRowGeom& g, int& m2, int& m3, int64_t& r) {
    const unsigned na = g.swap ? g.N[2] : g.N[1], nb = g.swap ? g.N[1] : g.N[2];
    int a, b;
    if (g.nlines <= 0xffffffffll) {  // uniform: 32-bit divisions
        const unsigned u = (unsigned)line, q = u / na, rr = q / nb;
        a = (int)(u - q * na);
        b = (int)(q - rr * nb);
        r = rr;
    } else {
        const int64_t q = line / na;
        a = (int)(line - q * na);
        r = q / nb;
        b = (int)(q - r * nb);
    }
    m2 = g.swap ? b : a;
    m3 = g.swap ? a : b;
}

// A thread's place among the lines of a row pass: line and first point with
// the lanes along the lines (li, tl), and on the image side (la, ta).
struct RowLanes {
    int li, tl, la, ta;
    bool act;
};
template <int K>
__device__ __forceinline__ RowLanes row_lanes(const FftRowGeom& g) {
    RowLanes p;
    const unsigned tid = threadIdx.x;
    const unsigned TL = K > 0 ? (unsigned)(K / kFftE<K>) : (unsigned)g.ax.TL;
    p.li = (int)(tid / TL);
    p.tl = (int)(tid - p.li * TL);
    p.act = K > 0 || p.li < g.lpw;
    p.la = p.li;
    p.ta = p.tl;
    if (g.across) {  // lpw is a power of two
        p.la = (int)(tid & (unsigned)(g.lpw - 1));
        p.ta = (int)(tid / (unsigned)g.lpw);
    }
    return p;
}

template <int K>
constexpr bool kRowPriv = K > 0 && (K / kFftE<K>) <= 64;
template <typename T, int K>
constexpr int kFftThreads = K == 0 ? (sizeof(T) == 8 ? 768 : 1024) : (fft_points(K > 0 ? K : 16) == 16 ? 512 : 1024);

// sn of one image point, as the reference forms it (deapod_factor)
template <typename T>
__device__ __forceinline__ T row_deapod(const double* sn0, int ndim, int t, double s1, double s2) {
    double s = 1.0 * sn0[t];
    if (ndim > 1) s = s * s1;
    if (ndim > 2) s = s * s2;
    return (T)s;
}

// Axis 0, forward: grid[r, n2, n3, :] = FFT_K0(pad(x[:, n2, n3, r] * sn)) for
// n2 < N1, n3 < N2 (sn as deapod_factor).
template <typename T, int K, int SIGN>
__global__ __launch_bounds__((kFftThreads<T, K>)) void fft_rows_pad_kernel(const cx<T>* __restrict__ x,
                                                                           cx<T>* __restrict__ grid, FftRowGeom g,
                                                                           const double* sn0, const double* sn1,
                                                                           const double* sn2, int ndim,
                                                                           const cx<T>* __restrict__ tw) {
    constexpr int E = kFftE<K>;
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem);
    const int KR = K > 0 ? K : g.ax.K;
    const FftSpan in_span = fft_span<K>(g.ax, false), out_span = fft_span<K>(g.ax, true);
    const RowLanes p = row_lanes<K>(g);
    const int64_t line0 = (int64_t)blockIdx.x * g.lpw;
    // image loads: along the line, or across neighbouring lines (consecutive
    // threads on consecutive lines, adjacent in memory)
    cx<T> v[E];
    {
        const int64_t line = line0 + p.la;
        const bool live = p.act && line < g.nlines;
        int m2 = 0, m3 = 0;
        int64_t r = 0;
        if (live) row_of_line(line, g, m2, m3, r);
        const cx<T>* xl = x + (int64_t)m2 * g.xs[1] + (int64_t)m3 * g.xs[2] + r * g.xs[3];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = p.ta + e * in_span.step;
            v[e] = (live && fft_has<K>(in_span, p.ta, e) && t < g.N[0]) ? xl[(int64_t)t * g.xs[0]] : mkcx<T>((T)0, (T)0);
        }
        if (sn0) {
            const double s1 = ndim > 1 ? sn1[m2] : 1.0, s2 = ndim > 2 ? sn2[m3] : 1.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int t = p.ta + e * in_span.step;
                if (fft_has<K>(in_span, p.ta, e) && t < g.N[0]) {
                    const T s = row_deapod<T>(sn0, ndim, t, s1, s2);
                    v[e].x = v[e].x * s;
                    v[e].y = v[e].y * s;
                }
            }
        }
    }
    cx<T>* tws = stage_twiddles<T>(lds, g.lpw, g.stride, g.ax.ntw, tw);  // after the data loads are in flight
    fft_lines<T, K, SIGN, kRowPriv<K>>(v, lds, g.stride, p.la, p.ta, p.li, p.tl, p.li, p.tl, p.act, false, g.ax, tws);
    const int64_t line = line0 + p.li;
    if (p.act && line < g.nlines) {
        int m2, m3;
        int64_t r;
        row_of_line(line, g, m2, m3, r);
        cx<T>* out = grid + r * g.nk + ((int64_t)m3 * g.K[1] + m2) * KR;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = p.tl + e * out_span.step;
            if (fft_has<K>(out_span, p.tl, e)) out[t] = v[e];
        }
    }
}

// Axis 0, adjoint: x[:N0, n2, n3, r] = IFFT_K0(grid[r, n2, n3, :])[:N0] *
// scale * sn for n2 < N1, n3 < N2 (the arithmetic of crop_deapod_kernel).
//   rezero: write zeros over the rows it read, so that a grid passed through
//   the adjoint with zero_tail set on every other pass ends all zero.
template <typename T, int K, int SIGN>
__global__ __launch_bounds__((kFftThreads<T, K>)) void fft_rows_crop_kernel(cx<T>* __restrict__ grid,
                                                                            cx<T>* __restrict__ x, FftRowGeom g,
                                                                            const double* sn0, const double* sn1,
                                                                            const double* sn2, int ndim, T scale,
                                                                            const cx<T>* __restrict__ tw,
                                                                            int rezero) {
    constexpr int E = kFftE<K>;
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem);
    const int KR = K > 0 ? K : g.ax.K;
    const FftSpan in_span = fft_span<K>(g.ax, false), out_span = fft_span<K>(g.ax, true);
    const RowLanes p = row_lanes<K>(g);
    const int64_t line0 = (int64_t)blockIdx.x * g.lpw;
    cx<T> v[E];
    {
        const int64_t line = line0 + p.li;
        const bool live = p.act && line < g.nlines;
        int m2 = 0, m3 = 0;
        int64_t r = 0;
        if (live) row_of_line(line, g, m2, m3, r);
        const int64_t row = ((int64_t)m3 * g.K[1] + m2) * KR;
        cx<T>* in = grid + r * g.nk + row;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = p.tl + e * in_span.step;
            v[e] = (live && fft_has<K>(in_span, p.tl, e)) ? in[t] : mkcx<T>((T)0, (T)0);
        }
        if (g.mult) {
            const cx<T>* mul = (const cx<T>*)g.mult + row;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int t = p.tl + e * in_span.step;
                if (live && fft_has<K>(in_span, p.tl, e)) v[e] = cmulc<T>(v[e], mul[t]);
            }
        }
        if (rezero && live) {  // each thread clears the points it loaded
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int t = p.tl + e * in_span.step;
                if (fft_has<K>(in_span, p.tl, e)) in[t] = mkcx<T>((T)0, (T)0);
            }
        }
    }
    cx<T>* tws = stage_twiddles<T>(lds, g.lpw, g.stride, g.ax.ntw, tw);
    // image stores: along the line, or across neighbouring lines
    fft_lines<T, K, SIGN, kRowPriv<K>>(v, lds, g.stride, p.li, p.tl, p.li, p.tl, p.la, p.ta, p.act, g.across != 0, g.ax,
                                       tws);
    const int64_t line = line0 + p.la;
    if (p.act && line < g.nlines) {
        int m2, m3;
        int64_t r;
        row_of_line(line, g, m2, m3, r);
        cx<T>* xl = x + (int64_t)m2 * g.xs[1] + (int64_t)m3 * g.xs[2] + r * g.xs[3];
        const double s1 = sn0 && ndim > 1 ? sn1[m2] : 1.0, s2 = sn0 && ndim > 2 ? sn2[m3] : 1.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = p.ta + e * out_span.step;
            if (fft_has<K>(out_span, p.ta, e) && t < g.N[0]) {
                const T s = sn0 ? row_deapod<T>(sn0, ndim, t, s1, s2) : (T)1;
                cx<T> o;
                o.x = (v[e].x * scale) * s;
                o.y = (v[e].y * scale) * s;
                xl[(int64_t)t * g.xs[0]] = o;
            }
        }
    }
}

struct FftColGeom {
    int64_t S;        // stride of the axis = number of lines side by side (prod of lower K)
    int n_in;         // points read per line (the rest is zero)
    int n_out;        // points written per line
    int A;            // active indices of the next higher axis (1 if none)
    int64_t st_a;     // grid stride of that axis
    int64_t nk;       // prod K (stride of an image)
    int64_t nouter;   // A * nimg
    int lpw;          // neighbouring lines per workgroup, a power of two
    int nchunk;       // ceil(S / lpw)
    int stride;       // LDS line stride
    int zero_tail;    // also write zeros at n_out <= t < K
    const void* mult; // complex T grid (one image) multiplying the loaded lines, or null
    // Last forward pass / first adjoint pass of an ndim >= 2 grid: pb = 1
    // multiplies what the pass writes by phase_before (then divides by
    // scale_ortho if ortho), pb = 2 multiplies what it loads by
    // conj(phase_before); the element's axis-0 (and axis-1) index comes from
    // the inner line index i0 = k0 + K0 * k1.
    int pb;
    int ortho;
    int pb_ndim;
    int K0;
    double pbc[3];      // phase_before coefficients, rounded to T in the kernel
    double scale_ortho;
    FftAxis ax;
};

// phase_before_arg of a line's lower axes; the pass's own axis adds c t
template <typename T>
__device__ __forceinline__ T fft_pb_base(const FftColGeom& g, unsigned i0) {
    if (g.pb_ndim == 2) return (T)g.pbc[0] * (T)(int)i0;
    const unsigned k1 = i0 / (unsigned)g.K0, k0 = i0 - k1 * (unsigned)g.K0;
    return (T)g.pbc[0] * (T)(int)k0 + (T)g.pbc[1] * (T)(int)k1;
}

// grid value times phase_before (then / scale_ortho): the arithmetic of the
// tiled gather's tile staging, so the staged values are unchanged
template <typename T>
__device__ __forceinline__ cx<T> fft_pb_apply(cx<T> w, const FftColGeom& g, T base, int t, bool conj) {
    cx<T> p = cis_tile(base + (T)g.pbc[g.pb_ndim - 1] * (T)t);
    if (conj) p.y = -p.y;
    cx<T> o;
    o.x = w.x * p.x - w.y * p.y;
    o.y = w.x * p.y + w.y * p.x;
    if (!conj && g.ortho) {
        o.x = o.x / (T)g.scale_ortho;
        o.y = o.y / (T)g.scale_ortho;
    }
    return o;
}

// Axis d >= 1 in place: lpw neighbouring lines (inner index i0..i0+lpw-1) of
// one outer index per workgroup; each row of the block is one contiguous
// lpw-element segment.
template <typename T, int K, int SIGN>
__global__ __launch_bounds__((kFftThreads<T, K>)) void fft_cols_kernel(cx<T>* __restrict__ grid, FftColGeom g,
                                                                       const cx<T>* __restrict__ tw) {
    constexpr int E = kFftE<K>;
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem);
    const FftSpan in_span = fft_span<K>(g.ax, false), out_span = fft_span<K>(g.ax, true);
    const unsigned bid = xcd_remap(blockIdx.x, gridDim.x);  // neighbouring chunks share 128-byte lines
    const unsigned o = bid / (unsigned)g.nchunk, chunk = bid - o * (unsigned)g.nchunk;
    const unsigned img = o / (unsigned)g.A, a = o - img * (unsigned)g.A;
    const int li = (int)(threadIdx.x & (unsigned)(g.lpw - 1)), t0 = (int)(threadIdx.x / (unsigned)g.lpw);
    const unsigned i0 = chunk * (unsigned)g.lpw + li;  // inner index of this thread's line
    const bool act = K > 0 || t0 < g.ax.TL;
    const bool live = act && i0 < g.S;
    const int64_t ibase = (int64_t)a * g.st_a + i0;  // within one image
    cx<T>* gp = grid + (int64_t)img * g.nk + ibase;
    const T pbase = g.pb ? fft_pb_base<T>(g, i0) : (T)0;
    cx<T> v[E];
    {
        const int64_t step = (int64_t)in_span.step * g.S;  // uniform
        const cx<T>* q = gp + (int64_t)t0 * g.S;
#pragma unroll
        for (int e = 0; e < E; ++e, q += step) {
            const int t = t0 + e * in_span.step;
            v[e] = (live && fft_has<K>(in_span, t0, e) && t < g.n_in) ? *q : mkcx<T>((T)0, (T)0);
        }
    }
    if (g.mult) {
        const cx<T>* mul = (const cx<T>*)g.mult + ibase;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = t0 + e * in_span.step;
            if (live && fft_has<K>(in_span, t0, e) && t < g.n_in) v[e] = cmulc<T>(v[e], mul[(int64_t)t * g.S]);
        }
    }
    if (g.pb == 2) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = t0 + e * in_span.step;
            if (fft_has<K>(in_span, t0, e) && t < g.n_in) v[e] = fft_pb_apply<T>(v[e], g, pbase, t, true);
        }
    }
    cx<T>* tws = stage_twiddles<T>(lds, g.lpw, g.stride, g.ax.ntw, tw);
    fft_lines<T, K, SIGN, false>(v, lds, g.stride, li, t0, li, t0, li, t0, act, false, g.ax, tws);
    if (!live) return;
    const int64_t step = (int64_t)out_span.step * g.S;
    cx<T>* q = gp + (int64_t)t0 * g.S;
#pragma unroll
    for (int e = 0; e < E; ++e, q += step) {
        if (!fft_has<K>(out_span, t0, e)) continue;
        const int t = t0 + e * out_span.step;
        if (t < g.n_out) {
            cx<T> w = v[e];
            if (g.pb == 1) w = fft_pb_apply<T>(w, g, pbase, t, false);
            *q = w;
        } else if (g.zero_tail) {
            *q = mkcx<T>((T)0, (T)0);
        }
    }
}

// Circulant embedding of a point-spread function given on the lattice
// d_e in [-N_e, N_e) (element q_e = d_e + N_e, strides ps): T[d mod K] =
// psf[d] * inv_nk for d_e > -N_e on every axis.  T must be zero beforehand;
// K_e >= 2 N_e keeps the wrapped indices distinct.
template <typename T>
__global__ __launch_bounds__(256) void toeplitz_embed_kernel(const cx<T>* __restrict__ psf, cx<T>* __restrict__ t,
                                                             int ndim, int N0, int N1, int N2, int K0, int K1,
                                                             int K2, int64_t ps0, int64_t ps1, int64_t ps2,
                                                             int64_t count, T inv_nk) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int L0 = 2 * N0, L1 = 2 * N1;
    const int q0 = (int)(i % L0);
    const int64_t r = i / L0;
    const int q1 = ndim > 1 ? (int)(r % L1) : 0;
    const int q2 = ndim > 2 ? (int)(r / L1) : 0;
    const int d0 = q0 - N0, d1 = ndim > 1 ? q1 - N1 : 0, d2 = ndim > 2 ? q2 - N2 : 0;
    if (d0 == -N0 || (ndim > 1 && d1 == -N1) || (ndim > 2 && d2 == -N2)) return;
    const int k0 = d0 < 0 ? d0 + K0 : d0;
    const int k1 = d1 < 0 ? d1 + K1 : d1;
    const int k2 = d2 < 0 ? d2 + K2 : d2;
    const cx<T> v = psf[(int64_t)q0 * ps0 + (int64_t)q1 * ps1 + (int64_t)q2 * ps2];
    t[((int64_t)k2 * K1 + k1) * K0 + k0] = mkcx<T>(v.x * inv_nk, v.y * inv_nk);
}

}  // namespace mi355
