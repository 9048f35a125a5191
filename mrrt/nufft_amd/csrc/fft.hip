// Dispatch of the fused pruned FFT passes (kernels_fft.hpp): one pass along
// axis 0 or along an axis d >= 1, for every supported length.
#include "internal.hpp"

namespace mi355host {

namespace {

// The radices of a mixed length k, each at most kFftMaxRadix: as few as
// possible, then the largest smallest one (a line takes k / that threads),
// then an odd one first (its outputs are written at that stride).
void radix_search(int k, int rmax, int* cur, int n, int* best, int* nbest) {
    if (k == 1) {
        if (*nbest == 0 || n < *nbest || (n == *nbest && cur[n - 1] > best[*nbest - 1])) {
            for (int i = 0; i < n; ++i) best[i] = cur[i];
            *nbest = n;
        }
        return;
    }
    if (n == kFftMaxPasses) return;
    for (int r = rmax < k ? rmax : k; r >= 2; --r)
        if (k % r == 0) {
            cur[n] = r;
            radix_search(k / r, r, cur, n + 1, best, nbest);
        }
}

bool radix_list(int k, int* R, int* np) {
    int cur[kFftMaxPasses];
    *np = 0;
    radix_search(k, kFftMaxRadix, cur, 0, R, np);
    for (int i = 0; i < *np; ++i)
        if (R[i] % 2) {
            const int r = R[i];
            for (int q = i; q > 0; --q) R[q] = R[q - 1];
            R[0] = r;
            break;
        }
    return *np > 0;
}

}  // namespace

bool fft_axis_init(int64_t K, FftAxis* ax) {
    if (K < kFftMinK || K > kFftMaxK) return false;
    std::memset(ax, 0, sizeof(*ax));
    ax->K = (int)K;
    if (fft_pow2(K)) {
        ax->TL = ax->K / fft_points(ax->K);
        for (int ns = 1; ns < ax->K; ns *= ax->R[ax->np++]) ax->R[ax->np] = fft_radix(ax->K, ns);
    } else {
        if (!radix_list(ax->K, ax->R, &ax->np)) return false;
        int rmin = kFftMaxRadix;
        for (int p = 0; p < ax->np; ++p) rmin = ax->R[p] < rmin ? ax->R[p] : rmin;
        ax->TL = ax->K / rmin;
        if (ax->TL > 512) return false;
    }
    int ns = 1;
    for (int p = 0; p < ax->np; ++p) {
        ax->off[p] = ax->ntw;
        ax->inv_ns[p] = 1.0f / (float)ns;
        if (ns > 1) ax->ntw += (ax->R[p] - 1) * ns;
        ns *= ax->R[p];
    }
    return true;
}

namespace {

FftRowGeom row_geom(const FftDev& f, const int64_t* xs, int32_t nimg) {
    FftRowGeom g;
    for (int d = 0; d < 3; ++d) {
        g.N[d] = (int)f.N[d];
        g.K[d] = (int)f.K[d];
    }
    g.nk = f.nk;
    for (int d = 0; d < 4; ++d) g.xs[d] = 0;
    for (int d = 0; d < f.ndim; ++d) g.xs[d] = xs[d];
    g.xs[3] = xs[f.ndim];
    g.nlines = (int64_t)g.N[1] * g.N[2] * nimg;
    g.mult = nullptr;
    // C-ordered images (the last axis contiguous): neighbouring lines are
    // adjacent in memory, so the image side is read / written across lines
    g.swap = (f.ndim == 3 && g.xs[0] != 1 && g.xs[1] != 1 && g.xs[2] == 1) ? 1 : 0;
    g.across = (f.ndim >= 2 && g.xs[0] != 1 && (g.xs[1] == 1 || g.swap)) ? 1 : 0;
    g.ax = f.ax[0];
    return g;
}

// lines of axis d >= 1: lpw neighbouring lines of prod(K_0..K_{d-1}) per
// workgroup, for every active index of the next axis and every image
FftColGeom col_geom(const FftDev& f, int d, bool adjoint, int32_t nimg) {
    FftColGeom g;
    g.S = 1;
    for (int e = 0; e < d; ++e) g.S *= f.K[e];
    g.n_in = (int)(adjoint ? f.K[d] : f.N[d]);
    g.n_out = (int)(adjoint ? f.N[d] : f.K[d]);
    g.A = d + 1 < f.ndim ? (int)f.N[d + 1] : 1;
    g.st_a = g.S * f.K[d];
    g.nk = f.nk;
    g.nouter = (int64_t)g.A * nimg;
    g.mult = nullptr;
    g.pb = 0;
    g.ortho = 0;
    g.pb_ndim = f.ndim;
    g.K0 = (int)f.K[0];
    g.pbc[0] = g.pbc[1] = g.pbc[2] = 0.0;
    g.scale_ortho = 1.0;
    g.ax = f.ax[d];
    return g;
}

// Workgroups a pass aims for (measured best on 512^2 grids): lines per workgroup grow only
// while the pass keeps at least this many workgroups.
constexpr int64_t kFftTargetBlocks = 128;
// LDS of one workgroup: two fit a CU's 160 KB
constexpr size_t kFftLds = 81920;

size_t fft_lds_bytes(const FftAxis& ax, int lpw, int cxs) {
    return ((size_t)lpw * fft_line_stride(ax.K, lpw, cxs) + ax.ntw) * cxs;
}
// threads of lpw lines: whole waves for the mixed lengths (surplus idle)
unsigned fft_threads(const FftAxis& ax, int lpw) {
    const int n = lpw * ax.TL;
    return (unsigned)(fft_pow2(ax.K) ? n : (n + 63) / 64 * 64);
}

template <typename T, int K>
int launch_fft_rows(const FftDev& f, bool adjoint, const void* x, void* xo, const int64_t* xs, void* grid,
                    int32_t nimg, T scale, FftPassOpts o) {
    constexpr int cxs = 2 * (int)sizeof(T);
    FftRowGeom g = row_geom(f, xs, nimg);
    g.mult = o.mult;
    // more lines per workgroup across C-ordered images, for longer contiguous
    // runs of the image side (16 lines of complex64: one 128-byte line)
    const int max_threads = g.across ? kFftThreads<T, K> : 256;
    const int max_lpw = g.across ? 128 / cxs : 64;
    int lpw = 1;
    while (2 * lpw <= max_lpw && 2 * lpw * g.ax.TL <= max_threads && fft_lds_bytes(g.ax, 2 * lpw, cxs) <= kFftLds &&
           g.nlines / (2 * lpw) >= kFftTargetBlocks)
        lpw *= 2;
    g.lpw = lpw;
    g.stride = fft_line_stride(g.ax.K, lpw, cxs);
    const int64_t nb = (g.nlines + lpw - 1) / lpw;
    const dim3 threads(fft_threads(g.ax, lpw));
    const size_t lds = fft_lds_bytes(g.ax, lpw, cxs);
    const double* s0 = f.sn ? f.sn[0] : nullptr;
    const double* s1 = f.sn && f.ndim > 1 ? f.sn[1] : s0;
    const double* s2 = f.sn && f.ndim > 2 ? f.sn[2] : s0;
    if (adjoint)
        hipLaunchKernelGGL((fft_rows_crop_kernel<T, K, 1>), dim3((unsigned)nb), threads, lds, f.stream, (cx<T>*)grid,
                           (cx<T>*)xo, g, s0, s1, s2, f.ndim, scale, (const cx<T>*)f.tw[0], o.rezero);
    else
        hipLaunchKernelGGL((fft_rows_pad_kernel<T, K, -1>), dim3((unsigned)nb), threads, lds, f.stream,
                           (const cx<T>*)x, (cx<T>*)grid, g, s0, s1, s2, f.ndim, (const cx<T>*)f.tw[0]);
    LAUNCH_CHECK();
    return MI355NUFFT_OK;
}

template <typename T, int K>
int launch_fft_cols(const FftDev& f, bool adjoint, int d, void* grid, int32_t nimg, FftPassOpts o) {
    constexpr int cxs = 2 * (int)sizeof(T);
    FftColGeom g = col_geom(f, d, adjoint, nimg);
    g.zero_tail = o.rezero;
    g.mult = o.mult;
    if (o.pb) {
        g.pb = o.pb;
        for (int e = 0; e < 3; ++e) g.pbc[e] = o.pbc ? o.pbc[e] : 0.0;
        g.ortho = o.ortho;
        g.scale_ortho = o.scale_ortho;
    }
    // up to 128 contiguous bytes per row, while the pass keeps its workgroups
    int lpw = 1;
    while (2 * lpw * cxs <= 128 && 2 * lpw <= g.S && 2 * lpw * g.ax.TL <= kFftThreads<T, K> &&
           fft_lds_bytes(g.ax, 2 * lpw, cxs) <= kFftLds &&
           (g.S / (2 * lpw)) * g.nouter >= kFftTargetBlocks)
        lpw *= 2;
    g.lpw = lpw;
    g.nchunk = (int)((g.S + lpw - 1) / lpw);
    g.stride = fft_line_stride(g.ax.K, lpw, cxs);
    const int64_t nb = g.nchunk * g.nouter;
    if (nb >= ((int64_t)1 << 32)) return fail(MI355NUFFT_EINVAL, "FFT launch too large");
    const dim3 threads(fft_threads(g.ax, lpw));
    const size_t lds = fft_lds_bytes(g.ax, lpw, cxs);
    auto kernel = adjoint ? fft_cols_kernel<T, K, 1> : fft_cols_kernel<T, K, -1>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)nb), threads, lds, f.stream, (cx<T>*)grid, g, (const cx<T>*)f.tw[d]);
    LAUNCH_CHECK();
    return MI355NUFFT_OK;
}

}  // namespace

#define MI355_FFT_SWITCH(KV, CALL)                                        \
    switch (fft_pow2(KV) ? (int)(KV) : 0) {                               \
        case 0: return CALL(0);                                           \
        case 16: return CALL(16);                                         \
        case 32: return CALL(32);                                         \
        case 64: return CALL(64);                                         \
        case 128: return CALL(128);                                       \
        case 256: return CALL(256);                                       \
        case 512: return CALL(512);                                       \
        case 1024: return CALL(1024);                                     \
        case 2048: return CALL(2048);                                     \
        default: return fail(MI355NUFFT_EINVAL, "no fused FFT for K=%d", (int)(KV)); \
    }

template <typename T>
int fft_rows(const FftDev& f, bool adjoint, const void* x, void* xo, const int64_t* xs, void* grid, int32_t nimg,
             T scale, FftPassOpts o) {
#define MI355_ROWS(KK) launch_fft_rows<T, KK>(f, adjoint, x, xo, xs, grid, nimg, scale, o)
    MI355_FFT_SWITCH((int)f.K[0], MI355_ROWS)
#undef MI355_ROWS
}

template <typename T>
int fft_cols(const FftDev& f, bool adjoint, int d, void* grid, int32_t nimg, FftPassOpts o) {
#define MI355_COLS(KK) launch_fft_cols<T, KK>(f, adjoint, d, grid, nimg, o)
    MI355_FFT_SWITCH((int)f.K[d], MI355_COLS)
#undef MI355_COLS
}

template int fft_rows<float>(const FftDev&, bool, const void*, void*, const int64_t*, void*, int32_t, float,
                             FftPassOpts);
template int fft_rows<double>(const FftDev&, bool, const void*, void*, const int64_t*, void*, int32_t, double,
                              FftPassOpts);
template int fft_cols<float>(const FftDev&, bool, int, void*, int32_t, FftPassOpts);
template int fft_cols<double>(const FftDev&, bool, int, void*, int32_t, FftPassOpts);

}  // namespace mi355host
