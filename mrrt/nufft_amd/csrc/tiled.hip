// Dispatch of the tiled gather, scatter and trajectory-gradient kernels
// (kernels_binned.hpp) for one value type and kernel kind, chosen at compile
// time: built once per (MI355_TILED_T, MI355_TILED_CK) in {float, double} x
// {real kernel 0, complex kernel 1}.
#include "internal.hpp"

#if !defined(MI355_TILED_T) || !defined(MI355_TILED_CK)
#error "build with -DMI355_TILED_T=float|double -DMI355_TILED_CK=0|1"
#endif

namespace mi355host {

template <typename T, bool CK, int NDIM, int JMAX, bool FIXED>
void launch_tiled(bool adjoint, const TiledArgs<T, CK>& a, unsigned nsub, unsigned threads, size_t lds,
                  hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    // coefficients cached across repetitions (and, with the fixed-point
    // tile, the sample read by the scale's sum): only when a subproblem fits
    // one point per thread (the cache costs registers even when unused:
    // 135 VGPRs against 110 for the 2-D J = 6 fixed-point scatter)
    const bool reps = (a.ia.nreps > 1 || a.cmax > 0.f) && a.bg.P <= (int)threads && !a.no_cache;
    // a.rc == 2 for the scatter: two repetitions' tiles per pass
    const bool pair = adjoint && a.rc == 2;
    auto spread = pair ? spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false, false, 2>
                       : reps ? spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false, true>
                              : spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false, false>;
    if constexpr (sizeof(T) == 4)
        if (a.cmax > 0.f)
            spread = pair ? spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, false, 2>
                          : reps ? spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, true>
                                 : spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, false>;
    if constexpr (sizeof(T) == 4 && NDIM == 2)  // finer steps in large bins
        if (a.cmax > 0.f && (pair || !reps) && a.bg.B[0] * a.bg.B[1] > 256 && a.bg.P <= kWindowMaxP)
            spread = pair ? spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, false, 2, true>
                          : spread_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, false, 1, true>;
    auto interp = a.rc > 1 ? interp_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true>
                           : interp_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false>;
    if constexpr (FIXED)  // fused tap sums unless the reference's roundings are asked for
        if (!a.exact)
            interp = a.rc > 1 ? interp_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true, true>
                              : interp_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false, true>;
    // one row of workgroups per pass over the repetitions (the coefficients are
    // formed again for each pass either way), so that few subproblems still
    // fill the chip: scatter of 12 repetitions at Kd 640^2, 128,640 points,
    // 197 -> 138 us, 8 at Kd 512^2 91 -> 70 us, 8 at Kd 128^2 54 -> 19 us,
    // gather 58 -> 45 us at the first.  The coefficient cache keeps its
    // passes in one workgroup.
    const int passes = (a.ia.nreps + a.rc - 1) / a.rc;
    const dim3 grid(nsub, adjoint && reps && !pair ? 1 : passes);
    if (ev1) {
        if (adjoint)
            hipExtLaunchKernelGGL(spread, grid, dim3(threads), (uint32_t)lds, s, ev0, ev1, 0u, a);
        else
            hipExtLaunchKernelGGL(interp, grid, dim3(threads), (uint32_t)lds, s, ev0, ev1, 0u, a);
        return;
    }
    if (adjoint)
        hipLaunchKernelGGL(spread, grid, dim3(threads), lds, s, a);
    else
        hipLaunchKernelGGL(interp, grid, dim3(threads), lds, s, a);
}

// Denser bins are left to the atomic kernel: one batch of points, or half a
// point per cell of larger bins.  Adjoint of 24 frames x 32 coils: 16x16 bins
// 2.06 ms with 256, 2.10 with 512, 2.45 with 1024; 32x32 bins 2.35 / 2.20 /
// 2.30; 4 frames x 32 coils 505 / 511 / 635 us, 511 / 488 / 525.
inline int owner_heavy(const mi355nufft_plan* p) {
    const int half = p->bg.B[0] * p->bg.B[1] / 2;
    return half > kOwnerBatch ? half : kOwnerBatch;
}

template <bool CK, int JMAX, bool FIXED>
int launch_owner(mi355nufft_plan* p, const TiledArgs<float, CK>& a, hipEvent_t ev0) {
    OwnerGeom og;
    og.nt0 = (int)((p->K[0] + kOwnerB - 1) / kOwnerB);
    og.nt1 = (int)((p->K[1] + kOwnerB - 1) / kOwnerB);
    og.S = owner_stride(p);
    og.R1 = kOwnerB + 2 * (p->J[1] - 1);
    og.ngrp = (a.ia.nreps + kOwnerReps - 1) / kOwnerReps;
    const int64_t nb = (int64_t)og.nt0 * og.nt1 * p->nframes * og.ngrp;
    if (nb >= ((int64_t)1 << 31)) return fail(MI355NUFFT_EINVAL, "scatter launch too large");
    auto kernel = spread_owner_kernel<CK, JMAX, FIXED>;
    const size_t lds = 2 * owner_plane_bytes(p);
    if (ev0)
        hipExtLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(256), (uint32_t)lds, p->stream, ev0, nullptr, 0u, a, og);
    else
        hipLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(256), lds, p->stream, a, og);
    LAUNCH_CHECK();
    return MI355NUFFT_OK;
}

template <bool CK>
int run_owner(mi355nufft_plan* p, const TiledArgs<float, CK>& a, hipEvent_t ev0) {
    const int j = p->J[0] == p->J[1] ? p->J[0] : 0;
    if (j == 4) return launch_owner<CK, 4, true>(p, a, ev0);
    if (j == 5) return launch_owner<CK, 5, true>(p, a, ev0);
    if (j == 6) return launch_owner<CK, 6, true>(p, a, ev0);
    if (p->J[0] <= 4 && p->J[1] <= 4) return launch_owner<CK, 4, false>(p, a, ev0);
    return launch_owner<CK, 8, false>(p, a, ev0);
}

// Repetitions staged together by the gather and the gradient where only one
// tile fits the chunk: two for the compiled tap loops (complex128 tiles of
// 32x32 bins, 22 KB).  8 coils on Kd 1024^2, J = 6, one / two tiles, 0.33 points
// per cell gather 165 / 108 us, gradient 217 / 176; forward of 4 frames x 32
// coils on Kd 512^2 977 / 749.  Not for two or three repetitions, whose single
// tiles run side by side (20,000 points on Kd 600^2, two, gather 13.4 / 15.1), nor
// for the generic loops (J = 7, eight: 40.7 / 46.1).
inline int pair_rather_than_one(const mi355nufft_plan* p, int rc, size_t one, size_t chunk, int32_t nreps) {
    const int32_t J[3] = {p->J[0], p->J[1], p->J[2]};
    return rc == 1 && nreps >= 4 && fixed_j(p->ndim, J) && 2 * one <= (chunk * 13) / 10 ? 2 : rc;
}

template <typename T, bool CK>
int run_tiled(mi355nufft_plan* p, bool adjoint, const void* samples_in, void* samples_out, const void* grid_in,
              void* grid_out, int32_t nreps) {
    TiledArgs<T, CK> a;
    std::memset(&a, 0, sizeof(a));
    int32_t J[3] = {p->J[0], p->J[1], p->J[2]};
    fill_interp_args<T, CK>(a.ia, p->ndim, p->K, J, p->L, (const void* const*)p->d_tab, p->d_tm, p->M, nreps);
    a.ia.grid = (const cx<T>*)grid_in;
    a.ia.grid_out = (cx<T>*)grid_out;
    a.ia.in = (const cx<T>*)samples_in;
    a.ia.out = (cx<T>*)samples_out;
    a.ia.phase = p->has_phase ? (const cx<T>*)p->d_phase : nullptr;
    a.bg = p->bg;
    a.bs = bin_state(p);
    a.use_pb = p->phasing == 0 && !p->fft_phased;
    for (int d = 0; d < 3; ++d) a.pb[d] = (T)p->phase_coef[d];
    a.ortho = adjoint ? 0 : (p->ortho && !p->fft_phased);
    a.scale_ortho = (T)p->scale_ortho;
    a.tiles = adjoint ? (cx<T>*)p->tiles_target : nullptr;
    a.tms = (const T*)p->d_tms;
    a.phs = p->has_phase ? (const cx<T>*)p->d_phs : nullptr;
    a.cmax = (adjoint && use_fxp(p)) ? (float)p->tab_cmax : 0.f;  // > 0: fixed-point scatter tile
    a.exact = p->exact_taps;
    a.own_ok = 1;
    for (int d = 0; d < p->ndim; ++d)
        if (p->K[d] % p->bg.B[d] != 0) a.own_ok = 0;
    const unsigned nsub = tiled_grid(p);
    // the gather stages up to kMaxRepChunk repetitions' tiles at once
    // (coefficients are then computed once per point for all of them),
    // within the LDS budget; the scatter one or two at a time
    const size_t one = adjoint ? tile_bytes(p) : gather_tile_bytes(p);
    const size_t chunk_lds = p->lds_limit < kRepChunkLds ? p->lds_limit : kRepChunkLds;
    int rc = adjoint ? 1 : (int)(chunk_lds / one);
    if (!adjoint) rc = pair_rather_than_one(p, rc, one, chunk_lds, nreps);
    rc = rc < kMaxRepChunk ? rc : kMaxRepChunk;
    rc = rc < nreps ? rc : nreps;
    a.rc = rc > 1 ? rc : 1;
    // the scatter takes two repetitions per pass when both tiles fit the
    // chunk budget and its points would not fit the coefficient cache, which
    // the default points per subproblem of large bins leave out (its scale is
    // the coarser one)
    a.no_cache = p->ndim == 2 && p->P_req == 0 && p->bg.B[0] * p->bg.B[1] > 256;
    if (adjoint && nreps >= 2 && kScatterPairs && 2 * one <= chunk_lds && (p->bg.P > p->bg_threads || a.no_cache))
        a.rc = 2;
    const size_t lds = one * (size_t)a.rc;
    const int jm = jmax_of(p->ndim, J);
    const int jf = fixed_j(p->ndim, J);
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    RET_IF(timing_events(p, adjoint ? 1 : 0, &ev0, &ev1));
    // counted with the timed launches when asked for (the count's final
    // atomics lengthen a short launch, so timing alone leaves it out)
    a.flush_count = (adjoint && ev0 && (p->timing & 2)) ? p->d_flush_count : nullptr;
    a.flush_slots = kFlushSlots;
    if constexpr (sizeof(T) == 4)
        if (adjoint && use_owner(p, nreps)) {
            // two launches, timed as one: from the first's start to the second's end
            a.heavy = owner_heavy(p);
            RET_IF(run_owner<CK>(p, a, ev0));
            ev0 = nullptr;
        }
#define MI355_FCASE(ND, JF)                                                    \
    if (p->ndim == ND && jf == JF) {                                           \
        launch_tiled<T, CK, ND, JF, true>(adjoint, a, nsub, p->bg_threads, lds, p->stream, ev0, ev1); \
        LAUNCH_CHECK();                                                        \
        return MI355NUFFT_OK;                                                  \
    }
    MI355_FCASE(1, 4) MI355_FCASE(2, 4) MI355_FCASE(3, 4)
    MI355_FCASE(1, 5) MI355_FCASE(2, 5) MI355_FCASE(3, 5)
    MI355_FCASE(1, 6) MI355_FCASE(2, 6) MI355_FCASE(3, 6)
#undef MI355_FCASE
#define MI355_TCASE(ND, JM)                                                  \
    if (p->ndim == ND && jm == JM) {                                         \
        launch_tiled<T, CK, ND, JM, false>(adjoint, a, nsub, p->bg_threads, lds, p->stream, ev0, ev1); \
        LAUNCH_CHECK();                                                      \
        return MI355NUFFT_OK;                                                \
    }
    MI355_TCASE(1, 4) MI355_TCASE(1, 8) MI355_TCASE(1, 16)
    MI355_TCASE(2, 4) MI355_TCASE(2, 8) MI355_TCASE(2, 16)
    MI355_TCASE(3, 4) MI355_TCASE(3, 8) MI355_TCASE(3, 16)
#undef MI355_TCASE
    return fail(MI355NUFFT_EINVAL, "unsupported ndim/J combination");
}

template <typename T, bool CK, int NDIM, int JMAX, bool FIXED>
void launch_grad(const TiledArgs<T, CK>& a, const GradArgs<T>& g, unsigned nsub, unsigned threads, size_t lds,
                 hipStream_t s) {
    if (a.rc > 1)
        hipLaunchKernelGGL((grad_tiled_kernel<T, NDIM, CK, JMAX, FIXED, true>), dim3(nsub), dim3(threads), lds, s, a,
                           g);
    else
        hipLaunchKernelGGL((grad_tiled_kernel<T, NDIM, CK, JMAX, FIXED, false>), dim3(nsub), dim3(threads), lds, s,
                           a, g);
}

template <typename T, bool CK>
int run_grad(mi355nufft_plan* p, const void* grid, const void* w, void* grad, int32_t nreps) {
    TiledArgs<T, CK> a;
    std::memset(&a, 0, sizeof(a));
    int32_t J[3] = {p->J[0], p->J[1], p->J[2]};
    fill_interp_args<T, CK>(a.ia, p->ndim, p->K, J, p->L, (const void* const*)p->d_tab, p->d_tm, p->M, nreps);
    a.ia.grid = (const cx<T>*)grid;
    a.ia.phase = p->has_phase ? (const cx<T>*)p->d_phase : nullptr;
    a.bg = p->bg;
    a.bs = bin_state(p);
    a.use_pb = p->phasing == 0;
    for (int d = 0; d < 3; ++d) a.pb[d] = (T)p->phase_coef[d];
    a.ortho = p->ortho;
    a.scale_ortho = (T)p->scale_ortho;
    a.tms = (const T*)p->d_tms;
    a.phs = p->has_phase ? (const cx<T>*)p->d_phs : nullptr;
    GradArgs<T> g;
    g.w = (const cx<T>*)w;
    g.grad = (T*)grad;
    for (int d = 0; d < 3; ++d) {
        g.dtdw[d] = (T)((double)p->K[d] / (2.0 * M_PI));
        g.shift[d] = (T)p->shift[d];
    }
    const unsigned nsub = tiled_grid(p);
    {  // repetitions staged per pass, as in the gather; up to 52 KB (three
       // workgroups per CU) where that takes all of them at once
        const size_t chunk = p->lds_limit < kRepChunkLds ? p->lds_limit : kRepChunkLds;
        const size_t one = gather_tile_bytes(p);
        int rc = (int)((nreps <= kMaxRepChunk && nreps * one <= (chunk * 13) / 10 ? nreps * one : chunk) / one);
        rc = pair_rather_than_one(p, rc, one, chunk, nreps);
        rc = rc < kMaxRepChunk ? rc : kMaxRepChunk;
        rc = rc < nreps ? rc : nreps;
        a.rc = rc > 1 ? rc : 1;
    }
    const size_t lds = gather_tile_bytes(p) * (size_t)a.rc;
    const int jm = jmax_of(p->ndim, J);
    const int jf = fixed_j(p->ndim, J);
#define MI355_GFCASE(ND, JF)                                           \
    if (p->ndim == ND && jf == JF) {                                   \
        launch_grad<T, CK, ND, JF, true>(a, g, nsub, p->bg_threads, lds, p->stream);  \
        LAUNCH_CHECK();                                                \
        return MI355NUFFT_OK;                                          \
    }
    MI355_GFCASE(1, 4) MI355_GFCASE(2, 4) MI355_GFCASE(3, 4)
    MI355_GFCASE(1, 5) MI355_GFCASE(2, 5) MI355_GFCASE(3, 5)
    MI355_GFCASE(1, 6) MI355_GFCASE(2, 6) MI355_GFCASE(3, 6)
#undef MI355_GFCASE
#define MI355_GCASE(ND, JM)                                            \
    if (p->ndim == ND && jm == JM) {                                   \
        launch_grad<T, CK, ND, JM, false>(a, g, nsub, p->bg_threads, lds, p->stream); \
        LAUNCH_CHECK();                                                \
        return MI355NUFFT_OK;                                          \
    }
    MI355_GCASE(1, 4) MI355_GCASE(1, 8) MI355_GCASE(1, 16)
    MI355_GCASE(2, 4) MI355_GCASE(2, 8) MI355_GCASE(2, 16)
    MI355_GCASE(3, 4) MI355_GCASE(3, 8) MI355_GCASE(3, 16)
#undef MI355_GCASE
    return fail(MI355NUFFT_EINVAL, "unsupported ndim/J combination");
}

template int run_tiled<MI355_TILED_T, (bool)MI355_TILED_CK>(mi355nufft_plan*, bool, const void*, void*, const void*,
                                                             void*, int32_t);
template int run_grad<MI355_TILED_T, (bool)MI355_TILED_CK>(mi355nufft_plan*, const void*, const void*, void*, int32_t);

}  // namespace mi355host
