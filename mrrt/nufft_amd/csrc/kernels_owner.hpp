// Scatter of many images onto 2-D grids without atomics on the grid: a
// workgroup owns kOwnerB x kOwnerB grid cells of up to kOwnerReps
// repetitions, collects every point whose taps reach them (the bins that hold
// first taps from J - 1 cells below the tile to its last cell), accumulates
// in LDS and writes each of its cells itself.
//
// What it replaces: the tile per bin subproblem (spread_tiled_kernel) adds
// its halo, and cells shared between subproblems, to the grid with one
// global float atomic per component, which needs a cleared grid.
// Here points near a tile's edge are evaluated by up to four workgroups
// ((32 + 5)^2 / 32^2 = 1.34 evaluations per point at J = 6), and the grid is
// written in whole lines with no clear.  24 frames x 32 coils of Kd 512^2
// (64x32 bins): 93.7 M -> 22.8 M global atomics per scatter and 1.85 -> 1.63
// ms.  The bytes do not fall (2.10 -> 2.62 GB by the HBM counters: samples are
// read again for each tile they reach, and the atomic kernel skips empty
// cells); what falls is the atomics and, because nothing has to be left zero,
// the stores of the inverse FFT passes (columns 626 -> 490 us, crop 386 ->
// 250 us).
//
// Points of bins with more than `heavy` points are left to the atomic kernel,
// launched afterwards on top of what this one stored, so that a dense
// k-space centre does not serialise on the one workgroup that owns it.
#pragma once

#include "kernels_binned.hpp"

namespace mi355 {

constexpr int kOwnerB = 32;        // cells per axis of an owned tile
constexpr int kOwnerBatch = 256;   // points accumulated at one fixed-point scale, one per thread
constexpr int kOwnerList = kOwnerBatch + 256;
constexpr int kOwnerSegs = 64;     // bins a tile may draw points from
constexpr int kOwnerMaxJ = 8;      // taps per axis
constexpr int kOwnerReps = 8;      // repetitions of a workgroup, two at a time in LDS

struct OwnerGeom {
    int nt0, nt1;  // tiles per axis
    int S;         // LDS row stride, congruent to the bin tiles' (keeps their bank order)
    int R1;        // LDS rows, kOwnerB + 2 (J1 - 1)
    int ngrp;      // groups of kOwnerReps repetitions
};

// Bins that hold first taps k in [lo, hi] along one axis, 0 <= lo <= hi < K.
__device__ __forceinline__ int owner_bins(int lo, int hi, int B) { return hi / B - lo / B + 1; }

// One point per thread: its coefficients serve all repetitions of the
// workgroup, whose samples are loaded together.
// The fixed-point scale is that of spread_tiled_kernel with a tighter bound
// of the cell sums: a cell collects samples whose first taps lie in J cells
// per axis, hence in two neighbouring blocks of b >= J - 1 cells per axis, so
// A is the largest sum of |Re y| + |Im y| over 2 x 2 blocks (10 x 10 cells at
// J = 6) instead of the sum over the whole 37 x 37 neighbourhood (the atomic
// kernel's is over a bin, 16 x 16 cells by default).  The block sums are
// integers in units of 2^-20 of the power of two above the batch's largest
// sample, each sample rounded up.
template <bool CK, int JMAX, bool FIXED>
__global__ __launch_bounds__(256) void spread_owner_kernel(TiledArgs<float, CK> a, OwnerGeom og) {
    constexpr int RC = 2, NR = kOwnerReps;
    constexpr int NB = 8;                              // blocks per axis: 37 first taps / 5, 38 / 6, 39 / 7
    constexpr int CELLS = kOwnerB * kOwnerB / 256;     // owned cells per thread
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_list[kOwnerList];
    __shared__ int s_start[kOwnerSegs], s_off[kOwnerSegs + 1];
    __shared__ int s_cnt;
    __shared__ float s_max[4 * NR];
    __shared__ unsigned s_blk[NR * NB * NB];
    __shared__ int s_shift[NR];
    const InterpArgs<float, CK>& ia = a.ia;
    const BinGeom& bg = a.bg;
    const AxisGeom ax[3] = {ia.ax[0], ia.ax[1], ia.ax[2]};
    const int K0 = ax[0].K, K1 = ax[1].K;
    const int J0 = FIXED ? JMAX : ax[0].J, J1 = FIXED ? JMAX : ax[1].J;
    const float inv_b0 = 1.0f / (float)max(J0 - 1, 5), inv_b1 = 1.0f / (float)max(J1 - 1, 5);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int S = og.S, plane = S * og.R1;
    int* const tiles = reinterpret_cast<int*>(smem);
    unsigned w = blockIdx.x;
    const int grp = (int)(w % (unsigned)og.ngrp);
    w /= (unsigned)og.ngrp;
    const int tx = (int)(w % (unsigned)og.nt0);
    w /= (unsigned)og.nt0;
    const int ty = (int)(w % (unsigned)og.nt1);
    const int frame = (int)(w / (unsigned)og.nt1);
    const int o0 = tx * kOwnerB, o1 = ty * kOwnerB;
    const int w0 = min(kOwnerB, K0 - o0), w1 = min(kOwnerB, K1 - o1);
    const int rbase = grp * NR, nr = min(NR, ia.nreps - rbase);

    // the light bins that hold this tile's first taps: [o - (J - 1), o + w)
    // is one interval of [0, K), or two where it wraps (K >= 32 + 2 (J - 1))
    if (wave == 0) {
        const int l0 = max(o0 - (J0 - 1), 0), h0 = o0 + w0 - 1, e0 = o0 - (J0 - 1) + K0;  // e0 < K0: wrapped part
        const int l1 = max(o1 - (J1 - 1), 0), h1 = o1 + w1 - 1, e1 = o1 - (J1 - 1) + K1;
        const int na0 = owner_bins(l0, h0, bg.B[0]), na1 = owner_bins(l1, h1, bg.B[1]);
        // a bin that holds both the wrapped part and the start of the range counts once
        const int wr0 = e0 < K0 ? max(e0 / bg.B[0], h0 / bg.B[0] + 1) : bg.nb[0];
        const int wr1 = e1 < K1 ? max(e1 / bg.B[1], h1 / bg.B[1] + 1) : bg.nb[1];
        const int n0 = na0 + (bg.nb[0] - wr0), n1 = na1 + (bg.nb[1] - wr1);
        int start = 0, len = 0;
        if (lane < n0 * n1) {
            const int q1 = lane / n0, q0 = lane - q1 * n0;
            const int b0 = q0 < na0 ? l0 / bg.B[0] + q0 : wr0 + (q0 - na0);
            const int b1 = q1 < na1 ? l1 / bg.B[1] + q1 : wr1 + (q1 - na1);
            const int bin = frame * bg.nbins_frame + b1 * bg.nb[0] + b0;
            const int c = a.bs.counts[bin];
            if (c <= a.heavy) {
                start = a.bs.bin_start[bin];
                len = c;
            }
        }
        int sum = len;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(sum, o);
            if (lane >= o) sum += v;
        }
        s_start[lane] = start;
        s_off[lane + 1] = sum;
        if (lane == 0) {
            s_off[0] = 0;
            s_cnt = 0;
        }
    }
    int4* const tiles4 = reinterpret_cast<int4*>(smem);  // 2 RC planes: a multiple of four ints
    for (int e = tid; e < RC * plane / 2; e += 256) tiles4[e] = make_int4(0, 0, 0, 0);
    for (int e = tid; e < NR * NB * NB; e += 256) s_blk[e] = 0;
    __syncthreads();
    const int total = s_off[kOwnerSegs];

    // first taps of sorted point i relative to the tile, J - 1 added (>= 0); false: none in the tile
    auto local = [&](float t0, float t1, int& l0, int& l1) {
        l0 = first_tap_mod(t0, J0, K0) - o0;
        l1 = first_tap_mod(t1, J1, K1) - o1;
        if (l0 >= w0) l0 -= K0;
        if (l1 >= w1) l1 -= K1;
        l0 += J0 - 1;
        l1 += J1 - 1;
        return l0 >= 0 && l1 >= 0 && l0 < w0 + J0 - 1 && l1 < w1 + J1 - 1;
    };

    int have = 0;       // points in the list (uniform)
    bool first = true;  // no batch has been stored yet
    for (int c0 = 0; c0 < total || have > 0 || first; c0 += 256) {
        if (c0 < total) {
            const int c = c0 + tid;
            int i = 0;
            bool keep = false;
            if (c < total) {
                int lo = 0;  // last segment with s_off[lo] <= c
#pragma unroll
                for (int step = kOwnerSegs / 2; step > 0; step >>= 1)
                    if (s_off[lo + step] <= c) lo += step;
                i = s_start[lo] + (c - s_off[lo]);
                int l0, l1;
                keep = local(a.tms[i], a.tms[ia.M + i], l0, l1);
            }
            const unsigned long long m = __ballot(keep);
            int base = 0;
            if (lane == 0 && m) base = atomicAdd(&s_cnt, __popcll(m));
            base = __shfl(base, 0);
            if (keep) s_list[base + __popcll(m & ((1ull << lane) - 1ull))] = i;
            __syncthreads();
            have = s_cnt;
        }
        if (have < kOwnerBatch && c0 + 256 < total) {
            __syncthreads();  // s_cnt is read before the next round adds to it
            continue;
        }
        if (have == 0 && !first) break;
        const int n = min(have, kOwnerBatch);

        // this thread's point, its coefficients and the size of its samples
        const int pi = tid < n ? s_list[tid] : -1;
        float mx[NR];
        PointTaps<float, CK, JMAX> pt;
        pt.l[0] = pt.l[1] = 0;
        pt.ph = make_float2(1.f, 0.f);
        const float2* yp = ia.in + (int64_t)rbase * ia.M;
#pragma unroll
        for (int k = 0; k < NR; ++k) mx[k] = 0.f;
        if (pi >= 0) {
            yp += a.bs.perm[pi];
            const float t[2] = {a.tms[pi], a.tms[ia.M + pi]};
            if (a.phs) pt.ph = a.phs[pi];
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (k < nr) {
                    const float2 y = yp[(int64_t)k * ia.M];
                    mx[k] = fabsf(y.x) + fabsf(y.y);
                }
            (void)local(t[0], t[1], pt.l[0], pt.l[1]);
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                if constexpr (CK)
                    (void)axis_coefs<float, JMAX, FIXED>(t[d], ia.L, ax[d], ia.h[d], pt.cr[d], pt.ci[d]);
                else
                    (void)axis_coefs<float, JMAX, FIXED>(t[d], ia.L, ax[d], ia.h[d], pt.cr[d]);
            }
        }
        // largest |Re y| + |Im y| of each repetition (NaN stays)
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (k >= nr) break;
            float v = mx[k];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const float u = __shfl_xor(v, o);
                v = u > v || !(u == u) ? u : v;
            }
            if (lane == 0) s_max[wave * NR + k] = v;
        }
        __syncthreads();
        unsigned bad = 0;  // bit k: a non-finite sample
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (k >= nr) break;
            float v = s_max[k];
#pragma unroll
            for (int q = 1; q < 4; ++q) {
                const float u = s_max[q * NR + k];
                v = u > v || !(u == u) ? u : v;
            }
            if (!(v <= 3.4e38f)) {
                bad |= 1u << k;
                continue;
            }
            int ev = 0;  // the largest sample is below 2^ev
            (void)frexpf(v, &ev);
            if (pi >= 0)
                atomicAdd(&s_blk[(k * NB + div_small(pt.l[1], inv_b1)) * NB + div_small(pt.l[0], inv_b0)],
                          (unsigned)ceilf(ldexpf(mx[k], 20 - ev)) + 1u);
            if (tid == k) s_shift[k] = ev;
        }
        __syncthreads();
        // wave w finds the scales of repetitions w, w + 4: A = (largest window) 2^(ev - 20) cmax 1.001 < 2^(31 - sh)
        for (int k = wave; k < nr; k += 4) {
            unsigned win = 0;
            if (lane < (NB - 1) * (NB - 1)) {
                const unsigned* q = s_blk + (k * NB + lane / (NB - 1)) * NB + lane % (NB - 1);
                win = q[0] + q[1] + q[NB] + q[NB + 1];
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) win = max(win, (unsigned)__shfl_xor((int)win, o));
            int e = 0;
            (void)frexpf((float)win * a.cmax * 1.001f, &e);
            if (lane < NB * NB) s_blk[k * NB * NB + lane] = 0;  // for the next batch
            if (lane == 0) s_shift[k] = 51 - s_shift[k] - e;
        }
        __syncthreads();
        // the samples again (cached), those of the next pass while this one's are spread
        float2 yn[RC];
#pragma unroll
        for (int k = 0; k < RC; ++k) yn[k] = pi >= 0 && k < nr ? yp[(int64_t)k * ia.M] : make_float2(0.f, 0.f);
#pragma unroll 1
        for (int p0 = 0; p0 < nr; p0 += RC) {
            float2 py[RC];
#pragma unroll
            for (int k = 0; k < RC; ++k) {
                py[k] = yn[k];
                if (pi >= 0 && p0 + RC + k < nr) yn[k] = yp[(int64_t)(p0 + RC + k) * ia.M];
            }
            if (pi >= 0) {
#pragma unroll
                for (int k = 0; k < RC; ++k) {
                    if (p0 + k >= nr || (bad >> (p0 + k) & 1)) continue;
                    const int sh = s_shift[p0 + k];
                    float2 f = times_conj_phase<float, CK, JMAX>(py[k], pt, a.phs);
                    f.x = ldexpf(f.x, sh);
                    f.y = ldexpf(f.y, sh);
                    int* tre = tiles + 2 * k * plane;
                    scatter_taps_fx<2, CK, JMAX, FIXED, false>(tre, tre + plane, pt, f, ax, S, og.R1);
                }
            }
            __syncthreads();
            // the owned cells to the grid
#pragma unroll
            for (int k = 0; k < RC; ++k) {
                if (p0 + k >= nr) break;
                int* tre = tiles + 2 * k * plane;
                const int sh = s_shift[p0 + k];
                const bool badk = bad >> (p0 + k) & 1;
                float2* g = ia.grid_out + ((int64_t)frame * ia.nreps + rbase + p0 + k) * ia.kstride;
#pragma unroll
                for (int c = 0; c < CELLS; ++c) {
                    const int e = tid + 256 * c, x = e % kOwnerB, y = e / kOwnerB;
                    const int q = (y + J1 - 1) * S + x + J0 - 1;
                    float vr = ldexpf((float)tre[q], -sh), vi = ldexpf((float)tre[plane + q], -sh);
                    if (badk) vr = vi = __int_as_float(0x7fc00000);
                    if (x < w0 && y < w1) {
                        if (a.use_pb) {  // * conj(phase_before)
                            const float pc[3] = {a.pb[0], a.pb[1], a.pb[2]};
                            const float2 p = cis_tile(phase_before_arg<float>(pc, 2, o0 + x, o1 + y, 0));
                            const float wr = vr * p.x + vi * p.y;
                            const float wi = vi * p.x - vr * p.y;
                            vr = wr;
                            vi = wi;
                        }
                        float2* o = g + (int64_t)(o1 + y) * K0 + o0 + x;
                        if (!first) {  // an earlier batch of this workgroup stored here
                            const float2 old = *o;
                            vr += old.x;
                            vi += old.y;
                        }
                        *o = make_float2(vr, vi);
                    }
                }
            }
            __syncthreads();
            for (int e = tid; e < RC * plane / 2; e += 256) tiles4[e] = make_int4(0, 0, 0, 0);
            __syncthreads();
        }
        first = false;
        // points beyond the batch to the list's front
        const int rest = have - n;
        const int moved = tid < rest ? s_list[n + tid] : 0;
        __syncthreads();
        if (tid < rest) s_list[tid] = moved;
        if (tid == 0) s_cnt = rest;
        have = rest;
        __syncthreads();
    }
}

}  // namespace mi355
