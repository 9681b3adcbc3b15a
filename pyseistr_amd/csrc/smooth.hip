// Stand-alone triangle and box smoothing of a volume's axes (smoothcf), the
// step before the slope estimate; the smoothing inside the estimate's CG is
// in dip.hip.
#include "dipcore.hpp"

#include <algorithm>
#include <cstdlib>

namespace {

using dipcore::fold_idx;

constexpr int TB = 256;

// ---------------------------------------------------------------------------
// Stand-alone smoothing (smoothcf, dip_cfuns.c:2006-2123): every line along
// axis `ax` smoothed `repeat` times by ps_smooth (adj: fold -> doubint ->
// triple) or ps_smooth2 (triple2 -> doubint2 -> fold2), with the box and
// derivative options (dip_cfuns.c:403-625).  One thread per line runs the
// reference's loops in its order of float (and, in triple, double)
// operations, so the result is bit-identical to the reference.  The line's
// work array is tmp[e * nl + line] (consecutive lines, consecutive words).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
smoothc_lines(float *__restrict__ x, float *__restrict__ tmp, int n1, int n2, int n3, int ax, int nb, int box,
              int der, int adj, int repeat) {
    const long n12 = (long)n1 * n2;
    const long nl = ax == 0 ? n12 / n1 * n3 : (ax == 1 ? (long)n1 * n3 : n12);
    const long line = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (line >= nl) return;
    long o, d;
    int nx;
    if (ax == 0) { o = line * n1; d = 1; nx = n1; }
    else if (ax == 1) { o = line % n1 + line / n1 * n12; d = n1; nx = n2; }
    else { o = line; d = n12; nx = n3; }
    const int np = nx + 2 * nb;
    const float wt = box ? (float)(1.0 / (2 * nb - 1)) : (float)(1.0 / (nb * nb));
    const bool one = box || der;
    float *t = tmp + line;
    auto T = [&](int e) -> float & { return t[(long)e * nl]; };
    for (int r = 0; r < repeat; r++) {
        if (adj) {
            for (int e = 0; e < np; e++) T(e) = x[o + (long)fold_idx(e - nb, nx) * d];  // fold
            float s = 0.0f;                                                          // doubint
            for (int i = np - 1; i >= 0; i--) { s += T(i); T(i) = s; }
            if (!one) {
                s = 0.0f;
                for (int i = 0; i < np; i++) { s += T(i); T(i) = s; }
            }
            for (int i = 0; i < nx; i++) {                                           // triple
                if (box) x[o + i * d] = (T(i + 1) - T(i + 2 * nb)) * wt;
                else x[o + i * d] = (float)((2. * T(i + nb) - T(i) - T(i + 2 * nb)) * wt);
            }
        } else {
            for (int e = 0; e < np; e++) T(e) = 0.0f;                                // triple2
            if (box) {
                const float mw = -wt;
                for (int i = 0; i < nx; i++) T(i + 1) += wt * x[o + i * d];
                for (int i = 0; i < nx; i++) T(i + 2 * nb) += mw * x[o + i * d];
            } else {
                const float mw = -wt, w2 = (float)(2. * wt);
                for (int i = 0; i < nx; i++) T(i) += mw * x[o + i * d];
                for (int i = 0; i < nx; i++) T(i + nb) += w2 * x[o + i * d];
                for (int i = 0; i < nx; i++) T(i + 2 * nb) += mw * x[o + i * d];
            }
            float s = 0.0f;                                                          // doubint2
            for (int i = 0; i < np; i++) { s += T(i); T(i) = s; }
            if (!one) {
                s = 0.0f;
                for (int i = np - 1; i >= 0; i--) { s += T(i); T(i) = s; }
            }
            for (int i = 0; i < nx; i++) x[o + i * d] = T(i + nb);                   // fold2
            for (int e = nb + nx; e < np; e++) x[o + (long)fold_idx(e - nb, nx) * d] += T(e);
            for (int e = nb - 1; e >= 0; e--) x[o + (long)fold_idx(e - nb, nx) * d] += T(e);
        }
    }
}

// smoothcf with adj != 0 (ps_smooth) in two sweeps per line: the fold
// feeds the backward running sum directly (its sums are stored once in the
// work plane, [sample][line]), and the forward sweep runs the second
// running sum and forms each output from a ring of the last 2*nb integrated
// values in LDS.  Every float operation of fold / doubint / triple happens
// in the reference's order, so results are bit-identical to smoothc_lines;
// the work plane is written and read once instead of five times.
__global__ void __launch_bounds__(64)
smoothc_sweep(float *__restrict__ x, float *__restrict__ tmp, int n1, int n2, int n3, int ax, int nb, int box,
              int der, int repeat) {
    extern __shared__ float ring[];  // [2 * nb][64]
    const long n12 = (long)n1 * n2;
    const long nl = ax == 0 ? n12 / n1 * n3 : (ax == 1 ? (long)n1 * n3 : n12);
    const long line = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (line >= nl) return;
    long o, d;
    int nx;
    if (ax == 0) { o = line * n1; d = 1; nx = n1; }
    else if (ax == 1) { o = line % n1 + line / n1 * n12; d = n1; nx = n2; }
    else { o = line; d = n12; nx = n3; }
    const int np = nx + 2 * nb, R = 2 * nb;
    const float wt = box ? (float)(1.0 / (2 * nb - 1)) : (float)(1.0 / (nb * nb));
    const bool one = box || der;
    float *t = tmp + line;
    float *rg = ring + threadIdx.x;
    for (int r = 0; r < repeat; r++) {
        float s = 0.0f;
        for (int e = np - 1; e >= 0; e--) {
            s += x[o + (long)fold_idx(e - nb, nx) * d];
            t[(long)e * nl] = s;
        }
        float s2 = 0.0f;
        int slot = 0;  // e % R
        for (int e = 0; e < np; e++) {
            float v = t[(long)e * nl];
            if (!one) {
                s2 += v;
                v = s2;
            }
            if (e >= R) {  // output i = e - 2 nb; the ring holds T(i) .. T(i + 2 nb - 1)
                const long oi = o + (long)(e - R) * d;
                if (box) {
                    const int s1 = slot + 1 == R ? 0 : slot + 1;
                    x[oi] = (rg[s1 * 64] - v) * wt;
                } else {
                    const int sm = slot + nb >= R ? slot + nb - R : slot + nb;
                    x[oi] = (float)((2. * rg[sm * 64] - rg[slot * 64] - v) * wt);
                }
            }
            rg[slot * 64] = v;
            slot = slot + 1 == R ? 0 : slot + 1;
        }
    }
}

// The same operations with L lines of a block resident in LDS (T[e][line],
// the pitch L + 1 keeps rows and columns free of bank conflicts): all
// threads load and fold, the two running sums alone run one lane per line,
// and all threads form the outputs.  One read and one write of the volume,
// no work plane.  500 x 250 x 150, radius 5: 216 us an axis before (its few
// hundred waves waited for one load a step), now 79, 62 and 51, of which the
// sums, which one wave of a block issues, take 34, 16 and 11 and the memory
// the rest (32 us at a copy's rate).  As wide rows as three blocks a CU
// allow, 16, 32 and 64 lines here; half of that measured 79, 100 and 57.
//
// One running sum of a line in LDS, forward or backward, in batches whose
// loads go ahead of the chain of additions.
template <int P, bool BACK>
__device__ inline void running_sum(float *t, int np) {
    constexpr int U = 16, STEP = BACK ? -P : P;
    float *p = t + (BACK ? (np - 1) * P : 0);
    float s = 0.0f, a[U], b[U];
    const int m = np / U;
    auto fetch = [&](float *v, const float *q) {
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = q[u * STEP];
    };
    auto add = [&](float *v, float *q) {
#pragma unroll
        for (int u = 0; u < U; u++) q[u * STEP] = s += v[u];
    };
    if (m) fetch(a, p);
    int i = 0;
    for (; i + 2 < m; i += 2, p += 2 * U * STEP) {
        fetch(b, p + U * STEP);
        add(a, p);
        fetch(a, p + 2 * U * STEP);
        add(b, p + U * STEP);
    }
    for (; i < m; i++, p += U * STEP) {
        if (i + 1 < m) fetch(b, p + U * STEP);
        add(a, p);
#pragma unroll
        for (int u = 0; u < U; u++) a[u] = b[u];
    }
    for (int e = m * U; e < np; e++, p += STEP) *p = s += *p;
}

template <int L>
__global__ void __launch_bounds__(TB)
smoothc_resident(const float *in, float *out, int n1, int n2, int n3, int ax, int nb, int box, int der, int adj,
                 int repeat) {
    extern __shared__ float T[];  // [np][P]
    constexpr int P = L + 1;
    const long n12 = (long)n1 * n2;
    const long nl = ax == 0 ? (long)n2 * n3 : (ax == 1 ? (long)n1 * n3 : n12);
    const long l0 = (long)blockIdx.x * L;
    const int live = (int)min((long)L, nl - l0), tid = threadIdx.x;
    const int nx = ax == 0 ? n1 : (ax == 1 ? n2 : n3), np = nx + 2 * nb;
    const long d = ax == 0 ? 1 : (ax == 1 ? n1 : n12);
    const float wt = box ? (float)(1.0 / (2 * nb - 1)) : (float)(1.0 / (nb * nb));
    const bool one = box || der;
    // f(line, e, address of sample e) for every e < ne of every line, along
    // the lines where they are contiguous, else across them
    auto each = [&](int ne, auto f) {
        if (ax == 0) {
            for (int l = tid / 64; l < live; l += TB / 64) {
                const long o = (l0 + l) * n1;
#pragma unroll 4
                for (int e = tid % 64; e < ne; e += 64) f(l, e, o + e);
            }
        } else {
            const int l = tid % L;
            if (l >= live) return;
            const long line = l0 + l, o = ax == 1 ? line % n1 + line / n1 * n12 : line;
#pragma unroll 8
            for (int e = tid / L; e < ne; e += TB / L) f(l, e, o + e * d);
        }
    };
    for (int r = 0; r < repeat; r++) {
        const float *x = r ? out : in;
        if (adj) {
            each(nx, [&](int l, int e, long i) { T[(nb + e) * P + l] = x[i]; });  // fold
            __syncthreads();
            for (int q = tid; q < 2 * nb * L; q += TB) {
                const int l = q % L, j = q / L, e = j < nb ? j : nx + j;
                if (l < live) T[e * P + l] = T[(nb + fold_idx(e - nb, nx)) * P + l];
            }
            __syncthreads();
            if (tid < live) {  // doubint
                running_sum<P, true>(T + tid, np);
                if (!one) running_sum<P, false>(T + tid, np);
            }
            __syncthreads();
            each(nx, [&](int l, int e, long i) {  // triple
                const float *t = T + e * P + l;
                if (box) out[i] = (t[P] - t[2 * nb * P]) * wt;
                else out[i] = (float)((2. * t[nb * P] - t[0] - t[2 * nb * P]) * wt);
            });
        } else {
            const float mw = -wt, w2 = (float)(2. * wt);
            each(np, [&](int l, int e, long i) {  // triple2: the terms of the three passes over T(e), in their order
                float v = 0.0f;
                const int e0 = box ? 1 : 0, e1 = box ? 2 * nb : nb, e2 = 2 * nb;
                const bool b0 = e >= e0 && e - e0 < nx, b1 = e >= e1 && e - e1 < nx, b2 = !box && e >= e2;
                const long o = i - e * d;  // the loads are unconditional, so that they go out together
                const float t0 = (box ? wt : mw) * x[b0 ? i - e0 * d : o], t1 = (box ? mw : w2) * x[b1 ? i - e1 * d : o],
                            t2 = mw * x[b2 ? i - e2 * d : o];
                v = b0 ? v + t0 : v;
                v = b1 ? v + t1 : v;
                v = b2 ? v + t2 : v;
                T[e * P + l] = v;
            });
            __syncthreads();
            if (tid < live) {  // doubint2
                running_sum<P, false>(T + tid, np);
                if (!one) running_sum<P, true>(T + tid, np);
            }
            __syncthreads();
            each(nx, [&](int l, int e, long i) {  // fold2 (nb <= nx: one sample of each overhang at most)
                const float *t = T + l;
                float v = t[(e + nb) * P];
                if (e >= nx - nb) v += t[(nb + 2 * nx - 1 - e) * P];
                if (e < nb) v += t[(nb - 1 - e) * P];
                out[i] = v;
            });
        }
        __syncthreads();
    }
}

// Lines a block holds, 0 if they do not fit (the kernels above take long
// lines, and radii beyond the axis in the adj = 0 form, whose overhangs then
// fold more than once).  At least four lines; three blocks a CU where 32 lines
// or more fit so, two with fewer.
int resident_lines(int nx, int nb, bool adj) {
    if (nx > 1 << 16 || nb > 1 << 16 || (!adj && nb > nx)) return 0;
    const long np = nx + 2L * nb;
    for (int L : {64, 32, 16, 8, 4})
        if (np * (L + 1) * (long)sizeof(float) <= (L > 16 ? 48 : 64) * 1024) return L;
    return 0;
}

}  // namespace

// Replaces dipcfun.smoothcf (pyseistr/src/dip_cfuns.c:2006-2123), the C
// entry behind smoothc (pyseistr/smooth.py:115).
extern "C" int sh_smooth(sh_ctx *ctx, const float *in, float *out, int n1, int n2, int n3, int repeat, int adj,
                         int r1, int r2, int r3, int diff1, int diff2, int diff3, int box1, int box2, int box3) {
    if (!ctx) return SH_ENULL;
    if (!in || !out) return sh_fail(ctx, SH_ENULL, "sh_smooth: NULL pointer");
    if (n1 < 1 || n2 < 1 || n3 < 1) return sh_fail(ctx, SH_EINVAL, "sh_smooth: bad shape %d x %d x %d", n1, n2, n3);
    if (repeat < 0) return sh_fail(ctx, SH_EINVAL, "sh_smooth: repeat must be >= 0");
    const long n = (long)n1 * n2 * n3;
    const int nn[3] = {n1, n2, n3}, rect[3] = {r1, r2, r3}, diff[3] = {diff1, diff2, diff3}, box[3] = {box1, box2, box3};
    // SH_SMOOTHC_LINES=1: the one-pass-per-step kernel for adj != 0 as well
    const bool lines_only = getenv("SH_SMOOTHC_LINES") != nullptr;
    const float *src = in;  // the copy is left to the first pass that can read elsewhere than it writes
    for (int ax = 0; ax < 3; ax++) {
        if (rect[ax] <= 1 || repeat == 0) continue;
        const long nl = n / nn[ax];
        const int L = lines_only ? 0 : resident_lines(nn[ax], rect[ax], adj != 0);
        if (L) {
            const size_t lds = (size_t)(nn[ax] + 2 * rect[ax]) * (L + 1) * sizeof(float);
            const dim3 grid((unsigned)ceil_div(nl, L));
#define SM_(LL)                                                                                                   \
    case LL:                                                                                                      \
        hipLaunchKernelGGL(smoothc_resident<LL>, grid, dim3(TB), lds, ctx->stream, src, out, n1, n2, n3, ax,      \
                           rect[ax], box[ax] != 0, diff[ax] != 0, adj != 0, repeat);                              \
        break;
            switch (L) { SM_(64) SM_(32) SM_(16) SM_(8) SM_(4) }
#undef SM_
            SH_TRY(sh_launch_check(ctx, "smoothc_resident"));
            src = out;
            continue;
        }
        if (src != out) {
            SH_HIP(ctx, hipMemcpyAsync(out, in, (size_t)n * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
            src = out;
        }
        float *tmp = nullptr;
        SH_TRY(sh_slot(ctx, SLOT_DIP0 + 5, (size_t)(nn[ax] + 2L * rect[ax]) * nl * sizeof(float), (void **)&tmp));
        const size_t ring = (size_t)2 * rect[ax] * 64 * sizeof(float);
        if (adj && ring <= 32768 && !lines_only) {
            hipLaunchKernelGGL(smoothc_sweep, dim3((unsigned)ceil_div(nl, 64)), dim3(64), ring, ctx->stream, out, tmp, n1,
                               n2, n3, ax, rect[ax], box[ax] != 0, diff[ax] != 0, repeat);
            SH_TRY(sh_launch_check(ctx, "smoothc_sweep"));
            continue;
        }
        hipLaunchKernelGGL(smoothc_lines, dim3((unsigned)ceil_div(nl, 256)), dim3(256), 0, ctx->stream, out, tmp, n1, n2,
                           n3, ax, rect[ax], box[ax] != 0, diff[ax] != 0, adj != 0, repeat);
        SH_TRY(sh_launch_check(ctx, "smoothc_lines"));
    }
    if (src != out) SH_HIP(ctx, hipMemcpyAsync(out, in, (size_t)n * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    return SH_OK;
}
