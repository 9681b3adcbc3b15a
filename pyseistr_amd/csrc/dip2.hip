// Dip estimation of 2-D sections, dipc with n3 == 1 (pyseistr/src/
// dip_cfuns.c:1694-1989), with a section's state held in registers.
//
// As a sequence of launches a 512 x 256 section took 711 of them, 3-4 us
// each and more than half no-ops of solves that had converged.  Here one
// block per tile runs the whole Gauss-Newton loop: it keeps what belongs to
// its tile (and the model, residual and weights of the tile's halo, which it
// updates itself) in registers, smooths both axes in LDS, and exchanges only
// the smoothed gradient and the conjugate directions with its neighbours.
// The float operations on a sample and their order are those of the launches
// (dip.hip), so the dips are the same; only the double sums are added in
// another order.  512 x 256, 5 x 20 iterations: 2800 -> 920 us (the kernel 775 in
// another run); 128 x 64: the kernel 390 us of about 2000 before.  What bounds
// it: dependent phases, each a round trip of the exchange, a barrier and the
// two stencils: two a CG iteration and two or three a Gauss-Newton step, 217 at
// most.  (A batch of sections
// as teams of blocks in one launch ran no faster than its launches: with the
// chip full both are bound by the work in the tiles.)
//
// Exchange goes through memory with agent-scope atomic loads and stores
// (they bypass the XCDs' L2s, which are not coherent with each other),
// ordered by the barrier: every wave waits for its own stores, then the block
// publishes its partial sums, each half of a double next to the barrier's
// number in one 8-byte store, and a wave of every block polls until all words
// carry that number.  A barrier takes 1.1 us with 8 blocks, 1.8 us with 128
// (with fences, which write back and invalidate a whole L2, 2.7 and 16 us).
// Every block adds up all sums in the same order and keeps its own copy of
// the scalar record, so all take the same decisions.  The launch is
// cooperative, so all blocks are on the chip at once; the wait is bounded all
// the same, and a block that gives up fills its dips with NaN and sets the
// context's flag, which the next call that synchronises (or the next
// estimate) turns into an error.
#include "dip2.hpp"

#include <algorithm>
#include <cstdlib>

namespace {

using namespace dipcore;

constexpr int TBR = 512;            // threads of a block
constexpr int LS_SUMS = 7;          // sums of the seven halved steps
constexpr int WAIT_MAX = 1 << 24;   // polls before a block gives up
constexpr size_t LDS_MAX = 60 * 1024;

struct Resident {
    int n1, n2, r1, r2, niter, liter;
    const float *x, *init;
    const unsigned char *mask;
    float *ex;                  // three exchanged fields of n1 * n2 samples
    unsigned long long *words;  // [2][blocks][2 * LS_SUMS]
    float *dip;
    int *rec;
    int polls;    // before a block gives up
    int *failed;  // set then (host memory)
};

// Element i of a section's field.  The index is hidden from the optimiser
// where it is used, so that it forms the address from the uniform base and a
// 32-bit offset there instead of keeping a 64-bit pointer for every element
// and field in registers over the whole solve (which spilled 150 of them).
__device__ inline size_t here(int i) {
    unsigned o = (unsigned)i * 4u;
    asm volatile("" : "+v"(o));
    return o;
}
__device__ inline void ex_put(float *f, int i, float v) {
    __hip_atomic_store(reinterpret_cast<float *>(reinterpret_cast<char *>(f) + here(i)), v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float ex_get(const float *f, int i) {
    return __hip_atomic_load(reinterpret_cast<const float *>(reinterpret_cast<const char *>(f) + here(i)),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Barrier with K sums: v[k] in, the totals out (tot, LDS).
// False: another block did not arrive.
template <int K>
__device__ inline bool meet(const Resident &R, unsigned epoch, double (&v)[K], double *sh, double *tot, int *ok) {
    block_sum_multi(v, sh);
    unsigned long long *const words = R.words + (size_t)(epoch & 1) * gridDim.x * (2 * LS_SUMS);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wave's stores have arrived
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < K; k++) {
            const unsigned long long b = (unsigned long long)__double_as_longlong(v[k]), tag = (unsigned long long)epoch << 32;
            unsigned long long *w = words + (size_t)blockIdx.x * (2 * LS_SUMS) + 2 * k;
            __hip_atomic_store(w, tag | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(w + 1, tag | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    if (threadIdx.x < 64) {
        double s[K] = {};
        bool all = false;
        for (int n = 0; n < R.polls && !all; n++) {
            bool here = true;
#pragma unroll
            for (int k = 0; k < K; k++) s[k] = 0.0;
            for (int b = threadIdx.x; b < (int)gridDim.x; b += 64) {
                const unsigned long long *w = words + (size_t)b * (2 * LS_SUMS);
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const unsigned long long lo = __hip_atomic_load(w + 2 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const unsigned long long hi =
                        __hip_atomic_load(w + 2 * k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    here = here && (unsigned)(lo >> 32) == epoch && (unsigned)(hi >> 32) == epoch;
                    s[k] += __longlong_as_double((long long)((hi << 32) | (lo & 0xffffffffull)));
                }
            }
            all = __all(here);
        }
#pragma unroll
        for (int k = 0; k < K; k++) s[k] = wave_sum(s[k]);
        if (threadIdx.x == 0) {
#pragma unroll
            for (int k = 0; k < K; k++) tot[k] = s[k];
            *ok = all;
        }
    }
    __syncthreads();
    return *ok != 0;
}

// LDS of a block: the tile with its halo, then the axis-1 result.  A row of
// the tile has one unused sample so that its pitch is odd: threads four
// samples apart and threads in neighbouring rows read different banks.
SH_HD inline int row_len(int t1, int r1) { return t1 + 2 * (r1 - 1) + 1; }
inline size_t res_lds(int t1, int t2, int r1, int r2) {
    return sizeof(float) * (t2 + 2 * ((size_t)r2 - 1)) * ((size_t)row_len(t1, r1) + t1);
}

// HE: elements of the tile with its halo a thread holds.
template <int NW, int T1, int T2, int HE>
__global__ void __launch_bounds__(TBR)
d2_resident(const Resident R) {
    extern __shared__ float lds[];
    __shared__ float w1[SM_HMAX + 1], w2[SM_HMAX + 1];
    __shared__ DipScal s;
    __shared__ double sh[16 * LS_SUMS], tot[LS_SUMS];
    __shared__ int ok;
    const int h1 = R.r1 - 1, h2 = R.r2 - 1, W1 = row_len(T1, R.r1), R2 = T2 + 2 * h2, ne = R2 * W1;
    float *const tile = lds, *const s1 = lds + R2 * W1;
    const int tid = threadIdx.x;
    for (int k = tid; k < R.r1; k += TBR) w1[k] = (float)((double)(R.r1 - k) / ((double)R.r1 * R.r1));
    for (int k = tid; k < R.r2; k += TBR) w2[k] = (float)((double)(R.r2 - k) / ((double)R.r2 * R.r2));
    const float pmax = 3.402823466e+38f, pmin = -3.402823466e+38f;
    // the four own samples of a thread, at (x0 + qk, y0 + qr .. + 3)
    const bool quad = tid < T2 / 4 * T1;
    const int qr = tid / T1 * 4, qk = tid % T1;
    // both smoothing axes of what the threads put into tile
    auto smooth = [&](float *o) {
        __syncthreads();
        for (int e = tid; e < R2 * (T1 / 4); e += TBR) {
            const int r = e / (T1 / 4), k = e % (T1 / 4) * 4;
            float q[4];
            tri4(tile + r * W1 + k + h1, 1, w1, h1, q);
#pragma unroll
            for (int j = 0; j < 4; j++) s1[r * T1 + k + j] = q[j];
        }
        __syncthreads();
        if (quad) tri4(s1 + (qr + h2) * T1 + qk, T1, w2, h2, o);
    };
    unsigned epoch = 0;
    bool fine = true;
    const int n1 = R.n1, n2 = R.n2, ntx = (n1 + T1 - 1) / T1;
    const int x0 = blockIdx.x % ntx * T1, y0 = blockIdx.x / ntx * T2;
    const long n = (long)n1 * n2;
    // exchanged fields: den, num of a solve's start, then the directions; the gradient
    float *const e0 = R.ex, *const e1 = R.ex + n, *const e2 = R.ex + 2 * n;
    if (tid == 0) s = DipScal{};
    int gi[HE];
#pragma unroll
    for (int j = 0; j < HE; j++) {
        const int e = tid + j * TBR, r = (int)((unsigned)e / (unsigned)W1), k = e - r * W1;
        gi[j] = e < ne ? fold_idx(x0 - h1 + k, n1) + n1 * fold_idx(y0 - h2 + r, n2) : 0;
    }
    auto held = [&](int j) { return tid + j * TBR < ne; };
    const int ix = x0 + qk, o0 = ix + n1 * (y0 + qr);
    const bool col = quad && ix < n1, in1 = ix >= NW && ix < n1 - NW;
    auto mine = [&](int j) { return col && y0 + qr + j < n2; };
    float p[4], u2[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        p[j] = R.init && mine(j) ? R.init[o0 + j * n1] : 0.0f;
        u2[j] = 0.0f;
    }
    // the stencil's sample j with taps a (pwd_sample)
    auto residual = [&](int j, const float *a) {
        float y = 0.0f;
        if (mine(j) && in1 && y0 + qr + j < n2 - 1) {
            const float *c = reinterpret_cast<const float *>(reinterpret_cast<const char *>(R.x) + here(o0 + j * n1));
#pragma unroll
            for (int iw = 0; iw <= 2 * NW; iw++) y += (c[iw - NW + n1] - c[NW - iw]) * a[iw];
        }
        return y;
    };
    // a step of the line search: slopes and residual of sample j
    auto trial = [&](int j, float dp, float lam, float &pv) {
        pv = p[j] + lam * dp;
        if (pv < pmin) pv = pmin;
        if (pv > pmax) pv = pmax;
        float a[2 * NW + 1];
        apf_pass<NW>(pv, a);
        return residual(j, a);
    };
    // one barrier with sums, then the scalar step
    auto step = [&](auto &v, int mode, int it) {
        fine = meet(R, ++epoch, v, sh, tot, &ok);
        if (tid == 0 && fine) dip_scalar_step(&s, tot, mode, it, n, 1.e-6f);
        __syncthreads();
    };
    {
        double v[1] = {0.0};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float a[2 * NW + 1];
            apf_pass<NW>(p[j], a);
            u2[j] = residual(j, a);
            v[0] += (double)u2[j] * u2[j];
        }
        if (fine) step(v, F_USUM, 0);
    }
    for (int it = 0; it < R.niter && fine; it++) {
        // derivative and the division's scaling (pwd_sample<NW, 1>)
        {
            double v[1] = {0.0};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (!mine(j)) continue;
                float a[2 * NW + 1];
                apf_der<NW>(p[j], a);
                float num = u2[j], den = residual(j, a);
                const int i = o0 + j * n1;
                if (R.mask && R.mask[i]) {
                    num = 0.0f;
                    den = 0.0f;
                }
                const double norm = 1.0 / hypot((double)den, 1.0);
                num = (float)(num * norm);
                den = (float)(den * norm);
                ex_put(e0, i, den);
                ex_put(e1, i, num);
                v[0] += (double)den * den;
            }
            step(v, F_DIVN, it);
            if (!fine) break;
        }
        // weights and residual of the tile and its halo (cg_start_sample); x = 0
        float w[HE], r[HE], x[HE], wq[4], xq[4], pq[4], gq[4], spq[4], sxq[4], srq[4];
        const bool zero = s.divn_zero != 0;
        const double nrm = zero ? 0.0 : s.divn_norm;
#pragma unroll
        for (int j = 0; j < HE; j++) {
            w[j] = held(j) && !zero ? (float)(ex_get(e0, gi[j]) * nrm) : 0.0f;
            r[j] = held(j) && !zero ? -(float)(ex_get(e1, gi[j]) * nrm) : 0.0f;
            x[j] = 0.0f;
        }
        double r0 = 0.0;  // the block's part of the residual's square sum
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool m = mine(j) && !zero;
            wq[j] = m ? (float)(ex_get(e0, o0 + j * n1) * nrm) : 0.0f;
            const float rv = m ? -(float)(ex_get(e1, o0 + j * n1) * nrm) : 0.0f;
            r0 += (double)rv * rv;
            xq[j] = pq[j] = gq[j] = spq[j] = sxq[j] = srq[j] = 0.0f;
        }
        for (int k = 0; k < R.liter && !s.cg_done; k++) {
            // gx = -x + w r after the pending update; gp = p + S gx
            const bool pend = s.pending != 0;
            const float a2 = pend ? (float)s.alpha2 : 0.0f;
#pragma unroll
            for (int j = 0; j < HE; j++)
                if (held(j)) {
                    if (pend) {
                        x[j] = x[j] + a2 * ex_get(e0, gi[j]);
                        r[j] = r[j] + a2 * ex_get(e1, gi[j]);
                    }
                    tile[tid + j * TBR] = (-x[j]) + r[j] * w[j];
                }
            float o[4];
            smooth(o);
            double v[2] = {0.0, r0};
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (mine(j)) {
                    if (pend) {
                        pq[j] = pq[j] + a2 * spq[j];
                        xq[j] = xq[j] + a2 * sxq[j];
                    }
                    gq[j] = pq[j] + o[j];
                    ex_put(e2, o0 + j * n1, gq[j]);
                    v[0] += (double)gq[j] * gq[j];
                }
            fine = meet(R, ++epoch, v, sh, tot, &ok);
            if (tid == 0 && fine) {
                if (k == 0) dip_scalar_step(&s, tot + 1, F_R0, it, n, 1.e-6f);  // zero residual: zero model
                dip_scalar_step(&s, tot, F_GN, k, n, 1.e-6f);
            }
            __syncthreads();
            if (!fine || s.cg_done) break;
            // gx = S gp, gr = w gx, the new directions
            const float a1 = (float)s.alpha;
#pragma unroll
            for (int j = 0; j < HE; j++)
                if (held(j)) tile[tid + j * TBR] = ex_get(e2, gi[j]);
            smooth(o);
            double v3[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (mine(j)) {
                    const float gr = o[j] * wq[j];
                    spq[j] = k == 0 ? gq[j] : gq[j] + a1 * spq[j];
                    sxq[j] = k == 0 ? o[j] : o[j] + a1 * sxq[j];
                    srq[j] = k == 0 ? gr : gr + a1 * srq[j];
                    ex_put(e0, o0 + j * n1, sxq[j]);
                    ex_put(e1, o0 + j * n1, srq[j]);
                    v3[0] += (double)srq[j] * srq[j];
                    v3[1] += (double)spq[j] * spq[j];
                    v3[2] += (double)sxq[j] * sxq[j];
                }
            step(v3, F_BETA, k);
            if (!fine) break;
        }
        if (!fine) break;
        // line search: the full step; if it is refused, all halved ones at once
        float pt[4], ut[4];
        {
            const bool pend = s.pending != 0;
            const float a2 = (float)s.alpha2;
            double v[1] = {0.0};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (pend) xq[j] = xq[j] + a2 * sxq[j];
                ut[j] = trial(j, xq[j], 1.0f, pt[j]);
                v[0] += (double)ut[j] * ut[j];
            }
            step(v, F_LS0, it);
            if (!fine) break;
        }
        if (!s.accepted) {
            double v[LS_SUMS];
            float lam = 0.5f;
#pragma unroll 1
            for (int k = 0; k < LS_SUMS; k++) {
                double t = 0.0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float pv;
                    const float y = trial(j, xq[j], lam, pv);
                    t += (double)y * y;
                }
#pragma unroll
                for (int q = 0; q < LS_SUMS; q++)
                    if (q == k) v[q] = t;
                lam *= 0.5f;
            }
            step(v, F_LS7, it);
            if (!fine) break;
            lam = ldexpf(1.0f, -(s.ls_k < 8 ? s.ls_k : 7));  // (none accepted: the last one is kept)
#pragma unroll
            for (int j = 0; j < 4; j++) ut[j] = trial(j, xq[j], lam, pt[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            p[j] = pt[j];
            u2[j] = ut[j];
        }
    }
    // the dips may be written over the data: all blocks have read theirs
    if (fine) {
        double v[1] = {0.0};
        fine = meet(R, ++epoch, v, sh, tot, &ok);
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (mine(j)) R.dip[o0 + j * n1] = fine ? p[j] : __builtin_nanf("");
    if (!fine && tid == 0) __hip_atomic_store(R.failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (R.rec && blockIdx.x == 0)
        for (int q = tid; q < 2 * min(R.niter, 64); q += TBR) R.rec[q] = s.rec[q];
}

__global__ void d2_zero(unsigned long long *words, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) words[i] = 0;
}

// The tiles on offer, smallest first.
constexpr int NT = 3;
constexpr int T_CFG[NT][2] = {{32, 16}, {32, 32}, {64, 32}};

template <int NW, int HE>
const void *res_kernel(int c) {
    return c == 0 ? (const void *)d2_resident<NW, 32, 16, HE>
                  : c == 1 ? (const void *)d2_resident<NW, 32, 32, HE> : (const void *)d2_resident<NW, 64, 32, HE>;
}

int tiles_of(int c, int n1, int n2) { return ceil_div(n1, T_CFG[c][0]) * ceil_div(n2, T_CFG[c][1]); }

// Elements a thread holds with tile c: 9, 16, or 0 if it does not fit.
int held_of(int c, int r1, int r2) {
    const long ne = (long)(T_CFG[c][1] + 2 * (r2 - 1)) * row_len(T_CFG[c][0], r1);
    if (res_lds(T_CFG[c][0], T_CFG[c][1], r1, r2) > LDS_MAX || ne > 16L * TBR) return 0;
    return ne <= 9L * TBR ? 9 : 16;
}

}  // namespace

int dip2_resident(sh_ctx *ctx, int n1, int n2, int r1, int r2, int order, const float *x, const unsigned char *mask,
                  const float *init, int niter, int liter, int *rec, float *dip, int *ran) {
    *ran = 0;
    const long n = (long)n1 * n2;
    if (n >= (1L << 30)) return SH_OK;  // (32-bit byte offsets)
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return SH_OK;
    int cus = 0;
    SH_HIP(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    // the smallest tile with at most a block on every second CU, else on
    // every CU (smaller tiles: shorter phases; more blocks: a longer barrier.
    // 512 x 256: 128 tiles of 32 x 32 835 us, 256 of 32 x 16 896 us, 64 of 64 x
    // 32 907 us)
    int c = -1;
    for (int most : {cus / 2, cus})
        for (int k = 0; k < NT && c < 0; k++)
            if (tiles_of(k, n1, n2) <= most && held_of(k, r1, r2)) c = k;
    if (c < 0) return SH_OK;
    const int nb = tiles_of(c, n1, n2), he = held_of(c, r1, r2);
    const void *fn = nullptr;
    SH_DISPATCH_NW6(ctx, order, NW, fn = he == 9 ? res_kernel<NW, 9>(c) : res_kernel<NW, 16>(c));
    if (!ctx->wait_failed) {
        const hipError_t e = hipHostMalloc((void **)&ctx->wait_failed, sizeof(int), hipHostMallocDefault);
        if (e != hipSuccess) {
            ctx->wait_failed = nullptr;
            return sh_fail(ctx, SH_EALLOC, "hipHostMalloc: %s", hipGetErrorString(e));
        }
        *ctx->wait_failed = 0;
    }
    // SH_DIP2_POLLS: fewer polls (0: give up at the first barrier)
    const char *pe = getenv("SH_DIP2_POLLS");
    const int polls = pe ? std::min(std::max(atoi(pe), 0), WAIT_MAX) : WAIT_MAX;
    Resident R{n1, n2, r1, r2, niter, liter, x, init, mask, nullptr, nullptr, dip, rec, polls, ctx->wait_failed};
    SH_TRY(sh_slot(ctx, SLOT_DIP0, (size_t)n * 3 * sizeof(float), (void **)&R.ex));
    const size_t nw = (size_t)2 * nb * 2 * LS_SUMS;
    SH_TRY(sh_slot(ctx, SLOT_RED, nw * sizeof(unsigned long long), (void **)&R.words));
    hipLaunchKernelGGL(d2_zero, dim3(1), dim3(1024), 0, ctx->stream, R.words, (int)nw);
    SH_TRY(sh_launch_check(ctx, "d2_zero"));
    void *args[] = {&R};
    PROF_A(ctx);
    const hipError_t e = hipLaunchCooperativeKernel(fn, dim3(nb), dim3(TBR), args,
                                                    (unsigned)res_lds(T_CFG[c][0], T_CFG[c][1], r1, r2), ctx->stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        // more blocks than this device holds at once, or none of the kind: the launches run
        if (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported) return SH_OK;
        return sh_fail(ctx, SH_EHIP, "launch of d2_resident failed: %s", hipGetErrorString(e));
    }
    // the three exchanged fields of an iteration, written and read, if every
    // solve takes all its iterations
    PROF_B(ctx, "d2_resident", 24.0 * (double)n * niter * liter);
    *ran = 1;
    return SH_OK;
}
