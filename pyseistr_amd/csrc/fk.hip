// FK dip filter: sh_fkdip replaces the pure-Python fkdip (pyseistr/fk.py:2-68),
// the step after somf2dc in the reference's DAS demo.  The data are padded
// to powers of two (nf samples, nk traces); a real FFT along time keeps the
// nf/2 + 1 non-negative frequencies, a complex FFT along space follows, and
// a cone around zero wavenumber is kept: frequency row i1 (1-based) and
// fftshift-ed wavenumber column i2 pass when i1 > (nn1/nw)*(i2 - nk/2) and
// i1 > (nn1/nw)*(nk/2 - i2), with nn1 = nf/2 + 1 and nw = w*nk, evaluated
// in double as the reference does (fk.py:51-55).  The inverse transforms
// undo both FFTs; the reference's explicit Hermitian extension followed by
// a complex inverse FFT and the real part (fk.py:57-65) is a complex-to-real
// inverse transform, which is what runs here.  Up to 16384 samples and 4096
// traces (after padding; from 128 and 64) three kernels do it all: real
// transforms of the traces, space transforms with the cone in between, real
// inverse transforms.  Other sizes run as library FFTs (hipFFT, float64)
// with kernels for the staging, the cone and the crop.  Agreement with the
// reference is to float64 rounding.
#include "common.hpp"

#include <hipfft/hipfft.h>

#include <algorithm>

#include <cstdlib>

namespace {

struct FkPlans {
    int n1 = 0, n2 = 0, two_d = 0;
    hipfftHandle t_fwd = nullptr, x = nullptr, t_inv = nullptr;  // time R2C, space C2C, time C2R
    hipfftHandle f2 = nullptr, i2 = nullptr;                     // both axes at once: R2C, C2R
    ~FkPlans() {
        for (hipfftHandle h : {t_fwd, x, t_inv, f2, i2})
            if (h) hipfftDestroy(h);
    }
};

int pow2_at_least(int n) {
    int p = 1;
    while (p < n) p *= 2;
    return p;
}

// R[c][i] (nf per trace, nc traces) = in[c][i] for i < n1 and c < n2, zero
// beyond
__global__ void fk_stage(const double *__restrict__ in, double *__restrict__ R, int n1, int nf, int n2, int nc) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)nf * nc) return;
    const int i = (int)(k % nf), c = (int)(k / nf);
    R[k] = i < n1 && c < n2 ? in[(long)c * n1 + i] : 0.0;
}

// n1 == 1: the length-1 time transform is the identity, so the spectrum
// columns take the samples directly
__global__ void fk_stage1(const double *__restrict__ in, double2 *__restrict__ C, int n2, int nk) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nk) return;
    C[c] = make_double2(c < n2 ? in[c] : 0.0, 0.0);
}

// zero the padded traces n2 .. nk-1 of the spectrum (nh rows per trace)
__global__ void fk_zero(double2 *__restrict__ C, int nh, int n2, int nk) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)nh * (nk - n2)) return;
    C[(long)n2 * nh + k] = make_double2(0.0, 0.0);
}

// whether frequency f, column col of the unshifted spectrum (at fftshift-ed
// position (col + nk/2) mod nk) is in the cone
__device__ inline bool in_cone(int f, int col, int nk, double slope) {
    const int nk2 = nk / 2, i1 = f + 1, i2 = (col + nk2) % nk + 1;
    return (double)i1 > slope * (double)(i2 - nk2) && (double)i1 > slope * (double)(nk2 - i2);
}

// keep the cone
__global__ void fk_cone(double2 *__restrict__ C, int nh, int nk, double slope) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)nh * nk) return;
    const int f = (int)(k % nh), col = (int)(k / nh);
    if (!in_cone(f, col, nk, slope)) C[k] = make_double2(0.0, 0.0);
}

// out[c][i] = R[c][i] * scale for i < n1 (R holds nf samples per trace)
__global__ void fk_crop(const double *__restrict__ R, double *__restrict__ out, int n1, int nf, int n2, double scale) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)n1 * n2) return;
    const int i = (int)(k % n1), c = (int)(k / n1);
    out[k] = R[(long)c * nf + i] * scale;
}

__global__ void fk_crop1(const double2 *__restrict__ C, double *__restrict__ out, int n2, double scale) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n2) return;
    out[c] = C[c].x * scale;
}

#include "fft64.hpp"

// ---------------------------------------------------------------------------
// The filter in three kernels.  The spectrum lies as [f / 8][trace][f % 8]
// (128-byte pieces, whole lines for both its writer and its reader), for the
// traces that exist alone: their padding is zeros on the way in and is not
// wanted on the way out, so neither is stored or transformed along time.
// Memory is the bound: the section and its half spectrum each four times
// less padding, 0.9 GB for 6000 x 2500; the library's two 2-D transforms
// with the staging, cone and crop kernels moved the padded arrays (0.27 GB
// each) fourteen times.  6000 x 2500 (8192 x 4096 padded): 1116 us before,
// now 86 (rows), 150 (space) and 70 (rows back), where the copy's rate takes
// 60, 70 and 60.  Error against long double, root mean square, over 129 x 33
// to 6000 x 200: 2.2e-16 to 3.7e-16 (the library's transforms: 4.0e-16 to
// 5.7e-16).
// ---------------------------------------------------------------------------
__device__ inline long spec_at(int f, long c, long n2) { return ((f >> 3) * n2 + c) * 8 + (f & 7); }

typedef double dpair __attribute__((ext_vector_type(2), aligned(8)));  // two samples of a trace of any length

template <int L>
struct RowCfg {
    static constexpr int N = 1 << L, T = N / 16;           // complex points, threads of a transform
    static constexpr int NB = T >= 256 ? T : 256, NT = NB / T;  // threads and traces of a block
};

// N + 1 frequencies of each trace of 2 N samples, from the transform of its
// even and odd samples as one complex sequence
template <int L>
__global__ void __launch_bounds__(RowCfg<L>::NB)
fk_rows(const double *__restrict__ in, double2 *__restrict__ C, const double2 *__restrict__ tw,
        const double2 *__restrict__ half, int n1, int n2) {
    using R = RowCfg<L>;
    constexpr int N = R::N, T = R::T;
    __shared__ double shm[R::NT * N];
    const int t = threadIdx.x % T, x = (threadIdx.x / T * T) & 31;
    double *sh = shm + threadIdx.x / T * N;
    const long tr = (long)blockIdx.x * R::NT + threadIdx.x / T, c = min(tr, (long)n2 - 1);
    const double *src = in + c * n1;
    double2 v[16];
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const int i = 2 * (t + m * T);
        if (i + 1 < n1) {
            const dpair p = *reinterpret_cast<const dpair *>(src + i);
            v[m] = make_double2(p.x, p.y);
        } else {
            v[m] = make_double2(i < n1 ? src[i] : 0.0, 0.0);
        }
    }
    fft_passes<L, false, 1>(v, sh, x, t, tw);
    // Z(N - k) of each of the thread's k
    double2 z[16];
    fft_mirror<L>(v, z, sh, x, t);
    if (tr >= n2) return;
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const int k = t + m * T;
        const double2 w = half[k];
        const double2 e = make_double2(0.5 * (v[m].x + z[m].x), 0.5 * (v[m].y - z[m].y));
        const double2 o = make_double2(0.5 * (v[m].y + z[m].y), 0.5 * (z[m].x - v[m].x));
        double2 X = cmul(o, w);
        X.x += e.x;
        X.y += e.y;
        if (k == 0) {
            X = make_double2(v[m].x + v[m].y, 0.0);
            C[spec_at(N, c, n2)] = make_double2(v[m].x - v[m].y, 0.0);
        }
        C[spec_at(k, c, n2)] = X;
    }
}

// the inverse of fk_rows, scaled; the imaginary parts of the first and last
// frequency are not used
template <int L>
__global__ void __launch_bounds__(RowCfg<L>::NB)
fk_rows_inv(const double2 *__restrict__ C, double *__restrict__ out, const double2 *__restrict__ tw,
            const double2 *__restrict__ half, int n1, int n2, double scale) {
    using R = RowCfg<L>;
    constexpr int N = R::N, T = R::T;
    __shared__ double shm[R::NT * N];
    const int t = threadIdx.x % T, x = (threadIdx.x / T * T) & 31;
    double *sh = shm + threadIdx.x / T * N;
    const long tr = (long)blockIdx.x * R::NT + threadIdx.x / T, c = min(tr, (long)n2 - 1);
    double2 v[16], z[16];
#pragma unroll
    for (int m = 0; m < 16; m++) v[m] = C[spec_at(t + m * T, c, n2)];
    fft_mirror<L>(v, z, sh, x, t);
    if (t == 0) {
        v[0].y = 0.0;
        z[0] = make_double2(C[spec_at(N, c, n2)].x, 0.0);
    }
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const double2 w = half[t + m * T];
        const double2 e = make_double2(v[m].x + z[m].x, v[m].y - z[m].y);
        const double2 d = make_double2(v[m].x - z[m].x, v[m].y + z[m].y);
        const double2 o = cmul(d, make_double2(w.x, -w.y));
        v[m] = make_double2(e.x - o.y, e.y + o.x);
    }
    fft_passes<L, true, 1>(v, sh, x, t, tw);
    if (tr >= n2) return;
    double *dst = out + c * n1;
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const int i = 2 * (t + m * T);
        if (i + 1 < n1) {
            dpair p;
            p.x = v[m].x * scale;
            p.y = v[m].y * scale;
            *reinterpret_cast<dpair *>(dst + i) = p;
        } else if (i < n1) {
            dst[i] = v[m].x * scale;
        }
    }
}

// The space transform of COLS frequencies, the cone, and back.  512 threads in
// 64 KB of LDS and 128 registers, so that two blocks share a CU and one loads
// while the other computes (one block with 227 registers: 180 us, two: 150,
// a few spills included).  Blocks whose
// frequencies share 128-byte pieces follow each other on one XCD (blocks are
// dealt to the eight in turn), so that its L2 holds the piece for them.
constexpr int COL_NB = 512;
template <int L>
__global__ void __launch_bounds__(COL_NB, 4)
fk_cols(double2 *__restrict__ C, const double2 *__restrict__ tw, int nh, int n2, double slope) {
    constexpr int N = 1 << L, T = N / 16, COLS = COL_NB / T, SHARE = COLS < 8 ? 8 / COLS : 1;
    __shared__ double shm[COLS * N];
    const int s = blockIdx.x / 8, blk = (s / SHARE * 8 + blockIdx.x % 8) * SHARE + s % SHARE;
    if (blk * COLS >= nh) return;
    const int t = threadIdx.x / COLS, f = blk * COLS + threadIdx.x % COLS, fc = min(f, nh - 1);
    const int x = (threadIdx.x % COLS * (COLS < 64 ? 64 / COLS : 1)) & 31;
    double *sh = shm + threadIdx.x % COLS * N;
    double2 v[16];
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const int c = t + m * T;
        v[m] = c < n2 ? C[spec_at(fc, c, n2)] : make_double2(0.0, 0.0);
    }
    fft_passes<L, false, 1>(v, sh, x, t, tw);
#pragma unroll
    for (int m = 0; m < 16; m++)
        if (!in_cone(fc, t + m * T, N, slope)) v[m] = make_double2(0.0, 0.0);
    fft_passes<L, true, 1>(v, sh, x, t, tw);
    if (f >= nh) return;
    int tt = t;
    here(tt);  // the addresses are formed again, not kept
#pragma unroll
    for (int m = 0; m < 16; m++) {
        const int c = tt + m * T;
        if (c < n2) C[spec_at(f, c, n2)] = v[m];
    }
}

// Twiddle tables of both axes, laid out once per pair of lengths on the context.
struct FkTables {
    int l1 = 0, l2 = 0;
    double2 *rows = nullptr, *half = nullptr, *cols = nullptr;
    ~FkTables() {
        if (rows) (void)hipFree(rows);
    }
};

int fk_tables(sh_ctx *ctx, int l1, int l2, FkTables *&out) {
    auto *p = static_cast<FkTables *>(ctx->fk_tables.get());
    if (p && p->l1 == l1 && p->l2 == l2) {
        out = p;
        return SH_OK;
    }
    ctx->fk_tables.reset();
    auto *q = new (std::nothrow) FkTables();
    if (!q) return sh_fail(ctx, SH_EALLOC, "sh_fkdip: out of host memory");
    std::shared_ptr<void> own(q, [](void *x) { delete static_cast<FkTables *>(x); });
    const size_t a = 1u << l1, b = 1u << l2;
    SH_HIP(ctx, hipMalloc((void **)&q->rows, (2 * a + b) * sizeof(double2)));
    q->half = q->rows + a;
    q->cols = q->half + a;
    const int T = 256;
    hipLaunchKernelGGL(fft_twiddles, dim3(ceil_div(a, T)), dim3(T), 0, ctx->stream, q->rows, l1);
    hipLaunchKernelGGL(fft_half_turns, dim3(ceil_div(a, T)), dim3(T), 0, ctx->stream, q->half, l1);
    hipLaunchKernelGGL(fft_twiddles, dim3(ceil_div(b, T)), dim3(T), 0, ctx->stream, q->cols, l2);
    SH_TRY(sh_launch_check(ctx, "fft_twiddles"));
    SH_HIP(ctx, hipStreamSynchronize(ctx->stream));  // later calls may come on another stream
    q->l1 = l1;
    q->l2 = l2;
    ctx->fk_tables = own;
    out = q;
    return SH_OK;
}

constexpr int FK_L1_MIN = 6, FK_L1_MAX = 13, FK_L2_MIN = 6, FK_L2_MAX = 12;

int fk_fused(sh_ctx *ctx, const double *in, double *out, int n1, int n2, int l1, int l2, double slope, double scale) {
    FkTables *tb;
    SH_TRY(fk_tables(ctx, l1, l2, tb));
    const int N = 1 << l1, nh = N + 1, nk = 1 << l2;
    double2 *C = nullptr;
    SH_TRY(sh_slot(ctx, SLOT_FK0 + 1, sizeof(double2) * (size_t)ceil_div(nh, 8) * 8 * n2, (void **)&C));
    hipStream_t st = ctx->stream;
    const int per = std::max(1, 4096 / N);  // traces of a block (RowCfg)
    const int cols = COL_NB * 16 / nk, share = cols < 8 ? 8 / cols : 1;
    const dim3 rg((unsigned)ceil_div(n2, per)), cg((unsigned)(ceil_div(ceil_div(nh, cols), 8 * share) * 8 * share));
#define FK_L1(K, ...)                                                                                              \
    switch (l1) {                                                                                                  \
    case 6: hipLaunchKernelGGL(K<6>, rg, dim3(RowCfg<6>::NB), 0, st, __VA_ARGS__); break;                          \
    case 7: hipLaunchKernelGGL(K<7>, rg, dim3(RowCfg<7>::NB), 0, st, __VA_ARGS__); break;                          \
    case 8: hipLaunchKernelGGL(K<8>, rg, dim3(RowCfg<8>::NB), 0, st, __VA_ARGS__); break;                          \
    case 9: hipLaunchKernelGGL(K<9>, rg, dim3(RowCfg<9>::NB), 0, st, __VA_ARGS__); break;                          \
    case 10: hipLaunchKernelGGL(K<10>, rg, dim3(RowCfg<10>::NB), 0, st, __VA_ARGS__); break;                       \
    case 11: hipLaunchKernelGGL(K<11>, rg, dim3(RowCfg<11>::NB), 0, st, __VA_ARGS__); break;                       \
    case 12: hipLaunchKernelGGL(K<12>, rg, dim3(RowCfg<12>::NB), 0, st, __VA_ARGS__); break;                       \
    case 13: hipLaunchKernelGGL(K<13>, rg, dim3(RowCfg<13>::NB), 0, st, __VA_ARGS__); break;                       \
    default: return sh_fail(ctx, SH_EINVAL, "sh_fkdip: transform of 2^%d", l1);                                    \
    }
#define FK_L2(LL)                                                                                                  \
    case LL: hipLaunchKernelGGL(fk_cols<LL>, cg, dim3(COL_NB), 0, st, C, tb->cols, nh, n2, slope); break;
    FK_L1(fk_rows, in, C, tb->rows, tb->half, n1, n2)
    SH_TRY(sh_launch_check(ctx, "fk_rows"));
    switch (l2) {
        FK_L2(6) FK_L2(7) FK_L2(8) FK_L2(9) FK_L2(10) FK_L2(11) FK_L2(12)
    default: return sh_fail(ctx, SH_EINVAL, "sh_fkdip: transform of 2^%d", l2);
    }
    SH_TRY(sh_launch_check(ctx, "fk_cols"));
    FK_L1(fk_rows_inv, C, out, tb->rows, tb->half, n1, n2, scale)
#undef FK_L1
#undef FK_L2
    return sh_launch_check(ctx, "fk_rows_inv");
}

int log2_of(int p) {
    int l = 0;
    while ((1 << l) < p) l++;
    return l;
}

int fft_fail(sh_ctx *ctx, const char *what, hipfftResult r) {
    return sh_fail(ctx, SH_EHIP, "sh_fkdip: %s failed (hipfftResult %d)", what, (int)r);
}

#define FK_FFT(ctx, what, call)                                \
    do {                                                       \
        hipfftResult r_ = (call);                              \
        if (r_ != HIPFFT_SUCCESS) return fft_fail(ctx, what, r_); \
    } while (0)

// plans for (n1, n2), cached on the context
int fk_plans(sh_ctx *ctx, int n1, int n2, FkPlans *&out) {
    auto *p = static_cast<FkPlans *>(ctx->fk.get());
    const int want_2d = pow2_at_least(n1) > 1 && pow2_at_least(n2) > 1 && !getenv("SH_FK_1D");
    if (p && p->n1 == n1 && p->n2 == n2 && p->two_d == want_2d) {
        out = p;
        return SH_OK;
    }
    ctx->fk.reset();
    auto *np_ = new (std::nothrow) FkPlans();
    if (!np_) return sh_fail(ctx, SH_EALLOC, "sh_fkdip: out of host memory");
    ctx->fk = std::shared_ptr<void>(np_, [](void *q) { delete static_cast<FkPlans *>(q); });
    const int nf = pow2_at_least(n1), nk = pow2_at_least(n2), nh = nf / 2 + 1;
    if (nf > 1 && nk > 1 && !getenv("SH_FK_1D")) {
        // the time transform of every padded trace followed by the space
        // transform of every frequency is the 2-D real transform of the
        // nk x nf array (time contiguous); the library then picks its own
        // column kernels for the space axis
        FK_FFT(ctx, "2-D plan", hipfftPlan2d(&np_->f2, nk, nf, HIPFFT_D2Z));
        FK_FFT(ctx, "2-D plan", hipfftPlan2d(&np_->i2, nk, nf, HIPFFT_Z2D));
        np_->two_d = 1;
        np_->n1 = n1;
        np_->n2 = n2;
        out = np_;
        return SH_OK;
    }
    if (nf > 1) {
        int n[1] = {nf}, re[1] = {nf}, ce[1] = {nh};
        FK_FFT(ctx, "time plan", hipfftPlanMany(&np_->t_fwd, 1, n, re, 1, nf, ce, 1, nh, HIPFFT_D2Z, n2));
        FK_FFT(ctx, "time plan", hipfftPlanMany(&np_->t_inv, 1, n, ce, 1, nh, re, 1, nf, HIPFFT_Z2D, n2));
    }
    if (nk > 1) {
        int n[1] = {nk}, e[1] = {nk};
        FK_FFT(ctx, "space plan", hipfftPlanMany(&np_->x, 1, n, e, nh, 1, e, nh, 1, HIPFFT_Z2Z, nh));
    }
    np_->n1 = n1;
    np_->n2 = n2;
    out = np_;
    return SH_OK;
}

}  // namespace

extern "C" int sh_fkdip(sh_ctx *ctx, const double *in, double *out, int n1, int n2, double w) {
    if (!ctx) return SH_ENULL;
    if (!in || !out) return sh_fail(ctx, SH_ENULL, "sh_fkdip: NULL pointer");
    if (n1 < 1 || n2 < 1 || n1 > (1 << 29) || n2 > (1 << 29))
        return sh_fail(ctx, SH_EINVAL, "sh_fkdip: bad shape %d x %d", n1, n2);
    const int nf = pow2_at_least(n1), nk = pow2_at_least(n2), nh = nf / 2 + 1;
    const double nw = w * nk;
    if (nw == 0.0) return sh_fail(ctx, SH_EINVAL, "sh_fkdip: w * nk is zero (the cone slope divides by it)");
    if ((long)nh * nk > (1L << 31) || (long)nf * nk > (1L << 31))
        return sh_fail(ctx, SH_EINVAL, "sh_fkdip: %d x %d spectrum exceeds one transform batch", nh, nk);
    const double slope = (double)nh / nw;
    const int l1 = log2_of(nf) - 1, l2 = log2_of(nk);  // complex points along time, points along space
    if (l1 >= FK_L1_MIN && l1 <= FK_L1_MAX && l2 >= FK_L2_MIN && l2 <= FK_L2_MAX && !getenv("SH_FK_1D"))
        return fk_fused(ctx, in, out, n1, n2, l1, l2, slope, 1.0 / ((double)nf * (double)nk));
    FkPlans *pl;
    SH_TRY(fk_plans(ctx, n1, n2, pl));
    void *rb = nullptr, *cb = nullptr;
    const int nc = pl->two_d ? nk : n2;  // traces held in the real buffer
    SH_TRY(sh_slot(ctx, SLOT_FK0, sizeof(double) * (size_t)nf * nc, &rb));
    SH_TRY(sh_slot(ctx, SLOT_FK0 + 1, sizeof(double2) * (size_t)nh * nk, &cb));
    double *R = (double *)rb;
    double2 *C = (double2 *)cb;
    hipStream_t st = ctx->stream;
    for (hipfftHandle h : {pl->t_fwd, pl->x, pl->t_inv, pl->f2, pl->i2})
        if (h) FK_FFT(ctx, "set stream", hipfftSetStream(h, st));
    const int T = 256;
    const double scale = 1.0 / ((double)nf * (double)nk);
    if (pl->two_d) {
        hipLaunchKernelGGL(fk_stage, dim3(ceil_div((long)nf * nk, T)), dim3(T), 0, st, in, R, n1, nf, n2, nk);
        SH_TRY(sh_launch_check(ctx, "fk_stage"));
        FK_FFT(ctx, "2-D transform", hipfftExecD2Z(pl->f2, R, (hipfftDoubleComplex *)C));
        hipLaunchKernelGGL(fk_cone, dim3(ceil_div((long)nh * nk, T)), dim3(T), 0, st, C, nh, nk, slope);
        SH_TRY(sh_launch_check(ctx, "fk_cone"));
        FK_FFT(ctx, "2-D transform", hipfftExecZ2D(pl->i2, (hipfftDoubleComplex *)C, R));
        hipLaunchKernelGGL(fk_crop, dim3(ceil_div((long)n1 * n2, T)), dim3(T), 0, st, R, out, n1, nf, n2, scale);
        return sh_launch_check(ctx, "fk_crop");
    }
    if (nf > 1) {
        hipLaunchKernelGGL(fk_stage, dim3(ceil_div((long)nf * n2, T)), dim3(T), 0, st, in, R, n1, nf, n2, n2);
        SH_TRY(sh_launch_check(ctx, "fk_stage"));
        if (nk > n2) {
            hipLaunchKernelGGL(fk_zero, dim3(ceil_div((long)nh * (nk - n2), T)), dim3(T), 0, st, C, nh, n2, nk);
            SH_TRY(sh_launch_check(ctx, "fk_zero"));
        }
        FK_FFT(ctx, "time transform", hipfftExecD2Z(pl->t_fwd, R, (hipfftDoubleComplex *)C));
    } else {
        hipLaunchKernelGGL(fk_stage1, dim3(ceil_div(nk, T)), dim3(T), 0, st, in, C, n2, nk);
        SH_TRY(sh_launch_check(ctx, "fk_stage1"));
    }
    if (nk > 1)
        FK_FFT(ctx, "space transform",
               hipfftExecZ2Z(pl->x, (hipfftDoubleComplex *)C, (hipfftDoubleComplex *)C, HIPFFT_FORWARD));
    hipLaunchKernelGGL(fk_cone, dim3(ceil_div((long)nh * nk, T)), dim3(T), 0, st, C, nh, nk, slope);
    SH_TRY(sh_launch_check(ctx, "fk_cone"));
    if (nk > 1)
        FK_FFT(ctx, "space transform",
               hipfftExecZ2Z(pl->x, (hipfftDoubleComplex *)C, (hipfftDoubleComplex *)C, HIPFFT_BACKWARD));
    if (nf > 1) {
        FK_FFT(ctx, "time transform", hipfftExecZ2D(pl->t_inv, (hipfftDoubleComplex *)C, R));
        hipLaunchKernelGGL(fk_crop, dim3(ceil_div((long)n1 * n2, T)), dim3(T), 0, st, R, out, n1, nf, n2, scale);
        return sh_launch_check(ctx, "fk_crop");
    }
    hipLaunchKernelGGL(fk_crop1, dim3(ceil_div(n2, T)), dim3(T), 0, st, C, out, n2, scale);
    return sh_launch_check(ctx, "fk_crop1");
}
