// Complex transforms of N = 2^L points in float64, N / 16 threads each:
// thread t holds points t + m N/16, m < 16, in registers, on the way in and
// out.  Stockham passes (self-sorting) of radix 16, the last one the
// remainder, which a thread runs as 16 / R butterflies; between passes the
// points change threads through LDS, real and imaginary parts in turn, so a
// transform needs N doubles of it.  Radix 16 halves the exchanges of radix 4
// and its 64 registers of points leave room for four waves a SIMD.
#pragma once
#include "common.hpp"

__device__ inline double2 cmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// a times -i (forward) or i
template <bool INV>
__device__ inline double2 cquarter(double2 a) {
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

template <bool INV>
__device__ inline void dft4(double2 &a, double2 &b, double2 &c, double2 &d) {
    const double2 s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = cquarter<INV>(csub(b, d));
    a = cadd(s0, s2);
    b = cadd(s1, s3);
    c = csub(s0, s2);
    d = csub(s1, s3);
}

// u[0..R) transformed in place, in natural order
template <int R, bool INV>
__device__ inline void dft(double2 *u) {
    constexpr double H = 0.70710678118654752440, C1 = 0.92387953251128675613, S1 = 0.38268343236508977173;
    auto w = [](double c, double s) { return make_double2(c, INV ? s : -s); };
    if constexpr (R == 2) {
        const double2 a = u[0];
        u[0] = cadd(a, u[1]);
        u[1] = csub(a, u[1]);
    } else if constexpr (R == 4) {
        dft4<INV>(u[0], u[1], u[2], u[3]);
    } else if constexpr (R == 8) {
        dft4<INV>(u[0], u[2], u[4], u[6]);
        dft4<INV>(u[1], u[3], u[5], u[7]);
        const double2 o0 = u[1], o1 = cmul(u[3], w(H, H)), o2 = cquarter<INV>(u[5]), o3 = cmul(u[7], w(-H, H));
        const double2 e0 = u[0], e1 = u[2], e2 = u[4], e3 = u[6];
        u[0] = cadd(e0, o0);
        u[1] = cadd(e1, o1);
        u[2] = cadd(e2, o2);
        u[3] = cadd(e3, o3);
        u[4] = csub(e0, o0);
        u[5] = csub(e1, o1);
        u[6] = csub(e2, o2);
        u[7] = csub(e3, o3);
    } else if constexpr (R == 16) {
#pragma unroll
        for (int i = 0; i < 4; i++) dft4<INV>(u[i], u[i + 4], u[i + 8], u[i + 12]);
        // u[i + 4 r] by exp(-2 pi i (i r) / 16)
        u[5] = cmul(u[5], w(C1, S1));
        u[6] = cmul(u[6], w(H, H));
        u[7] = cmul(u[7], w(S1, C1));
        u[9] = cmul(u[9], w(H, H));
        u[10] = cquarter<INV>(u[10]);
        u[11] = cmul(u[11], w(-H, H));
        u[13] = cmul(u[13], w(S1, C1));
        u[14] = cmul(u[14], w(-H, H));
        u[15] = cmul(u[15], w(-C1, -S1));
#pragma unroll
        for (int r = 0; r < 4; r++) dft4<INV>(u[4 * r], u[4 * r + 1], u[4 * r + 2], u[4 * r + 3]);
        // output r + 4 s is in u[4 r + s]
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int s = r + 1; s < 4; s++) {
                const double2 x = u[4 * r + s];
                u[4 * r + s] = u[4 * s + r];
                u[4 * s + r] = x;
            }
    }
}

// LDS place of point i: a pass's writes (16 points apart) and the reads in
// order both touch every bank once.  x (below 32) tells the transforms of a
// wave apart, whose regions start at the same bank.
__device__ inline int fft_place(int i, int x) { return i ^ ((i >> 4) & 31) ^ x; }

// Places of points whose numbers share no bit are each other's exclusive or,
// so a thread's 16 places are one of them and constants.  here: the compiler
// forms them anew where they are used instead of keeping 16 registers.
__device__ inline void here(int &p) { asm volatile("" : "+v"(p)); }

// The passes from NS = product of the radices so far; tw: the tables of the
// passes to come, (R - 1) x NS each, [r - 1][k] = exp(-2 pi i r k / (NS R)).
template <int L, bool INV, int NS>
__device__ inline void fft_passes(double2 (&v)[16], double *sh, int x, int t, const double2 *__restrict__ tw) {
    constexpr int N = 1 << L, T = N / 16, R = N / NS >= 16 ? 16 : N / NS, B = 16 / R;
#pragma unroll
    for (int q = 0; q < B; q++) {
        int k = (t + q * T) & (NS - 1);
        here(k);
        double2 u[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            u[r] = v[q + r * B];
            if (NS > 1 && r > 0) {
                const double2 w = tw[(r - 1) * NS + k];
                u[r] = cmul(u[r], make_double2(w.x, INV ? -w.y : w.y));
            }
        }
        dft<R, INV>(u);
#pragma unroll
        for (int r = 0; r < R; r++) v[q + r * B] = u[r];
    }
    if constexpr (NS * R < N) {  // R = 16, one butterfly
        const int k = t & (NS - 1);
        int pw = fft_place((t - k) * 16 + k, x), pr = fft_place(t, x);
#pragma unroll
        for (int part = 0; part < 2; part++) {
            here(pw);
            here(pr);
#pragma unroll
            for (int r = 0; r < 16; r++) sh[pw ^ fft_place(r * NS, 0)] = part ? v[r].y : v[r].x;
            __syncthreads();
#pragma unroll
            for (int m = 0; m < 16; m++) (part ? v[m].y : v[m].x) = sh[pr ^ fft_place(m * T, 0)];
            __syncthreads();
        }
        fft_passes<L, INV, NS * R>(v, sh, x, t, tw + (NS > 1 ? (R - 1) * NS : 0));
    }
}

// z[m] = point N - k of the thread's k = t + m T (point 0 for k = 0)
template <int L>
__device__ inline void fft_mirror(const double2 (&v)[16], double2 (&z)[16], double *sh, int x, int t) {
    constexpr int N = 1 << L, T = N / 16;
    // N - k = (T - t) + (15 - m) T; t = 0 wraps to (16 - m) T
    int pw = fft_place(t, x), pr = fft_place((T - t) & (T - 1), x);
#pragma unroll
    for (int part = 0; part < 2; part++) {
        here(pw);
        here(pr);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 16; m++) sh[pw ^ fft_place(m * T, 0)] = part ? v[m].y : v[m].x;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 16; m++)
            (part ? z[m].y : z[m].x) =
                sh[pr ^ (t ? fft_place((15 - m) * T, 0) : fft_place((16 - m) % 16 * T, 0))];
    }
    __syncthreads();
}

// the tables of fft_passes for 2^l points (fewer than 2^l entries)
__global__ void fft_twiddles(double2 *tw, int l) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    for (int ns = 16; ns < 1 << l; ns *= 16) {
        const int r = min(16, (1 << l) / ns), cnt = (r - 1) * ns;
        if (e >= 0 && e < cnt) {
            double s, c;
            sincospi(-2.0 * (double)((e / ns + 1) * (e % ns)) / (double)(ns * r), &s, &c);
            *(tw + blockIdx.x * blockDim.x + threadIdx.x) = make_double2(c, s);
        }
        e -= cnt;
    }
}

// exp(-pi i k / 2^l), k < 2^l
__global__ void fft_half_turns(double2 *w, int l) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 1 << l) return;
    double s, c;
    sincospi(-(double)k / (double)(1 << l), &s, &c);
    w[k] = make_double2(c, s);
}
