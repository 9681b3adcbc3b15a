// 2-D spray chains by a block of threads.
//
// A prediction is a right-hand side (two short filters), a forward and a
// backward substitution along the trace, and a division in between.  Only
// the substitutions are sequential: eight operations a sample each with four
// band entries, against about 75 instructions a sample for the whole step in
// one thread.  So a block takes `nt` neighbouring chains of one direction
// and slice, holds their traces in LDS, and every phase but the substitutions
// runs over all its threads (thread = trace, and a piece of its samples); for
// the substitutions lane t of the first wave walks trace t, with the factor
// rows loaded into a register ring ahead of use and four samples per LDS
// access.  The float operations of a sample and their order are those of
// solve_factored / predict_adj_factored (predict.hpp), so the results are
// identical.
//
// What bounds it: the dependent chain of the substitutions (about 10
// instructions a sample and wave), hidden by other blocks of the CU when
// there are more than one.
#include <algorithm>
#include <type_traits>

#include "predict.hpp"

namespace {

constexpr int CH_TB = 512;         // threads of a block, at most
constexpr int CH_LDS = 15 * 1024;  // floats of a block's traces and piece heads, at most

// floats of one trace's LDS row: whole groups of D samples for the
// substitutions, a multiple of 4 (16-byte accesses), odd in units of 4
// (neighbouring traces in different banks)
SH_HD int chain_row(int n1, int D) {
    const int q = (n1 + D - 1) / D * D / 4;
    return 4 * (q | 1);
}

struct ChainPlan {
    int D = 0;   // factor rows in a walker's register ring
    int nt = 0;  // chains of a block (0: the chains run one thread each)
    int np = 0;  // pieces of a trace, at least 8 samples each
    int nb = 0;  // blocks of one slice and direction
    int tb = 0;  // threads
    size_t lds = 0;
};

// How the chains of nslice slices of n2 traces (both directions) are
// divided.  A CU holds one block of 8 waves of the kernels with a ring of 32
// rows (or two of the 16-row ones).  Up to 8 chains a CU, each block takes 8
// chains and all its threads share their samples, so that the phases between
// the substitutions end soonest, and the ring is deep.  With more chains the
// blocks are smaller (32 samples a thread) and as many as the chip holds, so
// that one block's substitutions run beside another's phases.
// 512 x 256 gather, 8 predictions of 1024 chains: 8 chains and 8 samples a
// thread 358 us, 16 and 16 395 us, 16 and 32 438 us.  300 x 100 x 100, 3
// predictions of 20000 chains: 20 chains and 32 samples 245 us, 32 and 32
// 249 us, 50 and 48 266 us, 64 and 64 320 us, 16 and 24 364 us.  (One thread
// per chain: 1436 us and 515 us.)
ChainPlan chain_plan(int n1, int n2, long nslice, int nw) {
    ChainPlan p;
    const long chains = 2L * n2 * nslice;
    const bool few = chains <= 8L * 256;
    p.D = nw <= 2 ? (few ? 32 : 16) : 8;
    const int S = chain_row(n1, p.D);
    p.np = std::max(1, few ? std::min(n1 / 8, CH_TB / 8) : std::min(n1 / 32, CH_TB / 4));
    const int per = S + p.np * 2 * nw;
    long nt = few ? 8 : std::min(32L, std::max(8L, chains / 1024));
    nt = std::min<long>({nt, CH_TB / p.np, CH_LDS / per});
    if (nt < 1) return p;
    p.nb = (n2 + (int)nt - 1) / (int)nt;
    p.nt = (n2 + p.nb - 1) / p.nb;
    p.tb = (p.nt * p.np + 63) / 64 * 64;
    // (the substitutions read whole groups past the last row)
    p.lds = ((size_t)p.nt * per + 32) * sizeof(float);
    return p;
}

typedef float ch_f4 __attribute__((ext_vector_type(4)));

__device__ inline __amdgpu_buffer_rsrc_t chain_rsrc(const void *p, unsigned long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)(unsigned)bytes, 0x00020000);
}

// Rows of a plane of factor rows through a buffer resource, one after the
// other: the lane's offset in a register, the row's as the instruction's
// scalar offset.  The resource's range check does not cover that one, so the
// offset stops at the last row, in the loops that reach it (END), and at the
// first one by a step of zero (a scalar instruction a row each; with both in
// every row 512 x 256, eight predictions, takes 528 us, so 500).  The offset
// is hidden from the optimiser after every step, which otherwise keeps those
// of a whole ring in scalar registers and spills them (sint3d of 300 x 100 x
// 100 11.15 ms, 11.39 without).
template <int NB>
struct ChainRows {
    __amdgpu_buffer_rsrc_t r;
    int lane;            // byte offset of the trace's row 0
    unsigned row, last;  // bytes from one sample to the next; to the last one
    template <bool END = true>
    __device__ void up(unsigned &at) const {
        at = __builtin_amdgcn_readfirstlane(END ? min(at + row, last) : at + row);
        asm volatile("" : "+s"(at));
    }
    static __device__ void down(unsigned &at, unsigned step) {
        at = __builtin_amdgcn_readfirstlane(at - step);
        asm volatile("" : "+s"(at));
    }
    __device__ void load(unsigned at, float *o) const {
        const int so = (int)__builtin_amdgcn_readfirstlane(at);
        typedef float f2 __attribute__((ext_vector_type(2)));
        if constexpr (NB % 4 == 0) {
#pragma unroll
            for (int c = 0; c < NB / 4; c++) {
                const ch_f4 v =
                    __builtin_bit_cast(ch_f4, __builtin_amdgcn_raw_buffer_load_b128(r, lane + 16 * c, so, 0));
#pragma unroll
                for (int i = 0; i < 4; i++) o[4 * c + i] = v[i];
            }
        } else {
#pragma unroll
            for (int c = 0; c < NB / 2; c++) {
                const f2 v = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(r, lane + 8 * c, so, 0));
                o[2 * c] = v[0];
                o[2 * c + 1] = v[1];
            }
        }
    }
};

// Forward substitution in place over the LDS row y (banded_solve's first
// loop): y[k] -= o_m[k-1-m] y[k-1-m], m = 0 .. NB-1 in turn.  Entries before
// the trace are zeros (subtracting 0 * 0 changes nothing); the last group
// runs on into the row's padding, which nothing reads.
template <int NB, int D>
__device__ inline void chain_forward(const ChainRows<NB> &F, float *y, int n1) {
    float o[D][NB], b[NB];
    unsigned at = 0;
#pragma unroll
    for (int s = 0; s < D; s++) {
        if (s < D - NB) {
            F.load(at, o[s]);
            F.up(at);
        } else {
#pragma unroll
            for (int m = 0; m < NB; m++) o[s][m] = 0.0f;
        }
    }
#pragma unroll
    for (int m = 0; m < NB; m++) b[m] = 0.0f;
    constexpr int R = 2;  // groups of four samples read ahead
    ch_f4 r[R];
#pragma unroll
    for (int g = 0; g < R; g++) r[g] = reinterpret_cast<const ch_f4 *>(y)[g];
    auto group = [&](auto end, int k0) {
        constexpr bool END = decltype(end)::value;  // the rows to come reach the last one
#pragma unroll
        for (int g = 0; g < D / 4; g++) {
            ch_f4 v = r[g % R];
            r[g % R] = *reinterpret_cast<const ch_f4 *>(y + k0 + 4 * R + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int s = 4 * g + i;
                float t = v[i];
#pragma unroll
                for (int m = 0; m < NB; m++) t -= o[(s - 1 - m + 2 * D) % D][m] * b[m];
#pragma unroll
                for (int m = NB - 1; m > 0; m--) b[m] = b[m - 1];
                b[0] = t;
                v[i] = t;
                F.load(at, o[(s + D - NB) % D]);  // row k0 + s + D - NB
                F.template up<END>(at);
            }
            *reinterpret_cast<ch_f4 *>(y + k0 + 4 * g) = v;
        }
    };
    int k0 = 0;
    for (; k0 + 2 * D - NB < n1; k0 += D) group(std::false_type{}, k0);
    for (; k0 < n1; k0 += D) group(std::true_type{}, k0);
}

// Backward substitution in place (banded_solve's second loop after the
// division): y[k] -= o_m[k] y[k+1+m], from the end of the padding (zeros
// there, and the last row's entries, which its rows are read as, are zeros,
// since no sample lies beyond: its values stay zero).
template <int NB, int D>
__device__ inline void chain_backward(const ChainRows<NB> &F, float *y, int n1) {
    const int top = (n1 + D - 1) / D * D;
    float o[D][NB], x[NB];
    const unsigned start = (unsigned)(top - D) * F.row;
    unsigned at = start;
#pragma unroll
    for (int s = 0; s < D; s++) {
        F.load(at, o[s]);
        F.up(at);
    }
    at = start;
#pragma unroll
    for (int m = 0; m < NB; m++) x[m] = 0.0f;
    constexpr int R = 2;
    ch_f4 r[R];
#pragma unroll
    for (int g = 0; g < R; g++) r[g] = *reinterpret_cast<const ch_f4 *>(y + top - 4 * R + 4 * g);
    for (int k0 = top - D; k0 >= 0; k0 -= D) {
        const unsigned step = k0 ? F.row : 0;  // the first group has no rows before it
#pragma unroll
        for (int g = D / 4 - 1; g >= 0; g--) {
            ch_f4 v = r[g % R];
            r[g % R] = *reinterpret_cast<const ch_f4 *>(y + max(k0 - 4 * R + 4 * g, 0));
#pragma unroll
            for (int i = 3; i >= 0; i--) {
                const int s = 4 * g + i;
                float t = v[i];
#pragma unroll
                for (int m = 0; m < NB; m++) t -= o[s][m] * x[m];
#pragma unroll
                for (int m = NB - 1; m > 0; m--) x[m] = x[m - 1];
                x[0] = t;
                v[i] = t;
                F.down(at, step);
                F.load(at, o[s]);  // row k0 + s - D
            }
            *reinterpret_cast<ch_f4 *>(y + k0 + 4 * g) = v;
        }
    }
}

// What a block of chains works on: its direction, slice and traces, and
// this thread's trace and piece [k0, k0 + len).
struct ChainBlock {
    int dir, i0, nt, t, c, k0, len, most, n1, n2;
    bool live;         // the thread has a piece of a trace of the slice
    long slice, base;  // samples of a slice; the slice's first element
};
__device__ inline ChainBlock chain_block(int n1, int n2, int nt, int np, int nb) {
    ChainBlock B;
    B.n1 = n1;
    B.n2 = n2;
    B.nt = nt;
    B.dir = blockIdx.x / nb;
    B.i0 = (blockIdx.x % nb) * nt;
    B.t = threadIdx.x % nt;
    B.c = threadIdx.x / nt;
    B.k0 = (int)((long)B.c * n1 / np);
    B.len = (int)((long)(B.c + 1) * n1 / np) - B.k0;
    B.most = (n1 + np - 1) / np;
    B.live = B.c < np && B.i0 + B.t < n2;
    B.slice = (long)n1 * n2;
    B.base = (long)blockIdx.y * B.slice;
    return B;
}

// The normal-equation product of the block's traces, in place: row =
// A^T A row + e boundary(row), with the taps as given (the right-hand side,
// solve_factored) or reversed (the adjoint product, pred_adj_apply: both of
// its sums run over the taps in the other order).  A thread slides over
// its piece: sample kk's filter output goes, times its j-th tap, to row kk +
// NW - j, which so collects its products in ascending j.  The first 2 NW
// inputs of every piece are kept in heads, the piece before reads them there.
// q is the slope trace (q[k * n2]); the taps are formed from it here, on
// every thread: loading them ready-made (20 bytes a sample instead of 4)
// takes as long for a gather and longer for a volume, whose chains are bound
// by the memory they read.
template <int NW>
__device__ inline void chain_apply(const ChainBlock &B, const float *q, bool rev, bool act, float *row, float *heads,
                                   float e) {
    constexpr int NA = 2 * NW + 1, G = 4;
    const int n1 = B.n1, k0 = B.k0;
    float acc[NA], in[NA];  // rows and inputs kk - NW .. kk + NW
    float *const head = heads + (B.c * B.nt + B.t) * (2 * NW), *const next = head + B.nt * (2 * NW);
#pragma unroll
    for (int j = 0; j < NA; j++) acc[j] = 0.0f;
    in[0] = 0.0f;
    if (B.live)
#pragma unroll
        for (int j = 0; j < 2 * NW; j++) {
            in[j + 1] = k0 > 0 ? row[k0 - 2 * NW + j] : 0.0f;
            head[j] = row[k0 + j];
        }
    __syncthreads();
    if (!(act && B.live)) return;
    float qn[G];
    auto slope = [&](int s) { return q[(long)min(max(k0 - NW + s, 0), n1 - 1) * B.n2]; };
#pragma unroll
    for (int g = 0; g < G; g++) qn[g] = slope(g);
    for (int s0 = 0; s0 < B.most + 2 * NW; s0 += G) {
        float qc[G];
#pragma unroll
        for (int g = 0; g < G; g++) qc[g] = qn[g];
#pragma unroll
        for (int g = 0; g < G; g++) qn[g] = slope(s0 + G + g);
        float v[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int s = s0 + g;
            const float *p = s < B.len ? row + k0 + s : next + min(s - B.len, 2 * NW - 1);
            v[g] = k0 + s < n1 ? *p : 0.0f;
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int s = s0 + g, kk = k0 - NW + s, k = kk - NW;
#pragma unroll
            for (int j = 0; j < NA - 1; j++) in[j] = in[j + 1];
            in[NA - 1] = v[g];
            const bool in_trace = kk >= NW && kk < n1 - NW;
            float b[NA], a[NA];
            apf_pass<NW>(qc[g], b);
            tap_order<NA>(b, rev, a);
            float t = 0.0f;
#pragma unroll
            for (int j = 0; j < NA; j++) t += a[j] * in[j];
#pragma unroll
            for (int j = 0; j < NA; j++) {
                const float x = acc[NA - 1 - j] + a[j] * t;
                acc[NA - 1 - j] = in_trace ? x : acc[NA - 1 - j];
            }
            float o = acc[0];
            if (k < 2 || k >= n1 - 2) o += e * in[0];
            if (s >= 2 * NW && s - 2 * NW < B.len) row[k] = o;
#pragma unroll
            for (int j = 0; j < NA - 1; j++) acc[j] = acc[j + 1];
            acc[NA - 1] = 0.0f;
        }
    }
}

// Substitutions of the block's traces with the factors of their targets ip:
// forward, division by the diagonal, backward.  Every thread calls it.
template <int NB, int D>
__device__ inline void chain_solve(const ChainBlock &B, float *row, const float *Fv, long n, int ip, bool act,
                                   float *lds, int S) {
    // the variant's rows at this slice: off-diagonal entries, then the
    // diagonal plane behind those of all slices
    const float *fo = Fv + (long)NB * B.base, *fd = Fv + (long)NB * n + B.base;
    const bool walker = threadIdx.x < (unsigned)B.nt && act;
    const ChainRows<NB> F{chain_rsrc(fo, (unsigned long)B.slice * NB * 4), ip * NB * 4, (unsigned)B.n2 * NB * 4,
                          (unsigned)(B.n1 - 1) * (unsigned)B.n2 * NB * 4};
    __syncthreads();
    if (walker) {
        __builtin_amdgcn_s_setprio(3);
        chain_forward<NB, D>(F, lds + (int)threadIdx.x * S, B.n1);
        __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    if (act && B.live) {
#pragma unroll 8
        for (int s = 0; s < B.most; s++) {
            const int k = min(B.k0 + s, B.n1 - 1);
            const float v = row[k] / fd[(long)k * B.n2 + ip];
            if (s < B.len) row[k] = v;
        }
        if (B.k0 + B.len == B.n1)
            for (int k = B.n1; k < (B.n1 + D - 1) / D * D; k++) row[k] = 0.0f;
    }
    __syncthreads();
    if (walker) {
        __builtin_amdgcn_s_setprio(3);
        chain_backward<NB, D>(F, lds + (int)threadIdx.x * S, B.n1);
        __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
}

// Forward chains: block (direction, group of nt source traces) of slice
// blockIdx.y; blockIdx.z picks the input and the slot volume.  Same result as
// spray2_fwd.
template <int NW, int D>
__global__ void __launch_bounds__(CH_TB) __attribute__((amdgpu_waves_per_eu(NW <= 2 && D <= 16 ? 4 : 2)))
chain2_fwd(const float *__restrict__ x, const float *__restrict__ dip, const float *__restrict__ F, float *__restrict__ U, int n1, int n2, int n3,
           int ns, float e, int nt, int np, int nb, const int *stop, const float *__restrict__ x2,
           float *__restrict__ U2) {
    if (stop && *(volatile const int *)stop) return;
    extern __shared__ ch_f4 ch_lds[];
    float *const lds = reinterpret_cast<float *>(ch_lds);
    constexpr int NB = 2 * NW;
    if (blockIdx.z) {
        x = x2;
        U = U2;
    }
    const ChainBlock B = chain_block(n1, n2, nt, np, nb);
    const int i = B.i0 + B.t, S = chain_row(n1, D);
    const long n = B.slice * n3, pf = fac_plane_floats(NB, n);
    float *const row = lds + B.t * S, *const heads = lds + nt * S + 32;
    // the input, the centre slot (one direction writes it) and the slots of
    // this trace that no chain reaches
    if (B.live) {
#pragma unroll 8
        for (int s = 0; s < B.len; s++) {
            const long at = B.base + (long)(B.k0 + s) * n2 + i;
            const float v = x[at];
            row[B.k0 + s] = v;
            if (B.dir == 0) U[ns * n + at] = v;
        }
        for (int is = B.dir == 0 ? max(0, n2 - 1 - i) : min(i, ns); is < ns; is++) {
            float *z = U + (B.dir == 0 ? ns - is - 1 : ns + is + 1) * n + B.base + (long)B.k0 * n2 + i;
            for (int s = 0; s < B.len; s++) z[(long)s * n2] = 0.0f;
        }
    }
    __syncthreads();
    const int far = min(B.i0 + nt, n2) - 1;
    for (int is = 0; is < ns; is++) {
        if (B.dir == 0 ? far - is - 1 < 0 : B.i0 + is + 1 >= n2) break;  // none of the block's chains goes on
        const int ip = B.dir == 0 ? i - is - 1 : i + is + 1, iq = B.dir == 0 ? ip : ip - 1;
        const bool act = i < n2 && ip >= 0 && ip < n2;
        chain_apply<NW>(B, dip + B.base + iq, B.dir == 1, act, row, heads, e);
        chain_solve<NB, D>(B, row, F + B.dir * pf, n, ip, act, lds, S);
        if (act && B.live) {
            float *u = U + (B.dir == 0 ? ns - is - 1 : ns + is + 1) * n + B.base + (long)B.k0 * n2 + ip;
#pragma unroll 8
            for (int s = 0; s < B.len; s++) u[(long)s * n2] = row[B.k0 + s];
        }
    }
}

// Adjoint chains (see spray2_adj).  The slot a step adds is U's, or, with
// ww, formed from the smoothed field U as pwsmooth_adj_weight does:
// (U * w_slot) * ww.
template <int NW, int D>
__global__ void __launch_bounds__(CH_TB) __attribute__((amdgpu_waves_per_eu(NW <= 2 && D <= 16 ? 4 : 2)))
chain2_adj(const float *__restrict__ U, const float *__restrict__ ww, const float *__restrict__ dip,
           const float *__restrict__ F,
           float *__restrict__ C, int n1, int n2, int n3, int ns, float e, int nt, int np, int nb, const int *stop) {
    if (stop && *(volatile const int *)stop) return;
    extern __shared__ ch_f4 ch_lds[];
    float *const lds = reinterpret_cast<float *>(ch_lds);
    constexpr int NB = 2 * NW;
    const ChainBlock B = chain_block(n1, n2, nt, np, nb);
    const int i = B.i0 + B.t, S = chain_row(n1, D);
    const long n = B.slice * n3, pf = fac_plane_floats(NB, n);
    float *const row = lds + B.t * S, *const heads = lds + nt * S + 32;
    if (B.live)
        for (int s = 0; s < B.len; s++) row[B.k0 + s] = 0.0f;
    const int far = min(B.i0 + nt, n2) - 1;
    for (int is = ns - 1; is >= 0; is--) {
        if (B.dir == 1 ? B.i0 + is + 1 >= n2 : far - is - 1 < 0) continue;  // none of the block's chains has begun
        const int ip = B.dir == 1 ? i + is + 1 : i - is - 1, iq = B.dir == 1 ? ip - 1 : ip;
        const bool act = i < n2 && ip >= 0 && ip < n2;
        const int slot = B.dir == 1 ? ns + is + 1 : ns - is - 1;
        if (act && B.live) {
            const float w = (float)(ns + 1 - abs(slot - ns));
            const long at = B.base + (long)B.k0 * n2 + ip;
            if (ww) {
#pragma unroll 8
                for (int s = 0; s < B.len; s++) {
                    const float u = U[at + (long)s * n2] * w * ww[at + (long)s * n2];
                    row[B.k0 + s] = row[B.k0 + s] + u;
                }
            } else {
#pragma unroll 8
                for (int s = 0; s < B.len; s++) row[B.k0 + s] = row[B.k0 + s] + U[slot * n + at + (long)s * n2];
            }
        }
        chain_solve<NB, D>(B, row, F + B.dir * pf, n, ip, act, lds, S);
        chain_apply<NW>(B, dip + B.base + iq, B.dir == 0, act, row, heads, e);
        __syncthreads();
    }
    if (B.live) {
        float *c = C + B.dir * n + B.base + (long)B.k0 * n2 + i;
#pragma unroll 8
        for (int s = 0; s < B.len; s++) c[(long)s * n2] = row[B.k0 + s];
    }
}

// The chains' factors (factor_sweep's, identical), in two launches: the
// normal matrix's rows by one thread per 16 samples of a trace and direction,
// written where the factor will be, then the LDL^T recurrence alone, one
// thread per trace, in place with the rows loaded 8 samples ahead.  As one
// sweep per trace, forming the rows was half of its instructions.
constexpr int FR = 16;
template <int NW>
__global__ void __launch_bounds__(256)
chain2_rows(const float *__restrict__ dip, float *__restrict__ F, int n1, int n2, int n3, float e, int np) {
    constexpr int NA = 2 * NW + 1, NB = 2 * NW;
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(gid % n2), vc = (int)(gid / n2), v = vc / np, k0 = vc % np * FR;
    if (v > 1 || (v == 0 ? i > n2 - 2 : i < 1)) return;  // never a target in that direction
    const long slice = (long)n1 * n2, base = blockIdx.y * slice, n = slice * n3;
    const Acc q{dip + base + (v == 0 ? i : i - 1), n2};
    const FactorOut Fs = fac_out_at(F + v * fac_plane_floats(NB, n), NB, n, base + i, n2);
    float A[NA][NA];
#pragma unroll
    for (int w = 0; w < NA; w++) taps_at<NW>(q, k0 - NW + w, n1, v == 1, A[w]);
    for (int k = k0; k < min(k0 + FR, n1); k++) {
        float diag, offd[NB];
        reg_row<NB>(k, n1, e, diag, offd);
#pragma unroll
        for (int j = 0; j < NA; j++) {
            const int kk = k + j - NW;
            if (kk >= NW && kk < n1 - NW) diag += A[j][j] * A[j][j];
        }
#pragma unroll
        for (int m = 0; m < NB; m++)
#pragma unroll
            for (int j = m + 1; j < NA; j++) {
                const int kk = k + j - NW;
                if (kk >= NW && kk < n1 - NW) offd[m] += A[j][j - m - 1] * A[j][j];
            }
        fac_put<NB>(Fs, k, diag, offd);
#pragma unroll
        for (int w = 0; w < NA - 1; w++)
#pragma unroll
            for (int j = 0; j < NA; j++) A[w][j] = A[w + 1][j];
        taps_at<NW>(q, k + 1 + NW, n1, v == 1, A[NA - 1]);
    }
}

template <int NW>
__global__ void __launch_bounds__(64)
chain2_ldl(float *__restrict__ F, int n1, int n2, int n3) {
    constexpr int NB = 2 * NW, D = 8;
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(gid % n2), v = (int)(gid / n2);
    if (v > 1 || (v == 0 ? i > n2 - 2 : i < 1)) return;
    const long slice = (long)n1 * n2, base = blockIdx.y * slice, n = slice * n3;
    float *const Fv = F + v * fac_plane_floats(NB, n);
    const FactorOut Fo = fac_out_at(Fv, NB, n, base + i, n2);
    const Factor Fi{Fo.d, Fo.o, n2};
    float rd[D], ro[D][NB], Ld[NB], Lo[NB][NB];
    auto fetch = [&](int s, int k) {
        const long kc = k < n1 ? k : n1 - 1;
        rd[s] = fac_d(Fi, kc);
        fac_row<NB>(Fi, kc, ro[s]);
    };
#pragma unroll
    for (int r = 0; r < NB; r++) {
        Ld[r] = 0.0f;
#pragma unroll
        for (int m = 0; m < NB; m++) Lo[r][m] = 0.0f;
    }
#pragma unroll
    for (int s = 0; s < D; s++) fetch(s, s);
    auto step = [&](int s, int k) {
        // rows before the trace are zeros: subtracting 0 * 0 * 0 changes nothing
        float t = rd[s];
#pragma unroll
        for (int m = 0; m < NB; m++) t -= (Lo[m][m]) * (Lo[m][m]) * (Ld[m]);
        float ok[NB];
#pragma unroll
        for (int c = 0; c < NB; c++) {
            float w = ro[s][c];
#pragma unroll
            for (int m = 0; m < NB - c - 1; m++) w -= (Lo[m][m]) * (Lo[m][c + m + 1]) * (Ld[m]);
            ok[c] = c < n1 - k - 1 ? w / t : 0.0f;
        }
        fac_put<NB>(Fo, k, t, ok);
#pragma unroll
        for (int r = NB - 1; r > 0; r--) {
            Ld[r] = Ld[r - 1];
#pragma unroll
            for (int m = 0; m < NB; m++) Lo[r][m] = Lo[r - 1][m];
        }
        Ld[0] = t;
#pragma unroll
        for (int m = 0; m < NB; m++) Lo[0][m] = ok[m];
        fetch(s, k + D);
    };
    int k0 = 0;
    for (; k0 + D <= n1; k0 += D) {
#pragma unroll
        for (int s = 0; s < D; s++) step(s, k0 + s);
    }
#pragma unroll
    for (int s = 0; s < D; s++)
        if (k0 + s < n1) step(s, k0 + s);
}

}  // namespace

// Whether the blocks run (one thread per chain otherwise).  A block's walkers
// hold few chains at a time, so they lose where the chip would be full with
// a thread each, the more so the longer the traces (fewer of them fit a
// block) and the higher the order; and short traces leave nothing to share
// out.  Measured over traces of 8 to 15000 samples, 64 to 200000 chains and
// orders 1 to 4 (blocks' gain over one thread each, one spray): order 2,
// 128 x 2000 chains 1.71, 48 x 4000 0.59, 96 x 8000 1.00, 1000 x 20000 1.04,
// 1000 x 80000 0.76, 2000 x 8000 1.26, 3000 x 20000 0.58, 8000 x 4000 1.11,
// 8000 x 8000 0.69; order 3, 1000 x 8000 1.55, 1000 x 20000 0.65; order 4,
// 2000 x 2000 1.22, 2000 x 8000 0.49.  The lines run where it is about 1.
bool chain2_fits(int n1, int n2, int n3, int order, int sprays) {
    const long slices = (long)n3 * sprays;
    const double chains = 2.0 * n2 * slices;
    if (n1 < (chains > 2048 ? 96 : order == 1 ? 48 : 32)) return false;
    if (chains >= (order <= 3 ? 2000.0 : 1000.0) + (order <= 2 ? 18e6 : order == 3 ? 8e6 : 5e6) / n1) return false;
    // (a slice's factor rows are addressed with 32-bit offsets)
    return n3 <= 65535 && (double)n1 * n2 * 8 * order < 4294967295.0 && chain_plan(n1, n2, slices, order).nt > 0;
}

int chain2_factor(sh_ctx *ctx, const Pwsmooth2 &P) {
    const int np = ceil_div(P.n1, FR);
    SH_DISPATCH_NW(ctx, P.order, NW,
                   hipLaunchKernelGGL((chain2_rows<NW>), dim3(ceil_div(2L * P.n2 * np, 256), P.n3), dim3(256), 0,
                                      ctx->stream, P.dip, P.F, P.n1, P.n2, P.n3, P.e, np);
                   hipLaunchKernelGGL((chain2_ldl<NW>), dim3(ceil_div(2L * P.n2, 64), P.n3), dim3(64), 0, ctx->stream,
                                      P.F, P.n1, P.n2, P.n3));
    return sh_launch_check(ctx, "chain2_factor");
}

// NW and D of a plan (orders 3 and 4 keep a ring of 8 rows)
#define CHAIN_DISPATCH(ctx, order, D, ...)                    \
    SH_DISPATCH_NW(ctx, order, NW, {                          \
        if (NW > 2) {                                         \
            constexpr int DD = 8;                             \
            __VA_ARGS__;                                      \
        } else if ((D) == 32) {                               \
            constexpr int DD = NW > 2 ? 8 : 32;               \
            __VA_ARGS__;                                      \
        } else {                                              \
            constexpr int DD = NW > 2 ? 8 : 16;               \
            __VA_ARGS__;                                      \
        }                                                     \
    })

int chain2_forward(sh_ctx *ctx, const Pwsmooth2 &P, const float *x, const float *x2, float *U2) {
    const int sprays = x2 ? 2 : 1;
    const ChainPlan K = chain_plan(P.n1, P.n2, (long)P.n3 * sprays, P.order);
    if (K.nt < 1) return sh_fail(ctx, SH_EUNSUP, "chain2: traces of %d samples do not fit", P.n1);
    const dim3 grid(2 * K.nb, P.n3, sprays);
    CHAIN_DISPATCH(ctx, P.order, K.D,
                   hipLaunchKernelGGL((chain2_fwd<NW, DD>), grid, dim3(K.tb), K.lds, ctx->stream, x, P.dip, P.F, P.U, P.n1,
                                      P.n2, P.n3, P.ns, P.e, K.nt, K.np, K.nb, P.stop, x2, U2));
    return sh_launch_check(ctx, "chain2_fwd");
}

int chain2_adjoint(sh_ctx *ctx, const Pwsmooth2 &P, const float *U, const float *ww) {
    const ChainPlan K = chain_plan(P.n1, P.n2, P.n3, P.order);
    if (K.nt < 1) return sh_fail(ctx, SH_EUNSUP, "chain2: traces of %d samples do not fit", P.n1);
    const dim3 grid(2 * K.nb, P.n3);
    CHAIN_DISPATCH(ctx, P.order, K.D,
                   hipLaunchKernelGGL((chain2_adj<NW, DD>), grid, dim3(K.tb), K.lds, ctx->stream, U, ww, P.dip, P.F, P.C,
                                      P.n1, P.n2, P.n3, P.ns, P.e, K.nt, K.np, K.nb, P.stop));
    return sh_launch_check(ctx, "chain2_adj");
}
