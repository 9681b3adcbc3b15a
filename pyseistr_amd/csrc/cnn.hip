// Learned warm start for dip estimation: a 6-layer 3-D CNN (3x3x3 kernels,
// 32 channels, ReLU) that maps a normalised seismic volume to an initial
// (inline, crossline) dip field.  No counterpart in the reference; the dips
// it produces only seed the reference's Gauss-Newton loop (sh_dip init).
//
// Kernels: BF16 activations in channels-last layout [voxel][32] (voxel =
// F-order index), FP32 accumulation on the gfx950 matrix cores
// (v_mfma_f32_32x32x16_bf16) for the 32-channel layers, implicit GEMM with
// zero padding at the volume faces.  Backward: input gradients reuse the
// forward kernel with flipped/transposed weights and the ReLU mask of the
// layer below; weight gradients are per-block MFMA partials reduced in a
// fixed order.  Master weights and Adam state are FP32.
#include "common.hpp"

#include <algorithm>
#include <cstdlib>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Raw buffer access (32-bit byte offsets against a resource of known size):
// loads past the size return zeros and stores past it are dropped.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr unsigned BUF_OOB = 0xFFFFE000u;  // offset past every buffer used here
__device__ inline __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ inline bf16x8 ld_frag(__amdgpu_buffer_rsrc_t r, unsigned off, bool ok) {
    u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    u32x4 z = {0u, 0u, 0u, 0u};
    return __builtin_bit_cast(bf16x8, ok ? v : z);
}

namespace {

constexpr int C = 32, NT = 27, TB = 256;

// Parameter layout (FP32, flat): W1[27][32] b1[32] {Wl[27][32ci][32co] bl[32]} x4  W6[27][32][2] b6[2]
constexpr long OFF_W1 = 0, OFF_B1 = OFF_W1 + NT * C;
constexpr long L_SZ = (long)NT * C * C + C;
constexpr long OFF_L(int l) { return OFF_B1 + C + (long)(l - 2) * L_SZ; }  // l = 2..5
constexpr long OFF_W6 = OFF_B1 + C + 4 * L_SZ, OFF_B6 = OFF_W6 + NT * C * 2;
constexpr long NPARAM = OFF_B6 + 2;

__device__ inline void tap_offset(int t, int &d1, int &d2, int &d3) {
    d1 = t % 3 - 1;
    d2 = (t / 3) % 3 - 1;
    d3 = t / 9 - 1;
}

// ---------------------------------------------------------------------------
// Weight packing: master FP32 -> BF16 [27][32 co][32 ci] for the forward of
// layers 2..6 (layer 6 padded to 32 outputs with zeros) and the flipped,
// transposed [27][32 ci][32 co] for the input-gradient pass.
// ---------------------------------------------------------------------------
__global__ void pack_weights(const float *__restrict__ P, __bf16 *__restrict__ Wf, __bf16 *__restrict__ Wb) {
    // Wf, Wb: [5 layers][27][32][32]
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long per = (long)NT * C * C;
    if (i >= 5 * per) return;
    int l = (int)(i / per);  // 0..4 -> layers 2..6
    long r = i % per;
    int t = (int)(r / (C * C)), a = (int)((r / C) % C), b = (int)(r % C);
    // forward: Wf[l][t][co=a][ci=b] = W[t][ci=b][co=a]
    float wf, wb;
    if (l < 4) {
        const float *W = P + OFF_L(l + 2);
        wf = W[((long)t * C + b) * C + a];
        // backward: Wb[l][t'][co'=a (= ci)][ci'=b (= co)] = W[flip t'][ci=a][co=b]
        wb = W[((long)(NT - 1 - t) * C + a) * C + b];
    } else {
        const float *W = P + OFF_W6;  // [27][32 ci][2 co]
        wf = (a < 2) ? W[((long)t * C + b) * 2 + a] : 0.0f;
        wb = (b < 2) ? W[((long)(NT - 1 - t) * C + a) * 2 + b] : 0.0f;
    }
    Wf[i] = (__bf16)wf;
    Wb[i] = (__bf16)wb;
}

// ---------------------------------------------------------------------------
// Layer 1 (1 -> 32), FP32 input, ReLU, BF16 output.
// ---------------------------------------------------------------------------
// The weights and biases are read with wave-uniform indices from the
// read-only parameter vector, so they arrive through scalar loads and feed
// the FMAs as scalar operands (no LDS traffic per FMA).
__global__ void __launch_bounds__(TB) conv1_fwd(const float *__restrict__ x, float xscale, const float *__restrict__ P,
                                                __bf16 *__restrict__ out, int n1, int n2, int n3, int dil,
                                                FastDiv f1, FastDiv f2, const float *__restrict__ xsp) {
    if (xsp) xscale = xsp[0];  // the scale computed on the device
    const float *__restrict__ w = P + OFF_W1;
    const float *__restrict__ b = P + OFF_B1;
    long n = (long)n1 * n2 * n3;
    long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    int i1, i2, i3;
    if (n < (1L << 31)) {  // multiply-high division (no long division per voxel)
        const unsigned r = f1.div((unsigned)v), q = f2.div(r);
        i1 = (int)((unsigned)v - r * (unsigned)n1);
        i2 = (int)(r - q * (unsigned)n2);
        i3 = (int)q;
    } else {
        i1 = (int)(v % n1);
        const long r = v / n1;
        i2 = (int)(r % n2);
        i3 = (int)(r / n2);
    }
    float xv[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        int d1 = (t % 3 - 1) * dil, d2 = ((t / 3) % 3 - 1) * dil, d3 = (t / 9 - 1) * dil;
        int j1 = i1 + d1, j2 = i2 + d2, j3 = i3 + d3;
        bool in = j1 >= 0 && j1 < n1 && j2 >= 0 && j2 < n2 && j3 >= 0 && j3 < n3;
        xv[t] = in ? x[v + d1 + (long)n1 * (d2 + (long)n2 * d3)] * xscale : 0.0f;
    }
    __bf16 o[C];
#pragma unroll
    for (int co = 0; co < C; co++) {
        float s = b[co];
#pragma unroll
        for (int t = 0; t < NT; t++) s = fmaf(w[t * C + co], xv[t], s);
        o[co] = (__bf16)fmaxf(s, 0.0f);
    }
    bf16x8 *dst = (bf16x8 *)(out + v * C);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        bf16x8 pk;
#pragma unroll
        for (int i = 0; i < 8; i++) pk[i] = o[q * 8 + i];
        dst[q] = pk;
    }
}

// conv1_fwd for dilation 1 with the input staged in LDS: a block owns a
// 64 (i1) x 4 (i2) tile and marches along i3 over a segment of planes,
// keeping the scaled input planes o-1, o, o+1 (with their one-sample halo,
// zero outside the volume) in a ring of three LDS planes, so each input
// sample is read from HBM about once instead of through 27 global loads
// per voxel.  Same operations per output as conv1_fwd.
constexpr int C1_W = 66, C1_H = 6, C1_PL = C1_W * C1_H;

__global__ void __launch_bounds__(TB) conv1_fwd_tile(const float *__restrict__ x, float xscale,
                                                     const float *__restrict__ P, __bf16 *__restrict__ out, int n1,
                                                     int n2, int n3, int seg, const float *__restrict__ xsp) {
    if (xsp) xscale = xsp[0];
    __shared__ float pl[3 * C1_PL];
    const float *__restrict__ w = P + OFF_W1;
    const float *__restrict__ b = P + OFF_B1;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 x 4
    const int ntile1 = (n1 + 63) / 64;
    const int x0 = (blockIdx.x % ntile1) * 64, y0 = (blockIdx.x / ntile1) * 4;
    const int z0 = blockIdx.y * seg, z1 = min(n3, z0 + seg);
    const long n12 = (long)n1 * n2;
    const int i1 = x0 + tx, i2 = y0 + ty;
    for (int q = z0 - 1; q <= z1; q++) {
        // plane q into ring slot (q + 3) % 3
        float *dst = pl + ((q + 3) % 3) * C1_PL;
        for (int e = threadIdx.x; e < C1_PL; e += TB) {
            const int r = e / C1_W, c = e - r * C1_W;
            const int j1 = x0 - 1 + c, j2 = y0 - 1 + r;
            const bool in = q >= 0 && q < n3 && j1 >= 0 && j1 < n1 && j2 >= 0 && j2 < n2;
            dst[e] = in ? x[j1 + (long)n1 * j2 + n12 * q] * xscale : 0.0f;
        }
        __syncthreads();
        const int o = q - 1;
        if (o >= z0 && i1 < n1 && i2 < n2) {
            float xv[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int d1 = t % 3 - 1, d2 = (t / 3) % 3 - 1, d3 = t / 9 - 1;
                xv[t] = pl[((o + d3 + 3) % 3) * C1_PL + (ty + 1 + d2) * C1_W + tx + 1 + d1];
            }
            __bf16 ov[C];
#pragma unroll
            for (int co = 0; co < C; co++) {
                float s = b[co];
#pragma unroll
                for (int t = 0; t < NT; t++) s = fmaf(w[t * C + co], xv[t], s);
                ov[co] = (__bf16)fmaxf(s, 0.0f);
            }
            bf16x8 *dp = (bf16x8 *)(out + ((long)i1 + (long)n1 * i2 + n12 * o) * C);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                bf16x8 pk;
#pragma unroll
                for (int i = 0; i < 8; i++) pk[i] = ov[k * 8 + i];
                dp[k] = pk;
            }
        }
        __syncthreads();  // the slot of plane o - 1 is overwritten next
    }
}

// ---------------------------------------------------------------------------
// 32-channel 3x3x3 convolution on the matrix cores.
// Block = 4 waves, tile 64 (i1) x 4 (i2) voxels at one i3; wave w owns row
// i2 = y0 + w as two 32-voxel M-tiles.  Per tap and 16-channel half:
// A = input [32 voxels][16 ci] from global (zero outside the volume),
// B = W [16 ci][32 co] from LDS, D += A B in FP32.
// MODE 0: out = relu(D + b) BF16;  MODE 1: out[v][0..1] = D + b FP32;
// MODE 2: out = D * (aux > 0) BF16 (input gradient through the ReLU).
// ---------------------------------------------------------------------------
constexpr int CW = 8;          // waves per conv block (one i2 row of the tile each)
constexpr int CTB = 64 * CW;   // threads per conv block

// B operands in LDS: 16-byte entries [tap][h][hi][co] (h: which 8 of the
// lane's 16 input channels, hi = lane / 32, co = lane % 32), so the 64
// lanes of one fragment read cover 1 KB contiguously and hit distinct
// banks.  (Entries in [tap][co][ci] order put lanes co, co + 4, ... 64 B
// apart on the same banks; at 512x256x256 the layers ran equally fast
// either way, so bank conflicts are not what bounds them.)
__device__ inline void stage_weights(bf16x8 *wl, const __bf16 *__restrict__ Wg) {
    for (int i = threadIdx.x; i < NT * C * C / 8; i += blockDim.x) {
        const int co = i % 32, hi = (i / 32) % 2, h = (i / 64) % 2, t = i / 128;
        wl[i] = ((const bf16x8 *)Wg)[((t * C + co) * C + hi * 16 + h * 8) / 8];
    }
}
__device__ inline int wl_at(int t, int h, int hi, int co) { return ((t * 2 + h) * 2 + hi) * 32 + co; }

// A fragments of one (d2, d3) row of taps: [d1][m][half]
struct RowFrag {
    bf16x8 a[3][2][2];
};

__device__ inline void load_row(RowFrag &f, const __bf16 *__restrict__ in, bool plane, long rowbase, int x0,
                                int lane, int hi, int n1, int dil) {
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int m = 0; m < 2; m++) {
            int j1 = x0 + m * 32 + (lane & 31) + (d - 1) * dil;
            if (plane && j1 >= 0 && j1 < n1) {
                const bf16x8 *src = (const bf16x8 *)(in + (rowbase + j1) * C + hi * 16);
                f.a[d][m][0] = src[0];
                f.a[d][m][1] = src[1];
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    f.a[d][m][0][i] = (__bf16)0.0f;
                    f.a[d][m][1][i] = (__bf16)0.0f;
                }
            }
        }
}

template <int MODE>
__global__ void __launch_bounds__(CTB)
conv32(const __bf16 *__restrict__ in, const __bf16 *__restrict__ Wg, const float *__restrict__ bias,
       void *__restrict__ outp, const __bf16 *__restrict__ aux, int n1, int n2, int n3, int dil) {
    __shared__ bf16x8 wl[NT * C * C / 8];  // [27][h][hi][32 co] entries of 8 ci
    stage_weights(wl, Wg);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ntx = (n1 + 63) / 64, nty = (n2 + CW - 1) / CW;
    const long ntiles = (long)ntx * nty * n3;
    const long n12 = (long)n1 * n2;
    // tiles ordered column-major in i3 (item = column * n3 + i3); each block
    // walks a contiguous range, so consecutive tiles of a block share two of
    // their three input planes in its XCD's L2
    const long per = (ntiles + gridDim.x - 1) / gridDim.x;
    const long t_begin = (long)blockIdx.x * per, t_end = min(ntiles, t_begin + per);
    // K order of the two MFMAs of a tap: lane half hi holds input channels
    // hi*16 + [0, 8) for the first and hi*16 + [8, 16) for the second, so
    // each lane reads its 16 channels (32 bytes) of a voxel in one go.
    const int co = lane & 31, hi = lane >> 5;
    const float bco = (MODE == 2) ? 0.0f : bias[co];
    // the weights stay in LDS while the block walks over tiles; the A
    // fragments of the next (d2, d3) row of taps are loaded while the
    // current row's 12 MFMAs run
    for (long item = t_begin; item < t_end; item++) {
        const long col = item / n3;
        const int z = (int)(item % n3);
        const int x0 = (int)(col % ntx) * 64;
        const int y = (int)(col / ntx) * CW + w;
        f32x16 acc[2];
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[m][r] = 0.0f;
        const bool rowok = y < n2;
        RowFrag fa, fb;
        auto load = [&](RowFrag &f, int row) {
            int d2 = (row % 3 - 1) * dil, d3 = (row / 3 - 1) * dil;
            int j2 = y + d2, j3 = z + d3;
            bool plane = rowok && j2 >= 0 && j2 < n2 && j3 >= 0 && j3 < n3;
            load_row(f, in, plane, (long)j2 * n1 + (long)j3 * n12, x0, lane, hi, n1, dil);
        };
        auto compute = [&](const RowFrag &f, int row) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int t = row * 3 + d;
                const bf16x8 b0 = wl[wl_at(t, 0, hi, co)];
                const bf16x8 b1 = wl[wl_at(t, 1, hi, co)];
                // independent accumulators back to back (no dependent MFMA
                // pair); each accumulator still sums half 0 then half 1
#pragma unroll
                for (int m = 0; m < 2; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[d][m][0], b0, acc[m], 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 2; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[d][m][1], b1, acc[m], 0, 0, 0);
            }
        };
        load(fa, 0);
#pragma unroll 1
        for (int row = 0; row < 8; row += 2) {
            load(fb, row + 1);
            compute(fa, row);
            load(fa, row + 2);
            compute(fb, row + 1);
        }
        compute(fa, 8);
        if (!rowok) continue;
#pragma unroll
        for (int m = 0; m < 2; m++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                int rr = (r / 4) * 8 + hi * 4 + (r % 4);
                int i1 = x0 + m * 32 + rr;
                if (i1 >= n1) continue;
                long v = (long)i1 + (long)y * n1 + (long)z * n12;
                float s = acc[m][r] + bco;
                if (MODE == 0) {
                    ((__bf16 *)outp)[v * C + co] = (__bf16)fmaxf(s, 0.0f);
                } else if (MODE == 1) {
                    if (co < 2) ((float *)outp)[v * 2 + co] = s;
                } else {
                    float gate = (float)aux[v * C + co] > 0.0f ? 1.0f : 0.0f;
                    ((__bf16 *)outp)[v * C + co] = (__bf16)(s * gate);
                }
            }
        }
    }
}

// Wide-tile variant for small dilations: lane l of M-tile s holds voxel
// x0 + 4l + s (four interleaved M-tiles, 128 voxels along i1).  The input
// fragment of tile s and tap offset d1 is then the voxel group s + d1*dil,
// so one (d2, d3) row of taps needs only 4 + 2*dil distinct A fragments
// for its 12 MFMA pairs (against 12 in conv32): half the operand loads for
// dil = 1.  The accumulation order per output is that of conv32, so both
// give identical results.
template <int DIL>
struct RowFragW {
    bf16x8 a[4 + 2 * DIL][2];
};

template <int DIL>
__device__ inline void load_row_w(RowFragW<DIL> &f, const __bf16 *__restrict__ in, bool plane, long rowbase, int x0,
                                  int lane, int hi, int n1) {
#pragma unroll
    for (int g = 0; g < 4 + 2 * DIL; g++) {
        int j1 = x0 + 4 * (lane & 31) + g - DIL;
        if (plane && j1 >= 0 && j1 < n1) {
            const bf16x8 *src = (const bf16x8 *)(in + (rowbase + j1) * C + hi * 16);
            f.a[g][0] = src[0];
            f.a[g][1] = src[1];
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                f.a[g][0][i] = (__bf16)0.0f;
                f.a[g][1][i] = (__bf16)0.0f;
            }
        }
    }
}

template <int MODE, int DIL>
__global__ void __launch_bounds__(CTB)
conv32w(const __bf16 *__restrict__ in, const __bf16 *__restrict__ Wg, const float *__restrict__ bias,
        void *__restrict__ outp, const __bf16 *__restrict__ aux, int n1, int n2, int n3) {
    __shared__ bf16x8 wl[NT * C * C / 8];  // [27][h][hi][32 co] entries of 8 ci
    stage_weights(wl, Wg);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ntx = (n1 + 127) / 128, nty = (n2 + CW - 1) / CW;
    const long ntiles = (long)ntx * nty * n3;
    const long n12 = (long)n1 * n2;
    const long per = (ntiles + gridDim.x - 1) / gridDim.x;
    const long t_begin = (long)blockIdx.x * per, t_end = min(ntiles, t_begin + per);
    const int co = lane & 31, hi = lane >> 5;
    const float bco = (MODE == 2) ? 0.0f : bias[co];
    for (long item = t_begin; item < t_end; item++) {
        const long col = item / n3;
        const int z = (int)(item % n3);
        const int x0 = (int)(col % ntx) * 128;
        const int y = (int)(col / ntx) * CW + w;
        f32x16 acc[4];
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[m][r] = 0.0f;
        const bool rowok = y < n2;
        RowFragW<DIL> fa, fb;
        auto load = [&](RowFragW<DIL> &f, int row) {
            int d2 = (row % 3 - 1) * DIL, d3 = (row / 3 - 1) * DIL;
            int j2 = y + d2, j3 = z + d3;
            bool plane = rowok && j2 >= 0 && j2 < n2 && j3 >= 0 && j3 < n3;
            load_row_w<DIL>(f, in, plane, (long)j2 * n1 + (long)j3 * n12, x0, lane, hi, n1);
        };
        auto compute = [&](const RowFragW<DIL> &f, int row) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int t = row * 3 + d;
                const bf16x8 b0 = wl[wl_at(t, 0, hi, co)];
                const bf16x8 b1 = wl[wl_at(t, 1, hi, co)];
#pragma unroll
                for (int m = 0; m < 4; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[m + (d - 1) * DIL + DIL][0], b0, acc[m], 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 4; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[m + (d - 1) * DIL + DIL][1], b1, acc[m], 0, 0, 0);
            }
        };
        load(fa, 0);
#pragma unroll 1
        for (int row = 0; row < 8; row += 2) {
            load(fb, row + 1);
            compute(fa, row);
            load(fa, row + 2);
            compute(fb, row + 1);
        }
        compute(fa, 8);
        if (!rowok) continue;
#pragma unroll
        for (int m = 0; m < 4; m++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                int rr = (r / 4) * 8 + hi * 4 + (r % 4);
                int i1 = x0 + 4 * rr + m;
                if (i1 >= n1) continue;
                long v = (long)i1 + (long)y * n1 + (long)z * n12;
                float sv = acc[m][r] + bco;
                if (MODE == 0) {
                    ((__bf16 *)outp)[v * C + co] = (__bf16)fmaxf(sv, 0.0f);
                } else if (MODE == 1) {
                    if (co < 2) ((float *)outp)[v * 2 + co] = sv;
                } else {
                    float gate = (float)aux[v * C + co] > 0.0f ? 1.0f : 0.0f;
                    ((__bf16 *)outp)[v * C + co] = (__bf16)(sv * gate);
                }
            }
        }
    }
}

// Row of A fragments through a buffer resource: o1 = byte offset of voxel
// x0 + (lane & 31) of the row (+ the lane's channel half), BUF_OOB for a
// row outside the volume (the hardware returns zeros); xm bit m*3+d clears
// fragment (d, m) whose voxel lies outside [0, n1) along i1.
__device__ inline void load_row_b(RowFrag &f, __amdgpu_buffer_rsrc_t r, unsigned o1, unsigned xm) {
    const unsigned o0 = o1 - 64u;
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const unsigned o = (d == 0 ? o0 : o1) + m * 2048u + (d == 2 ? 64u : 0u);
            const bool ok = (xm >> (m * 3 + d)) & 1u;
            f.a[d][m][0] = ld_frag(r, o, ok);
            f.a[d][m][1] = ld_frag(r, o + 16u, ok);
        }
}

// Plane-scatter variant for dilation 1.  The block walks its z-range one
// INPUT plane at a time: the three (d2) rows of plane p are loaded once
// and feed the taps of the three outputs that read them, z = p + 1
// (d3 = -1), z = p (d3 = 0) and z = p - 1 (d3 = +1), held in three rolling
// accumulators; after plane p, output p - 1 is complete and is stored.
// Each input row is thus read once per block and z-range instead of three
// times, with 36 MFMAs per row load (12 in conv32).  Every output still
// sums its taps in conv32's order (rows (d3, d2) ascending, then d1, then
// the channel half), so both give identical results.  Rows are read and
// outputs written through buffer resources (one lane offset per row or
// plane plus immediates), which keeps the kernel within 256 VGPRs without
// spills; volumes need n * 64 bytes < 4e9.
template <int MODE>
__global__ void __launch_bounds__(CTB)
conv32z(const __bf16 *__restrict__ in, const __bf16 *__restrict__ Wg, const float *__restrict__ bias,
        void *__restrict__ outp, const __bf16 *__restrict__ aux, int n1, int n2, int n3) {
    __shared__ bf16x8 wl[NT * C * C / 8];  // [27][h][hi][32 co] entries of 8 ci
    stage_weights(wl, Wg);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ntx = (n1 + 63) / 64, nty = (n2 + CW - 1) / CW;
    const long ntiles = (long)ntx * nty * n3;
    const long n12 = (long)n1 * n2;
    const long per = (ntiles + gridDim.x - 1) / gridDim.x;
    const long t_begin = (long)blockIdx.x * per, t_end = min(ntiles, t_begin + per);
    const int co = lane & 31, hi = lane >> 5;
    const float bco = (MODE == 2) ? 0.0f : bias[co];
    const unsigned nvox = (unsigned)((long)n12 * n3);
    const __amdgpu_buffer_rsrc_t rin = buf_rsrc(in, nvox * 64u);
    const __amdgpu_buffer_rsrc_t rout = buf_rsrc(outp, nvox * (MODE == 1 ? 8u : 64u));
    const __amdgpu_buffer_rsrc_t raux = buf_rsrc(MODE == 2 ? (const void *)aux : (const void *)in, nvox * 64u);
    long item = t_begin;
    while (item < t_end) {
        // one segment: outputs z in [za, zb) of one column
        const long col = item / n3;
        const int za = (int)(item % n3);
        const int zb = (int)min<long>((long)n3, za + (t_end - item));
        item += zb - za;
        const int x0 = (int)(col % ntx) * 64;
        const int y = (int)(col / ntx) * CW + w;
        const bool rowok = y < n2;
        f32x16 alo[2], amid[2], ahi[2];  // outputs p - 1, p, p + 1
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                alo[m][r] = 0.0f;
                amid[m][r] = 0.0f;
                ahi[m][r] = 0.0f;
            }
        unsigned xm = 0;
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int d = 0; d < 3; d++)
                if ((unsigned)(x0 + m * 32 + (lane & 31) + d - 1) < (unsigned)n1) xm |= 1u << (m * 3 + d);
        const unsigned lb = (unsigned)(x0 + (lane & 31)) * 64u + (unsigned)hi * 32u;
        auto load = [&](RowFrag &f, int p, int r2) {
            int j2 = y + r2 - 1;
            bool plane = rowok && j2 >= 0 && j2 < n2 && p >= 0 && p < n3;
            unsigned o1 = plane ? lb + ((unsigned)j2 * (unsigned)n1 + (unsigned)p * (unsigned)n12) * 64u : BUF_OOB;
            load_row_b(f, rin, o1, xm);
        };
        // taps of row (d3, d2) = (row / 3 - 1, row % 3 - 1) into acc
        auto taps = [&](const RowFrag &f, int row, f32x16 *acc) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int t = row * 3 + d;
                const bf16x8 b0 = wl[wl_at(t, 0, hi, co)];
                const bf16x8 b1 = wl[wl_at(t, 1, hi, co)];
#pragma unroll
                for (int m = 0; m < 2; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[d][m][0], b0, acc[m], 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 2; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[d][m][1], b1, acc[m], 0, 0, 0);
            }
        };
        auto compute = [&](const RowFrag &f, int r2, bool dlo, bool dmid, bool dhi) {
            if (dhi) taps(f, r2, ahi);        // d3 = -1
            if (dmid) taps(f, 3 + r2, amid);  // d3 = 0
            if (dlo) taps(f, 6 + r2, alo);    // d3 = +1
        };
        // stores through buffer resources: one lane offset per plane plus
        // an immediate per element; the i1 tail tile checks each element
        const bool xfull = x0 + 64 <= n1;
        auto store = [&](const f32x16 *acc, int z) {
            if (!rowok) return;
            const unsigned vb = (unsigned)(x0 + hi * 4) + (unsigned)y * (unsigned)n1 + (unsigned)z * (unsigned)n12;
#pragma unroll
            for (int m = 0; m < 2; m++) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const unsigned e = (unsigned)(m * 32 + (r / 4) * 8 + (r % 4));
                    const bool ok = xfull || x0 + m * 32 + (r / 4) * 8 + hi * 4 + (r % 4) < n1;
                    float sv = acc[m][r] + bco;
                    if (MODE == 1) {
                        if (co < 2)
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sv), rout,
                                                                  ok ? (vb + e) * 8u + co * 4u : BUF_OOB, 0, 0);
                    } else {
                        const unsigned o = ok ? (vb + e) * 64u + co * 2u : BUF_OOB;
                        if (MODE == 2) {
                            unsigned short g = __builtin_amdgcn_raw_buffer_load_b16(raux, o, 0, 0);
                            sv = (float)__builtin_bit_cast(__bf16, g) > 0.0f ? sv : sv * 0.0f;
                        } else {
                            sv = fmaxf(sv, 0.0f);
                        }
                        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (__bf16)sv), rout, o, 0,
                                                              0);
                    }
                }
            }
        };
        // one input plane; f0 holds its row 0 on entry, f1 holds the next
        // plane's row 0 on exit
        auto plane = [&](RowFrag &f0, RowFrag &f1, int p) {
            const bool dlo = p - 1 >= za, dmid = p >= za && p < zb, dhi = p + 1 < zb;
            load(f1, p, 1);
            compute(f0, 0, dlo, dmid, dhi);
            load(f0, p, 2);
            compute(f1, 1, dlo, dmid, dhi);
            load(f1, p + 1, 0);
            compute(f0, 2, dlo, dmid, dhi);
            if (dlo) store(alo, p - 1);
#pragma unroll
            for (int m = 0; m < 2; m++) {
                alo[m] = amid[m];
                amid[m] = ahi[m];
#pragma unroll
                for (int r = 0; r < 16; r++) ahi[m][r] = 0.0f;
            }
        };
        RowFrag fa, fb;
        load(fa, za - 1, 0);
#pragma unroll 1
        for (int p = za - 1; p <= zb; p += 2) {
            plane(fa, fb, p);
            if (p + 1 > zb) break;
            plane(fb, fa, p + 1);
        }
    }
}

// Input gradient of layer 1's output when layer 2 is the consumer is given
// by conv32<2>; layer 1 needs no input gradient.

// ---------------------------------------------------------------------------
// Weight gradient of a 32-channel layer: dW[t][ci][co] = sum_v in[v+t][ci]
// g[v][co], on the matrix cores with K = voxels.
//
// Both operands have K along the slow axis of the channels-last layout, so
// the tiles are staged as they lie ([voxel][32], 16-byte copies) and the
// fragments come out of LDS through the transposing read
// (ds_read_b64_tr_b16): a tap's shift is then a whole-voxel offset and every
// read stays aligned.  A block walks tiles of 64 (i1) x 4 (i2) voxels along
// i3 and keeps its sums in registers: wave (d2, kh) holds the nine taps of
// one i2 shift (144 accumulators) for the rows of one half of the tile, so
// at most WG_BLOCKS partials are written and reduced, whatever the volume.
// For dilation 1 the three input planes are a ring in LDS and the next
// plane and gradient tile are loaded into registers while the current one is
// multiplied; larger dilations stage one plane at a time.
// 64^3, one layer: 144 us (2-byte staging, eight 2-byte LDS reads per
// fragment, 1024 partials) + 238 us (their serial sum) before.
// ---------------------------------------------------------------------------
constexpr int WG_X = 64, WG_Y = 4, WG_TB = 384, WG_BLOCKS = 256;
constexpr int MAX_DIL = 8;
constexpr int WG_PART = NT * C * C + C;  // one block's partial: weights, then bias
constexpr int WG_GCH = WG_X * WG_Y * 4;  // 16-byte chunks of a gradient tile

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// The 32 x 16 fragment (row = channel, k = voxel) of 16 consecutive voxels
// starting at p, p = [voxel][32] in LDS: lane l gets channel l & 31, voxels
// (l >> 5) * 8 + 0..7.  In each group of 16 lanes lane i supplies the 8 bytes
// of voxel i / 4, channels 4 (i % 4) .. +3, and receives channel i of the
// group's four voxels.  off = tr_off(lane), in elements.
__device__ inline int tr_off(int lane) {
    const int g = lane >> 4, i = lane & 15;
    return ((g >> 1) * 8 + (i >> 2)) * C + (g & 1) * 16 + (i & 3) * 4;
}
__device__ inline bf16x8 tr_frag(const __bf16 *p, int off) {
    const i16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + off));
    const i16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + off + 4 * C));
    const bf16x4 x = __builtin_bit_cast(bf16x4, a), y = __builtin_bit_cast(bf16x4, b);
    return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <bool RING>
__global__ void __launch_bounds__(WG_TB)
conv32_wgrad(const __bf16 *__restrict__ in, const __bf16 *__restrict__ g, float *__restrict__ part, int n1, int n2,
             int n3, int dil) {
    constexpr int RPL = (WG_X + 2) * (WG_Y + 2);  // voxels of a plane of the ring
    constexpr int NP = RING ? (RPL * 4 + WG_TB - 1) / WG_TB : 1, NG = (WG_GCH + WG_TB - 1) / WG_TB;
    __shared__ uint4 wg_lds[WG_GCH + (RING ? 3 * RPL : (WG_X + 2 * MAX_DIL) * (WG_Y + 2 * MAX_DIL)) * 4];
    const int HX = WG_X + 2 * dil, HY = WG_Y + 2 * dil, pl = HX * HY;
    uint4 *const gt = wg_lds, *const it = wg_lds + WG_GCH;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int d2 = w % 3, kh = w / 3;
    const int ntx = (n1 + WG_X - 1) / WG_X, nty = (n2 + WG_Y - 1) / WG_Y;
    const long n12 = (long)n1 * n2, ntiles = (long)ntx * nty * n3;
    const long per = (ntiles + gridDim.x - 1) / gridDim.x;
    long item = (long)blockIdx.x * per;
    const long end = min(ntiles, item + per);
    const int toff = tr_off(lane);
    const uint4 zero = {0u, 0u, 0u, 0u};
    f32x16 acc[9];
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    float bias = 0.0f;
    int x0 = 0, y0 = 0;
    // 16-byte chunk c of the input plane j3 / of the gradient tile at z
    auto in_chunk = [&](int c, int j3) -> uint4 {
        const int v = c >> 2, xx = v % HX, yy = v / HX;
        const int j1 = x0 - dil + xx, j2 = y0 - dil + yy;
        if (j1 < 0 || j1 >= n1 || j2 < 0 || j2 >= n2 || j3 < 0 || j3 >= n3) return zero;
        return reinterpret_cast<const uint4 *>(in)[((long)j1 + (long)j2 * n1 + (long)j3 * n12) * 4 + (c & 3)];
    };
    auto g_chunk = [&](int c, int z) -> uint4 {
        const int v = c >> 2, j1 = x0 + (v & (WG_X - 1)), j2 = y0 + v / WG_X;
        if (j1 >= n1 || j2 >= n2 || z >= n3) return zero;
        return reinterpret_cast<const uint4 *>(g)[((long)j1 + (long)j2 * n1 + (long)z * n12) * 4 + (c & 3)];
    };
    // the taps (d3 = zz - 1, this wave's d2) of the tile, its input plane at ip
    auto taps = [&](int zz, const __bf16 *ip) {
        const __bf16 *gp = reinterpret_cast<const __bf16 *>(gt);
#pragma unroll 1
        for (int yy = 2 * kh; yy < 2 * kh + 2; yy++)
#pragma unroll 2
            for (int xc = 0; xc < WG_X; xc += 16) {
                const bf16x8 b = tr_frag(gp + (yy * WG_X + xc) * C, toff);
                if (zz == 1 && d2 == 0) {
#pragma unroll
                    for (int i = 0; i < 8; i++) bias += (float)b[i];
                }
#pragma unroll
                for (int d1 = 0; d1 < 3; d1++) {
                    const bf16x8 a = tr_frag(ip + ((yy + d2 * dil) * HX + xc + d1 * dil) * C, toff);
                    if (zz == 0) acc[d1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[d1], 0, 0, 0);
                    else if (zz == 1) acc[3 + d1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[3 + d1], 0, 0, 0);
                    else acc[6 + d1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[6 + d1], 0, 0, 0);
                }
            }
    };
    while (item < end) {
        const long col = item / n3;
        const int za = (int)(item % n3), zb = (int)min<long>((long)n3, za + (end - item));
        item += zb - za;
        x0 = (int)(col % ntx) * WG_X;
        y0 = (int)(col / ntx) * WG_Y;
        if constexpr (RING) {
            __syncthreads();  // the previous column's readers are done
            for (int c = threadIdx.x; c < pl * 4; c += WG_TB) {
                it[((za + 2) % 3) * (RPL * 4) + c] = in_chunk(c, za - 1);
                it[(za % 3) * (RPL * 4) + c] = in_chunk(c, za);
            }
            uint4 pi[NP], pg[NG];
            auto fetch = [&](int z) {  // what tile z needs that is not in LDS yet
#pragma unroll
                for (int k = 0; k < NP; k++) {
                    const int c = threadIdx.x + k * WG_TB;
                    pi[k] = c < RPL * 4 ? in_chunk(c, z + 1) : zero;
                }
#pragma unroll
                for (int k = 0; k < NG; k++) {
                    const int c = threadIdx.x + k * WG_TB;
                    pg[k] = c < WG_GCH ? g_chunk(c, z) : zero;
                }
            };
            fetch(za);
#pragma unroll 1
            for (int z = za; z < zb; z++) {
                if (z > za) __syncthreads();
#pragma unroll
                for (int k = 0; k < NP; k++) {
                    const int c = threadIdx.x + k * WG_TB;
                    if (c < RPL * 4) it[((z + 1) % 3) * (RPL * 4) + c] = pi[k];
                }
#pragma unroll
                for (int k = 0; k < NG; k++) {
                    const int c = threadIdx.x + k * WG_TB;
                    if (c < WG_GCH) gt[c] = pg[k];
                }
                __syncthreads();
                if (z + 1 < zb) fetch(z + 1);
                const __bf16 *ip = reinterpret_cast<const __bf16 *>(it);
                taps(0, ip + ((z + 2) % 3) * (RPL * C));
                taps(1, ip + (z % 3) * (RPL * C));
                taps(2, ip + ((z + 1) % 3) * (RPL * C));
            }
        } else {
#pragma unroll 1
            for (int z = za; z < zb; z++) {
                auto plane = [&](int zz) {
                    __syncthreads();
                    if (zz == 0)
                        for (int c = threadIdx.x; c < WG_GCH; c += WG_TB) gt[c] = g_chunk(c, z);
                    for (int c = threadIdx.x; c < pl * 4; c += WG_TB) it[c] = in_chunk(c, z + (zz - 1) * dil);
                    __syncthreads();
                };
                plane(0);
                taps(0, reinterpret_cast<const __bf16 *>(it));
                plane(1);
                taps(1, reinterpret_cast<const __bf16 *>(it));
                plane(2);
                taps(2, reinterpret_cast<const __bf16 *>(it));
            }
        }
    }
    // the two halves' sums meet in LDS, three taps at a time (3 waves x 48 x
    // 64 floats = 36 KB, within the staging area)
    float *const sh = reinterpret_cast<float *>(wg_lds);
    float *const dst = part + (size_t)blockIdx.x * WG_PART;
    bias += __shfl_xor(bias, 32);  // the lane pair of a channel
    auto meet = [&](int zz, const f32x16 *a) {
        __syncthreads();
        if (kh == 1)
#pragma unroll
            for (int d1 = 0; d1 < 3; d1++)
#pragma unroll
                for (int r = 0; r < 16; r++) sh[(d2 * 48 + d1 * 16 + r) * 64 + lane] = a[d1][r];
        __syncthreads();
        if (kh == 0)
#pragma unroll
            for (int d1 = 0; d1 < 3; d1++)
#pragma unroll
                for (int r = 0; r < 16; r++) {  // D[row = ci][col = co]
                    const int ci = (r / 4) * 8 + (lane >> 5) * 4 + (r % 4), t = zz * 9 + d2 * 3 + d1;
                    dst[(t * C + ci) * C + (lane & 31)] = a[d1][r] + sh[(d2 * 48 + d1 * 16 + r) * 64 + lane];
                }
    };
    meet(0, acc);
    meet(1, acc + 3);
    meet(2, acc + 6);
    __syncthreads();
    if (d2 == 0 && kh == 1 && lane < C) sh[lane] = bias;
    __syncthreads();
    if (d2 == 0 && kh == 0 && lane < C) dst[NT * C * C + lane] = bias + sh[lane];
}

// Layer 1 weight gradient: dW1[t][co] = sum_v x[v+t] g1[v][co] in FP32 on the
// matrix cores (v_mfma_f32_32x32x2_f32): rows are the 27 taps and a row of
// ones for the bias, k = two voxels of a trace, columns the channels.  One
// wave takes whole traces, so the tests of a tap's i2 and i3 shift are made
// once a trace and its loads run along i1.  64^3: 408 us as one thread per
// (tap, channel) walking 256 voxels, before.
constexpr int C1_BLOCKS = 512;
constexpr int C1_PART = (NT + 1) * C;
__global__ void __launch_bounds__(TB)
conv1_wgrad(const float *__restrict__ x, float xscale, const __bf16 *__restrict__ g, float *__restrict__ part, int n1,
            int n2, int n3, int dil) {
    __shared__ float sh[4][C * C];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t = lane & 31, hi = lane >> 5, co = t;
    const int d1 = (t % 3 - 1) * dil, d2 = ((t / 3) % 3 - 1) * dil, d3 = (t / 9 - 1) * dil;
    const long rows = (long)n2 * n3;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    for (long row = (long)blockIdx.x * 4 + w; row < rows; row += (long)gridDim.x * 4) {
        const int i2 = (int)(row % n2), i3 = (int)(row / n2), j2 = i2 + d2, j3 = i3 + d3;
        const bool ok = t < NT && j2 >= 0 && j2 < n2 && j3 >= 0 && j3 < n3;
        const float *xr = x + (ok ? ((long)j3 * n2 + j2) * n1 : 0);
        const __bf16 *gr = g + row * n1 * C + co;
        for (int v0 = 0; v0 < n1; v0 += 16) {
            float a[8], b[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int i1 = v0 + 2 * k + hi, j1 = i1 + d1;
                const bool in1 = i1 < n1, tap = ok && in1 && j1 >= 0 && j1 < n1;
                const float gv = (float)gr[(long)(in1 ? i1 : 0) * C], xv = xr[tap ? j1 : 0] * xscale;
                a[k] = tap ? xv : (t == NT ? 1.0f : 0.0f);
                b[k] = in1 ? gv : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 8; k++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k], b[k], acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; r++) sh[w][((r / 4) * 8 + hi * 4 + (r % 4)) * C + co] = acc[r];
    __syncthreads();
    for (int i = threadIdx.x; i < C1_PART; i += TB)
        part[(size_t)blockIdx.x * C1_PART + i] = ((sh[0][i] + sh[1][i]) + sh[2][i]) + sh[3][i];
}

// Sum block partials (fixed order) and scatter into the gradient vector.
// A thread takes four neighbouring sums of every RG-th partial, the RG
// threads of those sums meet in LDS: the partials are read by enough threads
// to stream them (one thread per sum over all of them took 238 us for the
// 1024 partials of a 64^3 layer).
// mode 0: 32-channel layer: part [nblk][27][32 ci][32 co] + bias [32]
//         -> G[off + (t*32+ci)*32+co], G[off + 27*1024 + co] (bias)
// mode 1: final layer (co < 2): -> G[OFF_W6 + (t*32+ci)*2+co], G[OFF_B6+co]
// mode 2: layer 1: part [nblk][27*32 + 32] -> G[OFF_W1..], G[OFF_B1..]
constexpr int RG = 16;
__global__ void __launch_bounds__(TB)
reduce_wgrad(const float *__restrict__ part, int nblk, int size, int mode, long off, float *__restrict__ G) {
    __shared__ float4 sh[RG][TB / RG];
    const int u = threadIdx.x % (TB / RG), grp = threadIdx.x / (TB / RG);
    const int i4 = blockIdx.x * (TB / RG) + u;
    float4 s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i4 * 4 < size) {
        const float4 *p = reinterpret_cast<const float4 *>(part) + i4;
        const long st = size / 4;
#pragma unroll 8
        for (int b = grp; b < nblk; b += RG) {
            const float4 v = p[b * st];
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
    }
    sh[grp][u] = s;
    __syncthreads();
    if (grp || i4 * 4 >= size) return;
    float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k = 0; k < RG; k++) {
        const float4 v = sh[k][u];
        o[0] += v.x;
        o[1] += v.y;
        o[2] += v.z;
        o[3] += v.w;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int i = i4 * 4 + e;
        if (mode == 2) G[i < NT * C ? OFF_W1 + i : OFF_B1 + (i - NT * C)] = o[e];
        else if (mode == 0) G[off + i] = o[e];
        else if (i % C < 2) G[i < NT * C * C ? OFF_W6 + (i / C) * 2 + i % C : OFF_B6 + i % C] = o[e];
    }
}

// Loss gradient: gy = 2 (y - t) m / count (BF16, padded to 32 channels),
// partial sums of (y - t)^2 m.
__global__ void __launch_bounds__(TB)
loss_grad(const float *__restrict__ y, const float *__restrict__ tgt, const float *__restrict__ wt,
          __bf16 *__restrict__ gy, long n, float scale, double *part) {
    __shared__ double sh[16];
    long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double acc = 0.0;
    if (v < n) {
        float m = wt ? wt[v] : 1.0f;
        __bf16 *dst = gy + v * C;
        for (int c = 0; c < 2; c++) {
            float d = y[v * 2 + c] - tgt[c * n + v];
            dst[c] = (__bf16)(2.0f * d * m * scale);
            acc += (double)d * d * m;
        }
        for (int c = 2; c < C; c++) dst[c] = (__bf16)0.0f;
    }
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// Adam on the FP32 master parameters.
__global__ void adam_kernel(float *__restrict__ P, const float *__restrict__ G, float *__restrict__ M,
                            float *__restrict__ V, long n, float lr, float b1, float b2, float eps, float c1, float c2,
                            float wd) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float g = G[i] + wd * P[i];
    float m = b1 * M[i] + (1.0f - b1) * g;
    float v = b2 * V[i] + (1.0f - b2) * g * g;
    M[i] = m;
    V[i] = v;
    P[i] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

// 1 / RMS of x on the device (1 when x is all zero), in two launches: block
// partial sums of x^2 in double, then one block adds them in a fixed order.
__global__ void __launch_bounds__(TB) sumsq_partials(const float *__restrict__ x, long n, double *__restrict__ part) {
    __shared__ double sh[16];
    double s = 0.0;
    for (long i = (long)blockIdx.x * TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
        const double v = x[i];
        s += v * v;
    }
    const double t = block_sum(s, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ void __launch_bounds__(1024) inv_rms(const double *__restrict__ part, int nblk, long n,
                                                float *__restrict__ xs) {
    __shared__ double sh[16];
    double s = 0.0;
    for (int i = threadIdx.x; i < nblk; i += blockDim.x) s += part[i];
    const double t = block_sum(s, sh);
    if (threadIdx.x == 0) {
        const double rms = sqrt(t / (double)n);
        xs[0] = rms > 0.0 ? (float)(1.0 / rms) : 1.0f;
    }
}

// (y interleaved [v][2]) -> dips [2][v]
__global__ void split_dips(const float *__restrict__ y, float *__restrict__ out, long n) {
    long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    out[v] = y[v * 2];
    out[n + v] = y[v * 2 + 1];
}

struct CnnWork {
    __bf16 *Wf, *Wb;    // packed weights [5][27][32][32]
    __bf16 *act[6];     // layer outputs 1..5 (act[1..5]); act[0] unused
    float *y;           // [V][2]
    __bf16 *gA, *gB;    // gradient ping-pong [V][32]
    float *part;
    double *red, *dsum;
    int nblk_wg;
};

int cnn_work(sh_ctx *ctx, long n, bool train, CnnWork &W, int n1, int n2, int n3) {
    size_t wsz = (size_t)5 * NT * C * C * sizeof(__bf16);
    char *b = nullptr;
    size_t actsz = (size_t)n * C * sizeof(__bf16);
    size_t ysz = ((size_t)n * 2 * sizeof(float) + 255) / 256 * 256;  // keeps later buffers 16-byte aligned
    int nact = train ? 5 : 2;  // inference ping-pongs two buffers
    size_t need = 2 * wsz + (size_t)nact * actsz + ysz + (train ? 2 * actsz : 0);
    SH_TRY(sh_slot(ctx, SLOT_INTERP0 + 12, need, (void **)&b));
    W.Wf = (__bf16 *)b;
    W.Wb = (__bf16 *)(b + wsz);
    char *p = b + 2 * wsz;
    for (int l = 1; l <= 5; l++) W.act[l] = nullptr;
    if (train) {
        for (int l = 1; l <= 5; l++) { W.act[l] = (__bf16 *)p; p += actsz; }
    } else {
        W.act[1] = (__bf16 *)p; p += actsz;
        W.act[2] = (__bf16 *)p; p += actsz;
    }
    W.y = (float *)p; p += ysz;
    if (train) {
        W.gA = (__bf16 *)p; p += actsz;
        W.gB = (__bf16 *)p; p += actsz;
        const long tiles = (long)ceil_div(n1, WG_X) * ceil_div(n2, WG_Y) * n3;
        W.nblk_wg = (int)std::min<long>(tiles, WG_BLOCKS);
        SH_TRY(sh_slot(ctx, SLOT_INTERP0 + 13, (size_t)W.nblk_wg * WG_PART * sizeof(float), (void **)&W.part));
        SH_TRY(sh_slot(ctx, SLOT_INTERP0 + 14, (size_t)ceil_div(n, TB) * sizeof(double) + 64, (void **)&W.red));
        W.dsum = W.red + ceil_div(n, TB);
    }
    return SH_OK;
}

int conv_launch(sh_ctx *ctx, int mode, const __bf16 *in, const __bf16 *Wg, const float *bias, void *out,
                const __bf16 *aux, int n1, int n2, int n3, int dil, const char *name) {
    // persistent blocks: the 55 KB weight tile is staged once per block.
    // SH_CNN_CONV selects the dilation-1 kernel: z (default) plane-scatter,
    // w wide tiles, n the plain one (identical results, for timing)
    const char *cv = getenv("SH_CNN_CONV");
    const char kind = cv && cv[0] ? cv[0] : 'z';
    // (the plane-scatter kernel addresses its buffers with 32-bit offsets)
    if (dil == 1 && kind == 'z' && (double)n1 * n2 * n3 * 64.0 < 4.0e9) {
        long ntiles = (long)ceil_div(n1, 64) * ceil_div(n2, CW) * n3;
        // one block of 8 waves fits a CU: with fewer tiles than 4 per CU a
        // block takes at least two planes, so that it stages its weights
        // and reads shared input planes once for both (64^3: 512 tiles over
        // 256 blocks 28 us, over 512 blocks 40 us; over 128 blocks 36 us)
        const long want = std::max<long>(256, std::min<long>(1024, ntiles / 2));
        dim3 grid((unsigned)std::min<long>(ntiles, want));
        PROF_A(ctx);
        if (mode == 0)
            hipLaunchKernelGGL((conv32z<0>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3);
        else if (mode == 1)
            hipLaunchKernelGGL((conv32z<1>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3);
        else
            hipLaunchKernelGGL((conv32z<2>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3);
        double v = (double)n1 * n2 * n3;
        PROF_B(ctx, name, v * (64.0 + (mode == 1 ? 8.0 : 64.0) + (mode == 2 ? 64.0 : 0.0)));
        return sh_launch_check(ctx, name);
    }
    if (dil == 1 && kind == 'w') {  // wide tiles (half the operand loads)
        long ntiles = (long)ceil_div(n1, 128) * ceil_div(n2, CW) * n3;
        dim3 grid((unsigned)std::min<long>(ntiles, 1024));
        PROF_A(ctx);
#define CW_L(MM) hipLaunchKernelGGL((conv32w<MM, 1>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3)
        if (mode == 0) CW_L(0); else if (mode == 1) CW_L(1); else CW_L(2);
#undef CW_L
        double v = (double)n1 * n2 * n3;
        PROF_B(ctx, name, v * (64.0 + (mode == 1 ? 8.0 : 64.0) + (mode == 2 ? 64.0 : 0.0)));
        return sh_launch_check(ctx, name);
    }
    long ntiles = (long)ceil_div(n1, 64) * ceil_div(n2, CW) * n3;
    dim3 grid((unsigned)std::min<long>(ntiles, 1024));
    PROF_A(ctx);
    if (mode == 0)
        hipLaunchKernelGGL((conv32<0>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3, dil);
    else if (mode == 1)
        hipLaunchKernelGGL((conv32<1>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3, dil);
    else
        hipLaunchKernelGGL((conv32<2>), grid, dim3(CTB), 0, ctx->stream, in, Wg, bias, out, aux, n1, n2, n3, dil);
    double v = (double)n1 * n2 * n3;
    PROF_B(ctx, name, v * (64.0 + (mode == 1 ? 8.0 : 64.0) + (mode == 2 ? 64.0 : 0.0)));
    return sh_launch_check(ctx, name);
}

int cnn_forward(sh_ctx *ctx, const float *P, const float *x, float xscale, const int *D, int n1, int n2, int n3,
                CnnWork &W, bool train, const float *xsp = nullptr) {
    long n = (long)n1 * n2 * n3;
    long per = (long)NT * C * C;
    hipLaunchKernelGGL(pack_weights, dim3(ceil_div(5 * per, TB)), dim3(TB), 0, ctx->stream, P, W.Wf, W.Wb);
    SH_TRY(sh_launch_check(ctx, "pack_weights"));
    PROF_A(ctx);
    // SH_CNN_C1=g: the one-voxel-per-thread kernel with 27 global loads per
    // voxel instead of the LDS-staged one (identical results)
    const char *c1e = getenv("SH_CNN_C1");
    if (D[0] == 1 && !(c1e && c1e[0] == 'g')) {
        const long tiles = (long)ceil_div(n1, 64) * ceil_div(n2, 4);
        const int nseg = (int)std::max<long>(1, std::min<long>(n3 / 8, (2048 + tiles - 1) / tiles));
        const int seg = ceil_div(n3, nseg);
        hipLaunchKernelGGL(conv1_fwd_tile, dim3((unsigned)tiles, ceil_div(n3, seg)), dim3(TB), 0, ctx->stream, x, xscale,
                           P, W.act[1], n1, n2, n3, seg, xsp);
    } else {
        hipLaunchKernelGGL(conv1_fwd, dim3(ceil_div(n, TB)), dim3(TB), 0, ctx->stream, x, xscale, P, W.act[1], n1, n2,
                           n3, D[0], FastDiv((unsigned)n1), FastDiv((unsigned)n2), xsp);
    }
    PROF_B(ctx, "conv1_fwd", (double)n * (4.0 + 64.0));
    SH_TRY(sh_launch_check(ctx, "conv1_fwd"));
    __bf16 *cur = W.act[1];
    for (int l = 2; l <= 5; l++) {
        __bf16 *dst = train ? W.act[l] : (cur == W.act[1] ? W.act[2] : W.act[1]);
        SH_TRY(conv_launch(ctx, 0, cur, W.Wf + (size_t)(l - 2) * per, P + OFF_L(l) + per, dst, nullptr, n1, n2, n3,
                           D[l - 1], "conv32<relu>"));
        cur = dst;
    }
    return conv_launch(ctx, 1, cur, W.Wf + (size_t)4 * per, P + OFF_B6, W.y, nullptr, n1, n2, n3, D[5],
                       "conv32<final>");
}

// Per-layer dilations (NULL = all 1), each in [1, MAX_DIL].
int read_dil(sh_ctx *ctx, const int *dil, int *D) {
    for (int l = 0; l < 6; l++) {
        D[l] = dil ? dil[l] : 1;
        if (D[l] < 1 || D[l] > MAX_DIL) return sh_fail(ctx, SH_EINVAL, "cnn: dilation %d of layer %d not in 1..%d",
                                                       D[l], l + 1, MAX_DIL);
    }
    return SH_OK;
}

}  // namespace

extern "C" {

long sh_cnn_nparams(void) { return NPARAM; }

// Predict (inline, crossline) dips dip[2N] from the normalised volume x[N].
int sh_cnn_forward(sh_ctx *ctx, const float *params, const float *x, float xscale, const int *dil, int n1, int n2,
                   int n3, float *dip) {
    if (!ctx) return SH_ENULL;
    if (!params || !x || !dip) return sh_fail(ctx, SH_ENULL, "cnn_forward: NULL pointer");
    if (n1 < 1 || n2 < 1 || n3 < 1) return sh_fail(ctx, SH_EINVAL, "cnn_forward: bad shape");
    long n = (long)n1 * n2 * n3;
    int D[6];
    SH_TRY(read_dil(ctx, dil, D));
    CnnWork W{};
    SH_TRY(cnn_work(ctx, n, false, W, n1, n2, n3));
    float *xsp = nullptr;
    if (!(xscale > 0.0f)) {  // scale by 1 / RMS of x, computed here (no host round trip)
        const int nb = (int)std::min<long>(ceil_div(n, TB), 4096L);
        double *part = nullptr;
        SH_TRY(sh_slot(ctx, SLOT_INTERP0 + 16, (size_t)nb * sizeof(double) + 256, (void **)&part));
        xsp = (float *)(part + nb);
        hipLaunchKernelGGL(sumsq_partials, dim3(nb), dim3(TB), 0, ctx->stream, x, n, part);
        hipLaunchKernelGGL(inv_rms, dim3(1), dim3(1024), 0, ctx->stream, part, nb, n, xsp);
        SH_TRY(sh_launch_check(ctx, "inv_rms"));
    }
    SH_TRY(cnn_forward(ctx, params, x, xscale, D, n1, n2, n3, W, false, xsp));
    hipLaunchKernelGGL(split_dips, dim3(ceil_div(n, TB)), dim3(TB), 0, ctx->stream, W.y, dip, n);
    return sh_launch_check(ctx, "split_dips");
}

// Loss and gradient: loss = sum wt (y - target)^2 / count over both dip
// components (target [2][N], wt nullable weights [N]); grad[NPARAM] FP32.
int sh_cnn_grad(sh_ctx *ctx, const float *params, const float *x, float xscale, const int *dil, const float *target,
                const float *wt, int n1, int n2, int n3, float *grad, double *loss) {
    if (!ctx) return SH_ENULL;
    if (!params || !x || !target || !grad) return sh_fail(ctx, SH_ENULL, "cnn_grad: NULL pointer");
    if (n1 < 2 || n2 < 1 || n3 < 1) return sh_fail(ctx, SH_EINVAL, "cnn_grad: bad shape");
    long n = (long)n1 * n2 * n3;
    long per = (long)NT * C * C;
    int D[6];
    SH_TRY(read_dil(ctx, dil, D));
    CnnWork W{};
    SH_TRY(cnn_work(ctx, n, true, W, n1, n2, n3));
    SH_TRY(cnn_forward(ctx, params, x, xscale, D, n1, n2, n3, W, true));
    int nb = ceil_div(n, TB);
    float scale = 1.0f / (float)(2 * n);
    hipLaunchKernelGGL(loss_grad, dim3(nb), dim3(TB), 0, ctx->stream, W.y, target, wt, W.gA, n, scale, W.red);
    SH_TRY(sh_launch_check(ctx, "loss_grad"));
    if (loss) {
        double h = 0;
        SH_TRY(reduce_partials(ctx, W.red, nb, 1, W.dsum));
        SH_HIP(ctx, hipMemcpyAsync(&h, W.dsum, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        SH_HIP(ctx, hipStreamSynchronize(ctx->stream));
        *loss = h * (double)scale;
    }
    static_assert(WG_PART % 4 == 0 && C1_PART % 4 == 0, "the partials are read as float4");
    const int nred = ceil_div(WG_PART / 4, TB / RG);
    // layer 6 (input act5, output gradient gA)
    __bf16 *g = W.gA, *gn = W.gB;
    for (int l = 6; l >= 2; l--) {
        const __bf16 *ain = W.act[l - 1];
        const int dl = D[l - 1];
        PROF_A(ctx);
        if (dl == 1)
            hipLaunchKernelGGL(conv32_wgrad<true>, dim3(W.nblk_wg), dim3(WG_TB), 0, ctx->stream, ain, g,
                               W.part, n1, n2, n3, dl);
        else
            hipLaunchKernelGGL(conv32_wgrad<false>, dim3(W.nblk_wg), dim3(WG_TB), 0, ctx->stream, ain, g,
                               W.part, n1, n2, n3, dl);
        PROF_B(ctx, "conv32_wgrad", (double)n * 128.0);
        SH_TRY(sh_launch_check(ctx, "conv32_wgrad"));
        hipLaunchKernelGGL(reduce_wgrad, dim3(nred), dim3(TB), 0, ctx->stream, W.part, W.nblk_wg, WG_PART,
                           l == 6 ? 1 : 0, l == 6 ? 0L : OFF_L(l), grad);
        SH_TRY(sh_launch_check(ctx, "reduce_wgrad"));
        // input gradient through the ReLU of layer l-1
        SH_TRY(conv_launch(ctx, 2, g, W.Wb + (size_t)(l - 2) * per, nullptr, gn, ain, n1, n2, n3, D[l - 1],
                           "conv32<bwd>"));
        std::swap(g, gn);
    }
    // layer 1 weights
    const int nb1 = (int)std::min<long>(ceil_div((long)n2 * n3, 4), C1_BLOCKS);
    SH_TRY(sh_slot(ctx, SLOT_INTERP0 + 15, (size_t)nb1 * C1_PART * sizeof(float), (void **)&W.part));
    hipLaunchKernelGGL(conv1_wgrad, dim3(nb1), dim3(TB), 0, ctx->stream, x, xscale, g, W.part, n1, n2, n3, D[0]);
    SH_TRY(sh_launch_check(ctx, "conv1_wgrad"));
    hipLaunchKernelGGL(reduce_wgrad, dim3(ceil_div(C1_PART / 4, TB / RG)), dim3(TB), 0, ctx->stream, W.part, nb1,
                       C1_PART, 2, 0L, grad);
    return sh_launch_check(ctx, "reduce_wgrad");
}

int sh_cnn_adam(sh_ctx *ctx, float *params, const float *grad, float *m, float *v, float lr, float b1, float b2,
                float eps, int step, float wd) {
    if (!ctx) return SH_ENULL;
    if (!params || !grad || !m || !v || step < 1) return sh_fail(ctx, SH_EINVAL, "cnn_adam: bad arguments");
    float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(ceil_div(NPARAM, TB)), dim3(TB), 0, ctx->stream, params, grad, m, v, NPARAM,
                       lr, b1, b2, eps, c1, c2, wd);
    return sh_launch_check(ctx, "adam");
}

}  // extern "C"
