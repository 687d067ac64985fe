// nsg_cnn.hip -- BF16 MFMA kernels of the learned subgrid-stress network: convolution forward
// (implicit GEMM on v_mfma_f32_16x16x32_bf16), input gradients (the same kernel on flipped,
// transposed weights), weight gradients, MSE loss and Adam; the nsg_cnn_* C ABI.
//
// GEMM view of a convolution: M = points, N = output channels, K = 27 taps x CIN input channels,
// consumed 32 at a time.  MFMA operand layout (16x16x32 bf16): lane l holds A[l % 16][8 (l / 16) + j]
// and B[8 (l / 16) + j][l % 16], j = 0..7, and receives D[4 (l / 16) + i][l % 16], i = 0..3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "../../include/nsg.h"
#include "nsg_cnn.hpp"

using namespace nsgcnn;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned int)))) unsigned int u32x4;

namespace {

// weight gradients: tiles of 4 x 8 x 16 points (z fastest) and their halo
constexpr int TXT = 4, TYT = 8, TZT = 16;
constexpr int HX = TXT + 2, HY = TYT + 2, HZ = TZT + 2;
constexpr int TPTS = TXT * TYT * TZT;

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// the same rounding (to nearest, ties to even) by gfx950's conversion instruction
__device__ __forceinline__ uint16_t f2bf_hw(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// GELU of the forward convolution's epilogue, x Phi(x) = max(x, 0) - |x| erfc(|x| / sqrt 2) / 2,
// with erfc from Abramowitz & Stegun 7.1.26 (erfc(z) = t (a1 + t (a2 + t (a3 + t (a4 + t a5))))
// exp(-z^2), t = 1 / (1 + p z), absolute error <= 1.5e-7) written in w = x sqrt(log2(e) / 2), so
// that exp(-z^2) = exp2(-w^2) and p z = p' |w| with p' = p / sqrt(log2 e); the halves are folded
// into the coefficients.  One branch-free path of 14 instructions (hardware reciprocal and
// exponential); its difference from the erff form is far below half a bfloat16 unit of the
// rounded activation.
__device__ __forceinline__ float gelu_as(float x) {
    const float w = x * 0.84932180028801907f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.27273748087922250f, fabsf(w), 1.0f));
    const float q = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 0.5307027145f, -0.7265760135f), 0.7107068705f), -0.142248368f),
                             0.127414796f);
    const float e = __builtin_amdgcn_exp2f(-(w * w));
    return fmaf(-fabsf(x), q * e, fmaxf(x, 0.0f));
}
__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

__device__ __forceinline__ bf16x8 ld16(const uint16_t* p) { return __builtin_bit_cast(bf16x8, *(const u32x4*)p); }

// 16 bytes per lane from global memory to LDS at lds + 16 lane (lds wave-uniform), written in
// assembly so that the compiler does not track it: its own wait insertion treats any such copy as
// possibly aliasing every LDS read and would make the MFMA loop wait for the copies of the next
// item; the kernel waits for them itself.  No compiler-generated code in the kernels that use it
// keeps a value in M0.
__device__ __forceinline__ void dma16(const void* g, const uint16_t* lds) {
    const uint32_t off = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)lds;
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(off) : "memory");
}

// the same copy from base + off bytes (base wave-uniform, off < 2^32): the address is formed by
// the instruction (scalar base, 32-bit vector offset)
__device__ __forceinline__ void dma16o(const void* base, unsigned off, const uint16_t* lds) {
    const uint32_t l = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)lds;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(l) : "memory");
}

__device__ __forceinline__ int wrap(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

// decompose a tile index into its origin; tiles ordered z fastest
__device__ __forceinline__ void tile_origin(int t, int N, int& x0, int& y0, int& z0) {
    const int ntz = N / TZT, nty = N / TYT;
    z0 = (t % ntz) * TZT;
    t /= ntz;
    y0 = (t % nty) * TYT;
    x0 = (t / nty) * TXT;
}

enum Epi { EPI_GELU = 0, EPI_GELU_PRE = 1, EPI_LINEAR = 2, EPI_BWD_GELU = 3 };

struct ConvArgs {
    const uint16_t* in;   // [B][N^3][CIN] bf16
    const uint16_t* w;    // [COUT][27 CIN] bf16
    const float* bias;    // [COUT] (forward modes)
    const float* pre_in;  // EPI_BWD_GELU: pre-activation at the output points [B][N^3][COUT]
    uint16_t* act_out;    // bf16 output [B][N^3][COUT] (GELU modes, EPI_BWD_GELU)
    float* f_out;         // FP32 output [B][N^3][COUT] (EPI_GELU_PRE: pre-activation; EPI_LINEAR)
    int N;
};

// Convolution, persistent: the forward modes, and the input gradient (EPI_BWD_GELU: flipped,
// transposed weights, times GELU' of the stored pre-activation).  Blocks of 256 threads walk the (sample, tile)
// items of 4 x 4 x 16 output points, two blocks per CU.  The 6 x 6 x 18 periodic halo of an item
// goes from HBM to LDS through the global->LDS DMA (64 lanes x 16 bytes per instruction); a block
// has one halo buffer and a separate output tile, and copies the next item's halo as soon as every
// wavefront has read the current one, while its own epilogue (GELU, output tile, stores) runs; the
// two blocks of a CU drift apart, so one's epilogue and copies overlap the other's MFMAs.  The
// layer's weights stay in registers for the whole kernel: a wavefront holds 16 output channels'
// (with COUT = 32 the four wavefronts split them into two halves over 8 z-rows each, with 16 each
// holds them all over 4 z-rows), so LDS carries only the A operand.  The DMA writes each halo
// point's CIN channels contiguously (no padding), so the 16-byte chunks of a point are swizzled
// instead: chunk c of the point with halo z index hz sits in slot c ^ ((hz >> SH) & (CH - 1)),
// which puts the 8 points that one LDS cycle serves in distinct banks.  GEMM view per item:
// M = 256 points (16 z-rows), N = COUT, K = 27 taps x CIN in steps of 32.
// The input gradient's sums run over the taps in order (dx, dy, dz): walking the halo rows h = iy + dy
// of one dx, every z-row still meets its dy in order, and a fragment serves up to three z-rows while
// it is live.  Its pre-activations are read into registers before the next item's copies are issued.
// Input gradient, 64^3, batch 4: 226 -> 105 us (32 -> 32 channels), 139 -> 86 us (16 -> 32) against
// 512-thread blocks of one 4 x 8 x 16 tile, which staged halo and weights with every load waited for
// and read the pre-activations one by one; bound by the erff and expf of GELU' (33.5 M of each).
constexpr int PX = 4, PY = 4, PZ = 16;
constexpr int PHY = PY + 2, PHZ = PZ + 2, PHPTS = (PX + 2) * PHY * PHZ, PPTS = PX * PY * PZ;
constexpr int Q_THREADS = 256;

template <int CIN, int COUT, int EPI>
__global__ void __launch_bounds__(Q_THREADS, 2) conv3p_kernel(ConvArgs a, int ntile, int nitems) {
    constexpr bool BWD = EPI == EPI_BWD_GELU;
    constexpr int CH = CIN / 8;                  // 16-byte chunks per point
    constexpr int SH = (CH == 4) ? 1 : 2;        // swizzle shift (CH = 2 or 4)
    static_assert(CH == 2 || CH == 4, "CIN = 16 or 32");
    constexpr int KT = 27 * CIN, KSTEPS = (KT + 31) / 32, NH = COUT / 16;
    constexpr int NWAVE = Q_THREADS / 64;
    constexpr int HS = (NH >= 2) ? 2 : 1;        // channel groups of wavefronts
    constexpr int NHW = NH / HS;                 // 16-channel blocks per wavefront
    constexpr int SUB = PPTS / 16 / (NWAVE / HS);  // z-rows per wavefront
    constexpr int OS = COUT + 8;                 // output tile point stride (halfwords)
    constexpr int HB = PHPTS * CIN;              // halfwords of the halo buffer
    constexpr int NCHUNK = PHPTS * CH;
    constexpr int ROUNDS = (NCHUNK + Q_THREADS - 1) / Q_THREADS;
    constexpr int OT = (EPI != EPI_LINEAR) ? PPTS * OS : 8;  // bf16 output tile (GELU modes)
    __shared__ __attribute__((aligned(16))) uint16_t halo[HB];
    __shared__ __attribute__((aligned(16))) uint16_t outt[OT];
    const int N = a.N;
    const long long N3 = (long long)N * N * N;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int wrow = wv % (NWAVE / HS), hgrp = wv / (NWAVE / HS);  // z-rows wrow SUB .., channels hgrp NHW 16 ..

    // this thread's share of a halo copy, the same for every item: chunk f = (r NWAVE + wv) 64 + lane
    // is chunk src of halo point (hx, hy, hz), held as its byte offset from the point (x0 - 1,
    // y0 - 1, z0 - 1) without wrapping, 2 (((hx N + hy) N + hz) CIN + 8 src) (bits 0-25, N <= 256),
    // with flags for the halo faces that may wrap: hx = 0 (bit 26), hx = PX + 1 (27), hy = 0 (28),
    // hy = PY + 1 (29), hz = 0 (30), hz = PZ + 1 (31); ~0: past the halo.  Kept in LDS (each
    // thread reads back only its own entries): in registers they would spill, and a spill reload
    // waits for every copy in flight.
    const bool off32 = N <= 256;  // sample offsets fit 32 bits: 2 N^3 CIN bytes < 2^31
    constexpr int RFULL = NCHUNK / (NWAVE * 64);  // rounds with every lane inside the halo
    __shared__ unsigned hoff_t[ROUNDS * Q_THREADS];
    unsigned* hoff = hoff_t + threadIdx.x;  // entry r at hoff[r Q_THREADS]
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int f = (r * NWAVE + wv) * 64 + lane;
        if (f < NCHUNK) {
            const int q = f / CH, slot = f % CH;
            const int hz = q % PHZ, hy = (q / PHZ) % PHY, hx = q / (PHZ * PHY);
            const int src = slot ^ ((hz >> SH) & (CH - 1));
            hoff[r * Q_THREADS] = (unsigned)((2 * (((hx * N + hy) * N + hz) * CIN + src * 8)) & 0x3ffffff) |
                      ((unsigned)(hx == 0) << 26) | ((unsigned)(hx == PX + 1) << 27) | ((unsigned)(hy == 0) << 28) |
                      ((unsigned)(hy == PY + 1) << 29) | ((unsigned)(hz == 0) << 30) | ((unsigned)(hz == PZ + 1) << 31);
        } else {
            hoff[r * Q_THREADS] = ~0u;
        }
    }
    auto origin = [&](int item, int& b, int& x0, int& y0, int& z0) {
        b = item / ntile;
        int t = item % ntile;
        const int ntz = N / PZ, nty = N / PY;
        z0 = (t % ntz) * PZ;
        t /= ntz;
        y0 = (t % nty) * PY;
        x0 = (t / nty) * PX;
    };
    auto issue = [&](int item) {
        int b, x0, y0, z0;
        origin(item, b, x0, y0, z0);
        const uint16_t* in = a.in + (long long)b * N3 * CIN;
        if (off32) {
            // byte offset = the item's corner (x0 - 1, y0 - 1, z0 - 1), possibly negative, + the
            // lane's unwrapped offset + N along each axis whose face lies outside the box for this
            // item (0 or -1 masks from the face flags); three loops, by the axes that wrap
            const int ib = 2 * ((((x0 - 1) * N + (y0 - 1)) * N + (z0 - 1)) * CIN);
            const bool wxl = x0 == 0, wxh = x0 + PX == N, wyl = y0 == 0, wyh = y0 + PY == N;
            const bool wzl = z0 == 0, wzh = z0 + PZ == N;
            const int sx = 2 * N * N * CIN, sy = 2 * N * CIN, sz = 2 * CIN;
            auto one = [&](int r, unsigned d, unsigned off) {
                if (r < RFULL || d != ~0u) dma16o(in, off, halo + (r * NWAVE + wv) * 64 * 8);
            };
            if (!(wxl || wxh || wyl || wyh || wzl || wzh)) {
#pragma unroll
                for (int r = 0; r < ROUNDS; ++r) {
                    const unsigned d = hoff[r * Q_THREADS];
                    one(r, d, (d & 0x3ffffffu) + (unsigned)ib);
                }
            } else if (!(wxl || wxh || wyl || wyh) && wzl != wzh) {
                const int bz = wzl ? 30 : 31, cz = (wzl ? N : -N) * sz;
#pragma unroll
                for (int r = 0; r < ROUNDS; ++r) {
                    const unsigned d = hoff[r * Q_THREADS];
                    one(r, d, (d & 0x3ffffffu) + (unsigned)ib + (unsigned)(__builtin_amdgcn_sbfe((int)d, bz, 1) & cz));
                }
            } else {
                const int cxl = wxl ? N * sx : 0, cxh = wxh ? -N * sx : 0, cyl = wyl ? N * sy : 0;
                const int cyh = wyh ? -N * sy : 0, czl = wzl ? N * sz : 0, czh = wzh ? -N * sz : 0;
#pragma unroll
                for (int r = 0; r < ROUNDS; ++r) {
                    const unsigned d = hoff[r * Q_THREADS];
                    const int c = (__builtin_amdgcn_sbfe((int)d, 26, 1) & cxl) + (__builtin_amdgcn_sbfe((int)d, 27, 1) & cxh) +
                                  (__builtin_amdgcn_sbfe((int)d, 28, 1) & cyl) + (__builtin_amdgcn_sbfe((int)d, 29, 1) & cyh) +
                                  (__builtin_amdgcn_sbfe((int)d, 30, 1) & czl) + (__builtin_amdgcn_sbfe((int)d, 31, 1) & czh);
                    one(r, d, (d & 0x3ffffffu) + (unsigned)ib + (unsigned)c);
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const int f0 = (r * NWAVE + wv) * 64;
                int f = f0 + lane;
                asm volatile("" : "+v"(f));
                if (f < NCHUNK) {
                    const int q = f / CH, slot = f % CH;
                    const int hz = q % PHZ, hy = (q / PHZ) % PHY, hx = q / (PHZ * PHY);
                    const int src = slot ^ ((hz >> SH) & (CH - 1));
                    const int gx = wrap(x0 + hx - 1, N), gy = wrap(y0 + hy - 1, N), gz = wrap(z0 + hz - 1, N);
                    const uint16_t* gp = in + (((long long)gx * N + gy) * N + gz) * CIN + src * 8;
                    dma16((const void*)gp, halo + f0 * 8);
                }
            }
        }
    };

    // weights of K step ks: tap dx 9 + dy 3 + dz of the step's (dx, dz, dy) order for CIN = 32 (forward),
    // taps 2 ks, 2 ks + 1 for CIN = 16
    auto kmap = [](int ks) { return (CIN == 32) ? (ks / 9) * 9 + (ks % 3) * 3 + (ks / 3) % 3 : ks; };
    bf16x8 bw[KSTEPS][NHW];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        const int k0 = 32 * ks + 8 * g;
#pragma unroll
        for (int h = 0; h < NHW; ++h)
            bw[ks][h] = (k0 < KT) ? ld16(a.w + ((hgrp * NHW + h) * 16 + m) * KT + k0) : bf16x8{};
    }
    float bias[NHW];
#pragma unroll
    for (int h = 0; h < NHW; ++h) bias[h] = BWD ? 0.f : a.bias[(hgrp * NHW + h) * 16 + m];
    // halo z part of this lane's A fragment offsets: z index m + dz, chunk g (CIN = 32) or g % 2
    // (CIN = 16: lanes g >= 2 read the second tap of a K step)
    int zoff[3];
#pragma unroll
    for (int dz = 0; dz < 3; ++dz) {
        const int cc = (CH == 4) ? g : (g & 1);
        zoff[dz] = (m + dz) * CIN + ((cc ^ (((m + dz) >> SH) & (CH - 1))) * 8);
    }

    // Before an item: this wavefront's copies of its halo have landed (and its LDS accesses are
    // done), then every wavefront's.  The previous item's global stores, issued after those copies,
    // may stay in flight: the vector-memory counter completes in issue order, so waiting until at
    // most NST operations are outstanding (the stores one item issues) covers the copies.  The
    // first item also waits for the weight and bias reads.
    constexpr int NST = ((EPI != EPI_LINEAR) ? PPTS * (COUT / 8) / Q_THREADS : 0) + ((EPI == EPI_GELU_PRE || EPI == EPI_LINEAR) ? SUB * NHW * 4 : 0);
    static_assert(NST < 64, "vmcnt field");
    constexpr int WAIT_NST = (NST & 15) | (7 << 4) | ((NST >> 4) << 14);
    int item = blockIdx.x;
    if (item < nitems) issue(item);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    while (item < nitems) {
        __builtin_amdgcn_s_waitcnt(WAIT_NST);
        asm volatile("s_barrier" ::: "memory");
        floatx4 acc[SUB][NHW];
#pragma unroll
        for (int s2 = 0; s2 < SUB; ++s2)
#pragma unroll
            for (int h = 0; h < NHW; ++h) acc[s2][h] = floatx4{0.f, 0.f, 0.f, 0.f};
        floatx4 pre[BWD ? SUB : 1][BWD ? NHW : 1];
        if constexpr (BWD && CIN == 32) {
            static_assert(SUB % PY == 0, "whole x planes of z-rows per wavefront");
            constexpr int XP = SUB / PY;
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                for (int hy = 0; hy < PHY; ++hy) {
                    bf16x8 fr[XP][3];
#pragma unroll
                    for (int xp = 0; xp < XP; ++xp)
#pragma unroll
                        for (int dz = 0; dz < 3; ++dz)
                            fr[xp][dz] = ld16(halo + ((wrow * XP + xp + dx) * PHY + hy) * PHZ * CIN + zoff[dz]);
#pragma unroll
                    for (int iy = 0; iy < PY; ++iy) {
                        const int dy = hy - iy;
                        if (dy < 0 || dy > 2) continue;
#pragma unroll
                        for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                            for (int xp = 0; xp < XP; ++xp)
#pragma unroll
                                for (int h = 0; h < NHW; ++h)
                                    acc[xp * PY + iy][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                        fr[xp][dz], bw[dx * 9 + dy * 3 + dz][h], acc[xp * PY + iy][h], 0, 0, 0);
                    }
                }
        } else {
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            bf16x8 af[SUB];
#pragma unroll
            for (int s2 = 0; s2 < SUB; ++s2) {
                const int st = wrow * SUB + s2, ix = st / PY, iy = st % PY;
                if constexpr (CIN == 32) {
                    // K step ks = tap kmap(ks): the three dy taps of one (dx, dz) are consecutive,
                    // so a fragment shared by neighbouring z-rows is live for three steps only
                    const int dx = ks / 9, dz = (ks / 3) % 3, dy = ks % 3;
                    af[s2] = ld16(halo + ((ix + dx) * PHY + (iy + dy)) * PHZ * CIN + zoff[dz]);
                } else {
                    const int t0 = 2 * ks, t1 = 2 * ks + 1;
                    if (t1 < 27) {
                        const int o0 = ((ix + t0 / 9) * PHY + (iy + (t0 / 3) % 3)) * PHZ * CIN + zoff[t0 % 3];
                        const int o1 = ((ix + t1 / 9) * PHY + (iy + (t1 / 3) % 3)) * PHZ * CIN + zoff[t1 % 3];
                        af[s2] = ld16(halo + (g < 2 ? o0 : o1));
                    } else {
                        const int o0 = ((ix + t0 / 9) * PHY + (iy + (t0 / 3) % 3)) * PHZ * CIN + zoff[t0 % 3];
                        af[s2] = (g < 2) ? ld16(halo + o0) : bf16x8{};
                    }
                }
            }
#pragma unroll
            for (int s2 = 0; s2 < SUB; ++s2)
#pragma unroll
                for (int h = 0; h < NHW; ++h)
                    acc[s2][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[s2], bw[kmap(ks)][h], acc[s2][h], 0, 0, 0);
        }
        }
        if constexpr (BWD) {
            int b, x0, y0, z0;
            origin(item, b, x0, y0, z0);
#pragma unroll
            for (int s2 = 0; s2 < SUB; ++s2) {
                const int st = wrow * SUB + s2;
                const float* p = a.pre_in + ((long long)b * N3 + ((long long)(x0 + st / PY) * N + (y0 + st % PY)) * N + z0 + 4 * g) * COUT;
#pragma unroll
                for (int h = 0; h < NHW; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) pre[s2][h][i] = p[i * COUT + (hgrp * NHW + h) * 16 + m];
            }
        }
        if constexpr (BWD) {
            // the pre-activations have landed before the next item's copies are issued (a wait for them
            // afterwards would wait for the copies too)
#pragma unroll
            for (int s2 = 0; s2 < SUB; ++s2)
#pragma unroll
                for (int h = 0; h < NHW; ++h) asm volatile("" : "+v"(pre[s2][h]));
        }
        // every wavefront is done reading the halo: the next item's copy may overwrite it
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int nx = item + (int)gridDim.x;
        if (nx < nitems) issue(nx);
        int b, x0, y0, z0;
        origin(item, b, x0, y0, z0);
#pragma unroll
        for (int s2 = 0; s2 < SUB; ++s2) {
            const int st = wrow * SUB + s2, ix = st / PY, iy = st % PY;
            const long long row = (long long)b * N3 + ((long long)(x0 + ix) * N + (y0 + iy)) * N + z0;
#pragma unroll
            for (int h = 0; h < NHW; ++h) {
                const int co = (hgrp * NHW + h) * 16 + m;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const long long idx = (row + 4 * g + i) * COUT + co;
                    const int tp = st * PZ + 4 * g + i;
                    const float v = acc[s2][h][i] + bias[h];
                    if constexpr (BWD) {
                        outt[tp * OS + co] = f2bf_hw(acc[s2][h][i] * gelu_grad(pre[s2][h][i]));
                    } else if constexpr (EPI == EPI_GELU) {
                        outt[tp * OS + co] = f2bf_hw(gelu_as(v));
                    } else if constexpr (EPI == EPI_GELU_PRE) {
                        a.f_out[idx] = v;
                        outt[tp * OS + co] = f2bf_hw(gelu_as(v));
                    } else {
                        a.f_out[idx] = v;
                    }
                }
            }
        }
        if constexpr (EPI != EPI_LINEAR) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            constexpr int OC = COUT / 8;
#pragma unroll
            for (int j = 0; j < PPTS * OC / Q_THREADS; ++j) {
                const int i = j * Q_THREADS + threadIdx.x;
                const int tp = i / OC, c = i % OC;
                const int iz = tp % PZ, iy = (tp / PZ) % PY, ix = tp / (PZ * PY);
                const long long gp = (long long)b * N3 + ((long long)(x0 + ix) * N + (y0 + iy)) * N + (z0 + iz);
                *(u32x4*)(a.act_out + gp * COUT + c * 8) = *(const u32x4*)(outt + tp * OS + c * 8);
            }
        }
        item = nx;
    }
}

// Weight gradients: partial[blk][co][tap * CIN + ci] = sum over this block's points p of
// dp[p][co] * act[p + tap][ci], bpartial[blk][co] = sum dp[p][co].  GEMM view: M = COUT,
// N = 27 CIN, K = points (32 per MFMA, two z-rows).  Persistent over (tile, sample), one block per
// CU.  grid (wgrad_blocks); block 64 NWAVE
//
// Both MFMA operands run along the points, and the arrays are channels-last, so the tile is
// transposed on its way into LDS (a thread takes 8 channels of two z-neighbours and writes 8 dwords):
// lds [channel][halo row][24 z], ldd [channel][point].  An operand is then one 16-byte read per lane
// instead of eight 2-byte reads at a stride of CIN + 8 halfwords.  The three dz taps of one (dx, dy)
// share a read: dz = 0 is the 16 bytes at z0, dz = 2 the same shifted by a dword (one more dword
// read), dz = 1 a funnel shift of neighbouring dwords.  A wavefront owns GPW of the 9 CIN / 16
// (dx, dy, 16 channels) groups times QPW of the COUT / 16 row blocks; channel strides of 4 (mod 32)
// dwords put 8 consecutive channels' 16-byte reads in distinct banks.  The next tile's global reads
// are in flight (in registers) while this one is multiplied.  Every sum runs in the order of
// (tile, point): the wavefront layout does not enter the result.
// 64^3, batch 4: 201 -> 83 us (32 -> 32 channels; matrix-core time 23 us), 162 -> 56 (32 -> 16), 128
// -> 48 (16 -> 32), bound by the LDS operand reads and the staging writes between the two barriers of
// a tile; with the operands read in their own K step 139 / 82 / 63 us.
template <int CIN, int COUT> struct WgradShape {
    static constexpr int MT = COUT / 16;
    // 32 -> 32: 12 wavefronts of 3 groups and one row block (3 per SIMD); else 9 wavefronts
    static constexpr int NWAVE = (CIN == 32 && COUT == 32) ? 12 : 9;
    static constexpr int QPW = (CIN == 16) ? MT : 1;
    static constexpr int GPW = 9 * (CIN / 16) * (MT / QPW) / NWAVE;
    static constexpr int NT = 64 * NWAVE;
    static_assert(NWAVE * GPW * QPW == 9 * (CIN / 16) * MT, "every (group, row block) has one wavefront");
};

template <int CIN, int COUT>
__global__ void __launch_bounds__((WgradShape<CIN, COUT>::NT)) wgrad_kernel(const uint16_t* __restrict__ act,
                                                                          const uint16_t* __restrict__ dp,
                                                                          float* __restrict__ partial, float* __restrict__ bpartial,
                                                                          int N, int B) {
    using S = WgradShape<CIN, COUT>;
    constexpr int NT = S::NT, GPW = S::GPW, QPW = S::QPW, QSPLIT = S::MT / QPW;
    constexpr int KT = 27 * CIN;
    constexpr int ZS = 24;                       // halfwords per halo row (18 used)
    constexpr int SC = HX * HY * ZS + 8;         // halfwords per input channel
    constexpr int SPD = TPTS + 8;                // halfwords per output channel
    constexpr int CHI = CIN / 8, CHO = COUT / 8; // 16-byte chunks per point
    constexpr int HU = HX * HY * (HZ / 2) * CHI, HR = (HU + NT - 1) / NT;  // staging units (z pair, chunk), rounds
    constexpr int DU = (TPTS / 2) * CHO, DR = (DU + NT - 1) / NT;
    constexpr int BT = 512;                      // threads of the bias sums
    static_assert(NT >= BT, "bias sums");
    static_assert((SC / 2) % 32 % 8 == 4 && (SPD / 2) % 32 == 4 && HZ % 2 == 0, "bank spread");
    __shared__ __attribute__((aligned(16))) uint16_t lds[CIN * SC];
    __shared__ __attribute__((aligned(16))) uint16_t ldd[COUT * SPD];
    __shared__ float bred[BT];
    const long long N3 = (long long)N * N * N;
    const int ntiles = (N / TXT) * (N / TYT) * (N / TZT);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int q0 = (wv % QSPLIT) * QPW, g0 = (wv / QSPLIT) * GPW;  // first row block and group
    floatx4 acc[GPW][3][QPW];
#pragma unroll
    for (int u = 0; u < GPW; ++u)
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int q = 0; q < QPW; ++q) acc[u][z][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;
    const int bco = threadIdx.x % COUT;
    u32x4 ha[HR], hb[HR], da[DR], db[DR];  // the next tile's reads
    auto fetch = [&](int job) {
        const int b = job / ntiles, t = job % ntiles;
        int x0, y0, z0;
        tile_origin(t, N, x0, y0, z0);
        const uint16_t* src = act + (long long)b * N3 * CIN;
#pragma unroll
        for (int r = 0; r < HR; ++r) {
            const int i = r * NT + threadIdx.x;
            if (i < HU) {
                const int c = i % CHI, zp = (i / CHI) % (HZ / 2), row = i / (CHI * (HZ / 2));
                const int gx = wrap(x0 + row / HY - 1, N), gy = wrap(y0 + row % HY - 1, N);
                const int ga = wrap(z0 + 2 * zp - 1, N), gb = wrap(z0 + 2 * zp, N);
                const uint16_t* p = src + ((long long)gx * N + gy) * N * CIN + c * 8;
                ha[r] = *(const u32x4*)(p + ga * CIN);
                hb[r] = *(const u32x4*)(p + gb * CIN);
            }
        }
        const uint16_t* dsrc = dp + (long long)b * N3 * COUT;
#pragma unroll
        for (int r = 0; r < DR; ++r) {
            const int i = r * NT + threadIdx.x;
            if (i < DU) {
                const int c = i % CHO, p2 = 2 * (i / CHO);
                const int iz = p2 % TZT, iy = (p2 / TZT) % TYT, ix = p2 / (TZT * TYT);
                const uint16_t* p = dsrc + (((long long)(x0 + ix) * N + (y0 + iy)) * N + (z0 + iz)) * COUT + c * 8;
                da[r] = *(const u32x4*)p;
                db[r] = *(const u32x4*)(p + COUT);
            }
        }
    };
    // 8 channels of two z-neighbours -> one dword per channel
    auto spread = [](uint16_t* dst, int stride, u32x4 a, u32x4 b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *(uint32_t*)(dst + 2 * j * stride) = (a[j] & 0xffffu) | (b[j] << 16);
            *(uint32_t*)(dst + (2 * j + 1) * stride) = (a[j] >> 16) | (b[j] & 0xffff0000u);
        }
    };
    int job = blockIdx.x;
    if (job < ntiles * B) fetch(job);
    for (; job < ntiles * B; job += gridDim.x) {
        __syncthreads();  // previous tile's LDS reads are done
#pragma unroll
        for (int r = 0; r < HR; ++r) {
            const int i = r * NT + threadIdx.x;
            if (i < HU) {
                const int c = i % CHI, zp = (i / CHI) % (HZ / 2), row = i / (CHI * (HZ / 2));
                spread(lds + c * 8 * SC + row * ZS + 2 * zp, SC, ha[r], hb[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {
            const int i = r * NT + threadIdx.x;
            if (i < DU) spread(ldd + (i % CHO) * 8 * SPD + 2 * (i / CHO), SPD, da[r], db[r]);
        }
        __syncthreads();
        if (job + (int)gridDim.x < ntiles * B) fetch(job + gridDim.x);
        if (threadIdx.x < BT) {
            uint16_t d[COUT];  // read before they are added: the sum is a chain
#pragma unroll
            for (int k = 0; k < COUT; ++k) d[k] = ldd[bco * SPD + threadIdx.x / COUT + k * (BT / COUT)];
#pragma unroll
            for (int k = 0; k < COUT; ++k) bsum += bf2f(d[k]);
        }
        // this lane's 8 points: 32 ks + 8 g + j lie in one z-row (z = 8 (g & 1) + j)
        const uint16_t* pa = ldd + (q0 * 16 + m) * SPD + 8 * g;
        const uint16_t* pb[GPW];  // group: channels 16 (gr / 9) .., (dx, dy) = gr % 9
#pragma unroll
        for (int u = 0; u < GPW; ++u) {
            const int gr = g0 + u, xy = gr % 9;
            pb[u] = lds + ((gr / 9) * 16 + m) * SC + (xy / 3 * HY + xy % 3 + (g >> 1)) * ZS + (g & 1) * 8;
        }
        // operands of K step ks, read one step ahead of their use
        u32x4 af[2][QPW], w[2][GPW];
        uint32_t e[2][GPW];
        auto operands = [&](int ks) {
            const int ix = ks / (TYT / 2), iy = 2 * (ks % (TYT / 2));
#pragma unroll
            for (int q = 0; q < QPW; ++q) af[ks & 1][q] = *(const u32x4*)(pa + q * 16 * SPD + 32 * ks);
#pragma unroll
            for (int u = 0; u < GPW; ++u) {
                w[ks & 1][u] = *(const u32x4*)(pb[u] + (ix * HY + iy) * ZS);
                e[ks & 1][u] = *(const uint32_t*)(pb[u] + (ix * HY + iy) * ZS + 8);
            }
        };
        operands(0);
#pragma unroll
        for (int ks = 0; ks < TPTS / 32; ++ks) {
            if (ks + 1 < TPTS / 32) operands(ks + 1);
            const int k = ks & 1;
#pragma unroll
            for (int u = 0; u < GPW; ++u) {
                asm volatile("" : "+v"(w[k][u]), "+v"(e[k][u]));  // no second read of the shifted dwords
                const u32x4 a = w[k][u];
                const uint32_t x = e[k][u];
                const u32x4 f[3] = {a,
                                    u32x4{__builtin_amdgcn_alignbit(a[1], a[0], 16), __builtin_amdgcn_alignbit(a[2], a[1], 16),
                                          __builtin_amdgcn_alignbit(a[3], a[2], 16), __builtin_amdgcn_alignbit(x, a[3], 16)},
                                    u32x4{a[1], a[2], a[3], x}};
#pragma unroll
                for (int z = 0; z < 3; ++z)
#pragma unroll
                    for (int q = 0; q < QPW; ++q)
                        acc[u][z][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[k][q]),
                                                                              __builtin_bit_cast(bf16x8, f[z]), acc[u][z][q], 0, 0, 0);
            }
        }
    }
    // D[4 g + i][m] of (row block q, tap, 16 channels): co = 16 q + 4 g + i, column tap CIN + ci
    float* P = partial + (long long)blockIdx.x * COUT * KT;
#pragma unroll
    for (int u = 0; u < GPW; ++u)
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int q = 0; q < QPW; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int gr = g0 + u, col = ((gr % 9) * 3 + z) * CIN + (gr / 9) * 16 + m;
                    P[(long long)(16 * (q0 + q) + 4 * g + i) * KT + col] = acc[u][z][q][i];
                }
    if (threadIdx.x < BT) bred[threadIdx.x] = bsum;
    __syncthreads();
    if (threadIdx.x < COUT) {
        float s = 0.f;
        for (int k = threadIdx.x; k < BT; k += COUT) s += bred[k];
        bpartial[(long long)blockIdx.x * COUT + threadIdx.x] = s;
    }
}

// grad[e] = sum over blocks of layer l's partials (fixed order), e over every parameter of the master
// layout; layer l's partials are nblk copies of its lcount(l) entries at poff[l] (weights of all
// blocks, then biases of all blocks).  One element per thread, 64-thread blocks, 16 blocks' partials
// read before they are added: the sum is a chain over nblk values, and one read after another in 108
// blocks of 256 threads took 63 us per layer, this 8 (all four layers in one launch: 18 us)
constexpr int RED_T = 64;
struct ReduceArgs {
    const float* partial;
    long long poff[NLAYER];
    float* grad;
    int nblk;
};
__global__ void __launch_bounds__(RED_T) wgrad_reduce_kernel(ReduceArgs a) {
    const long long e = blockIdx.x * (long long)RED_T + threadIdx.x;
    if (e >= MASTER_COUNT) return;
    int l = 0;
    long long o = e;
#pragma unroll
    for (int q = 1; q < NLAYER; ++q)
        if (e >= loffset(q)) { l = q; o = e - loffset(q); }
    long long nw = wcount(0), nb = CPAD[1], po = a.poff[0];
#pragma unroll
    for (int q = 1; q < NLAYER; ++q)
        if (l == q) { nw = wcount(q); nb = CPAD[q + 1]; po = a.poff[q]; }
    const float* src = a.partial + po + (o < nw ? o : a.nblk * nw + (o - nw));
    const long long stride = o < nw ? nw : nb;
    constexpr int L = 16;
    float s = 0.f;
    int k = 0;
    for (; k + L <= a.nblk; k += L) {
        float v[L];
#pragma unroll
        for (int j = 0; j < L; ++j) v[j] = src[(k + j) * stride];
#pragma unroll
        for (int j = 0; j < L; ++j) s += v[j];
    }
    for (; k < a.nblk; ++k) s += src[k * stride];
    a.grad[e] = s;
}

// MSE: loss partials and dL/d(out) = 2 (out - t) / count as bf16 (16 channels, 6 used)
__global__ void __launch_bounds__(256) loss_kernel(const float* __restrict__ out, const float* __restrict__ t,
                                                   uint16_t* __restrict__ dp, double* __restrict__ lpart, long long npts,
                                                   double inv_count) {
    __shared__ double red[256];
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const floatx4 o4 = *(const floatx4*)(out + p * 16);
        const float2 o2 = *(const float2*)(out + p * 16 + 4);
        const float2 t0 = *(const float2*)(t + p * 6), t1 = *(const float2*)(t + p * 6 + 2), t2 = *(const float2*)(t + p * 6 + 4);
        const float d[6] = {o4[0] - t0.x, o4[1] - t0.y, o4[2] - t1.x, o4[3] - t1.y, o2.x - t2.x, o2.y - t2.y};
        uint32_t v[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            acc += (double)d[c] * d[c];
            v[c] = f2bf((float)(2.0 * d[c] * inv_count));
        }
        if (dp) {
            *(u32x4*)(dp + p * 16) = u32x4{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, 0u};
            *(u32x4*)(dp + p * 16 + 8) = u32x4{0u, 0u, 0u, 0u};
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

// loss[it] = mean over n partials (fixed tree).  A run of training steps is not interrupted to look
// at its losses: bad (if given) holds 1 + the first step of the run whose loss is not finite, 0 until
// then, and the updates from that step on leave the parameters alone
__global__ void __launch_bounds__(256) loss_sum_kernel(const double* __restrict__ p, int n, double inv_count, double* loss, int it,
                                                       int* bad) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += p[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double v = red[0] * inv_count;
        loss[it] = v;
        if (bad) {
            const int b = it == 0 ? 0 : *bad;
            *bad = b == 0 && !isfinite(v) ? it + 1 : b;
        }
    }
}

// Adam on the master parameters of every layer (padded entries are held at zero), then the bf16 copies
struct AdamArgs {
    float *p, *m, *v;
    const float* g;
    uint16_t *wf[NLAYER], *wb[NLAYER];
    const int* bad;                 // update only while *bad is 0
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 / (1 - b1^t), c2 = 1 / (1 - b2^t)
    int update;                     // 0: only refresh the bf16 copies
};
template <int L> __device__ __forceinline__ void adam_element(const AdamArgs& a, long long e) {
    constexpr int CI = CPAD[L], CO = CPAD[L + 1], KT = 27 * CI;
    constexpr int nw = CO * KT;
    const int o = (int)(e - loffset(L));
    bool valid;
    int co, K = 0;
    if (o < nw) {
        co = o / KT;
        K = o % KT;
        valid = co < CREAL[L + 1] && (K % CI) < CREAL[L];
    } else {
        co = o - nw;
        valid = co < CREAL[L + 1];
    }
    float p = a.p[e];
    if (a.update) {
        if (valid) {
            const float g = a.g[e];
            const float m = a.b1 * a.m[e] + (1.f - a.b1) * g;
            const float v = a.b2 * a.v[e] + (1.f - a.b2) * g * g;
            a.m[e] = m;
            a.v[e] = v;
            p -= a.lr * (m * a.c1) / (sqrtf(v * a.c2) + a.eps);
        } else {
            p = 0.f;
        }
        a.p[e] = p;
    }
    if (o < nw) {
        const uint16_t h = f2bf(p);
        a.wf[L][o] = h;
        const int tap = K / CI, ci = K % CI;
        a.wb[L][(long long)ci * 27 * CO + (26 - tap) * CO + co] = h;
    }
}
__global__ void adam_kernel(AdamArgs a) {
    const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (e >= MASTER_COUNT || (a.update && *a.bad)) return;
    if (e < loffset(1)) adam_element<0>(a, e);
    else if (e < loffset(2)) adam_element<1>(a, e);
    else if (e < loffset(3)) adam_element<2>(a, e);
    else adam_element<3>(a, e);
}

// a batch's inputs and targets from the resident samples: 16 bytes per thread and turn, sample
// blockIdx.y of the (at most GB) ones in the arguments (eight device-to-device copies took 96 us at
// 64^3, batch 4, one launch 20)
constexpr int GB = 16;
struct GatherArgs {
    const uint16_t* x[GB];
    const float* y[GB];
    uint16_t* dx;
    float* dy;
    long long N3;
};
__global__ void __launch_bounds__(256) gather_kernel(GatherArgs a) {
    const int b = blockIdx.y;
    const u32x4 *x = (const u32x4*)a.x[b], *y = (const u32x4*)a.y[b];
    u32x4 *dx = (u32x4*)a.dx + b * a.N3 * 2, *dy = (u32x4*)(a.dy + b * a.N3 * 6);
    const long long nx = a.N3 * 2, n = nx + a.N3 * 3 / 2;  // N^3 is a multiple of 4096
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += 256ll * gridDim.x) {
        if (i < nx) dx[i] = x[i];
        else dy[i - nx] = y[i - nx];
    }
}

// physical [n][9] -> normalised bf16 [n][16]; physical [n][6] -> normalised FP32 [n][6]
__global__ void pack_x_kernel(const float* __restrict__ x, uint16_t* __restrict__ out, long long n, float inv) {
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < n; p += (long long)gridDim.x * blockDim.x)
#pragma unroll
        for (int c = 0; c < 16; ++c) out[p * 16 + c] = c < 9 ? f2bf(x[p * 9 + c] * inv) : (uint16_t)0;
}
__global__ void pack_y_kernel(const float* __restrict__ y, float* __restrict__ out, long long n, float i0, float i1, float i2,
                              float i3, float i4, float i5) {
    const float inv[6] = {i0, i1, i2, i3, i4, i5};
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < n; p += (long long)gridDim.x * blockDim.x)
#pragma unroll
        for (int c = 0; c < 6; ++c) out[p * 6 + c] = y[p * 6 + c] * inv[c];
}
__global__ void unpack_out_kernel(const float* __restrict__ in, float* __restrict__ y, long long n) {
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < n; p += (long long)gridDim.x * blockDim.x)
#pragma unroll
        for (int c = 0; c < 6; ++c) y[p * 6 + c] = in[p * 16 + c];
}

int cfail(nsg_cnn* c, int code, const char* fmt, ...) __attribute__((format(printf, 3, 4)));
int cfail(nsg_cnn* c, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define CHK(c, expr)                                                                                           \
    do {                                                                                                       \
        hipError_t e_ = (expr);                                                                                \
        if (e_ != hipSuccess) return cfail((c), NSG_ERR_DEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)
#define LCHK(c) CHK(c, hipGetLastError())

constexpr int LOSS_BLOCKS = 1024;   // blocks of loss_kernel (64^3, batch 4: 52 us with 256 and scalar loads, 26 with 1024)

int ntiles(const nsg_cnn* c) { return (c->N / TXT) * (c->N / TYT) * (c->N / TZT); }

template <int CIN, int COUT, int EPI>
int launch_conv(nsg_cnn* c, hipStream_t s, int B, const ConvArgs& a) {
    const int nt = (c->N / PX) * (c->N / PY) * (c->N / PZ);
    const int items = nt * B;
    // two blocks per CU: one 64^3 forward took 0.071 ms against 0.081-0.087 ms with 1, 3, 4 or 6
    // blocks per CU, a batch of 8 0.355-0.360 ms against 0.37-0.51 ms
    const int blocks = std::min(items, 2 * c->ncu);
    hipLaunchKernelGGL((conv3p_kernel<CIN, COUT, EPI>), dim3(blocks), dim3(Q_THREADS), 0, s, a, nt, items);
    LCHK(c);
    return NSG_OK;
}

// blocks of the weight-gradient kernels (one without a tile would add zeros)
int wgrad_grid(const nsg_cnn* c, int B) { return std::min(c->wgrad_blocks, ntiles(c) * B); }
// layer l's partials start here (elements)
long long partial_offset(int nblk, int l) { return nblk * loffset(l); }

template <int CIN, int COUT>
int launch_wgrad(nsg_cnn* c, hipStream_t s, int B, const uint16_t* act, const uint16_t* dp, int layer) {
    const int nblk = wgrad_grid(c, B);
    float* part = c->partial + partial_offset(nblk, layer);
    hipLaunchKernelGGL((wgrad_kernel<CIN, COUT>), dim3(nblk), dim3((WgradShape<CIN, COUT>::NT)), 0, s, act, dp, part,
                       part + (size_t)nblk * COUT * 27 * CIN, c->N, B);
    LCHK(c);
    return NSG_OK;
}

int launch_reduce(nsg_cnn* c, hipStream_t s, int B) {
    ReduceArgs a;
    a.nblk = wgrad_grid(c, B);
    a.partial = c->partial;
    for (int l = 0; l < NLAYER; ++l) a.poff[l] = partial_offset(a.nblk, l);
    a.grad = c->grad;
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)((MASTER_COUNT + RED_T - 1) / RED_T)), dim3(RED_T), 0, s, a);
    LCHK(c);
    return NSG_OK;
}

int refresh_weights(nsg_cnn* c, hipStream_t s, bool update, float lr) {
    const float b1 = 0.9f, b2 = 0.999f;
    double c1 = 1.0, c2 = 1.0;
    if (update) {
        c->adam_t += 1;
        c1 = 1.0 / (1.0 - std::pow((double)b1, (double)c->adam_t));
        c2 = 1.0 / (1.0 - std::pow((double)b2, (double)c->adam_t));
    }
    AdamArgs a;
    a.p = c->master; a.m = c->adam_m; a.v = c->adam_v; a.g = c->grad;
    for (int l = 0; l < NLAYER; ++l) { a.wf[l] = c->wf[l]; a.wb[l] = c->wb[l]; }
    a.bad = c->bad;
    a.lr = lr; a.b1 = b1; a.b2 = b2; a.eps = 1e-8f; a.c1 = (float)c1; a.c2 = (float)c2;
    a.update = update ? 1 : 0;
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((MASTER_COUNT + 255) / 256)), dim3(256), 0, s, a);
    LCHK(c);
    return NSG_OK;
}

// loss of the batch into c->losses[it] and, if wanted, its gradient into dp[0]; no wait
int enqueue_loss(nsg_cnn* c, hipStream_t s, int B, bool want_grad, int it, int* bad) {
    const long long npts = (long long)B * c->N3;
    const double inv = 1.0 / (6.0 * (double)npts);
    hipLaunchKernelGGL(loss_kernel, dim3(LOSS_BLOCKS), dim3(256), 0, s, (const float*)c->out, (const float*)c->target,
                       want_grad ? c->dp[0] : (uint16_t*)nullptr, c->lpart, npts, inv);
    LCHK(c);
    hipLaunchKernelGGL(loss_sum_kernel, dim3(1), dim3(256), 0, s, (const double*)c->lpart, LOSS_BLOCKS, inv, c->losses, it, bad);
    LCHK(c);
    return NSG_OK;
}

int loss_dev(nsg_cnn* c, hipStream_t s, int B, bool want_grad, double* loss) {
    int rc = enqueue_loss(c, s, B, want_grad, 0, nullptr);
    if (rc) return rc;
    CHK(c, hipMemcpyAsync(loss, c->losses, sizeof(double), hipMemcpyDeviceToHost, s));
    CHK(c, hipStreamSynchronize(s));
    return NSG_OK;
}

// backward of the whole network from dp[0] = dL/d(out) (16 ch); gradients into c->grad
int backward_dev(nsg_cnn* c, hipStream_t s, int B) {
    int rc;
    // layer 4 (32 -> 16): weights, then dL/d(pre3) = (W4^T * dp) gelu'(pre3)
    if ((rc = launch_wgrad<32, 16>(c, s, B, c->act[3], c->dp[0], 3))) return rc;
    {
        ConvArgs a{c->dp[0], c->wb[3], nullptr, c->pre[2], c->dp[1], nullptr, c->N};
        if ((rc = launch_conv<16, 32, EPI_BWD_GELU>(c, s, B, a))) return rc;
    }
    if ((rc = launch_wgrad<32, 32>(c, s, B, c->act[2], c->dp[1], 2))) return rc;
    {
        ConvArgs a{c->dp[1], c->wb[2], nullptr, c->pre[1], c->dp[0], nullptr, c->N};
        if ((rc = launch_conv<32, 32, EPI_BWD_GELU>(c, s, B, a))) return rc;
    }
    if ((rc = launch_wgrad<32, 32>(c, s, B, c->act[1], c->dp[0], 1))) return rc;
    {
        ConvArgs a{c->dp[0], c->wb[1], nullptr, c->pre[0], c->dp[1], nullptr, c->N};
        if ((rc = launch_conv<32, 32, EPI_BWD_GELU>(c, s, B, a))) return rc;
    }
    if ((rc = launch_wgrad<16, 32>(c, s, B, c->act[0], c->dp[1], 0))) return rc;
    return launch_reduce(c, s, B);
}

// host parameter order (torch conv3d, unpadded) <-> padded master layout
void host_to_master(const float* in, std::vector<float>& m) {
    m.assign(MASTER_COUNT, 0.f);
    long long o = 0;
    for (int l = 0; l < NLAYER; ++l) {
        const int ci_r = CREAL[l], co_r = CREAL[l + 1], cin = CPAD[l];
        float* W = m.data() + loffset(l);
        for (int co = 0; co < co_r; ++co)
            for (int ci = 0; ci < ci_r; ++ci)
                for (int tap = 0; tap < 27; ++tap) W[(long long)co * 27 * cin + tap * cin + ci] = in[o++];
        for (int co = 0; co < co_r; ++co) W[wcount(l) + co] = in[o++];
    }
}
void master_to_host(const std::vector<float>& m, float* out) {
    long long o = 0;
    for (int l = 0; l < NLAYER; ++l) {
        const int ci_r = CREAL[l], co_r = CREAL[l + 1], cin = CPAD[l];
        const float* W = m.data() + loffset(l);
        for (int co = 0; co < co_r; ++co)
            for (int ci = 0; ci < ci_r; ++ci)
                for (int tap = 0; tap < 27; ++tap) out[o++] = W[(long long)co * 27 * cin + tap * cin + ci];
        for (int co = 0; co < co_r; ++co) out[o++] = W[wcount(l) + co];
    }
}

uint64_t splitmix(uint64_t& s) {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

void free_cnn(nsg_cnn* c) {
    void* bufs[] = {c->master, c->adam_m, c->adam_v, c->grad, c->out, c->target, c->partial, c->lpart, c->losses,
                    c->bad, c->dp[0], c->dp[1]};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    for (int l = 0; l < NLAYER; ++l) {
        if (c->wf[l]) (void)hipFree(c->wf[l]);
        if (c->wb[l]) (void)hipFree(c->wb[l]);
        if (c->act[l]) (void)hipFree(c->act[l]);
    }
    for (int l = 0; l < NLAYER - 1; ++l)
        if (c->pre[l]) (void)hipFree(c->pre[l]);
    for (auto* p : c->xs) (void)hipFree(p);
    for (auto* p : c->ys) (void)hipFree(p);
    for (auto& e : c->ev)
        if (e) (void)hipEventDestroy(e);
    if (c->s) (void)hipStreamDestroy(c->s);
}

int upload_batch(nsg_cnn* c, const float* x, const float* t, int B) {
    // host x [B][N^3][9] and t [B][N^3][6], already normalised
    const long long n = (long long)B * c->N3;
    float* hx = nullptr;
    CHK(c, hipMalloc(&hx, sizeof(float) * n * 9));
    hipError_t e = hipMemcpyAsync(hx, x, sizeof(float) * n * 9, hipMemcpyHostToDevice, c->s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(pack_x_kernel, dim3(1024), dim3(256), 0, c->s, (const float*)hx, c->act[0], n, 1.0f);
        e = hipGetLastError();
    }
    if (e == hipSuccess && t) e = hipMemcpyAsync(c->target, t, sizeof(float) * n * 6, hipMemcpyHostToDevice, c->s);
    if (e == hipSuccess) e = hipStreamSynchronize(c->s);
    (void)hipFree(hx);
    if (e != hipSuccess) return cfail(c, NSG_ERR_DEVICE, "batch upload failed: %s", hipGetErrorString(e));
    return NSG_OK;
}

}  // namespace

namespace nsgcnn {
int forward_dev(nsg_cnn* c, hipStream_t s, int B, bool train) {
    int rc;
    const float* bias[NLAYER];
    for (int l = 0; l < NLAYER; ++l) bias[l] = c->master + loffset(l) + wcount(l);
    if (train) {
        ConvArgs a1{c->act[0], c->wf[0], bias[0], nullptr, c->act[1], c->pre[0], c->N};
        if ((rc = launch_conv<16, 32, EPI_GELU_PRE>(c, s, B, a1))) return rc;
        ConvArgs a2{c->act[1], c->wf[1], bias[1], nullptr, c->act[2], c->pre[1], c->N};
        if ((rc = launch_conv<32, 32, EPI_GELU_PRE>(c, s, B, a2))) return rc;
        ConvArgs a3{c->act[2], c->wf[2], bias[2], nullptr, c->act[3], c->pre[2], c->N};
        if ((rc = launch_conv<32, 32, EPI_GELU_PRE>(c, s, B, a3))) return rc;
    } else {
        ConvArgs a1{c->act[0], c->wf[0], bias[0], nullptr, c->act[1], nullptr, c->N};
        if ((rc = launch_conv<16, 32, EPI_GELU>(c, s, B, a1))) return rc;
        ConvArgs a2{c->act[1], c->wf[1], bias[1], nullptr, c->act[2], nullptr, c->N};
        if ((rc = launch_conv<32, 32, EPI_GELU>(c, s, B, a2))) return rc;
        ConvArgs a3{c->act[2], c->wf[2], bias[2], nullptr, c->act[3], nullptr, c->N};
        if ((rc = launch_conv<32, 32, EPI_GELU>(c, s, B, a3))) return rc;
    }
    ConvArgs a4{c->act[3], c->wf[3], bias[3], nullptr, nullptr, c->out, c->N};
    return launch_conv<32, 16, EPI_LINEAR>(c, s, B, a4);
}
}  // namespace nsgcnn

// ------------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------------
long long nsg_cnn_param_count(void) { return PARAM_COUNT; }

const char* nsg_cnn_last_error(const nsg_cnn* c) { return c ? c->err.c_str() : "null network"; }

void nsg_cnn_destroy(nsg_cnn* c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->s) (void)hipStreamSynchronize(c->s);
    free_cnn(c);
    delete c;
}

int nsg_cnn_create(int N, int max_batch, uint64_t seed, int device, nsg_cnn** out) {
    if (!out) return NSG_ERR_INVALID;
    *out = nullptr;
    nsg_cnn* c = new (std::nothrow) nsg_cnn();
    if (!c) return NSG_ERR_OOM;
    *out = c;
    if (N < 16 || N % 16 != 0) return cfail(c, NSG_ERR_INVALID, "grid N=%d must be a multiple of 16", N);
    if (max_batch < 1) return cfail(c, NSG_ERR_INVALID, "max_batch must be >= 1");
    c->device = device;
    c->N = N;
    c->maxB = max_batch;
    c->N3 = (long long)N * N * N;
    CHK(c, hipSetDevice(device));
    CHK(c, hipStreamCreateWithFlags(&c->s, hipStreamNonBlocking));
    CHK(c, hipEventCreate(&c->ev[0]));
    CHK(c, hipEventCreate(&c->ev[1]));
    {
        hipDeviceProp_t prop;
        CHK(c, hipGetDeviceProperties(&prop, device));
        c->wgrad_blocks = std::max(64, prop.multiProcessorCount);
        c->ncu = std::max(1, prop.multiProcessorCount);
    }
    const long long np = (long long)max_batch * c->N3;
    auto alloc = [&](void** p, size_t bytes) -> int {
        hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) return cfail(c, NSG_ERR_OOM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
        return (int)NSG_OK;
    };
    int rc;
    for (float** p : {&c->master, &c->adam_m, &c->adam_v, &c->grad})
        if ((rc = alloc((void**)p, sizeof(float) * MASTER_COUNT))) return rc;
    for (int l = 0; l < NLAYER; ++l) {
        if ((rc = alloc((void**)&c->wf[l], 2 * wcount(l)))) return rc;
        if ((rc = alloc((void**)&c->wb[l], 2 * wcount(l)))) return rc;
        if ((rc = alloc((void**)&c->act[l], 2 * np * CPAD[l]))) return rc;
    }
    for (int l = 0; l < NLAYER - 1; ++l)
        if ((rc = alloc((void**)&c->pre[l], 4 * np * 32))) return rc;
    if ((rc = alloc((void**)&c->out, 4 * np * 16))) return rc;
    if ((rc = alloc((void**)&c->target, 4 * np * 6))) return rc;
    for (int k = 0; k < 2; ++k)
        if ((rc = alloc((void**)&c->dp[k], 2 * np * 32))) return rc;
    c->partial_n = (size_t)c->wgrad_blocks * MASTER_COUNT;
    if ((rc = alloc((void**)&c->partial, sizeof(float) * c->partial_n))) return rc;
    if ((rc = alloc((void**)&c->lpart, sizeof(double) * LOSS_BLOCKS))) return rc;
    c->losses_n = 64;  // grown by nsg_cnn_train
    if ((rc = alloc((void**)&c->losses, sizeof(double) * c->losses_n))) return rc;
    if ((rc = alloc((void**)&c->bad, sizeof(int)))) return rc;
    CHK(c, hipMemset(c->adam_m, 0, sizeof(float) * MASTER_COUNT));
    CHK(c, hipMemset(c->adam_v, 0, sizeof(float) * MASTER_COUNT));
    CHK(c, hipMemset(c->grad, 0, sizeof(float) * MASTER_COUNT));
    CHK(c, hipMemset(c->act[0], 0, 2 * np * 16));
    CHK(c, hipMemset(c->bad, 0, sizeof(int)));
    CHK(c, hipDeviceSynchronize());
    // torch's default conv initialisation: U(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
    std::vector<float> h(PARAM_COUNT);
    uint64_t st = seed;
    long long o = 0;
    for (int l = 0; l < NLAYER; ++l) {
        const double bound = 1.0 / std::sqrt(27.0 * CREAL[l]);
        for (long long k = 0; k < rcount(l); ++k) {
            const double u = (double)(splitmix(st) >> 11) * (1.0 / 9007199254740992.0);
            h[o++] = (float)((2.0 * u - 1.0) * bound);
        }
    }
    return nsg_cnn_set_params(c, h.data());
}

int nsg_cnn_set_params(nsg_cnn* c, const float* params) {
    if (!c || !params) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    std::vector<float> m;
    host_to_master(params, m);
    CHK(c, hipMemcpyAsync(c->master, m.data(), sizeof(float) * MASTER_COUNT, hipMemcpyHostToDevice, c->s));
    int rc = refresh_weights(c, c->s, false, 0.f);
    if (rc) return rc;
    CHK(c, hipStreamSynchronize(c->s));
    return NSG_OK;
}

int nsg_cnn_get_params(nsg_cnn* c, float* params) {
    if (!c || !params) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    std::vector<float> m(MASTER_COUNT);
    CHK(c, hipMemcpyAsync(m.data(), c->master, sizeof(float) * MASTER_COUNT, hipMemcpyDeviceToHost, c->s));
    CHK(c, hipStreamSynchronize(c->s));
    master_to_host(m, params);
    return NSG_OK;
}

int nsg_cnn_set_norm(nsg_cnn* c, double sigma_in, const double* sigma_out) {
    if (!c || !(sigma_in > 0.0) || !sigma_out) return NSG_ERR_INVALID;
    for (int k = 0; k < 6; ++k)
        if (!(sigma_out[k] > 0.0)) return cfail(c, NSG_ERR_INVALID, "sigma_out[%d] must be > 0", k);
    if (!c->xs.empty()) return cfail(c, NSG_ERR_INVALID, "set the normalisation before adding samples");
    c->sig_in = sigma_in;
    for (int k = 0; k < 6; ++k) c->sig_out[k] = sigma_out[k];
    return NSG_OK;
}

int nsg_cnn_get_norm(const nsg_cnn* c, double* sigma_in, double* sigma_out) {
    if (!c) return NSG_ERR_INVALID;
    if (sigma_in) *sigma_in = c->sig_in;
    if (sigma_out)
        for (int k = 0; k < 6; ++k) sigma_out[k] = c->sig_out[k];
    return NSG_OK;
}

int nsg_cnn_forward(nsg_cnn* c, const float* x, int B, float* y) {
    if (!c || !x || !y || B < 1 || B > c->maxB) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    int rc = upload_batch(c, x, nullptr, B);
    if (rc) return rc;
    if ((rc = forward_dev(c, c->s, B, false))) return rc;
    const long long n = (long long)B * c->N3;
    float* hy = nullptr;
    CHK(c, hipMalloc(&hy, sizeof(float) * n * 6));
    hipLaunchKernelGGL(unpack_out_kernel, dim3(1024), dim3(256), 0, c->s, (const float*)c->out, hy, n);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(y, hy, sizeof(float) * n * 6, hipMemcpyDeviceToHost, c->s);
    if (e == hipSuccess) e = hipStreamSynchronize(c->s);
    (void)hipFree(hy);
    if (e != hipSuccess) return cfail(c, NSG_ERR_DEVICE, "forward failed: %s", hipGetErrorString(e));
    return NSG_OK;
}

int nsg_cnn_loss_grad(nsg_cnn* c, const float* x, const float* t, int B, double* loss, float* grads) {
    if (!c || !x || !t || !loss || B < 1 || B > c->maxB) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    int rc = upload_batch(c, x, t, B);
    if (rc) return rc;
    if ((rc = forward_dev(c, c->s, B, true))) return rc;
    if ((rc = loss_dev(c, c->s, B, grads != nullptr, loss))) return rc;
    if (!grads) return NSG_OK;
    if ((rc = backward_dev(c, c->s, B))) return rc;
    std::vector<float> m(MASTER_COUNT);
    CHK(c, hipMemcpyAsync(m.data(), c->grad, sizeof(float) * MASTER_COUNT, hipMemcpyDeviceToHost, c->s));
    CHK(c, hipStreamSynchronize(c->s));
    master_to_host(m, grads);
    return NSG_OK;
}

int nsg_cnn_add_sample(nsg_cnn* c, const float* x, const float* tau) {
    if (!c || !x || !tau) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    uint16_t* dx = nullptr;
    float* dy = nullptr;
    float* tmp = nullptr;
    const long long n = c->N3;
    CHK(c, hipMalloc(&dx, 2 * n * 16));
    c->xs.push_back(dx);
    CHK(c, hipMalloc(&dy, 4 * n * 6));
    c->ys.push_back(dy);
    CHK(c, hipMalloc(&tmp, 4 * n * 9));
    hipError_t e = hipMemcpyAsync(tmp, x, 4 * n * 9, hipMemcpyHostToDevice, c->s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(pack_x_kernel, dim3(1024), dim3(256), 0, c->s, (const float*)tmp, dx, n, (float)(1.0 / c->sig_in));
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(tmp, tau, 4 * n * 6, hipMemcpyHostToDevice, c->s);
    if (e == hipSuccess) {
        const double* so = c->sig_out;
        hipLaunchKernelGGL(pack_y_kernel, dim3(1024), dim3(256), 0, c->s, (const float*)tmp, dy, n, (float)(1 / so[0]),
                           (float)(1 / so[1]), (float)(1 / so[2]), (float)(1 / so[3]), (float)(1 / so[4]), (float)(1 / so[5]));
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(c->s);
    (void)hipFree(tmp);
    if (e != hipSuccess) return cfail(c, NSG_ERR_DEVICE, "sample upload failed: %s", hipGetErrorString(e));
    return NSG_OK;
}

int nsg_cnn_sample_count(const nsg_cnn* c) { return c ? (int)c->xs.size() : 0; }

static int gather_batch(nsg_cnn* c, const int* idx, int B) {
    for (int b0 = 0; b0 < B; b0 += GB) {
        const int nb = std::min(GB, B - b0);
        GatherArgs a{};
        for (int b = 0; b < nb; ++b) { a.x[b] = c->xs[idx[b0 + b]]; a.y[b] = c->ys[idx[b0 + b]]; }
        a.dx = c->act[0] + (size_t)b0 * c->N3 * 16;
        a.dy = c->target + (size_t)b0 * c->N3 * 6;
        a.N3 = c->N3;
        const long long n = c->N3 * 7 / 2;  // 16-byte pieces of a sample
        hipLaunchKernelGGL(gather_kernel, dim3((unsigned)std::min<long long>((n + 255) / 256, 1024), nb), dim3(256), 0, c->s, a);
        LCHK(c);
    }
    return NSG_OK;
}

int nsg_cnn_train(nsg_cnn* c, int first, int count, int steps, int batch, double lr, uint64_t seed, double* loss_per_step) {
    if (!c || steps < 0 || batch < 1 || batch > c->maxB || !(lr > 0.0)) return NSG_ERR_INVALID;
    const int S = count;
    if (first < 0 || count < 1 || first + count > (int)c->xs.size())
        return cfail(c, NSG_ERR_INVALID, "sample range [%d, %d) outside the %d samples held", first, first + count, (int)c->xs.size());
    CHK(c, hipSetDevice(c->device));
    // the steps run to the end before the host looks at their losses (waiting for each step's loss
    // left the GPU idle for about 20 us a step); from a non-finite one on, the device leaves the
    // parameters alone, so they are what stopping at that step would leave
    constexpr int CHUNK = 4096;
    std::vector<double> h((size_t)std::min(steps, CHUNK));
    uint64_t st = seed;
    std::vector<int> idx(batch);
    for (int s0 = 0; s0 < steps; s0 += CHUNK) {
        const int n = std::min(CHUNK, steps - s0);
        if (c->losses_n < n) {
            double* p = nullptr;
            CHK(c, hipMalloc(&p, sizeof(double) * n));
            (void)hipFree(c->losses);
            c->losses = p;
            c->losses_n = n;
        }
        const long long t0 = c->adam_t;
        for (int it = 0; it < n; ++it) {
            for (int b = 0; b < batch; ++b) idx[b] = first + (int)(splitmix(st) % (uint64_t)S);
            int rc = gather_batch(c, idx.data(), batch);
            if (rc) return rc;
            if ((rc = forward_dev(c, c->s, batch, true))) return rc;
            if ((rc = enqueue_loss(c, c->s, batch, true, it, c->bad))) return rc;
            if ((rc = backward_dev(c, c->s, batch))) return rc;
            if ((rc = refresh_weights(c, c->s, true, (float)lr))) return rc;
        }
        int bad = 0;
        CHK(c, hipMemcpyAsync(h.data(), c->losses, sizeof(double) * n, hipMemcpyDeviceToHost, c->s));
        CHK(c, hipMemcpyAsync(&bad, c->bad, sizeof bad, hipMemcpyDeviceToHost, c->s));
        CHK(c, hipStreamSynchronize(c->s));
        const int done = bad ? bad - 1 : n;
        if (loss_per_step) std::copy(h.begin(), h.begin() + done, loss_per_step + s0);
        if (bad) {
            c->adam_t = t0 + done;
            return cfail(c, NSG_ERR_NONFINITE, "training loss is not finite at step %d", s0 + done);
        }
    }
    CHK(c, hipStreamSynchronize(c->s));
    return NSG_OK;
}

int nsg_cnn_eval(nsg_cnn* c, int first, int count, double* loss) {
    if (!c || !loss || first < 0 || count < 1 || first + count > (int)c->xs.size()) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    double tot = 0.0;
    for (int k = first; k < first + count; ++k) {
        int rc = gather_batch(c, &k, 1);
        if (rc) return rc;
        if ((rc = forward_dev(c, c->s, 1, false))) return rc;
        double l = 0.0;
        if ((rc = loss_dev(c, c->s, 1, false, &l))) return rc;
        tot += l;
    }
    *loss = tot / count;
    return NSG_OK;
}

int nsg_cnn_time_forward(nsg_cnn* c, int B, int iters, double* ms) {
    if (!c || !ms || B < 1 || B > c->maxB || iters < 1) return NSG_ERR_INVALID;
    CHK(c, hipSetDevice(c->device));
    int rc = forward_dev(c, c->s, B, false);
    if (rc) return rc;
    CHK(c, hipEventRecord(c->ev[0], c->s));
    for (int i = 0; i < iters; ++i)
        if ((rc = forward_dev(c, c->s, B, false))) return rc;
    CHK(c, hipEventRecord(c->ev[1], c->s));
    CHK(c, hipEventSynchronize(c->ev[1]));
    float f = 0.f;
    CHK(c, hipEventElapsedTime(&f, c->ev[0], c->ev[1]));
    *ms = f / iters;
    return NSG_OK;
}
