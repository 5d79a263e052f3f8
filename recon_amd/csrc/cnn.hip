// Pose-proposal network: forward and backward kernels on the CDNA4 matrix
// cores (bfloat16 operands, FP32 accumulation), Adam, and the C ABI of
// include/rt_cnn.h.
//
// Every convolution is an implicit GEMM over NHWC bfloat16 tensors. The
// forward pass of the default network (k_conv_fwd_mfma and its LDS-staged
// relatives) and the backward passes run on v_mfma_f32_16x16x32_bf16 (64-lane
// wave, A: 16 rows x 8 k per lane group, B: 8 k x 16 columns, D: 4 rows x 16
// columns per lane group); layers with 16 channels use
// v_mfma_f32_16x16x16_bf16 tiles (4 k per lane group):
//   forward      rows = output pixels (n, yo, xo), columns = Cout, k = (tap, Cin)
//   input grad   rows = input pixels (n, yi, xi),  columns = Cin,  k = (tap, Cout)
//   weight grad  rows = Cout, columns = (tap, Cin), k = output pixels, split
//                over workgroups and summed in a fixed order (deterministic)
// The head (global pooling, the 6-output dense layer, loss) is FP32.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/rt_cnn.h"
#include "cnn.hpp"
#include "rt_host.hpp"
#include "rt_stage.hpp"

namespace rt {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16 v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ bool bf_pos(bf16 v) { return !(v & 0x8000u) && v != 0; }

struct ConvGeom {
    int B, Hi, Wi, Ci, ci_shift, Ho, Wo, Co, co_shift, K, Kp;
};

__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

// ---------------------------------------------------------------- forward
// Block: 4 waves, 64 output pixels x 64 output channels; wave: 32 x 32.
__global__ __launch_bounds__(256) void k_conv_fwd(ConvGeom g, const bf16* __restrict__ X, const bf16* __restrict__ Wp,
                                                  const float* __restrict__ bias, bf16* __restrict__ Y) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = lane >> 4;
    const int M = g.B * g.Ho * g.Wo;
    const int row0 = blockIdx.x * 64 + (w & 1) * 32;
    const int col0 = blockIdx.y * 64 + (w >> 1) * 32;
    if (col0 >= g.Co || row0 >= M) return;
    const int HW = g.Ho * g.Wo;
    int nn[2], yo[2], xo[2];
    bool mv[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        int m = row0 + i * 16 + r16;
        mv[i] = m < M;
        int mm = mv[i] ? m : 0;
        nn[i] = mm / HW;
        int r = mm - nn[i] * HW;
        yo[i] = r / g.Wo;
        xo[i] = r - yo[i] * g.Wo;
    }
    f4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const s4 zero = {0, 0, 0, 0};
    for (int k0 = kq * 4; k0 < g.Kp; k0 += 16) {
        const int tap = k0 >> g.ci_shift, ci = k0 & (g.Ci - 1);
        const int ky = tap / 3, kx = tap - 3 * (tap / 3);
        s4 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            int yi = 2 * yo[i] - 1 + ky, xi = 2 * xo[i] - 1 + kx;
            bool ok = mv[i] && tap < 9 && yi >= 0 && yi < g.Hi && xi >= 0 && xi < g.Wi;
            a[i] = ok ? *(const s4*)(X + (((size_t)nn[i] * g.Hi + yi) * g.Wi + xi) * g.Ci + ci) : zero;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            int c = col0 + j * 16 + r16;
            b[j] = c < g.Co ? *(const s4*)(Wp + (size_t)c * g.Kp + k0) : zero;
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        int col = col0 + j * 16 + r16;
        if (col >= g.Co) continue;
        float bv = bias[col];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int m = row0 + i * 16 + kq * 4 + e;
                if (m < M) {
                    float v = acc[i][j][e] + bv;
                    Y[(size_t)m * g.Co + col] = f2bf(v > 0.0f ? v : 0.0f);
                }
            }
    }
}

// Forward on gfx950's v_mfma_f32_16x16x32_bf16 (A: row lane % 16, eight
// consecutive k per lane group lane / 16; B the same k for column lane % 16;
// D: rows 4 * (lane / 16) + i, column lane % 16). Each wave owns a 16*TM x
// 16*TN tile; four waves (WGM x WGN) form the workgroup. Operands come
// straight from global memory as 16-byte loads (an 8-channel run of one tap
// of one input pixel, or 8 k of one weight row; two taps of 4 channels when
// Cin = 4), the next k-step's loads issued before the current step's MFMAs.
// The bias, ReLU and bfloat16 rounding are applied to the accumulators, and
// the tile leaves through LDS as 16-byte row chunks.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f4 mfma32(bf8 a, bf8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <int TM, int TN, int WGM, int WGN, bool CI4>
__global__ __launch_bounds__(256) void k_conv_fwd_mfma(ConvGeom g, const bf16* __restrict__ X,
                                                       const bf16* __restrict__ Wp, const float* __restrict__ bias,
                                                       bf16* __restrict__ Y) {
    static_assert(WGM * WGN == 4, "four waves");
    constexpr int WM = 16 * TM, WN = 16 * TN, LDT = WN + 8;  // LDS row pitch (bf16)
    __shared__ __attribute__((aligned(16))) bf16 tile[4][WM * LDT];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int M = g.B * g.Ho * g.Wo, HW = g.Ho * g.Wo;
    const int row0 = blockIdx.x * (WM * WGM) + (w % WGM) * WM;
    const int col0 = blockIdx.y * (WN * WGN) + (w / WGM) * WN;
    int yb[TM], xb[TM];
    size_t nb[TM];
    bool mv[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) {
        const int m = row0 + 16 * t + r16;
        mv[t] = m < M;
        const int mm = mv[t] ? m : 0;
        const int n = mm / HW, r = mm - n * HW, yo = r / g.Wo, xo = r - yo * g.Wo;
        yb[t] = 2 * yo - 1;
        xb[t] = 2 * xo - 1;
        nb[t] = (size_t)n * g.Hi * g.Wi;
    }
    const bf16* wrow[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) wrow[j] = Wp + (size_t)(col0 + 16 * j + r16) * g.Kp + 8 * kg;
    auto tap_ok = [&](int t, int tap, size_t& off) {
        const int ky = tap / 3, kx = tap - 3 * (tap / 3);
        const int yi = yb[t] + ky, xi = xb[t] + kx;
        off = (nb[t] + (size_t)yi * g.Wi + xi) * g.Ci;
        return mv[t] && tap < 9 && yi >= 0 && yi < g.Hi && xi >= 0 && xi < g.Wi;
    };
    auto load = [&](int s, bf8* a, bf8* b) {
        const int k = 32 * s + 8 * kg;
        if constexpr (CI4) {
            const int tap0 = k >> 2;
#pragma unroll
            for (int t = 0; t < TM; t++) {
                size_t o0, o1;
                const bool ok0 = tap_ok(t, tap0, o0), ok1 = tap_ok(t, tap0 + 1, o1);
                const uint2 v0 = ok0 ? *(const uint2*)(X + o0) : make_uint2(0u, 0u);
                const uint2 v1 = ok1 ? *(const uint2*)(X + o1) : make_uint2(0u, 0u);
                const uint4 v = make_uint4(v0.x, v0.y, v1.x, v1.y);
                a[t] = __builtin_bit_cast(bf8, v);
            }
        } else {
            const int tap = k >> g.ci_shift, ci = k & (g.Ci - 1);
#pragma unroll
            for (int t = 0; t < TM; t++) {
                size_t o;
                const bool ok = tap_ok(t, tap, o);
                const uint4 v = ok ? *(const uint4*)(X + o + ci) : make_uint4(0u, 0u, 0u, 0u);
                a[t] = __builtin_bit_cast(bf8, v);
            }
        }
#pragma unroll
        for (int j = 0; j < TN; j++) b[j] = __builtin_bit_cast(bf8, *(const uint4*)(wrow[j] + 32 * s));
    };
    f4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const int steps = g.Kp / 32;
    bf8 a[TM], b[TN];
    load(0, a, b);
    for (int s = 0; s < steps; s++) {
        bf8 an[TM], bn[TN];
        if (s + 1 < steps) load(s + 1, an, bn);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
#pragma unroll
        for (int i = 0; i < TM; i++) a[i] = an[i];
#pragma unroll
        for (int j = 0; j < TN; j++) b[j] = bn[j];
    }
    bf16* T = tile[w];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const float bv = bias[col0 + 16 * j + r16];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float v = acc[i][j][e] + bv;
                T[(16 * i + 4 * kg + e) * LDT + 16 * j + r16] = f2bf(v > 0.0f ? v : 0.0f);
            }
    }
    __syncthreads();
    constexpr int CPR = WN / 8;          // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;        // rows per wave instruction
#pragma unroll
    for (int r = 0; r < WM; r += RPI) {
        const int rr = r + lane / CPR, c = lane % CPR;
        const int m = row0 + rr;
        const uint4 v = *(const uint4*)(T + rr * LDT + 8 * c);
        if (m < M) *(uint4*)(Y + (size_t)m * g.Co + col0 + 8 * c) = v;
    }
}

// Forward for Cin a multiple of 32 (the layers after the first): a workgroup
// tile of BM output pixels x BN output channels, k in steps of 32 (one tap, 32
// channels). Each step's A rows (64-byte runs of the input) and B rows (64
// bytes of weights) are staged in LDS by the whole workgroup, double-buffered:
// the next step's global loads are issued before this step's MFMAs and stored
// to the other buffer after them, one barrier per step. Waves (WGM x 4/WGM)
// take 16*TM x 16*TN sub-tiles with v_mfma_f32_16x16x32_bf16; the epilogue is
// the one of k_conv_fwd_mfma.
// D: stages whose loads are in flight in registers ahead of the one in LDS (the
// step count is a multiple of D). A layer of few rows has one or two
// workgroups per CU and waits on each stage's loads: with D = 3 they have two
// stages' time to arrive (64 samples, layers 3-6: 89 us with D = 1, 61 us;
// one sample: 66 and 45 us). Full layers hide them with D = 1.
typedef unsigned u4 __attribute__((ext_vector_type(4)));
template <int BM, int BN, int WGM, int KS = 32, int D = 1>
__global__ __launch_bounds__(256) void k_conv_fwd_lds32(ConvGeom g, const bf16* __restrict__ X,
                                                        const bf16* __restrict__ Wp, const float* __restrict__ bias,
                                                        bf16* __restrict__ Y) {
    constexpr int WGN = 4 / WGM, WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
    constexpr int LD = KS + 8;  // LDS row pitch in bf16: KS k + 8
    constexpr int STAGE = (BM + BN) * LD;
    constexpr int CR = KS / 8;  // 16-byte chunks per row and stage
    constexpr int AC = BM * CR, BC = BN * CR;
    constexpr int AQ = (AC + 255) / 256, BQ = (BC + 255) / 256;
    constexpr int TLD = BN + 8;  // epilogue tile pitch
    static_assert(BM * TLD <= 2 * STAGE, "epilogue tile fits in the stage buffers");
    __shared__ __attribute__((aligned(16))) bf16 lds[2 * STAGE];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r16 = lane & 15, kg = lane >> 4;
    const int M = g.B * g.Ho * g.Wo, HW = g.Ho * g.Wo;
    const int bm0 = blockIdx.x * BM, bn0 = blockIdx.y * BN;
    // Loads without branches, so that the compiler lets them stay in flight over
    // the MFMAs and barriers: a tap in the padding (bit `tap` of ok clear) reads
    // the row's centre pixel instead, which always exists, and is zeroed on its
    // way to LDS; the stages past the last repeat it.
    constexpr bool AF = AC % 256 == 0, BF = BC % 256 == 0;  // every thread loads every chunk
    static_assert(D == 1 || D == 3, "one or three stages");
    static_assert(BF, "weight chunks tile the threads");
    int arow[AQ], apart[AQ];
    const bf16* ap[AQ];  // the row's centre pixel, at the chunk's channels
    unsigned ok[AQ];
#pragma unroll
    for (int q = 0; q < AQ; q++) {
        const int e = t + 256 * q;
        arow[q] = (e / CR) % BM;
        apart[q] = e % CR;
        const int m = bm0 + arow[q];
        const bool v = (AF || e < AC) && m < M;
        const int mm = v ? m : 0;
        const int n = mm / HW, r = mm - n * HW, yo = r / g.Wo, xo = r - yo * g.Wo;
        ap[q] = X + (((size_t)n * g.Hi + 2 * yo) * g.Wi + 2 * xo) * g.Ci + 8 * apart[q];
        ok[q] = 0u;
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int yi = 2 * yo - 1 + tap / 3, xi = 2 * xo - 1 + tap % 3;
            ok[q] |= (v && yi >= 0 && yi < g.Hi && xi >= 0 && xi < g.Wi) ? 1u << tap : 0u;
        }
    }
    const bf16* bp[BQ];
#pragma unroll
    for (int q = 0; q < BQ; q++) {
        const int e = t + 256 * q;
        bp[q] = Wp + (size_t)(bn0 + e / CR) * g.Kp + 8 * (e % CR);
    }
    struct Regs {
        u4 a[AQ], b[BQ];
        unsigned z[AQ];  // all ones, or zero for a tap in the padding
    };
    const int steps = g.Kp / KS;
    auto gload = [&](int s, Regs& r) {
        const int k = KS * min(s, steps - 1);
        const int tap = k >> g.ci_shift, ci0 = k & (g.Ci - 1);
        const int toff = ((tap / 3 - 1) * g.Wi + tap % 3 - 1) * g.Ci;
#pragma unroll
        for (int q = 0; q < AQ; q++) {
            r.z[q] = 0u - ((ok[q] >> tap) & 1u);
            r.a[q] = *(const u4*)(ap[q] + (ci0 + (toff & (int)r.z[q])));
        }
#pragma unroll
        for (int q = 0; q < BQ; q++) r.b[q] = *(const u4*)(bp[q] + k);
    };
    auto sstore = [&](int buf, const Regs& r) {
        bf16* A = lds + buf * STAGE;
        bf16* Bs = A + BM * LD;
#pragma unroll
        for (int q = 0; q < AQ; q++) {
            if (AF || t + 256 * q < AC) *(u4*)(A + arow[q] * LD + 8 * apart[q]) = r.a[q] & r.z[q];
        }
#pragma unroll
        for (int q = 0; q < BQ; q++) {
            const int e = t + 256 * q;
            *(u4*)(Bs + (e / CR) * LD + 8 * (e % CR)) = r.b[q];
        }
    };
    const int wm0 = (w % WGM) * WM, wn0 = (w / WGM) * WN;
    f4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int s, Regs& load, const Regs& store) {
        const int cur = s & 1;
        gload(s + D, load);  // stage s went to LDS a step ago
        const bf16* A = lds + cur * STAGE;
        const bf16* Bs = A + BM * LD;
#pragma unroll
        for (int kk = 0; kk < KS; kk += 32) {
            bf8 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) a[i] = *(const bf8*)(A + (wm0 + 16 * i + r16) * LD + kk + 8 * kg);
#pragma unroll
            for (int j = 0; j < TN; j++) b[j] = *(const bf8*)(Bs + (wn0 + 16 * j + r16) * LD + kk + 8 * kg);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
        }
        sstore(cur ^ 1, store);  // after the last step: nothing reads it
        __syncthreads();
    };
    Regs r0, r1, r2;
    gload(0, r0);
    if constexpr (D == 3) {
        gload(1, r1);
        gload(2, r2);
    }
    sstore(0, r0);
    __syncthreads();
    if constexpr (D == 3) {
        for (int s = 0; s < steps; s += 3) {
            step(s, r0, r1);
            step(s + 1, r1, r2);
            step(s + 2, r2, r0);
        }
    } else {
        for (int s = 0; s < steps; s++) step(s, r0, r0);
    }
    bf16* T = lds;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const float bv = bias[bn0 + wn0 + 16 * j + r16];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float v = acc[i][j][e] + bv;
                T[(wm0 + 16 * i + 4 * kg + e) * TLD + wn0 + 16 * j + r16] = f2bf(v > 0.0f ? v : 0.0f);
            }
    }
    __syncthreads();
    constexpr int CPR = BN / 8;
#pragma unroll
    for (int e0 = 0; e0 < BM * CPR; e0 += 256) {
        const int e = e0 + t;
        if (e < BM * CPR) {
            const int rr = e / CPR, c = e - rr * CPR;
            const int m = bm0 + rr;
            if (m < M) *(uint4*)(Y + (size_t)m * g.Co + bn0 + 8 * c) = *(const uint4*)(T + rr * TLD + 8 * c);
        }
    }
}

// The first two forward layers fused: a workgroup of 8 waves per CU takes pairs
// in turn; the first layer (4 -> C1 channels) writes its H1 x W1 x C1 output to
// LDS with bias, ReLU and bfloat16 rounding, and the second layer (C1 = 32 ->
// 64) reads its operands from that map, so the intermediate never reaches HBM.
// There are two maps: while the second layer of a pair runs from one, the
// inputs of the next pair are in flight, and its first layer fills the other;
// one barrier a pair. The weights are the MFMA's row operand and the pixels
// its columns, so that a lane holds four consecutive channels of a pixel: one
// 8-byte store. A wave keeps the second layer's weights of 32 channels in
// registers for all its pairs and takes every fourth row tile. The map's
// 16-byte chunks are placed so that eight lanes that read every second pixel
// fall on different banks (f12_slot). 4096 samples: 217 us with pixels as rows
// (14 instructions a value to round and store), weights loaded per step and
// the map in pixel order (8-way conflicts); 188 us here, of which the vector
// instructions (addresses, rounding) fill 83 and the MFMAs 28; one sample 22 and
// 15 us.
constexpr int F12_C1 = 32;
constexpr int F12_LDS = 30 * 40 * F12_C1;  // bf16 elements: the default network's first-layer map
constexpr int F12_RT1 = 10;                // row tiles of 16 pixels per wave: first layer (80 tiles),
constexpr int F12_RT2 = 5;                 // second layer (20 tiles, each by two waves)
constexpr int F12_ZERO = 2 * F12_LDS;      // byte offset of 64 zero bytes behind the first map,
constexpr int F12_MAP = F12_ZERO + 64;     // of the second map
// byte offset of the 16-byte chunk c of pixel p in the map
__device__ __forceinline__ int f12_slot(int p, int c) { return ((p ^ ((p >> 3) & 1)) << 6) + ((c ^ ((p >> 1) & 3)) << 4); }
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
// max(v + bias, 0) of four channels as bfloat16, round to nearest even (a NaN gives 0)
__device__ __forceinline__ u2 relu4(f4 v, f4 bias) {
    v = v + bias;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
    const b2 lo = {(__bf16)v[0], (__bf16)v[1]}, hi = {(__bf16)v[2], (__bf16)v[3]};
    return u2{__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi)};
}
// v, of which the compiler knows nothing: addresses formed from it stay inside
// the loop over pairs instead of filling registers across it
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
__global__ __launch_bounds__(512, 2) void k_conv12_fused(ConvGeom g1, ConvGeom g2, const bf16* __restrict__ X,
                                                         const bf16* __restrict__ W1, const float* __restrict__ b1,
                                                         const bf16* __restrict__ W2, const float* __restrict__ b2,
                                                         bf16* __restrict__ Y) {
    constexpr int NW = 8;
    extern __shared__ __attribute__((aligned(16))) char lds12[];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), r16 = lane & 15, kg = lane >> 4;
    const int H1 = g1.Ho, Wd1 = g1.Wo, M1 = H1 * Wd1, H2 = g2.Ho, Wd2 = g2.Wo, M2 = H2 * Wd2;
    const float i1 = 1.0f / (float)Wd1, i2 = 1.0f / (float)Wd2;
    if (t < 4) ((u4*)(lds12 + F12_ZERO))[t] = u4{0u, 0u, 0u, 0u};  // what a tap in the padding reads
    // first layer: K = 36 in two steps of 32; lane group kg holds taps 2 kg and
    // 2 kg + 1 of the first step, tap 8 in group 0 of the second
    bf8 aw1[2][2];
    f4 bias1[2], bias2[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int s = 0; s < 2; s++)
            aw1[j][s] = __builtin_bit_cast(bf8, *(const u4*)(W1 + (size_t)(16 * j + r16) * g1.Kp + 32 * s + 8 * kg));
        bias1[j] = *(const f4*)(b1 + 16 * j + 4 * kg);
        bias2[j] = *(const f4*)(b2 + 32 * (w & 1) + 16 * j + 4 * kg);
    }
    int dy[3], dx[3], off[3];
    unsigned hl[3];  // rows of the input for the tap: none for tap 8 outside group 0
#pragma unroll
    for (int h = 0; h < 3; h++) {
        const int tap = h < 2 ? 2 * kg + h : 8;
        dy[h] = tap / 3 - 1;
        dx[h] = tap % 3 - 1;
        off[h] = (dy[h] * g1.Wi + dx[h]) * 4;
        hl[h] = h < 2 || kg == 0 ? (unsigned)g1.Hi : 0u;
    }
    // second layer: this wave's 32 channels, one tap of 32 channels per step
    bf8 aw2[2][9];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int s = 0; s < 9; s++)
            aw2[j][s] = __builtin_bit_cast(
                bf8, *(const u4*)(W2 + (size_t)(32 * (w & 1) + 16 * j + r16) * g2.Kp + 32 * s + 8 * kg));
    const int RT2 = (M2 + 15) / 16;
    // first layer of one pair: every tap of the wave's row tiles, without
    // branches; a tap in the padding reads eight of the weights' zero padding
    // bytes (k = 36 ..) instead, so no mask has to outlive its load
    const bf16* zero = W1 + 40;
    u2 v[F12_RT1][3];
    auto load1 = [&](int pair) {
        const bf16* Xp = X + (size_t)pair * g1.Hi * g1.Wi * 4;
        const int r = opaque(r16);
#pragma unroll
        for (int u = 0; u < F12_RT1; u++) {
            const int m = (w + NW * u) * 16 + r;
            const int yo = (int)(((float)m + 0.5f) * i1), xo = m - yo * Wd1;  // yo >= H1 past the last pixel
            const int base = (2 * yo * g1.Wi + 2 * xo) * 4;
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const int yi = 2 * yo + dy[h], xi = 2 * xo + dx[h];
                const bool ok = ((unsigned)yi < hl[h]) & ((unsigned)xi < (unsigned)g1.Wi) & (yo < H1);
                const bf16* q = Xp + (base + off[h]);
                q = ok ? q : zero;
                v[u][h] = *(const u2*)q;
            }
        }
    };
    auto layer1 = [&](char* map) {
        const int r = opaque(r16);
#pragma unroll
        for (int u = 0; u < F12_RT1; u++) {
            const int p = (w + NW * u) * 16 + r;
            const bf8 x0 = __builtin_bit_cast(bf8, u4{v[u][0].x, v[u][0].y, v[u][1].x, v[u][1].y});
            const bf8 x1 = __builtin_bit_cast(bf8, u4{v[u][2].x, v[u][2].y, 0u, 0u});
#pragma unroll
            for (int j = 0; j < 2; j++) {
                f4 acc = f4{0.f, 0.f, 0.f, 0.f};
                acc = mfma32(aw1[j][0], x0, acc);
                acc = mfma32(aw1[j][1], x1, acc);
                // channels 16 j + 4 kg .. + 3 of pixel p: half of chunk 2 j + kg / 2
                if (p < M1) *(u2*)(map + f12_slot(p, 2 * j + (kg >> 1)) + 8 * (kg & 1)) = relu4(acc, bias1[j]);
            }
        }
    };
    load1(blockIdx.x);
    layer1(lds12);
    __syncthreads();
    int cur = 0;
    for (int pair = blockIdx.x; pair < g1.B; pair += gridDim.x, cur = F12_MAP - cur) {
        const int next = pair + gridDim.x;
        if (next < g1.B) load1(next);  // in flight over this pair's second layer
        f4 acc[F12_RT2][2];
        int p0[F12_RT2], okm[F12_RT2];  // the centre tap's pixel; bit s: tap s is inside the map
        const int r = opaque(r16);
#pragma unroll
        for (int q = 0; q < F12_RT2; q++) {
            const int m = min(((w >> 1) + 4 * q) * 16 + r, M2 - 1);  // past the last pixel: read, not stored
            const int yo = (int)(((float)m + 0.5f) * i2), xo = m - yo * Wd2;
            p0[q] = 2 * yo * Wd1 + 2 * xo;
            const int rows = (yo > 0 ? 0x7 : 0) | 0x38 | (2 * yo + 1 < H1 ? 0x1c0 : 0);
            const int cols = (xo > 0 ? 0x49 : 0) | 0x92 | (2 * xo + 1 < Wd1 ? 0x124 : 0);
            okm[q] = rows & cols;
#pragma unroll
            for (int j = 0; j < 2; j++) acc[q][j] = f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int s = 0; s < 9; s++) {
            const int d = (s / 3 - 1) * Wd1 + s % 3 - 1;
#pragma unroll
            for (int q = 0; q < F12_RT2; q++) {
                const int at = cur + f12_slot(p0[q] + d, kg);
                const bf8 x = *(const bf8*)(lds12 + (okm[q] & (1 << s) ? at : F12_ZERO + 16 * kg));
#pragma unroll
                for (int j = 0; j < 2; j++) acc[q][j] = mfma32(aw2[j][s], x, acc[q][j]);
            }
        }
        bf16* Yp = Y + (size_t)pair * M2 * 64;
#pragma unroll
        for (int q = 0; q < F12_RT2; q++) {
            const int rt = (w >> 1) + 4 * q, m = rt * 16 + r;
            if (rt >= RT2 || m >= M2) continue;
#pragma unroll
            for (int j = 0; j < 2; j++)
                *(u2*)(Yp + (size_t)m * 64 + 32 * (w & 1) + 16 * j + 4 * kg) = relu4(acc[q][j], bias2[j]);
        }
        if (next < g1.B) layer1(lds12 + (F12_MAP - cur));  // the other map: last read before the previous barrier
        __syncthreads();
    }
}

// ---------------------------------------------------------------- input gradient
// dX = conv^T(dZ, W), masked by the ReLU of the layer input (X > 0), stored as
// the next (earlier) layer's dZ. WT: [Cin][9][Cout].
__global__ __launch_bounds__(256) void k_conv_bwd_data(ConvGeom g, const bf16* __restrict__ dZ,
                                                       const bf16* __restrict__ WT, const bf16* __restrict__ X,
                                                       bf16* __restrict__ dX) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = lane >> 4;
    const int M = g.B * g.Hi * g.Wi;
    const int row0 = blockIdx.x * 64 + (w & 1) * 32;
    const int col0 = blockIdx.y * 64 + (w >> 1) * 32;
    if (col0 >= g.Ci || row0 >= M) return;
    const int HW = g.Hi * g.Wi;
    int nn[2], yi[2], xi[2];
    bool mv[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        int m = row0 + i * 16 + r16;
        mv[i] = m < M;
        int mm = mv[i] ? m : 0;
        nn[i] = mm / HW;
        int r = mm - nn[i] * HW;
        yi[i] = r / g.Wi;
        xi[i] = r - yi[i] * g.Wi;
    }
    f4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const s4 zero = {0, 0, 0, 0};
    const int Kd = 9 * g.Co;
    for (int k0 = kq * 4; k0 < Kd; k0 += 16) {
        const int tap = k0 >> g.co_shift, co = k0 & (g.Co - 1);
        const int ky = tap / 3, kx = tap - 3 * (tap / 3);
        s4 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            int ty = yi[i] + 1 - ky, tx = xi[i] + 1 - kx;
            int yo = ty >> 1, xo = tx >> 1;
            bool ok = mv[i] && ty >= 0 && tx >= 0 && !(ty & 1) && !(tx & 1) && yo < g.Ho && xo < g.Wo;
            a[i] = ok ? *(const s4*)(dZ + (((size_t)nn[i] * g.Ho + yo) * g.Wo + xo) * g.Co + co) : zero;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            int c = col0 + j * 16 + r16;
            b[j] = c < g.Ci ? *(const s4*)(WT + ((size_t)c * 9 + tap) * g.Co + co) : zero;
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        int col = col0 + j * 16 + r16;
        if (col >= g.Ci) continue;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int m = row0 + i * 16 + kq * 4 + e;
                if (m < M) {
                    size_t o = (size_t)m * g.Ci + col;
                    dX[o] = f2bf(bf_pos(X[o]) ? acc[i][j][e] : 0.0f);
                }
            }
    }
}

// The input gradient by parity class (blockIdx.z = 2 py + px): with stride 2 an
// input pixel (yi, xi) receives only the taps of its parity, ky = 1 where yi
// is even and ky in {0, 2} where it is odd (likewise kx), so each class is a
// GEMM over its own pixels with 1, 2, 2 or 4 taps instead of nine taps masked
// to a quarter of them. A workgroup tile of BM pixels x BN input channels, k =
// (tap, Cout) in stages of KS staged through double-buffered LDS as in
// k_conv_fwd_lds32; the tile leaves through LDS as 16-byte row chunks, masked
// by the ReLU of the layer input (X > 0). 256 samples, five layers: 477 us in
// the general kernel (nine masked taps, operands gathered from global memory
// per MFMA), 78 us here; bound by the latency of the staged loads.
template <int BM, int BN, int WGM, int KS>
__global__ __launch_bounds__(256) void k_conv_bwd_data_lds(ConvGeom g, const bf16* __restrict__ dZ,
                                                           const bf16* __restrict__ WT, const bf16* __restrict__ X,
                                                           bf16* __restrict__ dX) {
    constexpr int WGN = 4 / WGM, WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
    constexpr int LD = KS + 8;
    constexpr int STAGE = (BM + BN) * LD;
    constexpr int CR = KS / 8;
    constexpr int AC = BM * CR, BC = BN * CR;
    constexpr int AQ = (AC + 255) / 256, BQ = (BC + 255) / 256;
    constexpr int TLD = BN + 8;
    static_assert(BM * TLD <= 2 * STAGE, "epilogue tile fits in the stage buffers");
    __shared__ __attribute__((aligned(16))) bf16 lds[2 * STAGE];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r16 = lane & 15, kg = lane >> 4;
    const int py = blockIdx.z >> 1, px = blockIdx.z & 1;
    const int Hc = (g.Hi + 1 - py) >> 1, Wc = (g.Wi + 1 - px) >> 1, HWc = Hc * Wc;  // the class's pixels
    const int M = g.B * HWc;
    const int bm0 = blockIdx.x * BM, bn0 = blockIdx.y * BN;
    if (bm0 >= M) return;
    // the class's pixel m as (n, yi, xi)
    auto pixel = [&](int m, int& n, int& yi, int& xi) {
        n = m / HWc;
        const int r = m - n * HWc, yc = r / Wc;
        yi = 2 * yc + py;
        xi = 2 * (r - yc * Wc) + px;
    };
    int arow[AQ], apart[AQ], ayi[AQ], axi[AQ];
    size_t anb[AQ];
    bool av[AQ], ae[AQ];
#pragma unroll
    for (int q = 0; q < AQ; q++) {
        const int e = t + 256 * q;
        ae[q] = e < AC;
        arow[q] = (e / CR) % BM;
        apart[q] = e % CR;
        const int m = bm0 + arow[q];
        av[q] = ae[q] && m < M;
        int n;
        pixel(av[q] ? m : 0, n, ayi[q], axi[q]);
        anb[q] = (size_t)n * g.Ho * g.Wo;
    }
    int brow[BQ], bpart[BQ];
    bool be[BQ];
    const bf16* bp[BQ];
#pragma unroll
    for (int q = 0; q < BQ; q++) {
        const int e = t + 256 * q;
        be[q] = e < BC;
        brow[q] = (e / CR) % BN;
        bpart[q] = e % CR;
        bp[q] = WT + (size_t)(bn0 + brow[q]) * 9 * g.Co + 8 * bpart[q];
    }
    uint4 ra[AQ], rb[BQ];
    auto gload = [&](int s) {
        const int k = KS * s;
        const int j = k >> g.co_shift, co0 = k & (g.Co - 1);  // tap j of the class
        const int jx = px ? (j & 1) : 0, jy = py ? (px ? j >> 1 : j) : 0;
        const int ky = py ? 2 * jy : 1, kx = px ? 2 * jx : 1;
#pragma unroll
        for (int q = 0; q < AQ; q++) {
            const int yo = (ayi[q] + 1 - ky) >> 1, xo = (axi[q] + 1 - kx) >> 1;  // exact: even by the class's taps
            const bool ok = av[q] && yo >= 0 && xo >= 0 && yo < g.Ho && xo < g.Wo;
            ra[q] = ok ? *(const uint4*)(dZ + (anb[q] + (size_t)yo * g.Wo + xo) * g.Co + co0 + 8 * apart[q])
                       : make_uint4(0u, 0u, 0u, 0u);
        }
        const size_t bo = (size_t)(3 * ky + kx) * g.Co + co0;
#pragma unroll
        for (int q = 0; q < BQ; q++) rb[q] = be[q] ? *(const uint4*)(bp[q] + bo) : make_uint4(0u, 0u, 0u, 0u);
    };
    auto sstore = [&](int buf) {
        bf16* A = lds + buf * STAGE;
        bf16* Bs = A + BM * LD;
#pragma unroll
        for (int q = 0; q < AQ; q++)
            if (ae[q]) *(uint4*)(A + arow[q] * LD + 8 * apart[q]) = ra[q];
#pragma unroll
        for (int q = 0; q < BQ; q++)
            if (be[q]) *(uint4*)(Bs + brow[q] * LD + 8 * bpart[q]) = rb[q];
    };
    const int wm0 = (w % WGM) * WM, wn0 = (w / WGM) * WN;
    f4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const int steps = (1 + py) * (1 + px) * g.Co / KS;
    gload(0);
    sstore(0);
    __syncthreads();
    for (int s = 0; s < steps; s++) {
        const int cur = s & 1;
        if (s + 1 < steps) gload(s + 1);
        const bf16* A = lds + cur * STAGE;
        const bf16* Bs = A + BM * LD;
#pragma unroll
        for (int kk = 0; kk < KS; kk += 32) {
            bf8 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) a[i] = *(const bf8*)(A + (wm0 + 16 * i + r16) * LD + kk + 8 * kg);
#pragma unroll
            for (int j = 0; j < TN; j++) b[j] = *(const bf8*)(Bs + (wn0 + 16 * j + r16) * LD + kk + 8 * kg);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
        }
        if (s + 1 < steps) sstore(cur ^ 1);
        __syncthreads();
    }
    bf16* T = lds;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                T[(wm0 + 16 * i + 4 * kg + e) * TLD + wn0 + 16 * j + r16] = f2bf(acc[i][j][e]);
    __syncthreads();
    constexpr int CPR = BN / 8;
#pragma unroll
    for (int e0 = 0; e0 < BM * CPR; e0 += 256) {
        const int e = e0 + t;
        if (e < BM * CPR) {
            const int rr = e / CPR, c = e - rr * CPR;
            const int m = bm0 + rr;
            if (m < M) {
                int n, yi, xi;
                pixel(m, n, yi, xi);
                const size_t o = (((size_t)n * g.Hi + yi) * g.Wi + xi) * g.Ci + bn0 + 8 * c;
                const uint4 xv = *(const uint4*)(X + o);
                uint4 v = *(const uint4*)(T + rr * TLD + 8 * c);
                auto mask = [](unsigned x, unsigned u) {
                    return (bf_pos((bf16)(x & 0xffffu)) ? u & 0xffffu : 0u) | (bf_pos((bf16)(x >> 16)) ? u & 0xffff0000u : 0u);
                };
                v = make_uint4(mask(xv.x, v.x), mask(xv.y, v.y), mask(xv.z, v.z), mask(xv.w, v.w));
                *(uint4*)(dX + o) = v;
            }
        }
    }
}

// ---------------------------------------------------------------- weight gradient
// ws[s][co][k] = sum over output pixels m of chunk s of dZ[m][co] * im2col(X)[m][k],
// and, from the first column tile, ws_b[s][co] = the chunk's sum of dZ[m][co]
// (the bias gradient). Workgroup tile: 64 output channels x 64 k, 128 pixels a
// stage. The reduction runs over m, the slow index of both operands, so each
// thread loads an 8 x 8 block (8 pixels x 8 channels, one 16-byte run per
// pixel), transposes it in registers and stores eight 16-byte runs of m to
// LDS, from which the MFMA operands are read whole; the next stage's loads
// are issued before this stage's MFMAs. 256 samples, six layers: 324 us with
// one wave per 32 x 32 tile and 2-byte gathers, plus 360 us of column sums;
// 101 us here for both.
constexpr int BW_M = 128, BW_LD = BW_M + 8;  // pixels a stage; LDS row pitch (bf16)
__global__ __launch_bounds__(256) void k_conv_bwd_w(ConvGeom g, const bf16* __restrict__ dZ, const bf16* __restrict__ X,
                                                    float* __restrict__ ws, float* __restrict__ ws_b, int chunk) {
    __shared__ __attribute__((aligned(16))) bf16 lds[2 * 64 * BW_LD];  // A: [co][m], B: [k][m]
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r16 = lane & 15, kg = lane >> 4;
    const int M = g.B * g.Ho * g.Wo, HW = g.Ho * g.Wo;
    const int co0 = blockIdx.x * 64, kc0 = blockIdx.y * 64, s = blockIdx.z;
    const int mbeg = s * chunk, mend = min(M, mbeg + chunk);
    // threads 0-127 stage dZ, 128-255 the im2col columns: pixel block mb, channel (or k) block cb
    const int half = t >> 7, mb = t & 15, cb = (t >> 4) & 7;
    const int col = (half ? kc0 : co0) + 8 * cb;
    const bool cv = col < (half ? g.K : g.Co);  // K is a multiple of 4, Co of 16
    const int tap0 = col >> g.ci_shift, tap1 = (col + 4) >> g.ci_shift;
    const int ky0 = tap0 / 3, kx0 = tap0 - 3 * ky0, ky1 = tap1 / 3, kx1 = tap1 - 3 * ky1;
    const int ci = col & (g.Ci - 1);
    const bool cv1 = col + 4 < g.K;
    uint4 r[8];
    float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const bool bias = blockIdx.y == 0 && !half;
    auto gload = [&](int m0) {
        const int mf = m0 + 8 * mb;
        int n = 0, yo = 0, xo = 0;
        if (half) {
            const int mm = min(mf, M - 1);
            n = mm / HW;
            const int q = mm - n * HW;
            yo = q / g.Wo;
            xo = q - yo * g.Wo;
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const bool mok = cv && mf + e < mend;
            r[e] = make_uint4(0u, 0u, 0u, 0u);
            if (!half) {
                if (mok) r[e] = *(const uint4*)(dZ + (size_t)(mf + e) * g.Co + col);
            } else {
                const bf16* Xn = X + (size_t)n * g.Hi * g.Wi * g.Ci;
                const int yi = 2 * yo - 1 + ky0, xi = 2 * xo - 1 + kx0;
                const bool ok = mok && yi >= 0 && yi < g.Hi && xi >= 0 && xi < g.Wi;
                if (g.Ci == 4) {  // two taps of 4 channels
                    const int yj = 2 * yo - 1 + ky1, xj = 2 * xo - 1 + kx1;
                    const bool okj = mok && cv1 && yj >= 0 && yj < g.Hi && xj >= 0 && xj < g.Wi;
                    const uint2 u = ok ? *(const uint2*)(Xn + ((size_t)yi * g.Wi + xi) * 4) : make_uint2(0u, 0u);
                    const uint2 v = okj ? *(const uint2*)(Xn + ((size_t)yj * g.Wi + xj) * 4) : make_uint2(0u, 0u);
                    r[e] = make_uint4(u.x, u.y, v.x, v.y);
                } else if (ok) {
                    r[e] = *(const uint4*)(Xn + ((size_t)yi * g.Wi + xi) * g.Ci + ci);
                }
                if (++xo == g.Wo) {
                    xo = 0;
                    if (++yo == g.Ho) { yo = 0; n++; }
                }
            }
        }
    };
    auto sstore = [&]() {
        bf16* base = lds + half * 64 * BW_LD + (8 * cb) * BW_LD + 8 * mb;
        const unsigned* rw = reinterpret_cast<const unsigned*>(r);
#pragma unroll
        for (int j = 0; j < 4; j++) {  // channels 2j, 2j + 1: the low and high halves of dword j of each pixel
            unsigned lo[4], hi[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                lo[i] = __builtin_amdgcn_perm(rw[4 * (2 * i + 1) + j], rw[4 * (2 * i) + j], 0x05040100u);
                hi[i] = __builtin_amdgcn_perm(rw[4 * (2 * i + 1) + j], rw[4 * (2 * i) + j], 0x07060302u);
            }
            *(uint4*)(base + (2 * j) * BW_LD) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            *(uint4*)(base + (2 * j + 1) * BW_LD) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        }
        if (bias) {
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    bsum[2 * j] += __uint_as_float(rw[4 * e + j] << 16);
                    bsum[2 * j + 1] += __uint_as_float(rw[4 * e + j] & 0xffff0000u);
                }
        }
    };
    const int wa0 = (w & 1) * 32, wb0 = (w >> 1) * 32;
    f4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const bf16* A = lds;
    const bf16* Bs = lds + 64 * BW_LD;
    gload(mbeg);
    for (int m0 = mbeg; m0 < mend; m0 += BW_M) {
        sstore();
        __syncthreads();
        if (m0 + BW_M < mend) gload(m0 + BW_M);
#pragma unroll
        for (int kk = 0; kk < BW_M; kk += 32) {
            bf8 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) a[i] = *(const bf8*)(A + (wa0 + 16 * i + r16) * BW_LD + kk + 8 * kg);
#pragma unroll
            for (int j = 0; j < 2; j++) b[j] = *(const bf8*)(Bs + (wb0 + 16 * j + r16) * BW_LD + kk + 8 * kg);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int k = kc0 + wb0 + 16 * j + r16;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int co = co0 + wa0 + 16 * i + kg * 4 + e;
                if (co < g.Co && k < g.Kp) ws[((size_t)s * g.Co + co) * g.Kp + k] = acc[i][j][e];
            }
        }
    if (blockIdx.y == 0) {  // the 16 pixel blocks' channel sums, in order
        float* part = reinterpret_cast<float*>(lds);  // [16][64]; every wave is past its last operand read
        if (!half) {
#pragma unroll
            for (int e = 0; e < 8; e++) part[mb * 64 + 8 * cb + e] = bsum[e];
        }
        __syncthreads();
        if (t < 64 && co0 + t < g.Co) {
            float v = 0.0f;
#pragma unroll
            for (int q = 0; q < 16; q++) v += part[q * 64 + t];
            ws_b[(size_t)s * g.Co + co0 + t] = v;
        }
    }
}

// Column sums of the backward pass's partial results, all in one launch: sum i
// adds the rows of an S x width matrix (width a multiple of 2) into out; a
// weight gradient's columns past K of each Kp-column group are padding. A
// workgroup of 1024 threads takes 2 * 64 * (16 / slices) columns; wave `slice`
// of a column group adds rows slice, slice + slices, ..., the slices then meet
// in order (deterministic). One thread per column over all rows took 690 us
// over the 14 sums of a 256-sample step; this launch takes 26 us.
struct RowSum {
    const float* src;
    float* out;
    int S, width, K, Kp, slices, block0;
};
constexpr int ROW_SUMS = 14;
struct RowSums {
    RowSum s[ROW_SUMS];
    int n;
};
__global__ __launch_bounds__(1024) void k_row_sums(RowSums a) {
    __shared__ float2 part[16][64];
    int i = 0;
    while (i + 1 < a.n && (int)blockIdx.x >= a.s[i + 1].block0) i++;
    const RowSum& r = a.s[i];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int slices = r.slices, groups = 16 / slices, grp = w / slices, slice = w - grp * slices;
    const int c = 2 * (64 * (((int)blockIdx.x - r.block0) * groups + grp) + lane);
    float2 v = make_float2(0.0f, 0.0f);
    if (c < r.width) {
        const float* p = r.src + c;
#pragma unroll 8
        for (int q = slice; q < r.S; q += slices) {
            const float2 u = *(const float2*)(p + (size_t)q * r.width);
            v.x += u.x;
            v.y += u.y;
        }
    }
    part[w][lane] = v;
    __syncthreads();
    if (slice == 0 && c < r.width) {
        for (int q = 1; q < slices; q++) {
            const float2 u = part[w + q][lane];
            v.x += u.x;
            v.y += u.y;
        }
        const int row = r.Kp ? c / r.Kp : 0, k = c - row * r.Kp;  // Kp is even: both columns in one row
        if (!r.Kp || k < r.K) r.out[r.Kp ? (size_t)row * r.K + k : (size_t)c] = v.x;
        if (!r.Kp || k + 1 < r.K) r.out[r.Kp ? (size_t)row * r.K + k + 1 : (size_t)c + 1] = v.y;
    }
}

// ---------------------------------------------------------------- head
// One block per sample: mean pool, dense 6 outputs; with targets also the loss,
// the dense-layer gradient contributions and dZ of the last convolution.
__global__ __launch_bounds__(256) void k_head(int P6, int C6, const bf16* __restrict__ A6, const float* __restrict__ Wfc,
                                              const float* __restrict__ bfc, const float* __restrict__ y,
                                              const float* __restrict__ wn, int nw, float* __restrict__ out,
                                              bf16* __restrict__ dZ6, float* __restrict__ ws_fc, float* __restrict__ ws_loss) {
    extern __shared__ float sh[];  // h[C6], dh[C6]
    __shared__ float red[4][6];
    __shared__ float o6[6], d6[6];
    const int n = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    // 1 / max(1, sum of the nw sample weights): every block forms the same sum
    float inv_norm = 0.0f;
    if (y) {
        float s = 0.0f;
        for (int i = t; i < nw; i += 256) s += wn[i];
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) red[wv][0] = s;
        __syncthreads();
        inv_norm = 1.0f / fmaxf(1.0f, (red[0][0] + red[1][0]) + (red[2][0] + red[3][0]));
        __syncthreads();
    }
    float* h = sh;
    for (int c = t; c < C6; c += 256) {
        float s = 0.0f;
        for (int p = 0; p < P6; p++) s += bf2f(A6[((size_t)n * P6 + p) * C6 + c]);
        h[c] = s / (float)P6;
    }
    __syncthreads();
    for (int j = 0; j < 6; j++) {
        float s = 0.0f;
        for (int c = t; c < C6; c += 256) s += Wfc[j * C6 + c] * h[c];
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) red[wv][j] = s;
    }
    __syncthreads();
    if (t < 6) {
        float v = bfc[t] + ((red[0][t] + red[1][t]) + (red[2][t] + red[3][t]));
        o6[t] = v;
        out[n * 6 + t] = v;
        if (y) d6[t] = 2.0f * wn[n] * (v - y[n * 6 + t]) * inv_norm;
    }
    __syncthreads();
    if (!y) return;
    if (t == 0) {
        float l = 0.0f;
        for (int j = 0; j < 6; j++) { float e = o6[j] - y[n * 6 + j]; l += e * e; }
        ws_loss[2 * n] = wn[n] * l * inv_norm;  // rows of 2 columns, for the column sums
        ws_loss[2 * n + 1] = 0.0f;
    }
    const int width = 6 * C6 + 6;
    float* dh = sh + C6;
    for (int c = t; c < C6; c += 256) {
        float s = 0.0f;
        for (int j = 0; j < 6; j++) {
            ws_fc[(size_t)n * width + j * C6 + c] = d6[j] * h[c];
            s += Wfc[j * C6 + c] * d6[j];
        }
        dh[c] = s;
    }
    if (t < 6) ws_fc[(size_t)n * width + 6 * C6 + t] = d6[t];
    __syncthreads();
    for (int q = t; q < P6 * C6; q += 256) {
        int c = q % C6;
        size_t o = (size_t)n * P6 * C6 + q;
        dZ6[o] = f2bf(bf_pos(A6[o]) ? dh[c] / (float)P6 : 0.0f);
    }
}

// ---------------------------------------------------------------- parameters
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       size_t n, float lr, float b1, float b2, float c1, float c2, float eps) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    float mi = b1 * m[i] + (1.0f - b1) * gi;
    float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi; v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
// bfloat16 copies of one layer's weights: Wp[co][Kp] (zero padded) and WT[ci][tap][co]
__global__ void k_pack(const float* __restrict__ W, int Co, int Ci, int Kp, bf16* __restrict__ Wp, bf16* __restrict__ WT) {
    int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= Co * Kp) return;
    int co = idx / Kp, k = idx - (idx / Kp) * Kp;
    int K = 9 * Ci;
    bf16 v = k < K ? f2bf(W[(size_t)co * K + k]) : (bf16)0;
    Wp[idx] = v;
    if (WT && k < K) {
        int tap = k / Ci, ci = k - (k / Ci) * Ci;
        WT[((size_t)ci * 9 + tap) * Co + co] = v;
    }
}

// ---------------------------------------------------------------- inputs and proposals
// The network's inputs, one cell of bw x bh = (W / IW) x (H / IH) pixels per
// thread and per frame (cell_features; the inverse depths by the hardware
// reciprocal: within 1 ulp, far below the bfloat16 rounding of the result).
// The inverse depths are summed per column over the rows in order; the
// column sums are merged pairwise by a stack (two sums of equal size merge,
// left + right; what remains at the end is added right to left), which for
// a power-of-two bw is the balanced tree ((c0 + c1) + (c2 + c3)) + ...
__global__ __launch_bounds__(256) void k_inputs(const FrameSrc* __restrict__ src, int IW, int IH, bf16* __restrict__ x) {
    const int n = blockIdx.y;
    const int cell = blockIdx.x * 256 + threadIdx.x;
    if (cell >= IW * IH) return;
    const FrameSrc s = src[n];
    const int bw = s.W / IW, bh = s.H / IH;
    const int cx = cell % IW, cy = cell / IW;
    bf16* o = x + ((size_t)n * IW * IH + cell) * 4;
    for (int f = 0; f < 2; f++) {
        const uint8_t* g8 = s.g8[f];
        const uint16_t* d16 = s.d16[f];
        const size_t row0 = (size_t)(cy * bh) * s.W + (size_t)cx * bw;
        if (bw == 8 && bh == 8 && !(((uintptr_t)(g8 + row0)) & 7) && !(((uintptr_t)(d16 + row0)) & 15) && !(s.W & 7)) {
            cell8_features(g8, d16, s.W, cx * 8, cy * 8, o + 2 * f);
            continue;
        }
        unsigned gs = 0, nv = 0;
        float sv[16];  // bw < 65536 columns: at most 16 pending sums
        int sl[16], sp = 0;
        for (int xx = 0; xx < bw; xx++) {
            float v = 0.0f;
            for (int yy = 0; yy < bh; yy++) {
                const size_t i = row0 + (size_t)yy * s.W + xx;
                gs += g8[i];
                unsigned d = d16[i];
                if (d) { v += inv_depth_m(d); nv++; }
            }
            int l = 0;
            while (sp > 0 && sl[sp - 1] == l) { v = sv[--sp] + v; l++; }
            sv[sp] = v; sl[sp] = l; sp++;
        }
        float ids = sv[sp - 1];
        for (int k = sp - 2; k >= 0; k--) ids = sv[k] + ids;
        cell_features(gs, ids, nv, bw * bh, o + 2 * f);
    }
}

// Training-set symmetries of a pinhole camera with a centred principal point.
// flags bit 0: mirror columns (camera x -> -x), bit 1: mirror rows (y -> -y),
// bit 2: swap reference and current frame (target = that of the inverse pose,
// y_inv). A mirror S maps Trel to S Trel S: rotation vector -S w, translation S t.
__global__ __launch_bounds__(256) void k_augment(const bf16* __restrict__ x, const float* __restrict__ y,
                                                 const float* __restrict__ y_inv, const int* __restrict__ flags, int IW,
                                                 int IH, bf16* __restrict__ xo, float* __restrict__ yo) {
    const int n = blockIdx.y;
    const int cell = blockIdx.x * 256 + threadIdx.x;
    const int f = flags[n];
    if (cell < IW * IH) {
        int cx = cell % IW, cy = cell / IW;
        int sx = (f & 1) ? IW - 1 - cx : cx, sy = (f & 2) ? IH - 1 - cy : cy;
        const bf16* src = x + ((size_t)n * IW * IH + (size_t)sy * IW + sx) * 4;
        bf16* dst = xo + ((size_t)n * IW * IH + cell) * 4;
        if (f & 4) { dst[0] = src[2]; dst[1] = src[3]; dst[2] = src[0]; dst[3] = src[1]; }
        else { dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2]; dst[3] = src[3]; }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const float* b = (f & 4) ? y_inv + 6 * n : y + 6 * n;
        float v[6] = {b[0], b[1], b[2], b[3], b[4], b[5]};
        if (f & 1) { v[1] = -v[1]; v[2] = -v[2]; v[3] = -v[3]; }
        if (f & 2) { v[0] = -v[0]; v[2] = -v[2]; v[4] = -v[4]; }
        for (int k = 0; k < 6; k++) yo[6 * n + k] = v[k];
    }
}

// Trel = [R(w) | t] from the scaled outputs (Rodrigues), FP64, stored FP32
__global__ void k_outputs_to_trel(const float* __restrict__ out, int n, float rot_scale_rad, float trans_scale,
                                  float* __restrict__ trel) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double w[3], t[3];
    for (int k = 0; k < 3; k++) { w[k] = (double)out[6 * i + k] * rot_scale_rad; t[k] = (double)out[6 * i + 3 + k] * trans_scale; }
    double th = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    double A = th > 1e-12 ? sin(th) / th : 1.0;
    double B = th > 1e-12 ? (1.0 - cos(th)) / (th * th) : 0.5;
    double K[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
    double K2[9];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) {
            double s = 0.0;
            for (int q = 0; q < 3; q++) s += K[3 * r + q] * K[3 * q + c];
            K2[3 * r + c] = s;
        }
    float* T = trel + 16 * (size_t)i;
    for (int r = 0; r < 3; r++) {
        for (int c = 0; c < 3; c++) T[4 * r + c] = (float)((r == c ? 1.0 : 0.0) + A * K[3 * r + c] + B * K2[3 * r + c]);
        T[4 * r + 3] = (float)t[r];
    }
    T[12] = 0.0f; T[13] = 0.0f; T[14] = 0.0f; T[15] = 1.0f;
}

}  // namespace rt

using namespace rt;

// ---------------------------------------------------------------- host object
struct rt_cnn {
    int device = 0, max_batch = 0, cus = 256;
    bool fused12 = false;       // k_conv12_fused may use the LDS it needs on this device
    rt_cnn_config cfg;
    hipStream_t stream = nullptr;
    rt::HostStage st_src, st_flags;  // pinned staging of the frame table and the augmentation flags
    int H[7], W[7];
    size_t w_off[6], b_off[6], fc_w, fc_b, nparams;
    int K[6], Kp[6];
    std::vector<void*> allocs;
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    bf16* Wp[6] = {};
    bf16* WT[6] = {};
    bf16* act[7] = {};          // act[0] is the caller's input during a call
    bf16 *dz_a = nullptr, *dz_b = nullptr;
    bf16* xin = nullptr;        // inputs built by rt_batch_propose
    float *ws = nullptr, *ws_b = nullptr, *ws_fc = nullptr, *ws_loss = nullptr, *out = nullptr, *loss = nullptr;
    size_t ws_off[6], wsb_off[6];  // of each layer in ws and ws_b
    FrameSrc* src_dev = nullptr;
    int* flags_dev = nullptr;
    float* trel_tmp = nullptr;
    int step = 0;
    bool packed = false;
};

static int ilog2(int v) {
    int s = 0;
    while ((1 << s) < v) s++;
    return (1 << s) == v ? s : -1;
}

extern "C" void rt_cnn_default_config(rt_cnn_config* c) {
    if (!c) return;
    c->in_width = 80; c->in_height = 60;
    const int ch[7] = {4, 32, 64, 128, 128, 256, 256};
    for (int l = 0; l < 7; l++) c->channels[l] = ch[l];
    c->rot_scale_deg = 10.0f;
    c->trans_scale_mm = 150.0f;
}

static ConvGeom geom(const rt_cnn* net, int l, int B) {
    ConvGeom g;
    g.B = B; g.Hi = net->H[l]; g.Wi = net->W[l]; g.Ci = net->cfg.channels[l]; g.ci_shift = ilog2(g.Ci);
    g.Ho = net->H[l + 1]; g.Wo = net->W[l + 1]; g.Co = net->cfg.channels[l + 1]; g.co_shift = ilog2(g.Co);
    g.K = net->K[l]; g.Kp = net->Kp[l];
    return g;
}

static size_t act_elems(const rt_cnn* net, int l, int B) {
    return (size_t)B * net->H[l] * net->W[l] * net->cfg.channels[l];
}

// Weight-gradient split of layer l: chunks of output pixels (multiples of the
// kernel's stage) so that the grid holds about two workgroups per CU; at most
// wsplit_max parts for any batch up to B.
static int wsplit_max(const rt_cnn* net, int l, int B) {
    const int M = B * net->H[l + 1] * net->W[l + 1];
    const int tiles = ((net->cfg.channels[l + 1] + 63) / 64) * ((net->Kp[l] + 63) / 64);
    return std::max(1, std::min(512 / tiles, (M + BW_M - 1) / BW_M));
}
static void wsplit(const rt_cnn* net, int l, int B, int* S, int* chunk) {
    const int M = B * net->H[l + 1] * net->W[l + 1], s = wsplit_max(net, l, B);
    *chunk = ((M + s - 1) / s + BW_M - 1) / BW_M * BW_M;
    *S = (M + *chunk - 1) / *chunk;
}

extern "C" int rt_cnn_create(int device, const rt_cnn_config* c, int max_batch, rt_cnn** out) {
    if (!out || max_batch < 1) return set_error(RT_ERR_ARG, "rt_cnn_create: bad argument");
    *out = nullptr;
    rt_cnn_config cfg;
    if (c) cfg = *c; else rt_cnn_default_config(&cfg);
    if (cfg.in_width < 2 || cfg.in_height < 2) return set_error(RT_ERR_ARG, "rt_cnn_create: input too small");
    if (cfg.channels[0] != 4) return set_error(RT_ERR_ARG, "rt_cnn_create: the input has 4 channels");
    for (int l = 1; l < 7; l++)
        if (ilog2(cfg.channels[l]) < 4 || cfg.channels[l] > 1024)
            return set_error(RT_ERR_ARG, "rt_cnn_create: conv channels must be powers of two in 16..1024");
    if (!(cfg.rot_scale_deg > 0) || !(cfg.trans_scale_mm > 0)) return set_error(RT_ERR_ARG, "rt_cnn_create: bad output scales");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return set_error(RT_ERR_ARG, "no such device");
    if (hipSetDevice(device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    rt_cnn* net = new rt_cnn();
    net->device = device; net->max_batch = max_batch; net->cfg = cfg;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0) net->cus = cus;
    net->fused12 = hipFuncSetAttribute((const void*)k_conv12_fused, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       F12_MAP + 2 * F12_LDS) == hipSuccess;
    net->H[0] = cfg.in_height; net->W[0] = cfg.in_width;
    for (int l = 1; l < 7; l++) { net->H[l] = (net->H[l - 1] + 1) / 2; net->W[l] = (net->W[l - 1] + 1) / 2; }
    size_t o = 0;
    for (int l = 0; l < 6; l++) {
        net->K[l] = 9 * cfg.channels[l];
        net->Kp[l] = (net->K[l] + 31) / 32 * 32;
        net->w_off[l] = o; o += (size_t)cfg.channels[l + 1] * net->K[l];
        net->b_off[l] = o; o += (size_t)cfg.channels[l + 1];
    }
    net->fc_w = o; o += 6 * (size_t)cfg.channels[6];
    net->fc_b = o; o += 6;
    net->nparams = o;
    // workspace sizes
    size_t wsf = 0, wsb = 0, maxact = 0;
    for (int l = 0; l < 6; l++) {  // every layer's parts at once: one launch sums them all
        const size_t S = wsplit_max(net, l, max_batch);
        net->ws_off[l] = wsf; wsf += S * cfg.channels[l + 1] * net->Kp[l];
        net->wsb_off[l] = wsb; wsb += S * cfg.channels[l + 1];
    }
    for (int l = 1; l < 7; l++) maxact = std::max(maxact, act_elems(net, l, max_batch));
    bool ok = hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking) == hipSuccess;
    auto al = [&](void** p, size_t bytes) {
        if (!ok) return;
        if (hipMalloc(p, std::max(bytes, (size_t)256)) != hipSuccess) { ok = false; return; }
        net->allocs.push_back(*p);
        if (hipMemset(*p, 0, std::max(bytes, (size_t)256)) != hipSuccess) ok = false;
    };
    al((void**)&net->params, 4 * o); al((void**)&net->grads, 4 * o);
    al((void**)&net->adam_m, 4 * o); al((void**)&net->adam_v, 4 * o);
    for (int l = 0; l < 6; l++) {
        al((void**)&net->Wp[l], 2 * (size_t)cfg.channels[l + 1] * net->Kp[l]);
        if (l > 0) al((void**)&net->WT[l], 2 * (size_t)cfg.channels[l + 1] * net->K[l]);
    }
    for (int l = 1; l < 7; l++) al((void**)&net->act[l], 2 * act_elems(net, l, max_batch));
    al((void**)&net->dz_a, 2 * maxact); al((void**)&net->dz_b, 2 * maxact);
    al((void**)&net->xin, 2 * act_elems(net, 0, max_batch));
    al((void**)&net->ws, 4 * wsf); al((void**)&net->ws_b, 4 * wsb);
    al((void**)&net->ws_fc, 4 * (size_t)max_batch * (6 * cfg.channels[6] + 6));
    al((void**)&net->ws_loss, 8 * (size_t)max_batch);
    al((void**)&net->out, 4 * 6 * (size_t)max_batch);
    al((void**)&net->loss, 256);
    al((void**)&net->src_dev, sizeof(FrameSrc) * (size_t)max_batch);
    al((void**)&net->flags_dev, 4 * (size_t)max_batch);
    if (!ok) {
        for (void* p : net->allocs) hipFree(p);
        if (net->stream) hipStreamDestroy(net->stream);
        delete net;
        return set_error(RT_ERR_NOMEM, "rt_cnn_create: device allocation");
    }
    *out = net;
    return RT_OK;
}

extern "C" void rt_cnn_destroy(rt_cnn* net) {
    if (!net) return;
    hipSetDevice(net->device);
    hipStreamSynchronize(net->stream);
    net->st_src.release();
    net->st_flags.release();
    for (void* p : net->allocs) hipFree(p);
    hipStreamDestroy(net->stream);
    delete net;
}

extern "C" size_t rt_cnn_num_params(const rt_cnn* net) { return net ? net->nparams : 0; }
extern "C" void* rt_cnn_stream(rt_cnn* net) { return net ? (void*)net->stream : nullptr; }

static int pack(rt_cnn* net, hipStream_t s) {
    for (int l = 0; l < 6; l++) {
        int Co = net->cfg.channels[l + 1], Ci = net->cfg.channels[l];
        int n = Co * net->Kp[l];
        k_pack<<<(n + 255) / 256, 256, 0, s>>>(net->params + net->w_off[l], Co, Ci, net->Kp[l], net->Wp[l], net->WT[l]);
    }
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "pack launch");
    net->packed = true;
    return RT_OK;
}

extern "C" int rt_cnn_set_params(rt_cnn* net, const float* params) {
    if (!net || !params) return set_error(RT_ERR_ARG, "rt_cnn_set_params: null argument");
    if (hipSetDevice(net->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    size_t b = 4 * net->nparams;
    if (hipMemcpyAsync(net->params, params, b, hipMemcpyHostToDevice, net->stream) != hipSuccess ||
        hipMemsetAsync(net->adam_m, 0, b, net->stream) != hipSuccess || hipMemsetAsync(net->adam_v, 0, b, net->stream) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_cnn_set_params: copy");
    net->step = 0;
    int rc = pack(net, net->stream);
    if (rc) return rc;
    if (hipStreamSynchronize(net->stream) != hipSuccess) return set_error(RT_ERR_HIP, "rt_cnn_set_params: sync");
    return RT_OK;
}

extern "C" int rt_cnn_get_params(rt_cnn* net, float* params) {
    if (!net || !params) return set_error(RT_ERR_ARG, "rt_cnn_get_params: null argument");
    if (hipSetDevice(net->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    if (hipMemcpyAsync(params, net->params, 4 * net->nparams, hipMemcpyDeviceToHost, net->stream) != hipSuccess ||
        hipStreamSynchronize(net->stream) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_cnn_get_params: copy");
    return RT_OK;
}

// One forward layer on the 16x16x32 MFMA kernel when its shape fits: Cin = 4
// or a power of two >= 8, Cout a multiple of 32 (Cin = 4) or 64. The wave tile
// is the tallest of 64, 32, 16 rows that still gives 2048 waves. Returns false
// when the layer needs the general kernels.
static bool forward_mfma(const ConvGeom& g, const bf16* X, const bf16* Wp, const float* bias, bf16* Y, hipStream_t s) {
    const int M = g.B * g.Ho * g.Wo;
    const bool pow2 = g.Ci >= 8 && (g.Ci & (g.Ci - 1)) == 0;
    if (g.Ci == 4 && g.Co % 32 == 0) {
        k_conv_fwd_mfma<4, 2, 4, 1, true><<<dim3((M + 255) / 256, g.Co / 32), 256, 0, s>>>(g, X, Wp, bias, Y);
        return true;
    }
    if (!pow2 || g.Co % 64) return false;
    if (g.Ci % 32 == 0) {
        // LDS-staged tiles: the largest workgroup tile that still gives 512 workgroups
        auto blocks = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * (g.Co / bn); };
        if (g.Co == 64) {
            if (blocks(256, 64) >= 512) k_conv_fwd_lds32<256, 64, 4><<<dim3((M + 255) / 256, 1), 256, 0, s>>>(g, X, Wp, bias, Y);
            else k_conv_fwd_lds32<128, 64, 4><<<dim3((M + 127) / 128, 1), 256, 0, s>>>(g, X, Wp, bias, Y);
            return true;
        }
        if (g.Co % 128 == 0) {
            const unsigned gy = g.Co / 128;
            if (blocks(128, 128) >= 512) k_conv_fwd_lds32<128, 128, 2><<<dim3((M + 127) / 128, gy), 256, 0, s>>>(g, X, Wp, bias, Y);
            else if (blocks(64, 128) >= 512) k_conv_fwd_lds32<64, 128, 2><<<dim3((M + 63) / 64, gy), 256, 0, s>>>(g, X, Wp, bias, Y);
            else if (g.Ci % 64 == 0)  // few rows and a long k: stages of 64 halve its barriers and load round trips
                k_conv_fwd_lds32<32, 128, 2, 64, 3><<<dim3((M + 31) / 32, gy), 256, 0, s>>>(g, X, Wp, bias, Y);
            else k_conv_fwd_lds32<32, 128, 2><<<dim3((M + 31) / 32, gy), 256, 0, s>>>(g, X, Wp, bias, Y);
            return true;
        }
    }
    auto waves = [&](int wm) { return (long)((M + wm - 1) / wm) * (g.Co / 64); };
    if (g.Co == 64) {  // one column tile: the four waves stacked over rows
        if (waves(64) >= 2048) k_conv_fwd_mfma<4, 4, 4, 1, false><<<dim3((M + 255) / 256, 1), 256, 0, s>>>(g, X, Wp, bias, Y);
        else if (waves(32) >= 2048) k_conv_fwd_mfma<2, 4, 4, 1, false><<<dim3((M + 127) / 128, 1), 256, 0, s>>>(g, X, Wp, bias, Y);
        else k_conv_fwd_mfma<1, 4, 4, 1, false><<<dim3((M + 63) / 64, 1), 256, 0, s>>>(g, X, Wp, bias, Y);
        return true;
    }
    if (g.Co % 128) return false;
    const dim3 gy(0, g.Co / 128);
    if (waves(64) >= 2048) k_conv_fwd_mfma<4, 4, 2, 2, false><<<dim3((M + 127) / 128, gy.y), 256, 0, s>>>(g, X, Wp, bias, Y);
    else if (waves(32) >= 2048) k_conv_fwd_mfma<2, 4, 2, 2, false><<<dim3((M + 63) / 64, gy.y), 256, 0, s>>>(g, X, Wp, bias, Y);
    else k_conv_fwd_mfma<1, 4, 2, 2, false><<<dim3((M + 31) / 32, gy.y), 256, 0, s>>>(g, X, Wp, bias, Y);
    return true;
}

// The first two layers in one launch when their shapes are the fused
// kernel's: 4 -> 32 -> 64 channels, the first layer's map within its LDS, the
// second layer's rows within a wave's row tiles.
static bool forward_fused12(rt_cnn* net, int n, hipStream_t s) {
    const ConvGeom g1 = geom(net, 0, n), g2 = geom(net, 1, n);
    if (g1.Ci != 4 || g1.Co != F12_C1 || g1.Kp != 64 || g2.Ci != F12_C1 || g2.Co != 64 || g2.Kp != 9 * F12_C1 ||
        g2.Hi != g1.Ho || g2.Wi != g1.Wo || (g1.Ho * g1.Wo + 1) / 2 * 2 * F12_C1 > F12_LDS ||
        (g1.Ho * g1.Wo + 15) / 16 > 8 * F12_RT1 || (g2.Ho * g2.Wo + 15) / 16 > 4 * F12_RT2 || !net->fused12)
        return false;
    k_conv12_fused<<<std::min(n, net->cus), 512, F12_MAP + 2 * F12_LDS, s>>>(g1, g2, net->act[0], net->Wp[0], net->params + net->b_off[0], net->Wp[1],
                                         net->params + net->b_off[1], net->act[2]);
    return true;
}

// keep: every layer's activation stays in net->act (training's backward pass
// reads them); otherwise the first two layers may run fused and the first
// layer's activation is not stored.
static int forward(rt_cnn* net, int n, const bf16* x, hipStream_t s, bool keep = false) {
    if (!net->packed) return set_error(RT_ERR_STATE, "rt_cnn: parameters not set");
    net->act[0] = const_cast<bf16*>(x);
    const bool fused = !keep && forward_fused12(net, n, s);
    for (int l = fused ? 2 : 0; l < 6; l++) {
        ConvGeom g = geom(net, l, n);
        int M = n * g.Ho * g.Wo;
        if (forward_mfma(g, net->act[l], net->Wp[l], net->params + net->b_off[l], net->act[l + 1], s)) continue;
        dim3 grid((M + 63) / 64, (g.Co + 63) / 64);
        k_conv_fwd<<<grid, 256, 0, s>>>(g, net->act[l], net->Wp[l], net->params + net->b_off[l], net->act[l + 1]);
    }
    return hipGetLastError() == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn forward launch");
}

// The input gradient of one layer. The parity-class kernel takes Cout and Cin
// that are multiples of 32 (a stage of k then lies in one tap, a tile's
// columns in the tensor); 16-channel layers run the general kernel. The tile
// is the largest that still gives 512 workgroups, since a workgroup's stages
// wait on their loads one after the other.
static void backward_data(const ConvGeom& g, const bf16* dZ, const bf16* WT, const bf16* X, bf16* dX, hipStream_t s) {
    if (g.Co % 32 || g.Ci % 32) {
        const int Mi = g.B * g.Hi * g.Wi;
        k_conv_bwd_data<<<dim3((Mi + 63) / 64, (g.Ci + 63) / 64), 256, 0, s>>>(g, dZ, WT, X, dX);
        return;
    }
    const int M = g.B * ((g.Hi + 1) / 2) * ((g.Wi + 1) / 2);  // the largest class
    const int bn = g.Ci % 64 ? 32 : 64;
    auto grid = [&](int bm) { return dim3((M + bm - 1) / bm, g.Ci / bn, 4); };
    auto blocks = [&](int bm) { return (long)grid(bm).x * grid(bm).y * 4; };
    if (bn == 32) {
        k_conv_bwd_data_lds<128, 32, 4, 32><<<grid(128), 256, 0, s>>>(g, dZ, WT, X, dX);
    } else if (blocks(128) >= 512) {
        k_conv_bwd_data_lds<128, 64, 4, 32><<<grid(128), 256, 0, s>>>(g, dZ, WT, X, dX);
    } else if (g.Co % 64) {
        k_conv_bwd_data_lds<64, 64, 2, 32><<<grid(64), 256, 0, s>>>(g, dZ, WT, X, dX);
    } else if (blocks(64) >= 512) {
        k_conv_bwd_data_lds<64, 64, 2, 64><<<grid(64), 256, 0, s>>>(g, dZ, WT, X, dX);
    } else {
        k_conv_bwd_data_lds<32, 64, 2, 64><<<grid(32), 256, 0, s>>>(g, dZ, WT, X, dX);
    }
}

// forward + backward into net->grads; loss into net->loss[0] (device)
static int loss_grad(rt_cnn* net, int n, const bf16* x, const float* y, const float* wn, hipStream_t s) {
    int rc = forward(net, n, x, s, true);
    if (rc) return rc;
    const int C6 = net->cfg.channels[6], P6 = net->H[6] * net->W[6];
    bf16* dz = net->dz_a;
    bf16* dz_other = net->dz_b;
    k_head<<<n, 256, 2 * C6 * 4, s>>>(P6, C6, net->act[6], net->params + net->fc_w, net->params + net->fc_b, y, wn, n,
                                      net->out, dz, net->ws_fc, net->ws_loss);
    RowSums sums;
    sums.n = 0;
    int blocks = 0;
    auto add = [&](const float* src, float* out, int S, int width, int K, int Kp) {
        int slices = 1;
        while (slices < 16 && slices < S) slices *= 2;
        sums.s[sums.n++] = RowSum{src, out, S, width, K, Kp, slices, blocks};
        const int cols = 2 * 64 * (16 / slices);
        blocks += (width + cols - 1) / cols;
    };
    for (int l = 5; l >= 0; l--) {
        ConvGeom g = geom(net, l, n);
        int S, chunk;
        wsplit(net, l, n, &S, &chunk);
        float* ws = net->ws + net->ws_off[l];
        float* ws_b = net->ws_b + net->wsb_off[l];
        dim3 gw((g.Co + 63) / 64, (g.Kp + 63) / 64, S);
        k_conv_bwd_w<<<gw, 256, 0, s>>>(g, dz, net->act[l], ws, ws_b, chunk);
        add(ws, net->grads + net->w_off[l], S, g.Co * g.Kp, g.K, g.Kp);
        add(ws_b, net->grads + net->b_off[l], S, g.Co, 0, 0);
        if (l > 0) {
            backward_data(g, dz, net->WT[l], net->act[l], dz_other, s);
            std::swap(dz, dz_other);
        }
    }
    add(net->ws_fc, net->grads + net->fc_w, n, 6 * C6 + 6, 0, 0);
    add(net->ws_loss, net->loss, n, 2, 0, 0);
    k_row_sums<<<blocks, 1024, 0, s>>>(sums);
    return hipGetLastError() == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn backward launch");
}

static int check_batch(rt_cnn* net, int n, const void* x) {
    if (!net || !x || n < 1 || n > net->max_batch) return set_error(RT_ERR_ARG, "rt_cnn: bad batch");
    if (hipSetDevice(net->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    return RT_OK;
}

extern "C" int rt_cnn_forward(rt_cnn* net, int n, const uint16_t* x_dev, float* out_dev) {
    int rc = check_batch(net, n, x_dev);
    if (rc) return rc;
    if (!out_dev) return set_error(RT_ERR_ARG, "rt_cnn_forward: null output");
    if ((rc = forward(net, n, x_dev, net->stream))) return rc;
    const int C6 = net->cfg.channels[6], P6 = net->H[6] * net->W[6];
    k_head<<<n, 256, 2 * C6 * 4, net->stream>>>(P6, C6, net->act[6], net->params + net->fc_w, net->params + net->fc_b,
                                                nullptr, nullptr, 0, out_dev, nullptr, nullptr, nullptr);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_cnn head launch");
    return RT_OK;
}

extern "C" int rt_cnn_loss_grad(rt_cnn* net, int n, const uint16_t* x_dev, const float* y_dev, const float* w_dev,
                                float* loss, float* out_host, float* grad_host) {
    int rc = check_batch(net, n, x_dev);
    if (rc) return rc;
    if (!y_dev || !w_dev) return set_error(RT_ERR_ARG, "rt_cnn_loss_grad: null targets");
    if ((rc = loss_grad(net, n, x_dev, y_dev, w_dev, net->stream))) return rc;
    bool ok = true;
    if (loss) ok = ok && hipMemcpyAsync(loss, net->loss, 4, hipMemcpyDeviceToHost, net->stream) == hipSuccess;
    if (out_host) ok = ok && hipMemcpyAsync(out_host, net->out, 24 * (size_t)n, hipMemcpyDeviceToHost, net->stream) == hipSuccess;
    if (grad_host) ok = ok && hipMemcpyAsync(grad_host, net->grads, 4 * net->nparams, hipMemcpyDeviceToHost, net->stream) == hipSuccess;
    ok = ok && hipStreamSynchronize(net->stream) == hipSuccess;
    return ok ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn_loss_grad: copy");
}

extern "C" int rt_cnn_train_step(rt_cnn* net, int n, const uint16_t* x_dev, const float* y_dev, const float* w_dev,
                                 float lr, float* loss) {
    int rc = check_batch(net, n, x_dev);
    if (rc) return rc;
    if (!y_dev || !w_dev || !(lr >= 0)) return set_error(RT_ERR_ARG, "rt_cnn_train_step: bad argument");
    if ((rc = loss_grad(net, n, x_dev, y_dev, w_dev, net->stream))) return rc;
    net->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    float c1 = (float)(1.0 - pow(0.9, net->step)), c2 = (float)(1.0 - pow(0.999, net->step));
    size_t P = net->nparams;
    k_adam<<<(unsigned)((P + 255) / 256), 256, 0, net->stream>>>(net->params, net->grads, net->adam_m, net->adam_v, P, lr, b1,
                                                                  b2, c1, c2, 1e-8f);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_cnn adam launch");
    if ((rc = pack(net, net->stream))) return rc;
    if (loss) {
        if (hipMemcpyAsync(loss, net->loss, 4, hipMemcpyDeviceToHost, net->stream) != hipSuccess ||
            hipStreamSynchronize(net->stream) != hipSuccess)
            return set_error(RT_ERR_HIP, "rt_cnn_train_step: loss copy");
    }
    return RT_OK;
}

extern "C" int rt_cnn_augment(rt_cnn* net, int n, const uint16_t* x_dev, const float* y_dev, const float* y_inv_dev,
                              const int* flags, uint16_t* x_out, float* y_out) {
    int rc = check_batch(net, n, x_dev);
    if (rc) return rc;
    if (!y_dev || !y_inv_dev || !flags || !x_out || !y_out) return set_error(RT_ERR_ARG, "rt_cnn_augment: null argument");
    if (net->cfg.channels[0] != 4) return set_error(RT_ERR_UNSUPPORTED, "rt_cnn_augment: 4-channel inputs only");
    if (!net->st_flags.upload(net->flags_dev, flags, 4 * (size_t)n, net->stream))
        return set_error(RT_ERR_HIP, "rt_cnn_augment: flags copy");
    int cells = net->cfg.in_width * net->cfg.in_height;
    k_augment<<<dim3((cells + 255) / 256, n), 256, 0, net->stream>>>(x_dev, y_dev, y_inv_dev, net->flags_dev, net->cfg.in_width,
                                                                     net->cfg.in_height, x_out, y_out);
    return hipGetLastError() == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn_augment launch");
}

static int make_inputs(rt_cnn* net, int n, const FrameSrc* src, bf16* x, hipStream_t s) {
    for (int i = 0; i < n; i++) {
        const FrameSrc& f = src[i];
        if (!f.g8[0] || !f.g8[1] || !f.d16[0] || !f.d16[1]) return set_error(RT_ERR_ARG, "rt_cnn: null frame");
        if (f.W < net->cfg.in_width || f.H < net->cfg.in_height || f.W % net->cfg.in_width || f.H % net->cfg.in_height)
            return set_error(RT_ERR_ARG, "rt_cnn: frame size must be a multiple of the network input size");
    }
    if (!net->st_src.upload(net->src_dev, src, sizeof(FrameSrc) * (size_t)n, s))
        return set_error(RT_ERR_HIP, "rt_cnn: frame table copy");
    int cells = net->cfg.in_width * net->cfg.in_height;
    k_inputs<<<dim3((cells + 255) / 256, n), 256, 0, s>>>(net->src_dev, net->cfg.in_width, net->cfg.in_height, x);
    return hipGetLastError() == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn inputs launch");
}

extern "C" int rt_cnn_make_inputs(rt_cnn* net, int n, const rt_pair* pairs, uint16_t* x_dev) {
    int rc = check_batch(net, n, x_dev);
    if (rc) return rc;
    if (!pairs) return set_error(RT_ERR_ARG, "rt_cnn_make_inputs: null pairs");
    std::vector<FrameSrc> src(n);
    for (int i = 0; i < n; i++) {
        src[i].W = pairs[i].width; src[i].H = pairs[i].height;
        src[i].g8[0] = pairs[i].ref_gray; src[i].g8[1] = pairs[i].cur_gray;
        src[i].d16[0] = pairs[i].ref_depth; src[i].d16[1] = pairs[i].cur_depth;
    }
    if ((rc = make_inputs(net, n, src.data(), x_dev, net->stream))) return rc;
    return hipStreamSynchronize(net->stream) == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_cnn_make_inputs: sync");
}

namespace rt {
bool cnn_cells8(const rt_cnn* net, int W, int H) {
    return net && net->cfg.in_width * 8 == W && net->cfg.in_height * 8 == H;
}

int cnn_propose(rt_cnn* net, int n, const FrameSrc* src, float* trel_dev, hipStream_t s, const bf16* x_ready) {
    if (!net || n < 1 || n > net->max_batch) return set_error(RT_ERR_ARG, "rt_batch_propose: batch larger than the network's max_batch");
    if (!net->packed) return set_error(RT_ERR_STATE, "rt_batch_propose: network parameters not set");
    if (hipSetDevice(net->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    const bf16* x = x_ready;
    int rc = 0;
    if (!x) {
        if ((rc = make_inputs(net, n, src, net->xin, s))) return rc;
        x = net->xin;
    }
    if ((rc = forward(net, n, x, s))) return rc;
    const int C6 = net->cfg.channels[6], P6 = net->H[6] * net->W[6];
    k_head<<<n, 256, 2 * C6 * 4, s>>>(P6, C6, net->act[6], net->params + net->fc_w, net->params + net->fc_b, nullptr,
                                      nullptr, 0, net->out, nullptr, nullptr, nullptr);
    k_outputs_to_trel<<<(n + 255) / 256, 256, 0, s>>>(net->out, n, net->cfg.rot_scale_deg * (float)(M_PI / 180.0),
                                                      net->cfg.trans_scale_mm, trel_dev);
    return hipGetLastError() == hipSuccess ? RT_OK : set_error(RT_ERR_HIP, "rt_batch_propose launch");
}
}  // namespace rt

// ---------------------------------------------------------------- host pose conversions
static void log_rotation(const double* T, double w[3]) {
    // rotation vector of the 3x3 block of a row-major 4x4
    double R[9] = {T[0], T[1], T[2], T[4], T[5], T[6], T[8], T[9], T[10]};
    double sx = R[7] - R[5], sy = R[2] - R[6], sz = R[3] - R[1];
    double s = 0.5 * sqrt(sx * sx + sy * sy + sz * sz);
    double c = 0.5 * (R[0] + R[4] + R[8] - 1.0);
    double th = atan2(s, c);
    if (th < 1e-9) { w[0] = 0.5 * sx; w[1] = 0.5 * sy; w[2] = 0.5 * sz; return; }
    if (M_PI - th < 1e-6) {
        // near pi: axis from the diagonal
        double ax[3] = {sqrt(std::max(0.0, (R[0] + 1) / 2)), sqrt(std::max(0.0, (R[4] + 1) / 2)), sqrt(std::max(0.0, (R[8] + 1) / 2))};
        if (R[1] < 0) ax[1] = -ax[1];
        if (R[2] < 0) ax[2] = -ax[2];
        for (int k = 0; k < 3; k++) w[k] = th * ax[k];
        return;
    }
    double f = th / (2.0 * s);
    w[0] = f * sx; w[1] = f * sy; w[2] = f * sz;
}

extern "C" int rt_cnn_pose_to_target(const rt_cnn_config* c, int n, const double* Trel, float* y) {
    if (!c || !Trel || !y || n < 0) return set_error(RT_ERR_ARG, "rt_cnn_pose_to_target: bad argument");
    double rs = c->rot_scale_deg * M_PI / 180.0;
    for (int i = 0; i < n; i++) {
        const double* T = Trel + 16 * (size_t)i;
        double w[3];
        log_rotation(T, w);
        for (int k = 0; k < 3; k++) {
            y[6 * i + k] = (float)(w[k] / rs);
            y[6 * i + 3 + k] = (float)(T[4 * k + 3] / c->trans_scale_mm);
        }
    }
    return RT_OK;
}

extern "C" int rt_cnn_target_to_pose(const rt_cnn_config* c, int n, const float* y, double* Trel) {
    if (!c || !Trel || !y || n < 0) return set_error(RT_ERR_ARG, "rt_cnn_target_to_pose: bad argument");
    double rs = c->rot_scale_deg * M_PI / 180.0;
    for (int i = 0; i < n; i++) {
        double w[3], t[3];
        for (int k = 0; k < 3; k++) { w[k] = y[6 * i + k] * rs; t[k] = (double)y[6 * i + 3 + k] * c->trans_scale_mm; }
        double th = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
        double A = th > 1e-12 ? sin(th) / th : 1.0, B = th > 1e-12 ? (1.0 - cos(th)) / (th * th) : 0.5;
        double K[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
        double* T = Trel + 16 * (size_t)i;
        for (int r = 0; r < 3; r++) {
            for (int q = 0; q < 3; q++) {
                double k2 = 0.0;
                for (int m = 0; m < 3; m++) k2 += K[3 * r + m] * K[3 * m + q];
                T[4 * r + q] = (r == q ? 1.0 : 0.0) + A * K[3 * r + q] + B * k2;
            }
            T[4 * r + 3] = t[r];
        }
        T[12] = 0; T[13] = 0; T[14] = 0; T[15] = 1;
    }
    return RT_OK;
}
