// Truncated signed distance fusion into a voxel grid and ray casting of the
// grid (the reference's VoxelGrid, kernels/VoxelGrid_cuda.cu). Every FP32
// value follows the reference's operation order (the library is built with
// -ffp-contract=off).
#include <hip/hip_runtime.h>

#include <float.h>
#include <math.h>
#include <string.h>

#include <cmath>
#include <type_traits>

#include "rt_device.hpp"
#include "rt_host.hpp"
#include "rt_tsdf.h"

#ifndef TSDF_AHEAD
#define TSDF_AHEAD 8  // voxels of a ray that are walked as one group (at most 8: the smallest skip block)
#endif

namespace rt {

struct TsdfArgs {
    int res, w, h;
    float ox, oy, oz;     // cube centre
    float dx, dy, dz;     // half-extent
    float vx, vy, vz;     // dim / res: half the voxel edge
    float mn, mx;
    float T[16];          // update: world -> camera; ray cast: camera -> world
    float K[9];
};

// Beside the voxels the grid keeps which of them are negative (behind a
// surface), so that a ray can pass empty space without reading voxels:
//   neg  one bit per voxel, x fastest, rows padded to 16 * nx bits
//   occ  one byte per 16 x 4 x 4 voxels: bit k if one of x 4 k .. 4 k + 3 is
//        negative
// Every kernel that writes voxels keeps both exact.
struct TsdfMap {
    uint16_t* neg;
    uint8_t* occ;
    int nx, ny;  // tiles of 16 along x, of 4 along y
};
__device__ __forceinline__ size_t map_tile(const TsdfMap& m, int xt, int y4, int z4) {
    return ((size_t)z4 * m.ny + y4) * m.nx + xt;
}
// which of the four nibbles of 16 signs hold one
__device__ __forceinline__ unsigned nibbles(unsigned r) {
    return ((r & 0xfu) ? 1u : 0u) | ((r & 0xf0u) ? 2u : 0u) | ((r & 0xf00u) ? 4u : 0u) | ((r & 0xf000u) ? 8u : 0u);
}
// the occ byte of a tile from its four slices' signs (16 bits per row of four
// rows), one per lane of a group of four lanes
__device__ __forceinline__ unsigned occ_of_words(unsigned long long w) {
    unsigned r = (unsigned)w | (unsigned)(w >> 32);
    r |= r >> 16;
    unsigned f = nibbles(r);
    f |= __shfl_xor(f, 1); f |= __shfl_xor(f, 2);
    return f;
}
// four rows' 16 signs of a tile's slice, in one word
__device__ __forceinline__ unsigned long long load_rows(const uint16_t* p, int nx) {
    return (unsigned long long)(p[0] | (unsigned)p[nx] << 16) |
           (unsigned long long)(p[2 * (size_t)nx] | (unsigned)p[3 * (size_t)nx] << 16) << 32;
}
__device__ __forceinline__ void store_rows(uint16_t* p, int nx, unsigned long long v) {
#pragma unroll
    for (int k = 0; k < 4; k++) p[k * (size_t)nx] = (uint16_t)(v >> 16 * k);
}

// What the update needs to pass over 16 x 4 voxels of a z slice that all
// project outside the image. u < 1 is f(p) / rz < 0 with the linear function
// f = K0 rx + (K2 - 1 / w) rz, and so on for the other three borders, so a
// slice is out where rz and f keep their signs over it: the value at its
// centre exceeds the reach ex0 .. of the slice, which holds a margin of 40
// times the rounding error of the projection (a slice that is kept for
// nothing costs time, not correctness).
struct TsdfCull {
    float cx0, cx1, cy0, cy1;    // K2 - 1 / w, K2 - (w - 2) / w, and the same of K5, h
    float ex0, ex1, ey0, ey1, ez;
    float umax, vmax;            // w - 2, h - 2, rounded up where float does not hold them
    float islope, nlo, nhi;      // RN(1 / slope) and the numerators for which it serves div_rn
};

// rx / rz and ry / rz, the IEEE quotients. With all three between 2^-60 and
// 2^60 in magnitude nothing over- or underflows, the reciprocal is RN(1 / rz)
// (rcp_rn's range) and div_rn is exact; a zero, a huge or a tiny value takes the
// divisions. Twelve instructions for about 22.
__device__ __forceinline__ void quotients(float rx, float ry, float rz, float& qx, float& qy) {
    const float big = 1152921504606846976.0f, small = 1.0f / 1152921504606846976.0f;
    const float y = rcp_rn(rz);
    qx = div_rn(rx, rz, y); qy = div_rn(ry, rz, y);
    const float hi = fmaxf(fmaxf(fabsf(rx), fabsf(ry)), fabsf(rz)), lo = fminf(fminf(fabsf(rx), fabsf(ry)), fabsf(rz));
    if (!(hi <= big && lo >= small)) { qx = rx / rz; qy = ry / rz; }
}

// updateVoxelsKernel (VoxelGrid_cuda.cu:944-1014)
// A wave takes 16 x 4 voxels (128-byte runs) of UPDATE_Z slices. Its lanes
// first test one slice each against the image (TsdfCull), then the slices that
// are left go through four at a time, their depth and voxel loads together in
// flight; the products that depend on z alone come from the lane that made
// them. The voxel is read and written only where it is updated, and a wave
// that changed any voxel brings the tile's signs and occ bytes up to date.
// Bound by vector instructions (about 110 per slice that is left, busy for four
// fifths of the time): 29 us at 256^3 and 320 x 240 with 40 % of the slices in
// the image, where one thread per voxel and two divisions each took 38. Grids of
// up to 128^3 take 1 us longer than so: bringing the signs up to date is a load
// and a store more, which the ray cast gives back (10 us and more from 64^3 on).
__device__ __forceinline__ float from_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
template <int UPDATE_Z>
__global__ __launch_bounds__(256) void k_tsdf_update(float2* __restrict__ tsdf, TsdfMap map, const float* __restrict__ dist,
                                                     TsdfArgs a, TsdfCull c) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xt = blockIdx.x, y4 = blockIdx.y * 4 + wave, z0 = blockIdx.z * UPDATE_Z;
    const int res = a.res;
    if (y4 >= map.ny) return;
    const float* K = a.K;
    const float* T = a.T;
    const int w = a.w;
    const float fw = (float)a.w, fh = (float)a.h;
    const float sx = a.ox - a.dx + a.vx, sy = a.oy - a.dy + a.vy, sz = a.oz - a.dz + a.vz;  // first voxel centre
    const float ex = a.vx * 2, ey = a.vy * 2, ez = a.vz * 2;                                // voxel edge
    // lane l: slice z0 + (l & 15)
    const int zl = z0 + (lane & (UPDATE_Z - 1));
    const float pzl = sz + (float)zl * ez;
    const float zx = T[2] * pzl, zy = T[6] * pzl, zz = T[10] * pzl;
    unsigned live;
    {
        const float cx = sx + ((float)(xt * 16) + 7.5f) * ex, cy = sy + ((float)(y4 * 4) + 1.5f) * ey;
        const float rx = T[0] * cx + T[1] * cy + zx + T[3], ry = T[4] * cx + T[5] * cy + zy + T[7],
                    rz = T[8] * cx + T[9] * cy + zz + T[11];
        const float x0 = K[0] * rx + c.cx0 * rz, x1 = K[0] * rx + c.cx1 * rz;
        const float y0 = K[4] * ry + c.cy0 * rz, y1 = K[4] * ry + c.cy1 * rz;
        const bool front = rz < -c.ez && (x0 > c.ex0 || x1 < -c.ex1 || y0 > c.ey0 || y1 < -c.ey1);
        const bool back = rz > c.ez && (x0 < -c.ex0 || x1 > c.ex1 || y0 < -c.ey0 || y1 > c.ey1);
        live = (unsigned)__ballot(!front && !back && zl < res) & ((1u << UPDATE_Z) - 1);
    }
    if (!live) return;
    const int x = xt * 16 + (lane & 15), y = y4 * 4 + (lane >> 4);
    const bool inx = x < res;
    const float px = sx + (float)x * ex, py = sy + (float)y * ey;
    const float ax = T[0] * px + T[1] * py, ay = T[4] * px + T[5] * py, az = T[8] * px + T[9] * py;
    const size_t slice = (size_t)res * res, base = (size_t)xt * 16 + (size_t)y4 * 4 * res + z0 * slice;
    const size_t own = base + (inx ? (lane & 15) + (size_t)(lane >> 4) * res : 0);
    const float vmin = a.vx * 2, tol = a.dx / 200.0f, slope = a.dx * 0.030f, far = -1.2501f * slope;
    unsigned long long myupd = 0, myneg = 0;  // lane l < UPDATE_Z: slice z0 + l
    for (int z4 = 0; z4 < UPDATE_Z; z4 += 4) {
        if (!(live >> z4 & 15u)) continue;
        float u[4], v[4], dz[4];
        bool ok[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float rx = ax + from_lane(zx, z4 + j) + T[3], ry = ay + from_lane(zy, z4 + j) + T[7],
                        rz = az + from_lane(zz, z4 + j) + T[11];
            float qx, qy;
            quotients(rx, ry, rz, qx, qy);
            dz[j] = -rz;  // the voxel's distance
            u[j] = (qx * K[0] + K[2]) * fw; v[j] = (qy * K[4] + K[5]) * fh;
            // 1 <= (int)u < w - 2; a projection that is not a number is out
            ok[j] = inx & (u[j] >= 1.0f) & (u[j] < c.umax) & (v[j] >= 1.0f) & (v[j] < c.vmax) & ((live >> (z4 + j) & 1u) != 0);
        }
        if (!__any(ok[0] | ok[1] | ok[2] | ok[3])) continue;
        float m[4][4], lo[4], hi[4], nt[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            u[j] = ok[j] ? u[j] : 1.0f; v[j] = ok[j] ? v[j] : 1.0f;
            const float* p = dist + ((size_t)(int)u[j] + (size_t)(int)v[j] * w);
            m[j][0] = p[0]; m[j][1] = p[1]; m[j][2] = p[w]; m[j][3] = p[w + 1];
        }
        // No depth near, or the voxel further behind the largest of the four than
        // the sdf below may be (the interpolated one is not above it by more than
        // its rounding): most of what projects into the image ends here.
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo[j] = fminf(fminf(m[j][0], m[j][1]), fminf(m[j][2], m[j][3]));
            hi[j] = fmaxf(fmaxf(m[j][0], m[j][1]), fmaxf(m[j][2], m[j][3]));
            ok[j] = ok[j] & !(lo[j] < vmin) & !(hi[j] * 1.00001f - dz[j] < far);
        }
        if (!__any(ok[0] | ok[1] | ok[2] | ok[3])) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float fu = u[j] - (int)u[j], fv = v[j] - (int)v[j];
            const float d = ((1 - fu) * (1 - fv) * m[j][0] + fu * (1 - fv) * m[j][1] + (1 - fu) * fv * m[j][2] +
                             fu * fv * m[j][3]);
            // the IEEE quotient; see quotients() for the range
            const float n = -(dz[j] - d);
            float sdf = div_rn(n, slope, c.islope);
            if (!(fabsf(n) >= c.nlo && fabsf(n) <= c.nhi)) sdf = n / slope;
            // |d - m| of all four at most tol: the largest is that of lo or hi
            ok[j] = ok[j] & !(fmaxf(d - lo[j], hi[j] - d) > tol) & !(sdf < -1.25f);
            nt[j] = fmaxf(fminf(1.0f, sdf), -1.0f);
        }
        if (!__any(ok[0] | ok[1] | ok[2] | ok[3])) continue;
        float2 t[4];
        // lanes without an update read the tile's first voxel
#pragma unroll
        for (int j = 0; j < 4; j++) t[j] = tsdf[ok[j] ? own + (z4 + j) * slice : base];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            t[j].x = (t[j].y * t[j].x + 1.0f * nt[j]) / (t[j].y + 1.0f);
            t[j].y = fminf(1.0f + t[j].y, 16.0f);
            if (ok[j]) tsdf[own + (z4 + j) * slice] = t[j];
            const unsigned long long upd = __ballot(ok[j]), neg = __ballot(ok[j] && t[j].x < 0.0f);
            myupd = lane == z4 + j ? upd : myupd;
            myneg = lane == z4 + j ? neg : myneg;
        }
    }
    if (!__any(myupd != 0)) return;
    if (lane >= UPDATE_Z || zl >= res) return;
    uint16_t* row = map.neg + ((size_t)zl * res + y4 * 4) * map.nx + xt;
    const unsigned long long old = load_rows(row, map.nx), now = (old & ~myupd) | myneg;
    if (now != old) store_rows(row, map.nx, now);
    const unsigned f = occ_of_words(now);
    if ((lane & 3) == 0) map.occ[map_tile(map, xt, y4, zl >> 2)] = (uint8_t)f;
}

__global__ __launch_bounds__(256) void k_tsdf_reset(float2* __restrict__ tsdf, TsdfMap map, size_t n, size_t words,
                                                    size_t tiles) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) tsdf[i] = make_float2(1.0f, 0.0f);
    if (i < words) map.neg[i] = 0;  // words, tiles <= n: at least eight voxels each
    if (i < tiles) map.occ[i] = 0;
}

// reconstructionKernel (VoxelGrid_cuda.cu:1088-1110): rows read bottom-up
__global__ __launch_bounds__(256) void k_tsdf_dist_rgbd(const float4* __restrict__ rgbd, int w, int h, float mn, float mx,
                                                        float* __restrict__ dist) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15), y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= w || y >= h) return;
    const float wv = rgbd[(size_t)x + (size_t)(h - 1 - y) * w].w;
    const float tol = 1e-4f;
    dist[(size_t)x + (size_t)y * w] = (wv > tol && wv < (1.0f - tol)) ? wv * (mx - mn) + mn : 0.0f;
}
__global__ __launch_bounds__(256) void k_tsdf_dist_u16(const uint16_t* __restrict__ d, size_t n, float* __restrict__ dist) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dist[i] = (float)d[i];
}

// trilinearDensity (VoxelGrid_cuda.cu:181-222) at grid coordinates p. The
// cell index and the eight addresses are the reference's; an address past the
// grid's last voxel (the reference reads beyond the array there) is held at
// the last voxel.
__device__ __forceinline__ float trilinear(const float2* __restrict__ g, int res, float px, float py, float pz) {
    const unsigned lim = (unsigned)res + 1;
    const unsigned ix = px > 0.0f ? min((unsigned)fminf(px, (float)lim), lim) : 0u;
    const unsigned iy = py > 0.0f ? min((unsigned)fminf(py, (float)lim), lim) : 0u;
    const unsigned iz = pz > 0.0f ? min((unsigned)fminf(pz, (float)lim), lim) : 0u;
    const float fx = px - ix, fy = py - iy, fz = pz - iz;
    const unsigned ys = res, zs = ys * ys, last = zs * ys - 1;  // res <= 1024: below 2^31 with the cell past the grid
    const unsigned o = ix + iy * ys + iz * zs;
    auto at = [&](unsigned a) { return g[min(a, last)].x; };
    const float d000 = at(o), d001 = at(o + zs), d010 = at(o + ys), d011 = at(o + ys + zs);
    const float d100 = at(o + 1), d101 = at(o + 1 + zs), d110 = at(o + 1 + ys), d111 = at(o + 1 + ys + zs);
    const float x00 = (1 - fx) * d000 + fx * d100, x01 = (1 - fx) * d001 + fx * d101;
    const float x10 = (1 - fx) * d010 + fx * d110, x11 = (1 - fx) * d011 + fx * d111;
    const float z0 = (1 - fy) * x00 + fy * x10, z1 = (1 - fy) * x01 + fy * x11;
    return (1 - fz) * z0 + fz * z1;
}
// resampleVoxelsKernel with trilinearDensity / trilinearWeight
// (VoxelGrid_cuda.cu:181-262, 897-939): T maps dst voxel centres into src
__host__ __device__ __forceinline__ int resample_xcds(int res) { return res > 256 ? 8 : 1; }
// The resampled voxel (ix, iy, iz); (1, 0) outside src.
__device__ __forceinline__ float2 resampled(const float2* __restrict__ src, const TsdfArgs& a, int ix, int iy, int iz) {
    const int res = a.res;
    const float* T = a.T;
    const float sx = a.ox - a.dx + a.vx, sy = a.oy - a.dy + a.vy, sz = a.oz - a.dz + a.vz;
    const float ex = a.vx * 2, ey = a.vy * 2, ez = a.vz * 2;
    const float px = sx + ix * ex, py = sy + iy * ey, pz = sz + iz * ez;
    const float rx = T[0] * px + T[1] * py + T[2] * pz + T[3];
    const float ry = T[4] * px + T[5] * py + T[6] * pz + T[7];
    const float rz = T[8] * px + T[9] * py + T[10] * pz + T[11];
    const float qx = (rx - sx) / ex, qy = (ry - sy) / ey, qz = (rz - sz) / ez;
    const float hi = (float)(res - 2);
    float2 out = make_float2(1.0f, 0.0f);
    // in range, so the cell index is at most res-2 on every axis and all eight reads are inside the grid
    if (qx >= 0 && qx <= hi && qy >= 0 && qy <= hi && qz >= 0 && qz <= hi) {
        const unsigned cx = (unsigned)qx, cy = (unsigned)qy, cz = (unsigned)qz;
        const float fx = qx - cx, fy = qy - cy, fz = qz - cz;
        const size_t ys = res, zs = (size_t)res * res;
        const size_t o = cx + cy * ys + cz * zs;
        const float2 d000 = src[o], d001 = src[o + zs], d010 = src[o + ys], d011 = src[o + ys + zs];
        const float2 d100 = src[o + 1], d101 = src[o + 1 + zs], d110 = src[o + 1 + ys], d111 = src[o + 1 + ys + zs];
        float r2[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float a000 = c ? d000.y : d000.x, a001 = c ? d001.y : d001.x, a010 = c ? d010.y : d010.x,
                        a011 = c ? d011.y : d011.x, a100 = c ? d100.y : d100.x, a101 = c ? d101.y : d101.x,
                        a110 = c ? d110.y : d110.x, a111 = c ? d111.y : d111.x;
            const float x00 = (1 - fx) * a000 + fx * a100, x01 = (1 - fx) * a001 + fx * a101;
            const float x10 = (1 - fx) * a010 + fx * a110, x11 = (1 - fx) * a011 + fx * a111;
            const float z0 = (1 - fy) * x00 + fy * x10, z1 = (1 - fy) * x01 + fy * x11;
            r2[c] = (1 - fz) * z0 + fz * z1;
        }
        out = make_float2(r2[0], r2[1]);
    }
    return out;
}
// A workgroup takes 64 x 4 x 4 voxels, a wave the rows of four slices: reads
// and writes run along x in 512 bytes, and the four tiles' occ bytes need no
// other workgroup. Bound by memory. What it costs beyond the voxels are the sign
// words, 8 bytes of a row per wave: past 256 voxels an axis the workgroups of a
// row run on one XCD (dispatch is round-robin over 8), so that they meet in one
// L2. us without the map, and with it in this order or x before y:
//   256^3 72, 76 / 73   384^3 251, 255 / 262   512^3 575, 586 / 615   768^3 1863, 1980 / 2088
// under a translation; 73, 76 at 256^3 and 605, 690 at 512^3 with a rotation, whose
// reads stray. (Tiles of 16 x 4 voxels and eight slices a wave took 94 and 926.)
__global__ __launch_bounds__(256) void k_tsdf_resample(float2* __restrict__ dst, TsdfMap map, const float2* __restrict__ src,
                                                       TsdfArgs a) {
    __shared__ unsigned long long rows[4];
    const int res = a.res, nxb = (res + 63) / 64, xcds = resample_xcds(res);
    const int b = blockIdx.x / xcds, xb = b % nxb, y4 = b / nxb * xcds + blockIdx.x % xcds, z4 = blockIdx.y;
    if (y4 >= map.ny) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, xt = xb * 4 + (threadIdx.x & 3);
    const int ix = xb * 64 + lane, iy = y4 * 4 + wave;
    unsigned long long any = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int iz = z4 * 4 + k;
        float2 out = make_float2(1.0f, 0.0f);
        if (ix < res) {
            out = resampled(src, a, ix, iy, iz);
            dst[ix + (size_t)iy * res + (size_t)iz * res * res] = out;
        }
        const unsigned long long neg = __ballot(out.x < 0.0f);
        any |= neg;
        if (lane < 4 && xt < map.nx) map.neg[((size_t)iz * res + iy) * map.nx + xt] = (uint16_t)(neg >> 16 * lane);
    }
    if (lane == 0) rows[wave] = any;
    __syncthreads();
    if (threadIdx.x < 4 && xt < map.nx) {
        const unsigned r = (unsigned)((rows[0] | rows[1] | rows[2] | rows[3]) >> 16 * lane);
        map.occ[map_tile(map, xt, y4, z4)] = (uint8_t)nibbles(r);
    }
}

// The skip table of a ray cast: for every block of (1 << LB)^3 voxels, whether
// one of the 27 blocks around it holds a negative voxel. A ray that stands in
// a block without one can move as many voxels as the block is wide along every
// axis and meet none. Blocks of 8 up to 512^3, of 16 above: at most 64 per
// row, so that the table (64 bits per row) fits into 32 KB of LDS. Blocks of 4
// at 256^3 read fewer voxels one by one, but took 107 us per ray cast for 79:
// the walk in between is the larger part.
// A row's bits stand in the order in which a wave makes them, lane l having
// the occ byte of voxels 16 l .. 16 l + 15; one wave per row.
__device__ __forceinline__ int skip_bit(int LB, int bx) { return LB == 3 ? (bx & 1) << 5 | bx >> 1 : bx; }
template <int LB>
__global__ __launch_bounds__(256) void k_tsdf_skip(TsdfMap map, int res, unsigned long long* __restrict__ skip) {
    const int lane = threadIdx.x & 63, nb = (res + (1 << LB) - 1) >> LB;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= nb * nb) return;
    const int bz = row / nb, by = row % nb;
    constexpr int S = LB - 2;  // tiles of four voxels of a block along y and z, as a shift
    const int z0 = max((bz - 1) << S, 0), z1 = min((bz + 2) << S, map.ny);
    const int y0 = max((by - 1) << S, 0), y1 = min((by + 2) << S, map.ny);
    unsigned f = 0;
    if (lane < map.nx)
        for (int z = z0; z < z1; z++)
#pragma unroll 3
            for (int y = y0; y < y1; y++) f |= map.occ[map_tile(map, lane, y, z)];
    const unsigned long long e = __ballot(f & 3u), o = __ballot(f & 12u);  // even and odd blocks of 8
    if (lane) return;
    if constexpr (LB == 3) {
        skip[row] = (unsigned)(e | o | o << 1) | (o | e | e >> 1) << 32;
    } else {
        const unsigned long long b = e | o;
        skip[row] = b | b << 1 | b >> 1;
    }
}

// estimateLinearZero (VoxelGrid_cuda.cu:558-561)
__device__ __forceinline__ float linear_zero(float tA, float dA, float tB, float dB) {
    const float s = fminf(fmaxf(dA / (dA - dB), 0.0f), 1.0f);
    return tA + s * (tB - tA);
}

// rayCastVoxelsKernel with initRay, intersectVoxelGridCuda and
// traverseVoxelsCuda (VoxelGrid_cuda.cu:118-164, 633-770)
//
// A ray's walk does not depend on what the voxels hold, and its time was the
// latency of reading them, then that of the walk itself: a 320 x 240 image is
// about one wave per SIMD, which waits for each result. A wave whose rays all
// stand in clear blocks of the skip table (in LDS) moves on by a block: the
// three axes advance each on their own, by the additions that the walk would
// make, up to a parameter that none of them overruns, so that what is left
// is a walk that went there voxel by voxel. Otherwise TSDF_AHEAD voxels are
// walked in turn, and their sign bits read together and tested in walk order.
// The voxel's centre, which only a negative voxel needs, is worked out there.
// 79 us at 256^3 and 320 x 240 (138 with every voxel of the walk read); a wave
// takes 44,000 cycles on average, the longest three times that.
//
// EXACT: no addition along the voxel centres rounds (see centres_exact), so a
// centre is its first coordinate plus a multiple of the edge. Otherwise it is
// carried along as the walk sums it, half as many instructions again.
template <int LB, bool EXACT>
__global__ __launch_bounds__(256) void k_tsdf_raycast(const float2* __restrict__ g, TsdfMap map,
                                                      const unsigned long long* __restrict__ skip, TsdfArgs a,
                                                      int refine, float4* __restrict__ out) {
    extern __shared__ unsigned long long rows[];
    const int nb = (a.res + (1 << LB) - 1) >> LB;
#pragma unroll 4
    for (int i = threadIdx.x; i < nb * nb; i += 256) rows[i] = skip[i];
    __syncthreads();
    const unsigned* tab = reinterpret_cast<const unsigned*>(rows);
    const int xi = blockIdx.x * 16 + (threadIdx.x & 15), yi = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (xi >= a.w || yi >= a.h) return;
    const float* K = a.K;
    const float* T = a.T;
    const int res = a.res;
    // initRay: the normalised pixel position through the inverse intrinsics, unit length
    const float pdx = (float)xi / (float)a.w, pdy = (float)yi / (float)a.h;
    float cx = -(pdx - K[2]) / K[0], cy = -(pdy - K[5]) / K[4], cz = -1.0f;
    float len = 0.0f;
    len += cx * cx; len += cy * cy; len += cz * cz;
    len = 1.0f / sqrtf(len);
    cx *= len; cy *= len; cz *= len;
    const float dx = T[0] * cx + T[1] * cy + T[2] * cz, dy = T[4] * cx + T[5] * cy + T[6] * cz,
                dz = T[8] * cx + T[9] * cy + T[10] * cz;
    const float ox = T[3], oy = T[7], oz = T[11];
    const int s0 = dx < 0, s1 = dy < 0, s2 = dz < 0;
    const float ivx = fabsf(dx) > 1e-6f ? 1.0f / dx : (1 - 2 * s0) * FLT_MAX;
    const float ivy = fabsf(dy) > 1e-6f ? 1.0f / dy : (1 - 2 * s1) * FLT_MAX;
    const float ivz = fabsf(dz) > 1e-6f ? 1.0f / dz : (1 - 2 * s2) * FLT_MAX;
    float4 result = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // intersectVoxelGridCuda: slab test against the cube
    const float bx[2] = {a.ox - a.dx, a.ox + a.dx}, by[2] = {a.oy - a.dy, a.oy + a.dy}, bz[2] = {a.oz - a.dz, a.oz + a.dz};
    const float x0 = (bx[s0] - ox) * ivx, x1 = (bx[1 - s0] - ox) * ivx;
    const float y0 = (by[s1] - oy) * ivy, y1 = (by[1 - s1] - oy) * ivy;
    const float z0 = (bz[s2] - oz) * ivz, z1 = (bz[1 - s2] - oz) * ivz;
    const float tmin = fmaxf(x0, fmaxf(y0, z0)), tmax = fminf(x1, fminf(y1, z1));
    if (!(tmin >= tmax || tmax <= 0)) {
        float enterT = tmin, exitT = tmax;
        const float vdx = 2.0f * a.vx, vdy = 2.0f * a.vy, vdz = 2.0f * a.vz;  // voxel edge
        const float ibx = a.ox - a.dx + a.vx, iby = a.oy - a.dy + a.vy, ibz = a.oz - a.dz + a.vz;
        enterT += vdx * 2; exitT -= vdx * 2;
        if (enterT < 0) enterT = 0;
        bool hit = false;
        float tHit = 0.0f;
        if (!(enterT + vdx * 2 > exitT)) {
            const float ivdx = 1.0f / vdx, ivdy = 1.0f / vdy, ivdz = 1.0f / vdz;
            // voxelize: the voxel the ray enters
            const float qx = (ox + enterT * dx - ibx) * ivdx, qy = (oy + enterT * dy - iby) * ivdy,
                        qz = (oz + enterT * dz - ibz) * ivdz;
            int vx = qx > 0.0f ? (int)fminf(qx, 2048.0f) : 0, vy = qy > 0.0f ? (int)fminf(qy, 2048.0f) : 0,
                vz = qz > 0.0f ? (int)fminf(qz, 2048.0f) : 0;  // 2048: past any grid
            float vpx = ibx + (float)vx * vdx, vpy = iby + (float)vy * vdy, vpz = ibz + (float)vz * vdz;
            const int gx = 1 - 2 * s0, gy = 1 - 2 * s1, gz = 1 - 2 * s2;
            const float stx = (float)gx * vdx, sty = (float)gy * vdy, stz = (float)gz * vdz;
            float tnx = (vpx + stx - ox) * ivx, tny = (vpy + sty - oy) * ivy, tnz = (vpz + stz - oz) * ivz;
            const float tsx = stx * ivx, tsy = sty * ivy, tsz = stz * ivz;
            int iter = refine ? 3 : 0;
            // t: the parameter of the last step, infinity once the ray's walk is over
            float t = vx < res && vy < res && vz < res ? enterT : INFINITY;
            // n <= N steps along an axis, one addition each
            constexpr int N = 8;  // at most a skip block's width, and TSDF_AHEAD
            static_assert(TSDF_AHEAD <= N, "a group's steps");
            auto along = [](float v, float st, int n) {
#pragma unroll
                for (int k = 0; k < N; k++) v = k < n ? v + st : v;
                return v;
            };
            // a group's voxels as one integer: x and y with 32 added, as a group
            // may leave the grid, in 12 bits each, above them its steps along z
            constexpr int BIAS = 32;
            int pos = 0;
            const int ix = gx, iy = gy * (1 << 12);
            auto px_of = [](int p) { return (p & 4095) - BIAS; };
            auto py_of = [](int p) { return (p >> 12 & 4095) - BIAS; };
            auto nz_of = [](int p) { return (int)((unsigned)p >> 24); };
            // bits of the sign map; at most 2^30
            const int pitch = map.nx * 16, plane = pitch * res, words = (int)((unsigned)plane * (unsigned)res / 32u);
            const int jx = gx, jy = gy * pitch, jz = gz * plane;
            const unsigned* neg = reinterpret_cast<const unsigned*>(map.neg);
            // The step to the nearest voxel wall: x if tnx < tny and tnx < tnz, else y if
            // tny <= tnx and tny < tnz, else z. The second comparison is with the nearer
            // of x and y, which is the same three-way choice (a NaN included). Each select
            // hangs on one comparison (no mask arithmetic, whose way through the scalar
            // unit costs a lone wave more than the two instructions it saves); adding 0
            // leaves a parameter as it is.
            bool wxy = false, wk = false;
            auto step = [&]() {
                wxy = tnx < tny;
                const float b = wxy ? tnx : tny;
                const float nx = tnx + (wxy ? tsx : 0.0f), ny = tny + (wxy ? 0.0f : tsy), nz = tnz + tsz;
                const int in = wxy ? ix : iy;
                wk = b < tnz;
                t = wk ? b : tnz;
                pos += wk ? in : 1 << 24;
                tnx = wk ? nx : tnx; tny = wk ? ny : tny; tnz = wk ? tnz : nz;
            };
            // A parameter that is not a number or -inf (rays along an axis, with a
            // start on a voxel wall) does not move by additions alone: such a ray
            // is always walked voxel by voxel.
            const float least = fminf(fminf(tnx, tny), tnz);
            const bool odd = !(least > -INFINITY) || isnan(tnx) || isnan(tny) || isnan(tnz) || isnan(tsx) || isnan(tsy) || isnan(tsz);
            // the grid check ends the walk within 3 * (res + 1) steps: each step moves one index one way
            while (true) {
                // The wave as a whole: a ray whose walk is over has nothing to step
                // below `until`, so that no lane leaves and the loop is two branches.
                bool fine = false;
                while (true) {
                    const bool in = (t < exitT) & (min(min(vx, vy), vz) >= 0) & (max(max(vx, vy), vz) < res);
                    const int row = (vz >> LB) * nb + (vy >> LB), bit = skip_bit(LB, vx >> LB), word = row * 2 + (bit >> 5);
                    const bool full = odd | (tab[in ? word : 0] >> (bit & 31) & 1u);
                    // the next steps are those below `until`: at most N along each axis
                    // (N - 1 by the sum, one more where the additions round)
                    const float next = fminf(fminf(tnx, tny), tnz);
                    const float bound = fminf(fminf(fminf(tnx + (N - 1) * tsx, tny + (N - 1) * tsy), tnz + (N - 1) * tsz), exitT);
                    // in a clear voxel that is the walk's last one: over
                    const bool on = in & (full | (next < exitT));
                    t = on ? t : INFINITY;
                    // no step below `bound`: the steps are too small for it
                    fine = on & (full | !(next < bound));
                    if (__any(fine) || !__any(on)) break;
                    const float until = on ? bound : -INFINITY;
                    int nx = 0, ny = 0, nz = 0;
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const bool bx = tnx < until, by = tny < until, bz = tnz < until;
                        const float ax = tnx + tsx, ay = tny + tsy, az = tnz + tsz;
                        tnx = bx ? ax : tnx; tny = by ? ay : tny; tnz = bz ? az : tnz;
                        nx += bx ? 1 : 0; ny += by ? 1 : 0; nz += bz ? 1 : 0;
                        if constexpr (!EXACT) {
                            vpx = bx ? vpx + stx : vpx; vpy = by ? vpy + sty : vpy; vpz = bz ? vpz + stz : vpz;
                        }
                    }
                    vx += gx * nx; vy += gy * ny; vz += gz * nz;
                    // t stays: like the parameter of the last step it is below exitT
                }
                if (!__any(fine)) break;
                if (t < exitT) {
                    pos = (vx + BIAS) | (vy + BIAS) << 12;
                    // the sign bits of the group, read back to back; a word past the
                    // map is held at its last one, and what lies past the exit or the
                    // grid is told when its bit is set
                    int at[TSDF_AHEAD];
                    float ta[TSDF_AHEAD];
                    unsigned word[TSDF_AHEAD];
                    int idx = vz * plane + vy * pitch + vx;
                    unsigned cand = 0;
#pragma unroll
                    for (int j = 0; j < TSDF_AHEAD; j++) {
                        at[j] = pos; ta[j] = t;
                        word[j] = neg[min((unsigned)idx >> 5, (unsigned)words - 1)] >> (idx & 31);
                        step();
                        idx += wk ? (wxy ? jx : jy) : jz;
                    }
                    const int vx0 = vx, vy0 = vy, vz0 = vz;
                    vx = px_of(pos); vy = py_of(pos); vz += gz * nz_of(pos);
                    const float cvx = vpx, cvy = vpy, cvz = vpz;
                    if constexpr (!EXACT) {
                        vpx = along(vpx, stx, abs(vx - vx0)); vpy = along(vpy, sty, abs(vy - vy0));
                        vpz = along(vpz, stz, abs(vz - vz0));
                    }
#pragma unroll
                    for (int j = 0; j < TSDF_AHEAD; j++) cand |= (word[j] & 1u) << j;
                    // the voxel's centre on the ray, and whether the walk comes there
                    auto centre = [&](int j, float& tc) {
                        int p = at[0];
                        float tp = ta[0];
#pragma unroll
                        for (int k = 1; k < TSDF_AHEAD; k++) { p = k == j ? at[k] : p; tp = k == j ? ta[k] : tp; }
                        const int hx = px_of(p), hy = py_of(p), hz = vz0 + gz * nz_of(p);
                        float px, py, pz;
                        if constexpr (EXACT) {
                            px = ibx + (float)hx * vdx; py = iby + (float)hy * vdy; pz = ibz + (float)hz * vdz;
                        } else {
                            px = along(cvx, stx, abs(hx - vx0)); py = along(cvy, sty, abs(hy - vy0));
                            pz = along(cvz, stz, abs(hz - vz0));
                        }
                        tc = fminf(fmaxf((px - ox) * dx + (py - oy) * dy + (pz - oz) * dz, enterT), exitT);
                        return tp < exitT && hx >= 0 && hy >= 0 && hz >= 0 && hx < res && hy < res && hz < res;
                    };
                    auto density = [&](float tt) {
                        return trilinear(g, res, (ox + tt * dx - ibx) * ivdx, (oy + tt * dy - iby) * ivdy,
                                         (oz + tt * dz - ibz) * ivdz);
                    };
                    // Two negative voxels at a time, and below three steps of the
                    // backward search: their samples do not depend on each other, and
                    // one round of reads costs a ray more than a sample made for nothing.
                    bool found = false;
                    while (cand && !found) {
                        const int ja = __builtin_ctz(cand);
                        cand &= cand - 1;
                        const int jb = cand ? __builtin_ctz(cand) : ja;
                        cand &= cand - 1;
                        float t1, tb;
                        const bool ina = centre(ja, t1), inb = centre(jb, tb);
                        float e1 = density(t1);
                        const float eb = density(tb);
                        if (!ina) break;
                        if (!(e1 < 0.0f)) {
                            if (!inb) break;
                            t1 = tb; e1 = eb;
                        }
                        if (e1 < 0.0f) {
                            found = true;  // or the surface was expected and not found
                            float t0 = t1 - vdx / 2;
                            // at most the cube's diagonal in half-voxel steps
                            for (int back = 0; t0 > enterT && !hit && back < 4 * res + 16; back += 3) {
                                float tk[3], ek[3];
#pragma unroll
                                for (int k = 0; k < 3; k++) { tk[k] = t0; t0 -= vdx * 0.5f; }
#pragma unroll
                                for (int k = 0; k < 3; k++) ek[k] = density(tk[k]);
                                float e0 = 0.0f;
#pragma unroll
                                for (int k = 0; k < 3; k++) {
                                    const bool on = !hit && tk[k] > enterT && back + k < 4 * res + 16;
                                    if (on && ek[k] > 0.0f) {
                                        hit = true; t0 = tk[k]; e0 = ek[k];
                                    } else if (on && ek[k] > e1) {
                                        t1 = tk[k]; e1 = ek[k];
                                    }
                                }
                                if (hit) {
                                    float tx = linear_zero(t0, e0, t1, e1);
                                    while (iter > 0) {
                                        const float exv = density(tx);
                                        if (exv < 0.0f) { t1 = tx; e1 = exv; } else { t0 = tx; e0 = exv; }
                                        tx = linear_zero(t0, e0, t1, e1);
                                        iter--;
                                    }
                                    tHit = tx;
                                }
                            }
                        }
                    }
                    if (found) t = INFINITY;
                }
            }
        }
        if (hit) result = make_float4(tHit * cx, tHit * cy, tHit * cz, (tHit > a.mn && tHit < a.mx) ? 1.0f : 0.0f);
    }
    out[(size_t)xi + (size_t)yi * a.w] = result;
}

// shadingKernel (VoxelGrid_cuda.cu:844-894): normals from the neighbouring points
__global__ __launch_bounds__(256) void k_tsdf_shade(const float4* __restrict__ xyz, int w, int h, float4* __restrict__ shade,
                                                    float4* __restrict__ normals) {
    const int xi = blockIdx.x * 16 + (threadIdx.x & 15), yi = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (xi >= w || yi >= h) return;
    const size_t off = (size_t)xi + (size_t)yi * w;
    float4 px = make_float4(0.0f, 0.0f, 0.0f, 1.0f), nm = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (!(xi >= w - 3 || yi >= h - 3 || xi < 3 || yi < 3)) {
        const float4 p1x = xyz[off + 1], p0x = xyz[off - 1], p1y = xyz[off + w], p0y = xyz[off - w];
        if (p1x.w > 0.0f && p0x.w > 0.0f && p1y.w > 0.0f && p0y.w > 0.0f) {
            const float ux = p1x.x - p0x.x, uy = p1x.y - p0x.y, uz = p1x.z - p0x.z;
            const float vx = p0y.x - p1y.x, vy = p0y.y - p1y.y, vz = p0y.z - p1y.z;
            float nx = uy * vz - uz * vy, ny = -(ux * vz - uz * vx), nz = ux * vy - uy * vx;
            float len = 0.0f;
            len += nx * nx; len += ny * ny; len += nz * nz;
            len = 1.0f / sqrtf(len);
            nx *= len; ny *= len; nz *= len;
            const float c = nx * 0.0f + ny * 0.0f + nz * 1.0f;
            if (c > 0.0f) {
                px = make_float4(c, c, c, 1.0f);
                nm = make_float4(nx, ny, nz, 0.0f);
            }
        }
    }
    if (shade) shade[off] = px;
    normals[off] = nm;
}

}  // namespace rt

using namespace rt;

struct rt_tsdf {
    int device = 0;
    rt_tsdf_params p;
    hipStream_t stream = nullptr;
    float2* grid = nullptr;
    float* dist = nullptr;
    unsigned long long* skip = nullptr;  // the ray cast's table, written by each ray cast
    TsdfMap map = {nullptr, nullptr, 0, 0};
    hipEvent_t done = nullptr;  // orders work between two grids' streams
};

static TsdfArgs tsdf_args(const rt_tsdf* g, const float* T, const float* K) {
    TsdfArgs a;
    a.res = g->p.resolution; a.w = g->p.width; a.h = g->p.height;
    a.ox = g->p.origin[0]; a.oy = g->p.origin[1]; a.oz = g->p.origin[2];
    a.dx = g->p.dim[0]; a.dy = g->p.dim[1]; a.dz = g->p.dim[2];
    a.vx = a.dx / a.res; a.vy = a.dy / a.res; a.vz = a.dz / a.res;  // VoxelGrid.cpp:106
    a.mn = g->p.min_dist; a.mx = g->p.max_dist;
    memcpy(a.T, T, sizeof(a.T));
    memcpy(a.K, K, sizeof(a.K));
    return a;
}

static size_t map_tiles(const rt_tsdf* g) { return (size_t)g->map.nx * g->map.ny * (g->p.resolution / 4); }
static size_t map_words(const rt_tsdf* g) { return (size_t)g->map.nx * g->p.resolution * g->p.resolution; }  // of 16 bits
static int skip_shift(int res) { return res <= 512 ? 3 : 4; }
static unsigned skip_rows(int res) {
    const unsigned nb = (unsigned)((res + (1 << skip_shift(res)) - 1) >> skip_shift(res));
    return nb * nb;
}

// the cull of k_tsdf_update; a value that is not finite culls nothing
static TsdfCull tsdf_cull(const TsdfArgs& a) {
    TsdfCull c;
    const double w = a.w, h = a.h, res = a.res;
    const double cx0 = a.K[2] - 1.0 / w, cx1 = a.K[2] - (w - 2) / w, cy0 = a.K[5] - 1.0 / h, cy1 = a.K[5] - (h - 2) / h;
    const double hx = 7.5 * 2 * a.vx, hy = 1.5 * 2 * a.vy;  // half a slice: 16 and 4 voxel centres
    // the largest sum of magnitudes behind a coordinate, tiles past the grid included
    const double px = fabs(a.ox) + a.dx * (1 + 32.0 / res), py = fabs(a.oy) + a.dy * (1 + 32.0 / res),
                 pz = fabs(a.oz) + a.dz * (1 + 32.0 / res);
    double big = 0;
    for (int i = 0; i < 3; i++)
        big = fmax(big, fabs(a.T[4 * i]) * px + fabs(a.T[4 * i + 1]) * py + fabs(a.T[4 * i + 2]) * pz + fabs(a.T[4 * i + 3]));
    auto reach = [&](double k, const float* row, double cz, double k2) {
        return fabs(k * row[0] + cz * a.T[8]) * hx + fabs(k * row[1] + cz * a.T[9]) * hy +
               1e-5 * big * (fabs(k) + fabs(k2) + 2);
    };
    c.cx0 = (float)cx0; c.cx1 = (float)cx1; c.cy0 = (float)cy0; c.cy1 = (float)cy1;
    c.ex0 = (float)reach(a.K[0], a.T, cx0, a.K[2]); c.ex1 = (float)reach(a.K[0], a.T, cx1, a.K[2]);
    c.ey0 = (float)reach(a.K[4], a.T + 4, cy0, a.K[5]); c.ey1 = (float)reach(a.K[4], a.T + 4, cy1, a.K[5]);
    c.ez = (float)(fabs(a.T[8]) * hx + fabs(a.T[9]) * hy + 2e-5 * big);
    // (int)u < w - 2 for a float u is u < the smallest float that is not below w - 2
    auto bound = [](int n) { const float f = (float)n; return (double)f < (double)n ? nextafterf(f, INFINITY) : f; };
    c.umax = bound(a.w - 2); c.vmax = bound(a.h - 2);
    const float slope = a.dx * 0.030f, top = 1152921504606846976.0f;  // 2^60
    const bool fits = slope >= 1.0f / top && slope <= top;
    c.islope = fits ? 1.0f / slope : 0.0f;
    c.nlo = fits ? 1.0f / top : INFINITY; c.nhi = fits ? top : 0.0f;
    return c;
}

// Whether every voxel centre first + i * edge, i < res, is a float, products
// and sums along the way included: with all of them multiples of 2^e and below
// 2^(e + 24) nothing rounds.
static bool centres_exact(float first, float edge, int res) {
    if (!std::isfinite(first) || !std::isfinite(edge)) return false;
    auto low = [](double v) {  // exponent of the lowest set bit
        if (v == 0) return 1024;
        int e;
        double m = frexp(fabs(v), &e);
        for (; m != floor(m); e--) m *= 2;
        return e;
    };
    const int e1 = low(edge), e = e1 < low(first) ? e1 : low(first);
    const double last = (double)first + (double)edge * (res - 1);
    return (double)edge * res < ldexp(1.0, e1 + 24) && fmax(fabs((double)first), fabs(last)) < ldexp(1.0, e + 24);
}

extern "C" void rt_tsdf_default_params(rt_tsdf_params* p) {
    if (!p) return;
    p->resolution = 256;
    p->origin[0] = 0.0f; p->origin[1] = 0.01f; p->origin[2] = -1600.01f;
    p->dim[0] = p->dim[1] = p->dim[2] = 1500.0f;
    p->width = 320; p->height = 240;
    p->min_dist = 300.0f; p->max_dist = 7000.0f;
}

extern "C" int rt_tsdf_create(int device, const rt_tsdf_params* p, rt_tsdf** out) {
    if (!p || !out || p->resolution < 8 || p->resolution % 8 || p->resolution > 1024 || p->width < 8 || p->height < 8 ||
        !(p->dim[0] > 0 && p->dim[1] > 0 && p->dim[2] > 0))
        return set_error(RT_ERR_ARG, "rt_tsdf_create: bad argument");
    if (hipSetDevice(device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    rt_tsdf* g = new rt_tsdf();
    g->device = device; g->p = *p;
    g->map.nx = (p->resolution + 15) / 16; g->map.ny = p->resolution / 4;
    const size_t nv = (size_t)p->resolution * p->resolution * p->resolution;
    if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess) { delete g; return set_error(RT_ERR_HIP, "stream"); }
    if (hipEventCreateWithFlags(&g->done, hipEventDisableTiming) != hipSuccess) {
        hipStreamDestroy(g->stream);
        delete g;
        return set_error(RT_ERR_HIP, "event");
    }
    if (hipMalloc((void**)&g->grid, nv * sizeof(float2)) != hipSuccess ||
        hipMalloc((void**)&g->dist, (size_t)p->width * p->height * sizeof(float)) != hipSuccess ||
        hipMalloc((void**)&g->map.neg, map_words(g) * sizeof(uint16_t)) != hipSuccess ||
        hipMalloc((void**)&g->map.occ, map_tiles(g)) != hipSuccess ||
        hipMalloc((void**)&g->skip, skip_rows(p->resolution) * sizeof(unsigned long long)) != hipSuccess) {
        hipFree(g->grid); hipFree(g->dist); hipFree(g->map.neg); hipFree(g->map.occ);
        hipEventDestroy(g->done);
        hipStreamDestroy(g->stream);
        delete g;
        return set_error(RT_ERR_NOMEM, "rt_tsdf_create: grid");
    }
    if (hipMemsetAsync(g->dist, 0, (size_t)p->width * p->height * sizeof(float), g->stream) != hipSuccess) {
        rt_tsdf_destroy(g);
        return set_error(RT_ERR_HIP, "rt_tsdf_create: clear");
    }
    int rc = rt_tsdf_reset(g);
    if (rc) { rt_tsdf_destroy(g); return rc; }
    *out = g;
    return RT_OK;
}

extern "C" void rt_tsdf_destroy(rt_tsdf* g) {
    if (!g) return;
    hipSetDevice(g->device);
    hipStreamSynchronize(g->stream);
    hipFree(g->grid);
    hipFree(g->dist);
    hipFree(g->map.neg);
    hipFree(g->map.occ);
    hipFree(g->skip);
    hipEventDestroy(g->done);
    hipStreamDestroy(g->stream);
    delete g;
}

extern "C" int rt_tsdf_reset(rt_tsdf* g) {
    if (!g) return set_error(RT_ERR_ARG, "rt_tsdf_reset: null");
    if (hipSetDevice(g->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    const size_t n = (size_t)g->p.resolution * g->p.resolution * g->p.resolution;
    k_tsdf_reset<<<(unsigned)((n + 255) / 256), 256, 0, g->stream>>>(g->grid, g->map, n, map_words(g), map_tiles(g));
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(g->stream) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_tsdf_reset");
    return RT_OK;
}

extern "C" int rt_tsdf_set_depth_rgbd(rt_tsdf* g, const float* rgbd) {
    if (!g || !rgbd) return set_error(RT_ERR_ARG, "rt_tsdf_set_depth_rgbd: null");
    if (hipSetDevice(g->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    dim3 grid((g->p.width + 15) / 16, (g->p.height + 15) / 16);
    k_tsdf_dist_rgbd<<<grid, 256, 0, g->stream>>>((const float4*)rgbd, g->p.width, g->p.height, g->p.min_dist,
                                                   g->p.max_dist, g->dist);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_tsdf_set_depth_rgbd");
    return RT_OK;
}

extern "C" int rt_tsdf_set_depth_u16(rt_tsdf* g, const uint16_t* depth) {
    if (!g || !depth) return set_error(RT_ERR_ARG, "rt_tsdf_set_depth_u16: null");
    if (hipSetDevice(g->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    const size_t n = (size_t)g->p.width * g->p.height;
    k_tsdf_dist_u16<<<(unsigned)((n + 255) / 256), 256, 0, g->stream>>>(depth, n, g->dist);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_tsdf_set_depth_u16");
    return RT_OK;
}

extern "C" int rt_tsdf_update(rt_tsdf* g, const float* T, const float* K) {
    if (!g || !T || !K) return set_error(RT_ERR_ARG, "rt_tsdf_update: null");
    if (hipSetDevice(g->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    float iT[16];
    invert_rt4f(T, iT);  // VoxelGrid::setCameraParams (VoxelGrid.cpp:275-282): the kernel maps world -> camera
    const TsdfArgs a = tsdf_args(g, iT, K);
    auto update = [&](auto slices) {
        constexpr int Z = decltype(slices)::value;
        const dim3 grid(g->map.nx, (g->map.ny + 3) / 4, (g->p.resolution + Z - 1) / Z);
        k_tsdf_update<Z><<<grid, 256, 0, g->stream>>>(g->grid, g->map, g->dist, a, tsdf_cull(a));
    };
    // Slices a wave: few where the grid has few waves, and one follows the other's
    // latency; many where they are plenty and share the wave's set-up. us of an
    // update at 4 and 16 slices: 64^3 5.1 10.3, 128^3 8.7 11.8, 192^3 14.6 17.8,
    // 256^3 29.0 29.4, 384^3 70.8 63.6, 512^3 214 190 (one thread per voxel 4.2,
    // 7.6, 17.4, 38, 117 and 298); of frames in flight, each with its ray cast,
    // 192^3 32.1 33.6, 256^3 49.3 47.6.
    if (g->p.resolution < 256) update(std::integral_constant<int, 4>());
    else update(std::integral_constant<int, 16>());
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_tsdf_update");
    return RT_OK;
}

extern "C" int rt_tsdf_raycast(rt_tsdf* g, const float* T, const float* K, int refine, float* xyz, float* normals,
                               float* shade) {
    if (!g || !T || !K || !xyz || !normals) return set_error(RT_ERR_ARG, "rt_tsdf_raycast: null");
    if (hipSetDevice(g->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    const TsdfArgs a = tsdf_args(g, T, K);  // the ray cast walks from the camera: camera -> world
    dim3 grid((g->p.width + 15) / 16, (g->p.height + 15) / 16);
    const bool exact = centres_exact(a.ox - a.dx + a.vx, 2.0f * a.vx, a.res) &&
                       centres_exact(a.oy - a.dy + a.vy, 2.0f * a.vy, a.res) &&
                       centres_exact(a.oz - a.dz + a.vz, 2.0f * a.vz, a.res);
    const unsigned rows = skip_rows(a.res), lds = rows * sizeof(unsigned long long);
    auto cast = [&](auto lb, auto ex) {
        constexpr int LB = decltype(lb)::value;
        k_tsdf_skip<LB><<<(rows + 3) / 4, 256, 0, g->stream>>>(g->map, a.res, g->skip);
        k_tsdf_raycast<LB, decltype(ex)::value>
            <<<grid, 256, lds, g->stream>>>(g->grid, g->map, g->skip, a, refine ? 1 : 0, (float4*)xyz);
    };
    const std::integral_constant<int, 3> small{};
    const std::integral_constant<int, 4> large{};
    if (skip_shift(a.res) == 3)
        exact ? cast(small, std::true_type()) : cast(small, std::false_type());
    else
        exact ? cast(large, std::true_type()) : cast(large, std::false_type());
    k_tsdf_shade<<<grid, 256, 0, g->stream>>>((const float4*)xyz, g->p.width, g->p.height, (float4*)shade,
                                               (float4*)normals);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_tsdf_raycast");
    return RT_OK;
}

extern "C" int rt_tsdf_resample(rt_tsdf* dst, const rt_tsdf* src, const float* T) {
    if (!dst || !src || !T || dst == src) return set_error(RT_ERR_ARG, "rt_tsdf_resample: null or same grid");
    const rt_tsdf_params &a = dst->p, &b = src->p;
    if (a.resolution != b.resolution || memcmp(a.origin, b.origin, sizeof(a.origin)) || memcmp(a.dim, b.dim, sizeof(a.dim)) ||
        dst->device != src->device)
        return set_error(RT_ERR_ARG, "rt_tsdf_resample: grids differ in resolution, origin, extent or device");
    if (hipSetDevice(dst->device) != hipSuccess) return set_error(RT_ERR_HIP, "hipSetDevice");
    float K[9] = {0};
    const TsdfArgs args = tsdf_args(dst, T, K);  // VoxelGrid::setCameraParams keeps T itself as iT
    // src's queued work is ordered before the resample
    if (hipEventRecord(src->done, src->stream) != hipSuccess || hipStreamWaitEvent(dst->stream, src->done, 0) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_tsdf_resample");
    const int xcds = resample_xcds(a.resolution);
    const dim3 grid((a.resolution + 63) / 64 * ((dst->map.ny + xcds - 1) / xcds * xcds), a.resolution / 4);
    k_tsdf_resample<<<grid, 256, 0, dst->stream>>>(dst->grid, dst->map, src->grid, args);
    if (hipGetLastError() != hipSuccess) return set_error(RT_ERR_HIP, "rt_tsdf_resample");
    // src's later work is ordered after the resample has read it
    if (hipEventRecord(dst->done, dst->stream) != hipSuccess || hipStreamWaitEvent(src->stream, dst->done, 0) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_tsdf_resample");
    return RT_OK;
}

extern "C" int rt_tsdf_read(rt_tsdf* g, float* host, size_t bytes) {
    if (!g || !host) return set_error(RT_ERR_ARG, "rt_tsdf_read: null");
    const size_t n = (size_t)g->p.resolution * g->p.resolution * g->p.resolution * sizeof(float2);
    if (bytes < n) return set_error(RT_ERR_ARG, "rt_tsdf_read: buffer too small");
    if (hipSetDevice(g->device) != hipSuccess || hipMemcpyAsync(host, g->grid, n, hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
        hipStreamSynchronize(g->stream) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_tsdf_read");
    return RT_OK;
}

extern "C" const float* rt_tsdf_data(rt_tsdf* g) { return g ? (const float*)g->grid : nullptr; }

extern "C" void* rt_tsdf_stream(rt_tsdf* g) { return g ? (void*)g->stream : nullptr; }

extern "C" int rt_tsdf_synchronize(rt_tsdf* g) {
    if (!g) return set_error(RT_ERR_ARG, "rt_tsdf_synchronize: null");
    if (hipSetDevice(g->device) != hipSuccess || hipStreamSynchronize(g->stream) != hipSuccess)
        return set_error(RT_ERR_HIP, "rt_tsdf_synchronize");
    return RT_OK;
}
