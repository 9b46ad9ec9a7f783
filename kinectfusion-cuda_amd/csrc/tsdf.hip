// TSDF volume: allocation, initialisation, projective fusion, and the raw
// interchange format (project/src/tsdf.cu, voxel_grid.h, voxel_grid.cpp).
//
// HBM layout: two planes (f, w) of n^3 voxels in 8^3 bricks (kf_device.hpp).
//   KF_VOXEL_F32        : f float, w float          (8 B / voxel)
//   KF_VOXEL_SNORM16_U8 : f snorm16, w uint8 count  (3 B / voxel)
// A cull pass lists the bricks whose bounding sphere meets the view frustum;
// then one wave fuses one listed brick at a time, one brick column (8 voxels
// along z, contiguous in the plane) per lane, so a wave reads and writes a
// brick's planes as contiguous 16-byte-per-lane accesses, and the listed
// bricks are spread evenly over the waves.  Bricks whose bounding sphere lies outside the view frustum
// are skipped before any voxel is visited; the test is conservative, so the
// result is identical to visiting every voxel.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <cmath>
#include <thread>
#include <vector>

#include "kf_device.hpp"
#include "kf_kernels.hpp"

namespace kf {

namespace {

// List entries name a brick by its coordinates, bi | bj << 10 | bk << 20
// (volumes are at most 1024^3 voxels: 128 bricks per axis), so the sweep
// forms its linear index with two multiply-adds instead of two divisions; bit 31
// marks a brick in free space (cube_test).
constexpr unsigned kFreeBrick = 1u << 31;
__host__ __device__ __forceinline__ unsigned pack_brick(int bi, int bj, int bk)
{
    return (unsigned)bi | (unsigned)bj << 10 | (unsigned)bk << 20;
}

// Whether a frame may update voxels of cube (bi, bj, bk) of SIDE voxels a side: 0 when
// it certainly updates none, else 1, and (FREE) kFreeBrick when it certainly updates
// all of them with f = 1.
template <int SIDE, bool FREE>
__device__ __forceinline__ unsigned cube_test(const FuseArgs& a, const float* ip, int bi, int bj, int bk)
{
    // Bounding sphere of the cube's voxel centres (span SIDE - 1 times res per axis).
    constexpr float kHalf = (SIDE - 1) * 0.5f;
    float cx = a.half + ((float)(bi * SIDE) + kHalf) * a.res;
    float cy = a.half + ((float)(bj * SIDE) + kHalf) * a.res;
    float cz = a.half + ((float)(bk * SIDE) + kHalf) * a.res;
    float r = kHalf * 1.7320508f * a.res * 1.01f + 1e-4f;
    float ex = (ip[0] * cx + ip[4] * cy) + (ip[8] * cz + ip[12]);
    float ey = (ip[1] * cx + ip[5] * cy) + (ip[9] * cz + ip[13]);
    float ez = (ip[2] * cx + ip[6] * cy) + (ip[10] * cz + ip[14]);
    if (ez + r < kMinDistance || ez - r >= kMaxDistance) return 0u;
    float fx = a.K[0], fy = a.K[4], px = a.K[6], py = a.K[7];
    float W = (float)a.w, H = (float)a.h;
    // pixel.x >= 0  <=>  fx*x + px*z >= 0 (z > 0);  pixel.x < W  <=>  (W-px)*z - fx*x > 0
    if ((fx * ex + px * ez) < -r * a.plane_norm[0]) return 0u;
    if (((W - px) * ez - fx * ex) < -r * a.plane_norm[1]) return 0u;
    if ((fy * ey + py * ez) < -r * a.plane_norm[2]) return 0u;
    if (((H - py) * ez - fy * ey) < -r * a.plane_norm[3]) return 0u;
    // Occlusion: a voxel is updated only if d - z >= -mue for the valid depth d
    // of its pixel.  With the sphere beyond the near plane its pixels lie in the
    // box below (x/z and y/z at the corners, one pixel of margin); if even the
    // largest valid depth there is more than mue (+1 mm for rounding) in front
    // of the sphere's nearest point, no voxel of the brick is updated.  The
    // quotients come from the hardware reciprocal: within a few 1e-7 of x/z,
    // which moves the box by under 1e-2 pixel (|x/z| is at most a few tens with
    // z > kMinDistance), far inside its one pixel of margin.
    const float zlo = ez - r;
    if (!a.drange || !(zlo > kMinDistance)) return 1u;
    const float zhi = ez + r, xa = ex - r, xb = ex + r, ya = ey - r, yb = ey + r;
    const float r0 = __builtin_amdgcn_rcpf(zlo), r1 = __builtin_amdgcn_rcpf(zhi);
    const float u0 = fx * fminf(xa * r0, xa * r1) + px - 1.0f, u1 = fx * fmaxf(xb * r0, xb * r1) + px + 1.0f;
    const float v0 = fy * fminf(ya * r0, ya * r1) + py - 1.0f, v1 = fy * fmaxf(yb * r0, yb * r1) + py + 1.0f;
    const int i0 = (int)fmaxf(u0, 0.0f), i1 = (int)fminf(u1, W - 1.0f);
    const int j0 = (int)fmaxf(v0, 0.0f), j1 = (int)fminf(v1, H - 1.0f);
    if (i1 < i0 || j1 < j0) return a.mue + 1e-3f >= zlo ? 1u : 0u;  // no pixel: no valid depth
    const float2* m;
    int shift, tx;
    if (i1 - i0 < 48 && j1 - j0 < 48) {
        m = a.drange;
        shift = 4;
        tx = a.tx16;
    } else if (i1 - i0 < 192 && j1 - j0 < 192) {
        m = a.drange + a.tx16 * a.ty16;
        shift = 6;
        tx = a.tx64;
    } else {
        return 1u;
    }
    // a box under 48 (192) pixels spans at most 4 x 4 tiles of 16 (64): all 16
    // reads are issued together, those past the box's last tile row or column
    // repeating it (the range is the same)
    const int ti0 = i0 >> shift, tj0 = j0 >> shift, ti1 = i1 >> shift, tj1 = j1 >> shift;
    float2 t[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const float2* e = m + (min(tj0 + (q >> 2), tj1) * tx + min(ti0 + (q & 3), ti1));
        if (FREE) t[q] = *e;
        else t[q].x = e->x;
    }
    float dm = 0.0f;
#pragma unroll
    for (int q = 0; q < 16; ++q) dm = fmaxf(dm, t[q].x);
    if (!(dm + a.mue + 1e-3f >= zlo)) return 0u;
    if (!FREE) return 1u;
    float dn = t[0].y;
#pragma unroll
    for (int q = 1; q < 16; ++q) dn = fminf(dn, t[q].y);
    // Free space: every voxel projects into the image (the box, with its margin, lies in
    // it) between the distance limits, on a valid depth more than mue (+1 mm) behind the
    // sphere's farthest point.
    const bool inside = u0 >= 0.0f && v0 >= 0.0f && u1 <= W - 1.0f && v1 <= H - 1.0f;
    return inside && zlo > kMinDistance + 1e-3f && zhi < kMaxDistance - 1e-3f && dn - zhi >= a.mue + 1e-3f ? kFreeBrick
                                                                                                          : 1u;
}

// Tile depth ranges of a depth map (FuseArgs::drange), the max only (the min, which
// only a batch's cull reads, is 0): one workgroup per 64x64 pixel region; lane group
// t/16 takes one 16x16 tile, each lane a 4x4 block.
// Invalid depths (isDepthValid false) count as 0.
__global__ __launch_bounds__(256) void depth_range_kernel(const float* __restrict__ depth, int w, int h, float2* drange,
                                                          int tx16, int ty16, int tx64)
{
    __shared__ float part[16];
    const int q = threadIdx.x >> 4, sub = threadIdx.x & 15;
    const int tx = blockIdx.x * 4 + (q & 3), ty = blockIdx.y * 4 + (q >> 2);
    const int x0 = tx * 16 + (sub & 3) * 4, y0 = ty * 16 + (sub >> 2) * 4;
    float m = 0.0f;
    for (int y = y0; y < y0 + 4; ++y)
        for (int x = x0; x < x0 + 4; ++x)
            if (x < w && y < h) {
                const float d = depth[(int64_t)y * w + x];
                if (is_depth_valid(d)) m = fmaxf(m, d);
            }
    // max over the 16 lanes of the tile (one 16-lane row)
    m = row_range(m, 0.0f).x;
    if (sub == 0) {
        part[q] = m;
        if (tx < tx16 && ty < ty16) drange[ty * tx16 + tx] = make_float2(m, 0.0f);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = 0.0f;
        for (int k = 0; k < 16; ++k) r = fmaxf(r, part[k]);
        drange[tx16 * ty16 + blockIdx.y * tx64 + blockIdx.x] = make_float2(r, 0.0f);
    }
}

// True when x may lie within a few ulp of an integer (0 and the image size
// included): x*rcp(z) is within 2^-22 |x/z| of the rounded quotient x/z
// (v_rcp_f32 is within 1 ulp), so outside a band of half-width band =
// 2^-21 max(w, h) both have the same sign, the same integer part and the same
// side of every integer bound wherever |x| <= 2 max(w, h); beyond that both
// lie outside the image, and the integer part is not used.
__device__ __forceinline__ bool near_integer(float x, float band)
{
    return fabsf(x - rintf(x)) <= band;
}

// A brick column's planes in registers: the 8 voxels (i, j, 0..7) are
// contiguous, so f and w move as one or two 16-byte accesses each (FP32: two
// float4 per plane; snorm16: 8 codes in a uint4, 8 counts in a uint2).
template <int FMT>
struct ColumnPlanes;

template <>
struct ColumnPlanes<KF_VOXEL_F32> {
    float f[8], w[8];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = w[k] = 0.0f;
    }
    __device__ __forceinline__ void load(const FuseArgs& a, int64_t base)
    {
        const float4* F = reinterpret_cast<const float4*>(static_cast<const float*>(a.f) + base);
        const float4* W = reinterpret_cast<const float4*>(static_cast<const float*>(a.wt) + base);
        const float4 f0 = F[0], f1 = F[1], w0 = W[0], w1 = W[1];
        f[0] = f0.x, f[1] = f0.y, f[2] = f0.z, f[3] = f0.w, f[4] = f1.x, f[5] = f1.y, f[6] = f1.z, f[7] = f1.w;
        w[0] = w0.x, w[1] = w0.y, w[2] = w0.z, w[3] = w0.w, w[4] = w1.x, w[5] = w1.y, w[6] = w1.z, w[7] = w1.w;
    }
    __device__ __forceinline__ void store(const FuseArgs& a, int64_t base) const
    {
        float4* F = reinterpret_cast<float4*>(static_cast<float*>(a.f) + base);
        float4* W = reinterpret_cast<float4*>(static_cast<float*>(a.wt) + base);
        F[0] = make_float4(f[0], f[1], f[2], f[3]);
        F[1] = make_float4(f[4], f[5], f[6], f[7]);
        W[0] = make_float4(w[0], w[1], w[2], w[3]);
        W[1] = make_float4(w[4], w[5], w[6], w[7]);
    }
};

template <>
struct ColumnPlanes<KF_VOXEL_SNORM16_U8> {
    uint4 f;  // codes 2m (low half) and 2m+1 (high half) in word m
    uint2 w;  // count k in byte k % 4 of word k / 4
    __device__ __forceinline__ void clear()
    {
        f = make_uint4(0u, 0u, 0u, 0u);
        w = make_uint2(0u, 0u);
    }
    __device__ __forceinline__ void load(const FuseArgs& a, int64_t base)
    {
        f = *reinterpret_cast<const uint4*>(static_cast<const int16_t*>(a.f) + base);
        w = *reinterpret_cast<const uint2*>(static_cast<const uint8_t*>(a.wt) + base);
    }
    __device__ __forceinline__ void store(const FuseArgs& a, int64_t base) const
    {
        *reinterpret_cast<uint4*>(static_cast<int16_t*>(a.f) + base) = f;
        *reinterpret_cast<uint2*>(static_cast<uint8_t*>(a.wt) + base) = w;
    }
    // Every code 32767 (F = 1): an update by f = 1 writes (1 W + 1) / (W + 1) = 1 again.
    __device__ __forceinline__ bool settled() const
    {
        return (f.x & f.y & f.z & f.w) == 0x7fff7fffu && (f.x | f.y | f.z | f.w) == 0x7fff7fffu;
    }
    // Every count + 1, at most 128, four bytes at a time.
    __device__ __forceinline__ static uint32_t count_word(uint32_t c)
    {
        const uint32_t full = c & 0x80808080u;  // counts of 128 (or more: 128 from here on)
        return full | (((c & 0x7f7f7f7fu) + 0x01010101u) & ~(full | (full - (full >> 7))));
    }
    __device__ __forceinline__ void count_all()
    {
        w.x = count_word(w.x);
        w.y = count_word(w.y);
    }
    __device__ __forceinline__ static uint32_t word(const uint4& v, int m)
    {
        return m == 0 ? v.x : (m == 1 ? v.y : (m == 2 ? v.z : v.w));
    }
    __device__ __forceinline__ int16_t code(int k) const
    {
        return (int16_t)(uint16_t)(word(f, k >> 1) >> (16 * (k & 1)));
    }
    __device__ __forceinline__ int count(int k) const
    {
        return (int)(((k < 4 ? w.x : w.y) >> (8 * (k & 3))) & 0xffu);
    }
    __device__ __forceinline__ void set(int k, int16_t q, int c)
    {
        const uint32_t sh = 16u * (uint32_t)(k & 1), m = 0xffffu << sh, v = (uint32_t)(uint16_t)q << sh;
        uint32_t& fw = (k >> 1) == 0 ? f.x : ((k >> 1) == 1 ? f.y : ((k >> 1) == 2 ? f.z : f.w));
        fw = (fw & ~m) | v;
        const uint32_t bs = 8u * (uint32_t)(k & 3), bm = 0xffu << bs;
        uint32_t& ww = k < 4 ? w.x : w.y;
        ww = (ww & ~bm) | ((uint32_t)c << bs);
    }
};

// The precision form's update of voxel kl by f: unit weight per observation, count
// capped at 128 (an upload or a reset may have stored any count up to 255).
__device__ __forceinline__ void update_voxel(ColumnPlanes<KF_VOXEL_SNORM16_U8>& v, int kl, float f,
                                             const float* inv_count, float& fmin, float& fk0)
{
    const int wc = v.count(kl);
    const float Wv = (float)wc;
    float Fv = snorm_decode(v.code(kl));
    Fv = div_by_exact_reciprocal(Fv * Wv + f, Wv + 1.0f, inv_count[wc]);
    const int16_t qf = snorm_encode(Fv);
    v.set(kl, qf, wc < 128 ? wc + 1 : 128);
    const float written = snorm_decode(qf);
    fmin = fminf(fmin, written);
    if (kl == 0) fk0 = written;
}

// tsdf.cu:20-75 for the 8 voxels (one per z-slice kl) of one lane's column of
// a brick (lane = (j, i) of the brick); returns the number of updated voxels.
// Projection (tsdf.cu:34-45): pe = inv_pose * (x, y, z, 1), pixel = K pe / pe.z;
// only the pixel's integer part and the range test use the quotient, so it is
// formed from the hardware reciprocal and recomputed by the correctly rounded
// division only near an integer (the decisions are the exact quotient's).
// Update (tsdf.cu:47-69): f = min(1, diff / mue) from the exact reciprocal of
// mue; the precision form divides by the observation count + 1 with the exact
// reciprocal of 1..256 from inv_count (LDS); every value written is the one the
// plain quotients give.  fmin takes the smallest value written, fk0 the value
// written to voxel 0 (the brick's k = 0 plane).  The column's planes are read
// when any of its voxels passes the depth test (after the depth gathers) and
// written back whole when any was updated (the others keep the bits they were
// read with; one wave owns the brick).
template <int FMT>
__device__ __forceinline__ int fuse_column(const FuseArgs& a, v3 col, const float4* zt, int64_t base, float& fmin,
                                           float& fk0, const float* inv_count)
{
    float dep[8], pz[8];
    unsigned pix[8];
    bool hit[8];
    const float fw = (float)a.w, fh = (float)a.h;
#pragma unroll
    for (int kl = 0; kl < 8; ++kl) {
        // pe = (m0*x + m1*y) + (m2*z + m3*1): the first pair is shared by the
        // column, the second by the slice (zt, formed once per fuse)
        v3 pe = mk3(col.x + zt[kl].x, col.y + zt[kl].y, col.z + zt[kl].z);
        bool ok = pe.z >= kMinDistance && pe.z < kMaxDistance;
        unsigned q = 0u;
        if (ok) {
            float px, py;
            if (a.cull) {
                // K pe for a pinhole K: the zero entries add exact zeros, so the product is
                // (fx x + cx z, fy y + cy z, z)
                const float vx = a.K[0] * pe.x + a.K[6] * pe.z, vy = a.K[4] * pe.y + a.K[7] * pe.z;
                const float r = __builtin_amdgcn_rcpf(pe.z);
                px = vx * r;
                py = vy * r;
                if (near_integer(px, a.band) || near_integer(py, a.band)) {
                    px = vx / pe.z;
                    py = vy / pe.z;
                }
            } else {
                const v3 pv = m3v(a.K, pe);
                px = pv.x / pv.z;
                py = pv.y / pv.z;
            }
            ok = px >= 0.0f && px < fw && py >= 0.0f && py < fh;
            // 0 <= px < w, 0 <= py < h: a 24-bit product (images are below 2^24 pixels a side)
            if (ok) q = __umul24((unsigned)py, (unsigned)a.w) + (unsigned)px;
        }
        hit[kl] = ok;
        pix[kl] = q;
        pz[kl] = pe.z;
    }
#pragma unroll
    for (int kl = 0; kl < 8; ++kl) {
        dep[kl] = 0.0f;
        if (hit[kl]) dep[kl] = a.depth[pix[kl]];
    }
    // the depth test first: the planes of a column none of whose voxels is
    // updated (behind the surface or on invalid depth) are not read
    bool upd[8], any = false;
#pragma unroll
    for (int kl = 0; kl < 8; ++kl) {
        upd[kl] = hit[kl] && is_depth_valid(dep[kl]) && dep[kl] - pz[kl] >= -a.mue;
        any = any || upd[kl];
    }
    ColumnPlanes<FMT> v;
    v.clear();
    if (any) v.load(a, base);
    int cnt = 0;
#pragma unroll
    for (int kl = 0; kl < 8; ++kl) {
        const float d = dep[kl];
        const float diff = d - pz[kl];
        if (!upd[kl]) continue;
        // f = min(1, diff / mue): diff >= mue makes the rounded quotient >= 1, so the
        // division (most updated voxels lie in front of the surface) is skipped there
        float f = 1.0f;
        if (diff < a.mue) {
            f = div_by_exact_reciprocal(diff, a.mue, a.inv_mue);
            f = (f < 1.0f) ? f : 1.0f;
        }
        if constexpr (FMT == KF_VOXEL_F32) {
            const float wt = 1.0f / d;
            float Fv = v.f[kl], Wv = v.w[kl];
            Fv = (Fv * Wv + f * wt) / (Wv + wt);
            Wv = Wv + wt;
            v.f[kl] = Fv;
            v.w[kl] = Wv;
            fmin = fminf(fmin, Fv);
            if (kl == 0) fk0 = Fv;
        } else {
            update_voxel(v, kl, f, inv_count, fmin, fk0);
        }
        ++cnt;
    }
    if (cnt) v.store(a, base);
    return cnt;
}

// Exact reciprocals for the count update: entry c is 1 / (c + 1), for every count
// a uint8 holds.
constexpr int kInvCount = 256;
__device__ __forceinline__ void fill_inv_count(float* t)
{
    for (int c = threadIdx.x; c < kInvCount; c += blockDim.x) t[c] = 1.0f / (float)(c + 1);
    __syncthreads();
}

__device__ __forceinline__ void load_inv_pose(const FuseArgs& a, float* ip)
{
    if (threadIdx.x < 16) ip[threadIdx.x] = a.dyn ? a.dyn->inv_pose[threadIdx.x] : a.inv_pose[threadIdx.x];
    __syncthreads();
}

// The z terms of slice k's projection, (m2 z + m3 * 1) per row of the inverse
// pose (the second pair of the reference's (m0 x + m1 y) + (m2 z + m3 * 1)),
// formed by the cull for every slice once per fuse and read by the sweep.
__device__ __forceinline__ void z_terms(const float* ip, const float* zk, float4* zt, int k)
{
    const float z = zk[k];
    zt[k] = make_float4(ip[8] * z + ip[12] * 1.0f, ip[9] * z + ip[13] * 1.0f, ip[10] * z + ip[14] * 1.0f, 0.0f);
}

// Pass 1: one lane per brick; bricks whose bounding sphere meets the view
// frustum are appended to `list`, one atomic per workgroup.  The list length
// lives in count[parity]; this pass also clears count[1 - parity], which the
// previous launch used, for the next launch (also when its own frame is not
// fused: the next launch appends to that count from zero).
constexpr int kCullThreads = 1024;

__global__ __launch_bounds__(kCullThreads) void fuse_cull_kernel(FuseArgs a, int64_t nbricks, int* list,
                                                                 unsigned int* count, int parity)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) count[1 - parity] = 0u;
    if (a.dyn && a.dyn->frame_skip_fuse) return;
    __shared__ float ip[16];
    __shared__ unsigned int wave_base[kCullThreads / 64 + 1];
    load_inv_pose(a, ip);
    for (int k = blockIdx.x * kCullThreads + threadIdx.x; k < a.n; k += gridDim.x * kCullThreads) z_terms(ip, a.zk, a.zt, k);
    const int64_t brick = (int64_t)blockIdx.x * kCullThreads + threadIdx.x;
    bool vis = false;
    unsigned packed = 0u;
    if (brick < nbricks) {
        // at most 128^3 bricks: 32-bit index arithmetic
        const unsigned ub = (unsigned)brick, nb = (unsigned)a.nb;
        const int bi = (int)(ub % nb), bj = (int)((ub / nb) % nb), bk = (int)(ub / (nb * nb));
        vis = !a.cull || cube_test<8, false>(a, ip, bi, bj, bk);
        packed = pack_brick(bi, bj, bk);
    }
    const uint64_t m = __ballot(vis);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wave_base[wave] = (unsigned int)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned int total = 0;
        for (int w = 0; w < kCullThreads / 64; ++w) {
            unsigned int c = wave_base[w];
            wave_base[w] = total;
            total += c;
        }
        wave_base[kCullThreads / 64] = total ? atomicAdd(&count[parity], total) : 0u;
    }
    __syncthreads();
    if (vis)
        list[wave_base[kCullThreads / 64] + wave_base[wave] + (unsigned int)__popcll(m & ((1ull << lane) - 1ull))] =
            (int)packed;
}

constexpr int kFuseWaves = 4;

// The free bits a fused brick may clear (kf_device.hpp): lane l < 8 loads those
// of brick (bi - (l & 1), bj - (l >> 1 & 1), bk - (l >> 2)), the brick itself
// and the 7 below it whose halos reach into it (bit 0: large steps, bit 1: small;
// 0 for a brick outside the volume), at the brick's start, so that the load
// shares the column loads' round trip.
__device__ __forceinline__ int load_free(const FuseArgs& a, int bi, int bj, int bk, int lane)
{
    int b = 0;
    if (lane < 8) {
        const int ni = bi - (lane & 1), nj = bj - ((lane >> 1) & 1), nk = bk - (lane >> 2);
        if (ni >= 0 && nj >= 0 && nk >= 0) {
            const unsigned long long* r = a.free_bits + free_word(a.nb, ni, nj, nk, 0);
            const unsigned long long large = r[0], small = r[a.nb > 64 ? 2 : 1];
            b = (int)((large >> (ni & 63)) & 1ull) | (int)((small >> (ni & 63)) & 1ull) << 1;
        }
    }
    return b;
}

// Clears the free bits the brick's written values end: every value counts for
// its brick, values on the local i = 0 plane (lanes with i == 0) for the -x
// neighbour too, on j = 0 (lanes with j == 0) for the -y neighbour, on k = 0
// (each lane's first voxel) for the -z neighbour, and the values on two or three
// of these planes for the diagonal neighbours.  A brick in front of the surface
// has no value below kSkipBound, and once the model has settled the bits at the
// surface are clear already: then no atomic is issued.
__device__ __forceinline__ void clear_free(const FuseArgs& a, int bi, int bj, int bk, int lane, int free,
                                           float lane_min, float lane_k0)
{
    if (!__ballot(lane_min < kSkipBound) || !__ballot(free != 0)) return;
    const bool i0 = (lane & 7) == 0, j0 = (lane >> 3) == 0;
#pragma unroll
    for (int l = 0; l < 8; ++l) {
        const int b = __builtin_amdgcn_readlane(free, l);
        if (b == 0) continue;  // uniform
        const int dx = l & 1, dy = (l >> 1) & 1, dz = l >> 2;
        const float v = ((!dx || i0) && (!dy || j0)) ? (dz ? lane_k0 : lane_min) : 1.0f;
        const bool large = (b & 1) && __ballot(v < kSkipBound), small = (b & 2) && __ballot(v < 0.0f);
        if (lane < 2 && (lane == 0 ? large : small)) {
            const int x = bi - dx;
            atomicAnd(&a.free_bits[free_word(a.nb, x, bj - dy, bk - dz, lane)], ~(1ull << (x & 63)));
        }
    }
}

// One wave fuses brick (bi, bj, bk) (lane = (j, i) inside the brick, its
// column of 8 voxels along z) and clears the free bits it ends.  Returns
// the lane's count of updated voxels.
//
// A brick in free space (kFreeBrick) needs no projection in the precision form, whose
// weights do not depend on the depth: every voxel is updated by f = 1, and where every
// code is 1 already only the counts change.  Sweep of a tick of 64 sessions of 512^3
// 920 -> 665 us.  Only a batch's cull marks bricks: one session's sweep is bound by its
// chain of dependent reads, and its cull and depth ranges took 1.5 us more for the test.
//
// The brick's z terms are uniform: they are read through the constant address
// space (scalar loads, issued together at the start).
typedef __attribute__((address_space(4))) const float ConstFloat;
typedef __attribute__((address_space(4))) const int ConstInt;
typedef __attribute__((address_space(4))) const unsigned int ConstUint;

template <int FMT, bool FREE>
__device__ __forceinline__ int fuse_brick(const FuseArgs& a, const float* ip, unsigned packed, int lane,
                                          const float* inv_count)
{
    const int bi = (int)(packed & 1023u), bj = (int)((packed >> 10) & 1023u), bk = (int)((packed >> 20) & 1023u);
    const int64_t brick = ((int64_t)bk * a.nb + bj) * a.nb + bi;
    if (FREE && (packed & kFreeBrick)) {  // uniform
        const int64_t base = brick * kBrickVoxels + lane * 8;
        ColumnPlanes<KF_VOXEL_SNORM16_U8> v;
        v.load(a, base);
        if (!__ballot(!v.settled())) {
            v.count_all();
            *reinterpret_cast<uint2*>(static_cast<uint8_t*>(a.wt) + base) = v.w;
            return 8;
        }
        const int free = load_free(a, bi, bj, bk, lane);
        float fmin = __int_as_float(0x7f800000), fk0 = fmin;
#pragma unroll
        for (int kl = 0; kl < 8; ++kl) update_voxel(v, kl, 1.0f, inv_count, fmin, fk0);
        v.store(a, base);
        clear_free(a, bi, bj, bk, lane, free, fmin, fk0);
        return 8;
    }
    float4 zt[8];
#pragma unroll
    for (int kl = 0; kl < 8; ++kl) {
        ConstFloat* z = (ConstFloat*)a.zt + (bk * 8 + kl) * 4;
        zt[kl] = make_float4(z[0], z[1], z[2], 0.0f);
    }
    const int i = bi * 8 + (lane & 7), j = bj * 8 + (lane >> 3);
    const float x = a.half + (float)i * a.res, y = a.half + (float)j * a.res;
    const v3 col = mk3(ip[0] * x + ip[4] * y, ip[1] * x + ip[5] * y, ip[2] * x + ip[6] * y);
    const int free = load_free(a, bi, bj, bk, lane);
    float fmin = __int_as_float(0x7f800000), fk0 = fmin;
    const int cnt = fuse_column<FMT>(a, col, zt, brick * kBrickVoxels + lane * 8, fmin, fk0, inv_count);
    clear_free(a, bi, bj, bk, lane, free, fmin, fk0);
    return cnt;
}

// Sums the lanes' counts of a workgroup into its own slot (slot b belongs to
// workgroup b; the add returns nothing, so the wave does not wait for it).
__device__ __forceinline__ void add_touched(unsigned long long* touched, int cnt, int* wave_cnt)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    cnt = wave_sum(cnt);
    if (lane == 0) wave_cnt[wave] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        int c = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) c += wave_cnt[w];
        if (c) atomicAdd(&touched[blockIdx.x], (unsigned long long)c);
    }
}

// Pass 2: waves stride over the visible bricks.  The skip flag, the pose, the
// list length and the wave's first list entry are uniform loads issued
// together (the list buffer holds an entry per brick of the volume, so reading
// an entry past the length stays inside it); the next entry is fetched while
// a brick is fused.

template <int FMT>
__global__ __launch_bounds__(64 * kFuseWaves, 7) void fuse_list_kernel(FuseArgs a, const int* list,
                                                                    const unsigned int* count)
{
    __shared__ int wave_cnt[kFuseWaves];
    __shared__ float inv_count[kInvCount];
    if (FMT != KF_VOXEL_F32) fill_inv_count(inv_count);
    // constant address space: no kernel writes the PoseState, the list or its
    // length while this one runs
    typedef __attribute__((address_space(4))) const PoseState ConstState;
    const int lane = threadIdx.x & 63;
    const unsigned int wave = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned int cap = (unsigned)a.nb * (unsigned)a.nb * (unsigned)a.nb;
    const unsigned int waves = gridDim.x * kFuseWaves;
    unsigned int item = blockIdx.x * kFuseWaves + wave;
    const int skip = a.dyn ? ((ConstState*)a.dyn)->frame_skip_fuse : 0;
    float ip[16];
    if (a.dyn) {
        ConstState* cs = (ConstState*)a.dyn;
#pragma unroll
        for (int q = 0; q < 16; ++q) ip[q] = cs->inv_pose[q];
    } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) ip[q] = a.inv_pose[q];
    }
    const unsigned int total = *(ConstUint*)count;
    unsigned brick = item < cap ? ((ConstUint*)list)[item] : 0u;
    if (skip) return;
    int cnt = 0;
    while (item < total) {
        const unsigned int next = item + waves;
        const unsigned next_brick = next < cap ? ((ConstUint*)list)[next] : 0u;
        cnt += fuse_brick<FMT, false>(a, ip, brick, lane, inv_count);
        item = next;
        brick = next_brick;
    }
    add_touched(a.touched, cnt, wave_cnt);
}

// ---- many sessions per launch (batch ticks).  The cull tests cubes of 4x4x4 bricks
// and the bricks of those it cannot drop.  Jobs are sorted by group0; global cube g of
// the tick belongs to the job whose range holds it.  List entries are job << 32 |
// pack_brick(bi, bj, bk) (the brick's coordinates in the job's volume), so the sweep
// needs no search.
//
// A lane tests a cube; then its wave tests, one after the other, the bricks of the
// cubes that are left, a lane each, and keeps which are listed and which are in free
// space as two masks per cube.  The workgroup takes one slot range of the list for all
// of its masks.  A wave's cubes lie a launch's waves apart, so each wave gets its part
// of every view (visible cubes lie together).  Bound: latency and the vector ALU; a
// test per brick instead (350 operations) took a tick of 64 sessions of 512^3 176 us,
// this form 98 us on 8192 workgroups.
constexpr int kBatchCullThreads = 256;
constexpr int kGroup = 4;  // bricks per cube and axis

template <class CJ>
__device__ __forceinline__ void load_cull_args(const CJ& j, FuseArgs& a)
{
    a.w = j.a.w;
    a.h = j.a.h;
    a.K[0] = j.a.K[0];
    a.K[4] = j.a.K[4];
    a.K[6] = j.a.K[6];
    a.K[7] = j.a.K[7];
    a.dyn = j.a.dyn;
    a.nb = j.a.nb;
    a.half = j.a.half;
    a.res = j.a.res;
    a.mue = j.a.mue;
    a.cull = j.a.cull;
#pragma unroll
    for (int q = 0; q < 4; ++q) a.plane_norm[q] = j.a.plane_norm[q];
    a.drange = j.a.drange;
    a.tx16 = j.a.tx16;
    a.ty16 = j.a.ty16;
    a.tx64 = j.a.tx64;
    a.ty64 = j.a.ty64;
}

__device__ __forceinline__ uint64_t lane_mask(uint64_t v, int lane)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), lane);
    return (uint64_t)hi << 32 | lo;
}

__global__ __launch_bounds__(kBatchCullThreads) void fuse_batch_cull_kernel(const BatchHeader* hd,
                                                                           const FuseJob* jobs)
{
    constexpr int kWaves = kBatchCullThreads / 64;
    typedef __attribute__((address_space(4))) const FuseJob ConstJob;
    typedef __attribute__((address_space(4))) const PoseState ConstState;
    __shared__ unsigned wave_sum_[kWaves], slot0;
    const unsigned total = hd->fuse_groups;
    const int njobs = hd->n_fuse;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned waves = gridDim.x * kWaves;
    // uniform trip count so every lane reaches the barriers
    for (unsigned start = 0; start < total; start += waves * 64) {
        const unsigned g = start + (unsigned)lane * waves + blockIdx.x * kWaves + (unsigned)wave;
        int j = 0;
        unsigned cube = 0u;  // pack_brick of its coordinates
        bool vis = false;
        if (g < total) {
            j = job_of(jobs, njobs, g, [](const FuseJob& x) { return x.group0; });
            const FuseArgs& a = jobs[j].a;
            if (!a.dyn->frame_skip_fuse) {
                const float* ip = a.dyn->inv_pose;
                const unsigned q = g - jobs[j].group0, ng = (unsigned)(a.nb + kGroup - 1) / kGroup;
                for (unsigned k = q; k < (unsigned)a.n; k += ng * ng * ng) z_terms(ip, a.zk, a.zt, (int)k);
                const int gi = (int)(q % ng), gj = (int)((q / ng) % ng), gk = (int)(q / (ng * ng));
                cube = pack_brick(gi, gj, gk);
                vis = !a.cull || cube_test<8 * kGroup, false>(a, ip, gi, gj, gk);
            }
        }
        uint64_t listed = 0, in_free = 0;  // of the lane's own cube
        for (uint64_t m = __ballot(vis); m; m &= m - 1) {
            const int l = __ffsll((unsigned long long)m) - 1;
            // the cube's job and pose in scalar registers (neither is written while the kernel runs)
            FuseArgs a;
            load_cull_args(((ConstJob*)jobs)[__builtin_amdgcn_readlane(j, l)], a);
            float ip[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) ip[q] = ((ConstState*)a.dyn)->inv_pose[q];
            const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)cube, l);
            const int bi = (int)(c & 1023u) * kGroup + (lane & 3), bj = (int)((c >> 10) & 1023u) * kGroup + ((lane >> 2) & 3),
                      bk = (int)(c >> 20) * kGroup + (lane >> 4);
            unsigned t = 0u;
            if (bi < a.nb && bj < a.nb && bk < a.nb) t = a.cull ? cube_test<8, true>(a, ip, bi, bj, bk) : 1u;
            const uint64_t any = __ballot(t != 0u), fr = __ballot((t & kFreeBrick) != 0u);
            if (lane == l) {
                listed = any;
                in_free = fr;
            }
        }
        // slots: by wave, then by cube (lane), then by brick
        const int mine = __popcll(listed);
        int before = mine;  // inclusive sum over the lanes
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(before, d);
            if (lane >= d) before += o;
        }
        if (lane == 63) wave_sum_[wave] = (unsigned)before;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned t = 0;
            for (int w = 0; w < kWaves; ++w) t += wave_sum_[w];
            slot0 = t ? atomicAdd(hd->fuse_count, t) : 0u;
        }
        __syncthreads();
        unsigned base = slot0 + (unsigned)(before - mine);
        for (int w = 0; w < wave; ++w) base += wave_sum_[w];
        for (uint64_t m = __ballot(listed != 0); m; m &= m - 1) {
            const int l = __ffsll((unsigned long long)m) - 1;
            const uint64_t any = lane_mask(listed, l);
            if (!((any >> lane) & 1ull)) continue;
            const uint64_t fr = lane_mask(in_free, l);
            const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)cube, l);
            const unsigned brick = pack_brick((int)(c & 1023u) * kGroup + (lane & 3),
                                              (int)((c >> 10) & 1023u) * kGroup + ((lane >> 2) & 3),
                                              (int)(c >> 20) * kGroup + (lane >> 4)) |
                                   (((fr >> lane) & 1ull) ? kFreeBrick : 0u);
            hd->fuse_list[(unsigned)__builtin_amdgcn_readlane((int)base, l) +
                          (unsigned)__popcll(any & ((1ull << lane) - 1ull))] =
                (unsigned long long)__builtin_amdgcn_readlane(j, l) << 32 | brick;
        }
        __syncthreads();  // the next trip's sums
    }
}

// Field-wise copy of a job's arguments read through the constant address
// space (scalar loads; the inverse pose comes from the session's PoseState).
template <class CJ>
__device__ __forceinline__ void load_fuse_args(const CJ& j, FuseArgs& a)
{
    a.depth = j.a.depth;
    a.w = j.a.w;
    a.h = j.a.h;
#pragma unroll
    for (int q = 0; q < 9; ++q) a.K[q] = j.a.K[q];
    a.dyn = j.a.dyn;
    a.n = j.a.n;
    a.nb = j.a.nb;
    a.half = j.a.half;
    a.res = j.a.res;
    a.mue = j.a.mue;
    a.inv_mue = j.a.inv_mue;
    a.zk = j.a.zk;
    a.zt = j.a.zt;
    a.band = j.a.band;
    a.f = j.a.f;
    a.wt = j.a.wt;
    a.free_bits = j.a.free_bits;
    a.cull = j.a.cull;
    a.format = j.a.format;
}

// Each wave sweeps a contiguous run of the list, in which the bricks of a cube (up
// to 64) follow one another and the next cube mostly belongs to another session
// (the cull's lanes take cubes a launch's waves apart): the job's arguments and
// pose are reloaded when the job changes, about once a cube, and the next entry is
// fetched while a brick is fused. Eight waves per SIMD: the
// job arguments otherwise hold 106 SGPRs (seven waves); at eight, 40 of them
// move to VGPR lanes, no scratch, and a 64-session tick measured 0.6 % faster.
__global__ __launch_bounds__(64 * kFuseWaves, 8) void fuse_batch_list_kernel(const BatchHeader* hd, const FuseJob* jobs)
{
    __shared__ int wave_cnt[kFuseWaves];
    __shared__ float inv_count[kInvCount];
    fill_inv_count(inv_count);
    // the tick's table, the list and its length are never written while the
    // kernel runs: read them with scalar loads through the constant address space
    typedef __attribute__((address_space(4))) const FuseJob ConstJob;
    typedef __attribute__((address_space(4))) const BatchHeader ConstHeader;
    typedef __attribute__((address_space(4))) const PoseState ConstState;
    typedef __attribute__((address_space(4))) const unsigned long long ConstEntry;
    ConstJob* cj = (ConstJob*)jobs;
    ConstHeader* ch = (ConstHeader*)hd;
    const int lane = threadIdx.x & 63;
    const unsigned int wave = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned int total = *(ConstUint*)ch->fuse_count;
    ConstEntry* list = (ConstEntry*)ch->fuse_list;
    const unsigned int waves = gridDim.x * kFuseWaves;
    const unsigned int per = (total + waves - 1) / waves;
    const unsigned long long first = (unsigned long long)(blockIdx.x * kFuseWaves + wave) * per;
    unsigned int item = first < total ? (unsigned)first : total;
    const unsigned int end = item + per < total ? item + per : total;
    unsigned long long e = item < end ? list[item] : 0ull;
    int cur = -1;
    FuseArgs a;
    float ip[16];
    int cnt = 0;
    while (item < end) {
        const unsigned long long ne = item + 1 < end ? list[item + 1] : 0ull;
        const int job = (int)(e >> 32);
        const unsigned brick = (unsigned)(e & 0xffffffffull);
        if (job != cur) {
            cur = job;
            load_fuse_args(cj[job], a);
            ConstState* cs = (ConstState*)a.dyn;
#pragma unroll
            for (int q = 0; q < 16; ++q) ip[q] = cs->inv_pose[q];
        }
        if (a.format == KF_VOXEL_F32) cnt += fuse_brick<KF_VOXEL_F32, false>(a, ip, brick, lane, inv_count);
        else cnt += fuse_brick<KF_VOXEL_SNORM16_U8, true>(a, ip, brick, lane, inv_count);
        e = ne;
        ++item;
    }
    add_touched(hd->touched, cnt, wave_cnt);
}

// Bound: HBM writes.  Stores of a voxel each took 12.6 us for 200^3 snorm16 voxels
// (1.9 TB/s), of 16 bytes 7.2 us; 512^3 FP32 takes 156 us either way (6.9 TB/s).
template <int FMT>
__global__ __launch_bounds__(256) void init_kernel(void* f, void* wt, int64_t count, float f0, float w0,
                                                   unsigned long long* free_bits, uint8_t* dist, int nb)
{
    int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * 256;
    const float fb = (FMT == KF_VOXEL_F32) ? f0 : snorm_decode(snorm_encode(f0));
    const bool large = fb >= kSkipBound, small = fb >= 0.0f;
    const int W = nb > 64 ? 2 : 1;
    for (int64_t r = q; r < (int64_t)nb * nb * 2 * W; r += stride)
        free_bits[r] = ((r / W) & 1 ? small : large) ? ~0ull : 0ull;
    const uint8_t db = (uint8_t)((large ? kDistMax : 0) | (small ? kDistMax << 4 : 0));
    for (int64_t b = q; b < (int64_t)nb * nb * nb; b += stride) dist[b] = db;
    // 16 bytes a store; count is a multiple of 512
    if (FMT == KF_VOXEL_F32) {
        const float4 fv = make_float4(f0, f0, f0, f0), wv = make_float4(w0, w0, w0, w0);
        for (; q < count / 4; q += stride) {
            static_cast<float4*>(f)[q] = fv;
            static_cast<float4*>(wt)[q] = wv;
        }
    } else {
        const unsigned c = (unsigned)(uint16_t)snorm_encode(f0) * 0x10001u;
        const unsigned k = (unsigned)(uint8_t)rintf(fminf(fmaxf(w0, 0.0f), 255.0f)) * 0x1010101u;
        const uint4 fv = make_uint4(c, c, c, c), wv = make_uint4(k, k, k, k);
        for (; q < count / 16; q += stride) {
            static_cast<uint4*>(f)[2 * q] = fv;
            static_cast<uint4*>(f)[2 * q + 1] = fv;
            static_cast<uint4*>(wt)[q] = wv;
        }
    }
}

// Raw interchange <-> bricked planes, for `count` voxels from q0 in the
// interchange's order (x fastest, then y and z).  slab: their interleaved (f, w)
// floats, in pinned host memory: the kernels move them over the host link themselves
// (8 bytes a lane, 512 contiguous bytes a wave).
template <int FMT>
__global__ __launch_bounds__(256) void slab_to_volume(const float2* __restrict__ slab, void* f, void* wt, int n, int nb,
                                                      int64_t q0, int64_t count)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= count) return;
    const int64_t q = q0 + e, row = q / n;
    const int i = (int)(q - row * n), k = (int)(row / n), j = (int)(row - (int64_t)k * n);
    const int64_t d = brick_index(nb, i, j, k);
    const float2 fw = slab[e];
    if (FMT == KF_VOXEL_F32) {
        static_cast<float*>(f)[d] = fw.x;
        static_cast<float*>(wt)[d] = fw.y;
    } else {
        static_cast<int16_t*>(f)[d] = snorm_encode(fw.x);
        static_cast<uint8_t*>(wt)[d] = (uint8_t)rintf(fminf(fmaxf(fw.y, 0.0f), 255.0f));
    }
}
template <int FMT>
__global__ __launch_bounds__(256) void volume_to_slab(float2* __restrict__ slab, const void* f, const void* wt, int n,
                                                      int nb, int64_t q0, int64_t count)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= count) return;
    const int64_t q = q0 + e, row = q / n;
    const int i = (int)(q - row * n), k = (int)(row / n), j = (int)(row - (int64_t)k * n);
    const int64_t d = brick_index(nb, i, j, k);
    if (FMT == KF_VOXEL_F32)
        slab[e] = make_float2(static_cast<const float*>(f)[d], static_cast<const float*>(wt)[d]);
    else
        slab[e] = make_float2(snorm_decode(static_cast<const int16_t*>(f)[d]),
                              (float)static_cast<const uint8_t*>(wt)[d]);
}

// Every free bit set (before free_bits_kernel clears the others).
__global__ void free_reset_kernel(unsigned long long* free_bits, int64_t words)
{
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q < words) free_bits[q] = ~0ull;
}

// Free bits from the voxels (after an upload): one wave per brick takes the 9^3
// voxels [8b, 8b + 8] per axis that lie in the volume.
template <int FMT>
__global__ __launch_bounds__(256) void free_bits_kernel(const void* f, unsigned long long* free_bits, int64_t nbricks,
                                                        int n, int nb)
{
    const int64_t brick = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (brick >= nbricks) return;
    const int lane = threadIdx.x & 63;
    const int bi = (int)(brick % nb), bj = (int)((brick / nb) % nb), bk = (int)(brick / ((int64_t)nb * nb));
    float m = __int_as_float(0x7f800000);
    for (int q = lane; q < 9 * 9 * 9; q += 64) {
        const int i = bi * 8 + q % 9, j = bj * 8 + (q / 9) % 9, k = bk * 8 + q / 81;
        if (i >= n || j >= n || k >= n) continue;
        const int64_t idx = brick_index(nb, i, j, k);
        const float v = (FMT == KF_VOXEL_F32) ? static_cast<const float*>(f)[idx]
                                              : snorm_decode(static_cast<const int16_t*>(f)[idx]);
        m = fminf(m, v);
    }
    m = wave_min(m);
    if (lane < 2 && m < (lane == 0 ? kSkipBound : 0.0f))
        atomicAnd(&free_bits[free_word(nb, bi, bj, bk, lane)], ~(1ull << (bi & 63)));
}

// ---- free distances (kf_device.hpp) from the free bits.
// One workgroup per 8 x 8 rows of bricks along x, one lane per row of the
// 24 x 24 window its distances depend on.  A row's free bits are one or two words
// (W) per kind of step, and a step of the distance is an erosion by one brick: two
// shifts along x, then the neighbouring rows along y and z through LDS.  A
// brick's distance is the number of steps it stays free, counted in four
// bit-sliced planes per row.  Rows past the window count as free; what they
// get wrong moves in one row per step and ends outside the 8 x 8 rows.
//
// Bound: latency (64 workgroups for 512^3): one load per lane, then kDistRadius
// steps of two barriers: 7.5 us for one 512^3 volume, 0.13 ms for 64 of them.
constexpr int kDistWin = 8 + 2 * kDistRadius;
constexpr int kDistThreads = kDistWin * kDistWin;
static_assert(kDistThreads % 64 == 0 && kDistMax < 16, "whole waves; distances fit four bits");
// Two words per row and exchange: both kinds of step at once for one-word rows,
// one kind after the other for two-word rows (their registers at once, 148,
// left room for one workgroup per CU).
template <int W>
struct DistRows {
    uint64_t a[kDistThreads][2], b[kDistThreads][2];
    uint64_t planes[64][2][4][W];
};
template <int W>
__device__ __forceinline__ void erode_x(uint64_t* m)
{
    if (W == 1) {
        m[0] &= ((m[0] >> 1) | (1ull << 63)) & ((m[0] << 1) | 1ull);
    } else {
        const uint64_t lo = m[0], hi = m[W - 1];
        m[0] = lo & ((lo >> 1) | (hi << 63)) & ((lo << 1) | 1ull);
        m[W - 1] = hi & ((hi >> 1) | (1ull << 63)) & ((hi << 1) | (lo >> 63));
    }
}
template <int W>
__device__ void brick_dist_tile(const unsigned long long* free_bits, uint8_t* dist, int nb, int tile, DistRows<W>& S)
{
    const int tid = threadIdx.x, tiles = (nb + 7) / 8, ty = tile % tiles, tz = tile / tiles;
    const int y = tid % kDistWin, z = tid / kDistWin;
    const int gy = ty * 8 - kDistRadius + y, gz = tz * 8 - kDistRadius + z;
    const bool in = gy >= 0 && gy < nb && gz >= 0 && gz < nb;
    const unsigned long long* r = free_bits + free_word(nb, 0, clampi(gy, 0, nb - 1), clampi(gz, 0, nb - 1), 0);
    const int ym = tid - (y > 0), yp = tid + (y < kDistWin - 1);
    const int zm = z > 0 ? tid - kDistWin : tid, zp = z < kDistWin - 1 ? tid + kDistWin : tid;
    constexpr int kKinds = 2 / W;  // kinds of step at once
    for (int h0 = 0; h0 < 2; h0 += kKinds) {
        uint64_t m[2], c[2][4];  // [kind][word], kKinds x W
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            m[q] = r[h0 * W + q];
            // bricks past the volume are free
            const int valid = nb - 64 * (q % W);
            if (valid < 64) m[q] |= ~0ull << valid;
            if (!in) m[q] = ~0ull;
            c[q][0] = m[q];
            c[q][1] = c[q][2] = c[q][3] = 0;
        }
        for (int s = 0; s < kDistRadius; ++s) {
#pragma unroll
            for (int h = 0; h < kKinds; ++h) erode_x<W>(m + h * W);
#pragma unroll
            for (int q = 0; q < 2; ++q) S.a[tid][q] = m[q];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                m[q] &= S.a[ym][q] & S.a[yp][q];
                S.b[tid][q] = m[q];
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                m[q] &= S.b[zm][q] & S.b[zp][q];
                uint64_t carry = m[q];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint64_t t = c[q][p] & carry;
                    c[q][p] ^= carry;
                    carry = t;
                }
            }
        }
        const int oy = y - kDistRadius, oz = z - kDistRadius;
        if (oy >= 0 && oy < 8 && oz >= 0 && oz < 8) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int p = 0; p < 4; ++p) S.planes[oz * 8 + oy][h0 + q / W][p][q % W] = c[q][p];
        }
    }
    __syncthreads();
    // one row of the tile per wave, a brick per lane
    const int lane = tid & 63;
    for (int o = __builtin_amdgcn_readfirstlane(tid >> 6); o < 64; o += kDistThreads / 64) {
        const int by = ty * 8 + (o & 7), bz = tz * 8 + (o >> 3);
        if (by >= nb || bz >= nb) continue;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            unsigned d = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    d |= (unsigned)((S.planes[o][h][p][w] >> lane) & 1ull) << (4 * h + p);
            if (w * 64 + lane < nb) dist[((int64_t)bz * nb + by) * nb + w * 64 + lane] = (uint8_t)d;
        }
    }
}
template <int W>
__global__ __launch_bounds__(kDistThreads) void brick_dist_kernel(const unsigned long long* free_bits, uint8_t* dist,
                                                                  int nb)
{
    __shared__ DistRows<W> S;
    brick_dist_tile<W>(free_bits, dist, nb, blockIdx.x, S);
}
// The same for every fused volume of a tick (workgroups stride over the tiles).
__global__ __launch_bounds__(kDistThreads) void brick_dist_batch_kernel(const BatchHeader* hd, const FuseJob* jobs)
{
    __shared__ union {
        DistRows<1> one;
        DistRows<2> two;
    } S;
    const int tiles = hd->dist_tiles, njobs = hd->n_fuse;
    for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
        const FuseJob& J = jobs[job_of(jobs, njobs, t, [](const FuseJob& x) { return x.dist_tile0; })];
        if (J.a.nb <= 64) brick_dist_tile<1>(J.a.free_bits, J.a.dist, J.a.nb, t - J.dist_tile0, S.one);
        else brick_dist_tile<2>(J.a.free_bits, J.a.dist, J.a.nb, t - J.dist_tile0, S.two);
        __syncthreads();  // the planes have been read
    }
}
int launch_brick_dist(const kf_volume* v, hipStream_t s)
{
    const unsigned blocks = (unsigned)dist_tiles(v->nb);
    if (v->nb <= 64) brick_dist_kernel<1><<<blocks, kDistThreads, 0, s>>>(v->free_bits, v->dist, v->nb);
    else brick_dist_kernel<2><<<blocks, kDistThreads, 0, s>>>(v->free_bits, v->dist, v->nb);
    KF_LAUNCHED("brick_dist_kernel");
    return KF_OK;
}
// Whether work enqueued on `s` goes into a graph (the query fails for the null stream
// while another stream is captured: taken as yes).
bool stream_captures(hipStream_t s)
{
    hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &c) == hipSuccess) return c != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

// z of each k slice: one lane, the host loop's repeated additions in order.
__global__ void z_table_kernel(float* zk, int n, float half, float res)
{
    float z = half + (-res);
    for (int k = 0; k < n; ++k) {
        z = z + res;
        zk[k] = z;
    }
}

bool is_pinhole(const float* K)
{
    return K[1] == 0.0f && K[2] == 0.0f && K[3] == 0.0f && K[5] == 0.0f && K[8] == 1.0f && K[0] > 0.0f &&
           K[4] > 0.0f;
}

// Moves voxels [q0, q1) between the volume and the host's side through two pinned
// chunks in turn, so the host fills or empties one while a kernel moves the other.
// host_side(q, count, chunk): reads or writes `count` voxels from q.
constexpr int64_t kChunkVoxels = 1 << 18;  // 2 MiB
template <class Fn>
int move_voxels(const kf_volume* v, bool to_volume, int64_t q0, int64_t q1, float2* pinned, const hipEvent_t* ev,
                Fn&& host_side)
{
    const auto launch = [&](int64_t q, int b) -> int {
        const int64_t count = std::min(kChunkVoxels, q1 - q);
        const unsigned blocks = (unsigned)((count + 255) / 256);
        float2* slab = pinned + b * kChunkVoxels;
        const bool f32 = v->format == KF_VOXEL_F32;
        if (to_volume && f32)
            slab_to_volume<KF_VOXEL_F32><<<blocks, 256>>>(slab, v->f, v->w, v->n, v->nb, q, count);
        else if (to_volume)
            slab_to_volume<KF_VOXEL_SNORM16_U8><<<blocks, 256>>>(slab, v->f, v->w, v->n, v->nb, q, count);
        else if (f32)
            volume_to_slab<KF_VOXEL_F32><<<blocks, 256>>>(slab, v->f, v->w, v->n, v->nb, q, count);
        else
            volume_to_slab<KF_VOXEL_SNORM16_U8><<<blocks, 256>>>(slab, v->f, v->w, v->n, v->nb, q, count);
        KF_LAUNCHED("volume transfer");
        if (ev[b]) KF_HIP(hipEventRecord(ev[b], nullptr));
        return KF_OK;
    };
    int st = KF_OK, b = 0;
    if (!to_volume && q0 < q1) st = launch(q0, 0);
    for (int64_t q = q0; q < q1 && st == KF_OK; q += kChunkVoxels, b ^= 1) {
        const int64_t count = std::min(kChunkVoxels, q1 - q);
        if (!to_volume && q + kChunkVoxels < q1) st = launch(q + kChunkVoxels, b ^ 1);
        // the chunk's last kernel is done (an event never recorded counts as done; a volume
        // of one chunk has no events)
        if (st == KF_OK && (ev[b] || !to_volume)) {
            const hipError_t e = ev[b] ? hipEventSynchronize(ev[b]) : hipStreamSynchronize(nullptr);
            if (e != hipSuccess) st = fail_hip(e, "volume transfer");
        }
        if (st == KF_OK) st = host_side(q, count, pinned + b * kChunkVoxels);
        if (st == KF_OK && to_volume) st = launch(q, b);
    }
    return st;
}

// The volume to or from the host.  `parallel`: host_side may run for several chunks
// at once, on threads of this call, each moving a part of the volume through chunks
// of its own: one core copies at a quarter of the host link's rate.  Small volumes
// are not worth the threads (about 50 us each).  A 256^3 FP32 volume from the host
// and back (268 MB), through one pageable layer, its staged copy and a device copy in
// turn -> now: 24.1 -> 6.2 ms, 43 GB/s.
template <class Fn>
int move_volume(const kf_volume* v, bool to_volume, bool parallel, Fn&& host_side)
{
    constexpr int kMovers = 4;
    const int64_t total = (int64_t)v->n * v->n * v->n;
    const int movers = parallel ? (int)std::min<int64_t>(kMovers, std::max<int64_t>(1, total / (2 * kChunkVoxels))) : 1;
    float2* pinned = nullptr;
    hipEvent_t ev[2 * kMovers] = {};
    // a volume of one chunk (up to 64^3) needs no second one
    const int64_t slots = total <= kChunkVoxels ? total : 2 * kChunkVoxels * movers;
    KF_HIP(hipHostMalloc(reinterpret_cast<void**>(&pinned), sizeof(float2) * (size_t)slots, hipHostMallocDefault));
    int st = KF_OK;
    for (int k = 0; k < 2 * movers && total > kChunkVoxels && st == KF_OK; ++k) {
        const hipError_t e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        if (e != hipSuccess) st = fail_hip(e, "volume transfer events");
    }
    if (st == KF_OK) {
        int device = 0;
        (void)hipGetDevice(&device);
        int status[kMovers] = {};
        std::string message[kMovers];
        const auto part = [&](int k) {  // whole chunks each
            const int64_t chunks = (total + kChunkVoxels - 1) / kChunkVoxels;
            const int64_t q0 = chunks * k / movers * kChunkVoxels;
            const int64_t q1 = std::min(total, chunks * (k + 1) / movers * kChunkVoxels);
            status[k] = move_voxels(v, to_volume, q0, q1, pinned + 2 * kChunkVoxels * k, ev + 2 * k, host_side);
        };
        std::vector<std::thread> threads;
        int started = 1;
        try {
            threads.reserve(kMovers);
            for (; started < movers; ++started) {
                const int k = started;
                threads.emplace_back([&, k] {
                    const hipError_t e = hipSetDevice(device);
                    if (e != hipSuccess) status[k] = fail_hip(e, "volume transfer");
                    else part(k);
                    if (status[k]) message[k] = kf_last_error();  // the thread's own
                });
            }
        } catch (const std::exception&) {
            // no more threads: this one moves the rest
        }
        part(0);
        for (int k = started; k < movers; ++k) part(k);
        for (std::thread& t : threads) t.join();
        for (int k = 0; k < movers && st == KF_OK; ++k)
            if (status[k]) st = message[k].empty() ? status[k] : fail(status[k], message[k]);
    }
    if (st == KF_OK && to_volume) {
        const int64_t nbricks = (int64_t)v->nb * v->nb * v->nb;
        const unsigned b = (unsigned)((nbricks + 3) / 4);
        const int64_t words = (int64_t)free_words(v->nb);
        free_reset_kernel<<<(unsigned)((words + 255) / 256), 256>>>(v->free_bits, words);
        if (v->format == KF_VOXEL_F32)
            free_bits_kernel<KF_VOXEL_F32><<<b, 256>>>(v->f, v->free_bits, nbricks, v->n, v->nb);
        else
            free_bits_kernel<KF_VOXEL_SNORM16_U8><<<b, 256>>>(v->f, v->free_bits, nbricks, v->n, v->nb);
        st = launch_brick_dist(v, nullptr);
        if (st == KF_OK) v->dist_stale = false;
    }
    const hipError_t e = hipDeviceSynchronize();  // nothing uses the chunks past this line
    if (st == KF_OK && e != hipSuccess) st = fail_hip(e, "volume transfer");
    for (hipEvent_t x : ev)
        if (x) (void)hipEventDestroy(x);
    (void)hipHostFree(pinned);
    return st;
}

}  // namespace

FuseArgs fuse_args(const float* depth, int w, int h, const kf_volume* v, const float* K, const float* inv_pose,
                   const PoseState* dyn_state)
{
    FuseArgs a{};
    a.depth = depth;
    a.w = w;
    a.h = h;
    memcpy(a.K, K, sizeof(a.K));
    if (inv_pose) memcpy(a.inv_pose, inv_pose, sizeof(a.inv_pose));
    a.dyn = dyn_state;
    a.n = v->n;
    a.nb = v->nb;
    a.half = -v->width * 0.5f;
    a.res = v->res;
    a.mue = v->mue;
    a.inv_mue = 1.0f / v->mue;
    a.zk = v->zk;
    a.zt = v->zt;
    a.band = (float)std::max(w, h) * 0x1p-21f;
    a.f = v->f;
    a.wt = v->w;
    a.touched = v->touched;
    a.free_bits = v->free_bits;
    a.dist = v->dist;
    a.cull = is_pinhole(K) ? 1 : 0;
    const double W = (double)w, H = (double)h;
    const double pn[4] = {std::hypot((double)K[0], (double)K[6]), std::hypot((double)K[0], W - (double)K[6]),
                          std::hypot((double)K[4], (double)K[7]), std::hypot((double)K[4], H - (double)K[7])};
    for (int q = 0; q < 4; ++q) a.plane_norm[q] = std::nextafter((float)pn[q], INFINITY);
    a.format = v->format;
    a.drange = nullptr;
    a.tx16 = (w + 15) / 16;
    a.ty16 = (h + 15) / 16;
    a.tx64 = (w + 63) / 64;
    a.ty64 = (h + 63) / 64;
    return a;
}

int launch_fuse_batch(const BatchHeader* hd, const FuseJob* jobs, unsigned cull_blocks, unsigned list_blocks,
                      hipStream_t s, hipEvent_t mid)
{
    fuse_batch_cull_kernel<<<cull_blocks, kBatchCullThreads, 0, s>>>(hd, jobs);
    KF_LAUNCHED("fuse_batch_cull_kernel");
    if (mid) KF_HIP(hipEventRecord(mid, s));
    fuse_batch_list_kernel<<<list_blocks, 64 * kFuseWaves, 0, s>>>(hd, jobs);
    KF_LAUNCHED("fuse_batch_list_kernel");
    // three workgroups of nine waves fit a CU
    brick_dist_batch_kernel<<<768, kDistThreads, 0, s>>>(hd, jobs);
    KF_LAUNCHED("brick_dist_batch_kernel");
    return KF_OK;
}

// Workgroups of the list sweep that are resident at once on the current
// device (at most kFuseBlocks, the size of the per-workgroup counters).
static int fuse_list_blocks(int format)
{
    static int cached[2] = {0, 0};
    int& c = cached[format == KF_VOXEL_F32 ? 0 : 1];
    if (!c) {
        int dev = 0, cus = 0, per_cu = 0;
        const void* k = format == KF_VOXEL_F32 ? reinterpret_cast<const void*>(&fuse_list_kernel<KF_VOXEL_F32>)
                                               : reinterpret_cast<const void*>(&fuse_list_kernel<KF_VOXEL_SNORM16_U8>);
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, 64 * kFuseWaves, 0) == hipSuccess && per_cu > 0 &&
            cus > 0)
            c = std::min<int>(kFuseBlocks, per_cu * cus);
        else
            c = kFuseBlocks;
    }
    return c;
}

float2* volume_depth_range(kf_volume* v, int w, int h, hipStream_t s)
{
    const size_t need = depth_range_tiles(w, h);
    if (v->drange_cap < need) {
        // grown outside the stream order: wait for work that may still read the old map
        if (hipStreamSynchronize(s) != hipSuccess) return nullptr;
        (void)hipFree(v->drange);
        v->drange = nullptr;
        v->drange_cap = 0;
        if (hipMalloc(&v->drange, sizeof(float2) * need) != hipSuccess) return nullptr;
        v->drange_cap = need;
    }
    return v->drange;
}

int launch_fuse(const float* depth, int w, int h, kf_volume* v, const float* K, const float* inv_pose,
                const PoseState* dyn_state, hipStream_t s, hipEvent_t* list_events, bool drange_ready)
{
    float2* drange = volume_depth_range(v, w, h, s);
    if (!drange) return fail(KF_ERR_OOM, "fuse: depth tile maps");
    if (stream_captures(s)) v->fuse_captured = true;
    else v->dist_stale = true;
    FuseArgs a = fuse_args(depth, w, h, v, K, inv_pose, dyn_state);
    a.drange = drange;
    if (!drange_ready) {
        depth_range_kernel<<<dim3((unsigned)a.tx64, (unsigned)a.ty64), 256, 0, s>>>(depth, w, h, drange, a.tx16, a.ty16,
                                                                                a.tx64);
        KF_LAUNCHED("depth_range_kernel");
    }
    const int64_t nbricks = (int64_t)v->nb * v->nb * v->nb;
    const int parity = (int)(v->fuse_launches & 1);
    fuse_cull_kernel<<<(unsigned)((nbricks + kCullThreads - 1) / kCullThreads), kCullThreads, 0, s>>>(
        a, nbricks, v->brick_list, v->list_count, parity);
    KF_LAUNCHED("fuse_cull_kernel");
    // every workgroup resident at once (no second round); fewer when the volume is small
    const unsigned blocks =
        (unsigned)std::min<int64_t>((nbricks + kFuseWaves - 1) / kFuseWaves, fuse_list_blocks(v->format));
    if (list_events) KF_HIP(hipEventRecord(list_events[0], s));
    if (v->format == KF_VOXEL_F32)
        fuse_list_kernel<KF_VOXEL_F32><<<blocks, 64 * kFuseWaves, 0, s>>>(a, v->brick_list, v->list_count + parity);
    else
        fuse_list_kernel<KF_VOXEL_SNORM16_U8><<<blocks, 64 * kFuseWaves, 0, s>>>(a, v->brick_list,
                                                                                 v->list_count + parity);
    KF_LAUNCHED("fuse_list_kernel");
    if (list_events) KF_HIP(hipEventRecord(list_events[1], s));
    v->fuse_launches += 1;
    return KF_OK;
}

// A fuse leaves the distances to the raycast that needs them (kf_fuse of 640x480 with
// them in every fuse -> now: 512^3 FP32 39.8 -> 32.0 us, 200^3 snorm16 24.7 -> 17.5).  A
// captured fuse may run again without a call here and a captured raycast after any
// fuse, so those always have the step.
int refresh_free_distances(const kf_volume* v, hipStream_t s)
{
    const bool captures = stream_captures(s);
    if (!v->dist_stale && !v->fuse_captured && !captures) return KF_OK;
    const int st = launch_brick_dist(v, s);
    if (st == KF_OK && !captures) v->dist_stale = false;
    return st;
}

int launch_initialize(kf_volume* v, float f, float wt, hipStream_t s)
{
    const int64_t count = (int64_t)v->n * v->n * v->n;
    const int64_t lanes = count / (v->format == KF_VOXEL_F32 ? 4 : 16);
    const unsigned blocks = (unsigned)std::min<int64_t>((lanes + 255) / 256, 65536);
    if (v->format == KF_VOXEL_F32)
        init_kernel<KF_VOXEL_F32><<<blocks, 256, 0, s>>>(v->f, v->w, count, f, wt, v->free_bits, v->dist, v->nb);
    else
        init_kernel<KF_VOXEL_SNORM16_U8><<<blocks, 256, 0, s>>>(v->f, v->w, count, f, wt, v->free_bits, v->dist,
                                                                v->nb);
    KF_LAUNCHED("init_kernel");
    return KF_OK;
}

// Allocates a volume and enqueues its initialisation on `s` (no host wait):
// the z table by repeated addition and every voxel at (2, 0).
int volume_create(int n, float width_m, float mue_m, int format, hipStream_t s, kf_volume** out)
{
    if (!out) return fail(KF_ERR_ARG, "kf_volume_create: null out");
    *out = nullptr;
    if (n < 8 || n % 8 != 0) return fail(KF_ERR_ARG, "kf_volume_create: n must be a positive multiple of 8");
    if (n > 1024) return fail(KF_ERR_ARG, "kf_volume_create: n must be at most 1024");
    if (!(width_m > 0.0f) || !(width_m < 1e4f)) return fail(KF_ERR_ARG, "kf_volume_create: width must be in (0, 1e4) m");
    // the raycast marches at >= 0.1 * mue; 1e-4 m keeps every march finite and short
    if (!(mue_m >= 1e-4f)) return fail(KF_ERR_ARG, "kf_volume_create: mue must be >= 1e-4 m");
    if (format != KF_VOXEL_F32 && format != KF_VOXEL_SNORM16_U8)
        return fail(KF_ERR_ARG, "kf_volume_create: unknown voxel format");
    kf_volume* v = new kf_volume();
    v->n = n;
    v->nb = n / 8;
    v->format = format;
    v->width = width_m;
    v->res = width_m / (float)(n - 1);  // voxel_grid.h:43
    v->mue = mue_m;
    const int64_t count = (int64_t)n * n * n;
    const size_t fb = (format == KF_VOXEL_F32) ? 4 : 2, wb = (format == KF_VOXEL_F32) ? 4 : 1;
    v->bytes = (size_t)count * (fb + wb);
    hipError_t e;
    if ((e = hipMalloc(&v->f, (size_t)count * fb)) != hipSuccess || (e = hipMalloc(&v->w, (size_t)count * wb)) != hipSuccess ||
        (e = hipMalloc(&v->zk, sizeof(float) * n)) != hipSuccess ||
        (e = hipMalloc(&v->zt, sizeof(float4) * n)) != hipSuccess ||
        (e = hipMalloc(&v->touched, sizeof(unsigned long long) * kFuseBlocks)) != hipSuccess ||
        (e = hipMemsetAsync(v->touched, 0, sizeof(unsigned long long) * kFuseBlocks, s)) != hipSuccess ||
        (e = hipMalloc(&v->brick_list, sizeof(int) * (size_t)v->nb * v->nb * v->nb)) != hipSuccess ||
        (e = hipMalloc(&v->free_bits, sizeof(unsigned long long) * free_words(v->nb))) != hipSuccess ||
        (e = hipMalloc(&v->dist, (size_t)v->nb * v->nb * v->nb)) != hipSuccess ||
        (e = hipMalloc(&v->list_count, 2 * sizeof(unsigned int))) != hipSuccess ||
        (e = hipMemsetAsync(v->list_count, 0, 2 * sizeof(unsigned int), s)) != hipSuccess) {
        kf_volume_destroy(v);
        return fail_hip(e, "kf_volume_create");
    }
    // tsdf.cu:27-31: z starts at -width/2 - res and advances by repeated addition
    z_table_kernel<<<1, 1, 0, s>>>(v->zk, n, -width_m * 0.5f, v->res);
    e = hipGetLastError();
    if (e != hipSuccess) {
        kf_volume_destroy(v);
        return fail_hip(e, "z_table_kernel");
    }
    // Voxel{} = (2, 0) (voxel_grid.h:10-16), as KinectFusion's constructor initialises it
    int st = launch_initialize(v, 2.0f, 0.0f, s);
    if (st != KF_OK) {
        kf_volume_destroy(v);
        return st;
    }
    *out = v;
    return KF_OK;
}

}  // namespace kf

// ------------------------------------------------------------------ C ABI
extern "C" {

int kf_volume_create(int n, float width_m, float mue_m, int format, kf_volume** out)
{
    int st = kf::volume_create(n, width_m, mue_m, format, nullptr, out);
    if (st) return st;
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        kf_volume_destroy(*out);
        *out = nullptr;
        return kf::fail_hip(e, "initialize");
    }
    return KF_OK;
}

int kf_volume_create_scaled(int n, float width_m, float mue_scale, int format, kf_volume** out)
{
    if (n < 2) return kf::fail(KF_ERR_ARG, "kf_volume_create_scaled: n too small");
    float res = width_m / (float)(n - 1);
    return kf_volume_create(n, width_m, mue_scale * res, format, out);  // voxel_grid.h:44
}

int kf_volume_destroy(kf_volume* v)
{
    if (!v) return KF_OK;
    (void)hipFree(v->f);
    (void)hipFree(v->w);
    (void)hipFree(v->zk);
    (void)hipFree(v->zt);
    (void)hipFree(v->touched);
    (void)hipFree(v->brick_list);
    (void)hipFree(v->free_bits);
    (void)hipFree(v->dist);
    (void)hipFree(v->list_count);
    (void)hipFree(v->drange);
    (void)hipFree(v->ray_list);
    (void)hipFree(v->ray_count);
    delete v;
    return KF_OK;
}

int kf_volume_info(const kf_volume* v, int* n, float* width_m, float* resolution, float* mue_m, int* format)
{
    if (!v) return kf::fail(KF_ERR_ARG, "kf_volume_info: null volume");
    if (n) *n = v->n;
    if (width_m) *width_m = v->width;
    if (resolution) *resolution = v->res;
    if (mue_m) *mue_m = v->mue;
    if (format) *format = v->format;
    return KF_OK;
}

int kf_volume_bytes(const kf_volume* v, size_t* bytes)
{
    if (!v || !bytes) return kf::fail(KF_ERR_ARG, "kf_volume_bytes: null argument");
    *bytes = v->bytes;
    return KF_OK;
}

int kf_volume_touched_total(const kf_volume* v, int64_t* count)
{
    if (!v || !count) return kf::fail(KF_ERR_ARG, "kf_volume_touched_total: null argument");
    std::vector<unsigned long long> part(kf::kFuseBlocks);
    KF_HIP(hipDeviceSynchronize());
    KF_HIP(hipMemcpy(part.data(), v->touched, sizeof(unsigned long long) * part.size(), hipMemcpyDeviceToHost));
    unsigned long long c = 0;
    for (auto x : part) c += x;
    *count = (int64_t)c;
    return KF_OK;
}

int kf_initialize_grid(kf_volume* v, float f, float w, kf_stream_t stream, float* elapsed_ms)
{
    if (!v) return kf::fail(KF_ERR_ARG, "initializeGrid: null volume");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_initialize(v, f, w, s))) return st;
    return t.finish();
}

int kf_fuse(const float* depth_m, int w, int h, kf_volume* v, const kf_sensor* sensor, kf_stream_t stream,
            float* elapsed_ms)
{
    if (!depth_m || !v || !sensor || w <= 0 || h <= 0) return kf::fail(KF_ERR_ARG, "fuse: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_fuse(depth_m, w, h, v, sensor->intr[0], sensor->inv_pose, nullptr, s, nullptr, false)))
        return st;
    return t.finish();
}

int kf_volume_download(const kf_volume* v, float* fw_host)
{
    if (!v || !fw_host) return kf::fail(KF_ERR_ARG, "kf_volume_download: null argument");
    KF_HIP(hipDeviceSynchronize());
    return kf::move_volume(v, false, true, [&](int64_t q, int64_t count, float2* chunk) {
        memcpy(fw_host + (size_t)q * 2, chunk, sizeof(float2) * (size_t)count);
        return (int)KF_OK;
    });
}

int kf_volume_upload(kf_volume* v, const float* fw_host)
{
    if (!v || !fw_host) return kf::fail(KF_ERR_ARG, "kf_volume_upload: null argument");
    KF_HIP(hipDeviceSynchronize());
    return kf::move_volume(v, true, true, [&](int64_t q, int64_t count, float2* chunk) {
        memcpy(chunk, fw_host + (size_t)q * 2, sizeof(float2) * (size_t)count);
        return (int)KF_OK;
    });
}

// voxel_grid.cpp:43-60
int kf_volume_save(const kf_volume* v, const char* path)
{
    if (!v || !path) return kf::fail(KF_ERR_ARG, "kf_volume_save: null argument");
    FILE* fp = fopen(path, "wb");
    if (!fp) return kf::fail(KF_ERR_IO, std::string("kf_volume_save: cannot open ") + path);
    KF_HIP(hipDeviceSynchronize());
    int st = kf::move_volume(v, false, false, [&](int64_t, int64_t count, float2* chunk) {
        return fwrite(chunk, sizeof(float2), (size_t)count, fp) == (size_t)count
                   ? (int)KF_OK
                   : kf::fail(KF_ERR_IO, "kf_volume_save: short write");
    });
    if (fclose(fp) != 0 && st == KF_OK) st = kf::fail(KF_ERR_IO, "kf_volume_save: close failed");
    return st;
}

// voxel_grid.cpp:62-80 (the reference reads without checking; a short file is an error here)
int kf_volume_load(kf_volume* v, const char* path)
{
    if (!v || !path) return kf::fail(KF_ERR_ARG, "kf_volume_load: null argument");
    FILE* fp = fopen(path, "rb");
    if (!fp) return kf::fail(KF_ERR_IO, std::string("kf_volume_load: cannot open ") + path);
    KF_HIP(hipDeviceSynchronize());
    int st = kf::move_volume(v, true, false, [&](int64_t, int64_t count, float2* chunk) {
        return fread(chunk, sizeof(float2), (size_t)count, fp) == (size_t)count
                   ? (int)KF_OK
                   : kf::fail(KF_ERR_IO, "kf_volume_load: short file");
    });
    fclose(fp);
    return st;
}

}  // extern "C"
