// Measurement step of the per-frame path (project/src/measurement.cu): raw
// depth codes -> metres, bilateral filter, depth pyramid, vertex and normal maps.
//
// Maps are plain row-major arrays in HBM (float depth, float4 vertex/normal with
// validity in .w).  Every kernel takes 16x16 lanes (4 waves of 64) a workgroup, one
// lane per output pixel of a 16x16 tile, or several per pixel of a larger region where
// its comment says so, with bounds checks, so any frame size works (the reference
// launches w/8 x h/8 blocks and skips the remainder).
#include <string.h>

#include "kf_device.hpp"
#include "kf_kernels.hpp"

namespace kf {

namespace {

constexpr int kTile = 16;

inline dim3 grid2d(int w, int h) { return dim3((w + kTile - 1) / kTile, (h + kTile - 1) / kTile); }

// measurement.cu:14-31
__global__ __launch_bounds__(256) void convert_kernel(const uint16_t* __restrict__ raw, float* __restrict__ out,
                                                      int w, int h, float scale, int unmirror)
{
    int i = blockIdx.x * kTile + threadIdx.x, j = blockIdx.y * kTile + threadIdx.y;
    if (i >= w || j >= h) return;
    float d = half_rne(raw[(int64_t)j * w + i]);
    int io = unmirror ? (w - 1 - i) : i;
    out[(int64_t)j * w + io] = d * scale;
}

// measurement.cu:33-66: 7x7, x outer / y inner, clamp-to-edge, sigma_s = 4, sigma_r = 0.25.
// The 22x22 input window of the tile is staged in LDS once, filled with
// clamp-to-edge reads, so tap (x, y) is simply the window element at the
// thread's offset.
typedef float BilateralTile[kTile + 6][kTile + 6 + 1];

// The weight's argument is -sd / sigma_s^2 - id / sigma_r^2 with
// 1 / sigma_s^2 = 1/16 and 1 / sigma_r^2 = 16: both products are exact (powers
// of two; 16 id overflows exactly when the product does), so it is one
// rounding of c - 16 id with c = -(x^2 + y^2) / 16 exact, i.e. one fused
// multiply-add on a per-tap constant.
//
// Bound: the vector ALU, 49 weights of 22 instructions (exp 16, argument 3,
// sums 3) and one LDS read per pixel; the 22x22 window costs under 2 reads and
// conversions per pixel.
//
// One column of taps.  CENTRE: the column holding the pixel itself, whose tap
// has weight exp(0) = 1; 0 * centre makes it NaN for a centre that is not
// finite, as its inf - inf would.
template <bool CENTRE>
__device__ __forceinline__ void bilateral_column(const BilateralTile& tile, int tx, int ty, int x, float center,
                                                 float& norm, float& acc)
{
    const float cx = (float)(x * x) * -0.0625f;
#pragma unroll
    for (int y = -3; y <= 3; ++y) {
        if (CENTRE && y == 0) {
            const float f = fmaf(center, 0.0f, 1.0f);
            norm = norm + f;
            acc = acc + f * center;
            continue;
        }
        const float cur = tile[ty + 3 + y][tx + 3 + x];
        float id = center - cur;
        id = id * id;
        const float f = kf_expf_nonpos(fmaf(id, -16.0f, cx + (float)(y * y) * -0.0625f));
        norm = norm + f;
        acc = acc + f * cur;
    }
}
__device__ __forceinline__ float bilateral_at(const BilateralTile& tile, int tx, int ty)
{
    const float center = tile[ty + 3][tx + 3];
    float norm = 0.0f, acc = 0.0f;
    // the loops over columns stay rolled: unrolled, all 49 taps' tile reads were
    // held at once (106 VGPRs, 4 waves per SIMD); rolled, under 32 and 8 waves
#pragma unroll 1
    for (int x = -3; x < 0; ++x) bilateral_column<false>(tile, tx, ty, x, center, norm, acc);
    bilateral_column<true>(tile, tx, ty, 0, center, norm, acc);
#pragma unroll 1
    for (int x = 1; x <= 3; ++x) bilateral_column<false>(tile, tx, ty, x, center, norm, acc);
    return acc / norm;
}

__global__ __launch_bounds__(256) void bilateral_kernel(const float* __restrict__ in, float* __restrict__ out, int w,
                                                        int h)
{
    __shared__ BilateralTile tile;
    const int i0 = blockIdx.x * kTile - 3, j0 = blockIdx.y * kTile - 3;
    const int t = threadIdx.y * kTile + threadIdx.x;
    for (int q = t; q < (kTile + 6) * (kTile + 6); q += kTile * kTile) {
        int ly = q / (kTile + 6), lx = q % (kTile + 6);
        int gi = clampi(i0 + lx, 0, w - 1), gj = clampi(j0 + ly, 0, h - 1);
        tile[ly][lx] = in[(int64_t)gj * w + gi];
    }
    __syncthreads();
    int i = blockIdx.x * kTile + threadIdx.x, j = blockIdx.y * kTile + threadIdx.y;
    if (i >= w || j >= h) return;
    out[(int64_t)j * w + i] = bilateral_at(tile, threadIdx.x, threadIdx.y);
}

// measurement.cu:68-102: the taps within 3 sigma_r of the top-left tap, averaged.
__device__ __forceinline__ float down4(float f1, float f2, float f3, float f4)
{
    const float tsd = 3.0f * 0.25f;
    float acc = f1;
    int cnt = 1;
    if (fabsf(f1 - f2) <= tsd) { acc = acc + f2; ++cnt; }
    if (fabsf(f1 - f3) <= tsd) { acc = acc + f3; ++cnt; }
    if (fabsf(f1 - f4) <= tsd) { acc = acc + f4; ++cnt; }
    return acc / (float)cnt;
}

__global__ __launch_bounds__(256) void down_sample_kernel(const float* __restrict__ in, int w, float* __restrict__ out,
                                                          int wo, int ho)
{
    int i = blockIdx.x * kTile + threadIdx.x, j = blockIdx.y * kTile + threadIdx.y;
    if (i >= wo || j >= ho) return;
    float f1 = in[(int64_t)(2 * j) * w + 2 * i], f2 = in[(int64_t)(2 * j) * w + 2 * i + 1];
    float f3 = in[(int64_t)(2 * j + 1) * w + 2 * i], f4 = in[(int64_t)(2 * j + 1) * w + 2 * i + 1];
    out[(int64_t)j * wo + i] = down4(f1, f2, f3, f4);
}

// measurement.cu:104-126
__device__ __forceinline__ float4 vertex_at(float d, int i, int j, const float* ki)
{
    float4 o = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
    if (is_depth_valid(d)) {
        v3 p = m3v(ki, mk3((float)i + 0.5f, (float)j + 0.5f, 1.0f));
        p = mul3s(p, d);
        o = make_float4(p.x, p.y, p.z, kValid);
    }
    return o;
}

struct Mat3 {
    float m[9];
};

__global__ __launch_bounds__(256) void vertex_kernel(const float* __restrict__ depth, float4* __restrict__ out, int w,
                                                     int h, Mat3 ki)
{
    int i = blockIdx.x * kTile + threadIdx.x, j = blockIdx.y * kTile + threadIdx.y;
    if (i >= w || j >= h) return;
    out[(int64_t)j * w + i] = vertex_at(depth[(int64_t)j * w + i], i, j, ki.m);
}

// ---- the measurement step in one launch (one session's frame without normals, whose
// 64x64 depth ranges are not asked for here: measure_one_pass_kernel), or in two (with
// normals or ranges: measure_kernel and pyramid_kernel; many sessions:
// measure_batch_kernel and pyramid_batch_kernel).  launch_measure chooses.
// The metres of the 22x22 window at (i0, j0), clamped to the image's edges.
// UNMIRROR: row j of the frame is read right to left (measurement.cu:22-25).
template <bool UNMIRROR>
__device__ __forceinline__ void fill_window(const PreJob& J, int i0, int j0, BilateralTile& tile)
{
    for (int q = threadIdx.y * kTile + threadIdx.x; q < (kTile + 6) * (kTile + 6); q += kTile * kTile) {
        const int ly = q / (kTile + 6), lx = q % (kTile + 6);
        int gi = clampi(i0 + lx, 0, J.w - 1);
        const int gj = clampi(j0 + ly, 0, J.h - 1);
        if (UNMIRROR) gi = J.w - 1 - gi;
        tile[ly][lx] = half_rne(J.raw[(int64_t)gj * J.w + gi]) * J.scale;
    }
}

// Pass 1, per level-0 16x16 tile lt of job J: raw codes -> metres in LDS (the
// fuse input is written back, with the tile's depth range when J.drange is
// set), bilateral filter, level-0 vertex map.
template <bool UNMIRROR>
__device__ __forceinline__ void measure_tile(const PreJob& J, int lt, BilateralTile& tile, float2* wave_range)
{
    const int t = threadIdx.y * kTile + threadIdx.x;
    const int i0 = (lt % J.tiles_x) * kTile - 3, j0 = (lt / J.tiles_x) * kTile - 3;
    __syncthreads();  // the previous tile's reads of the window are over
    fill_window<UNMIRROR>(J, i0, j0, tile);
    __syncthreads();
    const int i = i0 + 3 + threadIdx.x, j = j0 + 3 + threadIdx.y;
    float dv = 0.0f, dl = __int_as_float(0x7f800000);  // this pixel's part of the tile's range
    if (i < J.w && j < J.h) {
        const int64_t q = (int64_t)j * J.w + i;
        const float dm = tile[threadIdx.y + 3][threadIdx.x + 3];
        J.depth_m[q] = dm;
        dv = dl = is_depth_valid(dm) ? dm : 0.0f;
        const float d = bilateral_at(tile, threadIdx.x, threadIdx.y);
        J.d0[q] = d;
        J.v[0][q] = vertex_at(d, i, j, J.Kinv[0]);
    }
    if (!J.drange) return;
    dv = wave_max(dv);
    dl = wave_min(dl);
    if ((t & 63) == 0) wave_range[t >> 6] = make_float2(dv, dl);
    __syncthreads();
    if (t == 0) {
        const float2 a = wave_range[0], b = wave_range[1], c = wave_range[2], d = wave_range[3];
        J.drange[lt] = make_float2(fmaxf(fmaxf(a.x, b.x), fmaxf(c.x, d.x)), fminf(fminf(a.y, b.y), fminf(c.y, d.y)));
    }
}

// Pass 2 of many sessions (3 levels, no normals), one thread per level-2 pixel
// of level-2 tile lt: its 4x4 level-0 block (the frame's width is a multiple of
// 4, so each row is one 16-byte load) gives 4 level-1 depths (downSample) and
// those the level-2 depth; vertex maps of both levels.  A workgroup covers a
// 64x64 level-0 region and also writes its depth range.  Bound: HBM.
__device__ __forceinline__ void pyramid_tile(const PreJob& J, int lt)
{
    const int t = threadIdx.y * kTile + threadIdx.x;
    const int rx = lt % J.ptiles_x, ry = lt / J.ptiles_x;
    if (t < 64) region_range(J.drange, J.w, J.h, rx, ry);
    const int i2 = rx * kTile + threadIdx.x, j2 = ry * kTile + threadIdx.y;
    const int w1 = J.w >> 1, w2 = J.w >> 2;
    if (i2 >= w2 || j2 >= (J.h >> 2)) return;
    float4 r[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) r[y] = *reinterpret_cast<const float4*>(J.d0 + (int64_t)(4 * j2 + y) * J.w + 4 * i2);
    float l1[2][2];
#pragma unroll
    for (int dy = 0; dy < 2; ++dy) {
        const float4 a = r[2 * dy], b = r[2 * dy + 1];
        l1[dy][0] = down4(a.x, a.y, b.x, b.y);
        l1[dy][1] = down4(a.z, a.w, b.z, b.w);
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
            const int i1 = 2 * i2 + dx, j1 = 2 * j2 + dy;
            J.v[1][(int64_t)j1 * w1 + i1] = vertex_at(l1[dy][dx], i1, j1, J.Kinv[1]);
        }
    }
    const float d2 = down4(l1[0][0], l1[0][1], l1[1][0], l1[1][1]);
    J.v[2][(int64_t)j2 * w2 + i2] = vertex_at(d2, i2, j2, J.Kinv[2]);
}

// Pass 2 of one session, per RxR level-0 region lt: the depths of levels 1 and 2
// (downSample), their vertex maps and, when J.n is set, the normals of every
// level, all from the region's filtered depths in LDS.  A normal needs its right
// and lower neighbour (device_helper.cuh:81-110): one more column and row per
// level, so (for R = 32) 36x36 level-0 depths feed 18x18 of level 1 and 9x9 of level 2, and
// the neighbours' vertices are formed again from those depths (15 operations)
// instead of read back (48 bytes).  Depths outside the image are 0 here, which
// makes their vertices invalid as device_helper.cuh:43-50 has it.
//
// Bound: launch and memory latency.  16x16 regions give a 640x480 frame 1200
// workgroups, 32x32 ones 300, which leave the chip half idle but read less halo:
// kf_preprocess with normals by 32x32 -> 16x16 regions 484x372 16.2 -> 13.8 us, 640x480
// 19.0 -> 17.0, 800x600 24.6 -> 23.3, 1276x716 35.9 -> 35.5 (within the runs' spread),
// 1920x1080 65.5 -> 68.5: frames up to kSmallRegions pixels take 16x16, the line lying
// between the last size that gains (480000 pixels) and the one that does not (913616).  Many sessions fill the chip either
// way, and there the regions' barriers cost: 64 frames of 640x480 took 109 us by
// regions, 50 us by the form above (73 us with its depths read one by one).
constexpr int kSmallRegions = 600000;
template <int R>
struct PyramidTile {
    float d0[R + 4][R + 5];
    float d1[R / 2 + 2][R / 2 + 3];
    float d2[R / 4 + 1][R / 4 + 1];
};
template <class Row>
__device__ __forceinline__ float4 normal_from_depths(const Row& d, int x, int y, int i, int j, const float* ki)
{
    NormalStencil s;
    s.c = vertex_at(d[y][x], i, j, ki);
    s.r = vertex_at(d[y][x + 1], i + 1, j, ki);
    s.d = vertex_at(d[y + 1][x], i, j + 1, ki);
    return normal_of(s);
}

// The normals and coarser levels of the RxR region at (x0, y0), whose filtered depths
// (with the halo, when normals are asked for) are in T.d0.
template <int R>
__device__ __forceinline__ void region_levels(const PreJob& J, int x0, int y0, PyramidTile<R>& T)
{
    const int t = threadIdx.y * kTile + threadIdx.x;
    const bool normals = J.n[0] != nullptr;
    if (normals) {
#pragma unroll
        for (int q = 0; q < R * R / (kTile * kTile); ++q) {
            const int e = t + q * kTile * kTile, x = e % R, y = e / R, i = x0 + x, j = y0 + y;
            if (i < J.w && j < J.h) J.n[0][(int64_t)j * J.w + i] = normal_from_depths(T.d0, x, y, i, j, J.Kinv[0]);
        }
    }
    if (J.levels < 2) return;  // uniform
    const int w1 = J.w >> 1, h1 = J.h >> 1, e1 = R / 2 + (normals ? 2 : 0);
    for (int q = t; q < e1 * e1; q += kTile * kTile) {
        const int y = q / e1, x = q - y * e1;
        T.d1[y][x] = down4(T.d0[2 * y][2 * x], T.d0[2 * y][2 * x + 1], T.d0[2 * y + 1][2 * x], T.d0[2 * y + 1][2 * x + 1]);
    }
    __syncthreads();
    if (t < R * R / 4) {
        const int x = t % (R / 2), y = t / (R / 2), i = x0 / 2 + x, j = y0 / 2 + y;
        if (i < w1 && j < h1) {
            const int64_t q = (int64_t)j * w1 + i;
            const float d = T.d1[y][x];
            J.v[1][q] = vertex_at(d, i, j, J.Kinv[1]);
            if (J.d12[0]) J.d12[0][q] = d;
            if (normals) J.n[1][q] = normal_from_depths(T.d1, x, y, i, j, J.Kinv[1]);
        }
    }
    if (J.levels < 3) return;
    const int w2 = J.w >> 2, h2 = J.h >> 2, e2 = R / 4 + (normals ? 1 : 0);
    if (t < e2 * e2) {
        const int y = t / e2, x = t - y * e2;
        T.d2[y][x] = down4(T.d1[2 * y][2 * x], T.d1[2 * y][2 * x + 1], T.d1[2 * y + 1][2 * x], T.d1[2 * y + 1][2 * x + 1]);
    }
    __syncthreads();
    if (t < R * R / 16) {
        const int x = t % (R / 4), y = t / (R / 4), i = x0 / 4 + x, j = y0 / 4 + y;
        if (i < w2 && j < h2) {
            const int64_t q = (int64_t)j * w2 + i;
            const float d = T.d2[y][x];
            J.v[2][q] = vertex_at(d, i, j, J.Kinv[2]);
            if (J.d12[1]) J.d12[1][q] = d;
            if (normals) J.n[2][q] = normal_from_depths(T.d2, x, y, i, j, J.Kinv[2]);
        }
    }
}

template <int R>
__device__ __forceinline__ void pyramid_region(const PreJob& J, int lt, PyramidTile<R>& T)
{
    const int t = threadIdx.y * kTile + threadIdx.x;
    const int rtx = (J.w + R - 1) / R, rx = lt % rtx, ry = lt / rtx;
    const int x0 = rx * R, y0 = ry * R;
    const int e0 = R + (J.n[0] ? 4 : 0);
    for (int q = t; q < e0 * e0; q += kTile * kTile) {
        const int y = q / e0, x = q - y * e0;
        const bool in = x0 + x < J.w && y0 + y < J.h;
        T.d0[y][x] = in ? J.d0[(int64_t)(y0 + y) * J.w + (x0 + x)] : 0.0f;
    }
    constexpr int k64 = 64 / R;
    if (J.drange && rx % k64 == 0 && ry % k64 == 0 && t >= 192)
        region_range(J.drange, J.w, J.h, rx / k64, ry / k64);
    __syncthreads();
    region_levels(J, x0, y0, T);
}

// Both passes in one for a frame without normals, per 16x16 tile lt: its coarser levels
// need its own pixels only.  Two passes -> one: 160x120 8.9 -> 5.6 us, 640x480 14.4 ->
// 11.0, 1920x1080 55 -> 52.  (With normals the tile would filter their halo again:
// 160x120 9.5 us in two passes, 9.6 in one, 400x300 10.8 and 11.1, 1276x716 35 and 45.)
struct OnePassTile {
    BilateralTile window;
    PyramidTile<kTile> pyramid;
    float wave_max[4];
};
template <bool UNMIRROR>
__device__ __forceinline__ void one_pass_tile(const PreJob& J, int lt, OnePassTile& S)
{
    const int t = threadIdx.y * kTile + threadIdx.x;
    const int x0 = (lt % J.tiles_x) * kTile, y0 = (lt / J.tiles_x) * kTile;
    fill_window<UNMIRROR>(J, x0 - 3, y0 - 3, S.window);
    __syncthreads();
    const int i = x0 + threadIdx.x, j = y0 + threadIdx.y;
    const bool in = i < J.w && j < J.h;
    const float dm = S.window[threadIdx.y + 3][threadIdx.x + 3];
    const float d = in ? bilateral_at(S.window, threadIdx.x, threadIdx.y) : 0.0f;
    S.pyramid.d0[threadIdx.y][threadIdx.x] = d;
    if (in) {
        const int64_t q = (int64_t)j * J.w + i;
        J.depth_m[q] = dm;
        J.d0[q] = d;
        J.v[0][q] = vertex_at(d, i, j, J.Kinv[0]);
    }
    if (J.drange) {
        const float m = wave_max(in && is_depth_valid(dm) ? dm : 0.0f);
        if ((t & 63) == 0) S.wave_max[t >> 6] = m;
    }
    __syncthreads();
    // the max only: one session's cull does not read the min
    if (J.drange && t == 0)
        J.drange[lt] = make_float2(fmaxf(fmaxf(S.wave_max[0], S.wave_max[1]), fmaxf(S.wave_max[2], S.wave_max[3])), 0.0f);
    region_levels(J, x0, y0, S.pyramid);
}

// One session: one workgroup per tile, the job by value.
template <bool UNMIRROR>
__global__ __launch_bounds__(256) void measure_kernel(PreJob J)
{
    __shared__ BilateralTile tile;
    __shared__ float2 wave_range[4];
    measure_tile<UNMIRROR>(J, blockIdx.x, tile, wave_range);
}
template <int R>
__global__ __launch_bounds__(256) void pyramid_kernel(PreJob J)
{
    __shared__ PyramidTile<R> T;
    pyramid_region(J, blockIdx.x, T);
}
template <bool UNMIRROR>
__global__ __launch_bounds__(256) void measure_one_pass_kernel(PreJob J)
{
    __shared__ OnePassTile S;
    one_pass_tile<UNMIRROR>(J, blockIdx.x, S);
}

// Many sessions per launch (batch ticks), persistent over the tick's tiles.
// The first kernel also clears the tick's fuse-list counter and deferred-ray
// counts, which later passes of this tick use.
__global__ __launch_bounds__(256) void measure_batch_kernel(const BatchHeader* hd, const PreJob* jobs)
{
    __shared__ BilateralTile tile;
    __shared__ float2 wave_range[4];
    if (blockIdx.x == 0 && threadIdx.y == 0) {
        if (threadIdx.x == 0) *hd->fuse_count = 0u;
        hd->ray_count[threadIdx.x * kCountStride] = 0u;  // kTile == 16 deferred-ray counts
    }
    const int tiles = hd->pre_tiles, njobs = hd->n_pre;
    for (int tl = blockIdx.x; tl < tiles; tl += gridDim.x) {
        const PreJob& J = jobs[job_of(jobs, njobs, tl, [](const PreJob& x) { return x.tile0; })];
        measure_tile<false>(J, tl - J.tile0, tile, wave_range);
    }
}

__global__ __launch_bounds__(256) void pyramid_batch_kernel(const BatchHeader* hd, const PreJob* jobs)
{
    const int tiles = hd->pyr_tiles, njobs = hd->n_pre;
    for (int tl = blockIdx.x; tl < tiles; tl += gridDim.x) {
        const PreJob& J = jobs[job_of(jobs, njobs, tl, [](const PreJob& x) { return x.ptile0; })];
        pyramid_tile(J, tl - J.ptile0);
    }
}

// measurement.cu:128-135 with device_helper.cuh:81-110
__global__ __launch_bounds__(256) void normal_kernel(const float4* __restrict__ v, float4* __restrict__ out, int w,
                                                     int h)
{
    int i = blockIdx.x * kTile + threadIdx.x, j = blockIdx.y * kTile + threadIdx.y;
    if (i >= w || j >= h) return;
    out[(int64_t)j * w + i] = compute_normal(v, w, h, i, j);
}

}  // namespace

int launch_convert(const uint16_t* raw, float* out, int w, int h, float scale, int unmirror, hipStream_t s)
{
    convert_kernel<<<grid2d(w, h), dim3(kTile, kTile), 0, s>>>(raw, out, w, h, scale, unmirror);
    KF_LAUNCHED("convert_kernel");
    return KF_OK;
}
int launch_bilateral(const float* in, float* out, int w, int h, hipStream_t s)
{
    bilateral_kernel<<<grid2d(w, h), dim3(kTile, kTile), 0, s>>>(in, out, w, h);
    KF_LAUNCHED("bilateral_kernel");
    return KF_OK;
}
int launch_down_sample(const float* in, int w_in, int h_in, float* out, hipStream_t s)
{
    int wo = w_in / 2, ho = h_in / 2;
    down_sample_kernel<<<grid2d(wo, ho), dim3(kTile, kTile), 0, s>>>(in, w_in, out, wo, ho);
    KF_LAUNCHED("down_sample_kernel");
    return KF_OK;
}
int launch_vertex_map(const float* depth, float4* out, int w, int h, const float* inv_k, hipStream_t s)
{
    Mat3 ki;
    for (int q = 0; q < 9; ++q) ki.m[q] = inv_k[q];
    vertex_kernel<<<grid2d(w, h), dim3(kTile, kTile), 0, s>>>(depth, out, w, h, ki);
    KF_LAUNCHED("vertex_kernel");
    return KF_OK;
}
int launch_normal_map(const float4* v, float4* out, int w, int h, hipStream_t s)
{
    normal_kernel<<<grid2d(w, h), dim3(kTile, kTile), 0, s>>>(v, out, w, h);
    KF_LAUNCHED("normal_kernel");
    return KF_OK;
}

int launch_measure(PreJob& J, hipStream_t s)
{
    J.tiles_x = (J.w + kTile - 1) / kTile;
    const unsigned tiles = (unsigned)(J.tiles_x * ((J.h + kTile - 1) / kTile));
    if (J.levels > 1 && !J.n[0] && (!J.drange || J.late_regions)) {
        if (J.unmirror) measure_one_pass_kernel<true><<<tiles, dim3(kTile, kTile), 0, s>>>(J);
        else measure_one_pass_kernel<false><<<tiles, dim3(kTile, kTile), 0, s>>>(J);
        KF_LAUNCHED("measure_one_pass_kernel");
        return KF_OK;
    }
    if (J.unmirror) measure_kernel<true><<<tiles, dim3(kTile, kTile), 0, s>>>(J);
    else measure_kernel<false><<<tiles, dim3(kTile, kTile), 0, s>>>(J);
    KF_LAUNCHED("measure_kernel");
    // pass 2 has work for a pyramid, normals or the 64x64 depth ranges
    if (J.levels > 1 || J.n[0] || J.drange) {
        const int r = (int64_t)J.w * J.h <= kSmallRegions ? 16 : 32;
        const unsigned regions = (unsigned)(((J.w + r - 1) / r) * ((J.h + r - 1) / r));
        if (r == 16) pyramid_kernel<16><<<regions, dim3(kTile, kTile), 0, s>>>(J);
        else pyramid_kernel<32><<<regions, dim3(kTile, kTile), 0, s>>>(J);
        KF_LAUNCHED("pyramid_kernel");
    }
    return KF_OK;
}

int launch_preprocess_batch(const BatchHeader* hd, const PreJob* jobs, unsigned blocks, hipStream_t s)
{
    measure_batch_kernel<<<blocks, dim3(kTile, kTile), 0, s>>>(hd, jobs);
    KF_LAUNCHED("measure_batch_kernel");
    pyramid_batch_kernel<<<blocks, dim3(kTile, kTile), 0, s>>>(hd, jobs);
    KF_LAUNCHED("pyramid_batch_kernel");
    return KF_OK;
}

}  // namespace kf

// ------------------------------------------------------------------ C ABI
extern "C" {

int kf_convert_to_depth_meters(const uint16_t* raw, float* depth_m, int w, int h, float scale, int unmirror,
                               kf_stream_t stream, float* elapsed_ms)
{
    if (!raw || !depth_m || w <= 0 || h <= 0) return kf::fail(KF_ERR_ARG, "convertToDepthMeters: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_convert(raw, depth_m, w, h, scale, unmirror, s))) return st;
    return t.finish();
}

int kf_apply_bilateral_filter(const float* depth_m, float* filtered, int w, int h, kf_stream_t stream,
                              float* elapsed_ms)
{
    if (!depth_m || !filtered || w <= 0 || h <= 0) return kf::fail(KF_ERR_ARG, "applyBilateralFilter: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_bilateral(depth_m, filtered, w, h, s))) return st;
    return t.finish();
}

int kf_down_sample(const float* in, int w_in, int h_in, float* out, int w_out, int h_out, kf_stream_t stream,
                   float* elapsed_ms)
{
    if (!in || !out || w_out <= 0 || h_out <= 0) return kf::fail(KF_ERR_ARG, "downSample: bad argument");
    // measurement.cu:186-189
    if (w_in / w_out != 2 || h_in / h_out != 2 || w_in != 2 * w_out || h_in != 2 * h_out)
        return kf::fail(KF_ERR_DIMS, "downSample: output has to be half size of the input surface object!");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_down_sample(in, w_in, h_in, out, s))) return st;
    return t.finish();
}

int kf_create_vertex_map(const float* depth, float* vertex_map, int w, int h, const float inv_k[9],
                         kf_stream_t stream, float* elapsed_ms)
{
    if (!depth || !vertex_map || !inv_k || w <= 0 || h <= 0) return kf::fail(KF_ERR_ARG, "createVertexMap: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) ||
        (st = kf::launch_vertex_map(depth, reinterpret_cast<float4*>(vertex_map), w, h, inv_k, s)))
        return st;
    return t.finish();
}

int kf_create_normal_map(const float* vertex_map, float* normal_map, int w, int h, kf_stream_t stream,
                         float* elapsed_ms)
{
    if (!vertex_map || !normal_map || w <= 0 || h <= 0) return kf::fail(KF_ERR_ARG, "createNormalMap: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) || (st = kf::launch_normal_map(reinterpret_cast<const float4*>(vertex_map),
                                                        reinterpret_cast<float4*>(normal_map), w, h, s)))
        return st;
    return t.finish();
}

int kf_preprocess(const uint16_t* raw, int w, int h, float scale, int unmirror, int levels, const float inv_k[][9],
                  float* depth_m, float* const depth_pyr[], float* const vertex_pyr[], float* const normal_pyr[],
                  kf_stream_t stream, float* elapsed_ms)
{
    if (!raw || !depth_m || !depth_pyr || !vertex_pyr || !inv_k || levels < 1 || levels > 3 || w <= 0 || h <= 0)
        return kf::fail(KF_ERR_ARG, "kf_preprocess: bad argument");
    // grid_map_pyramid.h:63-72
    int e = 1 << (levels - 1);
    if (w % e || h % e)
        return kf::fail(KF_ERR_DIMS, "Can't construct pyramid. Dimensions must be divisible by 2^(m_n_layers - 1).");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    kf::PreJob J;
    memset(&J, 0, sizeof(J));
    J.raw = raw;
    J.depth_m = depth_m;
    J.d0 = depth_pyr[0];
    for (int l = 0; l < levels; ++l) {
        J.v[l] = reinterpret_cast<float4*>(vertex_pyr[l]);
        if (normal_pyr) J.n[l] = reinterpret_cast<float4*>(normal_pyr[l]);
        if (l > 0) J.d12[l - 1] = depth_pyr[l];
        memcpy(J.Kinv[l], inv_k[l], sizeof(J.Kinv[l]));
    }
    J.w = w;
    J.h = h;
    J.levels = levels;
    J.unmirror = unmirror;
    J.scale = scale;
    int st;
    if ((st = t.start()) || (st = kf::launch_measure(J, s))) return st;
    return t.finish();
}

}  // extern "C"
