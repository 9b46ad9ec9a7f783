// Raycaster (project/src/raycast.cu): per pixel of a pyramid level, march the
// TSDF from the sensor pose, find the zero crossing and write the world-space
// vertex and the normal (-grad F) of the surface.
//
// The reference samples the volume through a CUDA texture (normalized
// coordinates, linear filter, clamp; voxel_grid.cpp:24-33).  Here the same
// texel-centre rule is evaluated in software on the bricked f plane:
//   x = u*n - 1/2, i = floor(x), a = x - i, indices clamped to [0, n-1],
// with exact FP32 weights (the texture unit keeps 8 fractional bits).
//
// Launch: one lane per pixel, 8x8 pixel tiles per 64-lane wave (rays of a wave
// are coherent, so their trilinear stencils share bricks and cache lines);
// tiles are assigned so that neighbouring tiles run on the same XCD (the 8
// XCDs each have their own L2 and receive workgroups round-robin).
#include <string.h>

#include "kf_device.hpp"
#include "kf_kernels.hpp"

namespace kf {

namespace {

// Skipping: a sample is skipped when its stencil certainly lies in the box of
// free bricks around its brick (the free distances, kf_device.hpp): it can then
// neither end the march nor change its step.  A skipped sample only sets prev_t;
// its value is computed if and when the zero-crossing formula needs it.
//
// The test works on texel coordinates computed with a reciprocal instead of
// the exact division (a few 1e-5 voxel apart): a sample counts as inside a box
// only when its coordinate is at least kMargin voxel inside it, so its exact
// stencil is inside the box too.
constexpr float kMargin = 0.01f;

struct RaycastArgs {
    RaycastVolume vol;
    float pose[16];
    const PoseState* dyn;  // when set, the pose comes from dyn->pose
    RaycastLevel lv[3];
    int levels, tiles;
    DeferredRay* rays;  // rays handed to the finishing pass: 8 lists (XCDs) of at most cap
    unsigned* count;    // their counts for this launch, kCountStride apart
    unsigned* clear;    // the counts of the other launch parity, cleared for the next launch
    unsigned cap;
    RaycastSide side;
};


// Normalized texture coordinate x / width + 1/2 of a world coordinate, the
// quotient from the exact reciprocal (three operations; x / width in every
// bit: for an x so small that its residual underflows the sum is 1/2 either way).
__device__ __forceinline__ float tex(const RaycastVolume& a, float x)
{
    return div_by_exact_reciprocal(x, a.width, a.inv_width) + 0.5f;
}

// Approximate texel coordinate of a world coordinate for the skip tests only
// (they allow kMargin of error; this is within a few 1e-5 texel).
__device__ __forceinline__ float approx_texel(float x, float invw, float nf)
{
    return fmaf(fmaf(x, invw, 0.5f), nf, -0.5f);
}

// Texel coordinates of a trilinear sample at normalized (u, v, s):
// x = u*n - 1/2, i0 = floor(x) clamped to [0, n-1], i1 = i0 + 1 clamped.
struct Stencil {
    int i0, j0, k0, i1, j1, k1;
    float a, b, c;
};
// The floors are integers (sample positions are finite), so clamping them, and
// them plus one (exact below 2^24; beyond, both clamp to the same end), to
// [0, n-1] in float and converting gives the clamped indices: one median of
// three and a conversion per index.
__device__ __forceinline__ Stencil stencil_texel(int n, float x, float y, float z)
{
    Stencil st;
    float fx = floorf(x), fy = floorf(y), fz = floorf(z);
    st.a = x - fx;
    st.b = y - fy;
    st.c = z - fz;
    const float top = (float)(n - 1);
    st.i0 = (int)__builtin_amdgcn_fmed3f(fx, 0.0f, top);
    st.j0 = (int)__builtin_amdgcn_fmed3f(fy, 0.0f, top);
    st.k0 = (int)__builtin_amdgcn_fmed3f(fz, 0.0f, top);
    st.i1 = (int)__builtin_amdgcn_fmed3f(fx + 1.0f, 0.0f, top);
    st.j1 = (int)__builtin_amdgcn_fmed3f(fy + 1.0f, 0.0f, top);
    st.k1 = (int)__builtin_amdgcn_fmed3f(fz + 1.0f, 0.0f, top);
    return st;
}
// From normalized coordinates: x = u*n - 1/2 rounded twice; for a power-of-two
// n the product is exact, so one fused multiply-add rounds the same way (P2).
template <bool P2>
__device__ __forceinline__ Stencil stencil(int n, float u, float v, float s)
{
    const float nf = (float)n;
    if (P2) return stencil_texel(n, fmaf(u, nf, -0.5f), fmaf(v, nf, -0.5f), fmaf(s, nf, -0.5f));
    return stencil_texel(n, u * nf - 0.5f, v * nf - 0.5f, s * nf - 0.5f);
}

// Voxel q of the f plane (32-bit element offset from the plane's base).
template <int FMT>
__device__ __forceinline__ float voxel_at(const void* f, uint32_t q)
{
    const char* base = static_cast<const char*>(f);
    if (FMT == KF_VOXEL_F32) return *reinterpret_cast<const float*>(base + (size_t)(q * 4u));
    return snorm_decode(*reinterpret_cast<const int16_t*>(base + (size_t)(q * 2u)));
}

// Element offsets of the 8 corners of a stencil's cell, in the order
// c000 c100 c010 c110 c001 c101 c011 c111 (i fastest).
__device__ __forceinline__ void cell_offsets(int nb, const Stencil& t, uint32_t* o)
{
    const uint32_t x0 = brick_ox(t.i0), x1 = brick_ox(t.i1);
    const uint32_t y0 = brick_oy(nb, t.j0), y1 = brick_oy(nb, t.j1);
    const uint32_t z0 = brick_oz(nb, t.k0), z1 = brick_oz(nb, t.k1);
    const uint32_t y0z0 = y0 + z0, y1z0 = y1 + z0, y0z1 = y0 + z1, y1z1 = y1 + z1;
    o[0] = x0 + y0z0;
    o[1] = x1 + y0z0;
    o[2] = x0 + y1z0;
    o[3] = x1 + y1z0;
    o[4] = x0 + y0z1;
    o[5] = x1 + y0z1;
    o[6] = x0 + y1z1;
    o[7] = x1 + y1z1;
}

__device__ __forceinline__ float lerp_cell(const float* v, float a, float b, float c)
{
    const float e00 = (1.0f - a) * v[0] + a * v[1], e10 = (1.0f - a) * v[2] + a * v[3];
    const float e01 = (1.0f - a) * v[4] + a * v[5], e11 = (1.0f - a) * v[6] + a * v[7];
    const float g0 = (1.0f - b) * e00 + b * e10, g1 = (1.0f - b) * e01 + b * e11;
    return (1.0f - c) * g0 + c * g1;
}

template <int FMT>
__device__ __forceinline__ float trilinear(const void* F, int nb, const Stencil& t)
{
    uint32_t o[8];
    float v[8];
    cell_offsets(nb, t, o);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = voxel_at<FMT>(F, o[q]);
    return lerp_cell(v, t.a, t.b, t.c);
}

template <int FMT, bool P2>
__device__ __forceinline__ float sample_tsdf(const void* F, int n, int nb, float u, float v, float s)
{
    return trilinear<FMT>(F, nb, stencil<P2>(n, u, v, s));
}

// The ray of a march in texel space, for the skip test.
struct RaySpeed {
    float ix, iy, iz;  // large steps per texel along each axis, signed, at most 1e9
    float cap;         // most steps a run may take (see free_run)
};
__device__ __forceinline__ RaySpeed ray_speed(v3 dir, float large, float invw, float nf)
{
    // 1 / 0 is held at 1e9: such an axis never bounds a run
    const float k = invw * nf * large;
    RaySpeed r;
    r.ix = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(dir.x * k), -1e9f, 1e9f);
    r.iy = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(dir.y * k), -1e9f, 1e9f);
    r.iz = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(dir.z * k), -1e9f, 1e9f);
    // the smaller of 20000 width / n and the small steps in kMaxDistance
    r.cap = __builtin_amdgcn_rcpf(fmaxf(invw * nf * (1.0f / 20000.0f), large * (1.0f / (20.0f * kMaxDistance))));
    return r;
}

// The brick of a sample from its approximate texel coordinates: its index and
// its centre plane coordinates (8 b + 4) per axis.
struct BrickAt {
    int index;
    float cx, cy, cz;
};
__device__ __forceinline__ BrickAt brick_at(const RaycastVolume& a, float xa, float ya, float za)
{
    const int top = a.n - 1;
    const int x = clampi((int)xa, 0, top), y = clampi((int)ya, 0, top), z = clampi((int)za, 0, top);
    BrickAt b;
    b.index = grid_index(x >> 3, y >> 3, z >> 3, a.nb);
    b.cx = (float)((x & ~7) | 4);
    b.cy = (float)((y & ~7) | 4);
    b.cz = (float)((z & ~7) | 4);
    return b;
}

// Half the side of the box of free bricks around a brick of distance D, less
// 2 kMargin; negative for D = 0 (no sample is inside).
__device__ __forceinline__ float free_extent(int D) { return (float)(8 * D) - (4.0f + 2.0f * kMargin); }

__device__ __forceinline__ bool inside_box(const BrickAt& b, float xa, float ya, float za, float E)
{
    return fmaxf(fmaxf(fabsf(xa - b.cx), fabsf(ya - b.cy)), fabsf(za - b.cz)) <= E;
}

// Steps after a sample inside the box (scale: large steps 1, small steps
// large / small) whose samples certainly stay in it.  The march's approximate
// texel coordinates are linear in t up to rounding: t stays below 6 m, so each
// addition is off by at most 2^-22 m, and k of them by k * 2^-22 m * (texels
// per metre); the cap keeps k below kMargin / 2 of that.  (It also keeps k below
// the small steps in the march's whole range: where a voxel is much longer than a
// step, a run would otherwise go on long after the march has ended; an empty 128^3
// volume of 1000 m drawn at 640x480 265 -> 71 us.)  The reciprocals' relative error
// of a few 1e-7 on at most 140 texels moves the last counted sample by under 1e-4
// texel.  So a counted sample, 2 kMargin inside the box by the linear form, has a
// computed coordinate kMargin inside it.
__device__ __forceinline__ int free_run(const BrickAt& b, float xa, float ya, float za, float E, const RaySpeed& r,
                                        float scale)
{
    const float kx = fmaf(b.cx - xa, r.ix, E * fabsf(r.ix));
    const float ky = fmaf(b.cy - ya, r.iy, E * fabsf(r.iy));
    const float kz = fmaf(b.cz - za, r.iz, E * fabsf(r.iz));
    return (int)fminf(fminf(fminf(kx, ky), kz) * scale, r.cap);
}

// A lane takes at most this many trips in the large-step part of its march and
// in the small-step part (a trip skips a run of samples or evaluates one); a
// longer ray (about 1 in 40 grazes a surface and takes hundreds of small steps)
// is appended to a list that a second pass finishes with a whole wave per ray,
// so no wave of the first pass waits on one long ray.  The single-session
// pass's tail bounds the frame; the batch's persistent pass is throughput-bound.
// Small trips, first + finishing pass: one 640x480 frame (three levels) into 512^3
// FP32 12 59 + 15 us, 14 62 + 11, 16 65 + 10, into 256^3 snorm16 53 + 32, 57 + 27,
// 60 + 22, 8 of either 50 + 100 and more; 64 frames in a tick 16 2.11 + 0.41 ms, 20
// 2.18 + 0.37, 24 2.22 + 0.33, 28 2.31 + 0.30.  Large trips: 16 to 32 alike, but 16
// gives the batch's finishing pass 0.1 ms more.
constexpr int kLargeTrips = 24;
constexpr int kSmallTrips = 14;
constexpr int kBatchSmallTrips = 20;

__device__ __forceinline__ float lane_bcast(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Camera ray of pixel (i, j) and its march interval (raycast.cu:7-27, 44-73).
struct RayGeom {
    v3 o, dir;
    float nearv, farv;
    bool active;  // false: the pixel is left untouched (raycast.cu:61-73)
};
__device__ __forceinline__ RayGeom ray_geom(const RaycastVolume& a, const float* pose, const RaycastLevel& L, int i,
                                            int j, bool in_image)
{
    float Rm[9] = {pose[0], pose[1], pose[2], pose[4], pose[5], pose[6], pose[8], pose[9], pose[10]};
    float M[9];
    m3m3(Rm, L.Kinv, M);
    RayGeom g;
    g.o = mk3(pose[12], pose[13], pose[14]);
    const float hw = a.width * 0.5f;
    g.dir = m3v(M, mk3((float)i + 0.5f, (float)j + 0.5f, 1.0f));
    const v3 inv = mk3(1.0f / g.dir.x, 1.0f / g.dir.y, 1.0f / g.dir.z);
    float t0x = (-hw - g.o.x) * inv.x, t1x = (hw - g.o.x) * inv.x;
    float t0y = (-hw - g.o.y) * inv.y, t1y = (hw - g.o.y) * inv.y;
    float t0z = (-hw - g.o.z) * inv.z, t1z = (hw - g.o.z) * inv.z;
    float tmin = fminf(t0x, t1x), tmax = fmaxf(t0x, t1x);
    tmin = fmaxf(tmin, fminf(t0y, t1y));
    tmax = fminf(tmax, fmaxf(t0y, t1y));
    tmin = fmaxf(tmin, fminf(t0z, t1z));
    tmax = fminf(tmax, fmaxf(t0z, t1z));
    if (tmax < tmin) {
        tmin = -1.0f;
        tmax = -1.0f;
    }
    g.nearv = (kMinDistance < tmin) ? tmin : kMinDistance;
    g.farv = (tmax < kMaxDistance) ? tmax : kMaxDistance;
    g.active = in_image && !(tmax < 0.0f) && g.nearv < g.farv;
    return g;
}

// raycast.cu:29-42 and 119-145: the surface point at tstar (tstar == 0: no
// crossing) and its normal -grad F, written by one lane.  The 6 gradient
// samples' corner loads are issued together; x + 0 == x, so the samples are
// those of raycast.cu:33-38.
template <int FMT, bool P2>
__device__ __forceinline__ void write_surface(const RaycastVolume& a, const RaycastLevel& L, int i, int j,
                                              const RayGeom& g, float tstar)
{
    const int64_t q = (int64_t)j * L.w + i;
    if (tstar != 0.0f) {
        const float width = a.width;
        const v3 vtx = add3(g.o, mul3s(g.dir, tstar));
        const float r = a.mue * 0.5f / width;
        const float u = tex(a, vtx.x), v = tex(a, vtx.y), s = tex(a, vtx.z);
        // the 48 corner loads of the 6 samples are issued together (one round trip)
        const float gx = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u - r, v, s) - sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u + r, v, s);
        const float gy = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u, v - r, s) - sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u, v + r, s);
        const float gz = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u, v, s - r) - sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u, v, s + r);
        const v3 gg = div3s(mk3(gx, gy, gz), r);
        const float gn = len3(gg);
        if (is_depth_valid(gn)) {
            const v3 nn = div3s(gg, gn);
            L.vout[q] = make_float4(vtx.x, vtx.y, vtx.z, kValid);
            L.nout[q] = make_float4(nn.x, nn.y, nn.z, kValid);
            return;
        }
    }
    L.vout[q] = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
    L.nout[q] = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
}

// The same, with the 6 gradient samples taken by lanes 0-5 of the wave and the
// result written by lane 0 (the finishing pass: one ray per wave).
template <int FMT, bool P2>
__device__ __forceinline__ void write_surface_wave(const RaycastVolume& a, const RaycastLevel& L, int i, int j,
                                                   const RayGeom& g, float tstar)
{
    const int lane = threadIdx.x & 63;
    const int64_t q = (int64_t)j * L.w + i;
    if (tstar != 0.0f) {
        const float width = a.width;
        const v3 vtx = add3(g.o, mul3s(g.dir, tstar));
        const float r = a.mue * 0.5f / width;
        const float u = tex(a, vtx.x), v = tex(a, vtx.y), s = tex(a, vtx.z);
        float val = 0.0f;
        if (lane < 6) {
            const int ax = lane >> 1;
            const float du = ax == 0 ? r : 0.0f, dv = ax == 1 ? r : 0.0f, ds = ax == 2 ? r : 0.0f;
            if (lane & 1) val = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u - du, v - dv, s - ds);
            else val = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, u + du, v + dv, s + ds);
        }
        const float gx = lane_bcast(val, 1) - lane_bcast(val, 0);
        const float gy = lane_bcast(val, 3) - lane_bcast(val, 2);
        const float gz = lane_bcast(val, 5) - lane_bcast(val, 4);
        const v3 gg = div3s(mk3(gx, gy, gz), r);
        const float gn = len3(gg);
        if (is_depth_valid(gn)) {
            if (lane == 0) {
                const v3 nn = div3s(gg, gn);
                L.vout[q] = make_float4(vtx.x, vtx.y, vtx.z, kValid);
                L.nout[q] = make_float4(nn.x, nn.y, nn.z, kValid);
            }
            return;
        }
    }
    if (lane == 0) {
        L.vout[q] = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
        L.nout[q] = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
    }
}

// Where the first pass appends the rays it hands over.
struct RayQueue {
    DeferredRay* rays;
    unsigned* count;
    unsigned cap;
    int small_trips;  // small-step trips of a lane before it may hand its ray over
};

// t and prev_t after the sample at t and `run` more samples have been skipped,
// by the march's own repeated additions.
__device__ __forceinline__ void advance(float& t, float& prev_t, float step, int run)
{
    for (int k = 0; k < run; ++k) t = t + step;
    prev_t = t;
    t = t + step;
}

// raycast.cu:44-145 for pixel (i, j) of one level map, one lane per pixel,
// called by all 64 lanes of a wave together (in_image false past the map's
// edge).  The march takes large steps up to the first sample below 0.99, and
// small ones from there on, so it is two loops, each with the code of its step
// only.  A ray still marching after its trips is appended to rq with its exact
// march state and left to the finishing pass (when rq is full it marches on
// here); the lanes of a wave take their slots with one atomic (per-lane
// atomics on the launch's single counter serialise).
//
// Bound: the vector ALU and, in a launch that does not fill the chip, the
// chain of dependent reads of the longest ray.  With one loop for both steps and
// a skip test on one brick or one 64^3 super-brick at a time a lane took 20 trips
// of both steps' code; the boxes of free bricks leave 8 large-step and 7
// small-step ones.  First + finishing pass: 64 frames of 640x480 from 512^3
// snorm16 volumes 3.98 + 0.45 -> 3.14 + 0.28 ms, one frame from 512^3 FP32 105 + 22
// -> 86 + 17 us, its coarsest level alone (160x120) 52 -> 30 us.  Lists per XCD
// instead of one for the launch (their counters in lines of their own): 66 + 11 us,
// and 2.36 + 0.27 ms (raycast_batch_kernel).  Small steps that enter a cell load its
// corners along with the brick's distance, one round trip instead of two: 320x240
// from 200^3 40 -> 37 us, 640x480 from 256^3 61 -> 60 us, 64 frames 2.24 -> 2.19 ms.
template <int FMT, bool P2>
__device__ __forceinline__ void raycast_pixel(const RaycastVolume& a, const float* pose, const RaycastLevel& L, int i,
                                              int j, bool in_image, const RayQueue& rq, int job)
{
    const RayGeom g = ray_geom(a, pose, L, i, j, in_image);
    const v3 o = g.o, dir = g.dir;
    const float width = a.width, mue = a.mue;
    const float large = mue * 1.99f, small = mue * 0.1f;
    const float invw = 1.0f / width, nf = (float)a.n;
    const RaySpeed speed = ray_speed(dir, large, invw, nf);
    float t = g.nearv, prev = 0.0f, prev_t = 0.0f, fhit = 0.0f;
    bool prev_skipped = false, hit = false, can_defer = true;
    enum { kLarge, kSmall, kDone, kHandedOver };
    int phase = g.active ? kLarge : kDone;
    for (;;) {
        bool defer = false;
        int trips = 0;
        while (phase == kLarge) {
            if (!(t < g.farv)) {
                phase = kDone;
                break;
            }
            if (++trips > kLargeTrips && can_defer) {
                defer = true;
                break;
            }
            const v3 p = add3(o, mul3s(dir, t));
            const float xa = approx_texel(p.x, invw, nf), ya = approx_texel(p.y, invw, nf),
                        za = approx_texel(p.z, invw, nf);
            const BrickAt b = brick_at(a, xa, ya, za);
            const float E = free_extent(a.dist[b.index] & 15);
            if (inside_box(b, xa, ya, za, E)) {
                prev_skipped = true;
                advance(t, prev_t, large, free_run(b, xa, ya, za, E, speed, 1.0f));
                continue;
            }
            const float f = trilinear<FMT>(
                a.f, a.nb, P2 ? stencil_texel(a.n, xa, ya, za) : stencil<false>(a.n, tex(a, p.x), tex(a, p.y), tex(a, p.z)));
            if (f < 0.0f) {
                if (t == g.nearv) {
                    phase = kDone;
                    break;
                }
                t = t - mue;  // back off and march on with small steps
                t = t + small;
                phase = kSmall;
                break;
            }
            prev = f;
            prev_skipped = false;
            if (f < 0.99f) {
                t = t + small;
                phase = kSmall;
                break;
            }
            t = t + large;
        }
        trips = 0;
        // the corner values of the last cell (small steps often stay in one)
        float fi = -1e9f, fj = -1e9f, fk = -1e9f, c[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        while (phase == kSmall && !defer) {
            if (!(t < g.farv)) {
                phase = kDone;
                break;
            }
            if (++trips > rq.small_trips && can_defer) {
                defer = true;
                break;
            }
            const v3 p = add3(o, mul3s(dir, t));
            const float xa = approx_texel(p.x, invw, nf), ya = approx_texel(p.y, invw, nf),
                        za = approx_texel(p.z, invw, nf);
            const float x = P2 ? xa : tex(a, p.x) * nf - 0.5f, y = P2 ? ya : tex(a, p.y) * nf - 0.5f,
                        z = P2 ? za : tex(a, p.z) * nf - 0.5f;
            const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
            if (fx != fi || fy != fj || fz != fk) {
                // the corners and the brick's distance in one round trip: near a surface few
                // samples are free
                const BrickAt b = brick_at(a, xa, ya, za);
                const int dist = a.dist[b.index];
                fi = fx;
                fj = fy;
                fk = fz;
                uint32_t q[8];
                cell_offsets(a.nb, stencil_texel(a.n, x, y, z), q);
#pragma unroll
                for (int k = 0; k < 8; ++k) c[k] = voxel_at<FMT>(a.f, q[k]);
                const float E = free_extent(dist >> 4);
                if (inside_box(b, xa, ya, za, E)) {
                    prev_skipped = true;
                    advance(t, prev_t, small, free_run(b, xa, ya, za, E, speed, 19.9f));
                    continue;
                }
            }
            const float f = lerp_cell(c, x - fx, y - fy, z - fz);
            if (f < 0.0f) {
                hit = t != g.nearv;
                fhit = f;
                phase = kDone;
                break;
            }
            prev = f;
            prev_skipped = false;
            t = t + small;
        }
        const uint64_t dm = __ballot(defer);
        if (!dm) break;
        const int leader = __ffsll((unsigned long long)dm) - 1;
        unsigned base = 0u;
        if ((int)(threadIdx.x & 63) == leader) base = atomicAdd(rq.count, (unsigned)__popcll(dm));
        base = (unsigned)__builtin_amdgcn_readlane((int)base, leader);
        const unsigned slot = base + (unsigned)__popcll(dm & ((1ull << (threadIdx.x & 63)) - 1ull));
        if (defer && slot < rq.cap) {
            DeferredRay d;
            d.job = job;
            d.px = j * L.w + i;
            d.flags = (prev_skipped ? 1 : 0) | (phase == kSmall ? 2 : 0);
            d.t = t;
            d.prev = prev;
            d.prev_t = prev_t;
            d.pad[0] = d.pad[1] = 0.0f;
            rq.rays[slot] = d;
            phase = kHandedOver;
        } else if (defer) {
            can_defer = false;
        }
        if (!__ballot(phase == kLarge || phase == kSmall)) break;
    }
    if (!g.active || phase == kHandedOver) return;
    float tstar = 0.0f;
    if (hit) {
        if (prev_skipped) {
            const v3 pp = add3(o, mul3s(dir, prev_t));
            prev = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, tex(a, pp.x), tex(a, pp.y), tex(a, pp.z));
        }
        tstar = t - small * prev / (fhit - prev);
    }
    write_surface<FMT, P2>(a, L, i, j, g, tstar);
}

// Position of sample `lane` of a chunk of 64: t_0 = t and t_{k+1} = t_k + step,
// one rounded addition per sample as the march takes them.  The additions form
// a chain, but inside one binade of t they nearly always add the same rounded
// increment: each lane guesses t_{k-1} on the line t_b + (k - 1 - b) d through
// an exact t_b, takes one rounded step from the guess, and checks that the
// result is the line's next point (so the next lane's guess is exact).  The
// first lane whose check fails still got the exact value (its own guess was
// exact) and becomes the next t_b.  By induction every lane ends with the
// chained value; a chunk takes one pass per change of the increment (a binade
// crossing, the settling of a rounding tie) instead of 63 dependent additions.
__device__ __forceinline__ float chunk_position(float t, float step, int lane)
{
    float res = t;
    int b = 0;
    float tb = t;
    for (;;) {
        const float d = (tb + step) - tb;
        const float c = fmaf((float)(lane - b - 1), d, tb);  // t_{lane-1} when the guesses so far held
        const float tk = c + step;
        const bool on = tk == fmaf((float)(lane - b), d, tb);
        if (lane > b) res = tk;
        const uint64_t off = __ballot(lane > b && !on);
        if (!off) break;
        b = __ffsll((unsigned long long)off) - 1;
        tb = lane_bcast(res, b);
    }
    return res;
}

// The finishing pass for one handed-over ray: the wave marches it 64 samples
// at a time, lane k taking sample k of the chunk (its position by the same
// repeated additions t = t + step, chunk_position), and a ballot finds the first sample that
// ends the ray or changes the march (end of the interval, f < 0,
// or f < 0.99 on a large step).  The samples before it are consumed as the
// single-lane march would (prev from the last of them), the ones after it are
// discarded, so every sample position, value and decision is the sequential
// march's and the output is the same.
template <int FMT, bool P2>
__device__ __forceinline__ void finish_ray(const RaycastVolume& a, const float* pose, const RaycastLevel& L,
                                           const DeferredRay& r)
{
    const int lane = threadIdx.x & 63;
    const int i = r.px % L.w, j = r.px / L.w;
    const RayGeom g = ray_geom(a, pose, L, i, j, true);
    const float width = a.width, mue = a.mue;
    const float large = mue * 1.99f, small = mue * 0.1f;
    const float invw = 1.0f / width, nf = (float)a.n;
    float step = (r.flags & 2) ? small : large;
    float t = r.t, pv = r.prev, pt = r.prev_t;
    bool psk = (r.flags & 1) != 0;
    float tstar = 0.0f;
    for (;;) {
        const float tk = chunk_position(t, step, lane);
        const bool end = !(tk < g.farv);
        float f = 0.0f;
        int sk = 1;
        if (!end) {
            const v3 p = add3(g.o, mul3s(g.dir, tk));
            const float xa = approx_texel(p.x, invw, nf), ya = approx_texel(p.y, invw, nf),
                        za = approx_texel(p.z, invw, nf);
            const BrickAt b = brick_at(a, xa, ya, za);
            const int d = a.dist[b.index];
            sk = inside_box(b, xa, ya, za, free_extent(step == large ? d & 15 : d >> 4)) ? 1 : 0;
            if (!sk)
                f = trilinear<FMT>(a.f, a.nb, P2 ? stencil_texel(a.n, xa, ya, za)
                                                 : stencil<false>(a.n, tex(a, p.x), tex(a, p.y), tex(a, p.z)));
        }
        const bool neg = !end && !sk && f < 0.0f;
        const bool slow = !end && !sk && step == large && f < 0.99f;
        const uint64_t evm = __ballot(end || neg || slow);
        const int k = evm ? __ffsll((unsigned long long)evm) - 1 : 64;
        if (k > 0) {
            // sample k - 1 is the last one consumed: it sets prev
            if (__builtin_amdgcn_readlane(sk, k - 1)) {
                psk = true;
                pt = lane_bcast(tk, k - 1);
            } else {
                psk = false;
                pv = lane_bcast(f, k - 1);
            }
        }
        if (k == 64) {
            t = lane_bcast(tk, 63) + step;
            continue;
        }
        const float tkk = lane_bcast(tk, k), fk = lane_bcast(f, k);
        if (__builtin_amdgcn_readlane(end ? 1 : 0, k)) break;
        if (__builtin_amdgcn_readlane(neg ? 1 : 0, k)) {
            if (tkk == g.nearv) break;
            if (step == large) {
                t = tkk - mue;  // back off and march on with small steps
                step = small;
                t = t + step;
                continue;
            }
            float pk = pv;
            if (psk) {
                const v3 pp = add3(g.o, mul3s(g.dir, pt));
                pk = sample_tsdf<FMT, P2>(a.f, a.n, a.nb, tex(a, pp.x), tex(a, pp.y), tex(a, pp.z));
            }
            tstar = tkk - step * pk / (fk - pk);
            break;
        }
        // a large step found f < 0.99: small steps from the next sample on
        step = small;
        pv = fk;
        psk = false;
        t = tkk + step;
    }
    write_surface_wave<FMT, P2>(a, L, i, j, g, tstar);
}

// Workgroups of the first pass per level: its tile count rounded up to 8.
__host__ __device__ __forceinline__ int level_blocks(const RaycastArgs& a, int l)
{
    const int n = (l + 1 < a.levels ? a.lv[l + 1].tile0 : a.tiles) - a.lv[l].tile0;
    return (n + 7) & ~7;
}

// Dispatch order of the first pass: the coarsest level first (a tile of a
// coarse level covers more of the scene and its waves march longest; started
// last they made the kernel's tail), each level's tiles in 8 XCD-contiguous
// bands (workgroup g runs on XCD g % 8), so every XCD gets its share of every
// level.  Starting the tiles that marched longest in the previous launch first
// (recorded with an atomic per wave) gains nothing any more: most waves of a
// frame are resident at once, and it cost 1-2 % of the frame's raycasts.
// At least five waves per SIMD: the FP32 form compiles to 68 VGPRs (seven waves, no spill).
// A bound of eight (64 VGPRs, 20 bytes of spill per lane) made the three-level raycast 4 %
// slower.
template <int FMT>
__global__ __launch_bounds__(64, 5) void raycast_kernel(RaycastArgs a)
{
    if (blockIdx.x == 0 && threadIdx.x < 8) a.clear[threadIdx.x * kCountStride] = 0u;
    int g = blockIdx.x, l = a.levels - 1;
    for (; l >= 0; --l) {
        const int n8 = level_blocks(a, l);
        if (g < n8) break;
        g -= n8;
    }
    if (l < 0) return;
    const int x = g % 8, lt = x * (level_blocks(a, l) / 8) + g / 8;
    if (lt >= (l + 1 < a.levels ? a.lv[l + 1].tile0 : a.tiles) - a.lv[l].tile0) return;
    const RaycastLevel& L = a.lv[l];
    const int i = (lt % L.tiles_x) * 8 + (threadIdx.x & 7);
    const int j = (lt / L.tiles_x) * 8 + (threadIdx.x >> 3);
    const RayQueue rq{a.rays + (size_t)x * a.cap, a.count + x * kCountStride, a.cap, kSmallTrips};
    const float* pose = a.dyn ? a.dyn->pose : a.pose;
    if (a.vol.p2) raycast_pixel<FMT, true>(a.vol, pose, L, i, j, i < L.w && j < L.h, rq, l);
    else raycast_pixel<FMT, false>(a.vol, pose, L, i, j, i < L.w && j < L.h, rq, l);
}

// Waves of the finishing pass; each takes every kFinishWaves-th handed-over
// ray.  The batch's pass (hundreds of thousands of rays per tick) takes every
// kBatchFinishWaves-th: the rays' lengths vary, and the finer split shortens
// the tail (per 64-session tick, one wave per workgroup: 0.69 ms at 8192
// waves, 0.60 at 16384, 0.56 at 32768, 0.54 at 65536).  A single frame's few
// thousand rays gain nothing from more than 8192.  The waves are independent
// (no LDS, no barrier) and go kFinishPer to a workgroup: fewer workgroups to
// dispatch took the batch's pass from 0.54 to 0.51 ms (8 per workgroup gave
// 0.55, 16 gave 0.66 and slowed the single-frame pass).
constexpr unsigned kFinishWaves = 8192;
constexpr unsigned kBatchFinishWaves = 65536;
constexpr unsigned kFinishPer = 4;

// The 8 lists of a launch as one: ray r is number r - start of list x.  Every
// wave takes its rays from all lists alike, since a band of the image where the
// rays graze the floor hands over many times the rays of another (each XCD's waves
// on their own XCD's list: 16 instead of 11 us, 340 instead of 260 us in a tick of
// 64 sessions).  The counts are read through the constant address space (scalar
// loads; nothing writes them while a finishing pass runs).
struct RayLists {
    unsigned end[8];  // end[x]: rays of lists 0..x
};
__device__ __forceinline__ RayLists ray_lists(const unsigned* count, unsigned cap)
{
    typedef __attribute__((address_space(4))) const unsigned ConstCount;
    RayLists r;
    unsigned sum = 0;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
        const unsigned n = ((ConstCount*)count)[x * kCountStride];
        sum += n < cap ? n : cap;
        r.end[x] = sum;
    }
    return r;
}
__device__ __forceinline__ size_t ray_slot(const RayLists& l, unsigned cap, unsigned r)
{
    unsigned x = 0, start = 0;
#pragma unroll
    for (int q = 0; q < 7; ++q)
        if (r >= l.end[q]) {
            x = q + 1;
            start = l.end[q];
        }
    return (size_t)x * cap + (r - start);
}

template <int FMT>
__global__ __launch_bounds__(64 * kFinishPer) void raycast_finish_kernel(RaycastArgs a)
{
    typedef __attribute__((address_space(4))) const DeferredRay ConstRay;
    const RayLists lists = ray_lists(a.count, a.cap);
    const float* pose = a.dyn ? a.dyn->pose : a.pose;
    const unsigned w0 = blockIdx.x * kFinishPer + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.side.begin) {  // the last waves
        const unsigned waves = gridDim.x * kFinishPer, back = waves - 1 - w0;
        const unsigned rx = (unsigned)(a.side.w + 63) / 64, ry = (unsigned)(a.side.h + 63) / 64;
        if (back == 0) icp_begin_state(a.side.begin, a.side.carry, a.side.begin->pose);
        for (unsigned r = back; r < rx * ry; r += waves)
            region_range(a.side.drange, a.side.w, a.side.h, (int)(r % rx), (int)(r / rx));
    }
    for (unsigned r = w0; r < lists.end[7]; r += gridDim.x * kFinishPer) {
        ConstRay& cr = ((ConstRay*)a.rays)[ray_slot(lists, a.cap, r)];
        DeferredRay d;
        d.job = cr.job;
        d.px = cr.px;
        d.flags = cr.flags;
        d.t = cr.t;
        d.prev = cr.prev;
        d.prev_t = cr.prev_t;
        if (a.vol.p2) finish_ray<FMT, true>(a.vol, pose, a.lv[d.job], d);
        else finish_ray<FMT, false>(a.vol, pose, a.lv[d.job], d);
    }
}

// The handed-over rays of format FMT's tiles on XCD x.
template <int FMT, class Header>
__device__ __forceinline__ RayQueue ray_queue(const Header& hd, int x)
{
    const int k = (FMT == KF_VOXEL_F32 ? 0 : 8) + x;
    return RayQueue{hd.ray_list + (size_t)k * hd.ray_list_cap, hd.ray_count + k * kCountStride, hd.ray_list_cap,
                    kBatchSmallTrips};
}

// Field-wise copy of a job read through the constant address space.
template <class CJ>
__device__ __forceinline__ void copy_job(const CJ& j, RaycastVolume& vol, RaycastLevel& L)
{
    vol.f = j.vol.f;
    vol.dist = j.vol.dist;
    vol.n = j.vol.n;
    vol.nb = j.vol.nb;
    vol.format = j.vol.format;
    vol.width = j.vol.width;
    vol.mue = j.vol.mue;
    vol.inv_width = j.vol.inv_width;
    vol.p2 = j.vol.p2;
#pragma unroll
    for (int q = 0; q < 9; ++q) L.Kinv[q] = j.L.Kinv[q];
    L.vout = j.L.vout;
    L.nout = j.L.nout;
    L.w = j.L.w;
    L.h = j.L.h;
    L.tiles_x = j.L.tiles_x;
    L.tile0 = j.L.tile0;
}

// Many sessions and levels per launch, one launch per voxel format: the jobs of
// format FMT are jobs[j0, j1), their tiles padded to multiples of 8 and numbered
// [t0, t1) (jobs[k] has [jobs[k].L.tile0, jobs[k+1].L.tile0)).  As in
// raycast_kernel each job's tiles are cut into 8 bands, one per XCD, so every XCD
// gets its share of every job and keeps a part of each volume in its L2;
// workgroups on XCD x take the tiles of its bands in turn.
//
// March lengths vary by an order of magnitude between tiles, so a workgroup takes
// few of them and the hardware's dispatch levels the load.  Waves that claimed
// pairs of tiles from counters instead were bound by those: returning atomics of
// the whole device on one 128-byte line complete one in 11 ns, and 8192 waves
// that each look for work in all 8 bands make 65536 of them (0.74 ms) before a
// launch of any size ends.  First pass, claimed -> dispatched: 64 sessions of
// 640x480 from 512^3 snorm16 volumes 2.91 -> 2.36 ms, 16 uneven sessions 1.07 ->
// 0.39; the tick of 64 with 16384, 32768, 65536 workgroups 7.94, 7.71, 7.64 ms.
template <int FMT>
__global__ __launch_bounds__(64) void raycast_batch_kernel(const BatchHeader* hd, const RaycastJob* jobs)
{
    const int x = (int)(blockIdx.x & 7);
    const int nf = hd->n_ray_f32, tf = hd->ray_tiles_f32;
    const int j0 = FMT == KF_VOXEL_F32 ? 0 : nf, j1 = FMT == KF_VOXEL_F32 ? nf : hd->n_ray;
    const int t0 = FMT == KF_VOXEL_F32 ? 0 : tf, t1 = FMT == KF_VOXEL_F32 ? tf : hd->ray_tiles;
    const RayQueue rq = ray_queue<FMT>(*hd, x);
    // The table is read through the constant address space: it is never written
    // while the kernel runs, so its fields load with scalar loads into scalar
    // registers even after the kernel's stores (the vertex and normal maps).
    typedef __attribute__((address_space(4))) const RaycastJob ConstJob;
    ConstJob* cj = (ConstJob*)jobs;
    for (int t = t0 + (int)(blockIdx.x & ~7u); t < t1; t += (int)gridDim.x) {
        int lo = j0, hi = j1 - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (cj[mid].L.tile0 <= t) lo = mid;
            else hi = mid - 1;
        }
        const int jb = __builtin_amdgcn_readfirstlane(lo);
        RaycastVolume vol;
        RaycastLevel L;
        copy_job(cj[jb], vol, L);
        const float* pose = cj[jb].pose;
        const int tiles = L.tiles_x * ((L.h + 7) / 8);
        const int lt = x * ((tiles + 7) / 8) + (t - L.tile0) / 8;
        if (lt >= tiles) continue;  // padding of the last bands
        const int i = (lt % L.tiles_x) * 8 + (threadIdx.x & 7);
        const int j = (lt / L.tiles_x) * 8 + (threadIdx.x >> 3);
        if (vol.p2) raycast_pixel<FMT, true>(vol, pose, L, i, j, i < L.w && j < L.h, rq, jb);
        else raycast_pixel<FMT, false>(vol, pose, L, i, j, i < L.w && j < L.h, rq, jb);
    }
}

// The finishing pass of one voxel format over the rays its first pass handed
// over (each record names its job).
template <int FMT>
__global__ __launch_bounds__(64 * kFinishPer) void raycast_batch_finish_kernel(const BatchHeader* hd,
                                                                               const RaycastJob* jobs)
{
    typedef __attribute__((address_space(4))) const RaycastJob ConstJob;
    typedef __attribute__((address_space(4))) const BatchHeader ConstHeader;
    typedef __attribute__((address_space(4))) const DeferredRay ConstRay;
    ConstJob* cj = (ConstJob*)jobs;
    const RayQueue rq = ray_queue<FMT>(*(ConstHeader*)hd, 0);
    const RayLists lists = ray_lists(rq.count, rq.cap);
    ConstRay* rays = (ConstRay*)rq.rays;
    const unsigned w0 = blockIdx.x * kFinishPer + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (unsigned r = w0; r < lists.end[7]; r += gridDim.x * kFinishPer) {
        const size_t k = ray_slot(lists, rq.cap, r);
        DeferredRay d;
        d.job = rays[k].job;
        d.px = rays[k].px;
        d.flags = rays[k].flags;
        d.t = rays[k].t;
        d.prev = rays[k].prev;
        d.prev_t = rays[k].prev_t;
        RaycastVolume vol;
        RaycastLevel L;
        copy_job(cj[d.job], vol, L);
        if (vol.p2) finish_ray<FMT, true>(vol, cj[d.job].pose, L, d);
        else finish_ray<FMT, false>(vol, cj[d.job].pose, L, d);
    }
}

}  // namespace

RaycastVolume raycast_volume(const kf_volume* v)
{
    RaycastVolume r{};
    r.f = v->f;
    r.dist = v->dist;
    r.n = v->n;
    r.nb = v->nb;
    r.format = v->format;
    r.width = v->width;
    r.mue = v->mue;
    int e = 0;
    r.inv_width = 1.0f / v->width;
    r.p2 = frexpf(v->width, &e) == 0.5f && (v->n & (v->n - 1)) == 0 ? 1 : 0;
    return r;
}

// The two voxel formats use disjoint ray lists and maps, so both first passes run
// before both finishing passes.  A format without workgroups is not launched.
int launch_raycast_batch(const BatchHeader* hd, const RaycastJob* jobs, const unsigned blocks[2], hipStream_t s,
                         hipEvent_t mid)
{
    if (blocks[0]) {
        raycast_batch_kernel<KF_VOXEL_F32><<<blocks[0], 64, 0, s>>>(hd, jobs);
        KF_LAUNCHED("raycast_batch_kernel");
    }
    if (blocks[1]) {
        raycast_batch_kernel<KF_VOXEL_SNORM16_U8><<<blocks[1], 64, 0, s>>>(hd, jobs);
        KF_LAUNCHED("raycast_batch_kernel");
    }
    if (mid) KF_HIP(hipEventRecord(mid, s));
    constexpr unsigned finish = kBatchFinishWaves / kFinishPer;
    if (blocks[0]) {
        raycast_batch_finish_kernel<KF_VOXEL_F32><<<finish, 64 * kFinishPer, 0, s>>>(hd, jobs);
        KF_LAUNCHED("raycast_batch_finish_kernel");
    }
    if (blocks[1]) {
        raycast_batch_finish_kernel<KF_VOXEL_SNORM16_U8><<<finish, 64 * kFinishPer, 0, s>>>(hd, jobs);
        KF_LAUNCHED("raycast_batch_finish_kernel");
    }
    return KF_OK;
}

// The volume's deferred-ray list, grown to hold every ray of a launch of
// `rays` rays (grown outside the stream order: waits for work that may still
// use the old list).
static int ensure_ray_list(const kf_volume* v, size_t rays, hipStream_t s)
{
    if (!v->ray_count) {
        KF_HIP(hipMalloc(&v->ray_count, 2 * 8 * kCountStride * sizeof(unsigned)));
        KF_HIP(hipMemset(v->ray_count, 0, 2 * 8 * kCountStride * sizeof(unsigned)));
    }
    if (v->ray_cap >= rays) return KF_OK;
    KF_HIP(hipStreamSynchronize(s));
    (void)hipFree(v->ray_list);
    v->ray_list = nullptr;
    v->ray_cap = 0;
    KF_HIP(hipMalloc(&v->ray_list, sizeof(DeferredRay) * rays));
    v->ray_cap = rays;
    return KF_OK;
}

int launch_raycast_levels(const kf_volume* v, const float* pose, const PoseState* dyn_state, int levels,
                          const float (*inv_k)[9], float4* const* vout, float4* const* nout, int w0, int h0,
                          hipStream_t s, const RaycastSide* side)
{
    RaycastArgs a{};
    a.vol = raycast_volume(v);
    if (pose) memcpy(a.pose, pose, sizeof(a.pose));
    a.dyn = dyn_state;
    if (side) a.side = *side;
    a.levels = levels;
    int tiles = 0;
    for (int l = 0; l < levels; ++l) {
        RaycastLevel& L = a.lv[l];
        memcpy(L.Kinv, inv_k[l], sizeof(L.Kinv));
        L.vout = vout[l];
        L.nout = nout[l];
        L.w = w0 >> l;
        L.h = h0 >> l;
        L.tiles_x = (L.w + 7) / 8;
        L.tile0 = tiles;
        tiles += L.tiles_x * ((L.h + 7) / 8);
    }
    a.tiles = tiles;
    unsigned blocks = 0;
    for (int l = 0; l < levels; ++l) blocks += (unsigned)level_blocks(a, l);
    // every ray of an XCD's workgroups has a place in its list
    int st = ensure_ray_list(v, (size_t)blocks * 64, s);
    if (st == KF_OK) st = refresh_free_distances(v, s);
    if (st) return st;
    const int parity = (int)(v->ray_launches++ & 1);
    a.rays = static_cast<DeferredRay*>(v->ray_list);
    a.count = v->ray_count + parity * 8 * kCountStride;
    a.clear = v->ray_count + (1 - parity) * 8 * kCountStride;
    a.cap = (unsigned)(v->ray_cap / 8);
    if (v->format == KF_VOXEL_F32) {
        raycast_kernel<KF_VOXEL_F32><<<blocks, 64, 0, s>>>(a);
        KF_LAUNCHED("raycast_kernel");
        raycast_finish_kernel<KF_VOXEL_F32><<<kFinishWaves / kFinishPer, 64 * kFinishPer, 0, s>>>(a);
    } else {
        raycast_kernel<KF_VOXEL_SNORM16_U8><<<blocks, 64, 0, s>>>(a);
        KF_LAUNCHED("raycast_kernel");
        raycast_finish_kernel<KF_VOXEL_SNORM16_U8><<<kFinishWaves / kFinishPer, 64 * kFinishPer, 0, s>>>(a);
    }
    KF_LAUNCHED("raycast_finish_kernel");
    return KF_OK;
}

int launch_raycast(const kf_volume* v, const float* pose, const PoseState* dyn_state, const float* inv_k,
                   float4* vout, float4* nout, int w, int h, hipStream_t s)
{
    float ki[1][9];
    memcpy(ki[0], inv_k, sizeof(ki[0]));
    return launch_raycast_levels(v, pose, dyn_state, 1, ki, &vout, &nout, w, h, s);
}

}  // namespace kf

extern "C" int kf_raycast(const kf_volume* v, const kf_sensor* sensor, float* vertex_map, float* normal_map, int w,
                          int h, int level, kf_stream_t stream, float* elapsed_ms)
{
    if (!v || !sensor || !vertex_map || !normal_map || w <= 0 || h <= 0)
        return kf::fail(KF_ERR_ARG, "raycast: bad argument");
    if (level < 0 || level > 2) return kf::fail(KF_ERR_ARG, "raycast: level must be 0..2 (sensor.h:51-52)");
    hipStream_t s = kf::stream_of(stream);
    kf::CallTimer t(elapsed_ms, s);
    int st;
    if ((st = t.start()) ||
        (st = kf::launch_raycast(v, sensor->pose, nullptr, sensor->inv_intr[level], reinterpret_cast<float4*>(vertex_map),
                                 reinterpret_cast<float4*>(normal_map), w, h, s)))
        return st;
    return t.finish();
}
