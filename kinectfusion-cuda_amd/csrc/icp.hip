// Projective point-to-plane ICP (project/src/icp.cu, icp.cuh, icp.cpp,
// linear_least_squares.cpp), kept on the device for a whole frame.
//
// One iteration has two parts:
//   reduce   : 256 lanes x 4 pixels per workgroup.  Each lane associates its
//              pixels (icp.cu:7-82) and accumulates the 27 unique terms of the
//              normal equations (21 of A^T A, 6 of A^T b) in FP32 registers;
//              then a 64-lane shuffle tree and an LDS pass over the 4 waves, in
//              FP32 or (the compensated form) in FP64, and one partial row per
//              workgroup.  A and b are never materialised.
//   finalize : one workgroup sums the partial rows in a fixed order (so the
//              result is deterministic), solves the 6x6 system with an FP64
//              Cholesky, applies the pose update (icp.cpp:65-87) and the early
//              stop test (icp.cpp:45-53) to the device-resident PoseState.
// The kernel boundary between them is what makes every workgroup's partial row
// visible to the finalize across the 8 XCDs' L2s.  A frame's loop has one launch per
// iteration: every workgroup of the next reduce does the finalize for itself first.
// The reference instead writes A (N x 6) and b to HBM, runs cublasSgemm and
// cublasSgemv, copies 42 floats to the host and solves with Eigen's FP32 LLT,
// with a host synchronisation per iteration.
#include <math.h>
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

#include "kf_device.hpp"
#include "kf_kernels.hpp"

namespace kf {

namespace {

constexpr int kThreads = 256;
constexpr int kPixPerThread = 4;  // pixels per lane, at most (see icp_pix_for)
constexpr int kTerms = 27;
// The type the lanes' sums are added up in: FP32, or FP64 for the compensated
// form.  An FP64 addition issues at the rate of an FP32 one here, so it takes one
// instruction where FP32 sums that carry their rounding errors (TwoSum) take
// eight, and rounds at 2^-53.  Association of a tick of 64 sessions, sums with their
// errors -> FP64: 640x480 (4 pixels per lane) 247 -> 235 us, 320x240 (one) 117 -> 96;
// a whole compensated frame of 640x480 into 256^3 416 -> 388 us.
template <bool COMP>
struct SumType {
    using T = float;
};
template <>
struct SumType<true> {
    using T = double;
};
// Partial rows (component-major, of SumType): [0,27) sums, 27 the inlier count.

// Element e of M = K R_prev^T (both column-major), in m3m3's order.
__host__ __device__ __forceinline__ float projection_element(const float* K, const float* Rp, int e)
{
    const int c = e / 3, r = e % 3;
    return (K[r] * Rp[c] + K[3 + r] * Rp[3 + c]) + K[6 + r] * Rp[6 + c];
}

// icp.cu:7-82 split in two: what a pixel needs that does not depend on the
// pose (its vertex and its live normal, device_helper.cuh:81-110) and the
// pose-dependent association, so the loads of the first part can be issued
// before the pose of the iteration is known.
struct PixelIn {
    v3 vc;       // camera-space vertex
    v3 cr;       // live normal before normalization (device_helper.cuh:81-110's cross product)
    bool ok;     // vertex and normal valid
};
__device__ __forceinline__ PixelIn icp_pixel_from(float4 c, float4 r, float4 d, bool ok)
{
    PixelIn in;
    in.vc = xyz(c);
    in.cr = cross3(sub3(xyz(r), in.vc), sub3(xyz(d), in.vc));  // normal_of before its normalize3
    in.ok = ok && c.w == kValid && r.w == kValid && d.w == kValid;
    return in;
}

// The rejection tests decide a boolean only, so each is first decided from a
// cheap approximation and evaluated exactly (the reference arithmetic, correctly
// rounded square root and division) only when the approximation lies too close to
// the threshold to decide: the decision is the exact one always.
//
// Projection, icp.cuh:40-49: the floor of p.x / p.z and p.y / p.z.  The quotients
// from the hardware reciprocal (1 ulp) and the correctly rounded ones differ by
// less than 2^-21 of their size, so inside the map by less than band = 2^-21
// max(w, h): both have the same floor unless the former lies within band of an
// integer.  Outside the map both floors are outside.  A p.z that the hardware
// routine may flush takes the exact path.
__device__ __forceinline__ void floor_quotients(v3 p, float band, float& fu, float& fv)
{
    const float r = __builtin_amdgcn_rcpf(p.z);
    const float qx = p.x * r, qy = p.y * r;
    fu = floorf(qx);
    fv = floorf(qy);
    const float off = fmaxf(fabsf((qx - fu) - 0.5f), fabsf((qy - fv) - 0.5f)), az = fabsf(p.z);
    if (!(off <= 0.5f - band) || !(az >= 0x1p-100f && az <= 0x1p100f)) {
        fu = floorf(p.x / p.z);
        fv = floorf(p.y / p.z);
    }
}
// Distance, icp.cuh:57-60: reject iff RN(sqrt(D)) > T, D = dot(v, v) (the
// same bits on both paths).  D <= T^2 gives sqrt(D) <= T; D >= (T + ulp(T))^2
// gives RN(sqrt(D)) > T.  lo and hi below bound those squares from inside
// (lo <= T^2, hi >= T^2 (1 + 2^-21) > (T + ulp(T))^2); NaN takes the exact path.  A
// negative T keeps its sign in the square (no length is at most T), a square of 0
// accepts a length of 0 only, and an infinite D is never accepted unseen.
//
// Angle, icp.cuh:63-70 in its cosine form (acos(d) > th <=> d >= -1 && d < cos
// th), d = dot(normalize(Rc normalize(cr)), n).  The approximation da rotates cr
// as it is and takes one normalization, with the hardware reciprocal square root
// (1 ulp).  With u = 2^-24 and Rc a rotation: turning cr costs at most 3 sqrt(3) u
// of its length (three products and two sums per component), its squared length 3 u
// and the root of it half of that, the reciprocal root 2 u, the product with n 3 u and
// the last product u, 12.7 u |n| in all; d has the same, one more normalization (3 u)
// and a division per component, at most 17 u |n|: they differ by less than 30 u |n| <
// 2^-19 |n|_1 (measured worst case over 8M random rotations, normals and lengths with
// the reciprocal root off by one ulp either way: 2^-21.3).  A margin of 2^-16 |n|_1
// decides, eight times that, so also for a matrix that is a rotation only roughly; a
// squared length outside [2^-100, 2^100] (where the hardware routine may flush or
// overflow) and NaN take the exact path.
__device__ __forceinline__ bool pair_rejected(const IcpArgs& a, const float* Rc, v3 v, v3 cr, v3 n, bool live)
{
    const float D = dot3(v, v);
    const float T2 = a.dist_thresh * fabsf(a.dist_thresh);
    const float lo = fminf(T2 * (1.0f - 0x1p-22f), 0x1.fffffep127f), hi = T2 * (1.0f + 0x1p-20f);
    const v3 m = m3v(Rc, cr);
    const float mq = dot3(m, m);
    const float da = dot3(m, n) * __builtin_amdgcn_rsqf(mq);
    const float del = 0x1p-16f * (fabsf(n.x) + fabsf(n.y) + fabsf(n.z));
    const bool ranged = mq >= 0x1p-100f && mq <= 0x1p100f;
    const float c = a.cos_thresh;
    bool rejected = D > hi || (ranged && da < c - del && da >= -1.0f + del);
    const bool accepted = D <= lo && ranged && da >= c + del;
    if (live && !rejected && !accepted) {
        rejected = len3(v) > a.dist_thresh;
        const float dd = dot3(normalize3(m3v(Rc, normalize3(cr))), n);
        rejected = rejected || (dd >= -1.0f && dd < c);
    }
    return rejected;
}

// false = zero row (rejection reasons as icp.cu:29-70, evaluated in an order
// that does not change the result: every rejection writes the same zero row).
// Split in two so that the target loads of all of a lane's pixels are in
// flight together: icp_pixel_gather transforms and projects the pixel and
// issues the loads of its target vertex and normal (at an in-map index even
// when the projection is off the map, so no branch surrounds the loads);
// icp_pixel_finish applies the tests and builds the row.
struct PixelGather {
    v3 s;             // the vertex in the frame of the current estimate
    float4 tv, tn;    // target vertex and normal at the projection
    bool ok;          // the pixel is valid and projects into the map
};
// SMALL: the map has at most kMaxMapPixels pixels, so a pixel's index is exact in
// FP32 and its byte offset fits 32 bits (one register beside the map's address).
template <bool SMALL>
__device__ __forceinline__ PixelGather icp_pixel_gather(const IcpArgs& a, const PixelIn& in, const IterPose& P)
{
    PixelGather g;
    g.s = add3(m3v(P.R, in.vc), mk3(P.t[0], P.t[1], P.t[2]));
    // icp.cuh:40-49: (K * R_prev^T) * (s - t_prev), floor of the perspective division
    const v3 p = m3v(P.M, sub3(g.s, mk3(P.tp[0], P.tp[1], P.tp[2])));
    const float wf = (float)a.w, hf = (float)a.h;
    float fu, fv;
    floor_quotients(p, 0x1p-21f * fmaxf(wf, hf), fu, fv);
    g.ok = in.ok && fu >= 0.0f && fv >= 0.0f && fu < wf && fv < hf;
    if (SMALL) {
        const uint32_t o = g.ok ? (uint32_t)(int)fmaf(fv, wf, fu) * 16u : 0u;
        g.tv = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.TV) + o);
        g.tn = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.TN) + o);
    } else {
        const int64_t q = g.ok ? (int64_t)(int)fv * a.w + (int)fu : 0;
        g.tv = a.TV[q];
        g.tn = a.TN[q];
    }
    return g;
}
__device__ __forceinline__ bool icp_pixel_finish(const IcpArgs& a, const PixelIn& in, const PixelGather& g,
                                                 const float* Rc, float* row, float& b)
{
    const v3 s = g.s, d = xyz(g.tv), n = xyz(g.tn);
    const bool live = g.ok && g.tv.w == kValid && g.tn.w == kValid;
    if (pair_rejected(a, Rc, sub3(d, s), in.cr, n, live) || !live) return false;
    // icp.cuh:72-95
    row[0] = n.y * s.z - n.z * s.y;
    row[1] = n.z * s.x - n.x * s.z;
    row[2] = n.x * s.y - n.y * s.x;
    row[3] = n.x;
    row[4] = n.y;
    row[5] = n.z;
    b = ((((n.x * d.x + n.y * d.y) + n.z * d.z) - n.x * s.x) - n.y * s.y) - n.z * s.z;
    return true;
}

// Adds a pixel's row to the lane's FP32 sums of A^T A (upper triangle) and
// A^T b, each product fused into its sum (one rounding instead of two).  A lane
// sums at most kPixPerThread rows, so its few roundings are small against the
// total; the compensated form takes every addition after that (lanes, waves,
// workgroups: block_reduce_store and the partial-row sums) in FP64, where
// nearly all of the additions happen.
__device__ __forceinline__ void accumulate(float* s, const float* row, float b)
{
    int q = 0;
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int r = p; r < 6; ++r, ++q) s[q] = fmaf(row[p], row[r], s[q]);
#pragma unroll
    for (int p = 0; p < 6; ++p) s[21 + p] = fmaf(row[p], b, s[21 + p]);
}

// The lane exchanges of kf_device.hpp for both sum types.
template <int CTRL>
__device__ __forceinline__ float sum_partner(float v)
{
    return dpp_partner<CTRL>(v);
}
template <int CTRL>
__device__ __forceinline__ double sum_partner(double v)
{
    return __hiloint2double(dpp_partner<CTRL>(__double2hiint(v)), dpp_partner<CTRL>(__double2loint(v)));
}
template <int OFF>
__device__ __forceinline__ void sum_swap(float a, float b, float& lo, float& hi)
{
    swap_pair<OFF>(a, b, lo, hi);
}
template <int OFF>
__device__ __forceinline__ void sum_swap(double a, double b, double& lo, double& hi)
{
    float l0, l1, h0, h1;
    swap_pair<OFF>(__int_as_float(__double2loint(a)), __int_as_float(__double2loint(b)), l0, h0);
    swap_pair<OFF>(__int_as_float(__double2hiint(a)), __int_as_float(__double2hiint(b)), l1, h1);
    lo = __hiloint2double(__float_as_int(l1), __float_as_int(l0));
    hi = __hiloint2double(__float_as_int(h1), __float_as_int(h0));
}
// Sum over the 64 lanes, in every lane (the same pairing as wave_reduce).
template <class T>
__device__ __forceinline__ T wave_total(T v)
{
    T lo, hi;
    sum_swap<32>(v, v, lo, hi);
    v = lo + hi;
    sum_swap<16>(v, v, lo, hi);
    v = lo + hi;
    v = v + sum_partner<kDppRowMirror>(v);
    v = v + sum_partner<kDppRowHalfMirror>(v);
    v = v + sum_partner<kDppXor2>(v);
    return v + sum_partner<kDppXor1>(v);
}

// One halving step of the lane reduction: the first n/2 entries of s become, on
// the lane with the step's bit clear, its first half plus the partner's copy
// and, on the other lane, its second half plus the partner's copy.
template <int N, int OFF, class T>
__device__ __forceinline__ void halve_swap(T* s)
{
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        T lo, hi;
        sum_swap<OFF>(s[i], s[N / 2 + i], lo, hi);
        s[i] = lo + hi;
    }
}
template <int N, int CTRL, class T>
__device__ __forceinline__ void halve_dpp(T* s, bool upper)
{
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const T send = upper ? s[i] : s[N / 2 + i];
        const T keep = upper ? s[N / 2 + i] : s[i];
        s[i] = keep + sum_partner<CTRL>(send);
    }
}

// Reduces the lane values of a workgroup and writes one partial row.  The 27
// terms are halved across the lanes (28 -> 14 -> 7 -> 4 -> 2 -> 1, one zero
// pad at 27 and one at the 7 -> 8 step): lane L ends with term
// 14*b5 + 7*b4 + 4*b3 + 2*b2 + b1 of its bits, every pair (L, L^1) holding it
// (each step keeps the first half on the lane whose step bit is clear).
// The first step exchanges the lanes' FP32 sums and widens them as it adds.  cnt is
// the wave's count.
template <class T>
__device__ __forceinline__ void block_reduce_store(const float* s_in, int cnt, float* partials, int stride, int row)
{
    __shared__ T red[kThreads / 64][kTerms + 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T s[14];
#pragma unroll
    for (int q = 0; q < 14; ++q) {
        float lo, hi;
        swap_pair<32>(s_in[q], q < 13 ? s_in[14 + q] : 0.0f, lo, hi);
        s[q] = (T)lo + (T)hi;
    }
    halve_swap<14, 16>(s);
    s[7] = 0;
    halve_dpp<8, kDppRowMirror>(s, (lane & 8) != 0);
    halve_dpp<4, kDppRowHalfMirror>(s, (lane & 4) != 0);
    halve_dpp<2, kDppXor2>(s, (lane & 2) != 0);
    s[0] = s[0] + sum_partner<kDppXor1>(s[0]);  // both lanes of the pair add the same two operands
    const int sub = 4 * ((lane >> 3) & 1) + 2 * ((lane >> 2) & 1) + ((lane >> 1) & 1);
    const int q = 14 * ((lane >> 5) & 1) + 7 * ((lane >> 4) & 1) + sub;
    if ((lane & 1) == 0 && sub < 7 && q < kTerms) red[wave][q] = s[0];
    if (lane == 0) red[wave][kTerms] = (T)cnt;
    __syncthreads();
    if (threadIdx.x <= kTerms) {
        const int t = threadIdx.x;
        T ss = red[0][t];
        for (int wv = 1; wv < kThreads / 64; ++wv) ss = ss + red[wv][t];
        reinterpret_cast<T*>(partials)[(int64_t)t * stride + row] = ss;
    }
}

// The pixels of lane (block, k, lane), k < pix <= PIX, and their
// pose-independent inputs: pixel (block * pix + k) * kThreads + lane.
template <int PIX = kPixPerThread>
struct LanePixels {
    PixelIn in[PIX];
};
// Their vertex loads only, so the loads can be in flight while the workgroup
// finishes the previous iteration.  ok: the pixel has a right and a lower neighbour.
template <int PIX = kPixPerThread>
struct LaneLoads {
    float4 c[PIX], r[PIX], d[PIX];
    bool ok[PIX];
};
// Column of pixel px of a w-wide map, px < kMaxMapPixels: px is exact in FP32 and
// px * (1/w) is within one of px / w, so one correction each way gives the
// quotient (and 24-bit products suffice).
constexpr int kMaxMapPixels = 1 << 24;
__device__ __forceinline__ int pixel_column(int px, int w, float inv_w)
{
    int u = px - (int)__umul24((unsigned)((float)px * inv_w), (unsigned)w);
    if (u < 0) u += w;
    else if (u >= w) u -= w;
    return u;
}
// Only pixels up to `last` have a lower and (short of their row's end) a right
// neighbour; a pixel past it loads the last one's, so no select surrounds a load,
// and the three loads share one 32-bit offset.
__device__ __forceinline__ void issue_pixel_loads(const IcpArgs& a, int px, float4& c, float4& r, float4& d, bool& ok)
{
    const int last = a.w * a.h - a.w - 2;  // w x h <= kMaxMapPixels (checked on the host)
    const bool any = a.w > 1 && a.h > 1;   // uniform; else no pixel has both neighbours
    const float inv_w = 1.0f / (float)a.w;
    const char* row0 = reinterpret_cast<const char*>(a.V);
    const char* row1 = row0 + (size_t)a.w * 16;
    ok = any && px <= last && pixel_column(px, a.w, inv_w) + 1 < a.w;
    if (!any) {
        c = r = d = make_float4(0.0f, 0.0f, 0.0f, kInvalid);
        return;
    }
    const uint32_t o = (uint32_t)min(px, last) * 16u;
    c = *reinterpret_cast<const float4*>(row0 + o);
    r = *reinterpret_cast<const float4*>(row0 + o + 16);
    d = *reinterpret_cast<const float4*>(row1 + o);
}
template <int PIX>
__device__ __forceinline__ void issue_lane_loads(const IcpArgs& a, LaneLoads<PIX>& ll, int block, int pix)
{
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        if (k >= pix) break;  // uniform
        issue_pixel_loads(a, (block * pix + k) * kThreads + (int)threadIdx.x, ll.c[k], ll.r[k], ll.d[k], ll.ok[k]);
    }
}
template <int PIX>
__device__ __forceinline__ void finish_lane_pixels(const LaneLoads<PIX>& ll, LanePixels<PIX>& lp, int pix)
{
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        if (k >= pix) break;
        lp.in[k] = icp_pixel_from(ll.c[k], ll.r[k], ll.d[k], ll.ok[k]);
    }
}
template <int PIX>
__device__ __forceinline__ void load_lane_pixels(const IcpArgs& a, LanePixels<PIX>& lp, int block, int pix)
{
    LaneLoads<PIX> ll;
    issue_lane_loads(a, ll, block, pix);
    finish_lane_pixels(ll, lp, pix);
}

// Associates the lane's pixels at the iteration's pose and writes partial row
// `block` of a.partials.  Bound: latency in a frame, whose launches have a wave or two
// per SIMD; the vector ALU in a batch tick (0.91 busy at 320x240, 0.68 at 640x480,
// where the maps' bytes come at 4.4 TB/s).
// With the projection's quotients taken approximately, one normalization less in
// the angle test, offsets of 32 bits shared by a pixel's loads, the projection
// matrix formed once instead of by every lane, the batch's pose in scalar registers
// and counts by ballot, the association of a tick of 64 sessions took 142 instead of
// 154 us on average over its 19 iterations; sixteen uneven sessions 32 -> 25 us,
// a frame 333 -> 321 us (512^3, plain) and 365 -> 347 us (256^3, compensated).
template <bool COMP, int PIX>
__device__ __forceinline__ void associate_reduce(const IcpArgs& a, const LanePixels<PIX>& lp, const IterPose& P,
                                                 int block, int pix)
{
    float s[kTerms];
#pragma unroll
    for (int q = 0; q < kTerms; ++q) s[q] = 0.0f;
    int cnt = 0;  // of the wave
    PixelGather g[PIX];
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        if (k >= pix) break;
        g[k] = icp_pixel_gather<true>(a, lp.in[k], P);
    }
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        if (k >= pix) break;
        float row[6], b;
        const bool hit = icp_pixel_finish(a, lp.in[k], g[k], P.R, row, b);
        cnt += __popcll(__ballot(hit));
        if (hit) accumulate(s, row, b);
    }
    block_reduce_store<typename SumType<COMP>::T>(s, cnt, a.partials, a.stride, block);
}

template <bool COMP>
__device__ void reduce_body(const IcpArgs& a)
{
    PoseState* st = a.st;
    __shared__ IterPose pose;
    LanePixels<> lp;
    load_lane_pixels(a, lp, blockIdx.x, kPixPerThread);
    if (threadIdx.x < 9) pose.R[threadIdx.x] = st->R[threadIdx.x];
    else if (threadIdx.x < 12) pose.t[threadIdx.x - 9] = st->t[threadIdx.x - 9];
    else if (threadIdx.x < 21) pose.M[threadIdx.x - 12] = projection_element(a.K, st->Rp, threadIdx.x - 12);
    else if (threadIdx.x < 24) pose.tp[threadIdx.x - 21] = st->tp[threadIdx.x - 21];
    __syncthreads();
    associate_reduce<COMP>(a, lp, pose, blockIdx.x, kPixPerThread);
}

template <bool COMP>
__global__ __launch_bounds__(kThreads) void icp_reduce_kernel(IcpArgs a)
{
    if (a.st->status != 0 || a.st->level_done[a.level]) return;
    reduce_body<COMP>(a);
}

// Rows of a given A (n x 6 row-major) and b (LinearLeastSquares::solve).  The first
// workgroup clears what the solve that follows reports.
template <bool COMP>
__global__ __launch_bounds__(kThreads) void ab_reduce_kernel(const float* A, const float* B, int64_t n,
                                                             float* partials, int stride, PoseState* st)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->status = st->sticky_status = 0;
        for (int q = 0; q < 6; ++q) st->last_x[q] = 0.0f;
    }
    float s[kTerms];
#pragma unroll
    for (int q = 0; q < kTerms; ++q) s[q] = 0.0f;
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < kPixPerThread; ++k) {
        const int64_t r = ((int64_t)blockIdx.x * kPixPerThread + k) * kThreads + threadIdx.x;
        bool nz = false;
        if (r < n) {
            float row[6];
#pragma unroll
            for (int p = 0; p < 6; ++p) row[p] = A[r * 6 + p];
            const float b = B[r];
            accumulate(s, row, b);
            nz = b != 0.0f;
#pragma unroll
            for (int p = 0; p < 6; ++p) nz = nz || row[p] != 0.0f;
        }
        cnt += __popcll(__ballot(nz));
    }
    block_reduce_store<typename SumType<COMP>::T>(s, cnt, partials, stride, blockIdx.x);
}

// icp.cu:7-82, writing the rows (kernel::constructIcpResiduals).
__global__ __launch_bounds__(kThreads) void icp_rows_kernel(IcpArgs a, IterPose P, float* A, float* B)
{
    int64_t px = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (px >= (int64_t)a.w * a.h) return;
    int u = (int)(px % a.w), v = (int)(px / a.w);
    float row[6] = {0, 0, 0, 0, 0, 0}, b = 0.0f;
    const NormalStencil ns = load_normal_stencil(a.V, a.w, a.h, u, v);
    const PixelIn in = icp_pixel_from(ns.c, ns.r, ns.d, true);
    if (!icp_pixel_finish(a, in, icp_pixel_gather<false>(a, in, P), P.R, row, b)) {
#pragma unroll
        for (int p = 0; p < 6; ++p) row[p] = 0.0f;
        b = 0.0f;
    }
#pragma unroll
    for (int p = 0; p < 6; ++p) A[px * 6 + p] = row[p];
    B[px] = b;
}

// ---- FP64 6x6 Cholesky solve, unblocked, in the column order of Eigen's LLT
// (3rd/eigen/Eigen/src/Cholesky/LLT.h:306-326):
//   D = A(k,k) - sum_j<k L(k,j)^2,   i(k) = 1 / sqrt(D),
//   L(r,k) = (A(r,k) - sum_j<k L(r,j) L(k,j)) * i(k),
//   y(r) = (b(r) - sum_j<r L(r,j) y(j)) * i(r),
//   x(r) = (y(r) - sum_j>r L(j,r) x(j)) * i(r)
// (a reciprocal square root and multiplications instead of a square root and
// divisions by L(r,r), and fused multiply-adds in the sums: each value moves
// by a few ulp of FP64, far below the FP32 pose it feeds, and the FP64 square
// roots and divisions leave the dependent chain).  Every lane forms the whole matrix
// from the sums in LDS: the solve is one chain of dependent FP64 operations, and rows
// spread over lanes added a lane broadcast to each of its links.
// Returns 0 or the failing column + 1 and the solution in x.
__device__ __forceinline__ double bcast(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// index of A(p, q), p <= q, among the 21 sums: rows of the upper triangle
__device__ __forceinline__ int sym_index(int p, int q) { return p * 6 - (p * (p - 1)) / 2 + (q - p); }

__device__ __forceinline__ int chol6(const double* tot, double* x)
{
    double L[6][6], inv[6], y[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        double d = tot[sym_index(k, k)];
#pragma unroll
        for (int j = 0; j < k; ++j) d = fma(-L[k][j], L[k][j], d);
        if (!(d > 0.0)) return k + 1;
        inv[k] = rsqrt(d);  // 1/sqrt, within 2 ulp of FP64
#pragma unroll
        for (int r = k + 1; r < 6; ++r) {
            double v = tot[sym_index(k, r)];
#pragma unroll
            for (int j = 0; j < k; ++j) v = fma(-L[r][j], L[k][j], v);
            L[r][k] = v * inv[k];
        }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        double v = tot[21 + q];
#pragma unroll
        for (int j = 0; j < q; ++j) v = fma(-L[q][j], y[j], v);
        y[q] = v * inv[q];
    }
#pragma unroll
    for (int q = 5; q >= 0; --q) {
        double v = y[q];
#pragma unroll
        for (int j = q + 1; j < 6; ++j) v = fma(-L[j][q], x[j], v);
        x[q] = v * inv[q];
    }
    return 0;
}

// icp.cpp:65-87 in FP64: R_inc = R_y(x1) R_x(x0) R_z(x2) (glm orientate3(x0, x2, x1)),
// R <- R_inc^T R, t <- R_inc^T t + x[3..5].
//
// sin and cos in FP64 of an angle x: Cody-Waite reduction r = x - k pi/2 with
// pi/2 split in a 33-bit head (k * head exact for |k| < 2^20) and a tail,
// then the Taylor series of sin and cos on |r| <= pi/4 (terms through r^17
// and r^18: the next terms are below 2^-60 there; Horner steps fused).  Accurate to a few ulp of
// double for |x| < 2^20 pi/2, far beyond any ICP update; the library routines
// carry a huge-argument reduction whose registers every lane of the kernel
// would pay for.
__device__ __forceinline__ void sincos_small(double x, double* sn, double* cs)
{
    const double kHead = 1.57079632673412561417e+00;  // leading 33 bits of pi/2
    const double kTail = 6.07710050650619224932e-11;  // pi/2 - kHead
    const double k = rint(x * 0.636619772367581343076);
    const double r = (x - k * kHead) - k * kTail;
    const double z = r * r;
    double ps = 1.0 / 355687428096000.0;            // 1/17!
    ps = fma(ps, z, -1.0 / 1307674368000.0);        // 1/15!
    ps = fma(ps, z, 1.0 / 6227020800.0);            // 1/13!
    ps = fma(ps, z, -1.0 / 39916800.0);             // 1/11!
    ps = fma(ps, z, 1.0 / 362880.0);                // 1/9!
    ps = fma(ps, z, -1.0 / 5040.0);                 // 1/7!
    ps = fma(ps, z, 1.0 / 120.0);                   // 1/5!
    ps = fma(ps, z, -1.0 / 6.0);                    // 1/3!
    const double s = fma(r, z * ps, r);
    double pc = 1.0 / 6402373705728000.0;           // 1/18!
    pc = fma(pc, z, -1.0 / 20922789888000.0);       // 1/16!
    pc = fma(pc, z, 1.0 / 87178291200.0);           // 1/14!
    pc = fma(pc, z, -1.0 / 479001600.0);            // 1/12!
    pc = fma(pc, z, 1.0 / 3628800.0);               // 1/10!
    pc = fma(pc, z, -1.0 / 40320.0);                // 1/8!
    pc = fma(pc, z, 1.0 / 720.0);                   // 1/6!
    pc = fma(pc, z, -1.0 / 24.0);                   // 1/4!
    pc = fma(pc, z, 0.5);                           // 1/2!
    const double c = fma(-z, pc, 1.0);
    const int q = (int)((long long)k & 3);
    *sn = q == 0 ? s : (q == 1 ? c : (q == 2 ? -s : -c));
    *cs = q == 0 ? c : (q == 1 ? -s : (q == 2 ? -c : s));
}

// sin and cos of the three angles of an update, as update_pose uses them:
// yaw x[1] (sh, ch), pitch x[0] (sp, cp), roll x[2] (sb, cb).
struct SinCos3 {
    double sh, ch, sp, cp, sb, cb;
};
// Formed by lanes 0, 1, 2 of a wave, from the float update x (every lane of the wave
// calls it and receives all six values).
__device__ __forceinline__ SinCos3 angle_sincos_wave(const float* x)
{
    const int lane = threadIdx.x & 63;
    const float ang = lane == 0 ? x[1] : (lane == 1 ? x[0] : x[2]);
    double sn, cs;
    sincos_small(ang, &sn, &cs);
    SinCos3 a;
    a.sh = bcast(sn, 0);
    a.ch = bcast(cs, 0);
    a.sp = bcast(sn, 1);
    a.cp = bcast(cs, 1);
    a.sb = bcast(sn, 2);
    a.cb = bcast(cs, 2);
    return a;
}

// The updated pose, a float per lane: lane 3 c + r < 9 holds R(r, c), lanes 9 to 11 t.
// v: the same of the pose before.
__device__ __forceinline__ float update_pose_wave(float v, const float* x, const SinCos3& a)
{
    const double sh = a.sh, ch = a.ch, sp = a.sp, cp = a.cp, sb = a.sb, cb = a.cb;
    double Ri[9];
    Ri[0] = ch * cb + sh * sp * sb;  Ri[1] = sb * cp;  Ri[2] = -sh * cb + ch * sp * sb;
    Ri[3] = -ch * sb + sh * sp * cb; Ri[4] = cb * cp;  Ri[5] = sb * sh + ch * sp * cb;
    Ri[6] = sh * cp;                 Ri[7] = -sp;      Ri[8] = ch * cp;
    const int lane = threadIdx.x & 63, r = lane % 3, col = min(lane - r, 9);
    double s = 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const double e = r == 0 ? Ri[q] : (r == 1 ? Ri[3 + q] : Ri[6 + q]);
        s += e * (double)__shfl(v, col + q);
    }
    const float xt = r == 0 ? x[3] : (r == 1 ? x[4] : x[5]);
    return (float)(lane < 9 ? s : s + (double)xt);
}

// general_helper.cpp:11-21
__device__ void pose_error(const float* R1, const float* t1, const float* R2, const float* t2, float* out)
{
    v3 v = normalize3(mk3(1.0f, 1.0f, 1.0f));
    v3 a = m3v(R1, v), b = m3v(R2, v);
    out[0] = len3(sub3(b, a));
    out[1] = len3(sub3(mk3(t2[0], t2[1], t2[2]), mk3(t1[0], t1[1], t1[2])));
}

// Sums the partial rows (fixed order) into 27 doubles + count in LDS.  Wave w
// owns rows q = w, w + 4, ... (7 of the 28); lane l adds blocks l, l + 64, ...
// in that order, then the lanes combine (wave_total).  The loads of all of a
// wave's rows for a chunk of kRowHalves 64-block groups (RowChunk) are issued
// before any is added, so a row set costs one memory round trip per 320 blocks
// (a 640x480 level is 300); the first chunk can be loaded by the caller ahead
// of other loads (sum_loaded_partials).
constexpr int kRowsPerWave = (kTerms + 1 + 3) / 4;
constexpr int kRowHalves = 5;
template <class T>
struct RowChunk {
    T v[kRowHalves][kRowsPerWave];
};
// Needs nblocks > 0.  Lanes past the last block load the last block's entry
// (no divergent branch around the loads, so none waits for another);
// add_row_chunk skips them.  Groups wholly past the last block are not loaded
// (a wave-uniform test).
template <class T>
__device__ __forceinline__ void load_row_chunk(const float* partials, int stride, int nblocks, int b0, RowChunk<T>& ch)
{
    static_assert(kThreads == 256 && 3 + 4 * (kRowsPerWave - 1) == kTerms, "four waves own rows 0..kTerms");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const T* rows = reinterpret_cast<const T*>(partials);
#pragma unroll
    for (int h = 0; h < kRowHalves; ++h) {
        if (h > 0 && b0 + 64 * h >= nblocks) break;
        const int b = min(b0 + 64 * h + lane, nblocks - 1);
#pragma unroll
        for (int k = 0; k < kRowsPerWave; ++k) ch.v[h][k] = rows[(int64_t)(wave + 4 * k) * stride + b];
    }
}
template <class T>
__device__ __forceinline__ void add_row_chunk(int nblocks, int b0, const RowChunk<T>& ch, T* s)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int h = 0; h < kRowHalves; ++h) {
        if (h > 0 && b0 + 64 * h >= nblocks) break;
        const int b = b0 + 64 * h + lane;
#pragma unroll
        for (int k = 0; k < kRowsPerWave; ++k)
            if (b < nblocks) s[k] = s[k] + ch.v[h][k];
    }
}
// `first` = load_row_chunk(partials, stride, nblocks, 0, first); nblocks > 0.
template <class T>
__device__ void sum_loaded_partials(const float* partials, int stride, int nblocks, const RowChunk<T>& first,
                                    double* tot, double* count)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T s[kRowsPerWave];
#pragma unroll
    for (int k = 0; k < kRowsPerWave; ++k) s[k] = 0;
    add_row_chunk(nblocks, 0, first, s);
    for (int b0 = 64 * kRowHalves; b0 < nblocks; b0 += 64 * kRowHalves) {
        RowChunk<T> ch;
        load_row_chunk(partials, stride, nblocks, b0, ch);
        add_row_chunk(nblocks, b0, ch, s);
    }
#pragma unroll
    for (int k = 0; k < kRowsPerWave; ++k) {
        const int q = wave + 4 * k;
        const double t = (double)wave_total(s[k]);  // every lane: the same sum
        if (lane == 0) {
            if (q == kTerms) *count = t;  // wave-uniform
            else tot[q] = t;
        }
    }
    __syncthreads();
}
template <bool COMP>
__device__ void sum_partials(const float* partials, int stride, int nblocks, double* tot, double* count)
{
    RowChunk<typename SumType<COMP>::T> first = {};
    if (nblocks > 0) load_row_chunk(partials, stride, nblocks, 0, first);
    sum_loaded_partials(partials, stride, nblocks, first, tot, count);
}

// What a solve leaves in pinned host memory for a caller that waits.
struct SolveResult {
    float x[6];
    int status;
};

// The solution of the sums of partial rows (LinearLeastSquares::solve), recorded in the
// PoseState and, when given, in `out`.  Executed by every lane of one workgroup.
template <bool COMP>
__global__ __launch_bounds__(kThreads) void icp_finalize_kernel(PoseState* st, const float* partials, int stride,
                                                                int nblocks, SolveResult* out)
{
    __shared__ double tot[kTerms];
    __shared__ double count;
    sum_partials<COMP>(partials, stride, nblocks, tot, &count);
    if (threadIdx.x >= 64) return;
    double xd[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int rc = chol6(tot, xd) ? KF_ERR_NOT_PD : KF_OK;
    if (threadIdx.x != 0) return;
    for (int q = 0; q < kTerms; ++q) st->last_sums[q] = tot[q];
    st->last_inliers = (long long)count;
    const bool solved = rc == KF_OK;
    for (int q = 0; q < 6; ++q) {
        const float x = solved ? (float)xd[q] : 0.0f;
        if (solved && !isfinite(x)) rc = KF_ERR_NONFINITE;
        if (solved) st->last_x[q] = x;
        if (out) out->x[q] = x;
    }
    if (out) out->status = rc;
    if (rc != KF_OK) {
        if (st->status == 0) st->status = rc;
        if (st->sticky_status == 0) st->sticky_status = rc;
        st->frame_skip_fuse = 1;
    }
}

// ---- the device-resident coarse-to-fine loop: one launch per iteration.
// Launch k first finishes iteration k-1 (every workgroup sums launch k-1's
// partial rows in the same fixed order and solves, so all of them hold the same
// pose), then associates and reduces iteration k.  The carried state (IcpCarry)
// and the partial rows are double-buffered by launch parity, so no workgroup
// reads what another workgroup of the same launch writes.

// The carried state as a wave holds it: lane l has word l of the IcpCarry.
constexpr int kCarryWords = (int)(sizeof(IcpCarry) / sizeof(int));
constexpr int kWordStatus = (int)(offsetof(IcpCarry, status) / sizeof(int));
constexpr int kWordDone = (int)(offsetof(IcpCarry, level_done) / sizeof(int));
constexpr int kWordIterations = (int)(offsetof(IcpCarry, iterations) / sizeof(int));
constexpr int kWordPending = (int)(offsetof(IcpCarry, pending) / sizeof(int));
constexpr int kWordPendingLevel = (int)(offsetof(IcpCarry, pending_level) / sizeof(int));
constexpr int kWordPendingBlocks = (int)(offsetof(IcpCarry, pending_blocks) / sizeof(int));
static_assert(offsetof(IcpCarry, R) == 0 && offsetof(IcpCarry, t) == 36 && kWordStatus == 12 && kCarryWords <= 64,
              "the pose is the first twelve words");
__device__ __forceinline__ bool carry_pending(int word)
{
    return __builtin_amdgcn_readlane(word, kWordPending) != 0 && __builtin_amdgcn_readlane(word, kWordStatus) == 0;
}

// Applies the pending iteration of a carried state, solved from tot (icp.cpp:65-87, the
// early-stop test icp.cpp:45-53), by one wave; `record`: keeps the solve in st as well.
// Without a pending iteration the state stays as it is.
__device__ __forceinline__ int finish_iteration(int word, const double* tot, double count, PoseState* st, bool record,
                                                float stop_angle, float stop_dist)
{
    if (!carry_pending(word)) return word;  // uniform
    const int lane = threadIdx.x & 63;
    double xd[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int rc = chol6(tot, xd) ? KF_ERR_NOT_PD : KF_OK;
    float x[6];
    bool finite = true;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        x[q] = rc ? 0.0f : (float)xd[q];
        finite = finite && isfinite(x[q]);
    }
    if (!finite) rc = KF_ERR_NONFINITE;
    if (record) {
        if (lane < kTerms) st->last_sums[lane] = tot[lane];
        else if (lane == kTerms) st->last_inliers = (long long)count;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (lane == 32 + q) st->last_x[q] = x[q];
    }
    if (rc) return lane == kWordStatus ? rc : word;
    const float next = update_pose_wave(__int_as_float(word), x, angle_sincos_wave(x));
    // an error is at least 0: below a threshold of 0 or less it never is
    if (stop_angle > 0.0f && stop_dist > 0.0f) {  // uniform
        float was[12], is[12], err[2];
#pragma unroll
        for (int q = 0; q < 12; ++q) {
            was[q] = __int_as_float(__builtin_amdgcn_readlane(word, q));
            is[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(next), q));
        }
        pose_error(was, was + 9, is, is + 9, err);
        if (err[0] < stop_angle && err[1] < stop_dist &&
            lane == kWordDone + __builtin_amdgcn_readlane(word, kWordPendingLevel))
            word = 1;
    }
    if (lane < 12) word = __float_as_int(next);
    if (lane == kWordIterations) word += 1;
    return word;
}

// Opens an iteration at `level`: the state with its pending fields, and whether the
// session iterates.
__device__ __forceinline__ int open_iteration(int word, int level, int blocks, bool* run)
{
    const int lane = threadIdx.x & 63;
    *run = __builtin_amdgcn_readlane(word, kWordStatus) == 0 && !__builtin_amdgcn_readlane(word, kWordDone + level);
    if (lane == kWordPending) word = *run ? 1 : 0;
    if (lane == kWordPendingLevel) word = level;
    if (lane == kWordPendingBlocks) word = blocks;
    return word;
}

// Phase B of a launch for one session: finish the previous iteration from
// (cin, pin) and put the pose of this iteration in LDS.  `first` = this
// workgroup holds the session's partial row 0: it records the solve and writes
// the carried state for the next launch.  Returns (via run) whether the
// session iterates at `level` in this launch.  Ends with a barrier.
// Loads of phase B that do not depend on this launch's pose: the carried
// state (one word per lane of wave 0), the previous pose (lanes 64..75) and
// the first chunk of the previous launch's partial rows.  Issued before the
// pixel loads, so waiting for them does not wait for those (loads complete in
// issue order).
template <bool COMP>
struct BeginLoads {
    int cw;
    float pw;
    RowChunk<typename SumType<COMP>::T> rows;
};
template <bool COMP>
__device__ __forceinline__ void issue_begin_loads(const PoseState* st, const IcpCarry* cin, const float* pin,
                                                  int prev_blocks, BeginLoads<COMP>& bl)
{
    // every lane loads (indexes clamped; begin_iteration keeps the wanted
    // lanes' words), so no branch makes a load wait for the loads before it
    bl.cw = reinterpret_cast<const int*>(cin)[min((int)threadIdx.x & 63, kCarryWords - 1)];
    const int pi = min((int)threadIdx.x & 63, 11);
    bl.pw = *(pi < 9 ? st->Rp + pi : st->tp + (pi - 9));
    // no branch around the row loads either: with no previous launch
    // (prev_blocks = 0) every lane reads pin[0], and nothing is summed
    load_row_chunk(pin, prev_blocks, max(prev_blocks, 1), 0, bl.rows);
}

// Phase B of a launch for one session: finish the previous iteration from
// (cin, pin) and put the pose of this iteration in LDS.  `first` = this
// workgroup holds the session's partial row 0: it records the solve and writes
// the carried state for the next launch.  Returns (via run) whether the
// session iterates at `level` in this launch.  Ends with a barrier.  The rows
// are summed whether or not the previous launch left a pending iteration
// (prev_blocks is that launch's row count, known to the host; a sum nobody
// needs is discarded), so no load waits for the carry.
template <bool COMP>
__device__ void begin_iteration(const BeginLoads<COMP>& bl, PoseState* st, IcpCarry* cout, const float* pin,
                                int prev_blocks, int level, int blocks, bool first, float stop_angle, float stop_dist,
                                const float* K, IterPose* pose, int* run, double* tot, double* count)
{
    __shared__ float Rp[9];
    if (prev_blocks > 0) sum_loaded_partials(pin, prev_blocks, prev_blocks, bl.rows, tot, count);
    if (threadIdx.x >= 64 && threadIdx.x < 73) Rp[threadIdx.x - 64] = bl.pw;
    else if (threadIdx.x >= 73 && threadIdx.x < 76) pose->tp[threadIdx.x - 73] = bl.pw;
    __syncthreads();
    if (threadIdx.x >= 64 && threadIdx.x < 73)  // while wave 0 solves
        pose->M[threadIdx.x - 64] = projection_element(K, Rp, (int)threadIdx.x - 64);
    if (threadIdx.x < 64) {
        int word = finish_iteration(bl.cw, tot, *count, st, first, stop_angle, stop_dist);
        bool go;
        word = open_iteration(word, level, blocks, &go);
        if (threadIdx.x < 9) pose->R[threadIdx.x] = __int_as_float(word);
        else if (threadIdx.x < 12) pose->t[threadIdx.x - 9] = __int_as_float(word);
        if (threadIdx.x == 0) *run = go ? 1 : 0;
        if (first && threadIdx.x < kCarryWords) reinterpret_cast<int*>(cout)[threadIdx.x] = word;
    }
    __syncthreads();
}

template <bool COMP, int PIX>
__global__ __launch_bounds__(kThreads) void icp_step_kernel(IcpArgs a, const IcpCarry* cin, IcpCarry* cout,
                                                            const float* pin, int prev_blocks, float stop_angle,
                                                            float stop_dist)
{
    __shared__ IterPose pose;
    __shared__ int run;
    __shared__ double tot[kTerms];
    __shared__ double count;
    // phase A: the loads of phase B, then the pose-independent loads of this
    // lane's pixels (in flight during B)
    BeginLoads<COMP> bl;
    issue_begin_loads(a.st, cin, pin, prev_blocks, bl);
    LaneLoads<PIX> ll;
    issue_lane_loads(a, ll, blockIdx.x, PIX);
    __builtin_amdgcn_sched_barrier(0);  // nothing of phase B moves above the pixel loads
    // phase B: finish the previous iteration
    begin_iteration<COMP>(bl, a.st, cout, pin, prev_blocks, a.level, (int)gridDim.x, blockIdx.x == 0, stop_angle,
                          stop_dist, a.K, &pose, &run, tot, &count);
    if (!run) return;
    // phase C: live normals, association + reduction of this iteration
    LanePixels<PIX> lp;
    finish_lane_pixels(ll, lp, PIX);
    associate_reduce<COMP>(a, lp, pose, blockIdx.x, PIX);
}

// Starts a frame's ICP from a pose given by value.
struct Pose16 {
    float m[16];
};
__global__ __launch_bounds__(64) void icp_begin_kernel(PoseState* st, IcpCarry* c0, Pose16 pose)
{
    if (threadIdx.x < 16) st->pose[threadIdx.x] = pose.m[threadIdx.x];
    icp_begin_state(st, c0, pose.m);
}

// Commits the carried estimate as the sensor pose (Sensor::setPose,
// kinect_fusion.cpp:146-161, sensor.h:30-34); on failure the previous pose is
// kept and the frame is not fused.  By one wave; lane l holds word l of the state.
__device__ __forceinline__ void commit_state(PoseState* st, int word)
{
    const int lane = threadIdx.x & 63;
    const float v = __int_as_float(word);
    const int status = __builtin_amdgcn_readlane(word, kWordStatus);
    const int iterations = __builtin_amdgcn_readlane(word, kWordIterations);
    PoseMirror* out = st->mirror;
    const int r = lane % 3, c = lane / 3;  // lanes 0..8: element (r, c) of R; 9..11: t
    if (lane < 9) st->R[lane] = v;
    else if (lane < 12) st->t[r] = v;
    else if (lane >= kWordDone && lane < kWordDone + 4) st->level_done[lane - kWordDone] = word;
    else if (lane == kWordIterations) st->iterations = iterations;
    else if (lane == kWordStatus) st->status = status;
    if (out) {
        if (lane < 9) out->R[lane] = v;
        else if (lane < 12) out->t[r] = v;
        else if (lane == kWordIterations) out->iterations = iterations;
        else if (lane == kWordStatus) out->status = status;
    }
    if (status != 0) {
        if (lane == 0) {
            if (st->sticky_status == 0) st->sticky_status = status;
            st->frame_skip_fuse = 1;
        }
        return;
    }
    // the pose, its last row 0 0 0 1, and its inverse R^T, -R^T t
    double sum = 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) sum += (double)__shfl(v, r * 3 + q) * (double)__shfl(v, 9 + q);
    const bool top = lane < 12;
    const int e = lane < 15 ? (lane - 12) * 4 + 3 : 15;  // lanes 12..15: elements 3, 7, 11, 15
    const float p = top ? v : (lane == 15 ? 1.0f : 0.0f);
    if (lane < 16) {
        st->pose[top ? c * 4 + r : e] = p;
        if (out) out->pose[top ? c * 4 + r : e] = p;
        st->inv_pose[lane < 9 ? r * 4 + c : (top ? c * 4 + r : e)] = lane < 9 || !top ? p : (float)(-sum);
    }
}

// Finishes the last iteration and commits the estimate.
template <bool COMP>
__global__ __launch_bounds__(kThreads) void icp_commit_kernel(PoseState* st, const IcpCarry* cin, const float* pin,
                                                              int prev_blocks, float stop_angle, float stop_dist)
{
    __shared__ double tot[kTerms];
    __shared__ double count;
    const int word = reinterpret_cast<const int*>(cin)[min((int)threadIdx.x & 63, kCarryWords - 1)];
    // summed whether or not an iteration is pending, so no load waits for the state
    if (prev_blocks > 0) sum_partials<COMP>(pin, prev_blocks, prev_blocks, tot, &count);
    if (threadIdx.x >= 64) return;
    commit_state(st, finish_iteration(word, tot, count, st, true, stop_angle, stop_dist));
}

// ---- the same loop for many sessions per launch (batch ticks).  Each
// iteration is two launches: a solve launch (one workgroup per session)
// finishes the previous iteration from the session's partial rows and puts the
// pose of this iteration into its carry; an association launch reduces every
// block of every session (workgroup ranks own contiguous, XCD-contiguous block
// ranges).  Splitting keeps the FP64 solve out of the registers of the wide
// launch.  Partial rows are indexed by the session's own block number and
// summed in that order, so a session's result does not depend on the mix and
// equals the single-session loop's.
__global__ __launch_bounds__(64) void icp_batch_begin_kernel(const BatchHeader* hd, const IcpJob* jobs)
{
    for (int q = blockIdx.x; q < hd->n_icp; q += gridDim.x)
        icp_begin_state(jobs[q].a.st, jobs[q].carry, jobs[q].a.st->pose);
}

// final = 0: finish the pending iteration and open `level`; final = 1: finish
// the last iteration and commit the estimate (as icp_commit_kernel).
template <bool COMP>
__global__ __launch_bounds__(kThreads) void icp_batch_solve_kernel(const BatchHeader* hd, const IcpJob* jobs,
                                                                   int level, int final_, float stop_angle,
                                                                   float stop_dist)
{
    __shared__ double tot[kTerms];
    __shared__ double count;
    for (int q = blockIdx.x; q < hd->n_icp; q += gridDim.x) {
        const IcpJob& J = jobs[q];
        PoseState* st = J.a.st;
        int word = reinterpret_cast<const int*>(J.carry)[min((int)threadIdx.x & 63, kCarryWords - 1)];
        __syncthreads();  // every wave has read the carry before wave 0 rewrites it, and the previous sums
        if (carry_pending(word)) {
            const int blocks = __builtin_amdgcn_readlane(word, kWordPendingBlocks);
            sum_partials<COMP>(J.partials, blocks, blocks, tot, &count);
        }
        if (!final_) {  // of the association launch that follows
            if (threadIdx.x >= 64 && threadIdx.x < 73)
                J.pose->M[threadIdx.x - 64] = projection_element(J.a.K, st->Rp, (int)threadIdx.x - 64);
            else if (threadIdx.x >= 73 && threadIdx.x < 76)
                J.pose->tp[threadIdx.x - 73] = st->tp[threadIdx.x - 73];
        }
        if (threadIdx.x < 64) {
            word = finish_iteration(word, tot, count, st, true, stop_angle, stop_dist);
            if (!final_) {
                bool run;
                word = open_iteration(word, level, J.a.stride, &run);
                if (threadIdx.x < 9) J.pose->R[threadIdx.x] = __int_as_float(word);
                else if (threadIdx.x < 12) J.pose->t[threadIdx.x - 9] = __int_as_float(word);
            } else {
                commit_state(st, word);
                if (threadIdx.x == kWordPending) word = 0;
            }
            if (threadIdx.x < kCarryWords) reinterpret_cast<int*>(J.carry)[threadIdx.x] = word;
        }
    }
}

// A lane takes its pixels one after the other, the next one's loads issued ahead, so
// that few registers (84) hold them and other waves fill the waits: with its four
// pixels' loads in flight together the kernel held 102 and had four waves per SIMD.
// Five workgroups per CU resident, as many launched.  On average over the 19 iterations
// of a tick of 64 sessions 141 -> 135 us (22 -> 20.5 at 160x120, 77 -> 68 at 320x240,
// 221 -> 215 at 640x480, whose maps come at 4.4 TB/s), of 16 uneven sessions 26.8 ->
// 26.3; nothing issued ahead (70 registers, six waves) took 0.5 us more of the one and
// 0.3 of the other, two pixels at a time (96 registers) 3.5 and 1.
template <bool COMP>
__global__ __launch_bounds__(kThreads, 5) void icp_batch_assoc_kernel(const BatchHeader* hd, const IcpJob* jobs,
                                                                   int level)
{
    const int njobs = hd->n_icp, total = hd->icp_blocks[level];
    const int G = (int)gridDim.x;
    const int rank = xcd_rank((int)blockIdx.x, G);
    const int chunk = (total + G - 1) / G;
    int b = rank * chunk;
    const int end = min(total, b + chunk);
    if (b >= end) return;
    // the table, the carries and the iteration's poses are never written while the
    // kernel runs: scalar loads through the constant address space keep them in
    // scalar registers
    typedef __attribute__((address_space(4))) const IcpJob ConstJob;
    typedef __attribute__((address_space(4))) const IcpCarry ConstCarry;
    typedef __attribute__((address_space(4))) const IterPose ConstPose;
    ConstJob* cj = (ConstJob*)jobs;
    int j = job_of(jobs, njobs, b, [](const IcpJob& J) { return J.block0; });
    for (; b < end; ++b) {
        while (j + 1 < njobs && cj[j + 1].block0 <= b) ++j;
        j = __builtin_amdgcn_readfirstlane(j);
        if (!((ConstCarry*)cj[j].carry)->pending) continue;
        IcpArgs a;
        a.V = cj[j].a.V;
        a.TV = cj[j].a.TV;
        a.TN = cj[j].a.TN;
        a.w = cj[j].a.w;
        a.h = cj[j].a.h;
        a.dist_thresh = cj[j].a.dist_thresh;
        a.cos_thresh = cj[j].a.cos_thresh;
        a.partials = cj[j].partials;
        a.stride = cj[j].a.stride;
        a.pix = cj[j].a.pix;
        const int lb = b - cj[j].block0;
        ConstPose* cp = (ConstPose*)cj[j].pose;
        IterPose P;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            P.R[q] = cp->R[q];
            P.M[q] = cp->M[q];
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            P.t[q] = cp->t[q];
            P.tp[q] = cp->tp[q];
        }
        float s[kTerms];
#pragma unroll
        for (int q = 0; q < kTerms; ++q) s[q] = 0.0f;
        int cnt = 0;  // of the wave
        int px = lb * a.pix * kThreads + (int)threadIdx.x;
        float4 c, r, d;
        bool ok;
        issue_pixel_loads(a, px, c, r, d, ok);
#pragma unroll 1
        for (int k = 0; k < a.pix; ++k) {
            const PixelIn in = icp_pixel_from(c, r, d, ok);
            px += kThreads;
            if (k + 1 < a.pix) issue_pixel_loads(a, px, c, r, d, ok);
            const PixelGather g = icp_pixel_gather<true>(a, in, P);
            float row[6], rb;
            const bool hit = icp_pixel_finish(a, in, g, P.R, row, rb);
            cnt += __popcll(__ballot(hit));
            if (hit) accumulate(s, row, rb);
        }
        __syncthreads();  // the previous block's reduction LDS is free again
        block_reduce_store<typename SumType<COMP>::T>(s, cnt, a.partials, a.stride, lb);
    }
}

inline int blocks_for(int64_t n, int pix = kPixPerThread)
{
    return (int)((n + (int64_t)kThreads * pix - 1) / ((int64_t)kThreads * pix));
}

}  // namespace

// Pixels per lane of an iteration launch over an n-pixel map: the most (4, 2
// or 1) that still gives kFillBlocks workgroups, else 1.  An iteration's
// association is one lane's pixels in sequence, so a coarse level spread over
// more workgroups ends sooner.  A function of n alone: the batch and the
// single-session loop choose alike and sum the same partial rows.
int icp_pix_for(int64_t n)
{
    constexpr int kFillBlocks = 256;
    for (int pix = kPixPerThread; pix > 1; pix >>= 1)
        if (blocks_for(n, pix) >= kFillBlocks) return pix;
    return 1;
}
int64_t icp_max_map_pixels() { return kMaxMapPixels; }
int icp_level_blocks(int w, int h)
{
    const int64_t n = (int64_t)w * h;
    return blocks_for(n, icp_pix_for(n));
}
int icp_blocks_for(int w, int h)
{
    int m = 0;
    for (int l = 0; l < 3; ++l) m = std::max(m, icp_level_blocks(std::max(w >> l, 1), std::max(h >> l, 1)));
    return m;
}

static IcpCarry* carry_of(kf_icp* icp, int k) { return reinterpret_cast<IcpCarry*>(icp->carry) + (k & 1); }
static float* partials_of(kf_icp* icp, int k)
{
    return icp->partials + (size_t)(k & 1) * kPartialStride * (size_t)icp->max_blocks;
}

IcpCarry* icp_first_carry(kf_icp* icp) { return carry_of(icp, 0); }

int launch_icp_begin(kf_icp* icp, const float* pose16, hipStream_t s)
{
    Pose16 p;
    memcpy(p.m, pose16, sizeof(p.m));
    icp_begin_kernel<<<1, 64, 0, s>>>(icp->state, carry_of(icp, 0), p);
    KF_LAUNCHED("icp_begin_kernel");
    return KF_OK;
}

static IcpArgs level_args(const kf_icp* icp, const IcpLevel& L, int l)
{
    IcpArgs a{};
    a.V = L.V;
    a.TV = L.TV;
    a.TN = L.TN;
    a.w = L.w;
    a.h = L.h;
    memcpy(a.K, L.K, sizeof(a.K));
    a.dist_thresh = icp->cfg.distance_thresh;
    a.cos_thresh = icp->cos_thresh;
    a.st = icp->state;
    a.level = l;
    a.pix = icp_pix_for((int64_t)L.w * L.h);
    a.stride = blocks_for((int64_t)L.w * L.h, a.pix);
    return a;
}

// Enqueues the iteration launches and the commit; `before_commit` (optional) is
// recorded between them.  Returns the number of iterations in *launches.
static int enqueue_steps(kf_icp* icp, const IcpLevel* levels, int n_levels, hipStream_t s, hipEvent_t before_commit,
                         int* launches)
{
    const float sa = icp->cfg.iteration_stop_thresh_angle, sd = icp->cfg.iteration_stop_thresh_distance;
    int k = 0, prev_blocks = 0;  // row count of the previous launch (0: none this frame)
    for (int l = n_levels - 1; l >= 0; --l)
        for (int it = 0; it < icp->cfg.iters_per_layer[l]; ++it, ++k) {
            IcpArgs a = level_args(icp, levels[l], l);
            a.partials = partials_of(icp, k);
            const int blocks = a.stride;
            if (blocks > icp->max_blocks || (int64_t)a.w * a.h > kMaxMapPixels)
                return fail(KF_ERR_DIMS, "ICP: map larger than the configured width x height");
            using Step = void (*)(IcpArgs, const IcpCarry*, IcpCarry*, const float*, int, float, float);
            const Step steps[2][3] = {{icp_step_kernel<false, 1>, icp_step_kernel<false, 2>, icp_step_kernel<false, 4>},
                                      {icp_step_kernel<true, 1>, icp_step_kernel<true, 2>, icp_step_kernel<true, 4>}};
            const Step step = steps[icp->cfg.compensated ? 1 : 0][a.pix == 4 ? 2 : a.pix == 2 ? 1 : 0];
            step<<<blocks, kThreads, 0, s>>>(a, carry_of(icp, k), carry_of(icp, k + 1), partials_of(icp, k + 1),
                                             prev_blocks, sa, sd);
            KF_LAUNCHED("icp_step_kernel");
            prev_blocks = blocks;
        }
    if (before_commit) KF_HIP(hipEventRecord(before_commit, s));
    if (icp->cfg.compensated)
        icp_commit_kernel<true><<<1, kThreads, 0, s>>>(icp->state, carry_of(icp, k), partials_of(icp, k + 1), prev_blocks, sa, sd);
    else
        icp_commit_kernel<false><<<1, kThreads, 0, s>>>(icp->state, carry_of(icp, k), partials_of(icp, k + 1), prev_blocks, sa, sd);
    KF_LAUNCHED("icp_commit_kernel");
    if (launches) *launches = k;
    return KF_OK;
}

int launch_icp_loop(kf_icp* icp, const IcpLevel* levels, int n_levels, hipStream_t s)
{
    return enqueue_steps(icp, levels, n_levels, s, nullptr, nullptr);
}

int launch_icp_batch(const BatchHeader* hd, const IcpJob* jobs, const int* iters, int levels, int max_sessions,
                     int compensated, float stop_angle, float stop_dist, unsigned step_blocks, hipStream_t s)
{
    if (max_sessions <= 0) return KF_OK;
    icp_batch_begin_kernel<<<(unsigned)std::min(max_sessions, 1024), 64, 0, s>>>(hd, jobs);
    KF_LAUNCHED("icp_batch_begin_kernel");
    const IcpJob* level_jobs[3] = {jobs, jobs + max_sessions, jobs + 2 * max_sessions};
    const unsigned sb = (unsigned)std::min(max_sessions, 1024);
    for (int l = levels - 1; l >= 0; --l)
        for (int it = 0; it < iters[l]; ++it) {
            if (compensated) {
                icp_batch_solve_kernel<true><<<sb, kThreads, 0, s>>>(hd, level_jobs[l], l, 0, stop_angle, stop_dist);
                icp_batch_assoc_kernel<true><<<step_blocks, kThreads, 0, s>>>(hd, level_jobs[l], l);
            } else {
                icp_batch_solve_kernel<false><<<sb, kThreads, 0, s>>>(hd, level_jobs[l], l, 0, stop_angle, stop_dist);
                icp_batch_assoc_kernel<false><<<step_blocks, kThreads, 0, s>>>(hd, level_jobs[l], l);
            }
            KF_LAUNCHED("icp_batch_assoc_kernel");
        }
    if (compensated)
        icp_batch_solve_kernel<true><<<sb, kThreads, 0, s>>>(hd, jobs, 0, 1, stop_angle, stop_dist);
    else
        icp_batch_solve_kernel<false><<<sb, kThreads, 0, s>>>(hd, jobs, 0, 1, stop_angle, stop_dist);
    KF_LAUNCHED("icp_batch_solve_kernel");
    return KF_OK;
}

// ---- LinearLeastSquares::solve without allocation (kf_solve_normal_equations_noalloc).
// Its working memory -- the PoseState the solve writes and the per-block partial
// rows -- lives in one file-scope device array, `scratch`, of kNoAllocBytes on
// every GPU that runs it (held until the process ends).  Host code reaches a
// device's copy only through the address hipGetSymbolAddress returns for it
// (noalloc_scratch); the array's name is a host-side stand-in, not a device
// address.  Every call on a GPU shares that GPU's copy.
constexpr unsigned kNoAllocMaxEquations = 1u << 22;
constexpr int kNoAllocMaxBlocks = (int)((kNoAllocMaxEquations + kThreads * kPixPerThread - 1) /
                                        (kThreads * kPixPerThread));
constexpr size_t kNoAllocStateBytes = (sizeof(PoseState) + 255) & ~(size_t)255;
constexpr size_t kNoAllocBytes = kNoAllocStateBytes + sizeof(float) * kPartialStride * kNoAllocMaxBlocks;

__global__ void noalloc_result_kernel(const PoseState* st, float* x, int* status)
{
    if (threadIdx.x < 6) x[threadIdx.x] = st->last_x[threadIdx.x];
    if (threadIdx.x == 0 && status) *status = st->status;
}

}  // namespace kf

static __device__ __align__(256) unsigned char scratch[kf::kNoAllocBytes];
// A second one, for the calls that wait (kf_solve_normal_equations): a call that finds
// it in use by another thread allocates instead.
static __device__ __align__(256) unsigned char solve_scratch[kf::kNoAllocBytes];

namespace {

constexpr int kMaxDevices = 64;
std::atomic<bool> solve_scratch_used[kMaxDevices];
// Where a solve with solve_scratch leaves its result: 28 bytes of pinned host memory per
// GPU, allocated at its first use and, like the scratch, held until the process ends.
// Null where it could not be had (the result is copied then).  Called by the scratch's
// holder only.
kf::SolveResult* solve_result(int dev)
{
    static kf::SolveResult* ptr[kMaxDevices] = {};
    if (!ptr[dev] && hipHostMalloc(reinterpret_cast<void**>(&ptr[dev]), sizeof(kf::SolveResult), hipHostMallocDefault) !=
                         hipSuccess) {
        (void)hipGetLastError();
        ptr[dev] = nullptr;
    }
    return ptr[dev];
}

// The device address of this GPU's `scratch` or `solve_scratch`, looked up once per device.
int scratch_address(bool solve, char** out, int* device)
{
    static std::mutex mu;
    static char* ptr[2][kMaxDevices] = {};
    int dev = 0;
    KF_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return kf::fail(KF_ERR_ARG, "solve (no allocation): device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    char*& known = ptr[solve ? 1 : 0][dev];
    if (!known) {
        void* p = nullptr;
        hipError_t e = solve ? hipGetSymbolAddress(&p, HIP_SYMBOL(solve_scratch))
                             : hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return kf::fail_hip(e, "solve (no allocation): scratch address");
        known = static_cast<char*>(p);
    }
    *out = known;
    *device = dev;
    return KF_OK;
}

}  // namespace

// ------------------------------------------------------------------ C ABI
extern "C" {

int kf_construct_icp_residuals(const float* vertex_map, const float* target_vertex_map, const float* target_normal_map,
                               int w, int h, const float prev_rot[9], const float prev_transl[3],
                               const float cur_rot[9], const float cur_transl[3], const float intrinsics[9],
                               float distance_thresh, float angle_thresh, float* mat_a, float* vec_b,
                               kf_stream_t stream, float* elapsed_ms)
{
    if (!vertex_map || !target_vertex_map || !target_normal_map || !mat_a || !vec_b || w <= 0 || h <= 0 || !prev_rot ||
        !prev_transl || !cur_rot || !cur_transl || !intrinsics)
        return kf::fail(KF_ERR_ARG, "constructIcpResiduals: bad argument");
    hipStream_t s = kf::stream_of(stream);
    kf::IterPose P;  // passed by value
    memcpy(P.R, cur_rot, sizeof(P.R));
    memcpy(P.t, cur_transl, sizeof(P.t));
    for (int e = 0; e < 9; ++e) P.M[e] = kf::projection_element(intrinsics, prev_rot, e);
    memcpy(P.tp, prev_transl, sizeof(P.tp));
    kf::IcpArgs a{};
    a.V = reinterpret_cast<const float4*>(vertex_map);
    a.TV = reinterpret_cast<const float4*>(target_vertex_map);
    a.TN = reinterpret_cast<const float4*>(target_normal_map);
    a.w = w;
    a.h = h;
    a.dist_thresh = distance_thresh;
    a.cos_thresh = (float)cos((double)angle_thresh);
    kf::CallTimer t(elapsed_ms, s);
    int st = t.start();
    if (st == KF_OK) {
        const unsigned blocks = (unsigned)(((int64_t)w * h + kf::kThreads - 1) / kf::kThreads);
        kf::icp_rows_kernel<<<blocks, kf::kThreads, 0, s>>>(a, P, mat_a, vec_b);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) st = kf::fail_hip(e, "icp_rows_kernel");
    }
    if (st == KF_OK) st = t.finish();
    const hipError_t e = hipStreamSynchronize(s);
    if (st == KF_OK && e != hipSuccess) st = kf::fail_hip(e, "constructIcpResiduals");
    return st;
}

// Shared by kf_solve_normal_equations and kf_icp_reduce: partial rows -> sums/solve.
static int reduce_to_state(kf::PoseState** st_out, float** partials_out, int blocks)
{
    KF_HIP(hipMalloc(st_out, sizeof(kf::PoseState)));
    KF_HIP(hipMalloc(partials_out, sizeof(float) * kf::kPartialStride * (size_t)(blocks > 0 ? blocks : 1)));
    return KF_OK;
}

int kf_solve_normal_equations(const float* mat_a, const float* vec_b, unsigned int n_equations, float result[6],
                              kf_stream_t stream, float* elapsed_ms)
{
    if (!mat_a || !vec_b || !result || n_equations == 0)
        return kf::fail(KF_ERR_ARG, "LinearLeastSquares::solve: bad argument");
    hipStream_t s = kf::stream_of(stream);
    const int blocks = kf::blocks_for(n_equations);
    kf::PoseState* st = nullptr;
    float* partials = nullptr;
    char* base = nullptr;
    kf::SolveResult* pinned = nullptr;
    int dev = 0, rc = KF_OK;
    const bool shared = n_equations <= kf::kNoAllocMaxEquations && scratch_address(true, &base, &dev) == KF_OK &&
                        !solve_scratch_used[dev].exchange(true, std::memory_order_acquire);
    if (shared) {
        pinned = solve_result(dev);
        st = reinterpret_cast<kf::PoseState*>(base);
        partials = reinterpret_cast<float*>(base + kf::kNoAllocStateBytes);
    } else {
        rc = reduce_to_state(&st, &partials, blocks);
    }
    kf::CallTimer t(elapsed_ms, s);
    if (rc == KF_OK) rc = t.start();
    if (rc == KF_OK) {
        kf::ab_reduce_kernel<false><<<blocks, kf::kThreads, 0, s>>>(mat_a, vec_b, n_equations, partials, blocks, st);
        kf::icp_finalize_kernel<false><<<1, kf::kThreads, 0, s>>>(st, partials, blocks, blocks, pinned);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = kf::fail_hip(e, "solve kernels");
    }
    if (rc == KF_OK) rc = t.finish();
    kf::SolveResult r{};
    if (rc == KF_OK) {
        kf::PoseState hs;
        hipError_t e = pinned ? hipSuccess : hipMemcpyAsync(&hs, st, sizeof(hs), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            rc = kf::fail_hip(e, "solve readback");
        } else if (pinned) {
            r = *pinned;
        } else {
            memcpy(r.x, hs.last_x, sizeof(r.x));
            r.status = hs.status;
        }
    }
    if (rc == KF_OK) {
        for (int q = 0; q < 6; ++q) result[q] = r.x[q];
        if (r.status) rc = kf::fail(r.status, kf_status_string(r.status));
    } else {
        (void)hipStreamSynchronize(s);  // nothing uses the working memory past this call
    }
    if (shared) {
        solve_scratch_used[dev].store(false, std::memory_order_release);
    } else {
        (void)hipFree(st);
        (void)hipFree(partials);
    }
    return rc;
}

int kf_solve_normal_equations_noalloc(const float* mat_a, const float* vec_b, unsigned int n_equations,
                                      float* result_dev, int* status_dev, kf_stream_t stream)
{
    if (!mat_a || !vec_b || !result_dev || n_equations == 0)
        return kf::fail(KF_ERR_ARG, "solve (no allocation): bad argument");
    if (n_equations > kf::kNoAllocMaxEquations)
        return kf::fail(KF_ERR_ARG, "solve (no allocation): more than 2^22 equations");
    char* base = nullptr;
    int dev = 0;
    int rc = scratch_address(false, &base, &dev);
    if (rc) return rc;
    auto* st = reinterpret_cast<kf::PoseState*>(base);
    auto* partials = reinterpret_cast<float*>(base + kf::kNoAllocStateBytes);
    hipStream_t s = kf::stream_of(stream);
    const int blocks = kf::blocks_for(n_equations);
    kf::ab_reduce_kernel<false><<<blocks, kf::kThreads, 0, s>>>(mat_a, vec_b, n_equations, partials, blocks, st);
    kf::icp_finalize_kernel<false><<<1, kf::kThreads, 0, s>>>(st, partials, blocks, blocks, nullptr);
    kf::noalloc_result_kernel<<<1, 64, 0, s>>>(st, result_dev, status_dev);
    KF_HIP(hipGetLastError());
    return KF_OK;
}

int kf_icp_reduce(const float* vertex_map, const float* target_vertex_map, const float* target_normal_map, int w,
                  int h, const float prev_rot[9], const float prev_transl[3], const float cur_rot[9],
                  const float cur_transl[3], const float intrinsics[9], float distance_thresh, float angle_thresh,
                  int compensated, double sums_host[27], int64_t* inliers, kf_stream_t stream, float* elapsed_ms)
{
    if (!vertex_map || !target_vertex_map || !target_normal_map || !sums_host || w <= 0 || h <= 0)
        return kf::fail(KF_ERR_ARG, "kf_icp_reduce: bad argument");
    if ((int64_t)w * h > kf::kMaxMapPixels) return kf::fail(KF_ERR_DIMS, "kf_icp_reduce: map above 2^24 pixels");
    hipStream_t s = kf::stream_of(stream);
    const int blocks = kf::blocks_for((int64_t)w * h);
    kf::PoseState* st = nullptr;
    float* partials = nullptr;
    int rc = reduce_to_state(&st, &partials, blocks);
    kf::PoseState hs;
    memset(&hs, 0, sizeof(hs));
    memcpy(hs.R, cur_rot, sizeof(hs.R));
    memcpy(hs.t, cur_transl, sizeof(hs.t));
    memcpy(hs.Rp, prev_rot, sizeof(hs.Rp));
    memcpy(hs.tp, prev_transl, sizeof(hs.tp));
    if (rc == KF_OK) {
        hipError_t e = hipMemcpy(st, &hs, sizeof(hs), hipMemcpyHostToDevice);
        if (e != hipSuccess) rc = kf::fail_hip(e, "kf_icp_reduce state");
    }
    kf::IcpArgs a{};
    a.V = reinterpret_cast<const float4*>(vertex_map);
    a.TV = reinterpret_cast<const float4*>(target_vertex_map);
    a.TN = reinterpret_cast<const float4*>(target_normal_map);
    a.w = w;
    a.h = h;
    memcpy(a.K, intrinsics, sizeof(a.K));
    a.dist_thresh = distance_thresh;
    a.cos_thresh = (float)cos((double)angle_thresh);
    a.st = st;
    a.level = 0;
    a.partials = partials;
    a.stride = blocks;
    kf::CallTimer t(elapsed_ms, s);
    if (rc == KF_OK) rc = t.start();
    if (rc == KF_OK) {
        if (compensated) {
            kf::icp_reduce_kernel<true><<<blocks, kf::kThreads, 0, s>>>(a);
            kf::icp_finalize_kernel<true><<<1, kf::kThreads, 0, s>>>(st, partials, blocks, blocks, nullptr);
        } else {
            kf::icp_reduce_kernel<false><<<blocks, kf::kThreads, 0, s>>>(a);
            kf::icp_finalize_kernel<false><<<1, kf::kThreads, 0, s>>>(st, partials, blocks, blocks, nullptr);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = kf::fail_hip(e, "kf_icp_reduce kernels");
    }
    if (rc == KF_OK) rc = t.finish();
    if (rc == KF_OK) {
        hipError_t e = hipMemcpyAsync(&hs, st, sizeof(hs), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) rc = kf::fail_hip(e, "kf_icp_reduce readback");
    }
    if (rc == KF_OK) {
        for (int q = 0; q < 27; ++q) sums_host[q] = hs.last_sums[q];
        if (inliers) *inliers = hs.last_inliers;
    }
    (void)hipFree(st);
    (void)hipFree(partials);
    return rc;
}

int kf_icp_create(const kf_icp_config* config, kf_icp** out)
{
    if (!config || !out) return kf::fail(KF_ERR_ARG, "kf_icp_create: null argument");
    *out = nullptr;
    if (config->levels < 1 || config->levels > 3 || config->width <= 0 || config->height <= 0)
        return kf::fail(KF_ERR_ARG, "kf_icp_create: levels must be 1..3 and sizes positive");
    if ((int64_t)config->width * config->height > kf::icp_max_map_pixels())
        return kf::fail(KF_ERR_DIMS, "kf_icp_create: width x height above 2^24 pixels");
    for (int l = 0; l < config->levels; ++l)
        if (config->iters_per_layer[l] < 0) return kf::fail(KF_ERR_ARG, "kf_icp_create: negative iteration count");
    kf_icp* icp = new kf_icp();
    icp->cfg = *config;
    icp->cos_thresh = (float)cos((double)config->angle_thresh);
    icp->max_blocks = kf::icp_blocks_for(config->width, config->height);
    hipError_t e;
    if ((e = hipMalloc(&icp->state, sizeof(kf::PoseState))) != hipSuccess ||
        (e = hipMemset(icp->state, 0, sizeof(kf::PoseState))) != hipSuccess ||
        (e = hipMalloc(&icp->carry, 2 * sizeof(kf::IcpCarry))) != hipSuccess ||
        (e = hipMemset(icp->carry, 0, 2 * sizeof(kf::IcpCarry))) != hipSuccess ||
        (e = hipMalloc(&icp->partials, 2 * sizeof(float) * kf::kPartialStride * (size_t)icp->max_blocks)) != hipSuccess ||
        (e = hipHostMalloc(reinterpret_cast<void**>(&icp->mirror), sizeof(kf::PoseMirror), hipHostMallocDefault)) !=
            hipSuccess ||
        (e = hipMemcpy(&icp->state->mirror, &icp->mirror, sizeof(icp->mirror), hipMemcpyHostToDevice)) != hipSuccess) {
        kf_icp_destroy(icp);
        return kf::fail_hip(e, "kf_icp_create");
    }
    memset(icp->mirror, 0, sizeof(*icp->mirror));
    // the first two are for timing only: no system-scope cache write-back when they complete
    for (int q = 0; q < 3; ++q)
        if ((e = hipEventCreateWithFlags(&icp->ev[q], q < 2 ? hipEventDisableSystemFence : hipEventDefault)) !=
            hipSuccess) {
            kf_icp_destroy(icp);
            return kf::fail_hip(e, "kf_icp_create");
        }
    *out = icp;
    return KF_OK;
}

int kf_icp_destroy(kf_icp* icp)
{
    if (!icp) return KF_OK;
    for (hipEvent_t v : icp->ev)
        if (v) (void)hipEventDestroy(v);
    if (icp->mirror) (void)hipHostFree(icp->mirror);
    (void)hipFree(icp->state);
    (void)hipFree(icp->carry);
    (void)hipFree(icp->partials);
    delete icp;
    return KF_OK;
}

int kf_icp_compute_pose(kf_icp* icp, const float* const vertex_pyr[], const float* const target_vertex_pyr[],
                        const float* const target_normal_pyr[], const kf_sensor* sensor, float pose_out[16],
                        kf_stream_t stream, float* elapsed_ms)
{
    if (!icp || !vertex_pyr || !target_vertex_pyr || !target_normal_pyr || !sensor || !pose_out)
        return kf::fail(KF_ERR_ARG, "ICP::computePose: null argument");
    hipStream_t s = kf::stream_of(stream);
    kf::IcpLevel lv[3];
    for (int l = 0; l < icp->cfg.levels; ++l) {
        lv[l].V = reinterpret_cast<const float4*>(vertex_pyr[l]);
        lv[l].TV = reinterpret_cast<const float4*>(target_vertex_pyr[l]);
        lv[l].TN = reinterpret_cast<const float4*>(target_normal_pyr[l]);
        lv[l].w = icp->cfg.width >> l;
        lv[l].h = icp->cfg.height >> l;
        memcpy(lv[l].K, sensor->intr[l], sizeof(lv[l].K));
    }
    // ICP::getExecutionTimes: times[0] = the iteration launches (association, reduction
    // and the solve of the previous iteration), times[1] = the final solve and commit.
    int rc = kf::launch_icp_begin(icp, sensor->pose, s);
    if (rc == KF_OK && hipEventRecord(icp->ev[0], s) != hipSuccess) rc = kf::fail(KF_ERR_HIP, "ICP event record");
    int k = 0;
    if (rc == KF_OK) rc = kf::enqueue_steps(icp, lv, icp->cfg.levels, s, icp->ev[1], &k);
    if (rc == KF_OK && hipEventRecord(icp->ev[2], s) != hipSuccess) rc = kf::fail(KF_ERR_HIP, "ICP event record");
    if (rc == KF_OK) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) rc = kf::fail_hip(e, "ICP readback");
    }
    if (rc == KF_OK) {
        const kf::PoseMirror& hs = *icp->mirror;
        icp->times[0] = icp->times[1] = 0.0f;
        if (k > 0) (void)hipEventElapsedTime(&icp->times[0], icp->ev[0], icp->ev[1]);
        (void)hipEventElapsedTime(&icp->times[1], icp->ev[1], icp->ev[2]);
        if (elapsed_ms) (void)hipEventElapsedTime(elapsed_ms, icp->ev[0], icp->ev[2]);
        icp->last_iterations = hs.iterations;
        // the last good estimate (the commit does not run on failure)
        float P[16] = {0};
        for (int c = 0; c < 3; ++c)
            for (int r = 0; r < 3; ++r) P[c * 4 + r] = hs.R[c * 3 + r];
        for (int r = 0; r < 3; ++r) P[12 + r] = hs.t[r];
        P[15] = 1.0f;
        memcpy(pose_out, P, sizeof(P));
        if (hs.status) rc = kf::fail(hs.status, kf_status_string(hs.status));
    }
    return rc;
}

int kf_icp_execution_times(const kf_icp* icp, float times[2])
{
    if (!icp || !times) return kf::fail(KF_ERR_ARG, "kf_icp_execution_times: null argument");
    times[0] = icp->times[0];
    times[1] = icp->times[1];
    return KF_OK;
}

int kf_icp_iterations(const kf_icp* icp, int* iterations)
{
    if (!icp || !iterations) return kf::fail(KF_ERR_ARG, "kf_icp_iterations: null argument");
    *iterations = icp->last_iterations;
    return KF_OK;
}

}  // extern "C"
