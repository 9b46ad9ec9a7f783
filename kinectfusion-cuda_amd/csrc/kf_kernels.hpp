// Launch interfaces shared between the library's translation units.  Each
// launcher enqueues kernels on `s` and returns a kf_status.
#pragma once

#include "kf_internal.hpp"

namespace kf {

// ---- measurement (measurement.hip)
int launch_convert(const uint16_t* raw, float* out, int w, int h, float scale, int unmirror, hipStream_t s);
int launch_bilateral(const float* in, float* out, int w, int h, hipStream_t s);
int launch_down_sample(const float* in, int w_in, int h_in, float* out, hipStream_t s);
int launch_vertex_map(const float* depth, float4* out, int w, int h, const float* inv_k, hipStream_t s);
int launch_normal_map(const float4* v, float4* out, int w, int h, hipStream_t s);

// Counters that the waves of different XCDs add to lie this many words apart: a
// returning atomic on a 128-byte line that the whole device shares completes one
// in 11 ns.
constexpr int kCountStride = 32;

// ---- batch ticks (batch.hip): one table per tick in device memory, a header
// followed by the job arrays of every stage.  Counts are per tick; the fuse
// brick list, its counter and the touched slots belong to the batch.
struct BatchHeader {
    int n_pre, pre_tiles, pyr_tiles;  // preprocess jobs, L0 16x16 tiles, L2 16x16 tiles
    int n_ray, ray_tiles;             // raycast jobs (session x level), 8x8 tiles, each job's padded to 8
    int n_ray_f32, ray_tiles_f32;     // the FP32-volume jobs come first: their count and tiles
    int n_icp, icp_blocks[3];         // ICP sessions, blocks per level
    int n_fuse;                       // fuse jobs
    unsigned fuse_groups;             // cubes of 4x4x4 bricks over all fuse jobs
    int dist_tiles;                   // free-distance tiles over all fuse jobs
    unsigned* fuse_count;
    unsigned long long* fuse_list;    // job << 32 | brick of the job's volume
    unsigned long long* touched;
    unsigned* ray_count;  // 16 deferred-ray counts (8 XCDs of the F32 jobs, then of the snorm16 jobs),
                          // kCountStride apart, cleared by the first kernel
    struct DeferredRay* ray_list;  // 16 lists of ray_list_cap deferred rays, in the same order
    unsigned ray_list_cap;
};

// Preprocess of one session: raw codes -> metres (fuse input), bilateral L0,
// pyramid and vertex maps of `levels` levels, normal maps on request.
struct PreJob {
    const uint16_t* raw;
    float* depth_m;
    float* d0;         // bilateral-filtered level 0
    float2* drange;    // tile depth ranges of depth_m (FuseArgs::drange layout; optional)
    float4* v[3];      // camera-space vertex maps
    float4* n[3];      // camera-space normal maps (all levels or none)
    float* d12[2];     // one session: filtered depth of levels 1 and 2 (optional)
    int w, h;
    int levels;        // one session: 1..3, w and h divisible by 2^(levels - 1); a batch tick's jobs have 3
    int unmirror;      // one session: nonzero reads row j of the frame right to left
    int late_regions;  // one session: drange's 64x64 ranges are formed later (RaycastSide)
    float scale;
    float Kinv[3][9];
    int tile0, tiles_x;    // level-0 16x16 tiles of this job
    int ptile0, ptiles_x;  // batch ticks: level-2 16x16 tiles of this job
};
int launch_preprocess_batch(const BatchHeader* hd, const PreJob* jobs, unsigned blocks, hipStream_t s);
// The measurement of one session (fills in J.tiles_x).
int launch_measure(PreJob& J, hipStream_t s);

// ---- TSDF (tsdf.hip)
constexpr unsigned kFuseBlocks = 2048;  // fuse workgroups: 256 CUs x 8 resident workgroups of 4 waves
struct FuseArgs {
    const float* depth;
    int w, h;
    float K[9];
    float inv_pose[16];
    const PoseState* dyn;  // when set: inv_pose comes from dyn->inv_pose, skip if dyn->frame_skip_fuse
    int n, nb;
    float half, res, mue;
    float inv_mue;  // 1 / mue correctly rounded (the exact reciprocal the quotient diff / mue is formed from)
    const float* zk;
    float4* zt;     // (m2 z + m3) per row of the inverse pose for each k slice, written by the fuse's cull
    float band;     // near-integer band of the projection (2^-21 max(w, h))
    void* f;
    void* wt;
    unsigned long long* touched;
    unsigned long long* free_bits;  // per-brick free bits (kf_device.hpp)
    uint8_t* dist;  // per-brick free distances, formed from free_bits after the sweep
    int cull;     // 1 when K is a plain pinhole matrix (culling planes valid)
    // lengths of the culling planes' normals |(fx, cx)|, |(fx, w - cx)|, |(fy, cy)|,
    // |(fy, h - cy)|, rounded up (they scale the bounding-sphere radius)
    float plane_norm[4];
    int format;   // kf_voxel_format
    // occlusion and free-space tests: (max valid depth, min depth) per 16x16 tile (tx16 x
    // ty16) followed by the same per 64x64 tile (tx64 x ty64), an invalid depth counting
    // as 0 in both; null = frustum test only
    const float2* drange;
    int tx16, ty16, tx64, ty64;
};
// Tiles of the depth ranges of a w x h depth map.
inline size_t depth_range_tiles(int w, int h)
{
    return (size_t)((w + 15) / 16) * ((h + 15) / 16) + (size_t)((w + 63) / 64) * ((h + 63) / 64);
}
struct FuseJob {
    FuseArgs a;       // a.dyn set: the session's committed pose
    unsigned group0;  // first global cube (4x4x4 bricks) of this job
    int dist_tile0;   // first 8x8-row tile of this job's free distances
};
// Cubes of 4x4x4 bricks of a volume, those at its far faces cut off by them.
inline unsigned fuse_groups(int nb) { return (unsigned)((nb + 3) / 4) * ((nb + 3) / 4) * ((nb + 3) / 4); }
// Words of a volume's free bits (free_word).
inline size_t free_words(int nb) { return (size_t)nb * nb * 2 * (nb > 64 ? 2 : 1); }
// Workgroups of a volume's free distances: one per 8x8 rows of bricks.
inline int dist_tiles(int nb) { return ((nb + 7) / 8) * ((nb + 7) / 8); }
FuseArgs fuse_args(const float* depth, int w, int h, const kf_volume* v, const float* K, const float* inv_pose,
                   const PoseState* dyn_state);
// mid (optional): an event recorded between the brick cull and the sweep.
int launch_fuse_batch(const BatchHeader* hd, const FuseJob* jobs, unsigned cull_blocks, unsigned list_blocks,
                      hipStream_t s, hipEvent_t mid = nullptr);
// inv_pose: by-value world->camera matrix; dyn_state (may be null) overrides it
// with PoseState::inv_pose and skips the launch's work when the frame failed.
// list_events (optional): two events recorded around the brick-list kernel alone.
// drange_ready: the volume's tile depth ranges (volume_depth_range) already hold this
// depth map's (the measurement pass wrote them).
int launch_fuse(const float* depth, int w, int h, kf_volume* v, const float* K, const float* inv_pose,
                const PoseState* dyn_state, hipStream_t s, hipEvent_t* list_events, bool drange_ready);
// Forms the volume's free distances on `s` if a fuse may have changed the free bits
// since they were formed: every raycast's first step.
int refresh_free_distances(const kf_volume* v, hipStream_t s);
// The volume's tile depth range buffer sized for w x h (grown if needed); null on failure.
float2* volume_depth_range(kf_volume* v, int w, int h, hipStream_t s);
int launch_initialize(kf_volume* v, float f, float wt, hipStream_t s);
// kf_volume_create without the host wait: initialisation is enqueued on `s`.
int volume_create(int n, float width_m, float mue_m, int format, hipStream_t s, kf_volume** out);

// ---- raycast (raycast.hip)
struct RaycastVolume {
    const void* f;
    const uint8_t* dist;     // per-brick free distances (kf_device.hpp)
    int n, nb, format;
    float width, mue;
    float inv_width;  // 1 / width correctly rounded
    int p2;           // width and n are powers of two (the march's texel coordinates are then exact)
};
struct RaycastLevel {
    float Kinv[9];
    float4* vout;
    float4* nout;
    int w, h, tiles_x, tile0;  // tile0: first global tile of this level (batch ticks: a multiple of 8)
};
// A ray the per-lane march handed to the finishing pass: its march state
// before the sample at t.
struct DeferredRay {
    int job;    // pyramid level (single launch) or raycast job (batch)
    int px;     // j * w + i
    int flags;  // bit 0: the last sample was skipped (prev comes from prev_t), bit 1: small steps
    float t, prev, prev_t, pad[2];
};
// One (session, level) of a batched raycast; lives in device memory.
struct RaycastJob {
    RaycastVolume vol;
    const float* pose;   // device: camera-to-world pose of the session (PoseState::pose)
    RaycastLevel L;
};
RaycastVolume raycast_volume(const kf_volume* v);
// blocks: workgroups of the first pass per voxel format, 0 (no jobs of that format)
// or a multiple of 8.  mid (optional): an event recorded between the first pass and
// the finishing pass.
int launch_raycast_batch(const BatchHeader* hd, const RaycastJob* jobs, const unsigned blocks[2], hipStream_t s,
                         hipEvent_t mid = nullptr);
int launch_raycast(const kf_volume* v, const float* pose, const PoseState* dyn_state, const float* inv_k,
                   float4* vout, float4* nout, int w, int h, hipStream_t s);
// What a frame needs between its measurement and its tracking, done beside the
// finishing pass by waves that seldom get a ray (a launch of its own takes 5 us): the
// ICP's start and the 64x64 depth ranges of the w x h frame.
struct RaycastSide {
    PoseState* begin;  // null: nothing to do
    struct IcpCarry* carry;
    float2* drange;
    int w, h;
};
// All pyramid levels in one launch (level l is w0 >> l by h0 >> l).
int launch_raycast_levels(const kf_volume* v, const float* pose, const PoseState* dyn_state, int levels,
                          const float (*inv_k)[9], float4* const* vout, float4* const* nout, int w0, int h0,
                          hipStream_t s, const RaycastSide* side = nullptr);

// ---- ICP (icp.hip)
constexpr int kPartialStride = 64;  // floats per block partial: 27 sums and the count, FP32 or FP64
struct IcpArgs {
    const float4* V;
    const float4* TV;
    const float4* TN;
    int w, h;
    float K[9];
    float dist_thresh, cos_thresh;
    PoseState* st;  // pose source (R, t, Rp, tp) and early-stop flags
    int level;
    float* partials;
    int stride;     // partial-row count of this launch (or of this job)
    int pix;        // pixels per lane (icp_pix_for of the map's pixel count)
};
// State carried from one ICP launch to the next (double-buffered by launch parity).
struct IcpCarry {
    float R[9];
    float t[3];
    int status;
    int level_done[4];
    int iterations;
    int pending;         // the writing launch left partial rows that still need their solve
    int pending_level;
    int pending_blocks;  // partial-row count of that launch
    int pad[2];
};
// What the association of an iteration needs of its pose: the current estimate
// R, t, the projection M = K R_prev^T and t_prev.
struct IterPose {
    float R[9], t[3], M[9], tp[3];
};
// Starts a frame's ICP by one wave: the working and previous poses are the sensor pose
// (icp.cpp:27-29), P (st->pose or the same by value).
__device__ __forceinline__ void icp_begin_state(PoseState* st, IcpCarry* c0, const float* P)
{
    constexpr int kWords = (int)(sizeof(IcpCarry) / sizeof(int));
    const int lane = threadIdx.x & 63, r = lane % 3, c = lane / 3;
    int word = 0;  // of the carried state
    if (lane < 12) {  // R column by column, then t
        const float v = P[c * 4 + r];
        word = __float_as_int(v);
        if (lane < 9) st->R[lane] = st->Rp[lane] = v;
        else st->t[r] = st->tp[r] = v;
    } else if (lane < 16) {
        st->level_done[lane - 12] = 0;
    } else if (lane == 16) {
        st->status = 0;
        st->iterations = 0;
        st->frame_skip_fuse = 0;
    }
    if (lane < kWords) reinterpret_cast<int*>(c0)[lane] = word;
}
// One session at one level of a batched ICP launch.
struct IcpJob {
    IcpArgs a;         // a.stride = the session's blocks at this level; a.partials unused
    IcpCarry* carry;   // 2 entries, by launch parity
    IterPose* pose;    // of the iteration, written by its solve launch
    float* partials;   // 2 x kPartialStride x max_blocks, by launch parity
    int max_blocks;
    int block0;        // first block of this job in the launch
};
struct IcpLevel {
    const float4* V;
    const float4* TV;
    const float4* TN;
    int w, h;
    float K[9];
};
int icp_pix_for(int64_t n);
int64_t icp_max_map_pixels();         // largest w x h an ICP map may have
int icp_level_blocks(int w, int h);  // workgroups of one iteration launch over a w x h map
int icp_blocks_for(int w, int h);    // the most of icp_level_blocks over the three levels of a w x h frame
// Enqueues the whole coarse-to-fine loop on `s` with the state on the device,
// ending with the commit of the estimate into state->pose / inv_pose.
int launch_icp_loop(kf_icp* icp, const IcpLevel* levels, int n_levels, hipStream_t s);
// begin: starts the frame's ICP from pose16 (from state->pose: RaycastSide);
// launch_icp_loop then enqueues one launch per iteration and the final commit.
int launch_icp_begin(kf_icp* icp, const float* pose16, hipStream_t s);
IcpCarry* icp_first_carry(kf_icp* icp);  // the state the first launch reads
// Batched: begin, then steps k = 0.. over the levels coarse to fine, then commit.
int launch_icp_batch(const BatchHeader* hd, const IcpJob* jobs, const int* iters, int levels, int max_sessions,
                     int compensated, float stop_angle, float stop_dist, unsigned step_blocks, hipStream_t s);

// ---- visualisation (render.hip)
int launch_render(const float4* nmap, int w, int h, const float* mat9, int shading, uint32_t* out, hipStream_t s);
void shading_matrix(const float* pose16, const float* kinv9, float* out9);

}  // namespace kf
