// kernels.hpp - device data layout shared by the kernels and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <algorithm>
#include <stddef.h>
#include <stdint.h>

#include "../../include/vkr.h"
#include "bvh.hpp"

namespace vkr {

constexpr uint32_t kMiss = 0xFFFFFFFFu;

// Everything a kernel needs of one uploaded scene (device pointers).
struct DevScene {
    const BvhNode* nodes;
    const TriRecord* tris;          // leaf order
    const float4* sph;              // leaf order: centre, r
    const uint32_t* sph_key;        // leaf order: sphere scan index
    const vkr_triangle* tris_orig;  // scan order (std430, as uploaded)
    const vkr_sphere* spheres;      // scan order
    const vkr_plane* planes;        // scan order
    const vkr_material* tri_material;
    const vkr_material* materials;
    const uint32_t* emitters;       // scan indices of spheres with emissive != 0
    uint32_t n_tris, n_spheres, n_planes, n_emitters;
    uint32_t n_materials, flags, has_bvh, stack_needed;
    uint32_t emitters_bounded;      // every emitter: |emissive| < 2^20, 2^-20 <= r <= 2^20
    float sph_c[3], sph_r;          // every sphere centre lies within sph_r of sph_c
    float sph_rmin;                 // the least radius
    // Scenes of a few primitives, traced by scanning (scan.hpp, use_scan).
    uint32_t scan;                  // 1: the scan records exist
    float scan_reach;               // sph_r + the largest radius
    const float4* scan_sph;         // scan order: centre, r * r; padded (kScanRun)
    const float4* scan_planes;      // scan order: N, len; padded
    const TriRecord* scan_tris;     // scan order
};

// A scene is scanned rather than traversed when its tests cost less than the
// rounds of a tree: by spheres + 2 * triangles (a triangle's test is about two
// spheres' work).  4 bounces, 2 spp, tree against scan on one MI355X:
//   single rays (one emitter), 1280x720: 5 spheres 257 / 239 us, 33: 320 / 299,
//   49: 359 / 354, 65: 372 / 390, 101: 400 / 485;
//   ray pool (about a quarter emit), 1280x720: 25 spheres 766 / 637 us, 65:
//   1934 / 1754, 101: 3188 / 3014, 161: 5490 / 6450, but 512x512: 101: 1651 /
//   1859;
//   7 spheres and 16 triangles 350 / 306 us, 30 triangles 374 / 344.
// Spheres and planes are read kScanRun at a time and padded to whole runs, plus
// one that is read ahead, with primitives no ray hits.
constexpr uint32_t kScanRun = 4u;
constexpr uint32_t kScanUnits = 56u;       // single rays
constexpr uint32_t kScanUnitsPool = 80u;   // ray pool
// Single-ray waves of at most kQuadWidth pixels scan with four lanes a pixel;
// kQuadUnits is part of the rule that gives a wave so few (ctx.hpp).
constexpr uint32_t kQuadWidth = 16u;
constexpr uint32_t kQuadUnits = 24u;
inline uint32_t scan_units(uint32_t spheres, uint32_t tris)
{
    return (uint32_t)std::min<uint64_t>((uint64_t)spheres + 2ull * tris, 0xFFFFFFFFull);
}
inline bool use_scan(const DevScene& sc, bool pool)
{
    return sc.scan != 0u && scan_units(sc.n_spheres, sc.n_tris) <= (pool ? kScanUnitsPool : kScanUnits);
}

// One frame of work (a single trace call, or one job of a batch).
struct JobDesc {
    DevScene sc;
    float cam_pos[3];
    float aspect;
    float cam_dir[3];
    float seed;
    float cam_right[3];
    float eps;
    float cam_up[3];
    uint32_t flags;               // VKR_TRACE_*
    float light_pos[3];           // FrameData.light_pos (read by the Whitted kernel only)
    uint32_t kernel;              // VKR_KERNEL_*
    uint32_t W, H, spp, max_depth;
    uint32_t tiles_x, n_tiles, pool_base, pad;
    uint8_t* rgba8;
    float* radiance;
    uint32_t* prim_id;
    float* hit_t;
    uint32_t* ray_count;
    uint16_t* decisions;
    uint2* adj_samples;           // W*H*spp, pixel-major: (bits of the random-stream position at the
                                  // sample's start, clamp-saturation bits) for the adjoint; NULL: none
    uint2* adj_primary;           // W*H: (primary hit's primitive, bits of its t) for the adjoint; NULL: none
};

// Atomics on one address are served one after the other, 11.5 ns each
// whatever the number of waves; on 64 lines they take 0.4 ns each.  So a
// launch counts into kCounterBanks copies of the counters, one cache line
// each (a workgroup adds to bank blockIdx % banks), and the host sums them.
struct alignas(128) DevCounters {
    unsigned long long rays, shadow, traced, nodes, tris, spheres, planes, overflow;
    unsigned long long wave_nodes, wave_leaves, wave_steps;
};
constexpr uint32_t kCounterBanks = 64u;   // a power of two
static_assert(sizeof(DevCounters) == 128, "one bank per 128-byte line");
struct CounterRef {
    DevCounters* banks;
    uint32_t mask;                // number of banks - 1
};


// Most work items one launch's 32-bit pool cursor hands out.  A resident
// wave can add up to 64 to the cursor after the last item has gone (its one
// claim that finds the pool empty), and items are numbered from the resident
// lanes up, so the numbers stay below 2^32 while the resident lanes number
// under 2^23.
constexpr uint64_t kMaxPoolItems = 0xFF000000ull;

// One-pixel-per-lane launches cover at most this many lanes each, which
// bounds their ray records (2^21 x kLaneBytes = 2.7 GB).
constexpr uint32_t kMaxPlainLanes = 1u << 21;

// Ray records of the pooled path kernel, in global memory: one block of
// kWaveBytes per wave (64 lanes), laid out field by field so that the lanes
// of a wave reading or writing one field touch contiguous addresses.  Field
// f of lane l is at f + 16 l; per-slot fields hold slot k of lane l at
// f + 16 (64 k + l) (salts: f + 4 (64 k + l)).  Slot 0 is the path segment,
// slots 1.. are emitters ei0 + k - 1 of a next-event window.
//   kWPark   4 x float4: path state parked while the wave evaluates and
//            traces (acc, u) (mask, v) (e, random-stream position) and, once
//            per pixel, (bits of the primary hit's primitive, its t, -, -),
//            at kWPark + 1024 i
//   kWHead   the origin xyz of this step's rays
//   kWSlotD  per slot: the ray's (d xyz, t_max)
//   kWSlotC  per slot: the next-event contribution (xyz, 0); slot 0 (a
//            segment has none) holds kWPix, the sum of the pixel's finished
//            samples (xyz)
//   kWHit    4 x float4: the diffuse hit published for the wave's
//            next-event evaluation: (N xyz, u), (albedo xyz, roughness),
//            (V xyz, metalness), (bits of the kNee* flags, v, bits of ei0, -);
//            V = normalize(camera - P) is the same for every emitter
//   kWSalt   per slot: the random stream position before that emitter's
//            sample
constexpr uint32_t kRaySlots = 32;
constexpr uint32_t kNeeSlots = kRaySlots - 1u;   // emitters of one window
constexpr uint32_t kWPark = 0u;
constexpr uint32_t kWHead = kWPark + 4u * 1024u;
constexpr uint32_t kWSlotD = kWHead + 1024u;
constexpr uint32_t kWSlotC = kWSlotD + kRaySlots * 1024u;
constexpr uint32_t kWPix = kWSlotC;
constexpr uint32_t kWHit = kWSlotC + kRaySlots * 1024u;
constexpr uint32_t kWSalt = kWHit + 4u * 1024u;
constexpr uint32_t kWaveBytes = kWSalt + kRaySlots * 256u;
constexpr uint32_t kLaneBytes = kWaveBytes / 64u;   // what one lane of a launch needs
static_assert(kWaveBytes % 64u == 0u, "a wave's records split evenly over its lanes");

struct PathLaunch {
    JobDesc job;                  // single-frame launches (first: the kernel finds it at its arguments' start)
    const JobDesc* jobs;          // batched launches, and captured ones of one job; else NULL
    const uint32_t* job_start;    // n_jobs + 1 pool offsets (batched)
    uint32_t n_jobs;
    uint32_t total;               // pool indices (64 per 8x8 tile)
    uint32_t persistent;          // 0: one pixel per lane; 1: refill from pool
    uint32_t rays_only;           // count rays, nothing else (the adjoint's first pass)
    uint32_t base;                // one pixel per lane: pool index of the launch's lane 0
    uint32_t chunk;               // refill when at least this many lanes idle
    uint32_t width;               // lanes of a wave that take pixels (the others only help with its rays)
    uint32_t* pool;               // persistent pool cursor (device)
    CounterRef counters;
    char* lanes;                  // ray records: one kWaveBytes block per wave of the grid
};

static_assert(offsetof(PathLaunch, job) == 0, "uniform_job reads it there");

// Adjoint launch (path replay), see adjoint.hip.
struct AdjointLaunch {
    JobDesc job;
    const float* d_radiance;      // W*H*4
    float* d_params;              // 7 * n_spheres + 1
    const float* params;          // 7 * n_spheres + 1 (current values)
    CounterRef counters;
    uint32_t* pool;               // the pool cursor of the second pass
    uint32_t total;               // pool indices (64 per 8x8 tile and sample)
    // The first pass's records (JobDesc::adj_samples, adj_primary).
    const uint2* samples;
    const uint2* primary;
};

// One instantiation of the path kernel.  pool: a wave traces up to
// kRaySlots rays per lane and step from a shared pool (pays off with several
// emitters); else one ray per lane and step.  Results are identical.
struct PathVariant {
    uint32_t block, stack;
    bool count, batch, pool;
    bool scan = false;   // every job's scene is scanned: no tree, no stack (stack is ignored)
};

// Default pool refill threshold: a wave claims new pixels once at least this
// many of its lanes are idle.  A claim is an atomic on one address, 11.5 ns
// after the one before it, and takes all waves' turn; lanes idle meanwhile.
// Against 8 (one MI355X):
//   one frame of a tree or with the ray pool: 1 to 32 within 2%, 48 and 64 3-15%
//   slower (1080p heightfield, 100k-triangle soup), so 8;
//   one ray a lane over a scanned scene costs so little a pixel that the claims
//   bound it: 64 takes the 1024^2 reference scene, 4 spp, from 1115 to 854 us
//   (16: 867, 32: 942), 1 spp 428 to 233, 33 spheres 720p 404 to 363.  That
//   ends where spp times bounces reaches 32 (1024x768 reference scene 8 spp, 4
//   bounces 1232 / 1228 us, 6 spp, 8 bounces 1140 / 1146, 8 spp, 8 bounces
//   1355 / 1422);
//   batches, whose jobs' pixels differ more: 32 takes 64 mixed scenes from 1482
//   to 1352 ms, eight soups 265 to 255, two heightfields 1809 to 1795 us.
inline uint32_t default_chunk(const PathVariant& v, uint32_t spp, uint32_t max_depth)
{
    if (v.scan && !v.pool && (uint64_t)spp * max_depth <= 32u) return 64u;
    return v.batch ? 32u : 8u;
}

hipError_t launch_path(const PathLaunch& a, const PathVariant& v, uint32_t grid, hipStream_t s);
hipError_t launch_whitted(const JobDesc& j, CounterRef c, hipStream_t s);
hipError_t launch_filter(const uint8_t* cur, const uint8_t* prev, uint32_t sw, uint32_t sh, uint8_t* out,
                         uint32_t dw, uint32_t dh, hipStream_t s);
// The adjoint's second pass; a.samples and a.primary hold the first pass's
// records of this frame.  scan: the scene is scanned (use_scan).
hipError_t launch_adjoint(const AdjointLaunch& a, uint32_t stack, bool scan, hipStream_t s);
hipError_t launch_debug(uint32_t op, const float* in, float* out, uint32_t n, hipStream_t s);
hipError_t launch_zero_counters(CounterRef c, uint32_t* pool, hipStream_t s);
// Writes the per-frame fields of a job in a device job table (camera,
// aspect, seed, light position), in stream order.
hipError_t launch_set_frame(JobDesc* job, const vkr_frame_data& fd, hipStream_t s);
uint32_t compute_units(int device);
// Occupancy-derived persistent grid size for (block, stack).
uint32_t persistent_grid(const PathVariant& v, int device);

// The static scratch of vkr_trace_frame_static: counters at offset 0, the
// pool cursor at kStaticPoolOff, per-lane ray records from kStaticLanesOff.
constexpr size_t kStaticPoolOff = 256;
constexpr size_t kStaticLanesOff = 512;
constexpr size_t kStaticScratchBytes = kStaticLanesOff + (size_t)VKR_STATIC_SCRATCH_LANE_BYTES;
static_assert(sizeof(DevCounters) <= kStaticPoolOff, "counters fit below the pool cursor");
// Device address of this device's static scratch (looked up once per device
// with that device current, then cached).
hipError_t static_scratch(int device, char** out);
// Largest stack depth with a compiled kernel variant (0 when none fits).
uint32_t stack_variant(uint32_t needed);

// Device build of a triangle subtree (lbvh.hip): internal nodes go to
// d_nodes[node_off .. node_off + n - 2] (its root at node_off), one record
// per triangle to d_recs (Morton order; a leaf is a run of at most max_leaf
// records).  Returns, after a stream synchronisation, the subtree's height
// (its deepest leaf, the root's children at 1), its live node and leaf
// counts, and the exact bounds of the padded triangle boxes.  A tree higher
// than height_cap is rejected after its topology: only the height and counts
// are returned and the nodes' boxes and the records are not written.
struct LbvhRoot {
    float lo[3], hi[3];
    uint32_t height, nodes, leaves;
};
// Device scratch a build over n triangles needs (0 when n < 2); the caller
// passes at least that much to lbvh_build and may reuse it across builds.
size_t lbvh_scratch_bytes(uint32_t n);
hipError_t lbvh_build(const vkr_triangle* d_tris, uint32_t n, uint32_t node_off, uint32_t max_leaf,
                      uint32_t height_cap, void* scratch, size_t scratch_bytes, BvhNode* d_nodes, TriRecord* d_recs,
                      LbvhRoot* root, hipStream_t s);

}  // namespace vkr
