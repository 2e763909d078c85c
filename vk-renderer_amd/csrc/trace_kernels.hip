// trace_kernels.hip - gfx950 kernels for the vk-renderer compute path tracer.
//
// The reference (Assets/Tracer.comp) runs one invocation per pixel that
// loops SAMPLES paths of up to DEPTH bounces and scans every primitive
// linearly per ray.  Here:
//   * each lane runs one pixel as a small state machine; in every loop
//     iteration a lane at a diffuse vertex queues the shadow rays of up to
//     kNeeSlots emitters (with their contributions, evaluated first) and,
//     with the last of them, the next path segment, and the wave traces all
//     queued rays from a shared pool: a lane whose ray ends takes the next
//     one, so the wave waits for its total work, not for its longest lane;
//   * persistent waves refill idle lanes from a global pixel pool with one
//     wave-wide ballot + one atomic per refill (8x8 tiles in pool order);
//   * the linear scan is replaced by a BVH (two child boxes per 64-byte node,
//     128-bit loads) with a short per-lane stack in LDS;
//   * the reference's order-dependent acceptance rule
//     (`t > EPSILON && t < best + EPSILON` for triangles then spheres,
//     `t < best - EPSILON` for planes, Tracer.comp:378-428) is reproduced
//     exactly: the smallest hit t* is always accepted by the scan, so only
//     hits within a window above t* can still change the winner; they are
//     kept in a 4-entry list and replayed in scan order after traversal.
//     A window or list overflow is counted (documented near-tie).
#include <hip/hip_runtime.h>

#include <mutex>

#include "kernels.hpp"
#include "nee.hpp"
#include "scan.hpp"
#include "traverse.hpp"
#include "vkr_device.hpp"

namespace vkr {

// The job of a launch that has one: A.jobs in device memory (a captured graph's,
// whose frame data is replaced between replays) or A.job among the kernel's
// arguments (PathLaunch starts with it).  Constant memory through scalar
// loads; `at` is opaque, so a field is loaded where it is used and does not
// sit in scalar registers across the whole loop (some 140 of them were
// spilled).
__device__ __forceinline__ const JobDesc& uniform_job(unsigned long long at)
{
    asm volatile("" : "+s"(at));
    return *(const JobDesc*)reinterpret_cast<const __attribute__((address_space(4))) JobDesc*>(at);
}

// Runs body(job, mine) with a uniform job: once for a launch of one job, else
// once for each job that the wave's lanes hold (one, but for the waves at a
// job's edge); mine: the lane's own.  All lanes run it.  With a job of its own
// in every lane instead, the scene's pointers would be per-lane values that
// each node fetch loads, or holds eight registers for.
template <bool BATCH, class Body>
__device__ __forceinline__ void for_each_job(const PathLaunch& A, unsigned long long job_at, uint32_t job, bool active,
                                             Body&& body)
{
    if constexpr (!BATCH) {
        body(uniform_job(job_at), true);
    } else {
        unsigned long long todo = __ballot(active);
        while (todo) {
            const uint32_t j = (uint32_t)__builtin_amdgcn_readlane((int)job, __builtin_ctzll(todo));
            const bool mine = active && job == j;
            todo &= ~__ballot(mine);
            const unsigned long long at = (unsigned long long)(A.jobs + j);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32));
            body(uniform_job(((unsigned long long)hi << 32) | lo), mine);
        }
    }
}

// The path program of Assets/Tracer.comp:433-593 as a per-lane state machine.
// Each loop iteration takes every lane one vertex further:
//   (1) refill idle lanes (their first ray is the primary one);
//   (2) lanes at a diffuse vertex evaluate their next emitters; after the
//       last ones they draw Russian roulette, so the step's rays are those
//       emitters' shadow rays and the next path segment, which leaves the
//       same point.  Neither depends on the other: the stream position after
//       each sample is known (two draws an emitter), and the shadow rays'
//       outcomes only enter the sum.  One trace a vertex instead of two
//       halves the serial chain of a pixel and its wave's per-step work;
//   (3) trace the wave's rays together;
//   (4) add the unoccluded contributions, end the vertex, then take the
//       segment's hit or end the path and shade the next vertex.
// Every sample of a pixel starts with the same primary ray (:578-581), so its
// hit is traced once and kept; the counting variant traces it every time, as
// the reference does.
// Against one kind of ray a step and a primary ray a sample (same boxes, one
// MI355X): 1080p heightfield, 8 spp 9.12 -> 5.14 ms; 1024^2 reference scene,
// 4 spp 2.06 -> 1.49 ms; 1080p soup with 100k triangles 91.1 -> 84.0 ms;
// 256^2, 16 spp forward + backward 1.93 -> 1.48 ms.
template <int BLOCK, int STACK, bool COUNT, bool BATCH, bool POOL>
__device__ __forceinline__ void path_program(const PathLaunch& A)
{
    constexpr bool SCAN = STACK == 0;                // no tree: the scene is scanned
    __shared__ uint32_t s_stack[SCAN ? 1 : STACK * BLOCK];
    __shared__ uint32_t s_occ[BLOCK];                // per lane: occluded shadow rays (bit per slot)
    __shared__ uint2 s_res[BLOCK];                   // per lane: closest hit (prim, t)
    __shared__ uint32_t s_msk[BLOCK];                // per lane: slots holding a ray to trace
    __shared__ uint32_t s_cpre[BLOCK / 64 * kRaySlots];            // per wave and slot: items in lower slots
    __shared__ unsigned long long s_colm[BLOCK / 64 * kRaySlots];  // per wave and slot: lanes holding one
    uint32_t* stk = s_stack + (SCAN ? 0u : threadIdx.x);
    const uint32_t wbase = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
    const uint32_t wslot = (wbase >> 6) * kRaySlots;
    char* const wrec = A.lanes + ((size_t)blockIdx.x * (BLOCK / 64) + (wbase >> 6)) * kWaveBytes;
    // This lane's element of a one-per-lane field f is at wrec + (f + lo16):
    // a wave-uniform base and a 32-bit offset, one address form for all fields.
    const uint32_t lo16 = __lane_id() * 16u;

    const unsigned long long job_at =
        A.jobs ? (unsigned long long)A.jobs : (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();

    // Lane state.
    bool has = false;
    ItemPool pool;
    pool.start((uint32_t)blockIdx.x * (BLOCK / 64) + (wbase >> 6), gridDim.x * (BLOCK / 64), A.width, SCAN && !POOL && !BATCH && A.width <= kQuadWidth);
    uint32_t job = 0, px = 0, py = 0;
    float uvx = 0.0f, uvy = 0.0f, salt = 0.0f;
    uint32_t smp = 0, depth = 0;
    f3 ro{}, rd{}, acc{}, mask{}, accum{};
    f3 N{}, e{};
    const vkr_material* hm = nullptr;   // material of the current diffuse vertex
    uint32_t ei = 0;                    // its next emitter
    bool seg = false;                   // a path segment (ro, rd) is to be traced
    bool nee = false;                   // at a diffuse vertex that is not finished
    bool term = false;                  // ... and Russian roulette ended the path there
    bool ended = false;                 // the path ended with nothing left to trace
    uint32_t nee_flags = 0;             // kNee* of the vertex
    uint32_t prim0 = kMiss;             // the pixel's primary hit
    float t0 = 0.0f;
    uint32_t rays_px = 0, drec = 0, drep = 0;
    uint32_t c_rays = 0, c_shadow = 0, c_traced = 0, wave_steps = 0;
    WorkCnt wc{};

    // :561-574 the primary ray of the lane's pixel.
    auto primary = [&](const JobDesc& j) __attribute__((always_inline)) {
        const float tx = 2.0f * uvx - 1.0f;
        const float ty = 2.0f * uvy - 1.0f;
        f3 dir = add(add(ld3(j.cam_dir), muls(ld3(j.cam_right), tx)), muls(ld3(j.cam_up), ty));
        dir = mul(dir, f3{j.aspect, 1.0f, j.aspect});
        ro = ld3(j.cam_pos);
        rd = normalize(dir);
    };
    // The start of sample smp (:578-581).
    auto new_path = [&](const JobDesc& j) __attribute__((always_inline)) {
        acc = f3{0.0f, 0.0f, 0.0f};
        mask = f3{1.0f, 1.0f, 1.0f};
        depth = 0;
        drec = 0;
        drep = 0;
        if ((j.flags & VKR_TRACE_REPLAY_DECISIONS) && j.decisions)
            drep = j.decisions[((size_t)py * j.W + px) * j.spp + smp];
        // The adjoint's first pass, kept on request: where this sample's
        // random stream starts (its clamp bits follow, per bounce).
        if (j.adj_samples) j.adj_samples[((size_t)py * j.W + px) * j.spp + smp] = make_uint2(__float_as_uint(salt), 0u);
        ++rays_px;                                   // the primary ray
        ++c_rays;
    };
    // Russian roulette with throughput m (:545-549); true: the path ends.
    auto roulette = [&](const JobDesc& j, f3 m) __attribute__((always_inline)) {
        const float u = rng_next(salt, uvx, uvy);
        bool stop = u > max3(m);
        if (depth < 8u) {
            if (j.flags & VKR_TRACE_REPLAY_DECISIONS) stop = !((drep >> (2u * depth)) & 1u);
            if (!stop) drec |= 1u << (2u * depth);
        }
        return stop;
    };

    // Claims pool index g for this lane (no-op for indices outside the image).
    auto claim = [&](uint32_t g) __attribute__((always_inline)) {
        uint32_t local = g;
        if constexpr (BATCH) {
            uint32_t lo = 0, hi = A.n_jobs;
            while (hi - lo > 1u) {
                const uint32_t mid = (lo + hi) >> 1;
                if (A.job_start[mid] <= g) lo = mid; else hi = mid;
            }
            job = lo;
            local = g - A.job_start[lo];
        }
        const JobDesc& j = BATCH ? A.jobs[job] : uniform_job(job_at);
        const uint32_t tile = local >> 6, within = local & 63u;
        if (tile >= j.n_tiles) return;
        const uint32_t x = (tile % j.tiles_x) * 8u + (within & 7u);
        const uint32_t y = (tile / j.tiles_x) * 8u + (within >> 3);
        if (x >= j.W || y >= j.H) return;
        px = x;
        py = y;
        has = true;
        uvx = (float)x / (float)j.W;                 // :563
        uvy = (float)y / (float)j.H;
        salt = uvy / uvx + j.seed;                   // :565-566
        smp = 0;
        // The sum of finished samples: in the lane's record with the ray
        // pool (fewer registers live across the step), else in registers.
        if constexpr (POOL) *reinterpret_cast<float4*>(wrec + (kWPix + lo16)) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        else accum = f3{0.0f, 0.0f, 0.0f};
        rays_px = 0;
        new_path(j);
        primary(j);
        seg = true;
        nee = false;
        ended = false;
        ++c_traced;
    };

    if (!A.persistent) {
        const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
        const uint32_t g = A.base + b * BLOCK + threadIdx.x;
        if (g < A.total) claim(g);
    }

    while (true) {
        if (A.persistent) pool.refill(A.pool, A.total, A.chunk, has, claim);
        const unsigned long long live = __ballot(has);
        if (live == 0) {
            if (!A.persistent || pool.dry) break;
            continue;
        }
        if (COUNT && __lane_id() == 0) ++wave_steps;

        const JobDesc& jq = BATCH ? A.jobs[job] : uniform_job(job_at);

        // (2) Next-event samples (:464-469) and their unoccluded
        // contributions (:475-502), evaluated before the shadow rays
        // (nee_sample).  Rays that must be traced are added to e in emitter
        // order once their outcomes are known: the same additions in the same
        // order as the reference's loop.
        bool sh = false;     // !POOL: a shadow ray (sd, st), contribution c0
        f3 sd{}, c0{};
        float st = 0.0f;
        uint32_t nitem = 0;  // POOL: emitters this lane published for the wave to evaluate
        if (has && nee) {
            if constexpr (POOL) {
                // Publish the hit and its next window of up to kNeeSlots
                // emitters; the wave evaluates all (lane, emitter) pairs
                // together below.  Each sample draws twice (:464-465), so
                // the stream position before each one is known now.
                const uint32_t w = min(kNeeSlots, jq.sc.n_emitters - ei);
                if (ei == 0u) {
                    const f3 V = normalize(sub(ld3(jq.cam_pos), ro));
                    *reinterpret_cast<float4*>(wrec + (kWHit + lo16)) = make_float4(N.x, N.y, N.z, uvx);
                    *reinterpret_cast<float4*>(wrec + (kWHit + 1024u + lo16)) =
                        make_float4(hm->albedo[0], hm->albedo[1], hm->albedo[2], hm->roughness);
                    *reinterpret_cast<float4*>(wrec + (kWHit + 2048u + lo16)) = make_float4(V.x, V.y, V.z, hm->metalness);
                }
                *reinterpret_cast<float4*>(wrec + (kWHit + 3072u + lo16)) =
                    make_float4(__uint_as_float(nee_flags), uvy, __uint_as_float(ei), 0.0f);
                float* sk = reinterpret_cast<float*>(wrec + (kWSalt + 256u + __lane_id() * 4u));
                float sv = salt;
                for (uint32_t k = 0; k < w; ++k) {
                    sk[k * 64u] = sv;
                    sv = sv + 1.0f;
                    sv = sv + 1.0f;
                }
                salt = sv;
                rays_px += w;
                c_rays += w;
                c_shadow += w;
                ei += w;
                nitem = w;
            } else {
                NeeHit h;
                h.P = ro;
                h.N = N;
                h.V = normalize(sub(ld3(jq.cam_pos), ro));
                h.alb = ld3(hm->albedo);
                h.rough = hm->roughness;
                h.metal = hm->metalness;
                h.flags = nee_flags;
                while (ei < jq.sc.n_emitters) {
                    const float s0 = salt;
                    salt = salt + 1.0f;              // the sample's two draws (:464-465)
                    salt = salt + 1.0f;
                    ++rays_px;
                    ++c_rays;
                    ++c_shadow;
                    if (nee_sample(jq, h, ei++, s0, uvx, uvy, sd, st, c0)) {
                        ++c_traced;
                        sh = true;
                        break;
                    }
                }
            }
            if (ei >= jq.sc.n_emitters) {
                // The vertex's last emitters: its next segment goes along.
                term = roulette(jq, mul(mask, ld3(hm->albedo)));
                seg = !term && depth + 1u < jq.max_depth;
                if (seg) {
                    ++rays_px;
                    ++c_rays;
                    ++c_traced;
                }
            }
        }
        // t_max of the queued segment (:444), at the depth it leads to.
        const float dp1 = (float)(depth + (nee ? 2u : 1u));
        const float tmax = 3000.0f / (dp1 * dp1);

        TravOut tr{kMiss, 0.0f, false};
        if constexpr (!POOL) {
            // (3) At most a shadow ray and a segment per lane, from registers.
            bool occluded = false;
            for_each_job<BATCH>(A, job_at, job, has, [&](const JobDesc& jt, bool mine) __attribute__((always_inline)) {
                if (!mine) return;
                if constexpr (SCAN && !BATCH)
                    tr = A.width <= kQuadWidth
                             ? scan_pair_quad(jt.sc, ro, sh, sd, st, has && seg, rd, tmax, jt.eps, occluded)
                             : scan_pair(jt.sc, ro, sh, sd, st, has && seg, rd, tmax, jt.eps, occluded);
                else if constexpr (SCAN)
                    tr = scan_pair(jt.sc, ro, sh, sd, st, has && seg, rd, tmax, jt.eps, occluded);
                else
                    tr = traverse_pair<BLOCK, COUNT>(jt.sc, ro, sh, sd, st, has && seg, rd, tmax, jt.eps, stk, wc,
                                                     occluded);
            });
            if (sh && !occluded) e = add(e, c0);                     // :473, :502
        } else {
            // Path state that the wave's evaluation and tracing do not need
            // waits in the record, so it holds no registers meanwhile.
            float4* park = reinterpret_cast<float4*>(wrec + (kWPark + lo16));
            park[0] = make_float4(acc.x, acc.y, acc.z, uvx);
            park[64] = make_float4(mask.x, mask.y, mask.z, uvy);
            park[128] = make_float4(e.x, e.y, e.z, salt);
            *reinterpret_cast<float4*>(wrec + (kWHead + lo16)) = make_float4(ro.x, ro.y, ro.z, 0.0f);
            *reinterpret_cast<float4*>(wrec + (kWSlotD + lo16)) = make_float4(rd.x, rd.y, rd.z, tmax);
            s_msk[threadIdx.x] = has && seg ? 1u : 0u;
            s_occ[threadIdx.x] = 0u;
            auto fence = []() __attribute__((always_inline)) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            for_each_job<BATCH>(A, job_at, job, has, [&](const JobDesc& jt, bool mine) __attribute__((always_inline)) {
                // The wave evaluates every published (lane, emitter) pair,
                // slot by slot (neighbouring lanes take one emitter of
                // neighbouring owners, whose records are neighbours).  A
                // nonzero contribution goes to slot k of the owner (emitter
                // ei0 + k - 1) and sets bit k of its mask.
                const uint32_t tot = pool_columns(mine ? ((1u << nitem) - 1u) << 1u : 0u, s_cpre + wslot, s_colm + wslot);
                fence();
                for (uint32_t base = 0; base < tot; base += 64u) {
                    const uint32_t i = base + __lane_id();
                    if (i < tot) {
                        uint32_t k, lo;
                        pool_item(s_cpre + wslot, s_colm + wslot, i, k, lo);
                        const uint32_t oo = lo * 16u;
                        const float4 hd = *reinterpret_cast<const float4*>(wrec + (kWHead + oo));
                        const float4 h0 = *reinterpret_cast<const float4*>(wrec + (kWHit + oo));
                        const float4 h1 = *reinterpret_cast<const float4*>(wrec + (kWHit + 1024u + oo));
                        const float4 h2 = *reinterpret_cast<const float4*>(wrec + (kWHit + 2048u + oo));
                        const float4 h3 = *reinterpret_cast<const float4*>(wrec + (kWHit + 3072u + oo));
                        const float sk = *reinterpret_cast<const float*>(wrec + (kWSalt + (k * 64u + lo) * 4u));
                        NeeHit h;
                        h.P = f3{hd.x, hd.y, hd.z};
                        h.N = f3{h0.x, h0.y, h0.z};
                        h.V = f3{h2.x, h2.y, h2.z};
                        h.alb = f3{h1.x, h1.y, h1.z};
                        h.rough = h1.w;
                        h.metal = h2.w;
                        h.flags = __float_as_uint(h3.x);
                        f3 L, c;
                        float tl;
                        if (nee_sample(jt, h, __float_as_uint(h3.z) + k - 1u, sk, h0.w, h3.y, L, tl, c)) {
                            const uint32_t so = (k * 64u + lo) * 16u;
                            *reinterpret_cast<float4*>(wrec + (kWSlotD + so)) = make_float4(L.x, L.y, L.z, tl);
                            *reinterpret_cast<float4*>(wrec + (kWSlotC + so)) = make_float4(c.x, c.y, c.z, 0.0f);
                            atomicOr(s_msk + wbase + lo, 1u << k);
                        }
                    }
                }
                fence();
                // (3) The wave traces all queued rays together from its pool,
                // slot by slot: column k holds slot k of every lane that
                // queued one, lanes in order.  Neighbouring lanes then take
                // rays of one slot (the path segments, or one emitter) from
                // neighbouring pixels, which visit much the same nodes.
                const uint32_t msk = mine ? s_msk[threadIdx.x] : 0u;
                c_traced += (uint32_t)__popc(msk & ~1u);
                const uint32_t nrays = pool_columns(msk, s_cpre + wslot, s_colm + wslot);
                // The pool, the records and the result words are shared by
                // the wave's lanes: order the writes above before the reads
                // below.
                fence();
                if constexpr (SCAN)
                    scan_pool(jt, nrays, s_cpre + wslot, s_colm + wslot, s_occ + wbase, s_res + wbase, wrec);
                else
                    traverse_pool<BLOCK, COUNT>(jt, nrays, s_cpre + wslot, s_colm + wslot, s_occ + wbase, s_res + wbase,
                                                wrec, stk, wc);
                fence();
            });
            const float4 k0 = park[0], k1 = park[64], k2 = park[128];
            acc = f3{k0.x, k0.y, k0.z};
            mask = f3{k1.x, k1.y, k1.z};
            e = f3{k2.x, k2.y, k2.z};
            uvx = k0.w;
            uvy = k1.w;
            salt = k2.w;
            const float4 hd = *reinterpret_cast<const float4*>(wrec + (kWHead + lo16));
            const float4 sg = *reinterpret_cast<const float4*>(wrec + (kWSlotD + lo16));
            ro = f3{hd.x, hd.y, hd.z};
            rd = f3{sg.x, sg.y, sg.z};
            if (seg) {
                const uint2 r = s_res[threadIdx.x];
                tr.prim = r.x;
                tr.t = __uint_as_float(r.y);
                tr.hit = r.x != kMiss;
            }
            uint32_t bits = s_msk[threadIdx.x] & ~s_occ[threadIdx.x] & ~1u;   // unoccluded (:473), in emitter order
            while (bits) {
                const uint32_t k = (uint32_t)__builtin_ctz(bits);
                bits &= bits - 1u;
                const float4 c = *reinterpret_cast<const float4*>(wrec + (kWSlotC + k * 1024u + lo16));
                e = add(e, f3{c.x, c.y, c.z});                       // :502
            }
        }
        if (!has) continue;

        // (4) End of a diffuse vertex (:507-511) and of its roulette.
        const JobDesc& j = BATCH ? A.jobs[job] : uniform_job(job_at);
        bool path_end = ended;
        ended = false;
        if (nee) {
            if (ei < j.sc.n_emitters) continue;                      // more emitters
            nee = false;
            const f3 emis = ld3(hm->emissive);
            const bool all_pos = gmax(gsign(emis.x), 0.0f) == 1.0f && gmax(gsign(emis.y), 0.0f) == 1.0f &&
                                 gmax(gsign(emis.z), 0.0f) == 1.0f;
            const f3 em = all_pos ? normalize(emis) : f3{0.0f, 0.0f, 0.0f};
            acc = add(acc, mul(mask, add(em, e)));
            mask = mul(mask, ld3(hm->albedo));
            if (!term) {
                mask = muls(mask, recip_rn(max3(mask)));
                ++depth;
            }
            path_end = !seg;
        }

        bool hit = false;
        if (seg) {
            seg = false;
            if (j.adj_samples) {
                // Channels that clamp(acc) saturates at this bounce, 10 bits per channel.
                const uint32_t bit = 1u << depth;
                const uint32_t zb = ((acc.x > 1.0f || acc.x < 0.0f) ? bit : 0u) |
                                    ((acc.y > 1.0f || acc.y < 0.0f) ? bit << 10 : 0u) |
                                    ((acc.z > 1.0f || acc.z < 0.0f) ? bit << 20 : 0u);
                if (zb) j.adj_samples[((size_t)py * j.W + px) * j.spp + smp].y |= zb;
            }
            acc = clamps(acc, 0.0f, 1.0f);                           // :441
            if (smp == 0 && depth == 0) {                            // the primary hit, written at once
                const size_t pi = (size_t)py * j.W + px;
                if (j.prim_id) j.prim_id[pi] = tr.prim;
                if (j.hit_t) j.hit_t[pi] = tr.t;
                if (j.adj_primary) j.adj_primary[pi] = make_uint2(tr.prim, __float_as_uint(tr.t));
                if constexpr (POOL) {
                    *reinterpret_cast<float2*>(wrec + (kWPark + 3072u + lo16)) =
                        make_float2(__uint_as_float(tr.prim), tr.t);
                } else {
                    prim0 = tr.prim;
                    t0 = tr.t;
                }
            }
            hit = tr.hit;
            path_end = !tr.hit;                                      // :445
        }

        if (path_end) {                                              // :578-581
            if constexpr (POOL) {
                const float4 a = *reinterpret_cast<const float4*>(wrec + (kWPix + lo16));
                const float2 b = *reinterpret_cast<const float2*>(wrec + (kWPark + 3072u + lo16));
                accum = f3{a.x, a.y, a.z};
                prim0 = __float_as_uint(b.x);
                t0 = b.y;
            }
            // The next sample starts at the kept primary hit; where that is
            // a miss it ends there too.
            bool more;
            do {
                if ((j.flags & VKR_TRACE_RECORD_DECISIONS) && j.decisions)
                    j.decisions[((size_t)py * j.W + px) * j.spp + smp] = (uint16_t)drec;
                accum = add(accum, acc);
                ++smp;
                more = smp < j.spp;
                if (more) new_path(j);
            } while (!COUNT && more && prim0 == kMiss);
            if (more) {
                primary(j);
                if constexpr (COUNT) {
                    seg = true;
                    ++c_traced;
                } else {
                    hit = true;
                    tr.prim = prim0;
                    tr.t = t0;
                }
                if constexpr (POOL)
                    *reinterpret_cast<float4*>(wrec + (kWPix + lo16)) = make_float4(accum.x, accum.y, accum.z, 0.0f);
            } else {                                                 // :585-592
                const size_t pi = (size_t)py * j.W + px;
                f3 c = divs(accum, (float)j.spp);
                if (j.radiance) reinterpret_cast<float4*>(j.radiance)[pi] = make_float4(c.x, c.y, c.z, 1.0f);
                c = divv(c, adds(c, 1.0f));
                c = f3{pow_f(c.x, kInvGamma), pow_f(c.y, kInvGamma), pow_f(c.z, kInvGamma)};
                const float dither = rng_next(salt, uvx, uvy) / 64.0f;
                c = adds(c, dither);
                if (j.rgba8)
                    reinterpret_cast<uint32_t*>(j.rgba8)[pi] =
                        unorm8(c.x) | (unorm8(c.y) << 8) | (unorm8(c.z) << 16) | (255u << 24);
                if (j.ray_count) j.ray_count[pi] = rays_px;
                has = false;
                hit = false;
            }
        }

        if (hit) {                                                   // shade the vertex
            const f3 P = add(ro, muls(rd, tr.t));
            const uint32_t kind = tr.prim >> 30, idx = tr.prim & 0x3FFFFFFFu;
            const vkr_material* m;
            if (kind == 0) {
                const vkr_triangle* T = j.sc.tris_orig + idx;
                const f3 v0 = ld3(T->v0), v1 = ld3(T->v1), v2 = ld3(T->v2);
                const f3 u = sub(v1, v0), v = sub(v2, v0);
                N = f3{(u.y * v.z) - (u.z * v.y), (u.z * v.x) - (u.x * v.z), (u.x * v.y) - (u.y * v.x)};  // :392
                const uint32_t mi = T->mat_index;
                m = ((j.sc.flags & VKR_SCENE_TRI_MATERIAL_INDEX) && mi < j.sc.n_materials) ? j.sc.materials + mi
                                                                                           : j.sc.tri_material;
            } else if (kind == 1) {
                const vkr_sphere* S = j.sc.spheres + idx;
                N = divs(sub(P, ld3(S->P)), S->r);                   // :408
                m = &S->mat;
            } else {
                const vkr_plane* Q = j.sc.planes + idx;
                N = ld3(Q->N);                                       // :424
                m = &Q->mat;
            }
            const uint32_t type = m->type;
            if (type == VKR_MAT_DIFFUSE) {                           // :451-513
                const float r2 = rng_next(salt, uvx, uvy);
                const float phi = kTwoPi * rng_next(salt, uvx, uvy);
                const f3 dj = muls(jitter(N, phi, sqrt_rn(r2), sqrt_rn(1.0f - r2)), 1.0f - m->metalness);
                hm = m;
                ei = 0;
                e = f3{0.0f, 0.0f, 0.0f};
                rd = normalize(add(reflect(rd, N), dj));             // :512
                ro = P;
                nee = true;
                nee_flags = nee_flags_of(j.sc, N, m);
            } else {
                if (type == VKR_MAT_DIELECTRIC) {                    // :514-542
                    const f3 emis = ld3(m->emissive);
                    const float rough = m->roughness;
                    acc = add(acc, mul(emis, mask));
                    mask = mul(mask, ld3(m->albedo));
                    const float cosine = -dot(rd, N) / length(rd);
                    const f3 reflected = reflect(rd, N);
                    const f3 refracted = refract(rd, N, rough);
                    const float prob = eq3(refracted, f3{0.0f, 0.0f, 0.0f}) ? 1.0f : schlick(cosine, rough);
                    const float u = rng_next(salt, uvx, uvy);
                    bool refl = u < prob;
                    if (depth < 8u) {
                        if (j.flags & VKR_TRACE_REPLAY_DECISIONS) refl = (drep >> (2u * depth + 1u)) & 1u;
                        if (refl) drec |= 1u << (2u * depth + 1u);
                    }
                    rd = normalize(refl ? reflected : refracted);
                    ro = P;
                }
                // (a type outside the switch goes straight on to the roulette)
                if (!roulette(j, mask)) {
                    mask = muls(mask, recip_rn(max3(mask)));
                    ++depth;
                    seg = depth < j.max_depth;
                    if (seg) {
                        ++rays_px;
                        ++c_rays;
                        ++c_traced;
                    }
                }
                ended = !seg;
            }
        }
    }

    DevCounters* const cnt = counter_bank(A.counters, blockIdx.x);
    flush_counter(&cnt->rays, c_rays);
    if (A.rays_only) return;
    flush_counter(&cnt->shadow, c_shadow);
    flush_counter(&cnt->traced, c_traced);
    flush_counter(&cnt->overflow, wc.overflow);
    if (COUNT) {
        flush_counter(&cnt->nodes, wc.nodes);
        flush_counter(&cnt->tris, wc.tris);
        flush_counter(&cnt->spheres, wc.spheres);
        flush_counter(&cnt->planes, wc.planes);
        flush_counter(&cnt->wave_nodes, wc.wave_nodes);
        flush_counter(&cnt->wave_leaves, wc.wave_leaves);
        flush_counter(&cnt->wave_steps, wave_steps);
    }
}

// The timed kernel and the work-counting variant (same traversal order, more
// registers).  The traversal waits on dependent node fetches, so resident
// waves set the speed: with a 24-entry stack a 128-lane block needs 15.1 KB
// of LDS, ten fit a CU, and the pooled kernel is held to 96 VGPRs for 5 waves
// per SIMD (its spills are all in per-step code, outside the pool's traversal
// loops); with deeper stacks LDS allows 4 waves (128 VGPRs).  One ray a lane,
// 4 waves without the 69 spills are the faster ones: 1080p heightfield 4535 ->
// 4370 us (pooled, 100k-triangle soup 71.2 -> 73.5 ms).
template <int BLOCK, int STACK, bool BATCH, bool POOL>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(POOL && STACK > 0 && STACK <= 24 ? 5 : 4))) void k_path(const PathLaunch A)
{
    path_program<BLOCK, STACK, false, BATCH, POOL>(A);
}

template <int BLOCK, int STACK, bool BATCH, bool POOL>
__global__ __launch_bounds__(BLOCK) void k_path_count(const PathLaunch A)
{
    path_program<BLOCK, STACK, true, BATCH, POOL>(A);
}

// ---------------------------------------------------------------------------
// Whitted kernel, Assets/Raytracer.comp (its own constant scene, :98-127).
// ---------------------------------------------------------------------------
namespace whitted {
constexpr float kEps = 0.01f;  // :89
struct Sph { uint32_t mat; float o[3]; float r; };
struct Pln { uint32_t mat; float n[3]; float d; };
__constant__ Sph kSph[2] = {{5, {-14.0f, 12.0f, 32.0f}, 5.0f}, {4, {32.0f, 24.0f, 25.0f}, 12.0f}};
constexpr float kFloor = 0.0f, kCeiling = 128.0f, kWall = 64.0f;
__constant__ Pln kPln[5] = {{0, {0.0f, 1.0f, 0.0f}, kFloor},
                            {0, {0.0f, -1.0f, 0.0f}, kCeiling},
                            {2, {0.0f, 0.0f, -1.0f}, kWall},
                            {1, {1.0f, 0.0f, 0.0f}, kWall},
                            {3, {-1.0f, 0.0f, 0.0f}, kWall}};
__constant__ float kTri[9] = {10.0f, 10.0f, 0.0f, 0.0f, 20.0f, 0.0f, -10.0f, 10.0f, 0.0f};
__constant__ uint32_t kRefl[6] = {1, 0, 1, 0, 0, 0};
__constant__ float kDiff[18] = {1, 1, 1, 1, 0, 0, 0, 1, 0, 0, 0, 1, 1, 1, 0, 1, 0, 1};

// The nearest hit so far, and what is derived of it once the search is over.
struct Hit { float dist; uint32_t prim; uint32_t mat; f3 P, N; };

__device__ __forceinline__ float wplane_t(f3 o, f3 d, f3 n, float dist)  // :180-192
{
    const float dd = dot(d, n);
    if (dd == 0.0f) return 0.0f;
    return gmax(-(dist + dot(o, n)) / dd, 0.0f);
}

// The planes as they are: :253-275.
__device__ __forceinline__ void search_planes(f3 o, f3 d, Hit& h)
{
    for (int i = 0; i < 5; ++i) {
        const float t = wplane_t(o, d, ld3(kPln[i].n), kPln[i].d);
        if (t > kEps && t < h.dist) {
            h.dist = t;
            h.prim = (2u << 30) | (uint32_t)i;
        }
    }
}

// One axis: planes lo and hi (or hi alone) are num / dk away, whichever of them
// lies ahead.
__device__ __forceinline__ void search_axis(float num, float dk, bool ahead, uint32_t plane, Hit& h)
{
    const float t = num / dk;
    if (ahead && t > kEps && t < h.dist) {
        h.dist = t;
        h.prim = (2u << 30) | plane;
    }
}

// trace_ray (:224-278): the distance and primitive of the nearest hit.  The
// room's normals are axes, so for finite rays a plane's two dot products are one
// coordinate each, plus zeros, and opposite walls share the divisor: only the
// wall ahead has a distance above 0, one division an axis instead of one a
// wall.  Where both lie ahead (the ray starts outside the room) all are tested.
// 1024^2 frame 46.5 -> 45.0 us; bound by VALU issue and the waits for a hit's
// constants.
__device__ __forceinline__ bool search(f3 o, f3 d, Hit& h)
{
    h.prim = kMiss;
    const f3 v0 = ld3(kTri), v1 = ld3(kTri + 3), v2 = ld3(kTri + 6);
    {
        const float t = tri_t(o, d, v0, sub(v1, v0), sub(v2, v0), kEps);
        if (t > kEps && t < h.dist) {
            h.dist = t;
            h.prim = 0;
        }
    }
    for (int i = 0; i < 2; ++i) {
        const float t = sphere_t(o, d, ld3(kSph[i].o), kSph[i].r);
        if (t > kEps && t < h.dist) {
            h.dist = t;
            h.prim = (1u << 30) | (uint32_t)i;
        }
    }
    const float sum = fabsf(o.x) + fabsf(o.y) + fabsf(o.z) + fabsf(d.x) + fabsf(d.y) + fabsf(d.z);
    const float y0 = -(kFloor + o.y), y1 = kCeiling - o.y, z1 = kWall - o.z, x0 = -(kWall + o.x), x1 = kWall - o.x;
    const bool up = d.y > 0.0f, right = d.x > 0.0f, back = d.z > 0.0f;
    const bool y0a = y0 > 0.0f == up, y1a = y1 > 0.0f == up, x0a = x0 > 0.0f == right, x1a = x1 > 0.0f == right;
    if (!(sum < 3e38f) || (y0a && y1a) || (x0a && x1a)) {
        search_planes(o, d, h);
    } else {
        search_axis(y0a ? y0 : y1, d.y, (y0a || y1a) && d.y != 0.0f, y0a ? 0u : 1u, h);
        search_axis(z1, d.z, z1 > 0.0f == back && d.z != 0.0f, 2u, h);
        search_axis(x0a ? x0 : x1, d.x, (x0a || x1a) && d.x != 0.0f, x0a ? 3u : 4u, h);
    }
    return h.prim != kMiss;
}

// The hit's point, normal and material.
__device__ __forceinline__ void finish_hit(f3 o, f3 d, Hit& h)
{
    h.P = add(o, muls(d, h.dist));
    const uint32_t kind = h.prim >> 30, i = h.prim & 0x3FFFFFFFu;
    if (kind == 0) {
        const f3 v0 = ld3(kTri), v1 = ld3(kTri + 3), v2 = ld3(kTri + 6);
        const f3 u = sub(v1, v0), v = sub(v2, v0);
        h.mat = 1;
        h.N = f3{(u.y * v.z) - (u.z * v.y), (u.z * v.x) - (u.x * v.z), (u.x * v.y) - (u.y * v.x)};
    } else if (kind == 1) {
        h.mat = kSph[i].mat;
        h.N = divs(sub(h.P, ld3(kSph[i].o)), kSph[i].r);
    } else {
        h.mat = kPln[i].mat;
        h.N = ld3(kPln[i].n);
    }
}

struct C4 { float r, g, b, a; };

__device__ C4 render(const JobDesc& j, f3& ro, f3& rd, uint32_t& bounce, uint32_t& rays, bool& cap,
                     uint32_t& prim, float& pt)                             // :280-355
{
    Hit h;
    h.dist = 1000.0f;                                                       // :88,290
    ++rays;
    const bool hit = search(ro, rd, h);
    if (cap) { cap = false; prim = hit ? h.prim : kMiss; pt = h.dist; }
    if (!hit) return C4{0.0f, 0.0f, 0.0f, 1.0f};
    finish_hit(ro, rd, h);
    const f3 lp = ld3(j.light_pos);
    const f3 light_vec = normalize(sub(lp, h.P));
    const float dist_to_light = length(sub(lp, h.P));
    const f3 mdiff = ld3(kDiff + 3 * h.mat);
    const float li = 540.0f / (12.56637072f * dist_to_light);               // :308
    const f3 diffuse = muls(muls(mdiff, li), gmax(dot(h.N, light_vec), 0.0f));
    const f3 half_vec = normalize(add(light_vec, normalize(ld3(j.cam_pos))));
    const float spec = li * pow16(gclamp(dot(h.N, half_vec), 0.0f, 1.0f));
    f3 color = adds(diffuse, spec);
    Hit sh;
    sh.dist = dist_to_light;
    ++rays;
    if (search(h.P, light_vec, sh)) {                                        // :322-340
        color = muls(color, 0.5f);
        bounce = 3;
    }
    if (kRefl[h.mat]) {                                                     // :343-351
        rd = sub(rd, muls(h.N, 2.0f * dot(h.N, rd)));
        ro = h.P;
    } else {
        bounce = 3;
    }
    return C4{color.x, color.y, color.z, 1.0f};
}
}  // namespace whitted

__global__ __launch_bounds__(256) void k_whitted(const JobDesc j, CounterRef counters)
{
    const uint32_t x = blockIdx.x * 16u + (threadIdx.x & 15u);
    const uint32_t y = blockIdx.y * 16u + (threadIdx.x >> 4);
    uint32_t rays = 0;
    if (x < j.W && y < j.H) {
        const float uvx = (float)x / (float)j.W, uvy = (float)y / (float)j.H;   // :362
        const float tx = 2.0f * uvx - 1.0f, ty = 2.0f * uvy - 1.0f;             // :366
        f3 dir = add(add(ld3(j.cam_dir), muls(ld3(j.cam_right), tx)), muls(ld3(j.cam_up), ty));
        dir = mul(dir, f3{j.aspect, 1.0f, j.aspect});                           // :370
        f3 ro = ld3(j.cam_pos), rd = normalize(dir);
        uint32_t bounce = 0, prim = kMiss;
        bool cap = true;
        float pt = 0.0f;
        whitted::C4 fc = whitted::render(j, ro, rd, bounce, rays, cap, prim, pt);
        float s = 0.4f;                                                         // :382
        while (++bounce <= 2u) {                                                // :384-394
            const whitted::C4 rc = whitted::render(j, ro, rd, bounce, rays, cap, prim, pt);
            const float a = 1.0f - s;
            const float ma = 1.0f - a;
            const whitted::C4 m = {rc.r * ma + fc.r * a, rc.g * ma + fc.g * a, rc.b * ma + fc.b * a,
                                   rc.a * ma + fc.a * a};
            fc = whitted::C4{fc.r * (1.0f - s) + m.r * s, fc.g * (1.0f - s) + m.g * s,
                             fc.b * (1.0f - s) + m.b * s, fc.a * (1.0f - s) + m.a * s};
            s = s * 0.5f;
        }
        const size_t pi = (size_t)y * j.W + x;
        if (j.radiance) reinterpret_cast<float4*>(j.radiance)[pi] = make_float4(fc.r, fc.g, fc.b, fc.a);
        if (j.rgba8)
            reinterpret_cast<uint32_t*>(j.rgba8)[pi] =
                unorm8(fc.r) | (unorm8(fc.g) << 8) | (unorm8(fc.b) << 16) | (unorm8(fc.a) << 24);
        if (j.prim_id) j.prim_id[pi] = prim;
        if (j.hit_t) j.hit_t[pi] = pt;
        if (j.ray_count) j.ray_count[pi] = rays;
    }
    DevCounters* const cnt = counter_bank(counters, blockIdx.y * gridDim.x + blockIdx.x);
    flush_counter(&cnt->rays, rays);
    flush_counter(&cnt->traced, rays);
}

// ---------------------------------------------------------------------------
// Present pass, Assets/Fullscreen.frag:14-31 (+ Fullscreen.vert:6-11).
//
// Six bilinear samples, 24 texels a pixel, each channel over 255: the VALU
// bounds it (its bytes take 3 us of a 1024^2 -> 1080p pass).  A channel's
// t / 255 is two operations (below) instead of a division's ten; the samples'
// rows and columns are set up once each, for the centre and the two steps;
// texels outside the image are read as zero instead of branched around, and
// only in the waves that touch the border; and a wave in which the picture
// holds still everywhere takes no neighbour samples.
// 1024^2 -> 1920x1080: 61.6 -> 21.5 us.
// ---------------------------------------------------------------------------
// One axis of a sample at texture coordinate c (VK_FILTER_LINEAR): the lower
// texel and the upper one's weight.
struct TexAxis {
    int i;
    float a;
    __device__ __forceinline__ TexAxis(float c, uint32_t n)
    {
        const float x = c * (float)n - 0.5f;
        const float f = floorf(x);
        i = (int)f;
        a = x - f;
    }
    __device__ __forceinline__ bool inside(uint32_t n) const { return i >= 0 && i + 1 < (int)n; }
};

// t / 255 of a byte, rounded as the division: 1/255 as the sum of two floats
// (equal for all 256 bytes).
__device__ __forceinline__ float unit_byte(uint32_t t)
{
    const float v = (float)t;
    return __builtin_fmaf(v, 0x1.010102p-8f, v * -0x1.fdfdfep-33f);
}

// CLAMP_TO_BORDER with opaque black (GraphicsDevice.cpp:770-790) unless the
// sample's texels are known to lie inside.  A texel of zero adds +0, which
// leaves the sum as it is.
template <bool INSIDE>
__device__ __forceinline__ f3 sample_bilinear(const uint32_t* __restrict__ img, uint32_t w, uint32_t h, const TexAxis& x,
                                              const TexAxis& y)
{
    f3 acc{0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int dy = 0; dy < 2; ++dy) {
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
            const int xi = x.i + dx, yi = y.i + dy;
            const float wgt = (dx ? x.a : 1.0f - x.a) * (dy ? y.a : 1.0f - y.a);
            uint32_t t = 0u;
            if (INSIDE || (xi >= 0 && yi >= 0 && xi < (int)w && yi < (int)h)) t = img[(uint32_t)yi * w + (uint32_t)xi];
            acc.x = acc.x + unit_byte(t & 255u) * wgt;
            acc.y = acc.y + unit_byte((t >> 8) & 255u) * wgt;
            acc.z = acc.z + unit_byte((t >> 16) & 255u) * wgt;
        }
    }
    return acc;
}

template <bool INSIDE>
__device__ __forceinline__ f3 filter_pixel(const uint32_t* cur, const uint32_t* prev, uint32_t w, uint32_t h,
                                           const TexAxis& x, const TexAxis& xm, const TexAxis& xp, const TexAxis& y,
                                           const TexAxis& ym, const TexAxis& yp)
{
    const f3 c0 = sample_bilinear<INSIDE>(cur, w, h, x, y);
    const f3 c1 = sample_bilinear<INSIDE>(prev, w, h, x, y);
    const f3 dl = sub(c0, c1);
    const float vT = dot(dl, dl);                                           // :26
    if (!(vT > 0.0005f)) return c0;
    const f3 n = sample_bilinear<INSIDE>(cur, w, h, x, yp);                 // :20-23
    const f3 s = sample_bilinear<INSIDE>(cur, w, h, x, ym);
    const f3 e = sample_bilinear<INSIDE>(cur, w, h, xp, y);
    const f3 v = sample_bilinear<INSIDE>(cur, w, h, xm, y);
    return muls(add(add(add(n, s), e), v), 0.25f);                          // :28
}

__global__ __launch_bounds__(256) void k_filter(const uint32_t* __restrict__ cur, const uint32_t* __restrict__ prev,
                                                uint32_t sw, uint32_t sh, uint32_t* __restrict__ out, uint32_t dw,
                                                uint32_t dh)
{
    const uint32_t px = blockIdx.x * 16u + (threadIdx.x & 15u);
    const uint32_t py = blockIdx.y * 16u + (threadIdx.x >> 4);
    if (px >= dw || py >= dh) return;
    const float inv_size = 1.0f / 2048.0f;                                  // :12
    const float u = ((float)px + 0.5f) / (float)dw;
    const float v = 1.0f - ((float)py + 0.5f) / (float)dh;                   // :16
    const TexAxis x(u, sw), xm(u + -1.0f * inv_size, sw), xp(u + 1.0f * inv_size, sw);
    const TexAxis y(v, sh), ym(v + -1.0f * inv_size, sh), yp(v + 1.0f * inv_size, sh);
    const bool inside = xm.inside(sw) && xp.inside(sw) && ym.inside(sh) && yp.inside(sh);
    const f3 fin = __ballot(!inside) == 0ull ? filter_pixel<true>(cur, prev, sw, sh, x, xm, xp, y, ym, yp)
                                             : filter_pixel<false>(cur, prev, sw, sh, x, xm, xp, y, ym, yp);
    out[(size_t)py * dw + px] = unorm8(fin.x) | (unorm8(fin.y) << 8) | (unorm8(fin.z) << 16) | (255u << 24);
}

// ---------------------------------------------------------------------------
// Building-block evaluation for parity tests (op codes in vkr.h).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_debug(uint32_t op, const float* in, float* out, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float* a = in + (size_t)i * 16;
    float* r = out + (size_t)i * 8;
    switch (op) {
    case VKR_DEBUG_RAND: {  // in: cx cy salt0 -> out: 8 successive rand()
        float salt = a[2];
        for (int k = 0; k < 8; ++k) r[k] = rng_next(salt, a[0], a[1]);
        break;
    }
    case VKR_DEBUG_TRI:     // in: o(3) d(3) v0(3) v1(3) eps ... (v2 at 12..14 via a[12]) -> t
        r[0] = tri_t(f3{a[0], a[1], a[2]}, f3{a[3], a[4], a[5]}, f3{a[6], a[7], a[8]},
                     sub(f3{a[9], a[10], a[11]}, f3{a[6], a[7], a[8]}),
                     sub(f3{a[12], a[13], a[14]}, f3{a[6], a[7], a[8]}), a[15]);
        break;
    case VKR_DEBUG_SPHERE:  // in: o(3) d(3) c(3) r -> t
        r[0] = sphere_t(f3{a[0], a[1], a[2]}, f3{a[3], a[4], a[5]}, f3{a[6], a[7], a[8]}, a[9]);
        break;
    case VKR_DEBUG_PLANE:   // in: o(3) d(3) N(3) len -> t
        r[0] = plane_t(f3{a[0], a[1], a[2]}, f3{a[3], a[4], a[5]}, f3{a[6], a[7], a[8]}, a[9]);
        break;
    case VKR_DEBUG_BRDF: {  // in: N(3) H(3) V(3) L(3) rough cos F0 -> NDF, G, F(3), schlick(cos, rough)
        const f3 Nn{a[0], a[1], a[2]}, H{a[3], a[4], a[5]}, V{a[6], a[7], a[8]}, L{a[9], a[10], a[11]};
        r[0] = distribution_ggx(Nn, H, a[12]);
        r[1] = geometry_smith(Nn, V, L, a[12]);
        const f3 F = fresnel_schlick(a[13], f3{a[14], a[14], a[14]});
        r[2] = F.x; r[3] = F.y; r[4] = F.z;
        r[5] = schlick(a[13], a[12]);
        break;
    }
    case VKR_DEBUG_JITTER: {  // in: d(3) phi sina cosa -> out(3)
        const f3 v = jitter(f3{a[0], a[1], a[2]}, a[3], a[4], a[5]);
        r[0] = v.x; r[1] = v.y; r[2] = v.z;
        break;
    }
    case VKR_DEBUG_COS:     // in: x -> cos, sin, pow(x, 1/2.2)
        r[0] = cos_f(a[0]);
        r[1] = sin_f(a[0]);
        r[2] = pow_f(a[0], kInvGamma);
        break;
    default:
        break;
    }
}

__global__ __launch_bounds__(256) void k_zero(CounterRef c, uint32_t* pool)
{
    unsigned long long* w = reinterpret_cast<unsigned long long*>(c.banks);
    const uint32_t n = (c.mask + 1u) * (uint32_t)(sizeof(DevCounters) / sizeof(unsigned long long));
    for (uint32_t i = threadIdx.x; i < n; i += 256u) w[i] = 0ull;
    if (pool && threadIdx.x < 2u) pool[threadIdx.x] = 0u;   // [1]: the adjoint's second pass
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
namespace {
template <int BLOCK, int STACK, bool COUNT, bool BATCH, bool POOL>
const void* fn()
{
    if constexpr (COUNT) return reinterpret_cast<const void*>(&k_path_count<BLOCK, STACK, BATCH, POOL>);
    else return reinterpret_cast<const void*>(&k_path<BLOCK, STACK, BATCH, POOL>);
}

template <int BLOCK, int STACK, bool COUNT, bool BATCH>
const void* fn_pool(bool pool) { return pool ? fn<BLOCK, STACK, COUNT, BATCH, true>() : fn<BLOCK, STACK, COUNT, BATCH, false>(); }

template <int BLOCK, int STACK>
const void* fn_flags(const PathVariant& v)
{
    if (v.count) return v.batch ? fn_pool<BLOCK, STACK, true, true>(v.pool) : fn_pool<BLOCK, STACK, true, false>(v.pool);
    return v.batch ? fn_pool<BLOCK, STACK, false, true>(v.pool) : fn_pool<BLOCK, STACK, false, false>(v.pool);
}

// The scanning kernels have no stack and no counting variant.
template <int BLOCK>
const void* fn_scan(const PathVariant& v)
{
    return v.batch ? fn_pool<BLOCK, 0, false, true>(v.pool) : fn_pool<BLOCK, 0, false, false>(v.pool);
}

const void* kernel_ptr(const PathVariant& v)
{
    if (v.scan) return v.block == 64 ? fn_scan<64>(v) : v.block == 128 ? fn_scan<128>(v) : fn_scan<256>(v);
    if (v.block == 64) return v.stack <= 24 ? fn_flags<64, 24>(v) : v.stack <= 32 ? fn_flags<64, 32>(v) : fn_flags<64, 64>(v);
    if (v.block == 128) return v.stack <= 24 ? fn_flags<128, 24>(v) : v.stack <= 32 ? fn_flags<128, 32>(v) : fn_flags<128, 64>(v);
    return v.stack <= 24 ? fn_flags<256, 24>(v) : v.stack <= 32 ? fn_flags<256, 32>(v) : fn_flags<256, 64>(v);
}
}  // namespace

uint32_t stack_variant(uint32_t needed)
{
    if (needed <= 24) return 24;   // 5 waves per SIMD
    if (needed <= 32) return 32;
    if (needed <= 64) return 64;
    return 0;
}

hipError_t launch_path(const PathLaunch& a, const PathVariant& v, uint32_t grid, hipStream_t s)
{
    void* args[] = {const_cast<PathLaunch*>(&a)};
    return hipLaunchKernel(kernel_ptr(v), dim3(grid), dim3(v.block), args, 0, s);
}

uint32_t compute_units(int device)
{
    static thread_local int dev = -1, cus = 0;
    if (dev != device) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 256;
        dev = device;
    }
    return (uint32_t)cus;
}

uint32_t persistent_grid(const PathVariant& v, int device)
{
    // Resident workgroups per CU x CUs, cached per (device, variant).
    struct Entry { int device; PathVariant v; uint32_t grid; };
    static thread_local Entry cache[64];
    static thread_local int n = 0;
    for (int i = 0; i < n; ++i) {
        const Entry& c = cache[i];
        if (c.device == device && c.v.block == v.block && c.v.stack == v.stack && c.v.count == v.count &&
            c.v.batch == v.batch && c.v.pool == v.pool && c.v.scan == v.scan)
            return c.grid;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel_ptr(v), (int)v.block, 0) != hipSuccess ||
        per_cu < 1)
        per_cu = 1;
    const uint32_t grid = (uint32_t)per_cu * compute_units(device);
    if (n < 64) cache[n++] = Entry{device, v, grid};
    return grid;
}

hipError_t launch_whitted(const JobDesc& j, CounterRef c, hipStream_t s)
{
    hipLaunchKernelGGL(k_whitted, dim3((j.W + 15) / 16, (j.H + 15) / 16), dim3(256), 0, s, j, c);
    return hipGetLastError();
}

hipError_t launch_filter(const uint8_t* cur, const uint8_t* prev, uint32_t sw, uint32_t sh, uint8_t* out,
                         uint32_t dw, uint32_t dh, hipStream_t s)
{
    hipLaunchKernelGGL(k_filter, dim3((dw + 15) / 16, (dh + 15) / 16), dim3(256), 0, s,
                       reinterpret_cast<const uint32_t*>(cur), reinterpret_cast<const uint32_t*>(prev), sw, sh,
                       reinterpret_cast<uint32_t*>(out), dw, dh);
    return hipGetLastError();
}

hipError_t launch_debug(uint32_t op, const float* in, float* out, uint32_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_debug, dim3((n + 255) / 256), dim3(256), 0, s, op, in, out, n);
    return hipGetLastError();
}

__global__ void k_set_frame(JobDesc* job, vkr_frame_data fd)
{
    if (threadIdx.x != 0) return;
    for (int k = 0; k < 3; ++k) {
        job->cam_pos[k] = fd.camera.pos[k];
        job->cam_dir[k] = fd.camera.dir[k];
        job->cam_right[k] = fd.camera.right[k];
        job->cam_up[k] = fd.camera.up[k];
        job->light_pos[k] = fd.light_pos[k];
    }
    job->aspect = fd.aspect_ratio;
    job->seed = fd.seed;
}

hipError_t launch_set_frame(JobDesc* job, const vkr_frame_data& fd, hipStream_t s)
{
    hipLaunchKernelGGL(k_set_frame, dim3(1), dim3(64), 0, s, job, fd);
    return hipGetLastError();
}

// Scratch for callers that cannot allocate (vkr_trace_frame_static): one
// array per device, held until the process ends.  Host code never passes
// `scratch` itself to a kernel: its name is a host-side stand-in, and the
// device address comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) char scratch[kStaticScratchBytes];

hipError_t static_scratch(int device, char** out)
{
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static char* addr[kMaxDevices] = {};
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        addr[device] = static_cast<char*>(p);
    }
    *out = addr[device];
    return hipSuccess;
}

hipError_t launch_zero_counters(CounterRef c, uint32_t* pool, hipStream_t s)
{
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(256), 0, s, c, pool);
    return hipGetLastError();
}

}  // namespace vkr
