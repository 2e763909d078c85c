// adjoint.hip - path-replay adjoint of the path kernel (build extension).
//
// Parameters (vkr_scene_set_sphere_params): per sphere s albedo a_s (3),
// emission e_s (3) and roughness r_s, plus one light scale L; the traced
// emissive is E_s = L * e_s.  Given dLoss/d(mean radiance) per pixel, the
// kernel returns dLoss/dparams with every branch decision held fixed (the
// emitter set, Russian roulette, the dielectric choice), i.e. the exact
// derivative of the per-sample estimate of Assets/Tracer.comp:433-593.
//
// Path replay: each sample is traced twice from its RNG state; of the path
// only 8 bytes per sample, and 8 per pixel, are stored between the two passes.
//   pass 1 records which channels of clamp(acc) (Tracer.comp:441) saturate,
//          3 bits per bounce; a saturated channel blocks every earlier term.
//          A pixel's samples share one random stream, so this pass runs them
//          in order and keeps for each sample the stream position at its
//          start and its saturation bits, and per pixel the primary hit that
//          all its samples share.  It is the path kernel itself (k_path with
//          JobDesc::adj_samples), whose images nobody asked for;
//   pass 2 re-traces the same path (same random numbers, same shadow rays)
//          from that position, one lane per (pixel, sample), and accumulates,
//          with W_k = dLoss/dL masked by the later clamps:
//   * direct terms of q_k (normalize(emissive), the next-event term, the
//     dielectric emissive) in a_s, r_s, e, L at each vertex k;
//   * the throughput chain.  Because Russian roulette divides the mask by
//     its largest channel (:545-549), mask_k = P_k / max3(P_k) with P_k the
//     product of the albedos hit before k, so
//       d mask_k,c / d a_s,c' = mask_k,c * n_s (delta_cc' - delta_c'c*) / a_s,c'
//     (c* = argmax3 P_k, n_s = occurrences of s before k), a closed form that
//     needs only the sphere ids of earlier vertices.
// Gradients are reduced per workgroup in LDS and added once per block.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "nee.hpp"
#include "scan.hpp"
#include "traverse.hpp"
#include "vkr_device.hpp"

namespace vkr {

constexpr uint32_t kMaxAdjDepth = 10;

__device__ __forceinline__ uint32_t argmax3(f3 v)
{
    return (v.x >= v.y && v.x >= v.z) ? 0u : (v.y >= v.z ? 1u : 2u);
}

// Pass 2.  Work items: per 8x8 tile, sample by sample, so a wave replays one
// sample of 64 neighbouring pixels.  As in the path kernel, a lane takes one
// vertex per iteration: it shades the hit, evaluates the vertex's emitters up
// to the first whose shadow ray must be traced, and with the last of them
// queues the next segment along.  STACK 0: the scene is scanned.
template <int BLOCK, int STACK, bool LDSGRAD>
__global__ __launch_bounds__(BLOCK) void k_adjoint(const AdjointLaunch A)
{
    constexpr bool SCAN = STACK == 0;
    extern __shared__ uint32_t s_dyn[];
    uint32_t* stk = s_dyn + threadIdx.x;
    uint32_t* chain = s_dyn + STACK * BLOCK + threadIdx.x;          // kMaxAdjDepth entries, stride BLOCK
    float* sgrad = reinterpret_cast<float*>(s_dyn + (STACK + kMaxAdjDepth) * BLOCK);
    const JobDesc& j = A.job;
    const uint32_t ns = j.sc.n_spheres;
    const uint32_t np = 7u * ns + 1u;
    const float* th = A.params;
    const float lscale = th[7u * ns];
    float* grad = LDSGRAD ? sgrad : A.d_params;
    if (LDSGRAD) {
        for (uint32_t i = threadIdx.x; i < np; i += BLOCK) sgrad[i] = 0.0f;
        __syncthreads();
    }

    bool has = false;
    ItemPool pool;
    pool.start((uint32_t)blockIdx.x * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
               gridDim.x * (BLOCK / 64), 64u);
    float uvx = 0.0f, uvy = 0.0f, salt = 0.0f;
    uint32_t depth = 0, zb = 0, nchain = 0, cstar = 0, hs = kMiss;
    f3 ro{}, rd{}, mask{}, N{}, e{}, gp{};
    f3 gA{}, gE{};
    float gR = 0.0f, gL = 0.0f;
    float sum_l = 0.0f;                 // dLoss/dL of this lane's items: every lane adds to it
    uint32_t emi = 0;
    const vkr_material* hm = nullptr;
    uint32_t ei = 0, nee_flags = 0;
    bool hit = false, seg = false, nee = false, term = false;
    uint32_t hprim = kMiss;
    float ht = 0.0f;
    uint32_t c_rays = 0;
    WorkCnt wc{};

    auto claim = [&](uint32_t g) __attribute__((always_inline)) {
        const uint32_t tile = g / (64u * j.spp), s = (g >> 6) % j.spp, within = g & 63u;
        if (tile >= j.n_tiles) return;
        const uint32_t x = (tile % j.tiles_x) * 8u + (within & 7u);
        const uint32_t y = (tile / j.tiles_x) * 8u + (within >> 3);
        if (x >= j.W || y >= j.H) return;
        ++c_rays;                                   // the primary ray, traced by pass 1
        const uint32_t pix = y * j.W + x;
        const uint2 pr = A.primary[pix];
        if (pr.x == kMiss) return;                  // the path ends there
        has = true;
        hit = true;
        hprim = pr.x;
        ht = __uint_as_float(pr.y);
        uvx = (float)x / (float)j.W;
        uvy = (float)y / (float)j.H;
        const uint2 rec = A.samples[(size_t)pix * j.spp + s];
        salt = __uint_as_float(rec.x);
        zb = rec.y;
        const float4 g4 = reinterpret_cast<const float4*>(A.d_radiance)[pix];
        const float inv = 1.0f / (float)j.spp;      // d(mean)/d(sample) (:585)
        gp = f3{g4.x * inv, g4.y * inv, g4.z * inv};
        const float tx = 2.0f * uvx - 1.0f;
        const float ty = 2.0f * uvy - 1.0f;
        f3 dir = add(add(ld3(j.cam_dir), muls(ld3(j.cam_right), tx)), muls(ld3(j.cam_up), ty));
        dir = mul(dir, f3{j.aspect, 1.0f, j.aspect});
        ro = ld3(j.cam_pos);
        rd = normalize(dir);
        mask = f3{1.0f, 1.0f, 1.0f};
        depth = 0;
        nchain = 0;
        cstar = 0;
        seg = false;
        nee = false;
    };
    // W_k: dLoss/dL masked by the clamps that follow vertex k.
    auto weight = [&](uint32_t k) __attribute__((always_inline)) {
        const uint32_t above = (0x3FFu >> (k + 1u)) << (k + 1u);
        return f3{((zb >> 0) & above) ? 0.0f : gp.x, ((zb >> 10) & above) ? 0.0f : gp.y,
                  ((zb >> 20) & above) ? 0.0f : gp.z};
    };
    auto gadd = [&](uint32_t i, float v) __attribute__((always_inline)) {
        if (v != 0.0f) atomicAdd(grad + i, v);
    };
    // Throughput chain at vertex k with term T = mask_k (.) q_k.
    auto chain_grad = [&](f3 W, f3 T) __attribute__((always_inline)) {
        const float tot = W.x * T.x + W.y * T.y + W.z * T.z;
        for (uint32_t i = 0; i < nchain; ++i) {
            const uint32_t s = chain[i * BLOCK];
            const float* a = th + 7u * s;
            const float t0 = W.x * T.x - (cstar == 0 ? tot : 0.0f);
            const float t1 = W.y * T.y - (cstar == 1 ? tot : 0.0f);
            const float t2 = W.z * T.z - (cstar == 2 ? tot : 0.0f);
            if (a[0] != 0.0f) gadd(7u * s + 0u, t0 / a[0]);
            if (a[1] != 0.0f) gadd(7u * s + 1u, t1 / a[1]);
            if (a[2] != 0.0f) gadd(7u * s + 2u, t2 / a[2]);
        }
    };

    while (true) {
        pool.refill(A.pool, A.total, 32u, has, claim);
        if (__ballot(has) == 0) {
            if (pool.dry) break;
            continue;
        }

        // Shade the hit.
        if (has && hit) {
            hit = false;
            const f3 P = add(ro, muls(rd, ht));
            const uint32_t kind = hprim >> 30, idx = hprim & 0x3FFFFFFFu;
            const vkr_material* m;
            hs = kMiss;
            if (kind == 0) {
                const vkr_triangle* T = j.sc.tris_orig + idx;
                const f3 v0 = ld3(T->v0), v1 = ld3(T->v1), v2 = ld3(T->v2);
                const f3 u = sub(v1, v0), v = sub(v2, v0);
                N = f3{(u.y * v.z) - (u.z * v.y), (u.z * v.x) - (u.x * v.z), (u.x * v.y) - (u.y * v.x)};
                const uint32_t mi = T->mat_index;
                m = ((j.sc.flags & VKR_SCENE_TRI_MATERIAL_INDEX) && mi < j.sc.n_materials) ? j.sc.materials + mi
                                                                                           : j.sc.tri_material;
            } else if (kind == 1) {
                const vkr_sphere* S = j.sc.spheres + idx;
                N = divs(sub(P, ld3(S->P)), S->r);
                m = &S->mat;
                hs = idx;
            } else {
                const vkr_plane* Q = j.sc.planes + idx;
                N = ld3(Q->N);
                m = &Q->mat;
            }
            const uint32_t type = m->type;
            if (type == VKR_MAT_DIFFUSE) {
                const float r2 = rng_next(salt, uvx, uvy);
                const float phi = kTwoPi * rng_next(salt, uvx, uvy);
                const f3 dj = muls(jitter(N, phi, sqrt_rn(r2), sqrt_rn(1.0f - r2)), 1.0f - m->metalness);
                hm = m;
                e = f3{0.0f, 0.0f, 0.0f};
                ei = 0;
                rd = normalize(add(reflect(rd, N), dj));
                ro = P;
                nee = true;
                nee_flags = nee_flags_of(j.sc, N, m);
            } else {
                if (type == VKR_MAT_DIELECTRIC) {
                    const f3 emis = ld3(m->emissive);
                    const float rough = m->roughness;
                    const f3 W = weight(depth);
                    const f3 u = mul(W, mask);
                    if (hs != kMiss) {
                        const float* eo = th + 7u * hs + 3u;
                        gadd(7u * hs + 3u, u.x * lscale);
                        gadd(7u * hs + 4u, u.y * lscale);
                        gadd(7u * hs + 5u, u.z * lscale);
                        sum_l += u.x * eo[0] + u.y * eo[1] + u.z * eo[2];
                    }
                    chain_grad(W, mul(mask, emis));
                    mask = mul(mask, ld3(m->albedo));
                    if (hs != kMiss && nchain < kMaxAdjDepth) chain[(nchain++) * BLOCK] = hs;
                    const float cosine = -dot(rd, N) / length(rd);
                    const f3 reflected = reflect(rd, N);
                    const f3 refracted = refract(rd, N, rough);
                    const float prob = eq3(refracted, f3{0.0f, 0.0f, 0.0f}) ? 1.0f : schlick(cosine, rough);
                    const float u2 = rng_next(salt, uvx, uvy);
                    rd = normalize(u2 < prob ? reflected : refracted);
                    ro = P;
                }
                const float p = max3(mask);
                cstar = argmax3(mask);
                const float u = rng_next(salt, uvx, uvy);
                if (!(u > p)) {
                    mask = muls(mask, 1.0f / p);
                    ++depth;
                    seg = depth < j.max_depth;
                }
                has = seg;
            }
        }

        // The vertex's emitters up to the next shadow ray to trace; after the
        // last one the roulette, and the next segment goes along.
        bool sh = false;
        f3 sd{}, cnee{};
        float st = 0.0f;
        if (has && nee) {
            NeeHit h;
            h.P = ro;
            h.N = N;
            h.V = normalize(sub(ld3(j.cam_pos), ro));
            h.alb = ld3(hm->albedo);
            h.rough = hm->roughness;
            h.metal = hm->metalness;
            h.flags = nee_flags;
            while (ei < j.sc.n_emitters && !sh) {
                const float s0 = salt;
                salt = salt + 1.0f;
                salt = salt + 1.0f;
                ++c_rays;
                emi = j.sc.emitters[ei++];
                const vkr_sphere* S = j.sc.spheres + emi;
                if (h.flags && nee_certified(h, S)) continue;
                const NeeEval q = nee_eval(h, S, s0, uvx, uvy);
                cnee = q.c;
                sh = !(cnee.x == 0.0f && cnee.y == 0.0f && cnee.z == 0.0f);
                if (sh) {
                    sd = q.L;
                    st = q.tl;
                    // Pending gradient of this next-event term (added if unoccluded).
                    const f3 u = mul(weight(depth), mask);
                    // albedo of the shaded sphere: kD*a/pi and F0 = mix(0.04, a, metal)
                    const float dF = h.metal * (1.0f - q.p5);
                    const float dkd = -(1.0f - h.metal) * dF;
                    const float sp = q.NDF * q.G / q.den;
                    const f3 al = h.alb;
                    gA = f3{u.x * (((q.kD.x + al.x * dkd) / kPi + sp * dF) * q.att.x * q.NdotL),
                            u.y * (((q.kD.y + al.y * dkd) / kPi + sp * dF) * q.att.y * q.NdotL),
                            u.z * (((q.kD.z + al.z * dkd) / kPi + sp * dF) * q.att.z * q.NdotL)};
                    // roughness: NDF (a2 = r^4) and Smith-Schlick (k = (r+1)^2/8)
                    const float rough = h.rough;
                    const float a2 = rough * rough * rough * rough;
                    const float NdotH = gmax(dot(N, q.H), 0.0f);
                    const float nh2 = NdotH * NdotH;
                    const float dd = nh2 * (a2 - 1.0f) + 1.0f;
                    const float dNdf = (dd - 2.0f * a2 * nh2) / (kPi * dd * dd * dd) * 4.0f * rough * rough * rough;
                    const float k = (rough + 1.0f) * (rough + 1.0f) / 8.0f;
                    const float qv = q.NdotV * (1.0f - k) + k, ql = q.NdotL * (1.0f - k) + k;
                    const float gv = q.NdotV / qv, gl = q.NdotL / ql;
                    const float dgv = -q.NdotV * (1.0f - q.NdotV) / (qv * qv), dgl = -q.NdotL * (1.0f - q.NdotL) / (ql * ql);
                    const float dG = (dgv * gl + gv * dgl) * (rough + 1.0f) / 4.0f;
                    const float dsp = (dNdf * q.G + q.NDF * dG) / q.den;
                    gR = (u.x * q.F.x * q.att.x + u.y * q.F.y * q.att.y + u.z * q.F.z * q.att.z) * dsp * q.NdotL;
                    // emitter emission and light scale through att = (L e / x^2 - 0.001) / 0.999
                    const float* eo = th + 7u * emi + 3u;
                    const float s = 1.0f / (q.x2 * kAttDiv);
                    const f3 w = muls(mul(u, q.brdf), q.NdotL);
                    gE = f3{q.att.x > 0.0f ? w.x * lscale * s : 0.0f, q.att.y > 0.0f ? w.y * lscale * s : 0.0f,
                            q.att.z > 0.0f ? w.z * lscale * s : 0.0f};
                    gL = (q.att.x > 0.0f ? w.x * eo[0] * s : 0.0f) + (q.att.y > 0.0f ? w.y * eo[1] * s : 0.0f) +
                         (q.att.z > 0.0f ? w.z * eo[2] * s : 0.0f);
                }
            }
            if (ei >= j.sc.n_emitters) {
                const float u = rng_next(salt, uvx, uvy);
                term = u > max3(mul(mask, h.alb));
                seg = !term && depth + 1u < j.max_depth;
            }
        }

        // Trace.
        const float dp1 = (float)(depth + (nee ? 2u : 1u));
        const float tmax = 3000.0f / (dp1 * dp1);
        const bool sg = has && seg;
        if (sg) ++c_rays;
        bool occluded = false;
        TravOut tr;
        if constexpr (SCAN) tr = scan_pair(j.sc, ro, sh, sd, st, sg, rd, tmax, j.eps, occluded);
        else tr = traverse_pair<BLOCK, false>(j.sc, ro, sh, sd, st, sg, rd, tmax, j.eps, stk, wc, occluded);
        if (!has) continue;

        if (sh && !occluded) {
            e = add(e, cnee);
            if (hs != kMiss) {
                gadd(7u * hs + 0u, gA.x);
                gadd(7u * hs + 1u, gA.y);
                gadd(7u * hs + 2u, gA.z);
                gadd(7u * hs + 6u, gR);
            }
            gadd(7u * emi + 3u, gE.x);
            gadd(7u * emi + 4u, gE.y);
            gadd(7u * emi + 5u, gE.z);
            sum_l += gL;
        }
        if (nee) {
            if (ei < j.sc.n_emitters) continue;
            nee = false;
            const f3 emis = ld3(hm->emissive);
            const bool all_pos = gmax(gsign(emis.x), 0.0f) == 1.0f && gmax(gsign(emis.y), 0.0f) == 1.0f &&
                                 gmax(gsign(emis.z), 0.0f) == 1.0f;
            const f3 em = all_pos ? normalize(emis) : f3{0.0f, 0.0f, 0.0f};
            const f3 W = weight(depth);
            if (all_pos && hs != kMiss) {
                // d normalize(L e)/de = (I - n n^T) / |e|
                const float* eo = th + 7u * hs + 3u;
                const f3 ev{eo[0], eo[1], eo[2]};
                const float len = length(ev);
                const f3 n = divs(ev, len);
                const f3 u = mul(W, mask);
                const float un = dot(u, n);
                gadd(7u * hs + 3u, (u.x - un * n.x) / len);
                gadd(7u * hs + 4u, (u.y - un * n.y) / len);
                gadd(7u * hs + 5u, (u.z - un * n.z) / len);
            }
            chain_grad(W, mul(mask, add(em, e)));
            mask = mul(mask, ld3(hm->albedo));
            if (hs != kMiss && nchain < kMaxAdjDepth) chain[(nchain++) * BLOCK] = hs;
            cstar = argmax3(mask);
            if (!term) {
                mask = muls(mask, recip_rn(max3(mask)));
                ++depth;
            }
        }
        hit = seg && tr.hit;
        hprim = tr.prim;
        ht = tr.t;
        seg = false;
        has = hit;
    }

    flush_counter(&counter_bank(A.counters, blockIdx.x)->rays, c_rays);
    for (int off = 32; off > 0; off >>= 1) sum_l += __shfl_xor(sum_l, off, 64);
    if (__lane_id() == 0) gadd(7u * ns, sum_l);
    if (LDSGRAD) {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < np; i += BLOCK)
            if (sgrad[i] != 0.0f) atomicAdd(A.d_params + i, sgrad[i]);
    }
}

namespace {
template <int BLOCK, int STACK, bool LDSGRAD>
hipError_t go(const AdjointLaunch& a, size_t lds, hipStream_t s)
{
    const void* fn = reinterpret_cast<const void*>(&k_adjoint<BLOCK, STACK, LDSGRAD>);
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, BLOCK, lds) != hipSuccess || per_cu < 1) per_cu = 1;
    int dev = 0;
    (void)hipGetDevice(&dev);
    const uint32_t need = (a.total + BLOCK - 1u) / BLOCK;
    const uint32_t grid = std::max(1u, std::min((uint32_t)per_cu * compute_units(dev), need));
    hipLaunchKernelGGL((k_adjoint<BLOCK, STACK, LDSGRAD>), dim3(grid), dim3(BLOCK), lds, s, a);
    return hipGetLastError();
}

template <int STACK>
hipError_t go_stack(const AdjointLaunch& a, hipStream_t s)
{
    constexpr int kBlock = 128;
    const size_t base = (size_t)(STACK + kMaxAdjDepth) * kBlock * 4u;
    const size_t grad = (size_t)(7u * a.job.sc.n_spheres + 1u) * 4u;
    return base + grad <= 60u * 1024u ? go<kBlock, STACK, true>(a, base + grad, s) : go<kBlock, STACK, false>(a, base, s);
}
}  // namespace

hipError_t launch_adjoint(const AdjointLaunch& a, uint32_t stack, bool scan, hipStream_t s)
{
    return scan ? go_stack<0>(a, s) : stack <= 32 ? go_stack<32>(a, s) : go_stack<64>(a, s);
}

}  // namespace vkr
