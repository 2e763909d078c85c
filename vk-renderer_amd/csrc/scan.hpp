// scan.hpp - trace_ray over scenes of a few primitives, without a tree.
//
// A tree costs a small scene more than it saves: a dozen dependent node and
// leaf rounds, each about 50 VALU instructions for whichever lanes take part,
// against 25 per sphere with every lane busy, no stack and no divergence.  So
// small scenes (use_scan has the line and what both sides measured) are
// scanned as the reference scans them (Assets/Tracer.comp:374-431).  The
// primitives come through scalar loads (every lane tests the same one), a
// shadow ray and the segment from the same point share what depends on the
// point only, and the square roots and divisions that only rank the hits are
// the hardware's one-ulp estimates:
//   * pass 1 keeps the least and the second least hit distance beyond eps;
//   * the least hit is always accepted by the reference's rule, and only hits
//     within eps above it can replace it.  When the second least is further
//     away than that, and no distance is nearer to eps or to t_max than the
//     estimates' error, the least one wins and its distance is computed once,
//     exactly;
//   * otherwise the lane runs the reference's own loop.
// What bounds it: VALU issue.  Against the tree on the same kernels: 64^2
// reference scene 127 -> 98 us, 1024^2 with present filter 1291 -> 1146 us,
// 256^2, 16 spp, 33 spheres forward + backward 1536 -> 1154 us.  The smallest
// images are bound by a pixel's serial chain instead, see scan_pair_quad.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "traverse.hpp"
#include "vkr_device.hpp"

namespace vkr {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) v4f* cv4f;

__device__ __forceinline__ cv4f const_rows(const void* p) { return (cv4f) reinterpret_cast<unsigned long long>(p); }

// Calls body(row, i) for rows 0 .. n - 1 of a padded array (the padding rows of
// the last run included).  A run is loaded while the one before it is worked
// on: a wave that has its SIMD to itself would otherwise wait out a scalar
// load, as long as three sphere tests, for every row (65 spheres 512^2
// 394 -> 369 us).
template <class Body>
__device__ __forceinline__ void for_rows(const void* rows, uint32_t n, Body&& body)
{
    const cv4f p = const_rows(rows);
    v4f a = p[0], b = p[1], c = p[2], d = p[3];
    for (uint32_t i = 0; i < n; i += kScanRun) {
        const v4f a1 = p[i + 4u], b1 = p[i + 5u], c1 = p[i + 6u], d1 = p[i + 7u];
        body(a, i);
        body(b, i + 1u);
        body(c, i + 2u);
        body(d, i + 3u);
        a = a1;
        b = b1;
        c = c1;
        d = d1;
    }
}

// The least two of a ray's hit distances beyond `lo`, and the least one's key.
struct Nearest {
    float best, second;
    uint32_t key;
    __device__ __forceinline__ void clear()
    {
        best = second = __builtin_huge_valf();
        key = kMiss;
    }
    __device__ __forceinline__ void add(float t, float lo, uint32_t k)
    {
        const float v = t > lo ? t : __builtin_huge_valf();   // NaN: no hit
        key = v < best ? k : key;
        second = __builtin_amdgcn_fmed3f(v, best, second);    // best <= second
        best = fminf(v, best);
    }
};

// A sphere test is h = (oc . d)^2 - (|oc|^2 - r^2), t = -(oc . d) - sqrt(h): the
// reference's b^2 - 4c and (-b - sqrt) / 2 scaled by powers of two, so the same
// floats (DevScene::scan bounds the coordinates well below overflow).
struct SphereTerms {
    float dt, h;
    __device__ __forceinline__ SphereTerms(f3 oc, float cc, f3 d)
    {
        dt = dot(oc, d);
        h = dt * dt - cc;
    }
    __device__ __forceinline__ float near() const { return -dt - __builtin_amdgcn_sqrtf(h); }   // NaN when h < 0
    __device__ __forceinline__ float exact() const { return h < 0.0f ? -1.0f : -dt - sqrt_rn(h); }
};

// The reference's loop over triangles and spheres.  any: stops at the first
// accepted primitive.
__device__ __forceinline__ void scan_exact(const DevScene& sc, f3 o, f3 d, float tmax, float eps, bool any, float& best,
                                           uint32_t& key)
{
    best = tmax;
    key = kMiss;
    for (uint32_t i = 0; i < sc.n_tris && !(any && key != kMiss); ++i) {
        const cv4f p = const_rows(sc.scan_tris) + 3u * i;
        const v4f a = p[0], b = p[1], c = p[2];
        const float t = tri_t(o, d, f3{a.x, a.y, a.z}, f3{b.x, b.y, b.z}, f3{c.x, c.y, c.z}, eps);
        if ((t > eps) && (t < best + eps)) {
            best = t;
            key = i;
        }
    }
    for (uint32_t i = 0; i < sc.n_spheres && !(any && key != kMiss); ++i) {
        const v4f s = const_rows(sc.scan_sph)[i];
        const f3 oc = sub(o, f3{s.x, s.y, s.z});
        const float t = SphereTerms(oc, dot(oc, oc) - s.w, d).exact();
        if ((t > eps) && (t < best + eps)) {
            best = t;
            key = (1u << 30) | i;
        }
    }
}

// Planes: the least two of -(len + o.N) / (d.N) beyond eps, by estimates of
// relative error 2^-22.
__device__ __forceinline__ void scan_planes(const DevScene& sc, f3 o, f3 d, float eps, Nearest& n)
{
    const float lo = eps * (1.0f - 0x1p-18f);
    for_rows(sc.scan_planes, sc.n_planes, [&](v4f q, uint32_t i) __attribute__((always_inline)) {
        const f3 N{q.x, q.y, q.z};
        const float num = q.w + dot(o, N);
        n.add(-num * __builtin_amdgcn_rcpf(dot(d, N)), lo, i);
    });
}

// Whether a plane stops a shadow ray of length tmax (t in (eps, tmax - eps)), n
// its planes from scan_planes.
__device__ __forceinline__ bool scan_plane_stops(const DevScene& sc, f3 o, f3 d, float tmax, float eps, const Nearest& n)
{
    const float lim = tmax - eps, slack = fabsf(lim) * 0x1p-18f;
    if (!(n.best < lim + slack)) return false;
    if (n.best > eps * (1.0f + 0x1p-18f) && n.best < lim - slack) return true;
    WorkCnt wc{};
    return plane_stops<false>(sc, o, d, tmax, eps, wc);
}

// The planes (n, from scan_planes) after triangles and spheres gave (best, prim).
__device__ __forceinline__ void scan_plane_hits(const DevScene& sc, f3 o, f3 d, float eps, const Nearest& n, float& best,
                                                uint32_t& prim)
{
    const float lim = best - eps, slack = (fabsf(best) + eps) * 0x1p-18f;
    if (!(n.best < lim + slack)) return;
    if (n.best > eps * (1.0f + 0x1p-18f) && n.best < lim - slack && n.second > n.best + eps + eps + slack) {
        const float4 q = reinterpret_cast<const float4*>(sc.planes)[4u * n.key + 3u];
        best = plane_t(o, d, f3{q.x, q.y, q.z}, q.w);
        prim = (2u << 30) | n.key;
        return;
    }
    for (uint32_t i = 0; i < sc.n_planes; ++i) {
        const v4f q = const_rows(sc.planes)[4u * i + 3u];
        const float t = plane_t(o, d, f3{q.x, q.y, q.z}, q.w);
        if ((t > eps) && (t < best - eps)) {
            best = t;
            prim = (2u << 30) | i;
        }
    }
}

// How far an estimated sphere distance can be from the exact one: one ulp of
// a root of at most |o - c| + r, and the last rounding.
__device__ __forceinline__ float scan_error(const DevScene& sc, f3 o)
{
    const f3 oc = sub(o, f3{sc.sph_c[0], sc.sph_c[1], sc.sph_c[2]});
    return 5e-7f * (__builtin_amdgcn_sqrtf(dot(oc, oc)) * 1.0001f + sc.scan_reach);
}

// Ends a shadow ray / a closest-hit ray after pass 1.
__device__ __forceinline__ bool scan_end_any(const DevScene& sc, f3 o, f3 d, float tmax, float eps, float err,
                                             const Nearest& n)
{
    const float lim = tmax + eps;
    if (!(n.best < lim + err)) {
        if (n.best >= lim + err) return false;
    } else if (n.best > eps + err && n.best < lim - err) {
        return true;
    }
    float t;
    uint32_t key;
    scan_exact(sc, o, d, tmax, eps, true, t, key);
    return key != kMiss;
}
__device__ __forceinline__ void scan_end_closest(const DevScene& sc, f3 o, f3 d, float tmax, float eps, float err,
                                                 const Nearest& n, float& best, uint32_t& prim)
{
    const float lim = tmax + eps;
    best = tmax;
    prim = kMiss;
    if (!(n.best >= lim + err)) {
        if (n.best > eps + err && n.best < lim - err && !(n.second < n.best + (eps + 2.0f * err))) {
            prim = n.key;
            best = n.best;   // a triangle's distance is exact
            if (n.key >> 30) {
                const float4 s = sc.scan_sph[n.key & 0x3FFFFFFFu];
                const f3 oc = sub(o, f3{s.x, s.y, s.z});
                best = SphereTerms(oc, dot(oc, oc) - s.w, d).exact();
            }
        } else {
            scan_exact(sc, o, d, tmax, eps, false, best, prim);
        }
    }
}

// One ray per lane (active: the lane has one).  sc is uniform.
__device__ __forceinline__ TravOut scan_ray(const DevScene& sc, f3 o, f3 d, float tmax, float eps, bool any, bool active)
{
    const float err = scan_error(sc, o), lo = eps - err;
    Nearest n;
    n.clear();
    for (uint32_t i = 0; i < sc.n_tris; ++i) {
        const cv4f p = const_rows(sc.scan_tris) + 3u * i;
        const v4f a = p[0], b = p[1], c = p[2];
        n.add(tri_t(o, d, f3{a.x, a.y, a.z}, f3{b.x, b.y, b.z}, f3{c.x, c.y, c.z}, eps), eps, i);
    }
    for_rows(sc.scan_sph, sc.n_spheres, [&](v4f s, uint32_t i) __attribute__((always_inline)) {
        const f3 oc = sub(o, f3{s.x, s.y, s.z});
        n.add(SphereTerms(oc, dot(oc, oc) - s.w, d).near(), lo, (1u << 30) | i);
    });
    TravOut r{kMiss, tmax, false};
    if (!active) return r;
    if (any) {
        r.hit = scan_end_any(sc, o, d, tmax, eps, err, n);
        if (r.hit) return r;
    } else {
        scan_end_closest(sc, o, d, tmax, eps, err, n, r.t, r.prim);
    }
    n.clear();
    scan_planes(sc, o, d, eps, n);
    if (any) {
        r.hit = scan_plane_stops(sc, o, d, tmax, eps, n);
    } else {
        scan_plane_hits(sc, o, d, eps, n, r.t, r.prim);
        r.hit = r.prim != kMiss;
    }
    return r;
}

// The wave's queued rays, as traverse_pool takes them: 64 at a time.
__device__ __forceinline__ void scan_pool(const JobDesc& j, uint32_t total, const uint32_t* cpre,
                                          const unsigned long long* colm, uint32_t* occ, uint2* res,
                                          const char* __restrict__ wrec)
{
    for (uint32_t base = 0; base < total; base += 64u) {
        const uint32_t i = base + __lane_id();
        const bool act = i < total;
        uint32_t slot = 0, lo = 0;
        float4 h{}, r{};
        if (act) {
            pool_item(cpre, colm, i, slot, lo);
            h = *reinterpret_cast<const float4*>(wrec + (kWHead + lo * 16u));
            r = *reinterpret_cast<const float4*>(wrec + (kWSlotD + (slot * 64u + lo) * 16u));
        }
        const TravOut t = scan_ray(j.sc, f3{h.x, h.y, h.z}, f3{r.x, r.y, r.z}, r.w, j.eps, slot != 0u, act);
        if (act) {
            if (slot == 0u) res[lo] = make_uint2(t.prim, __float_as_uint(t.t));
            else if (t.hit) atomicOr(occ + lo, 1u << slot);
        }
    }
}

// A shadow ray (sh) and a path segment (seg) from one origin, as traverse_pair.
__device__ __forceinline__ TravOut scan_pair(const DevScene& sc, f3 o, bool sh, f3 sd, float st, bool seg, f3 d,
                                             float tmax, float eps, bool& occluded)
{
    const float err = scan_error(sc, o), lo = eps - err;
    Nearest n, m;
    n.clear();
    m.clear();
    for (uint32_t i = 0; i < sc.n_tris; ++i) {
        const cv4f p = const_rows(sc.scan_tris) + 3u * i;
        const v4f a = p[0], b = p[1], c = p[2];
        const f3 v0{a.x, a.y, a.z}, e1{b.x, b.y, b.z}, e2{c.x, c.y, c.z};
        n.add(tri_t(o, d, v0, e1, e2, eps), eps, i);
        m.add(tri_t(o, sd, v0, e1, e2, eps), eps, i);
    }
    for_rows(sc.scan_sph, sc.n_spheres, [&](v4f s, uint32_t i) __attribute__((always_inline)) {
        const f3 oc = sub(o, f3{s.x, s.y, s.z});
        const float cc = dot(oc, oc) - s.w;
        n.add(SphereTerms(oc, cc, d).near(), lo, (1u << 30) | i);
        m.add(SphereTerms(oc, cc, sd).near(), lo, i);
    });
    occluded = sh && scan_end_any(sc, o, sd, st, eps, err, m);
    TravOut r{kMiss, tmax, false};
    if (seg) scan_end_closest(sc, o, d, tmax, eps, err, n, r.t, r.prim);
    n.clear();
    m.clear();
    scan_planes(sc, o, d, eps, n);
    if (sh && !occluded) {
        scan_planes(sc, o, sd, eps, m);
        occluded = scan_plane_stops(sc, o, sd, st, eps, m);
    }
    if (seg) scan_plane_hits(sc, o, d, eps, n, r.t, r.prim);
    r.hit = r.prim != kMiss;
    return r;
}

// scan_pair by four lanes: lane 4k has the rays (sh, seg; its three neighbours
// none), each of the four tests every fourth primitive for them, and two
// exchanges bring the least two together.  For images so small that lanes are
// idle anyway and the time is a pixel's serial chain, of which the tests of 33
// spheres are a third (256^2, 16 spp, 33 spheres, forward + backward
// 1134 -> 1032 us; 64^2 reference scene 90.5 -> 84.7).
__device__ __forceinline__ float quad_first(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x00, 0xF, 0xF, true));
}
__device__ __forceinline__ f3 quad_first(f3 v) { return f3{quad_first(v.x), quad_first(v.y), quad_first(v.z)}; }
template <int PERM>
__device__ __forceinline__ void quad_merge(Nearest& n)
{
    const float b = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(n.best), PERM, 0xF, 0xF, true));
    const float s = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(n.second), PERM, 0xF, 0xF, true));
    const uint32_t k = (uint32_t)__builtin_amdgcn_mov_dpp((int)n.key, PERM, 0xF, 0xF, true);
    n.second = fminf(fmaxf(n.best, b), fminf(n.second, s));
    n.key = b < n.best ? k : n.key;
    n.best = fminf(n.best, b);
}
__device__ __forceinline__ void quad_merge(Nearest& n)
{
    quad_merge<0xB1>(n);   // lanes 1 0 3 2
    quad_merge<0x4E>(n);   // lanes 2 3 0 1
}
// Calls body(row, i) for this lane's quarter of the rows.
template <class Body>
__device__ __forceinline__ void for_quad_rows(const float4* rows, uint32_t n, uint32_t q, Body&& body)
{
    float4 a = rows[q];
    for (uint32_t i = 0; i < n; i += kScanRun) {
        const float4 a1 = rows[i + kScanRun + q];
        body(a, i + q);
        a = a1;
    }
}
__device__ __forceinline__ TravOut scan_pair_quad(const DevScene& sc, f3 o, bool sh, f3 sd, float st, bool seg, f3 d,
                                                  float tmax, float eps, bool& occluded)
{
    const uint32_t q = __lane_id() & 3u;
    const f3 qo = quad_first(o), qd = quad_first(d), qs = quad_first(sd);
    const float err = scan_error(sc, qo), lo = eps - err;
    Nearest n, m, np, mp;
    n.clear();
    m.clear();
    np.clear();
    mp.clear();
    for (uint32_t i = q; i < sc.n_tris; i += 4u) {
        const float4* p = reinterpret_cast<const float4*>(sc.scan_tris + i);
        const float4 a = p[0], b = p[1], c = p[2];
        const f3 v0{a.x, a.y, a.z}, e1{b.x, b.y, b.z}, e2{c.x, c.y, c.z};
        n.add(tri_t(qo, qd, v0, e1, e2, eps), eps, i);
        m.add(tri_t(qo, qs, v0, e1, e2, eps), eps, i);
    }
    for_quad_rows(sc.scan_sph, sc.n_spheres, q, [&](float4 s, uint32_t i) __attribute__((always_inline)) {
        const f3 oc = sub(qo, f3{s.x, s.y, s.z});
        const float cc = dot(oc, oc) - s.w;
        n.add(SphereTerms(oc, cc, qd).near(), lo, (1u << 30) | i);
        m.add(SphereTerms(oc, cc, qs).near(), lo, i);
    });
    const float lop = eps * (1.0f - 0x1p-18f);
    for_quad_rows(sc.scan_planes, sc.n_planes, q, [&](float4 p, uint32_t i) __attribute__((always_inline)) {
        const f3 N{p.x, p.y, p.z};
        const float num = p.w + dot(qo, N);
        np.add(-num * __builtin_amdgcn_rcpf(dot(qd, N)), lop, i);
        mp.add(-num * __builtin_amdgcn_rcpf(dot(qs, N)), lop, i);
    });
    quad_merge(n);
    quad_merge(m);
    quad_merge(np);
    quad_merge(mp);
    occluded = sh && (scan_end_any(sc, o, sd, st, eps, err, m) || scan_plane_stops(sc, o, sd, st, eps, mp));
    TravOut r{kMiss, tmax, false};
    if (!seg) return r;
    scan_end_closest(sc, o, d, tmax, eps, err, n, r.t, r.prim);
    scan_plane_hits(sc, o, d, eps, np, r.t, r.prim);
    r.hit = r.prim != kMiss;
    return r;
}

}  // namespace vkr
