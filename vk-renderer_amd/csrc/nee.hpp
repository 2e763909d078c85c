// nee.hpp - next-event estimation at a diffuse hit (Assets/Tracer.comp:458-504),
// shared by the path kernel and the adjoint.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "vkr_device.hpp"

namespace vkr {

// A diffuse hit as next-event estimation sees it.
constexpr uint32_t kNeeZero = 1u;     // every emitter contributes exactly +-0 (mirror, |N|^2 < 0.9999)
constexpr uint32_t kNeeFin = 2u;      // the BRDF factor is bounded for any sample
constexpr uint32_t kNeeMirror = 4u;   // metalness 1, roughness 0: zero unless (N.H)^2 rounds to 1
struct NeeHit {
    f3 P, N, V, alb;
    float rough, metal;
    uint32_t flags;                   // kNee*
};

// The kNee* flags of a hit with normal N on material m.
//
// Metalness 1 and roughness 0 (the reference's `mirror`):
// kD = (1 - F) * 0 and NDF = 0 / (pi * denom^2), where
// denom = 1 - NdotH^2 >= 8e-5 once |N|^2 < 0.9999 (|H| = 1),
// so with finite albedo, F, G and attenuation an emitter's
// contribution is exactly +-0 whatever its sample (F is
// finite when V stays outside the emitter's cone, which is
// checked per emitter).
//
// More generally, with |albedo|, |metalness| <= 16,
// k = (r+1)^2/8 in [2^-10, 1], |N|^2 <= 2^10 and the GGX
// denominator 1 - NdotH^2 (1 - a2) >= 2^-10 for every
// |H| = 1 (or a2 >= 1), the factor (kD alb/pi + specular)
// is below 2^72 for any sample: F <= 2^10, G <= 2^30,
// NDF <= 2^22.  An emitter whose attenuation is exactly 0,
// or whose whole sampling cone lies below the horizon
// (NdotL = +0), then contributes exactly +-0 as well.
__device__ __forceinline__ uint32_t nee_flags_of(const DevScene& sc, f3 N, const vkr_material* m)
{
    const f3 alb = ld3(m->albedo);
    const float nn = dot(N, N);
    const float rough = m->roughness, metal = m->metalness;
    const bool nee_zero = sc.emitters_bounded && metal == 1.0f && rough == 0.0f &&
               fabsf(alb.x) < 1e30f && fabsf(alb.y) < 1e30f && fabsf(alb.z) < 1e30f &&
               nn < 0.9999f;
    const float rp = rough + 1.0f;
    const float k = (rp * rp) / 8.0f;
    const float a = rough * rough;
    const float a2 = a * a;
    const bool nee_fin = sc.emitters_bounded && fabsf(alb.x) <= 16.0f && fabsf(alb.y) <= 16.0f &&
              fabsf(alb.z) <= 16.0f && fabsf(metal) <= 16.0f && k >= 0x1p-10f && k <= 1.0f &&
              nn <= 1024.0f &&
              (a2 >= 1.0f || 1.0f - (nn * (1.0f + 0x1p-16f)) * (1.0f - a2) >= 0x1p-10f);
    // Other mirror hits: kD = 0 and NDF = 0 / (pi (1 - NdotH^2)^2)
    // is 0 unless NdotH^2 rounds to exactly 1 (then NaN).
    const bool nee_mirror = !nee_zero && sc.emitters_bounded && metal == 1.0f &&
                            rough == 0.0f && fabsf(alb.x) <= 16.0f && fabsf(alb.y) <= 16.0f &&
                            fabsf(alb.z) <= 16.0f && nn <= 1024.0f;
    return (nee_zero ? kNeeZero : 0u) | (nee_fin ? kNeeFin : 0u) | (nee_mirror ? kNeeMirror : 0u);
}

// Whether emitter S contributes exactly +-0 at hit h whatever its sample.  An
// emitter so certified needs no draws and no shadow ray.  The tests carry
// margins far above the rounding of the fast reciprocal / square-root
// estimates they use; an emitter they cannot certify is evaluated in full.
__device__ __forceinline__ bool nee_certified(const NeeHit& h, const vkr_sphere* S)
{
    const f3 P = h.P, N = h.N, V = h.V;
    const float nn = dot(N, N);
    const f3 l0 = sub(ld3(S->P), P);
    const float sr = S->r;
    const float ll2 = dot(l0, l0);
    // Attenuation < 2^41: the hit point is at least 2^-9 radii from the centre.
    if (!(ll2 >= (sr * sr) * 0x1p-18f)) return false;
    // A sample L has cosa >= cos_a_max and sina <= sig, sig^2 = s2 + 1e-6
    // >= the kernel's 1 - cos_a_max^2, so it lies within t = 1.5708 sig of
    // w = l0 / |l0|.
    const float il = __builtin_amdgcn_rsqf(ll2);
    const float sw = sr * il;
    const float sig2 = fminf(sw * sw + 1e-6f, 1.0f);
    const float sig = __builtin_amdgcn_sqrtf(sig2) * (1.0f + 1e-6f);
    const float t = 1.5708f * sig;
    // Every certificate needs the Fresnel term finite: with V at least
    // 0.01 rad outside the cone, dot(H, V) <= 1 - 1e-5, so
    // pow(1 - dot(H, V), 5) never sees a negative base (NaN, :276).
    const f3 w = muls(l0, il);
    const float cph = dot(V, w);
    const float tv = t + 0.01f;
    if (!(tv < 1.5f && cph < 1.0f - 0.5f * tv * tv - 1e-6f)) return false;
    if (h.flags & kNeeZero) return true;
    if (h.flags & kNeeFin) {
        // (b) cone below the horizon: with c = cos(N, l0) < 0 and
        // s = sin(N, l0) (from |N x l0|, no cancellation),
        // cos(N, L) <= sig s + cl c < -1e-4.
        const float inv = __builtin_amdgcn_rsqf(nn * ll2);
        const float cc = dot(N, l0) * inv;
        const f3 cr = cross(N, l0);
        const float ss = __builtin_amdgcn_sqrtf(dot(cr, cr)) * inv;
        const float cl = __builtin_amdgcn_sqrtf(1.0f - sig2) * (1.0f - 1e-6f);
        if (cc < 0.0f && sig * ss + cl * cc < -1e-4f) return true;
    }
    if (h.flags & kNeeMirror) {
        // (c) mirror hits: H = normalize(V + L) stays within
        // dl >= t / (2 cos((phi0 + t) / 2)) of H0 = normalize(V + w)
        // (|dH| <= |dL| / |V + L|; phi0 = angle(V, w) < 107.5 deg, t < 1,
        // so the path never nears V + L = 0).  If |N| cos(N, H) then stays
        // at least 2e-4 away from 1, NdotH^2 cannot round to 1 and the
        // sample is +-0.
        const f3 vw = cross(V, w);
        const float sph = __builtin_amdgcn_sqrtf(dot(vw, vw));
        const float csum = (cph >= 0.0f ? cph * (1.0f - 0.5f * t * t) : cph) - sph * t;
        const float half = __builtin_amdgcn_sqrtf(fmaxf(0.5f * (1.0f + csum), 0.0f));
        if (cph > -0.3f && half >= 0.05f && t < 1.0f) {
            const float dl = t * __builtin_amdgcn_rcpf(2.0f * half) * 1.001f + 1e-5f;
            const f3 hv = add(V, w);
            const float hh = dot(hv, hv);
            const float ihn = __builtin_amdgcn_rsqf(hh * nn);
            const float c0 = dot(N, hv) * ihn;
            const f3 nh = cross(N, hv);
            const float s0 = __builtin_amdgcn_sqrtf(dot(nh, nh)) * ihn;
            const float nrm = __builtin_amdgcn_sqrtf(nn);
            const float cd = 1.0f - 0.5f * dl * dl;
            const float hi = c0 >= cd - 1e-4f ? 1.0f : (c0 >= 0.0f ? c0 : c0 * cd) + s0 * dl;
            const float lo = (c0 >= 0.0f ? c0 * cd : c0) - s0 * dl;
            if (dl < 1.0f && hh > 1e-6f && (nrm * hi < 1.0f - 2e-4f || nrm * lo > 1.0f + 2e-4f)) return true;
        }
    }
    if (h.flags & kNeeFin) {
        // (a) attenuation exactly 0 (:478-479): with the kernel's own x,
        // emis / x^2 <= kAttSub in every channel, tested with a 2^-16 margin.
        const float tl0 = length(l0) - sr;
        const float x = tl0 / sr + 1.0f;
        const float lim = (kAttSub * (x * x)) * (1.0f - 0x1p-16f);
        const f3 em = ld3(S->mat.emissive);
        if (em.x <= lim && em.y <= lim && em.z <= lim) return true;
    }
    return false;}

// Emitter S's next-event sample at hit h, evaluated in full
// (Assets/Tracer.comp:464-502), with the random stream at `salt` before its
// two draws.
struct NeeEval {
    f3 L;                  // the shadow ray's direction
    float tl;              // and its length
    f3 c;                  // the contribution added when it is unoccluded
    // Its factors, for the adjoint: c = (kD albedo / pi + F NDF G / den) att NdotL.
    f3 att, F, kD, brdf, H;
    float x2, p5, NDF, G, den, NdotV, NdotL;
};
__device__ __forceinline__ NeeEval nee_eval(const NeeHit& h, const vkr_sphere* S, float salt, float uvx, float uvy)
{
    NeeEval q;
    const f3 P = h.P, N = h.N, V = h.V;
    const f3 sP = ld3(S->P);
    const float sr = S->r;
    const f3 l0 = sub(sP, P);
    float dist;
    const f3 w0 = normalize_len(l0, dist);
    q.tl = dist - sr;
    const float cos_a_max = sqrt_rn(1.0f - gclamp(sr * sr / dot(l0, l0), 0.0f, 1.0f));
    const float cosa = gmix(cos_a_max, 1.0f, rng_next(salt, uvx, uvy));
    const float phi = kTwoPi * rng_next(salt, uvx, uvy);
    q.L = jitter_w(w0, phi, sqrt_rn(1.0f - cosa * cosa), cosa);

    const float x = q.tl / sr + 1.0f;
    q.x2 = x * x;
    f3 att = divs(muls(ld3(S->mat.emissive), 1.0f), q.x2);
    att = mul_recip(subs(att, kAttSub), kd(kAttDivR));
    q.att = maxs(att, 0.0f);
    const f3 F0 = mix3(f3{0.04f, 0.04f, 0.04f}, h.alb, h.metal);
    q.H = normalize(add(V, q.L));
    q.NDF = distribution_ggx(N, q.H, h.rough);
    q.G = geometry_smith(N, V, q.L, h.rough);
    q.p5 = pow5(1.0f - gmax(dot(q.H, V), 0.0f));
    q.F = fresnel_schlick_p(q.p5, F0);
    q.kD = muls(ssub(1.0f, q.F), 1.0f - h.metal);
    q.NdotV = gmax(dot(N, V), 0.0f);
    q.NdotL = gmax(dot(N, q.L), 0.0f);
    q.den = gmax(4.0f * q.NdotV * q.NdotL, 0.001f);
    const f3 specular = divs(muls(q.F, q.NDF * q.G), q.den);
    q.brdf = add(mul_recip(mul(q.kD, h.alb), kd(kPiR)), specular);
    q.c = muls(mul(q.brdf, q.att), q.NdotL);
    return q;
}

// The next-event sample of emitter `ei` at hit h with the random stream at
// `salt` before its two draws (the caller advances its own copy).  Returns
// false when the contribution is exactly +-0: then adding it cannot change e
// whatever the shadow ray finds, so the ray is not traced.  Else L is the
// shadow ray's direction, tl its length and c the contribution added when it
// is unoccluded.
__device__ __forceinline__ bool nee_sample(const JobDesc& j, const NeeHit& h, uint32_t ei, float salt, float uvx,
                                           float uvy, f3& L, float& tl, f3& c)
{
    const vkr_sphere* S = j.sc.spheres + j.sc.emitters[ei];
    if (h.flags && nee_certified(h, S)) return false;
    const NeeEval q = nee_eval(h, S, salt, uvx, uvy);
    L = q.L;
    tl = q.tl;
    c = q.c;
    return !(c.x == 0.0f && c.y == 0.0f && c.z == 0.0f);
}

}  // namespace vkr
