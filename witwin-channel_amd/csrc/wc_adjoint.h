// Reverse-mode (adjoint) forms of the transport operators of wc_em.h. One
// reverse sweep gives every derivative of one path at about the cost of two or
// three evaluations, where forward mode repeats each operation for every
// parameter and keeps every intermediate that many times over.
//
// Conventions: a real loss l; the cotangent of a real x is dl/dx, of a complex
// z the number g with dl = Re(conj(g) dz), so for holomorphic w = f(z)
// g_z += conj(f'(z)) g_w. Functions named *_adj add into their g_ outputs.
// Clamps pass the derivative on the side that w_max / w_min of the dual
// numbers select, and the fallback branches of safe_normalize and
// stable_perp_basis differentiate the fallback.
#pragma once

#include "wc_em.h"

namespace wc {

template <typename R> WC_HD Cx<R> conj(const Cx<R>& a) { return {a.re, -a.im}; }
WC_HD Cx<float> cmulj(const Cx<float>& a, const Cx<float>& g) {  // conj(a) * g
    return {a.re * g.re + a.im * g.im, a.re * g.im - a.im * g.re};
}
WC_HD float cdotr(const Cx<float>& a, const Cx<float>& g) { return a.re * g.re + a.im * g.im; }  // Re(conj(a) g)
WC_HD Cx<float> cinv(const Cx<float>& a) {
    const float inv = 1.0f / (a.re * a.re + a.im * a.im);
    return {a.re * inv, -a.im * inv};
}
WC_HD void acc(Cx<float>& a, const Cx<float>& b) {
    a.re += b.re;
    a.im += b.im;
}
WC_HD void acc(V3<float>& a, const V3<float>& b) {
    a.x += b.x;
    a.y += b.y;
    a.z += b.z;
}
// cotangent of a real axis v in c3_axis(v, s) or c3_dot_real(., v)
WC_HD V3<float> c3_axis_adj(const C3<float>& g, const Cx<float>& s) {
    return {cdotr(s, g.x), cdotr(s, g.y), cdotr(s, g.z)};
}
WC_HD V3<float> zero3() { return {0.0f, 0.0f, 0.0f}; }

// y = v / (|v| + EPS)
WC_HD void normalize_adj(const V3<float>& v, float n, const V3<float>& gy, V3<float>& gv) {
    const float inv = 1.0f / (n + kEpsF);
    const float c = n > 0.0f ? dot(v, gy) * inv * inv / n : 0.0f;
    gv.x += gy.x * inv - c * v.x;
    gv.y += gy.y * inv - c * v.y;
    gv.z += gy.z * inv - c * v.z;
}

// |v|: zero derivative at the origin
WC_HD void norm_adj(const V3<float>& v, float n, float g, V3<float>& gv) {
    const float c = n > 0.0f ? g / n : 0.0f;
    gv.x += c * v.x;
    gv.y += c * v.y;
    gv.z += c * v.z;
}

// safe_normalize(v, fallback); true when v was normalized (gv), false when the
// fallback was (gfb)
WC_HD bool safe_normalize_adj(const V3<float>& v, const V3<float>& fallback, const V3<float>& gy, V3<float>& gv,
                              V3<float>& gfb) {
    const float n = norm(v);
    if (n > kSmallEpsF) {
        normalize_adj(v, n, gy, gv);
        return true;
    }
    normalize_adj(fallback, norm(fallback), gy, gfb);
    return false;
}

// transverse(dir, pol) = pol - dir (pol . dir)
WC_HD void transverse_adj(const V3<float>& dir, const V3<float>& pol, const V3<float>& gy, V3<float>& gdir,
                          V3<float>& gpol) {
    const float pd = dot(pol, dir), dg = dot(dir, gy);
    acc(gpol, gy - dir * dg);
    acc(gdir, -(gy * pd) - pol * dg);
}

WC_HD void stable_perp_adj(const V3<float>& ray, const V3<float>& preferred, const V3<float>& gy, V3<float>& gray,
                           V3<float>& gpref) {
    const V3<float> proj = preferred - ray * dot(preferred, ray);
    const V3<float> alt = fabsf(ray.z) < 0.9f ? V3<float>{0.f, 0.f, 1.f} : V3<float>{0.f, 1.f, 0.f};
    const V3<float> alt_proj = alt - ray * dot(alt, ray);
    V3<float> gp = zero3(), ga = zero3(), none = zero3();
    if (safe_normalize_adj(proj, alt_proj, gy, gp, ga)) transverse_adj(ray, preferred, gp, gray, gpref);
    else transverse_adj(ray, alt, ga, gray, none);
}

// cross(a, b) normalized, falling back to stable_perp_basis(b, a): the s / p
// axes of a bounce
WC_HD void perp_axis_adj(const V3<float>& a, const V3<float>& b, const V3<float>& gy, V3<float>& ga, V3<float>& gb) {
    const V3<float> v = cross(a, b);
    const float n = norm(v);
    if (n > kSmallEpsF) {
        V3<float> gv = zero3();
        normalize_adj(v, n, gy, gv);
        acc(ga, cross(b, gv));
        acc(gb, cross(gv, a));
        return;
    }
    const V3<float> fb = stable_perp_basis(b, a);
    V3<float> gfb = zero3();
    normalize_adj(fb, norm(fb), gy, gfb);
    stable_perp_adj(b, a, gfb, gb, ga);
}

// Adjoint of slab_fresnel. With i the interface coefficient, ph = e^{-2jq}:
//   r = gain i (1 - ph) / (1 - i^2 ph)
//   dr/di = gain (1 - ph)(1 + i^2 ph) / den^2,  dr/dph = gain i (i^2 - 1) / den^2
//   i = (A - root) / (A + root): di/dA = 2 root / (A + root)^2, di/droot = -2 A / (A + root)^2
struct SlabGrad {
    float ct, eps, sig, gain, thick, freq;
};
WC_HD void slab_fresnel_adj(float cos_theta, float eps_r, float sigma_e, float mu_r, float gain, float thickness,
                            float frequency_hz, const Cx<float>& g_te, const Cx<float>& g_tm, SlabGrad& g) {
    const float w_raw = frequency_hz * (float)kTwoPi;
    const float omega = fmaxf(w_raw, kSmallEpsF);
    const float wl_raw = (float)kC0 / frequency_hz;
    const float wavelength = fmaxf(wl_raw, kSmallEpsF);
    const float ca = fabsf(cos_theta);
    const float ct = fminf(fmaxf(ca, kSmallEpsF), 1.0f);
    const float sin2 = fmaxf(1.0f - ct * ct, 0.0f);
    const float eps = fmaxf(eps_r, kSmallEpsF);
    const float sig = fmaxf(sigma_e, 0.0f);
    const float mu = fmaxf(mu_r, kSmallEpsF);
    const Cx<float> eta{eps, -(sig / omega) * (float)(1.0 / kEps0)};
    const Cx<float> z{eta.re * mu - sin2, eta.im * mu};
    const Cx<float> root = csqrt(z);
    const float q_scale = fmaxf(thickness, 0.0f) * (float)kTwoPi / wavelength;
    const Cx<float> ph = scale(cexpj(-(root.re * q_scale * 2.0f)), expf(root.im * q_scale * 2.0f));
    const Cx<float> one{1.0f, 0.0f};
    const Cx<float> one_ph = one - ph;
    Cx<float> g_root{0.0f, 0.0f}, g_ph{0.0f, 0.0f};
    // one polarization: returns the cotangent of A
    auto polarization = [&](const Cx<float>& A, const Cx<float>& g_r) {
        const Cx<float> inv = cinv(A + root);
        const Cx<float> i = (A - root) / (A + root);
        const Cx<float> i2ph = i * i * ph;
        const Cx<float> dinv = cinv(one - i2ph);
        g.gain += cdotr(i * one_ph * dinv, g_r);
        const Cx<float> h = cmulj(dinv * dinv, scale(g_r, gain));
        const Cx<float> g_i = cmulj(one_ph * (one + i2ph), h);
        acc(g_ph, cmulj(i * (i * i - one), h));
        const Cx<float> k = cmulj(inv * inv, scale(g_i, 2.0f));
        acc(g_root, -cmulj(A, k));
        return cmulj(root, k);
    };
    const Cx<float> g_ate = polarization(Cx<float>{mu * ct, 0.0f}, g_te);
    const Cx<float> g_atm = polarization(scale(eta, ct), g_tm);
    float g_ct = mu * g_ate.re + cdotr(eta, g_atm);
    Cx<float> g_eta = scale(g_atm, ct);
    // ph = exp(-2j root q_scale)
    const Cx<float> g_q = cmulj(Cx<float>{2.0f * ph.im, -2.0f * ph.re}, g_ph);
    acc(g_root, scale(g_q, q_scale));
    const float g_qs = cdotr(root, g_q);
    // root = sqrt(z), z = eta mu - sin2
    if (root.re != 0.0f || root.im != 0.0f) {
        const Cx<float> g_z = cmulj(cinv(scale(root, 2.0f)), g_root);
        acc(g_eta, scale(g_z, mu));
        g_ct += 2.0f * ct * g_z.re;  // -d sin2 = 2 ct dct
    }
    if (ca >= kSmallEpsF && ca <= 1.0f) g.ct += cos_theta < 0.0f ? -g_ct : g_ct;
    if (eps_r >= kSmallEpsF) g.eps += g_eta.re;
    if (sigma_e >= 0.0f) g.sig -= g_eta.im / omega * (float)(1.0 / kEps0);
    if (thickness >= 0.0f) g.thick += g_qs * (float)kTwoPi / wavelength;
    float g_f = 0.0f;
    if (w_raw >= kSmallEpsF) g_f -= g_eta.im * eta.im / omega * (float)kTwoPi;
    if (wl_raw >= kSmallEpsF) g_f += g_qs * q_scale / frequency_hz;
    g.freq += g_f;
}

// Adjoint of reflect_c3 at one bounce: g_out / g_dir are the cotangents of the
// reflected field and direction; adds to those of the incoming field (returned
// in g_value), the incident direction, the normal and the slab parameters
// (grad.ct is scratch).
WC_HD void reflect_c3_adj(const C3<float>& value, const V3<float>& incident, const V3<float>& normal_in, float eps_r,
                          float sigma_e, float mu_r, float gain, float thickness, float frequency_hz,
                          const C3<float>& g_out, const V3<float>& g_dir, C3<float>& g_value, V3<float>& g_inc,
                          V3<float>& g_normal, SlabGrad& grad) {
    const V3<float> ez{0.f, 0.f, 1.f};
    const V3<float> n0 = safe_normalize(normal_in, ez);
    const bool flip = dot(incident, n0) > 0.0f;
    const V3<float> n = flip ? -n0 : n0;
    const float din = dot(incident, n);
    const V3<float> rv = incident - n * (din * 2.0f);
    const V3<float> refl = safe_normalize(rv, -incident);
    const V3<float> s = safe_normalize(cross(n, incident), stable_perp_basis(incident, n));
    const V3<float> p_in = safe_normalize(cross(s, incident), stable_perp_basis(incident, s));
    const V3<float> p_out = safe_normalize(cross(s, refl), stable_perp_basis(refl, s));
    Cx<float> te, tm;
    slab_fresnel(fabsf(din), eps_r, sigma_e, mu_r, gain, thickness, frequency_hz, te, tm);
    const Cx<float> e_s = c3_dot_real(value, s), e_p = c3_dot_real(value, p_in);
    // out = s (te e_s) + p_out (tm e_p)
    const Cx<float> g_ts = c3_dot_real(g_out, s), g_tp = c3_dot_real(g_out, p_out);
    V3<float> g_s = c3_axis_adj(g_out, te * e_s);
    const V3<float> g_po = c3_axis_adj(g_out, tm * e_p);
    grad.ct = 0.0f;
    slab_fresnel_adj(fabsf(din), eps_r, sigma_e, mu_r, gain, thickness, frequency_hz, cmulj(e_s, g_ts),
                     cmulj(e_p, g_tp), grad);
    const Cx<float> g_es = cmulj(te, g_ts), g_ep = cmulj(tm, g_tp);
    g_value = c3_axis(s, g_es) + c3_axis(p_in, g_ep);
    acc(g_s, c3_axis_adj(value, g_es));
    const V3<float> g_pi = c3_axis_adj(value, g_ep);
    V3<float> g_refl = g_dir, g_n = zero3();
    perp_axis_adj(s, refl, g_po, g_s, g_refl);
    perp_axis_adj(s, incident, g_pi, g_s, g_inc);
    perp_axis_adj(n, incident, g_s, g_n, g_inc);
    V3<float> g_rv = zero3(), g_fb = zero3();
    if (!safe_normalize_adj(rv, -incident, g_refl, g_rv, g_fb)) acc(g_inc, -g_fb);
    acc(g_inc, g_rv);
    acc(g_n, g_rv * (-2.0f * din));
    const float g_din = (din < 0.0f ? -grad.ct : grad.ct) - 2.0f * dot(n, g_rv);
    acc(g_inc, n * g_din);
    acc(g_n, incident * g_din);
    if (flip) g_n = -g_n;
    const float nn = norm(normal_in);
    if (nn > kSmallEpsF) normalize_adj(normal_in, nn, g_n, g_normal);
}

// prop = amp e^{j ph}, ph = -k L (value reduced in double), amp = 1 / (2 k La):
// cotangents of k, of the phase length L and of the amplitude length La. The
// clamped flags say whether k / La sit on their lower bound.
WC_HD void carrier_adj(const Cx<float>& prop, float k, float k_amp, float L, float La, bool k_free, bool la_free,
                       const Cx<float>& g_prop, float& g_k, float& g_L, float& g_la) {
    // amp g_amp = Re(conj(prop) g), g_ph = Re(conj(j prop) g)
    const float ag = cdotr(prop, g_prop);
    const float g_ph = prop.re * g_prop.im - prop.im * g_prop.re;
    g_k -= L * g_ph;
    g_L -= k * g_ph;
    if (k_free) g_k -= ag / k_amp;
    if (la_free) g_la -= ag / La;
}

}  // namespace wc
