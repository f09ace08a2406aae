// Geometry adjoints of the stored paths of a radiomap: the reflecting planes
// and wall normals of one path by a reverse sweep over its interactions.
// Values follow the rounding steps of wc_tangent.h; the carrier phase is
// reduced in double.
#pragma once

#include "wc_adjoint.h"
#include "wc_paths.h"
#include "wc_tangent.h"

namespace wc {

// Cotangent of one path's projected coefficient. Coherent sums fix it per
// (cell, slot); incoherent ones weight the path's own field.
struct PathCotangent {
    Cx<float> a;     // coherent: of the path field
    float inc;       // incoherent: 2 dL/dgain plus the root-power share
    bool coherent;
    float sp;        // sqrt of the transmit power
};
__device__ __forceinline__ Cx<float> coefficient_cotangent(const PathCotangent& w, const Cx<float>& coef) {
    if (w.coherent) return scale(w.a, w.sp);
    return scale(coef, w.inc * w.sp * w.sp);
}

// field = value prop, coefficient = field . transverse(dir, rx_pol): the
// cotangents of value, prop and dir
__device__ __forceinline__ void receive_adj(const C3<float>& value, const Cx<float>& prop, const V3<float>& dir,
                                            const V3<float>& rx_pol, const PathCotangent& w, C3<float>& g_value,
                                            Cx<float>& g_prop, V3<float>& g_dir) {
    const C3<float> field = c3_scale(value, prop);
    const V3<float> tr = transverse(dir, rx_pol);
    const Cx<float> g_coef = coefficient_cotangent(w, c3_dot_real(field, tr));
    V3<float> none = zero3();
    transverse_adj(dir, rx_pol, c3_axis_adj(field, g_coef), g_dir, none);
    const C3<float> g_field = c3_axis(tr, g_coef);
    g_prop = cmulj(value.x, g_field.x) + cmulj(value.y, g_field.y) + cmulj(value.z, g_field.z);
    g_value = {cmulj(prop, g_field.x), cmulj(prop, g_field.y), cmulj(prop, g_field.z)};
}

// prop = e^{j ph} / (2 k La), ph = -k L
__device__ __forceinline__ void propagation_adj(const Cx<float>& prop, float k, float L, float La,
                                                const Cx<float>& g_prop, float& g_k, float& g_L, float& g_la) {
    carrier_adj(prop, k, k, L, La, true, true, g_prop, g_k, g_L, g_la);
}

template <int DM> struct PlaneGrad {
    V3<float> nrm[DM];  // plane or wall normal
    float off[DM];      // plane offset
};

// Planes of a reflection chain of `depth` <= DM bounces. The loops are
// unrolled over DM with the bounces past the depth switched off, so every
// per-bounce value is in registers and lanes of different depths share the
// code.
template <int DM>
__device__ __forceinline__ void reflection_planes(const SceneView& s, int depth, const int* groups, const int* mats,
                                                   const V3<float>& tx, const V3<float>& rx, const V3<float>& tx_pol,
                                                   const V3<float>& rx_pol, float freq, double k_d, double length_d,
                                                   const PathCotangent& w, PlaneGrad<DM>& out) {
    const V3<float> ez{0.f, 0.f, 1.f};
    V3<float> nrm[DM], img[DM], hit[DM], inc[DM], fall[DM];
    float off[DM];
    C3<float> val_in[DM];
    // values in the rounding steps of reflection_tangent
    V3<Q> p = lq(tx);
#pragma unroll
    for (int j = 0; j < DM; ++j) {
        out.off[j] = 0.0f;
        out.nrm[j] = zero3();
        if (j >= depth) continue;
        double o;
        nrm[j] = to_f(group_normal(s, groups[j], o));
        off[j] = (float)o;
        const Q d = dot(p, lq(nrm[j])) - off[j];
        p = p - scale3<Q>(nrm[j], d * 2.0f);
        img[j] = vq(p);
    }
    const V3<float> last_img = vq(p);
    V3<Q> next = lq(rx);
#pragma unroll
    for (int j = DM - 1; j >= 0; --j) {
        if (j >= depth) continue;
        const V3<Q> n = lq(nrm[j]), im = lq(img[j]);
        const Q si = dot(n, im) - off[j], sn = dot(n, next) - off[j];
        next = im + (next - im) * (si / (si - sn));
        hit[j] = vq(next);
    }
    const V3<float> first = vq(safe_normalize(lq(hit[0]) - lq(tx), lq(ez)));
    C3<float> value = vq(c3_from_real(transverse(lq(first), lq(tx_pol))));
    V3<float> prev = tx, outgoing = first;
#pragma unroll
    for (int b = 0; b < DM; ++b) {
        if (b >= depth) continue;
        const int m = mats[b];
        fall[b] = outgoing;
        inc[b] = vq(safe_normalize(lq(hit[b]) - lq(prev), lq(outgoing)));
        val_in[b] = value;
        value = reflect_value(value, inc[b], nrm[b], s.mat_eps[m], s.mat_sigma[m], s.mat_mu[m], s.mat_gain[m],
                              s.mat_thickness[m], freq, outgoing);
        prev = hit[b];
    }
    const V3<float> last = rx - prev;
    const V3<float> dir = vq(safe_normalize(lq(rx) - lq(prev), lq(outgoing)));
    const V3<float> unfolded = rx - last_img;
    const Q Lq = norm(lq(rx) - lq(last_img)), kq = wave_number(lq(freq));
    const float L = Lq.v, k = kq.v;
    const Cx<float> prop = vq(scale(cexpj(lq(neg_kd_phase(k_d, length_d))), lq(1.0f) / (kq * Lq * 2.0f)));

    C3<float> g_value;
    Cx<float> g_prop;
    V3<float> g_dir = zero3(), g_out = zero3(), g_point = zero3();
    float g_k = 0.0f, g_L = 0.0f;
    receive_adj(value, prop, dir, rx_pol, w, g_value, g_prop, g_dir);
    propagation_adj(prop, k, L, L, g_prop, g_k, g_L, g_L);
    {
        V3<float> g_seg = zero3();
        safe_normalize_adj(last, outgoing, g_dir, g_seg, g_out);
        g_point = -g_seg;
    }
    V3<float> g_hit[DM], g_img[DM];
#pragma unroll
    for (int b = DM - 1; b >= 0; --b) {
        if (b >= depth) continue;
        const int m = mats[b];
        V3<float> g_inc = zero3(), g_nrm = zero3();
        C3<float> g_in;
        SlabGrad sg{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        reflect_c3_adj<true>(val_in[b], inc[b], nrm[b], s.mat_eps[m], s.mat_sigma[m], s.mat_mu[m], s.mat_gain[m],
                       s.mat_thickness[m], freq, g_value, g_out, g_in, g_inc, g_nrm, sg);
        g_value = g_in;
        out.nrm[b] = g_nrm;
        g_out = zero3();
        const V3<float> seg = hit[b] - (b ? hit[b ? b - 1 : 0] : tx);
        V3<float> g_seg = zero3(), none = zero3();
        if (b == 0) {
            // the launch polarization is transverse to the first direction
            const V3<float> g_t{g_value.x.re, g_value.y.re, g_value.z.re};
            transverse_adj(first, tx_pol, g_t, g_out, none);
        }
        safe_normalize_adj(seg, fall[b], g_inc, g_seg, g_out);
        if (b == 0) safe_normalize_adj(seg, ez, g_out, g_seg, none);
        g_hit[b] = g_point + g_seg;
        g_point = -g_seg;
    }
    // hits from images: h = img + (next - img) t, t = si / (si - sn)
#pragma unroll
    for (int j = 0; j < DM; ++j) {
        if (j >= depth) continue;
        const V3<float> nx = j + 1 < depth ? hit[j + 1 < DM ? j + 1 : j] : rx;
        const float si = dot(nrm[j], img[j]) - off[j], sn = dot(nrm[j], nx) - off[j];
        const float inv = 1.0f / (si - sn), t = si * inv;
        const float g_t = dot(g_hit[j], nx - img[j]) * inv * inv;
        const float g_si = -sn * g_t, g_sn = si * g_t;
        g_img[j] = g_hit[j] * (1.0f - t) + nrm[j] * g_si;
        acc(out.nrm[j], img[j] * g_si + nx * g_sn);
        out.off[j] -= g_si + g_sn;
        if (j + 1 < depth && j + 1 < DM) acc(g_hit[j + 1 < DM ? j + 1 : j], g_hit[j] * t + nrm[j] * g_sn);
    }
    // images from the transmitter: p' = p - 2 n (p . n - off)
    V3<float> g_p = zero3();
    norm_adj(unfolded, L, -g_L, g_p);
#pragma unroll
    for (int j = DM - 1; j >= 0; --j) {
        if (j >= depth) continue;
        const V3<float> g = g_img[j] + g_p;
        const float ng = 2.0f * dot(nrm[j], g);
        g_p = g - nrm[j] * ng;
        const V3<float> q = j ? img[j ? j - 1 : 0] : tx;
        acc(out.nrm[j], g * (-2.0f * (dot(q, nrm[j]) - off[j])) - q * ng);
        out.off[j] += ng;
    }
}

// Wall normals of a straight segment through `depth` <= DM layered walls. A
// wall's two coefficients depend on its normal through the incidence cosine,
// so the layer recursion carries one tangent and the rest is swept back.
template <int DM>
__device__ __forceinline__ void straight_normals(const SceneView& s, int depth, const Hit* hits, const V3<float>& tx,
                                                 const V3<float>& rx, const V3<float>& tx_pol,
                                                 const V3<float>& rx_pol, float freq, double k_d, double carrier_d,
                                                 const PathCotangent& w, PlaneGrad<DM>& out) {
    const V3<float> ez{0.f, 0.f, 1.f};
    // values in the rounding steps of transmission_tangent
    const V3<Q> segq = lq(rx) - lq(tx);
    const Q distq = norm(segq);
    const V3<Q> dirq = segq * (lq(1.0f) / distq);
    const float dist = distq.v;
    const V3<float> dir = vq(dirq);
    C3<Q> value = c3_from_real(transverse(dirq, lq(tx_pol)));
    C3<float> val_in[DM];
    Q carrierq = distq;
    auto wall_frame = [&](int group, V3<float>& raw, bool& flip, float& cosine) {
        double o;
        raw = to_f(group_normal(s, group, o));
        V3<Q> n = safe_normalize(lq(raw), lq(ez));
        flip = dot(dirq, n).v > 0.0f;
        if (flip) n = -n;
        cosine = dot(dirq, n).v;
        return vq(n);
    };
    auto layers = [&](int face, int& lo, int& lc, float& thickness) {
        const int m = s.face_material[face];
        lo = s.mat_layer_offset[m];
        lc = s.mat_layer_count[m];
        thickness = 0.0f;
        for (int l = 0; l < lc; ++l) thickness += fmaxf(s.layer_thickness[lo + l], 0.0f);
    };
#pragma unroll
    for (int j = 0; j < DM; ++j) {
        out.off[j] = 0.0f;
        out.nrm[j] = zero3();
        if (j >= depth) continue;
        V3<float> raw;
        bool flip;
        float cosine, thickness;
        int lo, lc;
        const V3<float> n = wall_frame(hits[j].group, raw, flip, cosine);
        const float ct = fminf(fmaxf(fabsf(cosine), kSmallEpsF), 1.0f);
        layers(hits[j].face, lo, lc, thickness);
        const int lcc = lc < 4 ? lc : 4;
        const Cx<Q> t_te = stack_t<Q>(lq(ct), s.layer_thickness + lo, s.layer_eps + lo, s.layer_sigma + lo,
                                      s.layer_mu + lo, lcc, lq(freq), 0, nullptr, nullptr);
        const Cx<Q> t_tm = stack_t<Q>(lq(ct), s.layer_thickness + lo, s.layer_eps + lo, s.layer_sigma + lo,
                                      s.layer_mu + lo, lcc, lq(freq), 1, nullptr, nullptr);
        const V3<Q> nq = lq(n);
        const V3<Q> sax = safe_normalize(cross(nq, dirq), stable_perp_basis(dirq, nq));
        const V3<Q> pax = safe_normalize(cross(sax, dirq), stable_perp_basis(dirq, sax));
        val_in[j] = vq(value);
        const Cx<Q> e_s = c3_dot_real(value, sax), e_p = c3_dot_real(value, pax);
        value = c3_axis(sax, t_te * e_s) + c3_axis(pax, t_tm * e_p);
        carrierq = carrierq - lq(ct) * thickness;
    }
    const Q kq = wave_number(lq(freq));
    const float k = kq.v, carrier = carrierq.v;
    const Cx<float> prop = vq(scale(cexpj(lq(neg_kd_phase(k_d, carrier_d))), lq(1.0f) / (kq * distq * 2.0f)));
    C3<float> g_value;
    Cx<float> g_prop;
    V3<float> g_dir = zero3();
    float g_k = 0.0f, g_carrier = 0.0f, g_dist = 0.0f;
    receive_adj(vq(value), prop, dir, rx_pol, w, g_value, g_prop, g_dir);
    propagation_adj(prop, k, carrier, dist, g_prop, g_k, g_carrier, g_dist);
#pragma unroll
    for (int j = DM - 1; j >= 0; --j) {
        if (j >= depth) continue;
        using D1 = Dual<1>;  // incidence cosine
        V3<float> raw;
        bool flip;
        float cosine, thickness;
        int lo, lc;
        const V3<float> n = wall_frame(hits[j].group, raw, flip, cosine);
        const float ca = fabsf(cosine);
        const float ct = fminf(fmaxf(ca, kSmallEpsF), 1.0f);
        layers(hits[j].face, lo, lc, thickness);
        const int lcc = lc < 4 ? lc : 4;
        Cx<D1> t[2];
#pragma unroll 1
        for (int pol = 0; pol < 2; ++pol)
            t[pol] = stack_t<D1>(seed<1>(ct, 0), s.layer_thickness + lo, s.layer_eps + lo, s.layer_sigma + lo,
                                 s.layer_mu + lo, lcc, lift<D1>(freq), pol, nullptr, nullptr);
        const V3<float> sax = safe_normalize(cross(n, dir), stable_perp_basis(dir, n));
        const V3<float> pax = safe_normalize(cross(sax, dir), stable_perp_basis(dir, sax));
        const Cx<float> te = cval(t[0]), tm = cval(t[1]);
        const Cx<float> e_s = c3_dot_real(val_in[j], sax), e_p = c3_dot_real(val_in[j], pax);
        const Cx<float> g_ts = c3_dot_real(g_value, sax), g_tp = c3_dot_real(g_value, pax);
        V3<float> g_s = c3_axis_adj(g_value, te * e_s), g_pa = c3_axis_adj(g_value, tm * e_p);
        const Cx<float> g_te = cmulj(e_s, g_ts), g_tm = cmulj(e_p, g_tp);
        const float d_cos =
            g_te.re * t[0].re.d[0] + g_te.im * t[0].im.d[0] + g_tm.re * t[1].re.d[0] + g_tm.im * t[1].im.d[0];
        const Cx<float> g_es = cmulj(te, g_ts), g_ep = cmulj(tm, g_tp);
        g_value = c3_axis(sax, g_es) + c3_axis(pax, g_ep);
        acc(g_s, c3_axis_adj(val_in[j], g_es));
        acc(g_pa, c3_axis_adj(val_in[j], g_ep));
        V3<float> g_n = zero3();
        perp_axis_adj(sax, dir, g_pa, g_s, g_dir);
        perp_axis_adj(n, dir, g_s, g_n, g_dir);
        if (ca >= kSmallEpsF && ca <= 1.0f) {
            const float g_ct = d_cos - thickness * g_carrier;
            const float g_cos = cosine < 0.0f ? -g_ct : g_ct;
            acc(g_dir, n * g_cos);
            acc(g_n, dir * g_cos);
        }
        if (flip) g_n = -g_n;
        const float nn = norm(raw);
        if (nn > kSmallEpsF) normalize_adj(raw, nn, g_n, out.nrm[j]);
    }
}

}  // namespace wc
