// Stored paths whose reflecting planes (n, c) or wall normals carry the
// derivatives, as the adjoint checks evaluate them: with dual numbers in the
// rounding steps of the kernels' own tangents (wc_tangent.h), or in double.
// Endpoints, frequency and materials are constants.
#pragma once

#include "../../witwin-channel_amd/csrc/wc_tangent.h"

namespace wc {

// in double the phase follows the length itself
template <> struct PhaseOf<double> {
    static double make(double, double L, double k_d, double) { return -(k_d * L); }
};

template <typename R>
__device__ inline C3<R> reflection_tangent_planes(const SceneView& s, int depth, const int* faces, const V3<R>* nrm,
                                                  const R* off, const V3<float>& tx, const V3<float>& rx,
                                                  const V3<float>& tx_pol, float freq, double k_d, double length_d,
                                                  V3<R>& arrival) {
    V3<R> img[kMaxDepth];
    V3<R> p = lift3<R>(tx);
    for (int j = 0; j < depth; ++j) {
        const R dist = dot(p, nrm[j]) - off[j];
        p = p - nrm[j] * (dist * 2.0f);
        img[j] = p;
    }
    V3<R> hits[kMaxDepth];
    V3<R> next = lift3<R>(rx);
    for (int j = depth - 1; j >= 0; --j) {
        const R si = dot(nrm[j], img[j]) - off[j];
        const R sn = dot(nrm[j], next) - off[j];
        const R t = si / (si - sn);
        hits[j] = img[j] + (next - img[j]) * t;
        next = hits[j];
    }
    const R fr = lift<R>(freq);
    const V3<R> ez = v3c<R>(0.f, 0.f, 1.f);
    V3<R> prev = lift3<R>(tx);
    V3<R> incident = safe_normalize(hits[0] - prev, ez);
    C3<R> value = c3_from_real(transverse(incident, lift3<R>(tx_pol)));
    V3<R> outgoing = incident;
    for (int b = 0; b < depth; ++b) {
        incident = safe_normalize(hits[b] - prev, outgoing);
        const int m = s.face_material[faces[b]];
        value = reflect_c3(value, incident, nrm[b], lift<R>(s.mat_eps[m]), lift<R>(s.mat_sigma[m]),
                           lift<R>(s.mat_mu[m]), lift<R>(s.mat_gain[m]), lift<R>(s.mat_thickness[m]), fr, outgoing);
        prev = hits[b];
    }
    arrival = safe_normalize(lift3<R>(rx) - prev, outgoing);
    const R L = norm(lift3<R>(rx) - img[depth - 1]);
    const R k = wave_number(fr);
    const R amp = lift<R>(1.0f) / (k * L * 2.0f);
    return c3_scale(value, scale(cexpj(PhaseOf<R>::make(k, L, k_d, length_d)), amp));
}

template <typename R>
__device__ inline C3<R> transmission_tangent_walls(const SceneView& s, int count, const Hit* hits,
                                                   const V3<R>* wall_n, const V3<float>& tx, const V3<float>& rx,
                                                   const V3<float>& tx_pol, float freq, double k_d, double carrier_d,
                                                   V3<R>& arrival) {
    const V3<R> ez = v3c<R>(0.f, 0.f, 1.f);
    const V3<R> seg = lift3<R>(rx - tx);
    const R dist = norm(seg);
    const V3<R> dir = seg * (lift<R>(1.0f) / dist);
    const R fr = lift<R>(freq);
    C3<R> value = c3_from_real(transverse(dir, lift3<R>(tx_pol)));
    R carrier = dist;
    for (int w = 0; w < count; ++w) {
        V3<R> n = safe_normalize(wall_n[w], ez);
        if (val(dot(dir, n)) > 0.0f) n = -n;
        const R ct = w_min(w_max(w_abs(dot(dir, n)), kSmallEpsF), 1.0f);
        const int m = s.face_material[hits[w].face];
        const int lo = s.mat_layer_offset[m], lc = s.mat_layer_count[m];
        const int lcc = lc < 4 ? lc : 4;
        const Cx<R> t_te = stack_t<R>(ct, s.layer_thickness + lo, s.layer_eps + lo, s.layer_sigma + lo,
                                      s.layer_mu + lo, lcc, fr, 0, nullptr, nullptr);
        const Cx<R> t_tm = stack_t<R>(ct, s.layer_thickness + lo, s.layer_eps + lo, s.layer_sigma + lo,
                                      s.layer_mu + lo, lcc, fr, 1, nullptr, nullptr);
        const V3<R> sax = safe_normalize(cross(n, dir), stable_perp_basis(dir, n));
        const V3<R> pax = safe_normalize(cross(sax, dir), stable_perp_basis(dir, sax));
        const Cx<R> e_s = c3_dot_real(value, sax);
        const Cx<R> e_p = c3_dot_real(value, pax);
        value = c3_axis(sax, t_te * e_s) + c3_axis(pax, t_tm * e_p);
        float wall = 0.0f;
        for (int l = 0; l < lc; ++l) wall += fmaxf(s.layer_thickness[lo + l], 0.0f);
        carrier = carrier - ct * wall;
    }
    arrival = dir;
    const R k = wave_number(fr);
    const R amp = lift<R>(1.0f) / (k * dist * 2.0f);
    return c3_scale(value, scale(cexpj(PhaseOf<R>::make(k, carrier, k_d, carrier_d)), amp));
}

}  // namespace wc
