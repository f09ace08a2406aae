// CPU run of the reflection rows' adjoint kernel (wc_rows.hip, built as host
// C++ through the shim in hip/) against forward-mode tangents of the same row
// function, one dual pass per eight input scalars. Rows are random street
// geometries; some carry the degenerate forms the fallbacks exist for (normal
// incidence, coincident points, zero normals) and some have zero cotangents
// over values that are not numbers. Prints "depth kind errors" per input kind:
// the 2-norm of the difference over the 2-norm of the tangent contraction over
// the ordinary rows and over the degenerate ones, and the number of non-zeros
// in masked rows.
#include "hip/hip_runtime.h"
#include "../../witwin-channel_amd/csrc/wc_rows.hip"

#include <cstdio>
#include <random>
#include <vector>

int wc_fail(const char*, ...) { return 1; }
int wc_fail_hip(const char*, hipError_t) { return 1; }

using namespace wc;

template <int D> static void check(int n, double freq) {
    std::mt19937 gen(100 + D);
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    auto fill = [&](size_t k, float lo, float hi) {
        std::vector<float> v(k);
        for (auto& x : v) x = lo + (hi - lo) * 0.5f * (u(gen) + 1.0f);
        return v;
    };
    auto src = fill(3 * n, 0, 300), tgt = fill(3 * n, 0, 300), pos = fill((size_t)3 * n * D, 0, 300);
    auto nrm = fill((size_t)3 * n * D, -1, 1), power = fill(n, 0.1f, 2), txp = fill(3 * n, -1, 1), rxp = fill(3 * n, -1, 1);
    auto eps = fill((size_t)n * D, 1.5f, 7), sig = fill((size_t)n * D, 0.001f, 0.05f), mu = fill((size_t)n * D, 1, 1.2f);
    auto gain = fill((size_t)n * D, 0.5f, 1), thick = fill((size_t)n * D, 0.02f, 0.3f);
    const int degenerate = n / 4, masked = n / 8;
    for (int i = 0; i < degenerate; ++i) {
        float* p = &pos[(size_t)3 * i * D];
        if (i % 3 == 0) {  // normal incidence at the first bounce
            for (int c = 0; c < 3; ++c) nrm[(size_t)3 * i * D + c] = src[3 * i + c] - p[c];
        } else if (i % 3 == 1) {  // coincident points
            if (D > 1) for (int c = 0; c < 3; ++c) p[3 + c] = p[c];
            else for (int c = 0; c < 3; ++c) tgt[3 * i + c] = p[c];
        } else {
            for (int c = 0; c < 3; ++c) nrm[(size_t)3 * i * D + c] = 0.0f;
        }
    }
    auto gf = fill(6 * n, -1, 1), gc = fill(2 * n, -1, 1), gp = fill(2 * n, -1, 1), gg = fill(n, -1, 1);
    auto gl = fill(n, -1e-7f, 1e-7f), gd = fill(n, -1, 1), gdir = fill(3 * n, -1e-6f, 1e-6f);
    for (int i = n - masked; i < n; ++i) {
        for (int c = 0; c < 6; ++c) gf[6 * i + c] = 0;
        for (int c = 0; c < 2; ++c) gc[2 * i + c] = gp[2 * i + c] = 0;
        for (int c = 0; c < 3; ++c) gdir[3 * i + c] = 0;
        gg[i] = gl[i] = gd[i] = 0;
        pos[(size_t)3 * i * D] = NAN;
    }
    ReflIn in{D, src.data(), tgt.data(), pos.data(), nrm.data(), power.data(), txp.data(), rxp.data(), eps.data(),
              sig.data(), mu.data(), gain.data(), thick.data()};
    FieldGrads fg{gf.data(), gc.data(), gp.data(), gg.data(), gl.data(), gd.data(), gdir.data()};
    std::vector<float> o_src(3 * n), o_tgt(3 * n), o_pos(3 * n * D), o_nrm(3 * n * D), o_eps(n * D), o_sig(n * D),
        o_gain(n * D), o_thick(n * D), o_f(n);
    ReflGrads out{o_src.data(), o_tgt.data(), o_pos.data(), o_nrm.data(), o_eps.data(), o_sig.data(), o_gain.data(),
                  o_thick.data(), o_f.data()};
    blockIdx = {}; threadIdx = {}; blockDim = {1, 1, 1}; gridDim = {1, 1, 1};
    refl_vjp_kernel<D>(n, in, freq, fg, out);

    const char* names[] = {"source", "target", "positions", "normals", "eps", "sigma", "gain", "thickness", "frequency"};
    double num[2][9] = {{0}}, den[2][9] = {{0}};
    long nonzero = 0;
    for (int i = 0; i < n; ++i) {
        double rn[9] = {0}, rd[9] = {0};
        for (int pass = 0; pass * 8 < 7 + 10 * D; ++pass) {
            auto v3 = [&](const float* p, size_t k, int s0) {
                return V3<R8>{sv(p[3 * k], s0, pass), sv(p[3 * k + 1], s0 + 1, pass), sv(p[3 * k + 2], s0 + 2, pass)};
            };
            V3<R8> P[D], N[D];
            R8 E[D], S[D], G[D], T[D];
            for (int b = 0; b < D; ++b) {
                const size_t k = (size_t)i * D + b;
                const int s = 7 + 10 * b;
                P[b] = v3(in.pos, k, s);
                N[b] = v3(in.nrm, k, s + 3);
                E[b] = sv(eps[k], s + 6, pass);
                S[b] = sv(sig[k], s + 7, pass);
                G[b] = sv(gain[k], s + 8, pass);
                T[b] = sv(thick[k], s + 9, pass);
            }
            RowOut<R8> r;
            reflection_row<R8>(D, v3(in.src, i, 0), v3(in.tgt, i, 3), P, N, E, S, &mu[(size_t)i * D], G, T,
                               ld3(in.txp + 3 * i), ld3(in.rxp + 3 * i), std::sqrt(power[i]),
                               sv((float)freq, 6, pass), freq, r);
            float d[8];
            contract_row(fg, i, r, d);
            for (int j = 0; j < 8; ++j) {
                const int s = 8 * pass + j;
                if (s >= 7 + 10 * D) break;
                int kind;
                float got;
                if (s < 3) { kind = 0; got = o_src[3 * i + s]; }
                else if (s < 6) { kind = 1; got = o_tgt[3 * i + s - 3]; }
                else if (s == 6) { kind = 8; got = o_f[i]; }
                else {
                    const int q = (s - 7) % 10;
                    const size_t k = (size_t)i * D + (s - 7) / 10;
                    if (q < 3) { kind = 2; got = o_pos[3 * k + q]; }
                    else if (q < 6) { kind = 3; got = o_nrm[3 * k + q - 3]; }
                    else { kind = q - 2; got = q == 6 ? o_eps[k] : q == 7 ? o_sig[k] : q == 8 ? o_gain[k] : o_thick[k]; }
                }
                if (i >= n - masked) {
                    nonzero += got != 0.0f || d[j] != 0.0f;
                    continue;
                }
                rn[kind] += ((double)got - d[j]) * ((double)got - d[j]);
                rd[kind] += (double)d[j] * d[j];
            }
        }
        for (int k = 0; k < 9; ++k) {
            const int c = i < degenerate ? 1 : 0;
            num[c][k] += rn[k];
            den[c][k] += rd[k];
            if (!(rn[k] == rn[k])) std::printf("nan row %d kind %s\n", i, names[k]);
        }
    }
    for (int k = 0; k < 9; ++k)
        std::printf("%d %s %.3e %.3e %ld\n", D, names[k], std::sqrt(num[0][k] / den[0][k]),
                    std::sqrt(num[1][k] / den[1][k]), nonzero);
}

int main() {
    check<1>(2000, 3.5e9);
    check<2>(2000, 3.5e9);
    check<3>(2000, 3.5e9);
    check<4>(1000, 3.5e9);
    check<5>(1000, 3.5e9);
    return 0;
}
