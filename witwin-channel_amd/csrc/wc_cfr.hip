// Channel frequency response of padded per-pair path sets.
//
//   out[b, s, k] = sum_p valid[b,p] a[b,p,s] exp(-j 2 pi f_k (tau[b,p] - tau0[b]))
//
// One wavefront per (pair b, time step s, block of 1,024 subcarriers). The
// phase argument f * tau is reduced modulo one cycle in float64 before the
// float32 sine and cosine, which keeps the phase error near 1e-7 rad at the
// ~1e4-cycle arguments of km paths at mmWave; the sums run in float32 over
// paths in index order.
//
// Uniform grid f_k = f0 + k df (cfr_grid_kernel): with k = k0 + 32 i + j the
// phasor factors into e(f0 + (k0 + 32 i) df) e(j df), so the block is a product
// of a 32 x P matrix (path amplitudes times row phasors) and a P x 32 matrix
// (column phasors): a complex contraction over the paths, which runs on the
// float32 matrix units. A path costs one float64 phase and one sine / cosine
// per lane and two 32x32x2 instructions (its real and imaginary part are the
// K = 2 entries) instead of 1,024 rotations, 16 per lane, on the vector units.
// An arbitrary frequency list (cfr_list_kernel) evaluates every phasor.
// Measured on 45,221 pairs of up to 199 paths (18 on average) x 1,024
// subcarriers: 551 us with the rotations, 195 us with the matrix product (2.5 TB/s),
// for 0.49 GB of paths read and responses written; error against 64 bits 9.3e-7
// before, 1.6e-7 now.
#include "wc_api_internal.h"
#include "../../include/wcmi.h"

namespace wc {
namespace {

constexpr int kPerLane = 16;
constexpr int kBlock = 64 * kPerLane;  // subcarriers per wavefront
constexpr double kTwoPiD = 6.283185307179586476925286766559;

__device__ __forceinline__ void phasor(double cycles, float& c, float& s) {
    const double frac = cycles - floor(cycles);
    // exp(-j 2 pi frac)
    __sincosf(-(float)(kTwoPiD * frac), &s, &c);
}

// (pair, time step, first subcarrier) of this wavefront; false past the end
__device__ __forceinline__ bool wave_task(int pairs, int time_steps, int blocks_per_row, long long& row, int& b, int& s,
                                          int& k0) {
    const long long wave = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wave >= (long long)pairs * time_steps * blocks_per_row) return false;
    row = wave / blocks_per_row;  // b * S + s
    k0 = (int)(wave - row * blocks_per_row) * kBlock;
    b = (int)(row / time_steps);
    s = (int)(row - (long long)b * time_steps);
    return true;
}

// earliest valid delay of a pair (0 when it has none), the same in every lane
__device__ __forceinline__ double earliest_delay(const float* tau, const unsigned char* valid, int paths, int lane) {
    float m = INFINITY;
    for (int p = lane; p < paths; p += 64)
        if (valid[p]) m = fminf(m, tau[p]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fminf(m, __shfl_xor(m, off));
    return m < INFINITY ? (double)m : 0.0;
}

__global__ void __launch_bounds__(256) cfr_list_kernel(const float* __restrict__ a, const float* __restrict__ tau,
                                                       const unsigned char* __restrict__ valid, int pairs,
                                                       int max_paths, int time_steps,
                                                       const double* __restrict__ frequencies, int freq_count,
                                                       int blocks_per_row, int normalize, float* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    long long row;
    int b, s, k0;
    if (!wave_task(pairs, time_steps, blocks_per_row, row, b, s, k0)) return;
    const float* tau_b = tau + (size_t)b * max_paths;
    const unsigned char* valid_b = valid + (size_t)b * max_paths;
    const double tau0 = normalize ? earliest_delay(tau_b, valid_b, max_paths, lane) : 0.0;
    float acc_re[kPerLane], acc_im[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        acc_re[i] = 0.0f;
        acc_im[i] = 0.0f;
    }
    for (int p = 0; p < max_paths; ++p) {
        if (!valid_b[p]) continue;
        // tau - tau0 in float32, as the reference normalizes its float32 delays
        const double t = (double)((float)((double)tau_b[p] - tau0));
        const size_t ai = ((size_t)b * max_paths + p) * time_steps + s;
        const float ar = a[2 * ai], aim = a[2 * ai + 1];
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) {
            const int k = k0 + lane + 64 * i;
            if (k < freq_count) {
                float c, sn;
                phasor(frequencies[k] * t, c, sn);
                acc_re[i] = fmaf(ar, c, fmaf(-aim, sn, acc_re[i]));
                acc_im[i] = fmaf(ar, sn, fmaf(aim, c, acc_im[i]));
            }
        }
    }
    float* o = out + 2 * ((size_t)row * freq_count);
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        const int k = k0 + lane + 64 * i;
        if (k < freq_count) {
            o[2 * k] = acc_re[i];
            o[2 * k + 1] = acc_im[i];
        }
    }
}

// exp(-j 2 pi cycles) to the last bit or two: reduced to an eighth of a turn in
// float64, Taylor polynomials in float32 (remainders x^11 / 11! and x^12 / 12!,
// below 2e-9 at pi / 4). A subcarrier's phasor is a product of two of these, so
// each has to be better than the one the hardware sine gives (1e-7).
__device__ __forceinline__ void phasor_factor(double cycles, float& c, float& s) {
    const double quarters = rint(4.0 * cycles);
    const float x = (float)(kTwoPiD * (cycles - 0.25 * quarters));
    const float z = x * x;
    const float sn = fmaf(x * z, fmaf(z, fmaf(z, fmaf(z, 1.0f / 362880.0f, -1.0f / 5040.0f), 1.0f / 120.0f),
                                      -1.0f / 6.0f), x);
    const float cs = fmaf(z, fmaf(z, fmaf(z, fmaf(z, fmaf(z, -1.0f / 3628800.0f, 1.0f / 40320.0f), -1.0f / 720.0f),
                                          1.0f / 24.0f), -0.5f), 1.0f);
    // the quarter turn's index modulo 4, exact for every finite double
    const int k = (int)(quarters - 4.0 * floor(0.25 * quarters));
    const bool odd = (k & 1) != 0;
    const float a = odd ? sn : cs, b = odd ? cs : sn;
    c = (k == 1 || k == 2) ? -a : a;
    s = (k & 2) ? b : -b;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// swap the upper half of x with the lower half of y
__device__ __forceinline__ void swap_halves(float& x, float& y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(r[0]);
    y = __uint_as_float(r[1]);
}

// Lanes 0..31 carry row i = lane of the block (subcarriers k0 + 32 i + j) and
// lanes 32..63 column j = lane - 32. Each lane forms its one phasor; two half
// swaps arrange them as the operands of the 32x32x2 product, whose K = 2
// entries are (re, im) of the row factor u against (re, -im) of the column
// factor v for the real part and (im, re) for the imaginary part. Accumulator
// r of a lane is row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
cfr_grid_kernel(const float* __restrict__ a, const float* __restrict__ tau,
                const unsigned char* __restrict__ valid, int pairs,
                int max_paths, int time_steps, double f0, double df,
                int freq_count, int blocks_per_row, int normalize,
                float* __restrict__ out){
    const int lane = threadIdx.x & 63;
    const bool upper = lane >= 32;
    const int half = lane & 31;
    long long row;
    int b, s, k0;
    if (!wave_task(pairs, time_steps, blocks_per_row, row, b, s, k0)) return;
    const float* tau_b = tau + (size_t)b * max_paths;
    const unsigned char* valid_b = valid + (size_t)b * max_paths;
    const double tau0 = normalize ? earliest_delay(tau_b, valid_b, max_paths, lane) : 0.0;
    const double f_lane = upper ? df * (double)half : f0 + df * (double)(k0 + 32 * half);
    f32x16 acc_re = {0.0f}, acc_im = {0.0f};
    for (int p0 = 0; p0 < max_paths; p0 += 64) {
        // the chunk's 64 paths, one per lane; the valid ones in index order
        const int mine = p0 + lane;
        const bool on = mine < max_paths && valid_b[mine];
        unsigned long long left = __ballot(on);
        float my_t = 0.0f, my_re = 0.0f, my_im = 0.0f;
        if (on) {
            // tau - tau0 in float32, as the reference normalizes its float32 delays
            my_t = (float)((double)tau_b[mine] - tau0);
            const size_t ai = ((size_t)b * max_paths + mine) * time_steps + s;
            my_re = a[2 * ai];
            my_im = a[2 * ai + 1];
        }
        while (left) {
            const int l = __ffsll(left) - 1;
            left &= left - 1;
            const float t = __shfl(my_t, l), ar = __shfl(my_re, l), ai = __shfl(my_im, l);
            if (!isfinite(fabsf(ar) + fabsf(ai))) {
                // a product of phasors would turn one infinite part into NaN in both, as it
                // would a finite amplitude whose row factor overflows
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int k = k0 + 32 * (8 * (r >> 2) + 4 * (upper ? 1 : 0) + (r & 3)) + half;
                    float c, sn;
                    phasor((f0 + df * (double)k) * (double)t, c, sn);
                    acc_re[r] = fmaf(ar, c, fmaf(-ai, sn, acc_re[r]));
                    acc_im[r] = fmaf(ar, sn, fmaf(ai, c, acc_im[r]));
                }
                continue;
            }
            float c, sn;
            phasor_factor(f_lane * (double)t, c, sn);
            const float wr = upper ? 1.0f : ar, wi = upper ? 0.0f : ai;
            float u = fmaf(wr, c, -wi * sn), v = fmaf(wr, sn, wi * c);
            // u: u_re | v_re, v: u_im | v_im  ->  u: u_re | u_im, v: v_re | v_im
            swap_halves(u, v);
            float vr = v, vi = v;  // -> vr: v_re | v_re, vi: v_im | v_im
            swap_halves(vr, vi);
            acc_re = __builtin_amdgcn_mfma_f32_32x32x2f32(u, upper ? -vi : vr, acc_re, 0, 0, 0);
            acc_im = __builtin_amdgcn_mfma_f32_32x32x2f32(u, upper ? vr : vi, acc_im, 0, 0, 0);
        }
    }
    float2* o = reinterpret_cast<float2*>(out) + (size_t)row * freq_count;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int k = k0 + 32 * (8 * (r >> 2) + 4 * (upper ? 1 : 0) + (r & 3)) + half;
        if (k < freq_count) o[k] = make_float2(acc_re[r], acc_im[r]);
    }
}

}  // namespace
}  // namespace wc

using namespace wc;

extern "C" int wc_paths_cfr(const float* a, const float* tau, const unsigned char* valid, int pairs, int max_paths,
                            int time_steps, const double* frequencies, double f0, double df, int freq_count,
                            int normalize_delays, float* out, void* stream) {
    if (pairs < 0 || max_paths < 0 || time_steps <= 0 || freq_count < 0)
        return wc_fail("wc_paths_cfr: invalid sizes (pairs %d, paths %d, time steps %d, frequencies %d)", pairs,
                       max_paths, time_steps, freq_count);
    if (pairs == 0 || freq_count == 0) return 0;
    if (!out) return wc_fail("wc_paths_cfr: out is null");
    if (max_paths > 0 && (!a || !tau || !valid)) return wc_fail("wc_paths_cfr: path tensors are null");
    const int blocks_per_row = (freq_count + kBlock - 1) / kBlock;
    const long long waves = (long long)pairs * time_steps * blocks_per_row;
    const long long blocks = (waves + 3) / 4;
    if (blocks > 0x7fffffffLL) return wc_fail("wc_paths_cfr: launch too large (%lld waves)", waves);
    if (frequencies)
        hipLaunchKernelGGL(cfr_list_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a, tau, valid,
                           pairs, max_paths, time_steps, frequencies, freq_count, blocks_per_row, normalize_delays,
                           out);
    else
        hipLaunchKernelGGL(cfr_grid_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a, tau, valid,
                           pairs, max_paths, time_steps, f0, df, freq_count, blocks_per_row, normalize_delays, out);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? 0 : wc_fail_hip("wc_paths_cfr", err);
}
