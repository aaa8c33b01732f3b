// pm_device.h -- gfx950 (CDNA4, wave64) device code of libpmhip.so.
//
// Numerical contract (restating the reference, PorousMaterials.jl v0.4.2):
//   LJ pair        src/vdw_energetics.jl:19-22    4 eps s^3 (s^3 - 1), s = sigma^2/r^2
//   pair loop      src/vdw_energetics.jl:25-47    nearest image, strict r^2 < rc^2,
//                                                 overlap r^2 < 0.1 -> +Inf
//   real space     src/electrostatics.jl:377-386  q erfc(alpha r) / (4 pi eps0 r), r < rc
//   Fourier        src/electrostatics.jl:354-372  sum_k wt_k sum_c q_c cos(k.(x_c - x)),
//                                                 here from the unit-cell structure
//                                                 factor (the same sum, reorganised)
//   Widom          src/henry.jl:212-243           per-block sum e^{-E/T}, E e^{-E/T}
//   energy grid    src/grid.jl:313-355            point (i,j,k)/(n-1) ./ rep
//
// Two execution schemes:
//   pm_poses.h    one workgroup per pose, every replicated atom, nearest image
//                 per pair; serves the explicit-pose API (vdw_energy,
//                 electrostatic_potential_energy, forces).
//   pm_points.h   every probe site is an independent point.  Points are grouped
//                 into spatially compact chunks (one cell of a counting sort, or
//                 one brick of a grid) of <= 256 per workgroup, evaluated against
//                 an image list of the framework that covers every image within
//                 r_c of any point: no per-pair wrap or basis change, ~1/4 of the
//                 pairs.  The Fourier part runs in its own FP64 kernel.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "pmhip.h"

namespace pmk {

constexpr int WG = 256;      // work-items per workgroup (4 waves)
constexpr int TILE = 256;    // framework atoms per LDS tile
constexpr double R2_OVERLAP = 0.1;  // src/vdw_energetics.jl:2

enum { MODE_WIDOM = 0, MODE_GRID = 2 };

struct KVec {
    double ma, mb, mc, are, aim;
    double wnr;  // wt * N_R (the factor of the structure factor in A)
};

struct Site {
    double ox, oy, oz;  // Cartesian offset from the centre of mass (template)
    double q;           // point charge (e), 0 if none
    int lj;             // 1 if an LJ sphere
    int pad;
};

template <typename Real>
struct LJP {
    Real sig2, eps4;
};

// ---------------------------------------------------------------- RNG ----
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11).  Insertion g draws three
// blocks: counter (g_lo, g_hi, w, 0x57494430), key (seed_lo, seed_hi), w = 0,1,2.
__device__ inline void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        // one 32 x 32 -> 64-bit product per multiplier (v_mad_u64_u32)
        const uint64_t m0 = (uint64_t)0xD2511F53u * c[0], m1 = (uint64_t)0xCD9E8D57u * c[2];
        uint32_t hi0 = (uint32_t)(m0 >> 32), lo0 = (uint32_t)m0;
        uint32_t hi1 = (uint32_t)(m1 >> 32), lo1 = (uint32_t)m1;
        uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ inline double u53(uint32_t a, uint32_t b) {
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

__device__ inline void insertion_uniforms(unsigned long long seed, unsigned long long g, double u[6]) {
#pragma unroll
    for (uint32_t w = 0; w < 3; ++w) {
        uint32_t c[4] = {(uint32_t)g, (uint32_t)(g >> 32), w, 0x57494430u};
        philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        u[2 * w] = u53(c[0], c[1]);
        u[2 * w + 1] = u53(c[2], c[3]);
    }
}

// Arvo rotation (src/molecule.jl:233-244): R = -H Rz(2 pi u0), H = I - 2 v v^T,
// v = (cos(2 pi u1) sqrt(u2), sin(2 pi u1) sqrt(u2), sqrt(1 - u2)); column-major.
__device__ inline void arvo_rotation(const double* u, double R[9]) {
    double s1, c1, s2, c2;
    sincospi(2.0 * u[0], &s1, &c1);
    sincospi(2.0 * u[1], &s2, &c2);
    double sq = sqrt(u[2]);
    double v0 = c2 * sq, v1 = s2 * sq, v2 = sqrt(1.0 - u[2]);
    double H[9] = {1.0 - 2.0 * v0 * v0, -2.0 * v1 * v0,       -2.0 * v2 * v0,
                   -2.0 * v0 * v1,       1.0 - 2.0 * v1 * v1, -2.0 * v2 * v1,
                   -2.0 * v0 * v2,       -2.0 * v1 * v2,       1.0 - 2.0 * v2 * v2};
    // Rz columns: (c1, -s1, 0), (s1, c1, 0), (0, 0, 1)
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        R[r] = -(H[r] * c1 - H[r + 3] * s1);
        R[r + 3] = -(H[r] * s1 + H[r + 3] * c1);
        R[r + 6] = -H[r + 6];
    }
}

// ---------------------------------------------------------- pair maths ----
// FP32 erfc: Numerical Recipes "erfcc" Chebyshev fit (Press et al., Numerical
// Recipes in C, 2nd ed., section 6.2), fractional error < 1.2e-7 for x >= 0.
__device__ inline float erfc_f32(float x) {
    float t = __builtin_amdgcn_rcpf(1.0f + 0.5f * x);
    float p = 0.17087277f;
    p = fmaf(p, t, -0.82215223f);
    p = fmaf(p, t, 1.48851587f);
    p = fmaf(p, t, -1.13520398f);
    p = fmaf(p, t, 0.27886807f);
    p = fmaf(p, t, -0.18628806f);
    p = fmaf(p, t, 0.09678418f);
    p = fmaf(p, t, 0.37409196f);
    p = fmaf(p, t, 1.00002368f);
    p = fmaf(p, t, -1.26551223f);
    float y = p - x * x;  // exponent, natural-log units
    return t * __builtin_amdgcn_exp2f(y * 1.4426950408889634f);
}

// 4 eps s^3 (s^3 - 1), s = sigma^2 / r^2, in FP32
__device__ inline float lj_f32(double r2, float sig2, float eps4) {
    float s = sig2 * __builtin_amdgcn_rcpf((float)r2);
    float s3 = s * s * s;
    return eps4 * fmaf(s3, s3, -s3);
}

// q erfc(alpha r) / r in FP32
__device__ inline float coul_f32(double r2, double q, double alpha) {
    float rf2 = (float)r2;
    float rinv = __builtin_amdgcn_rsqf(rf2);
    float r = rf2 * rinv;
    return (float)q * erfc_f32((float)alpha * r) * rinv;
}

// --------------------------------------------------------- reductions ----
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Fixed-order workgroup sum of three values into out[0..2] (thread 0 writes).
__device__ inline void block_sum3(double v0, double v1, double v2, double* out) {
    __shared__ double red[3][WG / 64];
    v0 = wave_sum(v0);
    v1 = wave_sum(v1);
    v2 = wave_sum(v2);
    int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (lane == 0) { red[0][wave] = v0; red[1][wave] = v1; red[2][wave] = v2; }
    __syncthreads();
    if (tid == 0) {
        double t0 = 0.0, t1 = 0.0, t2 = 0.0;
        for (int w = 0; w < WG / 64; ++w) { t0 += red[0][w]; t1 += red[1][w]; t2 += red[2][w]; }
        out[0] = t0; out[1] = t1; out[2] = t2;
    }
}

// Unit-cell structure factor per kept k-vector: one wave per k-vector,
// lanes stride over the unit-cell charges, FP64 phases and sums.
__global__ __launch_bounds__(64) void structure_factor_kernel(const double4* uq, long long n,
                                                              const int* m, const double* wt,
                                                              double nr, KVec* out) {
    int k = blockIdx.x, lane = threadIdx.x;
    double ma = m[3 * k], mb = m[3 * k + 1], mc = m[3 * k + 2];
    double sre = 0.0, sim = 0.0;
    for (long long c = lane; c < n; c += 64) {
        double4 p = uq[c];
        double t = ma * p.x + mb * p.y + mc * p.z;
        t -= rint(t);
        double sn, cs;
        sincospi(2.0 * t, &sn, &cs);
        sre += p.w * cs;
        sim += p.w * sn;
    }
    sre = wave_sum(sre);
    sim = wave_sum(sim);
    if (lane == 0) {
        KVec kv;
        kv.ma = ma; kv.mb = mb; kv.mc = mc;
        kv.are = wt[k] * nr * sre;
        kv.aim = wt[k] * nr * sim;
        kv.wnr = wt[k] * nr;
        out[k] = kv;
    }
}

// Dense Fourier box from the kept k-vectors: A[(ma*(2Mb+1) + mb+Mb)*(2Mc+1) + mc+Mc].
__global__ void fourier_box_kernel(const KVec* kv, int nk, int Mb, int Mc, double2* box) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nk) return;
    KVec v = kv[k];
    long long idx = ((long long)v.ma * (2 * Mb + 1) + (long long)v.mb + Mb) * (2 * Mc + 1) + (long long)v.mc + Mc;
    box[idx] = make_double2(v.are, v.aim);
}

}  // namespace pmk
