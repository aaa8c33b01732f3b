// pm_poses.h -- energies and forces of explicit poses (libpmhip.so, gfx950).
//
// One workgroup per pose, every atom of the replicated box, nearest image per pair (src/vdw_energetics.jl:25-47,
// src/electrostatics.jl:331-388); serves vdw_energy,
// electrostatic_potential_energy and the minimiser's forces.
#pragma once

#include "pm_points.h"

namespace pmk {

struct PoseArgs {
    int ns, n_atoms, n_types, nk;
    int Ma, Mb, Mc;                       // largest |m| of the kept k-vectors per axis
    int nz;                               // phase powers per site, Ma + Mb + Mc + 3; 0: too many for LDS, the
                                          // phases come from sincospi per site and k-vector
    long long n_items;
    double f11, f12, f13, f22, f23, f33;  // replicated-box f_to_c (upper triangular)
    double c2f[9];                        // replicated-box c_to_f, column-major (forces)
    double repd[3];                       // replication factors (unit-cell phases)
    double r2_lj, r2_sr, alpha, inv4pe;
    double erfc64_inv_h;
    float r2_keep;                        // FP32 squared distance below which a pair is looked at in FP64
    Site site[PM_MAX_SITES];
    const double4* atoms;   // replicated atoms: fractional xyz + charge
    const float4* atoms_f;  // the same positions in FP32, wrapped into [0, 1)
    const int* species;
    const void* ljtab;      // [n_types][ns] of LJP<Real>
    const KVec* kv;
    const double2* erfc64_tab;
    const double* pose_xf;  // n_items x ns x 3
    double* out_e;          // n_items x 3: (vdw, sr, lr)
    double* out_g;          // GRAD: n_items x ns x 3, dE/d(site Cartesian xyz) in K/A
};

// queued pairs per wave: fewer than 64, and 64 for every site of a round
__host__ __device__ constexpr int pose_queue(int ns) { return 64 * (ns + 1); }

// Whether a pose kernel takes erfc in FP64: energies in FP64, and forces.  From the
// table (its template argument TABLE) only where that is as exact as the function,
// erfc64_table_exact().
template <bool ES, typename Real, bool GRAD>
constexpr bool pose_erfc64() {
    return ES && (sizeof(Real) == 8 || GRAD);
}

// LDS: the erfc table, the phase powers (z_a^0.., z_b^0.., z_c^0.. per site, or
// without them a phase per work-item and site), the
// LJ table, the pose's sites (position, charge), each wave's partial
// sums, the waves' queues.
struct PoseLds {
    int z, lj, site, red, queue, bytes;
};
__host__ __device__ inline PoseLds pose_lds(bool es, bool table, int nz, int n_types, int ns, bool fp64, bool grad) {
    PoseLds L{};
    L.z = table ? ERFC64_TAB * 16 : 0;
    L.lj = L.z + (es ? (nz > 0 ? nz : WG) * ns * 16 : 0);
    L.site = L.lj + ((n_types > 0 ? n_types : 1) * ns * (fp64 ? 16 : 8) + 15) / 16 * 16;
    L.red = L.site + ns * 32;
    L.queue = L.red + (WG / 64) * (4 + (grad ? 3 * ns : 0)) * 8;
    L.bytes = L.queue + (WG / 64) * pose_queue(ns) * 8;
    return L;
}

// 1/sqrt(r2): v_rsq_f64 and one third-order step; +inf below the smallest normal.
__device__ inline double rsq64(double r2) {
    double y = __builtin_amdgcn_rsq(r2);
    const double e = fma(-(r2 * y), y, 1.0);
    y = fma(e * y, fma(e, 0.375, 0.5), y);
    return r2 >= 2.2250738585072014e-308 ? y : INFINITY;
}

// erfc(alpha r) from the FP64 table (r = NaN, from r2 = 0, reads its start).
__device__ inline double erfc_tab64(double r, double inv_h, const double2* tab) {
    constexpr double MAGIC = 6755399441055744.0;  // 1.5 2^52: the sum's low word is the nearest integer
    const double x = r < 1e300 ? r : 0.0;
    const double xm = fma(x, inv_h, MAGIC);
    const double t = fma(x, inv_h, -(xm - MAGIC));
    const double2* e = tab + 3 * __double2loint(xm);
    const double2 c01 = e[0], c23 = e[1], c45 = e[2];
    return fma(fma(fma(fma(fma(c45.y, t, c45.x), t, c23.y), t, c23.x), t, c01.y), t, c01.x);
}

// The pair terms cost 10 to 20 times the distance, and about one pair in eight
// lies inside the cutoff, so a wave first takes its share of the atoms in FP32,
// one atom per lane and site after site, and queues the pairs within the cutoff
// (and a margin above the FP32 rounding of a distance) in LDS; 64 queued pairs at
// a time, one per lane, then get the FP64 nearest image, the exact cutoff and
// overlap tests and the pair terms with every lane at work.  One queue for all
// sites: a queue per site needs the pair terms' code once per site and leaves a
// last, partly filled round per site (190 us below).  A workgroup takes one pose:
// in a loop over poses the compiler keeps the constants of sincospi and exp in
// registers throughout (163 instead of 116; 127 us).  The Fourier part takes the
// phases z_a^m, z_b^m, z_c^m of every site from LDS (one sincospi per site, axis
// and power instead of one per site and k-vector).  4096 CO2 poses with forces,
// FP64, 4800 atoms, 461 k-vectors: 521 us with every pair and k-vector evaluated
// in full, one wave per pose; 105 us so.  Energies of 2048 poses: 191 -> 47 us
// (Ewald), 59 -> 31 us (LJ).  Bound by instruction issue and the latency of the
// queue's gathers at four waves per SIMD.
//   LJ      d/dx_s = 6 eps4 (2u^2 - u) / r^2 * d,   u = (sigma^2 / r^2)^3
//   real    d/dx_s = q_s q_a [erfc(a r) / r + 2a/sqrt(pi) e^{-a^2 r^2}] / r^2 * d / (4 pi eps0)
//   Fourier d/dx_s = q_s 2 pi C^T sum_k (-A_re sin th + A_im cos th) (m o rep),  th = 2 pi m.(rep o x)
// with d = x_atom - x_s (nearest image, Cartesian) and C the replicated box's c_to_f.
template <int NS, bool ES, typename Real, bool GRAD, bool TABLE>
__global__ __launch_bounds__(WG) void pose_kernel(PoseArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NV = 3 + (GRAD ? 3 * NS : 0);  // sums per pose
    const PoseLds L = pose_lds(ES, TABLE, a.nz, a.n_types, NS, sizeof(Real) == 8, GRAD);
    double2* const s_tab = reinterpret_cast<double2*>(smem);
    double2* const s_z = reinterpret_cast<double2*>(smem + L.z);
    LJP<Real>* const s_lj = reinterpret_cast<LJP<Real>*>(smem + L.lj);
    double* const s_red = reinterpret_cast<double*>(smem + L.red);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double4* const s_site = reinterpret_cast<double4*>(smem + L.site);
    int2* const queue = reinterpret_cast<int2*>(smem + L.queue) + wave * pose_queue(NS);

    const LJP<Real>* gtab = reinterpret_cast<const LJP<Real>*>(a.ljtab);
    for (int i = tid; i < a.n_types * NS; i += WG) s_lj[i] = gtab[i];
    if constexpr (TABLE)
        for (int i = tid; i < ERFC64_TAB; i += WG) s_tab[i] = a.erfc64_tab[i];

    const double f11 = a.f11, f12 = a.f12, f13 = a.f13, f22 = a.f22, f23 = a.f23, f33 = a.f33;
    const float g11 = (float)f11, g12 = (float)f12, g13 = (float)f13, g22 = (float)f22, g23 = (float)f23,
                g33 = (float)f33;
    const double r2lj = a.r2_lj, r2sr = a.r2_sr, alpha = a.alpha;
    const double two_a_rpi = 2.0 * alpha * 0.56418958354775628;  // 2 alpha / sqrt(pi)
    const int n_atoms = a.n_atoms;
    unsigned lj_mask = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) lj_mask |= a.site[s].lj != 0 ? 1u << s : 0u;

    const long long item = blockIdx.x;
    if (tid < NS) {
        const double* p = a.pose_xf + (item * NS + tid) * 3;
        s_site[tid] = make_double4(p[0], p[1], p[2], a.site[tid].q);
    }
    if constexpr (ES) {
        const int nz = a.nz;
        for (int i = tid; i < nz * NS; i += WG) {
            const int s = i / nz;
            int m = i - s * nz, d = 0;
            if (m > a.Ma) { m -= a.Ma + 1; d = 1; }
            if (d == 1 && m > a.Mb) { m -= a.Mb + 1; d = 2; }
            double t = (double)m * (a.pose_xf[(item * NS + s) * 3 + d] * a.repd[d]);
            t -= rint(t);
            double sn, cs;
            sincospi(2.0 * t, &sn, &cs);
            s_z[i] = make_double2(cs, sn);
        }
    }
    __syncthreads();  // the tables, sites and phases

    double acc_lj = 0.0, acc_sr = 0.0, acc_lr = 0.0;
    double gx[NS], gy[NS], gz[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) { gx[s] = 0.0; gy[s] = 0.0; gz[s] = 0.0; }
    bool ovl = false;
    if constexpr (ES) {
        const int nz = a.nz, ob = a.Ma + 1, oc = ob + a.Mb + 1;
        double hx[NS], hy[NS], hz[NS];  // gradient in (m o rep) space
#pragma unroll
        for (int s = 0; s < NS; ++s) { hx[s] = 0.0; hy[s] = 0.0; hz[s] = 0.0; }
        auto add = [&](const KVec& v, int s, double2 w) {  // w = e^{i 2 pi m.(rep o x_s)}
            acc_lr += s_site[s].w * (v.are * w.x + v.aim * w.y);
            if constexpr (GRAD) {
                const double d = v.aim * w.x - v.are * w.y;
                hx[s] += d * v.ma;
                hy[s] += d * v.mb;
                hz[s] += d * v.mc;
            }
        };
        if (nz > 0) {
#pragma unroll 1
            for (int k = tid; k < a.nk; k += WG) {
                const KVec v = a.kv[k];
                const int ma = (int)v.ma, mb = (int)v.mb, mc = (int)v.mc;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const double2* z = s_z + s * nz;
                    double2 zb = z[ob + abs(mb)], zc = z[oc + abs(mc)];
                    zb.y = mb < 0 ? -zb.y : zb.y;
                    zc.y = mc < 0 ? -zc.y : zc.y;
                    add(v, s, cmul(cmul(z[ma], zb), zc));
                }
            }
        } else {
#pragma unroll 1
            for (int k = tid; k < a.nk; k += WG) {
                const KVec v = a.kv[k];
#pragma unroll 1
                for (int s = 0; s < NS; ++s) {
                    const double4 x = s_site[s];
                    double t = v.ma * (x.x * a.repd[0]) + v.mb * (x.y * a.repd[1]) + v.mc * (x.z * a.repd[2]);
                    t -= rint(t);
                    double sn, cs;
                    sincospi(2.0 * t, &sn, &cs);
                    s_z[s * WG + tid] = make_double2(cs, sn);
                }
#pragma unroll
                for (int s = 0; s < NS; ++s) add(v, s, s_z[s * WG + tid]);
            }
        }
        if constexpr (GRAD) {
            const double* C = a.c2f;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                // 2 pi q_s C^T (h o rep)
                const double q2p = 2.0 * M_PI * a.site[s].q;
                const double vx = hx[s] * a.repd[0] * q2p, vy = hy[s] * a.repd[1] * q2p, vz = hz[s] * a.repd[2] * q2p;
                gx[s] += C[0] * vx + C[1] * vy + C[2] * vz;
                gy[s] += C[3] * vx + C[4] * vy + C[5] * vz;
                gz[s] += C[6] * vx + C[7] * vy + C[8] * vz;
            }
        }
    }

    float tx[NS], ty[NS], tz[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const double4 x = s_site[s];
        tx[s] = (float)(x.x - floor(x.x));
        ty[s] = (float)(x.y - floor(x.y));
        tz[s] = (float)(x.z - floor(x.z));
    }
    // atom round by atom round, then what is left in the queue
    int cnt = 0;
    for (int base = 0;;) {
        const bool done = base >= n_atoms;
        if (!done) {
            const int j = base + tid;
            const bool have = j < n_atoms;
            const float4 at = a.atoms_f[have ? j : 0];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                float dx = at.x - tx[s], dy = at.y - ty[s], dz = at.z - tz[s];
                dx -= rintf(dx);
                dy -= rintf(dy);
                dz -= rintf(dz);
                const float cx = fmaf(g13, dz, fmaf(g12, dy, g11 * dx)), cy = fmaf(g23, dz, g22 * dy), cz = g33 * dz;
                const bool keep = have && fmaf(cz, cz, fmaf(cy, cy, cx * cx)) < a.r2_keep;
                const unsigned long long m = __ballot(keep);
                if (keep) queue[cnt + __popcll(m & ((1ull << lane) - 1ull))] = make_int2(j, s);
                cnt += __popcll(m);
            }
            base += WG;
        } else if (cnt == 0) {
            break;
        }
        for (const int least = done ? 1 : 64; cnt >= least;) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int n = min(cnt, 64);
            cnt -= n;
            if (lane < n) {
                const int2 q = queue[cnt + lane];
                const double4 p = a.atoms[q.x];
                const double4 x = s_site[q.y];
                const LJP<Real> c = s_lj[a.species[q.x] * NS + q.y];
                double ex = p.x - x.x, ey = p.y - x.y, ez = p.z - x.z;
                ex -= rint(ex);
                ey -= rint(ey);
                ez -= rint(ez);
                const double px = f11 * ex + f12 * ey + f13 * ez;
                const double py = f22 * ey + f23 * ez;
                const double pz = f33 * ez;
                const double r2 = px * px + py * py + pz * pz;
                const bool in = r2 < r2lj;
                ovl |= in & (r2 < R2_OVERLAP) & (((lj_mask >> q.y) & 1u) != 0u);
                const double y = rsq64(r2);
                const double i2 = y * y;
                if constexpr (sizeof(Real) == 4) {
                    acc_lj += in ? (double)lj_f32(r2, c.sig2, c.eps4) : 0.0;
                } else {
                    const double w = c.sig2 * i2;
                    const double u = w * w * w;
                    acc_lj += in ? c.eps4 * u * (u - 1.0) : 0.0;
                }
                double f = 0.0;  // the pair's force is f times (px, py, pz)
                if constexpr (GRAD) {
                    const double w = (double)c.sig2 * i2;
                    const double u = w * w * w;
                    f = in ? 6.0 * (double)c.eps4 * u * (2.0 * u - 1.0) * i2 : 0.0;
                }
                if constexpr (ES) {
                    const bool ins = (r2 < r2sr) & (p.w != 0.0);
                    double t = 0.0;  // erfc(alpha r) / r
                    if constexpr (TABLE) {
                        t = y * erfc_tab64(ins ? r2 * y : 0.0, a.erfc64_inv_h, s_tab);
                    } else if constexpr (pose_erfc64<ES, Real, GRAD>()) {
                        const double r = sqrt(r2);
                        t = erfc(alpha * r) / r;
                    }
                    if constexpr (sizeof(Real) == 4)
                        acc_sr += ins ? x.w * (double)coul_f32(r2, p.w, alpha) : 0.0;
                    else
                        acc_sr += ins ? x.w * (p.w * t) : 0.0;
                    if constexpr (GRAD)
                        f += ins ? p.w * (t + two_a_rpi * exp(-alpha * alpha * r2)) * i2 * x.w * a.inv4pe : 0.0;
                }
                if constexpr (GRAD) {
                    const double ux = f * px, uy = f * py, uz = f * pz;
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        gx[s] += q.y == s ? ux : 0.0;
                        gy[s] += q.y == s ? uy : 0.0;
                        gz[s] += q.y == s ? uz : 0.0;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }

    // fixed-order sums over the lanes, then over the waves
    double v[NV];
    v[0] = acc_lj;
    v[1] = acc_sr;
    v[2] = acc_lr;
    if constexpr (GRAD)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            v[3 + 3 * s] = gx[s];
            v[4 + 3 * s] = gy[s];
            v[5 + 3 * s] = gz[s];
        }
    const bool hit = __ballot(ovl) != 0ull;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const double t = wave_sum(v[i]);
        if (lane == 0) s_red[wave * (NV + 1) + i] = t;
    }
    if (lane == 0) s_red[wave * (NV + 1) + NV] = hit ? 1.0 : 0.0;
    __syncthreads();
    if (tid < NV) {
        double t = 0.0;
        bool o = false;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) {
            t += s_red[w * (NV + 1) + tid];
            o |= s_red[w * (NV + 1) + NV] != 0.0;
        }
        if (tid == 0) a.out_e[3 * item] = o ? INFINITY : t;
        else if (tid == 1) a.out_e[3 * item + 1] = t * a.inv4pe;
        else if (tid == 2) a.out_e[3 * item + 2] = t;
        else if constexpr (GRAD) a.out_g[item * (3 * NS) + tid - 3] = t;
    }
}

}  // namespace pmk
