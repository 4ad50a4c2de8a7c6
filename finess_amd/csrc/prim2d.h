// prim2d.h -- the fused FP64 face: characteristic WENO5-LLF on primitive cell
// records (lib/2d/ConstructL.cpp:63-208 for x, :215-358 for y), for 2D Euler
// and shallow water.  Used by the plain and batched FP64 stages and, with
// given fluxes, by the Lax-Wendroff and RK4-PIF stages.
//
// The stage is bound by FP64 instruction issue, so the face is arranged for
// the fewest instructions and LDS reads.  With (u1, u2, u3) the mean velocity
// and d = u - u1 etc. the differences of a stencil cell's velocity from it,
// the left eigenvectors of the mean state act on q and on
// f = u q + p (e_2 + u e_5) through three numbers per cell,
//     t  = p / (g-1) + rho |d|^2 / 2,    m = rho d1,    tv = rho d2 (tw = rho d3),
// and, for a split part v = f + s q with l = u + s,
//     T = l t + p d1,   M = l m + p,
//     w_1,5 = (g-1) T / (2 c^2) -+ M / (2 c),   w_2 = l rho - (g-1) T / c^2,
//     w_3 = l tv,  w_4 = l tw
// (t and m are the energy and the normal momentum of the cell in the frame of
// the mean velocity, which also keeps them free of the cancellation of
// E - u.m + rho u^2 / 2).  So a record is (rho, u, v, w, p, c) and a stencil
// cell is four LDS reads and, for both parts, 27 FP64 instructions, where the
// conserved records took six reads and 56.  The two parts run one after the
// other in a rolled loop (unrolled, both parts' values are live and the kernel
// takes 194 registers instead of 128).
//
// Euler, Runge-Kutta, 1024^2: 25.6 M VALU instructions and 59 us per stage
// (40.6 M and 88 us with conserved records and the reconstruction of weno5);
// shallow water 43 us (71; its flux divided by h at every stencil cell).
#pragma once
#include <type_traits>

#include "physics.h"
#include "weno.h"

namespace finess {

// max(|s1|, |s2|), at least the global speed of the direction where
// global_alpha is set (lib/2d/ConstructL.cpp:172,323).  `sp` is a sum that is
// NaN whenever the face's state is: fmin and fmax drop NaNs, and a NaN speed
// has to stay one.
__host__ __device__ __forceinline__ double face_speed(double s1, double s2, double sp, const double* galpha)
{
    const double ws = fma(0.0, sp, fmax(fabs(s1), fabs(s2)));
    if (!galpha) return ws;
    const double amin = *galpha;
    return amin > ws ? amin : ws;
}

struct EulerPrim : Euler2D {
    static constexpr bool PRIM = true;
    static constexpr int NV = 6;  // rho, u, v, w, p, c

    __host__ __device__ __forceinline__ static void cell_record(const double q[5], const PhysParams& pp, double v[6])
    {
        const double ir = rcp_d(q[0]);
        const double u = q[1] * ir, vv = q[2] * ir, w = q[3] * ir;
        const double p = (pp.gamma - 1.0) * (q[4] - 0.5 * (q[1] * u + q[2] * vv + q[3] * w));
        v[0] = q[0]; v[1] = u; v[2] = vv; v[3] = w; v[4] = p;
        v[5] = sqrt_d(fabs(pp.gamma * p * ir));
    }

    // Flux of one face; cv: records, the stencil cell s at base + s * stride
    // (cells i-3..i+2).  LXW: the stencil fluxes are given (flux of cell s
    // and field k at lflux[k * lplane + lbase + s * lstride]; the tile keeps
    // them in LDS).
    // SKIP3: every stencil cell (and flux) has zero rho w.  Returns alpha.
    template <int WK, bool LXW, bool SKIP3, int NC>
    __device__ __host__ __forceinline__ static double face(const double (*cv)[NC], int base, int stride, int dir,
                                                           const double* lflux, long long lbase, long long lstride,
                                                           long long lplane, const PhysParams& pp, double eps,
                                                           double power, double ascale, double fh[5], const double* galpha)
    {
        const int iu = 1 + dir, iv = 2 - dir;
        const double gam = pp.gamma, gm1 = gam - 1.0;
        double u1, u2, u3 = 0.0, c2, alpha;
        {
            const int l = base + 2 * stride, r = base + 3 * stride;
            const double rl = cv[0][l], ul = cv[iu][l], vl = cv[iv][l], pl = cv[4][l];
            const double rr = cv[0][r], ur = cv[iu][r], vr = cv[iv][r], pr = cv[4][r];
            // the mean state (lib/2d/ConstructL.cpp:72-77) in primitive terms:
            // density-weighted velocities, and the pressure of the mean
            // energy, p = (p_l + p_r)/2 + (g-1) rho_l rho_r |du|^2 / (8 rho)
            const double irs = rcp_d(rl + rr);
            const double fl = rl * irs, fr = rr * irs;
            u1 = fma(fl, ul, fr * ur);
            u2 = fma(fl, vl, fr * vr);
            const double du = ur - ul, dv = vr - vl;
            double dd = fma(du, du, dv * dv);
            if (!SKIP3) {
                const double wl = cv[3][l], wr = cv[3][r];
                u3 = fma(fl, wl, fr * wr);
                dd = fma(wr - wl, wr - wl, dd);
            }
            const double gp = gam * ((pl + pr) * irs);
            c2 = fma(0.5 * gam * gm1 * (fl * fr), dd, gp);
            // SetWaveSpd (apps/2d/euler/lib/SetWaveSpd.cpp:47-69)
            const double un = 0.5 * (ul + ur), cm = sqrt_d(fabs(gp)), sp = un + cm;
            const double s1 = fmin(ul - cv[5][l], un - cm), s2 = fmax(ur + cv[5][r], sp);
            alpha = face_speed(s1, s2, sp, galpha);
        }
        const double la = ascale * alpha;
        const double ic = rsqrt_d(c2), c = c2 * ic;
        const double hic = 0.5 * ic, b = gm1 * (ic * ic), b2 = 0.5 * b, ig = 1.0 / gm1;
        double hu = fma(u1, u1, u2 * u2);
        if (!SKIP3) hu = fma(u3, u3, hu);
        hu *= 0.5;
        double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        // part +: f + la q over cells 0..4; part -: f - la q over cells 5..1
        double sl = la;
        int k0 = base, ks = stride;
        long long f0_ = lbase, fs_ = lstride;
#pragma unroll 1
        for (int part = 0; part < 2; part++) {
            double g0[5], g1[5], g2[5], g4[5];
#pragma unroll
            for (int n = 0; n < 5; n++) {
                const int k = k0 + n * ks;
                const double rho = cv[0][k], u = cv[iu][k], p = cv[4][k];
                const double d1 = u - u1, d2 = cv[iv][k] - u2;
                const double m = rho * d1, tv = rho * d2;
                double e = fma(tv, d2, m * d1);
                if (!SKIP3) {
                    const double d3 = cv[3][k] - u3;
                    e = fma(rho * d3, d3, e);
                }
                const double t = fma(0.5, e, p * ig);
                double T, M;
                if (LXW) {
                    const double* f = lflux + f0_ + n * fs_;
                    const double f0 = f[0], f1 = f[iu * lplane], f2 = f[iv * lplane], f4 = f[4 * lplane];
                    double tf = fma(-u2, f2, fma(-u1, f1, fma(hu, f0, f4)));
                    if (!SKIP3) tf = fma(-u3, f[3 * lplane], tf);
                    T = fma(sl, t, tf);
                    M = fma(sl, m, fma(-u1, f0, f1));
                    g1[n] = fma(sl, rho, fma(-b, T, f0));
                    if (SKIP3) g2[n] = fma(sl, tv, fma(-u2, f0, f2));
                } else {
                    const double l = u + sl;
                    T = fma(l, t, p * d1);
                    M = fma(l, m, p);
                    g1[n] = fma(l, rho, -(b * T));
                    if (SKIP3) g2[n] = l * tv;
                }
                const double hm = hic * M;
                g0[n] = fma(b2, T, -hm);
                g4[n] = fma(b2, T, hm);
            }
            w[0] += weno5_fp64<WK>(g0, 4.0 * eps, power);
            w[4] += weno5_fp64<WK>(g4, 4.0 * eps, power);
            w[1] += weno5_fp64<WK>(g1, 4.0 * eps, power);
            if (!SKIP3) {
                // both shear fields in a second pass over the stencil: the
                // fields of the first pass are done, so the registers stay
                // those of the form without rho w (the empty asm keeps the
                // compiler from carrying the stencil over instead)
                asm volatile("" ::: "memory");
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    const int k = k0 + n * ks;
                    const double rho = cv[0][k], tv = rho * (cv[iv][k] - u2), tw = rho * (cv[3][k] - u3);
                    if (LXW) {
                        const double* f = lflux + f0_ + n * fs_;
                        g2[n] = fma(sl, tv, fma(-u2, f[0], f[iv * lplane]));
                        g4[n] = fma(sl, tw, fma(-u3, f[0], f[3 * lplane]));
                    } else {
                        const double l = cv[iu][k] + sl;
                        g2[n] = l * tv;
                        g4[n] = l * tw;
                    }
                }
                w[3] += weno5_fp64<WK>(g4, 4.0 * eps, power);
            }
            w[2] += weno5_fp64<WK>(g2, 4.0 * eps, power);
            sl = -sl;
            k0 += 5 * stride;
            ks = -stride;
            f0_ += 5 * lstride;
            fs_ = -lstride;
        }
        // back through the right eigenvectors (ProjectRightEig.cpp), with the
        // 1/2 of the splitting; H = c^2/(g-1) + |u|^2/2
        const double y = 0.5 * (w[0] + w[4]), x = 0.5 * c * (w[4] - w[0]), s = fma(0.5, w[1], y);
        const double h2 = 0.5 * w[2];
        fh[0] = s;
        fh[iu] = fma(u1, s, x);
        fh[iv] = fma(u2, s, h2);
        double en = fma(hu, s, fma(c2 * ig, y, fma(u1, x, u2 * h2)));
        if (SKIP3) {
            fh[3] = 0.0;
        } else {
            const double h3 = 0.5 * w[3];
            fh[3] = fma(u3, s, h3);
            en = fma(u3, h3, en);
        }
        fh[4] = en;
        return alpha;
    }
};

// Shallow water (g = 1): records (h, u, v, sqrt h); with m = h (u - u1) and
// M = l m + h^2/2 the split characteristic values are (l h -+ M/c)/2 and
// l h (v - u2).
struct ShallowWaterPrim : ShallowWater2D {
    static constexpr bool PRIM = true;
    static constexpr int NV = 4;

    __host__ __device__ __forceinline__ static void cell_record(const double q[3], const PhysParams&, double v[4])
    {
        const double ih = rcp_d(q[0]);
        v[0] = q[0]; v[1] = q[1] * ih; v[2] = q[2] * ih;
        v[3] = sqrt_d(q[0]);
    }

    template <int WK, bool LXW, bool SKIP3, int NC>
    __device__ __host__ __forceinline__ static double face(const double (*cv)[NC], int base, int stride, int dir,
                                                           const double* lflux, long long lbase, long long lstride,
                                                           long long lplane, const PhysParams& pp, double eps,
                                                           double power, double ascale, double fh[3], const double* galpha)
    {
        const int iu = 1 + dir, iv = 2 - dir;
        double u1, u2, c, ic, alpha;
        {
            const int l = base + 2 * stride, r = base + 3 * stride;
            const double hl = cv[0][l], ul = cv[iu][l], vl = cv[iv][l], sl = cv[3][l];
            const double hr = cv[0][r], ur = cv[iu][r], vr = cv[iv][r], sr = cv[3][r];
            const double irs = rcp_d(hl + hr), hm = 0.5 * (hl + hr);
            const double fl = hl * irs, fr = hr * irs;
            u1 = fma(fl, ul, fr * ur);
            u2 = fma(fl, vl, fr * vr);
            ic = rsqrt_d(hm);
            c = hm * ic;
            // SetWaveSpd, with its u_r = (hu)_r / h_l when sw_compat_hl is set
            const double unr = pp.sw_compat_hl ? hr * ur * rcp_d(hl) : ur;
            const double un = fma(sl, ul, sr * unr) * rcp_d(sl + sr);
            const double s1 = fmin(un - c, ul - sl), s2 = fmax(un + c, unr + sr);
            alpha = face_speed(s1, s2, un + c, galpha);
        }
        const double la = ascale * alpha, hic = 0.5 * ic;
        double w[3] = {0.0, 0.0, 0.0};
        double sl = la;
        int k0 = base, ks = stride;
        long long f0_ = lbase, fs_ = lstride;
#pragma unroll 1
        for (int part = 0; part < 2; part++) {
            double g0[5], g1[5], g2[5];
#pragma unroll
            for (int n = 0; n < 5; n++) {
                const int k = k0 + n * ks;
                const double h = cv[0][k], u = cv[iu][k];
                const double m = h * (u - u1), tv = h * (cv[iv][k] - u2);
                double H, M;
                if (LXW) {
                    const double* f = lflux + f0_ + n * fs_;
                    const double f0 = f[0];
                    H = fma(sl, h, f0);
                    M = fma(sl, m, fma(-u1, f0, f[iu * lplane]));
                    g1[n] = fma(sl, tv, fma(-u2, f0, f[iv * lplane]));
                } else {
                    const double l = u + sl;
                    H = l * h;
                    M = fma(l, m, 0.5 * h * h);
                    g1[n] = l * tv;
                }
                const double hm = hic * M;
                g0[n] = fma(0.5, H, -hm);
                g2[n] = fma(0.5, H, hm);
            }
            auto add = [&](int k, const double* g) {
                const double v = weno5_fp64<WK>(g, 4.0 * eps, power);
                w[k] += v;
            };
            add(0, g0);
            add(2, g2);
            add(1, g1);
            sl = -sl;
            k0 += 5 * stride;
            ks = -stride;
            f0_ += 5 * lstride;
            fs_ = -lstride;
        }
        const double s = 0.5 * (w[0] + w[2]), x = 0.5 * c * (w[2] - w[0]);
        fh[0] = s;
        fh[iu] = fma(u1, s, x);
        fh[iv] = fma(u2, s, 0.5 * w[1]);
        return alpha;
    }
};

} // namespace finess
