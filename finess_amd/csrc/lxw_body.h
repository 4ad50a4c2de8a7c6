// lxw_body.h -- time-integrated fluxes of the third-order Lax-Wendroff
// (Picard integral) step, lib/2d/ConstructIntegratedR.cpp:59-296:
//
//   F = f + dt/2 (f_t + dt/3 f_tt),   G = g + dt/2 (g_t + dt/3 g_tt)
//   S = f_x + g_y,   f_t = -A1 S,   g_t = -A2 S
//   q_tt = H1(q_x, S) + H2(q_y, S) + A1 (f_xx + g_xy) + A2 (f_xy + g_yy)
//   f_tt = A1 q_tt + H1(S, S),   g_tt = A2 q_tt + H2(S, S)
//
// with A_d the flux Jacobians and H_d(a, b) their second derivatives applied
// to two vectors.  The reference forms A and H as explicit tensors from the
// app's DFluxFunc / D2FluxFunc and contracts them.  The FP64 form of the
// unlimited step writes the products out (lxw64_cell); in the FP32 form and the
// limited step every product is a directional derivative of the flux itself,
// evaluated exactly with
// hyper-dual numbers (x + a e1 + b e2 + ab e1e2, e1^2 = e2^2 = 0): one flux
// evaluation at q + a e1 + b e2 yields A a (e1 part), A b (e2 part) and
// H(a, b) (e1e2 part).  Derivatives: 5-point central differences Diff1/Diff2
// (lib/WenoReconstruct.cpp:702-716, 791-806) and the 4-point cross
// derivative of ConstructIntegratedR.cpp:202-213.
#pragma once
#include "physics.h"
#include "stage2d_body.h"

namespace finess {

template <typename T>
struct HD {
    T v, a, b, ab;
};
template <typename T>
__host__ __device__ __forceinline__ HD<T> operator+(HD<T> x, HD<T> y) { return {x.v + y.v, x.a + y.a, x.b + y.b, x.ab + y.ab}; }
template <typename T>
__host__ __device__ __forceinline__ HD<T> operator-(HD<T> x, HD<T> y) { return {x.v - y.v, x.a - y.a, x.b - y.b, x.ab - y.ab}; }
template <typename T>
__host__ __device__ __forceinline__ HD<T> operator*(HD<T> x, HD<T> y)
{
    return {x.v * y.v, x.v * y.a + x.a * y.v, x.v * y.b + x.b * y.v, x.v * y.ab + x.a * y.b + x.b * y.a + x.ab * y.v};
}
template <typename T>
__host__ __device__ __forceinline__ HD<T> operator*(T s, HD<T> x) { return {s * x.v, s * x.a, s * x.b, s * x.ab}; }
template <typename T>
__host__ __device__ __forceinline__ HD<T> hinv(HD<T> x)
{
    const T i = T(1) / x.v, i2 = i * i;
    return {i, -x.a * i2, -x.b * i2, (T(2) * x.a * x.b * i - x.ab) * i2};
}

// Flux of each physics in any number type (same expressions as FluxFunc).
template <typename T>
__host__ __device__ __forceinline__ void euler_flux(const T q[5], T gm1, T F[5], T G[5])
{
    const T rho = q[0];
    const T ir = hinv(rho);
    const T u1 = q[1] * ir, u2 = q[2] * ir, u3 = q[3] * ir;
    const T e = q[4];
    const T press = gm1 * (e - typename T::scalar(0.5) * (rho * (u1 * u1 + u2 * u2 + u3 * u3)));
    const T ru1 = rho * u1, ru2 = rho * u2, ep = e + press;
    F[0] = ru1; F[1] = ru1 * u1 + press; F[2] = ru1 * u2; F[3] = ru1 * u3; F[4] = u1 * ep;
    G[0] = ru2; G[1] = ru2 * u1; G[2] = ru2 * u2 + press; G[3] = ru2 * u3; G[4] = u2 * ep;
}

// Hyper-dual number of scalar type T (double for the plain form, float for
// the FP32 stencil form).
template <typename T>
struct HDs : HD<T> {
    using scalar = T;
    __host__ __device__ HDs() {}
    __host__ __device__ HDs(const HD<T>& x) : HD<T>(x) {}
    __host__ __device__ HDs(T v_, T a_, T b_, T ab_) : HD<T>{v_, a_, b_, ab_} {}
};
template <typename T>
__host__ __device__ __forceinline__ HDs<T> operator+(HDs<T> x, HDs<T> y) { return HDs<T>(HD<T>(x) + HD<T>(y)); }
template <typename T>
__host__ __device__ __forceinline__ HDs<T> operator-(HDs<T> x, HDs<T> y) { return HDs<T>(HD<T>(x) - HD<T>(y)); }
template <typename T>
__host__ __device__ __forceinline__ HDs<T> operator*(HDs<T> x, HDs<T> y) { return HDs<T>(HD<T>(x) * HD<T>(y)); }
template <typename T>
__host__ __device__ __forceinline__ HDs<T> operator*(T s, HDs<T> x) { return HDs<T>(s * HD<T>(x)); }
template <typename T>
__host__ __device__ __forceinline__ HDs<T> hinv(HDs<T> x) { return HDs<T>(hinv(HD<T>(x))); }
using HDd = HDs<double>;

template <class P>
struct LxwPhys;

template <>
struct LxwPhys<Euler2D> {
    static constexpr int M = 5;
    template <typename R>
    __host__ __device__ __forceinline__ static void flux(const R q[5], const PhysParams& pp, R F[5], R G[5])
    {
        const R rho = q[0];
        const R u1 = div_lp(q[1], rho), u2 = div_lp(q[2], rho), u3 = div_lp(q[3], rho);
        const R e = q[4];
        const R press = R(pp.gamma - 1.0) * (e - R(0.5) * rho * (u1 * u1 + u2 * u2 + u3 * u3));
        F[0] = rho * u1; F[1] = rho * u1 * u1 + press; F[2] = rho * u1 * u2; F[3] = rho * u1 * u3; F[4] = u1 * (e + press);
        G[0] = rho * u2; G[1] = rho * u2 * u1; G[2] = rho * u2 * u2 + press; G[3] = rho * u2 * u3; G[4] = u2 * (e + press);
    }
    // hyper-dual flux at q + a e1 + b e2
    template <typename R>
    __host__ __device__ __forceinline__ static void flux_hd(const R q[5], const R a[5], const R b[5],
                                                            const PhysParams& pp, HDs<R> F[5], HDs<R> G[5])
    {
        HDs<R> x[5];
        for (int m = 0; m < 5; m++) x[m] = HDs<R>(q[m], a[m], b[m], R(0));
        euler_flux<HDs<R>>(x, HDs<R>(R(pp.gamma - 1.0), R(0), R(0), R(0)), F, G);
    }
};

struct LxwArgs {
    const double* q;     // state planes (mx*my), boundary-mapped on load
    void* F;             // out: planes (mx+6)*(my+6), extended index (i+3)*(my+6)+(j+3),
    void* G;             //      of R (the kernel's arithmetic: FP64, or FP32 for the FP32 form)
    int mx, my;
    long long plane;
    int bc[4];
    int time_order;
    double dt, dx, dy;
    PhysParams pp;
    int src_ghosts;      // >0: q planes include that many ghosts per side (drop-in mode)
    int limited;         // the fluxes go to the limited step
    double idx, idy;     // 1/dx, 1/dy (the FP64 form)
    // device-controlled stepping (null: off): dt = *dtp, and the kernels
    // return at once while *halt is non-zero
    const double* dtp;
    const unsigned long long* halt;
};

__host__ __device__ __forceinline__ double lxw_dt(const LxwArgs& a) { return a.dtp ? *a.dtp : a.dt; }
__host__ __device__ __forceinline__ bool lxw_halted(const LxwArgs& a) { return a.halt && *a.halt != 0ull; }

// R: the arithmetic of the differences and Taylor terms (double in the plain
// form, float in the FP32 stencil form, whose stage reads these fluxes as FP32).
template <int TI, int TJ, int M, typename R = double>
struct LxwSmem {
    static constexpr int HI = TI + 4, HJ = TJ + 4, NC = HI * HJ;
    R q[M][NC];
    R f[M][NC];
    R g[M][NC];
};

template <class P>
__host__ __device__ __forceinline__ void lxw_load_state(const LxwArgs& a, int gi, int gj, double q[P::MEQN])
{
    if (a.src_ghosts) {
        const int g = a.src_ghosts;
        const long long ld = a.my + 2 * g;
        const long long pl = (long long)(a.mx + 2 * g) * ld;
        const long long idx = (long long)(gi + g) * ld + (gj + g);
        for (int m = 0; m < P::MEQN; m++) q[m] = a.q[m * pl + idx];
        return;
    }
    int fi, fj;
    const int si = bc_map(a.bc[0], a.bc[1], gi, a.mx, fi);
    const int sj = bc_map(a.bc[2], a.bc[3], gj, a.my, fj);
    const long long idx = (long long)si * a.my + sj;
    for (int m = 0; m < P::MEQN; m++) q[m] = a.q[m * a.plane + idx];
    if (fi) q[P::NORMAL_X] = -q[P::NORMAL_X];
    if (fj) q[P::NORMAL_Y] = -q[P::NORMAL_Y];
}

// The states of this thread's cells (number tid, tid + TI TJ, ...) of the tile
// and its 2-cell halo.  Every load is issued before the first is used, and a
// tile whose halo lies inside the grid (most of them) is read directly, by
// 32-bit offsets from the halo's first cell (2048^2: FP64 flux kernel 143 ->
// 135 us, FP32 123 -> 116).
template <class P, int TI, int TJ>
struct LxwCells {
    static constexpr int HI = TI + 4, HJ = TJ + 4, NC = HI * HJ, NT = TI * TJ, K = (NC + NT - 1) / NT;
    double q[K][P::MEQN];
    bool ok[K];

    __host__ __device__ __forceinline__ void load(int tid, int e0i, int e0j, const LxwArgs& a)
    {
        const int i0 = e0i - 5, j0 = e0j - 5;
        const bool inner = !a.src_ghosts && i0 >= 0 && j0 >= 0 && i0 + HI <= a.mx && j0 + HJ <= a.my && a.my < (1 << 24);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int c = tid + k * NT, ci = c / HJ, cj = c - ci * HJ;
            ok[k] = c < NC;
            if (inner) {
                if (ok[k]) {
                    const unsigned off = (unsigned)(ci * a.my + cj) * 8u;
                    const double* s = a.q + ((long long)i0 * a.my + j0);
                    for (int m = 0; m < P::MEQN; m++)
                        q[k][m] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(s + m * a.plane) + off);
                }
            } else {
                ok[k] = ok[k] && i0 + ci <= a.mx + 4 && j0 + cj <= a.my + 4;
                if (ok[k]) lxw_load_state<P>(a, i0 + ci, j0 + cj, q[k]);
            }
        }
    }
};

// Phase 1: states and point fluxes of the tile plus a 2-cell halo (corners
// included: the cross derivatives read the diagonal neighbours).
template <class P, int TI, int TJ, typename R = double>
__host__ __device__ __forceinline__ void lxw_phase_load(int tid, int e0i, int e0j, const LxwArgs& a,
                                                        LxwSmem<TI, TJ, P::MEQN, R>& sm)
{
    LxwCells<P, TI, TJ> cells;
    cells.load(tid, e0i, e0j, a);
#pragma unroll
    for (int k = 0; k < cells.K; k++) {
        if (!cells.ok[k]) continue;
        const int c = tid + k * cells.NT;
        R q[P::MEQN], f[P::MEQN], g[P::MEQN];
        for (int m = 0; m < P::MEQN; m++) q[m] = R(cells.q[k][m]);
        LxwPhys<P>::flux(q, a.pp, f, g);
        for (int m = 0; m < P::MEQN; m++) { sm.q[m][c] = q[m]; sm.f[m][c] = f[m]; sm.g[m][c] = g[m]; }
    }
}

// The same for a workgroup of nthreads threads (at most TI TJ, whose shares of
// the cells they take in turn).
template <class P, int TI, int TJ, typename R = double>
__host__ __device__ __forceinline__ void lxw_phase_load(int tid, int nthreads, int e0i, int e0j, const LxwArgs& a,
                                                        LxwSmem<TI, TJ, P::MEQN, R>& sm)
{
    do {
        lxw_phase_load<P, TI, TJ, R>(tid, e0i, e0j, a, sm);
        tid += nthreads;
    } while (tid < TI * TJ);
}

template <typename R>
__host__ __device__ __forceinline__ R d1(R h, R f0, R f1, R f3, R f4)
{
    R t = (f0 - f4) * R(1.0 / 12.0);
    t += (-f1 + f3) * R(2.0 / 3.0);
    return div_lp(t, h);
}
template <typename R>
__host__ __device__ __forceinline__ R d2(R h, R f0, R f1, R f2, R f3, R f4)
{
    R t = (-f0 - f4) * R(1.0 / 12.0);
    t += (f1 + f3) * R(4.0 / 3.0);
    t += (-f2) * R(5.0 / 2.0);
    return div_lp(t, h * h);
}

// Phase 2: one output cell per thread.
template <class P, int TI, int TJ, typename R = double>
__host__ __device__ __forceinline__ void lxw_phase_cell(int tid, int e0i, int e0j, const LxwArgs& a,
                                                        const LxwSmem<TI, TJ, P::MEQN, R>& sm)
{
    using S = LxwSmem<TI, TJ, P::MEQN, R>;
    constexpr int M = P::MEQN;
    const int ci = tid / TJ, cj = tid - ci * TJ;
    const int ei = e0i + ci, ej = e0j + cj;              // extended index, gi = ei - 3
    if (ci >= TI || ei >= a.mx + 6 || ej >= a.my + 6) return;
    const int c = (ci + 2) * S::HJ + (cj + 2);
    const int X = S::HJ, Y = 1;
    const R dx = R(a.dx), dy = R(a.dy), dt = R(lxw_dt(a));
    R q[M], fx[M], gy[M], qx[M], qy[M], S_[M];
    for (int m = 0; m < M; m++) {
        q[m] = sm.q[m][c];
        fx[m] = d1(dx, sm.f[m][c - 2 * X], sm.f[m][c - X], sm.f[m][c + X], sm.f[m][c + 2 * X]);
        qx[m] = d1(dx, sm.q[m][c - 2 * X], sm.q[m][c - X], sm.q[m][c + X], sm.q[m][c + 2 * X]);
        gy[m] = d1(dy, sm.g[m][c - 2 * Y], sm.g[m][c - Y], sm.g[m][c + Y], sm.g[m][c + 2 * Y]);
        qy[m] = d1(dy, sm.q[m][c - 2 * Y], sm.q[m][c - Y], sm.q[m][c + Y], sm.q[m][c + 2 * Y]);
        S_[m] = fx[m] + gy[m];
    }
    HDs<R> F1[M], G1[M];
    LxwPhys<P>::flux_hd(q, qx, S_, a.pp, F1, G1);      // A S (e2), H1(qx, S) (e1e2)
    R f_t[M], g_t[M], f_tt[M], g_tt[M];
    for (int m = 0; m < M; m++) { f_t[m] = -F1[m].b; g_t[m] = -G1[m].b; f_tt[m] = R(0); g_tt[m] = R(0); }
    if (a.time_order > 2) {
        HDs<R> F2[M], G2[M], F3[M], G3[M];
        LxwPhys<P>::flux_hd(q, qy, S_, a.pp, F2, G2);  // H2(qy, S)
        R sx[M], sy[M];
        for (int m = 0; m < M; m++) {
            const R fxx = d2(dx, sm.f[m][c - 2 * X], sm.f[m][c - X], sm.f[m][c], sm.f[m][c + X], sm.f[m][c + 2 * X]);
            const R gyy = d2(dy, sm.g[m][c - 2 * Y], sm.g[m][c - Y], sm.g[m][c], sm.g[m][c + Y], sm.g[m][c + 2 * Y]);
            R t1 = div_lp(R(0.5) * (sm.f[m][c + X + Y] - sm.f[m][c - X + Y]), dx);
            t1 -= div_lp(R(0.5) * (sm.f[m][c + X - Y] - sm.f[m][c - X - Y]), dx);
            t1 *= div_lp(R(0.5), dy);
            R t2 = div_lp(R(0.5) * (sm.g[m][c + X + Y] - sm.g[m][c - X + Y]), dx);
            t2 -= div_lp(R(0.5) * (sm.g[m][c + X - Y] - sm.g[m][c - X - Y]), dx);
            t2 *= div_lp(R(0.5), dy);
            sx[m] = fxx + t2;  // f_xx + g_xy
            sy[m] = t1 + gyy;  // f_xy + g_yy
        }
        LxwPhys<P>::flux_hd(q, sx, sy, a.pp, F3, G3);  // A1 sx (e1 of F), A2 sy (e2 of G)
        R qtt[M];
        for (int m = 0; m < M; m++) qtt[m] = F1[m].ab + G2[m].ab + F3[m].a + G3[m].b;
        HDs<R> F4[M], G4[M], F5[M], G5[M];
        LxwPhys<P>::flux_hd(q, qtt, S_, a.pp, F4, G4); // A q_tt (e1)
        LxwPhys<P>::flux_hd(q, S_, S_, a.pp, F5, G5);  // H(S, S) (e1e2)
        for (int m = 0; m < M; m++) {
            f_tt[m] = F4[m].a + F5[m].ab;
            g_tt[m] = G4[m].a + G5[m].ab;
        }
    }
    const long long lld = a.my + 6, lpl = (long long)(a.mx + 6) * lld;
    const long long o = (long long)ei * lld + ej;
    for (int m = 0; m < M; m++) {
        static_cast<R*>(a.F)[m * lpl + o] = sm.f[m][c] + R(0.5) * dt * (f_t[m] + div_lp(dt, R(3)) * f_tt[m]);
        static_cast<R*>(a.G)[m * lpl + o] = sm.g[m][c] + R(0.5) * dt * (g_t[m] + div_lp(dt, R(3)) * g_tt[m]);
    }
}

// ---- the FP64 form ---------------------------------------------------------
//
// The same fluxes with the derivatives of the flux written out.  In terms of
// the changes that a direction a makes to the primitive variables,
//     u_a = (a_1 - u a_0)/rho (v_a, w_a alike),
//     p_a = (g-1) (a_4 - u a_1 - v a_2 - w a_3 + |u|^2 a_0 / 2),  e_a = a_4 + p_a,
// the Jacobian products are
//     A1 a = (a_1, u a_1 + m_1 u_a + p_a, v a_1 + m_1 v_a, w a_1 + m_1 w_a, (E+p) u_a + u e_a),
// and the second derivatives, since those of m m'/rho and of |m|^2/(2 rho) are
// products of the velocity changes,
//     H1(a, b) = (0, 2 rho u_a u_b + p_ab, rho (u_a v_b + v_a u_b), rho (u_a w_b + w_a u_b),
//                 u_a e_b + u_b e_a + u p_ab - (E+p) (u_a b_0 + u_b a_0)/rho),
//     p_ab = -(g-1) rho (u_a u_b + v_a v_b + w_a w_b)
// (shallow water: p = h^2/2, p_a = h a_0, p_ab = a_0 b_0, no energy).  A cell
// takes 400 FP64 instructions, where five hyper-dual flux evaluations and the
// divisions of the differences by dx and dy took 1,250 and 224 registers.
// The limited step (mpp2d.hip), whose decisions follow the rounding of these
// fluxes, and the FP32 form keep the phases above.
//
// Records in LDS: q, then the fluxes that are not a momentum already
// (f_0 = q_1, g_0 = q_2, g_1 = f_2).
template <class P, int TI, int TJ>
struct LxwSmem64 {
    static constexpr int M = P::MEQN, HI = TI + 4, HJ = TJ + 4, NC = HI * HJ;
    static constexpr int NA = M == 5 ? 12 : 6;
    double a[NA][NC];
    // plane of q_k, f_k, g_k
    __host__ __device__ static constexpr int q(int k) { return k; }
    __host__ __device__ static constexpr int f(int k) { return k == 0 ? 1 : M + k - 1; }
    __host__ __device__ static constexpr int g(int k) { return k == 0 ? 2 : k == 1 ? f(2) : 2 * M + k - 3; }
};

// Returns whether a cell has a nonzero third momentum.
template <class P, int TI, int TJ>
__host__ __device__ __forceinline__ bool lxw64_load(int tid, int e0i, int e0j, const LxwArgs& a,
                                                    LxwSmem64<P, TI, TJ>& sm)
{
    using S = LxwSmem64<P, TI, TJ>;
    constexpr int M = S::M;
    bool nz3 = false;
    LxwCells<P, TI, TJ> cells;
    cells.load(tid, e0i, e0j, a);
#pragma unroll
    for (int k = 0; k < cells.K; k++) {
        if (!cells.ok[k]) continue;
        const int c = tid + k * cells.NT;
        const double* const q = cells.q[k];
        const double ir = rcp_d(q[0]);
        const double u = q[1] * ir, v = q[2] * ir;
        for (int m = 0; m < M; m++) sm.a[S::q(m)][c] = q[m];
        sm.a[S::f(2)][c] = q[1] * v;
        if constexpr (M == 5) {
            const double w = q[3] * ir;
            const double p = (a.pp.gamma - 1.0) * (q[4] - 0.5 * (q[1] * u + q[2] * v + q[3] * w));
            nz3 = nz3 || q[3] != 0.0;
            sm.a[S::f(1)][c] = fma(q[1], u, p);
            sm.a[S::f(3)][c] = q[1] * w;
            sm.a[S::f(4)][c] = u * (q[4] + p);
            sm.a[S::g(2)][c] = fma(q[2], v, p);
            sm.a[S::g(3)][c] = q[2] * w;
            sm.a[S::g(4)][c] = v * (q[4] + p);
        } else {
            const double p = 0.5 * q[0] * q[0];
            sm.a[S::f(1)][c] = fma(q[1], u, p);
            sm.a[S::g(2)][c] = fma(q[2], v, p);
        }
    }
    return nz3;
}

// A state and what its derivatives need.
template <class P>
struct LxwBase {
    double rho, ir, u, v, w, m1, m2, ep, hu, gm1;
};

// A direction: its components and the changes of the primitive variables.
template <class P, bool SKIP3>
struct LxwDir {
    static constexpr int M = P::MEQN;
    double a[M], du, dv, dw, dp, e;

    __host__ __device__ __forceinline__ void set(const LxwBase<P>& b)
    {
        du = fma(-b.u, a[0], a[1]) * b.ir;
        dv = fma(-b.v, a[0], a[2]) * b.ir;
        dw = 0.0;
        if constexpr (M == 5) {
            double t = fma(b.hu, a[0], fma(-b.u, a[1], fma(-b.v, a[2], a[4])));
            if (!SKIP3) {
                dw = fma(-b.w, a[0], a[3]) * b.ir;
                t = fma(-b.w, a[3], t);
            }
            dp = b.gm1 * t;
            e = a[4] + dp;
        } else {
            dp = b.rho * a[0];
            e = 0.0;
        }
    }
    // r += s A1 a and r += s A2 a (s = 1 or -1)
    __host__ __device__ __forceinline__ void a1(const LxwBase<P>& b, double r[M]) const
    {
        r[0] += a[1];
        r[1] += fma(b.u, a[1], fma(b.m1, du, dp));
        r[2] += fma(b.v, a[1], b.m1 * dv);
        if constexpr (M == 5) {
            if (!SKIP3) r[3] += fma(b.w, a[1], b.m1 * dw);
            r[4] += fma(b.ep, du, b.u * e);
        }
    }
    __host__ __device__ __forceinline__ void a2(const LxwBase<P>& b, double r[M]) const
    {
        r[0] += a[2];
        r[1] += fma(b.u, a[2], b.m2 * du);
        r[2] += fma(b.v, a[2], fma(b.m2, dv, dp));
        if constexpr (M == 5) {
            if (!SKIP3) r[3] += fma(b.w, a[2], b.m2 * dw);
            r[4] += fma(b.ep, dv, b.v * e);
        }
    }
};

// r += H1(x, y) (DIM 0) or H2(x, y) (DIM 1).
template <class P, bool SKIP3, int DIM>
__host__ __device__ __forceinline__ void lxw64_h(const LxwBase<P>& b, const LxwDir<P, SKIP3>& x,
                                                 const LxwDir<P, SKIP3>& y, double r[P::MEQN])
{
    constexpr int M = P::MEQN;
    const double guu = b.rho * (x.du * y.du), gvv = b.rho * (x.dv * y.dv);
    double p2;
    if constexpr (M == 5) {
        double g = guu + gvv;
        if (!SKIP3) g = fma(b.rho, x.dw * y.dw, g);
        p2 = -(b.gm1 * g);
    } else {
        p2 = x.a[0] * y.a[0];
    }
    const double guv = b.rho * fma(x.du, y.dv, x.dv * y.du);
    const double xn = DIM ? x.dv : x.du, yn = DIM ? y.dv : y.du;
    r[DIM ? 2 : 1] += fma(2.0, DIM ? gvv : guu, p2);
    r[DIM ? 1 : 2] += guv;
    if constexpr (M == 5) {
        if (!SKIP3) r[3] = fma(b.rho, fma(xn, y.dw, x.dw * yn), r[3]);
        const double d2 = fma(xn, y.a[0], yn * x.a[0]) * b.ir;
        r[4] += fma(xn, y.e, fma(yn, x.e, fma(DIM ? b.v : b.u, p2, -(b.ep * d2))));
    }
}

// One output cell per thread.
template <class P, int TI, int TJ, bool SKIP3>
__host__ __device__ __forceinline__ void lxw64_cell(int tid, int e0i, int e0j, const LxwArgs& a,
                                                    const LxwSmem64<P, TI, TJ>& sm)
{
    using S = LxwSmem64<P, TI, TJ>;
    using D = LxwDir<P, SKIP3>;
    constexpr int M = P::MEQN;
    const int ci = tid / TJ, cj = tid - ci * TJ;
    const int ei = e0i + ci, ej = e0j + cj;  // extended index, gi = ei - 3
    if (ci >= TI || ei >= a.mx + 6 || ej >= a.my + 6) return;
    const int c = (ci + 2) * S::HJ + (cj + 2);
    constexpr int X = S::HJ, Y = 1;
    const double rx = a.idx, ry = a.idy;
    const double x1 = (2.0 / 3.0) * rx, x2 = (1.0 / 12.0) * rx, y1 = (2.0 / 3.0) * ry, y2 = (1.0 / 12.0) * ry;
    auto live = [](int m) { return !(SKIP3 && M == 5 && m == 3); };
    // Diff1 along x or y of plane k
    auto dx1 = [&](int k) { return fma(x1, sm.a[k][c + X] - sm.a[k][c - X], x2 * (sm.a[k][c - 2 * X] - sm.a[k][c + 2 * X])); };
    auto dy1 = [&](int k) { return fma(y1, sm.a[k][c + Y] - sm.a[k][c - Y], y2 * (sm.a[k][c - 2 * Y] - sm.a[k][c + 2 * Y])); };
    LxwBase<P> b;
    b.rho = sm.a[0][c];
    b.ir = rcp_d(b.rho);
    b.m1 = sm.a[1][c];
    b.m2 = sm.a[2][c];
    b.u = b.m1 * b.ir;
    b.v = b.m2 * b.ir;
    b.w = 0.0;
    b.gm1 = a.pp.gamma - 1.0;
    b.hu = b.ep = 0.0;
    if constexpr (M == 5) {
        b.hu = fma(b.u, b.u, b.v * b.v);
        if (!SKIP3) {
            b.w = sm.a[3][c] * b.ir;
            b.hu = fma(b.w, b.w, b.hu);
        }
        b.hu *= 0.5;
        const double e = sm.a[4][c];
        b.ep = fma(b.gm1, fma(-b.hu, b.rho, e), e);
    }
    D s, d;
    double qtt[M];
    for (int m = 0; m < M; m++) {
        qtt[m] = 0.0;
        s.a[m] = live(m) ? dx1(S::f(m)) + dy1(S::g(m)) : 0.0;
    }
    s.set(b);
    double ft[M], gt[M];  // minus the first time derivatives
    for (int m = 0; m < M; m++) ft[m] = gt[m] = 0.0;
    s.a1(b, ft);
    s.a2(b, gt);
    double f2[M], g2[M];
    for (int m = 0; m < M; m++) f2[m] = g2[m] = 0.0;
    if (a.time_order > 2) {
        for (int m = 0; m < M; m++) d.a[m] = live(m) ? dx1(S::q(m)) : 0.0;
        d.set(b);
        lxw64_h<P, SKIP3, 0>(b, d, s, qtt);
        for (int m = 0; m < M; m++) d.a[m] = live(m) ? dy1(S::q(m)) : 0.0;
        d.set(b);
        lxw64_h<P, SKIP3, 1>(b, d, s, qtt);
        const double xx = rx * rx, yy = ry * ry, xy = 0.25 * (rx * ry);
        // Diff2 and the 4-point cross derivative
        auto dd = [&](int k, int o, double h) {
            const double n = sm.a[k][c + o] + sm.a[k][c - o], f = sm.a[k][c + 2 * o] + sm.a[k][c - 2 * o];
            return h * fma(4.0 / 3.0, n, fma(-1.0 / 12.0, f, -2.5 * sm.a[k][c]));
        };
        auto cross = [&](int k) {
            return (sm.a[k][c + X + Y] - sm.a[k][c - X + Y]) - (sm.a[k][c + X - Y] - sm.a[k][c - X - Y]);
        };
        for (int m = 0; m < M; m++) d.a[m] = live(m) ? fma(xy, cross(S::g(m)), dd(S::f(m), X, xx)) : 0.0;
        d.set(b);
        d.a1(b, qtt);
        for (int m = 0; m < M; m++) d.a[m] = live(m) ? fma(xy, cross(S::f(m)), dd(S::g(m), Y, yy)) : 0.0;
        d.set(b);
        d.a2(b, qtt);
        for (int m = 0; m < M; m++) d.a[m] = qtt[m];
        d.set(b);
        d.a1(b, f2);
        d.a2(b, g2);
        lxw64_h<P, SKIP3, 0>(b, s, s, f2);
        lxw64_h<P, SKIP3, 1>(b, s, s, g2);
    }
    const long long lld = a.my + 6, lpl = (long long)(a.mx + 6) * lld;
    const long long o = (long long)ei * lld + ej;
    const double dt = lxw_dt(a), h = 0.5 * dt, h2 = dt * (1.0 / 3.0);
    for (int m = 0; m < M; m++) {
        (static_cast<double*>(a.F) + m * lpl)[o] = live(m) ? fma(h, fma(h2, f2[m], -ft[m]), sm.a[S::f(m)][c]) : 0.0;
        (static_cast<double*>(a.G) + m * lpl)[o] = live(m) ? fma(h, fma(h2, g2[m], -gt[m]), sm.a[S::g(m)][c]) : 0.0;
    }
}

} // namespace finess
