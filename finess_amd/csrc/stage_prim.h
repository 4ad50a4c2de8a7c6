// stage_prim.h -- one tile of the fused FP64 stage on primitive records
// (prim2d.h), for the plain stage kernel and the batched one.
//
// A workgroup of 256 threads owns a TI x TJ tile of cells.  The records of the
// tile and its 3-cell cross-shaped halo go to LDS, then come the faces:
//
//   two passes  (TI+1) TJ and TI (TJ+1) up to 256 faces: every thread takes an
//               x face, then a y face.  15 x 16 cells have 511 faces, the
//               fewest per cell (2.13), and 32 KB of LDS leave room for four
//               workgroups per CU: the form for grids that fill the chip.
//   one pass    up to 128 faces of each direction: the first 128 threads take
//               the x faces, the others the y faces.  7 x 16 cells have 247
//               faces (2.2 per cell), but a workgroup lives half as long and
//               there are twice as many: the form for small grids, where the
//               length of one workgroup is the length of the launch.
//
// The stage is bound by FP64 issue (85% of the cycles at 1024^2), so loads and
// index arithmetic are kept short: cells of the halo's corners are not
// visited, and the maxima of the wave speeds are reduced by one wave per
// direction from LDS instead of by every wave.
#pragma once
#include "prim2d.h"
#include "stage2d_body.h"

namespace finess {

constexpr int PRIM_NT = 256;
template <class P, int TI, int TJ, bool TWO, bool LXW = false>
struct PrimSmem {
    static constexpr int HJ = TJ + 6, NC = (TI + 6) * HJ;
    static constexpr int NFX = (TI + 1) * TJ, NFY = TI * (TJ + 1), NT1 = TWO ? PRIM_NT : PRIM_NT / 2;
    static_assert(NFX <= NT1 && NFY <= NT1, "one face per thread and pass");
    struct Late {  // what the update reads besides the x fluxes
        double fy[P::MEQN][NFY];
        double speed[2][NT1];
    };
    // two passes: the y fluxes and the speeds take the records' place once
    // every face has been computed
    struct Records {
        double cv[P::NV][NC];
    };
    union Both {
        Records r;
        Late l;
    };
    struct Apart {
        Records r;
        Late l;
    };
    std::conditional_t<TWO, Both, Apart> u;
    // Lax-Wendroff: the time-integrated fluxes that the faces read, F along
    // the x stencils and G along the y stencils; in two passes the x fluxes
    // take F's place
    static constexpr int NF = (TI + 6) * TJ, NG = TI * (TJ + 6);
    struct Flux {
        double fx[P::MEQN][NFX];
    };
    union FluxBoth {
        double fx[P::MEQN][NFX];
        double F[P::MEQN][NF];
    };
    struct FluxApart {
        double fx[P::MEQN][NFX];
        double F[P::MEQN][NF];
    };
    std::conditional_t<!LXW, Flux, std::conditional_t<TWO, FluxBoth, FluxApart>> x;
    double G[LXW ? P::MEQN : 1][LXW ? NG : 1];
};

// Records of the tile's cells and of its halo without the corners: first the
// six halo rows of TJ cells, then the TI rows of TJ + 6.  Returns whether a
// cell has a nonzero third momentum (5-field systems).
template <class P, int TI, int TJ, int NC>
__host__ __device__ __forceinline__ bool prim_load(int t, int i0, int j0, const StageArgs& a, double (*cv)[NC])
{
    constexpr int M = P::MEQN, HJ = TJ + 6, NH = 6 * TJ, N = NH + TI * HJ, K = (N + PRIM_NT - 1) / PRIM_NT;
    // A tile whose halo lies inside the grid (most of them) reads its cells
    // directly, by 32-bit offsets from the halo's first cell; the others go
    // through the boundary map.
    const bool inner = !a.src_ghosts && i0 >= 3 && j0 >= 3 && i0 + TI + 3 <= a.mx && j0 + TJ + 3 <= a.my && a.my < (1 << 24);
    bool nz3 = false;
    double q[K][M];
    int at[K];
    bool ok[K];
#pragma unroll
    for (int k = 0; k < K; k++) {  // every load is issued before a record is formed
        const int c = t + k * PRIM_NT, d = c - NH;
        const int hr = c / TJ, rr = d / HJ;
        const int ci = c < NH ? (hr < 3 ? hr : hr + TI) : rr + 3;
        const int cj = c < NH ? c - hr * TJ + 3 : d - rr * HJ;
        at[k] = ci * HJ + cj;
        ok[k] = c < N;
        if (inner) {
            if (ok[k]) {
                const unsigned off = (unsigned)(ci * a.my + cj) * 8u;
                const double* s = a.src + ((long long)(i0 - 3) * a.my + (j0 - 3));
                for (int m = 0; m < M; m++)
                    q[k][m] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(s + m * a.plane) + off);
            }
        } else {
            const int gi = i0 + ci - 3, gj = j0 + cj - 3;
            ok[k] = ok[k] && gi <= a.mx + 2 && gj <= a.my + 2;
            if (ok[k]) load_state<P>(a, gi, gj, q[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (!ok[k]) continue;
        if constexpr (M == 5) nz3 = nz3 || q[k][3] != 0.0;
        double rec[P::NV];
        P::cell_record(q[k], a.pp, rec);
        for (int v = 0; v < P::NV; v++) cv[v][at[k]] = rec[v];
    }
    return nz3;
}

// The time-integrated fluxes of the tile's stencils, F on rows i0-3..i0+TI+2 of
// the tile's columns and G on columns j0-3..j0+TJ+2 of its rows, once each
// into LDS (read from memory at every stencil point they took 40 million L2
// requests of 128 bytes per 2048^2 stage, and the stage twice as long).
// Returns whether one of the third momentum is nonzero.
template <class P, int TI, int TJ, int NF, int NG>
__host__ __device__ __forceinline__ bool prim_load_fluxes(int t, int i0, int j0, const StageArgs& a, double (*F)[NF],
                                                          double (*G)[NG])
{
    constexpr int M = P::MEQN, HJ = TJ + 6;
    constexpr int KF = (NF + PRIM_NT - 1) / PRIM_NT, KG = (NG + PRIM_NT - 1) / PRIM_NT;
    const long long lld = a.my + 6, lpl = (long long)(a.mx + 6) * lld;
    const double* const gF = static_cast<const double*>(a.lxw_F);
    const double* const gG = static_cast<const double*>(a.lxw_G);
    double v[KF + KG][M];
    bool ok[KF + KG], nz3 = false;
#pragma unroll
    for (int k = 0; k < KF + KG; k++) {
        const int c = t + (k < KF ? k : k - KF) * PRIM_NT;
        if (k < KF) {
            const int r = c / TJ, col = c - r * TJ;
            ok[k] = c < NF && i0 + r <= a.mx + 5 && j0 + col < a.my;
            if (ok[k])
                for (int m = 0; m < M; m++) v[k][m] = (gF + m * lpl)[(i0 + r) * lld + (j0 + col + 3)];
        } else {
            const int r = c / HJ, col = c - r * HJ;
            ok[k] = c < NG && i0 + r < a.mx && j0 + col <= a.my + 5;
            if (ok[k])
                for (int m = 0; m < M; m++) v[k][m] = (gG + m * lpl)[(i0 + r + 3) * lld + (j0 + col)];
        }
    }
#pragma unroll
    for (int k = 0; k < KF + KG; k++) {
        if (!ok[k]) continue;
        const int c = t + (k < KF ? k : k - KF) * PRIM_NT;
        if constexpr (M == 5) nz3 = nz3 || v[k][3] != 0.0;
        for (int m = 0; m < M; m++) {
            if (k < KF) F[m][c] = v[k][m];
            else G[m][c] = v[k][m];
        }
    }
    return nz3;
}

// Face number f of direction DIR: its flux into fh; returns its wave speed
// when GetCFL counts it (lib/2d/GetCFL.cpp:54-58), else zero.
template <class P, int WK, bool LXW, int TI, int TJ, int DIR, int NC>
__host__ __device__ __forceinline__ double prim_face(int f, int i0, int j0, const StageArgs& a,
                                                     const double (*cv)[NC], const double* flux, bool skip3,
                                                     double fh[P::MEQN])
{
    const FaceGeom g = face_geom<TI, TJ>(f, DIR, i0, j0, a);
    if (!g.valid) return 0.0;
    // (flux: prim_load_fluxes' planes of the direction)
    const int lpl = DIR ? TI * (TJ + 6) : (TI + 6) * TJ, lst = DIR ? 1 : TJ;
    const int lb = DIR ? g.fi * (TJ + 6) + g.fj : f;
    const double* galpha = a.galpha ? a.galpha + DIR : nullptr;
    double alpha;
    // (a tile-uniform choice between two forms of the face code)
    if (P::MEQN == 5 && skip3)
        alpha = P::template face<WK, LXW, true, NC>(cv, g.base, g.stride, DIR, flux, lb, lst, lpl, a.pp,
                                                    a.eps, a.power, a.alpha_scaling, fh, galpha);
    else
        alpha = P::template face<WK, LXW, false, NC>(cv, g.base, g.stride, DIR, flux, lb, lst, lpl, a.pp,
                                                     a.eps, a.power, a.alpha_scaling, fh, galpha);
    const int gi = i0 + g.fi, gj = j0 + g.fj;
    if (DIR == 0 && a.smax_faces_x) a.smax_faces_x[(long long)gi * a.my + gj] = alpha;
    if (DIR == 1 && a.smax_faces_y) a.smax_faces_y[(long long)gi * (a.my + 1) + gj] = alpha;
    return g.count ? alpha : 0.0;
}

// Fields M0..M1-1 of the cell of thread tc: L = -(F(i+1) - F(i))/dx -
// (G(j+1) - G(j))/dy (lib/2d/ConstructL.cpp:388-399) and the stage update.
// The update's operands are read in `load`, before the barrier that the
// fluxes wait for.
template <class P, int TI, int TJ, int M0, int M1>
struct PrimUpdate {
    static constexpr int KM = M1 - M0;
    bool on;
    int ci, cj, gi, gj;
    long long idx;
    double pa[KM], pb[KM];

    __host__ __device__ __forceinline__ void load(int tc, int i0, int j0, const StageArgs& a)
    {
        ci = tc / TJ;
        cj = tc - ci * TJ;
        gi = i0 + ci;
        gj = j0 + cj;
        on = ci < TI && gi < a.mx && gj < a.my;
        idx = (long long)gi * a.my + gj;
        for (int k = 0; k < KM; k++) pa[k] = pb[k] = 0.0;
        if (!on || !a.out) return;
        for (int k = 0; k < KM; k++) pa[k] = (a.qa + (M0 + k) * a.plane)[idx];
        if (a.use_b)
            for (int k = 0; k < KM; k++) pb[k] = (a.qb + (M0 + k) * a.plane)[idx];
    }

    __host__ __device__ __forceinline__ void store(const StageArgs& a, double bdt, const double (*fx)[(TI + 1) * TJ],
                                                   const double (*fy)[TI * (TJ + 1)]) const
    {
        if (!on) return;
        constexpr int M = P::MEQN;
        double psi[M];
        if (a.src_kind != SRC_OFF) {
            double qs[M];
            load_state<P>(a, gi, gj, qs);
            source_psi<M>(a.src_kind, a.src_coef, qs, a.aux ? a.aux + idx : nullptr, a.plane, psi);
        }
        const int x = ci * TJ + cj, y = ci * (TJ + 1) + cj;
        double L[KM];
        for (int k = 0; k < KM; k++) {
            const int m = M0 + k;
            L[k] = -(fx[m][x + TJ] - fx[m][x]) * a.idx;
            L[k] = L[k] - (fy[m][y + 1] - fy[m][y]) * a.idy;
            if (a.src_kind != SRC_OFF) L[k] = psi[m] + L[k];  // Lstar = psi + tmp (lib/2d/ConstructL.cpp:378-386)
        }
        if (a.Lout)
            for (int k = 0; k < KM; k++) (a.Lout + (M0 + k) * a.plane)[idx] = L[k];
        if (!a.out) return;
        for (int k = 0; k < KM; k++) {
            double v = a.a1 * pa[k];
            if (a.use_b) v = v + a.a2 * pb[k];
            (a.out + (M0 + k) * a.plane)[idx] = v + bdt * L[k];
        }
    }
};

// The maximum of n speeds in LDS, by one wave, folded into *word (bit patterns
// of non-negative doubles).  A NaN speed must not vanish: it counts as +inf.
template <int N>
__device__ __forceinline__ void prim_fold_speed(const double* s, int lane, unsigned long long* word)
{
    double v = 0.0, bad = 0.0;
    for (int k = 0; k < N / 64; k++) {
        const double x = s[lane + 64 * k];
        v = fmax(v, x);
        bad = fma(0.0, x, bad);
    }
    if (bad != bad) v = __builtin_inf();
    v = wave_max64(v);
    if (lane == 0) atomicMax(word, (unsigned long long)__double_as_longlong(v));
}

// The tile at (i0, j0).  smax: the words that take the maxima of the x and
// (swy words further) y wave speeds, null for none.
template <class P, int WK, bool LXW, int TI, int TJ, bool TWO>
__device__ __forceinline__ void prim_tile(int t, int i0, int j0, const StageArgs& a,
                                          PrimSmem<P, TI, TJ, TWO, LXW>& sm, unsigned long long* smax, int swy)
{
    using S = PrimSmem<P, TI, TJ, TWO, LXW>;
    constexpr int M = P::MEQN, NT1 = S::NT1, MH = (M + 1) / 2;
    // a tile whose cells (and, for Lax-Wendroff, fluxes) have no rho w skips
    // that field's reconstructions
    bool nz = false;
    // beta dt is read before the tile's cells, not where the update needs it: the
    // registers then fit without spills (450^2 61.2 -> 58.8 us per step, 128^2
    // 22.1 -> 21.7, 2048^2 652 -> 645)
    const double bdt = stage_bdt(a);
    const double *lF = nullptr, *lG = nullptr;
    if constexpr (LXW) {
        nz = prim_load_fluxes<P, TI, TJ, S::NF, S::NG>(t, i0, j0, a, sm.x.F, sm.G);
        lF = &sm.x.F[0][0];
        lG = &sm.G[0][0];
    }
    nz = prim_load<P, TI, TJ, S::NC>(t, i0, j0, a, sm.u.r.cv) || nz;
    bool skip3 = false;
    if constexpr (M == 5) skip3 = !__syncthreads_or(nz);
    else __syncthreads();
    double fh[M];
    if constexpr (TWO) {
        const double ax = prim_face<P, WK, LXW, TI, TJ, 0, S::NC>(t, i0, j0, a, sm.u.r.cv, lF, skip3, fh);
        if constexpr (LXW) __syncthreads();  // the last read of F
        if (t < S::NFX)
            for (int m = 0; m < M; m++) sm.x.fx[m][t] = fh[m];
        const double ay = prim_face<P, WK, LXW, TI, TJ, 1, S::NC>(t, i0, j0, a, sm.u.r.cv, lG, skip3, fh);
        PrimUpdate<P, TI, TJ, 0, M> u;
        u.load(t, i0, j0, a);
        __syncthreads();  // the last read of the records
        if (t < S::NFY)
            for (int m = 0; m < M; m++) sm.u.l.fy[m][t] = fh[m];
        sm.u.l.speed[0][t] = ax;
        sm.u.l.speed[1][t] = ay;
        __syncthreads();
        u.store(a, bdt, sm.x.fx, sm.u.l.fy);
    } else {
        const int th = t & (NT1 - 1);
        const bool second = __builtin_amdgcn_readfirstlane(t) >= NT1;
        PrimUpdate<P, TI, TJ, 0, MH> u0;
        PrimUpdate<P, TI, TJ, MH, M> u1;
        if (second) {
            sm.u.l.speed[1][th] = prim_face<P, WK, LXW, TI, TJ, 1, S::NC>(th, i0, j0, a, sm.u.r.cv, lG, skip3, fh);
            if (th < S::NFY)
                for (int m = 0; m < M; m++) sm.u.l.fy[m][th] = fh[m];
            u1.load(th, i0, j0, a);
        } else {
            sm.u.l.speed[0][th] = prim_face<P, WK, LXW, TI, TJ, 0, S::NC>(th, i0, j0, a, sm.u.r.cv, lF, skip3, fh);
            if (th < S::NFX)
                for (int m = 0; m < M; m++) sm.x.fx[m][th] = fh[m];
            u0.load(th, i0, j0, a);
        }
        __syncthreads();
        if (second) u1.store(a, bdt, sm.x.fx, sm.u.l.fy);
        else u0.store(a, bdt, sm.x.fx, sm.u.l.fy);
    }
    // two of the four waves fold a direction each
    if (smax && t >= PRIM_NT - 128) {
        const int dir = __builtin_amdgcn_readfirstlane(t) >= PRIM_NT - 64;
        prim_fold_speed<NT1>(sm.u.l.speed[dir], t & 63, smax + (dir ? swy : 0));
    }
}

} // namespace finess
