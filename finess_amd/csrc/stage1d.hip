// stage1d.hip -- the 1D path: lib/1d/ConstructL.cpp:16-224 with the
// advection callbacks of apps/1d/advection/lib (f = aux(1) q, identity
// eigenvectors, s1 = min(a_l, (a_l+a_r)/2), s2 = max(a_r, (a_l+a_r)/2)),
// UpdateSoln (lib/1d/UpdateSoln.cpp:17-54) and the periodic halo
// (apps/1d/advection/smooth_example/SetBndValues.cpp:6-63).
//
// 1D grids are small (the advection case has 200 cells): up to
// small1d_cells<WK>() cells a stage is one workgroup (faces, barrier, cells),
// and a time step's stages run in one launch of that workgroup; beyond it
// each stage is two plain launches, one thread per face, then one thread
// per cell.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "kernels.h"
#include "stage1d_body.h"
#include "step_control_body.h"

namespace finess {

template <int WK>
__global__ __launch_bounds__(256) void k_faces1d(Stage1DArgs a)
{
    if (halted1d(a)) return;
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    double alpha = 0.0;
    if (f <= a.mx) alpha = face1d_any<WK>(f, a);
    if (a.smax_slot) {
        if (alpha != alpha) alpha = __builtin_inf();
        // GetCFL (lib/1d/GetCFL.cpp:30-33) reads faces 1..mx (1-based), i.e. f < mx
        if (f < a.mx)
            atomicMax(a.smax_slot + blockIdx.x % CFL_SPREAD, (unsigned long long)__double_as_longlong(alpha));
    }
}

__global__ __launch_bounds__(256) void k_update1d(Stage1DArgs a)
{
    if (halted1d(a)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.mx) update1d(i, a);
}

// GlobalWaveSpd (lib/1d/GlobalWaveSpd.cpp): max |aux(1)| over the interior
// (the advection SetWaveSpd with both sides equal), one workgroup.
__global__ __launch_bounds__(256) void k_global_speed1d(Stage1DArgs a)
{
    if (halted1d(a)) return;
    double v = 0.0;
    for (int i = threadIdx.x; i < a.mx; i += 256) {
        const double s = fabs(a.aux[idx1d(a, i)]);
        v = s != s ? __builtin_inf() : (v > s ? v : s);
    }
    v = wave_max64(v);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int k = 1; k < 4; k++) m = red[k] > m ? red[k] : m;
        *a.galpha = m;
    }
}

// Grids up to small1d_cells<WK>() cells run the whole stage in one
// workgroup: the faces, a workgroup barrier (which orders the face fluxes
// written to global memory before they are read), then the cells.  One
// launch instead of two, but one CU: the limits are the measured crossovers
// with the two-launch path, which takes 31-34 us per SSP-RK3 step (with the
// controller) at any size up to 8192 cells.  WENO5: 21.5 against 30.6 us
// at 1024 cells, 34.6 against 31.0 at 2048; WENO11: 31.6 against 33.2 at
// 512, 44.2 against 33.6 at 1024.  Orders 7 and 9 lie between.
template <int WK>
constexpr int small1d_cells()
{
#ifdef FINESS_SMALL1D
    return FINESS_SMALL1D;
#else
    return WK == WENO_JS11                                       ? 512
           : (WK == WENO_JS9 || WK == WENO_Z9 || WK == WENO_FD9) ? 768
           : (WK == WENO_JS7 || WK == WENO_Z7 || WK == WENO_FD7) ? 1024
                                                                 : 1536;
#endif
}

constexpr int SMALL1D_NT = 512;  // 2 waves per SIMD: the wide orders fit without spilling

#ifndef FINESS_PAIR1D
#define FINESS_PAIR1D 1
#endif

// One stage on a single workgroup: faces, barrier, cells, the CFL maximum.
template <int WK>
__device__ __forceinline__ void stage1d_small_body(const Stage1DArgs& a, double* red)
{
    double amax = 0.0;
    bool paired = false;
    if constexpr (WK < WENO_JS7) paired = FINESS_PAIR1D && 2 * (a.mx + 1) <= SMALL1D_NT;
    if (paired) {
        // a grid of at most SMALL1D_NT / 2 faces: two lanes per face, one
        // split part each, so that a face's two reconstructions run side by
        // side; the even lane adds them in face1d's order
        const int f = threadIdx.x >> 1, part = threadIdx.x & 1;
        if (f <= a.mx) {
            double alpha;
            const double w = face1d_part<WK < WENO_JS7 ? WK : WENO_JS5_P2>(f, a, part, alpha);
            // the partner lane's part (quad_perm [1,0,3,2]: both lanes of a
            // pair take this branch together)
            const long long wb = __double_as_longlong(w);
            const int lo = dpp_move<0xB1>((int)wb), hi = dpp_move<0xB1>((int)(wb >> 32));
            const double wo = __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
            if (!part) {
                a.fhat[f] = w + wo;
                if (a.smax_faces) a.smax_faces[f] = alpha;
                if (alpha != alpha) alpha = __builtin_inf();
                // GetCFL (lib/1d/GetCFL.cpp:30-33) reads faces 1..mx (1-based), i.e. f < mx
                if (f < a.mx) amax = alpha > amax ? alpha : amax;
            }
        }
    } else {
        for (int f = threadIdx.x; f <= a.mx; f += SMALL1D_NT) {
            double alpha = face1d_any<WK>(f, a);
            if (alpha != alpha) alpha = __builtin_inf();
            // GetCFL (lib/1d/GetCFL.cpp:30-33) reads faces 1..mx (1-based), i.e. f < mx
            if (f < a.mx) amax = alpha > amax ? alpha : amax;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < a.mx; i += SMALL1D_NT) update1d(i, a);
    if (!a.smax_slot) return;
    amax = wave_max64(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int k = 1; k < SMALL1D_NT / 64; k++) m = red[k] > m ? red[k] : m;
        atomicMax(a.smax_slot, (unsigned long long)__double_as_longlong(m));
    }
}

template <int WK>
__global__ __launch_bounds__(SMALL1D_NT) void k_stage1d_small(Stage1DArgs a)
{
    if (halted1d(a)) return;
    __shared__ double red[SMALL1D_NT / 64];
    stage1d_small_body<WK>(a, red);
}

// Every stage of one time step in one workgroup: the barrier after each stage
// orders its cell writes (and its reads of the shared face fluxes) before the
// next stage's faces.  One launch per step instead of one per stage.
template <int WK>
__global__ __launch_bounds__(SMALL1D_NT) void k_step1d_small(Stage1DStep s)
{
    if (halted1d(s.stage[0])) return;
    __shared__ double red[SMALL1D_NT / 64];
    for (int k = 0; k < s.n; k++) {
        stage1d_small_body<WK>(s.stage[k], red);
        __syncthreads();
    }
    // wave 0 runs the controller on the last stage's maxima; the barrier
    // above has ordered the stages' reads of dt before the block changes
    if (s.ctl && threadIdx.x < 64) step_control_wave(s.ctl, s.stage[s.n - 1].smax_slot, s.cp, threadIdx.x);
}

// A run of steps (Stage1DRun) of the wide orders.  Every thread takes the controller's decision
// from the block after the barrier that follows it: a step that raised the
// accepted count rotates the plane sets (an nv stop happens after its step
// is accepted, as on the host); a rejection is cleared here and retried.
//
// The run works in LDS (run1d_lds_bytes): the three plane sets, the face
// fluxes, the advection speeds, the CFL words and the controller block.  The stage code reaches
// them through the same pointers it takes for global memory (generic
// addresses), the state at entry and the block are read once, and the state
// at exit, the CFL words and the block are written back once: each stage
// then waits on LDS instead of on a round trip through L2 after every
// barrier.
#ifndef FINESS_RUN1D_LDS
#define FINESS_RUN1D_LDS 1
#endif
template <int WK>
__global__ __launch_bounds__(SMALL1D_NT) void k_run1d_small(Stage1DRun r)
{
    __shared__ double red[SMALL1D_NT / 64];
    int cur = r.cur;
#if FINESS_RUN1D_LDS
    extern __shared__ double lds1d[];
    __shared__ StepCtl lctl;
    __shared__ unsigned long long lsmax[2 * CFL_SPREAD];
    const int mx = r.base.mx;
    double* const buf[3] = {lds1d, lds1d + mx, lds1d + 2 * mx};
    double* const laux = lds1d + 4 * mx + 1;
    for (int i = threadIdx.x; i < mx; i += SMALL1D_NT) {
        buf[cur][i] = r.buf[cur][i];
        laux[i] = r.base.aux[i];
    }
    for (int k = threadIdx.x; k < 2 * CFL_SPREAD; k += SMALL1D_NT) lsmax[k] = r.smax_slot[k];
    if (threadIdx.x == 0) lctl = *r.ctl;
    __syncthreads();
    StepCtl* const ctl = &lctl;
    unsigned long long* const smax = lsmax;
    Stage1DArgs base = r.base;
    base.fhat = lds1d + 3 * mx;
    base.aux = laux;
    base.dtp = &lctl.dt;
    base.halt = &lctl.halt;
#else
    double* const* const buf = r.buf;
    StepCtl* const ctl = r.ctl;
    unsigned long long* const smax = r.smax_slot;
    const Stage1DArgs base = r.base;
#endif
    for (int att = 0; att < r.max_attempts; att++) {
        if (__hip_atomic_load(&ctl->halt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != HALT_NONE) break;
        const long long acc0 = __hip_atomic_load(&ctl->acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int k = 0; k < r.n; k++) {
            const SspStage g = ssp_stage(r.n, k);
            Stage1DArgs a = base;
            a.src = buf[(cur + g.src) % 3];
            a.qa = buf[(cur + g.qa) % 3];
            a.qb = g.qb >= 0 ? buf[(cur + g.qb) % 3] : nullptr;
            a.use_b = g.qb >= 0 && g.a2 != 0.0;
            a.out = buf[(cur + g.out) % 3];
            a.a1 = g.a1;
            a.a2 = g.a2;
            a.beta = g.beta;
            a.smax_slot = k == r.n - 1 ? smax : nullptr;
            stage1d_small_body<WK>(a, red);
            __syncthreads();
        }
        if (threadIdx.x < 64) step_control_wave(ctl, smax, r.cp, threadIdx.x);
        __syncthreads();
        const unsigned long long h = __hip_atomic_load(&ctl->halt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__hip_atomic_load(&ctl->acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != acc0)
            cur = (cur + ssp_result(r.n)) % 3;
        if (h == HALT_REJECT) {
            __syncthreads();  // every thread has read the halt word before it is cleared
            if (threadIdx.x == 0) __hip_atomic_store(&ctl->halt, (unsigned long long)HALT_NONE, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            continue;
        }
        if (h != HALT_NONE) break;
    }
#if FINESS_RUN1D_LDS
    for (int i = threadIdx.x; i < mx; i += SMALL1D_NT) r.buf[cur][i] = buf[cur][i];
    for (int k = threadIdx.x; k < 2 * CFL_SPREAD; k += SMALL1D_NT) r.smax_slot[k] = lsmax[k];
    if (threadIdx.x == 0) {
        lctl.buf = cur;
        *r.ctl = lctl;
    }
#else
    if (threadIdx.x == 0) r.ctl->buf = cur;
#endif
}

// The run of steps of the fifth-order kinds on one workgroup, for grids up to
// RUN1D_CELLS: one barrier per stage and none for the controller.
//
// A pair of lanes takes a face, one split part each; a wave's 32 faces are
// those around 31 cells, whose fluxes then come from the next pair by lane
// moves, so no flux passes through LDS.  A cell's state stays in its pair's
// registers through the step; LDS holds two copies of the stage's source with
// its ghosts, written in turn.  The speeds of advection do not change during
// the run, so the CFL maximum is taken once and every thread makes the
// controller's decision for itself.  NCH: chunks of 31 cells per wave.
//
// 200 cells take 2.1 us per step; the kernel above took 6.9 (two barriers, flux
// and state through generic pointers and the boundary map per stencil cell,
// the controller behind a third barrier): a chain of latencies, on one CU.
// 400 cells 3.1 (8.6), 1000 5.8 (13.3), 2000 9.6 and 2700 11.7 (32 with
// two launches per stage), which RUN1D_CELLS takes as far as the 64 KB of LDS
// that a launch gets without an attribute.
//
// More than 16 x 31 cells take all 16 waves, whose last chunks may hold no
// cells and are then left out: four waves on each SIMD share the chunks evenly
// (1000 cells in nine waves of four chunks: 7.4 us; 520 cells 3.9, now 3.4).
//
// The kinds with pow, which are bound by its instructions on the one CU, stop
// at RUN1D_CELLS_POW, the limit of the step kernels: 1000 cells take 34.7 us
// (41.7 in the kernel above), 1536 48.6 (65.6).  Beyond, two launches per stage
// take 31 to 38; the run took 60 at 1600 cells and 89 at 2700 (before the even
// sharing of the chunks, which gave a fifth at most).
constexpr int RUN1D_CELLS = 2700, RUN1D_CELLS_POW = 1536, RUN1D_WAVES = 16, RUN1D_CHUNK = 31;

// lane i takes lane i + 1's value (the last keeps its own)
__device__ __forceinline__ double wave_next(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_move<0x130>((int)b), hi = dpp_move<0x130>((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// the other lane of the pair
__device__ __forceinline__ double pair_other(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_move<0xB1>((int)b), hi = dpp_move<0xB1>((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Cell i's value into the copy X (cell i at X[i + 3]) and into the ghosts
// that the boundary rules (bc_map) take from it.
__device__ __forceinline__ void run1d_store(double* X, int i, double v, int n, int lo, int hi)
{
    X[i + 3] = v;
    if (i >= 3 && i < n - 3) return;
    if (lo == BC_PERIODIC) {
        if (i >= n - 3) X[i - n + 3] = v;
    } else if (lo == BC_REFLECT) {
        if (i < 3) X[2 - i] = v;
    } else if (i == 0) {
        X[0] = X[1] = X[2] = v;
    }
    if (hi == BC_PERIODIC) {
        if (i < 3) X[n + i + 3] = v;
    } else if (hi == BC_REFLECT) {
        if (i >= n - 3) X[2 * n + 2 - i] = v;
    } else if (i == n - 1) {
        X[n + 3] = X[n + 4] = X[n + 5] = v;
    }
}

template <int WK, int NCH>
__global__ __launch_bounds__(RUN1D_WAVES * 64) void k_run1d_wave(Stage1DRun r)
{
    extern __shared__ double run1d_lds[];
    __shared__ double red[RUN1D_WAVES];
    const Stage1DArgs& a = r.base;
    const int n = a.mx, ld = n + 6, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int part = lane & 1;
    // the wave's chunks that hold cells; the first FULL always do (launch_run1d)
    constexpr int FULL = NCH <= 2 ? NCH - 1 : NCH - 2;
    const int first = RUN1D_CHUNK * __builtin_amdgcn_readfirstlane(wave);
    const int chunks = first < n ? (n - first + nw * RUN1D_CHUNK - 1) / (nw * RUN1D_CHUNK) : 0;
    double* const X = run1d_lds;             // the two copies, ld apart
    double* const haux = run1d_lds + 2 * ld; // half the advection speeds
    for (int i = (int)threadIdx.x - 3; i < n + 3; i += blockDim.x) {
        const long long k = idx1d(a, i);
        X[i + 3] = r.buf[r.cur][k];
        haux[i + 3] = 0.5 * a.aux[k];
    }
    double hla[NCH], qn[NCH], x[NCH], sx = 0.0;
    int face[NCH];
    bool cell[NCH];
    for (int c = 0; c < NCH; c++) {
        const int f = (c * nw + wave) * RUN1D_CHUNK + (lane >> 1);
        cell[c] = (lane >> 1) < RUN1D_CHUNK && f < n;
        face[c] = f <= n ? f : n;  // pairs past the end repeat the last face
        double alpha;
        hla[c] = face1d_speed(face[c], a, alpha) * (part ? -0.5 : 0.5);
        if (alpha != alpha) alpha = __builtin_inf();
        // GetCFL (lib/1d/GetCFL.cpp:30-33) reads faces 1..mx (1-based), i.e. f < mx
        if (face[c] < n) sx = alpha > sx ? alpha : sx;
    }
    sx = wave_max64(sx);
    if (lane == 0) red[wave] = sx;
    __syncthreads();
    for (int w = 0; w < nw; w++) sx = red[w] > sx ? red[w] : sx;
    for (int c = 0; c < NCH; c++) qn[c] = x[c] = X[face[c] + 3];
    const double idx = 1.0 / a.dx;
    StepCtl h = *r.ctl;
    int s = 0;  // the copy that holds the step's start
    for (int att = 0; att < r.max_attempts && h.halt == HALT_NONE; att++) {
        const double dt = h.dt;
        for (int k = 0; k < r.n; k++) {
            const SspStage g = ssp_stage(r.n, k);
            const double bdt = g.beta * dt;
            const double* const S = X + s * ld;
            s ^= 1;
            double* const D = X + s * ld;
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                if (NCH > 1 && c >= FULL && c >= chunks) continue;
                // part 0: cells f-3..f+1, part 1: f+2..f-2
                const int i0 = part ? face[c] + 5 : face[c], st = part ? -1 : 1;
                double v[5];
                for (int m = 0; m < 5; m++) v[m] = S[i0 + m * st] * (haux[i0 + m * st] + hla[c]);
                const double w = weno5_fp64<WK>(v, a.eps, a.power);
                const double F = w + pair_other(w), Fn = wave_next(wave_next(F));
                double L = -(Fn - F) * idx;
                if (a.src_kind != SRC_OFF) L = source1d(a, x[c], L);
                // (the operands are the source or the step's start)
                const double qa = g.qa == g.src ? x[c] : qn[c], qb = g.qb == g.src ? x[c] : qn[c];
                x[c] = combine1d(g.a1, qa, g.qb >= 0 && g.a2 != 0.0, g.a2, qb, bdt, L);
                if (cell[c] && !part) run1d_store(D, face[c], x[c], n, a.bc_lo, a.bc_hi);
            }
            __syncthreads();
        }
        const long long acc = h.acc;
        step_control_decide(h, r.cp, sx, 0.0);
        if (h.acc != acc) {
            for (int c = 0; c < NCH; c++) qn[c] = x[c];
        } else {
            // rejected (retried with the controller's dt) or failed: the
            // step's start again
            for (int c = 0; c < NCH; c++) {
                x[c] = qn[c];
                if (cell[c] && !part) run1d_store(X + s * ld, face[c], x[c], n, a.bc_lo, a.bc_hi);
            }
            __syncthreads();
            if (h.halt == HALT_REJECT) h.halt = HALT_NONE;
        }
    }
    for (int c = 0; c < NCH; c++)
        if (cell[c] && !part) r.buf[r.cur][face[c]] = qn[c];
    if (threadIdx.x == 0) {
        h.buf = r.cur;
        *r.ctl = h;
    }
}

template <int WK, int NCH>
static void launch_run1d_wave(const Stage1DRun& r, hipStream_t st)
{
    const int nw = NCH > 1 ? RUN1D_WAVES : (r.base.mx + RUN1D_CHUNK - 1) / RUN1D_CHUNK;
    hipLaunchKernelGGL((k_run1d_wave<WK, NCH>), dim3(1), dim3(nw * 64), 3 * (r.base.mx + 6) * sizeof(double), st, r);
}

// Dynamic LDS of the run kernel: three plane sets of mx cells, mx + 1 face
// fluxes and mx advection speeds (61 KB at the largest single-workgroup
// grid, 1536 cells).
static size_t run1d_lds_bytes(int mx)
{
    return FINESS_RUN1D_LDS ? (size_t)(5 * mx + 1) * sizeof(double) : 0;
}

template <int WK>
static int launch_wk(const Stage1DArgs& a, hipStream_t st)
{
    if (a.galpha) hipLaunchKernelGGL(k_global_speed1d, dim3(1), dim3(256), 0, st, a);
    if (a.mx <= small1d_cells<WK>()) {
        hipLaunchKernelGGL(k_stage1d_small<WK>, dim3(1), dim3(SMALL1D_NT), 0, st, a);
        return hipGetLastError() == hipSuccess ? 0 : -4;
    }
    hipLaunchKernelGGL(k_faces1d<WK>, dim3((a.mx + 1 + 255) / 256), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_update1d, dim3((a.mx + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// GlobalWaveSpd in 1D reads aux only, which no stage changes: one launch
// serves all stages of a step.
template <int WK>
static int launch_step_wk(const Stage1DStep& s, hipStream_t st)
{
    if (s.stage[0].mx > small1d_cells<WK>()) {
        for (int k = 0; k < s.n; k++)
            if (const int rc = launch_wk<WK>(s.stage[k], st)) return rc;
        return s.ctl ? launch_step_control(s.ctl, s.stage[s.n - 1].smax_slot, s.cp, st) : 0;
    }
    if (s.stage[0].galpha) hipLaunchKernelGGL(k_global_speed1d, dim3(1), dim3(256), 0, st, s.stage[0]);
    hipLaunchKernelGGL(k_step1d_small<WK>, dim3(1), dim3(SMALL1D_NT), 0, st, s);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// Time-integrated fluxes of the 1D Lax-Wendroff step on the extended cells.
__global__ __launch_bounds__(256) void k_lxw_flux1d(Stage1DArgs a, double dt, int time_order, double* F)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < a.mx + 6) F[e] = integrated_f1d(e - 3, a, dt, time_order);
}

int launch_lxw_flux1d(const Stage1DArgs& a, double dt, int time_order, double* F, hipStream_t st)
{
    hipLaunchKernelGGL(k_lxw_flux1d, dim3((a.mx + 6 + 255) / 256), dim3(256), 0, st, a, dt, time_order, F);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <class F>
static int with_kind(int wk, F f)
{
    switch (wk) {
    case WENO_JS5_P2: return f(std::integral_constant<int, WENO_JS5_P2>());
    case WENO_JS5_POW: return f(std::integral_constant<int, WENO_JS5_POW>());
    case WENO_Z5: return f(std::integral_constant<int, WENO_Z5>());
    case WENO_Z5_P2: return f(std::integral_constant<int, WENO_Z5_P2>());
    case WENO_FD5: return f(std::integral_constant<int, WENO_FD5>());
    case WENO_JS7: return f(std::integral_constant<int, WENO_JS7>());
    case WENO_JS9: return f(std::integral_constant<int, WENO_JS9>());
    case WENO_JS11: return f(std::integral_constant<int, WENO_JS11>());
    case WENO_Z7: return f(std::integral_constant<int, WENO_Z7>());
    case WENO_Z9: return f(std::integral_constant<int, WENO_Z9>());
    case WENO_FD7: return f(std::integral_constant<int, WENO_FD7>());
    case WENO_FD9: return f(std::integral_constant<int, WENO_FD9>());
    case WENO_O1: return f(std::integral_constant<int, WENO_O1>());
    default: return -1;
    }
}

int launch_stage1d(int wk, const Stage1DArgs& a, hipStream_t st)
{
    return with_kind(wk, [&](auto k) { return launch_wk<decltype(k)::value>(a, st); });
}

int launch_run1d(int wk, const Stage1DRun& r, hipStream_t st)
{
    if (r.n < 1 || r.n > 3 || !run1d_fits(wk, r.base.mx)) return -1;
    if (r.base.galpha) hipLaunchKernelGGL(k_global_speed1d, dim3(1), dim3(256), 0, st, r.base);
    return with_kind(wk, [&](auto k) {
        constexpr int WK = decltype(k)::value;
        if constexpr (WK < WENO_JS7) {
            // chunks per wave: as many as 16 waves need
            const int ch = (r.base.mx + RUN1D_WAVES * RUN1D_CHUNK - 1) / (RUN1D_WAVES * RUN1D_CHUNK);
            if (ch <= 1) launch_run1d_wave<WK, 1>(r, st);
            else if (ch <= 2) launch_run1d_wave<WK, 2>(r, st);
            else if (ch <= 4) launch_run1d_wave<WK, 4>(r, st);
            else launch_run1d_wave<WK, 6>(r, st);
        } else {
            hipLaunchKernelGGL(k_run1d_small<WK>, dim3(1), dim3(SMALL1D_NT), run1d_lds_bytes(r.base.mx), st, r);
        }
        return hipGetLastError() == hipSuccess ? 0 : -4;
    });
}

bool run1d_fits(int wk, int mx)
{
    if (wk == WENO_JS5_POW || wk == WENO_Z5) return mx <= RUN1D_CELLS_POW;
    if (wk < WENO_JS7) return mx <= RUN1D_CELLS;
    // (and the run's LDS within the 64 KB a launch gets without an attribute)
    return run1d_lds_bytes(mx) + 2048 <= 65536 &&
           with_kind(wk, [&](auto k) { return mx <= small1d_cells<decltype(k)::value>() ? 1 : 0; }) == 1;
}

int launch_step1d(int wk, const Stage1DStep& s, hipStream_t st)
{
    if (s.n < 1 || s.n > 3) return -1;
    return with_kind(wk, [&](auto k) { return launch_step_wk<decltype(k)::value>(s, st); });
}

} // namespace finess
