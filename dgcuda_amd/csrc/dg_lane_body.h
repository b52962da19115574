// One Euler element per lane, p <= 3: the fused stage body of the lane
// kernels (single solve and batch), with the state in the vector layout.
//
// What bounds it: a wavefront's loads at small sizes, the state's bytes at
// large ones.  With mode-major rows the kernel issued 126 (p = 1) and 252
// (p = 2) vector loads of 4 bytes per lane and wavefront and waited on them
// for half of its wavefronts' time.  Here a lane moves one mode of its
// element's four variables per access (FP32 one 16-byte access, FP64 two),
// the geometry comes in packed records, the neighbours' modes are requested
// ahead of the arithmetic that covers them, and the neighbour's table rows
// are read from LDS instead of selected: 19.5-20.5 and 34-36 loads by stage,
// 889-1,100 and 2,067-2,339 vector instructions (counters, the step's dt and
// wave speeds included) instead of 1,163 and 2,608.  The sums of a face are
// pinned before the next begins (LANE_KEEP); moved down by the compiler they
// kept every face's values live (FP32 p = 2 168 registers and spills, pinned
// 128; FP64 p = 2 512, pinned 250).
// Per stage of a step, mode-major -> this layout: FP32 p = 1 at 524,288
// triangles 40.2 -> 24.1 us (111 MB, 4.6 TB/s), p = 2 71.6 -> 46.1 (187 MB,
// 4.1 TB/s; by kernel trace) and at 32,768 17.0 -> 9.9; FP64 p = 2 at 131,072
// 55.2 -> 27.2, at 32,768 24.1 -> 14.3.
//
// A face is evaluated in the element's own orientation (point j of the face
// against point p - j of the neighbour's), so only the neighbour's face
// number selects table entries at run time.  The normal-flux form is the
// matrix-core kernels': the side's sign is folded into the wave speed and
// the scale, so the two elements of a side get bit-identical point fluxes
// with opposite signs.
#pragma once
#include "dg_kernels.h"

namespace dgmi {

// keeps the scheduler from merging the faces (their loads and tables would
// all be live at once)
#ifndef LANE_FENCE  // a host build defines both empty
#define LANE_FENCE() __builtin_amdgcn_sched_barrier(0)
#define LANE_KEEP(x) asm volatile("" : "+v"(x))
#endif

// 16-byte pieces of an element's mode (V, W values), and a geometry record
template <typename R>
struct LaneV;
template <>
struct LaneV<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    typedef V G;
    static constexpr int W = 4;
    __device__ __forceinline__ static int word(float x) { return __float_as_int(x); }
};
template <>
struct LaneV<double> {
    typedef double V __attribute__((ext_vector_type(2)));
    typedef double G __attribute__((ext_vector_type(4)));
    static constexpr int W = 2;
    __device__ __forceinline__ static int word(double x) { return (int)x; }
};

// piece `row` (uniform) of element e: a scalar row base and a 32-bit byte
// offset per lane (e < 2^28 elements of 16 bytes)
template <typename R>
__device__ __forceinline__ const DG_GLOBAL typename LaneV<R>::V* lane_at(const R* x, int row, int Kp, int e) {
    const char DG_GLOBAL* b = (const char DG_GLOBAL*)(const DG_GLOBAL R*)x + (size_t)row * Kp * 16;
    return (const DG_GLOBAL typename LaneV<R>::V*)(b + (unsigned)e * 16u);
}
template <typename R>
__device__ __forceinline__ DG_GLOBAL typename LaneV<R>::V* lane_at(R* x, int row, int Kp, int e) {
    char DG_GLOBAL* b = (char DG_GLOBAL*)(DG_GLOBAL R*)x + (size_t)row * Kp * 16;
    return (DG_GLOBAL typename LaneV<R>::V*)(b + (unsigned)e * 16u);
}

// NT: the single-use streams (the RK operands and the outputs) carry the
// non-temporal hint.  FP64 always: p = 2 at 524,288 triangles 93.9 -> 83.5 us
// per stage, 32,768 15.1 -> 14.5.  FP32 when the solve's arrays exceed the
// 256 MB memory-side cache (StageArgs::stream): p = 2 at 1,048,352 triangles
// 84.2 -> 77.3 us; below, the next stage finds them there and the hint costs
// (p = 1 at 500,000 22.7 -> 24.8 us, p = 2 at 524,288 40.0 -> 43.0 us).  A
// template argument: the compiler merges the two forms of a branch and drops
// the hint.
template <bool NT, typename V>
__device__ __forceinline__ V lane_get(const DG_GLOBAL V* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    return *p;
}
template <bool NT, typename V>
__device__ __forceinline__ void lane_put(V x, DG_GLOBAL V* p) {
    if constexpr (NT)
        __builtin_nontemporal_store(x, p);
    else
        *p = x;
}

// the RK operands of element e that stage KIND reads from memory
template <int NP, int KIND, bool NT, typename R, typename V, int NG>
__device__ __forceinline__ void lane_rk_load(const StageArgs<R>& a, int e, V (&cv)[NP][NG], V (&av)[NP][NG]) {
    using RK = RkNeeds<KIND>;
#pragma unroll
    for (int m = 0; m < NP; m++)
#pragma unroll
        for (int g = 0; g < NG; g++) {
            if constexpr (RK::LOAD_C) cv[m][g] = lane_get<NT>(lane_at(a.c, m * NG + g, a.Kp, e));
            if constexpr (RK::LOAD_ACC) av[m][g] = lane_get<NT>(lane_at((const R*)a.acc, m * NG + g, a.Kp, e));
        }
}

template <int NP, int KIND, bool NT, typename R, typename V, int NG>
__device__ __forceinline__ void lane_rk_store(const StageArgs<R>& a, int e, const V (&o)[NP][NG],
                                              const V (&w)[NP][NG]) {
#pragma unroll
    for (int m = 0; m < NP; m++)
#pragma unroll
        for (int g = 0; g < NG; g++) {
            if constexpr (KIND == ST_RK4_2) lane_put<NT>(w[m][g], lane_at(a.acc, m * NG + g, a.Kp, e));
            lane_put<NT>(o[m][g], lane_at(a.out, m * NG + g, a.Kp, e));
        }
}

// all modes of element e of a state array in the vector layout
template <int NP, typename R>
__device__ __forceinline__ void lane_load(const R* __restrict__ x, int Kp, int e, R (&o)[4][NP]) {
    using V = typename LaneV<R>::V;
    constexpr int W = LaneV<R>::W, NG = 4 / W;
#pragma unroll
    for (int m = 0; m < NP; m++)
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const V q = *lane_at(x, m * NG + g, Kp, e);
#pragma unroll
            for (int i = 0; i < W; i++) o[g * W + i][m] = q[i];
        }
}

// all modes of caller's element o of an FP64 array in the reference layout
template <int NP, typename R>
__device__ __forceinline__ void lane_load_ref(const double* __restrict__ x, int K, int o, R (&u)[4][NP]) {
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
        for (int m = 0; m < NP; m++) u[v][m] = (R)*ref_at(x, v * NP + m, K, o);
}

// Neighbour-side trace table of order P in LDS: row (face, own point j)
// holds phi_m at the neighbour's point NQ1-1-j, the modes of a row
// contiguous (16-byte reads).  The neighbour's face differs from lane to lane; reading the
// row it names replaces two selects per entry.
template <int P>
struct LaneTab {
    static constexpr int NP = n_modes(P), NQ1 = P + 1;
    static constexpr int ROW = (NP + 3) / 4 * 4;          // values per (face, point)
    static constexpr int SIZE = 3 * NQ1 * ROW;
    template <typename R>
    __device__ __forceinline__ static void fill(R* t, int i0, int stride) {
        const TabP<R, P>& T = tab<R, P>();
        for (int i = i0; i < SIZE; i += stride) {
            const int f = i / (NQ1 * ROW), j = i / ROW % NQ1, m = i % ROW;
            t[i] = m < NP ? T.S[f][m][NQ1 - 1 - j] : R(0);
        }
    }
};

// Processes element e (clamped for loads when past the mesh, no stores
// then) of RK stage KIND; returns its cell wave speed after the last stage
// of a step, else 0, or -1 if `gate` (asked once the element's own loads are
// requested; it also makes `ltab` ready) finds the stage inactive.  stage_dt
// gives the stage's dt where it is used.  BND: the variant for meshes with boundary sides;
// without it the face loop carries no branch.
template <int P, int KIND, typename R, bool BND, bool NT, typename GATE, typename DT>
__device__ __forceinline__ double lane_process(const StageArgs<R>& a, int e, const R* ltab, const GATE& gate,
                                               const DT& stage_dt) {
    using L = LaneV<R>;
    using V = typename L::V;
    using G4 = typename L::G;
    using RK = RkNeeds<KIND>;
    constexpr int N = 4, NP = n_modes(P), NQ = n_quad_vol(P), NQ1 = P + 1, W = L::W, NG = N / W;
    constexpr bool LAST = (KIND == ST_RK4_4 || KIND == ST_RK2_2);
    const TabP<R, P>& T = tab<R, P>();
    const bool valid = e < a.K;
    const int ee = valid ? e : a.K - 1;
    const int Kp = a.Kp;
    constexpr bool REF = KIND == ST_RHS_REF;
    // (element e of the kernel's order: from the stage's input in the vector
    // layout, or from the caller's array)
    const auto load = [&](int x, R (&o)[N][NP]) {
        if constexpr (REF)
            lane_load_ref<NP, R>(a.ref_u, a.K, ref_elem(a, x), o);
        else
            lane_load<NP, R>(a.u, Kp, x, o);
    };

    G4 rec[3];
#pragma unroll
    for (int f = 0; f < 3; f++) rec[f] = ((const DG_GLOBAL G4*)a.lface)[(size_t)f * Kp + ee];
    R u[N][NP];
    load(ee, u);
    const G4 me = ((const DG_GLOBAL G4*)a.lmetric)[ee];
    const R ij = gp(a.geo_e)[4 * (size_t)Kp + ee];
    DG_LOADS_FIRST();
    if (!gate()) return -1.0;

    int wd[3], nb[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        wd[f] = L::word(rec[f][3]);
        nb[f] = wd[f] & NB_ELEM_MASK;
        if constexpr (BND)
            if (wd[f] < 0) nb[f] = ee;  // boundary side: the ghost replaces what is read
    }
    // neighbours' modes: the first face's ahead of the volume integral, then
    // one face ahead of its use
    constexpr bool AHEAD = sizeof(R) == 4 ? P <= 2 : P <= 1;
    R nu[AHEAD ? 2 : 1][N][NP];
    if constexpr (AHEAD) load(nb[0], nu[0]);

    R tot[N][NP];
#pragma unroll
    for (int v = 0; v < N; v++)
#pragma unroll
        for (int m = 0; m < NP; m++) tot[v][m] = R(0);

    // ---- volume: fluxes contracted with the inverse map, then with the
    // weighted basis gradients ----
    {
        const R xr = me[0], yr = me[1], xs = me[2], ys = me[3];
#pragma unroll 2
        for (int q = 0; q < NQ; q++) {
            R U[N];
#pragma unroll
            for (int v = 0; v < N; v++) U[v] = R(0);
#pragma unroll
            for (int m = 0; m < NP; m++)
#pragma unroll
                for (int v = 0; v < N; v++) U[v] += u[v][m] * T.B[m][q];
            R fr[N], fs[N];
            metric_flux<R>(a.phys, U, xr, yr, xs, ys, fr, fs);
#pragma unroll
            for (int m = 0; m < NP; m++) {
                const R gx = T.Gx[m][q], gy = T.Gy[m][q];
#pragma unroll
                for (int v = 0; v < N; v++) tot[v][m] += fr[v] * gx + fs[v] * gy;
            }
        }
    }

    // ---- the three faces ----
    V cv[NP][NG], av[NP][NG];  // RK operands read from memory
#pragma unroll
    for (int f = 0; f < 3; f++) {
        // the sums so far are formed here, not moved down to their last use
#pragma unroll
        for (int v = 0; v < N; v++)
#pragma unroll
            for (int m = 0; m < NP; m++) LANE_KEEP(tot[v][m]);
        LANE_FENCE();
        if constexpr (AHEAD) {
            if (f < 2) load(nb[f + 1], nu[(f + 1) & 1]);
        } else {
            load(nb[f], nu[0]);
        }
        if (f == 2) {
            // the stage update's operands, under the last face's arithmetic
            // and before any store (the output may be the base state itself)
            lane_rk_load<NP, KIND, NT>(a, ee, cv, av);
        }
        const R (&un)[N][NP] = nu[AHEAD ? f & 1 : 0];
        // (a boundary word's bits 28..29 hold its kind: 1..3)
        int fn = (wd[f] >> 28) & 3;
        if constexpr (BND) fn = wd[f] < 0 ? 0 : fn;
        const R* row = ltab + fn * (NQ1 * LaneTab<P>::ROW);
        const bool left = (wd[f] >> 30) & 1;
        const R nx = rec[f][0], ny = rec[f][1];
        const R cf = left ? R(-0.25) * rec[f][2] : R(0.25) * rec[f][2];
#pragma unroll
        for (int j = 0; j < NQ1; j++) {
            R Uo[N], Un[N];
#pragma unroll
            for (int v = 0; v < N; v++) {
                Uo[v] = R(0);
                Un[v] = R(0);
            }
#pragma unroll
            for (int m = 0; m < NP; m++) {
                const R so = T.S[f][m][j], sn = row[j * LaneTab<P>::ROW + m];
#pragma unroll
                for (int v = 0; v < N; v++) {
                    Uo[v] += u[v][m] * so;
                    Un[v] += un[v][m] * sn;
                }
            }
            if constexpr (BND)
                if (wd[f] < 0) boundary_ghost<N, NQ1, R>(a.bnd, wd[f], j, Uo, Un);
            R Fo[N], Fb[N], so, sb;
            normal_flux_speed<R>(a.phys, Uo, nx, ny, Fo, so);
            normal_flux_speed<R>(a.phys, Un, nx, ny, Fb, sb);
            const R lm = fmax(so, sb);
            const R lms = left ? lm : -lm;
            const R cw = cf * T.W1[j];
#pragma unroll
            for (int v = 0; v < N; v++) {
                const R g = cw * fma(lms, Uo[v] - Un[v], Fo[v] + Fb[v]);
#pragma unroll
                for (int m = 0; m < NP; m++) {
                    tot[v][m] += g * T.S[f][m][j];
                    if constexpr (sizeof(R) == 8 && P >= 2) LANE_KEEP(tot[v][m]);
                }
            }
        }
    }

    // ---- inverse mass (M = J*I; 1/J precomputed in FP64) and the RK stage update ----
    if constexpr (REF) {
        const R cj = ij * (R)a.ref_dt;
        if (valid) {
            const int o = ref_elem(a, e);
#pragma unroll
            for (int v = 0; v < N; v++)
#pragma unroll
                for (int m = 0; m < NP; m++) *ref_at(a.ref_k, v * NP + m, a.K, o) = (double)(cj * tot[v][m]);
        }
        return 0.0;
    }
    const R cj = ij * stage_dt();
    double lam = 0.0;
    V o[NP][NG], w[NP][NG];
#pragma unroll
    for (int m = 0; m < NP; m++)
#pragma unroll
        for (int g = 0; g < NG; g++) {
#pragma unroll
            for (int i = 0; i < W; i++) {
                const int v = g * W + i;
                R c = R(0), aa = R(0), t = R(0);
                if constexpr (RK::C_FROM_INPUT) c = u[v][m];
                if constexpr (RK::ACC_FROM_INPUT) aa = u[v][m];
                if constexpr (RK::LOAD_C) c = cv[m][g][i];
                if constexpr (RK::LOAD_ACC) aa = av[m][g][i];
                o[m][g][i] = rk_update<KIND, R>(c, aa, cj * tot[v][m], &t);
                w[m][g][i] = t;
            }
        }
    if (valid) lane_rk_store<NP, KIND, NT>(a, ee, o, w);
    if constexpr (LAST) {
        double U[4];
        const double b0 = tab<double, P>().B[0][0];
#pragma unroll
        for (int v = 0; v < N; v++) U[v] = (double)o[0][v / W][v % W] * b0;
        lam = valid ? cell_speed<N>(a.phys, U) : 0.0;
    }
    return lam;
}

}  // namespace dgmi
