// Fused element kernels on the vector ALUs: one lane per element.
//
// One launch per RK stage does what the reference does with four
// (eval_surface, eval_volume, eval_rhs, rk_tempstorage;
// src/2d/conservation/time_integrator.cu:274-307):
//   volume integral    (conserv_kernels.cu:766-811)
//   LLF surface terms  (conserv_kernels.cu:628-758) evaluated for the three
//                      faces of the element, each face flux computed in the
//                      side's canonical left->right orientation so both
//                      elements of a side obtain bit-identical fluxes
//                      (race-free, no atomics, no face buffers)
//   gather + M^-1      (time_integrator.cu:130-188, M = J*I)
//   RK stage update    (time_integrator.cu:194-218, 445-464)
//   CFL wave speeds    (euler.cu:252-278) of the new state on the last stage,
//                      reduced per workgroup with wavefront shuffles.
#include <algorithm>

#include "dg_lane_body.h"
#include "dg_valu_body.h"

namespace dgmi {

DGMI_TABLE_UPLOADER(upload_tables_kernels)

// BND: the variant for meshes with boundary sides (p <= VALU_BOUNDARY_MAX_P)
// REF: the right-hand side on the caller's arrays
// (advection p = 5 FP32 is held to the two wavefronts per SIMD it misses by
// one register: 320,000 triangles 935 -> 656 us a step; the others spill if held)
template <int N, int P, typename R, bool BND = false, bool REF = false>
__global__ void __launch_bounds__(128, (N == 1 && P == 5 && sizeof(R) == 4 ? 2 : 1)) k_stage_valu(StageArgs<R> a) {
    __shared__ double sh[8];
    if constexpr (REF) {
        const int t = tile_of_block(blockIdx.x, gridDim.x, a.xcd_remap);
        if (t < a.ntiles) valu_process<N, P, R, BND, true>(a, t * blockDim.x + threadIdx.x, ST_RHS);
        return;
    }
    const int kind = a.kind;
    const StageStep<R> step(a, kind);
    if (!step.active()) return;
    const int tile = tile_of_block(blockIdx.x, gridDim.x, a.xcd_remap);
    if (tile >= a.ntiles) return;
    const double lam =
        valu_process<N, P, R, BND, false>(a, tile * blockDim.x + threadIdx.x, kind, [&] { return step.dt(); });
    if (last_stage(kind)) {
        const double mx = block_max(lam, sh);
        if (threadIdx.x == 0) stage_commit(a, mx);
    }
}

// Euler, p <= 3: the lane body on the vector layout, one instance per stage
// kind (the RK operands' loads and the update are fixed at compile time)
// Wavefronts per SIMD the registers are held to: the most that fit without
// spills in the loops (FP32 p = 1, 2: 5 and 4; FP64 p = 1, 2: 2).  FP32 p = 2
// spills 3 registers in the first stage, 17-26 with boundary sides, and 16 on
// the caller's arrays.
template <int P, typename R>
constexpr int lane_minw() {
    if (sizeof(R) == 4) return P <= 1 ? 5 : P == 2 ? 4 : 2;
    return P <= 2 ? 2 : 1;
}
template <int P, int KIND, typename R, bool BND, bool NT>
__global__ void __launch_bounds__(128, (lane_minw<P, R>())) k_stage_lane(StageArgs<R> a) {
    __shared__ double sh[8];
    __shared__ __align__(16) R ltab[LaneTab<P>::SIZE];
    const int tile = tile_of_block(blockIdx.x, gridDim.x, a.xcd_remap);
    if (tile >= a.ntiles) return;
    const StageStep<R> step(a, KIND);
    const auto gate = [&] {
        LaneTab<P>::fill(ltab, threadIdx.x, blockDim.x);
        __syncthreads();
        return KIND == ST_RHS_REF || step.active();
    };
    const double lam = lane_process<P, KIND, R, BND, NT>(a, tile * blockDim.x + threadIdx.x, ltab, gate,
                                                         [&] { return step.dt(); });
    if (lam < 0.0) return;  // inactive: every lane of the launch
    if constexpr (last_stage(KIND)) {
        const double mx = block_max(lam, sh);
        if (threadIdx.x == 0) stage_commit(a, mx);
    }
}

// Packs the geometry of the vector layout (one thread per element).
template <typename R>
__global__ void __launch_bounds__(256) k_lane_pack(const R* __restrict__ geo_e, const R* __restrict__ geo_f,
                                                  const int* __restrict__ nbr, int Kp,
                                                  typename LaneV<R>::G* __restrict__ lface,
                                                  typename LaneV<R>::G* __restrict__ lmetric) {
    using G4 = typename LaneV<R>::G;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= Kp) return;
    const size_t kp = (size_t)Kp;
    for (int f = 0; f < 3; f++) {
        const int wd = nbr[f * kp + e];
        R wv;
        if constexpr (sizeof(R) == 4)
            wv = __int_as_float(wd);
        else
            wv = (R)wd;
        lface[f * kp + e] = G4{geo_f[3 * f * kp + e], geo_f[(3 * f + 1) * kp + e], geo_f[(3 * f + 2) * kp + e], wv};
    }
    lmetric[e] = G4{geo_e[e], geo_e[kp + e], geo_e[2 * kp + e], geo_e[3 * kp + e]};
}

template <typename R>
hipError_t launch_lane_pack(const R* geo_e, const R* geo_f, const int* nbr, int Kp, void* lface, void* lmetric,
                            hipStream_t st) {
    using G4 = typename LaneV<R>::G;
    hipLaunchKernelGGL((k_lane_pack<R>), dim3((Kp + 255) / 256), dim3(256), 0, st, geo_e, geo_f, nbr, Kp, (G4*)lface,
                       (G4*)lmetric);
    return hipGetLastError();
}
template hipError_t launch_lane_pack<float>(const float*, const float*, const int*, int, void*, void*, hipStream_t);
template hipError_t launch_lane_pack<double>(const double*, const double*, const int*, int, void*, void*, hipStream_t);

// Maximum cell wave speed of a state without stepping it (first step of a
// run, dg_cfl_dt): grid-stride over elements, workgroup max, one atomic max.
template <int N, typename R>
__global__ void __launch_bounds__(256) k_lambda(const R* u, StateIx ix, int K, double b0, PhysP ph, Ctrl* ctrl) {
    __shared__ double sh[8];
    double mx = 0.0;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < K; e += gridDim.x * blockDim.x) {
        double U[4];
#pragma unroll
        for (int v = 0; v < N; v++) U[v] = (double)u[ix.at(v, 0, e)] * b0;
        mx = fmax(mx, cell_speed<N>(ph, U));
    }
    mx = block_max(mx, sh);
    if (threadIdx.x == 0) lam_commit(mx, lam_slots(ctrl) + lam_side(ctrl)->current * LAM_SIDE);
}

__global__ void k_reset_lam(Ctrl* ctrl) {
    lam_clear(lam_slots(ctrl) + lam_side(ctrl)->current * LAM_SIDE);  // LAM_SLOTS threads
}

// host-chosen step: activate the stages with the given dt
__global__ void k_set_dt(Ctrl* ctrl, double dt, int advance) {
    const int side = lam_side(ctrl)->current;
    lam_clear(lam_slots(ctrl) + side * LAM_SIDE);  // LAM_SLOTS threads
    if (threadIdx.x == 0) {
        ctrl->dt = dt;
        ctrl->active = 1;
        lam_side(ctrl)->commit = side;
        if (advance) {
            ctrl->t += dt;
            ctrl->steps += 1;
        }
    }
}

// ---------------------------------------------------------------------------
// Initial conditions: c_i = sum_j w_j U0(x_j) phi_i(x_j) in FP64
// (conserv_kernels.cu:167-187, euler.cu:31-59), stored in the bulk precision.
// ---------------------------------------------------------------------------
template <int N, int P, typename R>
__global__ void __launch_bounds__(128) k_project_ic(R* c, StateIx ix, const double* V, int K, IcP ic) {
    constexpr int NP = n_modes(P), NQ = n_quad_vol(P);
    const int Kp = ix.Kp;
    const TabP<double, P>& T = tab<double, P>();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= K) return;
    const double v1x = V[e], v1y = V[Kp + e], v2x = V[2 * Kp + e], v2y = V[3 * Kp + e];
    const double v3x = V[4 * Kp + e], v3y = V[5 * Kp + e];
    double u0[NQ][N];
    for (int j = 0; j < NQ; j++) {
        const double r1 = T.R1[j], r2 = T.R2[j];
        const double x = r1 * v2x + r2 * v3x + (1 - r1 - r2) * v1x;
        const double y = r1 * v2y + r2 * v3y + (1 - r1 - r2) * v1y;
        double U[4];
        ic_point(ic, x, y, U);
        for (int n = 0; n < N; n++) u0[j][n] = U[n];
    }
    for (int i = 0; i < NP; i++) {
        double U[N];
        for (int n = 0; n < N; n++) U[n] = 0.;
        for (int j = 0; j < NQ; j++)
            for (int n = 0; n < N; n++) U[n] += T.W[j] * u0[j][n] * T.B[i][j];
        for (int n = 0; n < N; n++) c[ix.at(n, i, e)] = (R)U[n];
    }
    for (int i = NP; i < ix.slots(); i++)  // padding modes of the tile layouts
        for (int n = 0; n < N; n++) c[ix.at(n, i, e)] = R(0);
}

// ---------------------------------------------------------------------------
// FP64 audit partials per workgroup: mass of each variable, minimum cell-mean
// density and pressure, count of non-finite / non-positive cells.
// part[blk*8 + 0..3] mass, +4 min rho, +5 min p, +6 bad count.
// ---------------------------------------------------------------------------
template <int N, typename R>
__global__ void __launch_bounds__(256) k_audit(const R* c, StateIx ix, const double* Jd, int K, double b0,
                                              double gamma, double* part) {
    __shared__ double sm[256];
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double mass[4] = {0, 0, 0, 0}, rho = 1e300, pr = 1e300, bad = 0;
    if (e < K) {
        double U[4];
        const double J = Jd[e];
        for (int v = 0; v < N; v++) {
            double c0 = (double)c[ix.at(v, 0, e)];
            mass[v] = J * c0 * b0 * 0.5;
            U[v] = c0 * b0;
        }
        rho = U[0];
        bool ok = isfinite(U[0]);
        if (N == 4) {
            for (int v = 1; v < 4; v++) ok = ok && isfinite(U[v]);
            pr = (gamma - 1.) * (U[3] - (U[1] * U[1] + U[2] * U[2]) / 2. / U[0]);
            ok = ok && U[0] > 0 && pr > 0;
        }
        bad = ok ? 0 : 1;
    }
    // fixed-shape tree reduction: deterministic
    double vals[7] = {mass[0], mass[1], mass[2], mass[3], rho, pr, bad};
    for (int k = 0; k < 7; k++) {
        sm[threadIdx.x] = vals[k];
        __syncthreads();
        for (int s = blockDim.x / 2; s > 0; s >>= 1) {
            if (threadIdx.x < s) {
                double x = sm[threadIdx.x], y = sm[threadIdx.x + s];
                sm[threadIdx.x] = (k == 4 || k == 5) ? fmin(x, y) : x + y;
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) part[blockIdx.x * 8 + k] = sm[0];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int P, typename R, bool BND, bool NT>
static hipError_t launch_stage_lane(const StageArgs<R>& a, dim3 grid, hipStream_t st) {
    switch (a.kind) {
        case ST_RHS: hipLaunchKernelGGL((k_stage_lane<P, ST_RHS, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK4_1: hipLaunchKernelGGL((k_stage_lane<P, ST_RK4_1, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK4_2: hipLaunchKernelGGL((k_stage_lane<P, ST_RK4_2, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK4_3: hipLaunchKernelGGL((k_stage_lane<P, ST_RK4_3, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK4_4: hipLaunchKernelGGL((k_stage_lane<P, ST_RK4_4, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK2_1: hipLaunchKernelGGL((k_stage_lane<P, ST_RK2_1, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RK2_2: hipLaunchKernelGGL((k_stage_lane<P, ST_RK2_2, R, BND, NT>), grid, dim3(128), 0, st, a); break;
        case ST_RHS_REF:
            if constexpr (NT) {  // (its streams are the caller's arrays)
                hipLaunchKernelGGL((k_stage_lane<P, ST_RHS_REF, R, BND, NT>), grid, dim3(128), 0, st, a);
                break;
            } else {
                return hipErrorInvalidValue;
            }
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// advection at every order (boundary sides up to p = 3), Euler at p = 4, 5
template <int N, int P, typename R>
static hipError_t launch_stage_valu_np(const StageArgs<R>& a, dim3 grid, hipStream_t st) {
    if (a.kind == ST_RHS_REF) {
        if constexpr (ref_rhs_supported(N, P, 1)) {
            if constexpr (P <= VALU_BOUNDARY_MAX_P)
                if (a.bnd) {
                    hipLaunchKernelGGL((k_stage_valu<N, P, R, true, true>), grid, dim3(128), 0, st, a);
                    return hipGetLastError();
                }
            if (a.bnd) return hipErrorInvalidValue;  // refused on the host before this
            hipLaunchKernelGGL((k_stage_valu<N, P, R, false, true>), grid, dim3(128), 0, st, a);
            return hipGetLastError();
        } else {
            return hipErrorInvalidValue;
        }
    }
    if (a.bnd) {
        if constexpr (P <= VALU_BOUNDARY_MAX_P)
            hipLaunchKernelGGL((k_stage_valu<N, P, R, true>), grid, dim3(128), 0, st, a);
        else
            return hipErrorInvalidValue;  // refused on the host before this
    } else {
        hipLaunchKernelGGL((k_stage_valu<N, P, R>), grid, dim3(128), 0, st, a);
    }
    return hipGetLastError();
}

template <int P, typename R>
static hipError_t launch_euler(const StageArgs<R>& a, dim3 grid, hipStream_t st) {
    if constexpr (lane_vec(4, P)) {
        static_assert(P <= VALU_BOUNDARY_MAX_P, "the vector layout's kernels carry boundary sides");
        if constexpr (sizeof(R) == 4)
            if (!a.stream && a.kind != ST_RHS_REF)
                return a.bnd ? launch_stage_lane<P, R, true, false>(a, grid, st)
                             : launch_stage_lane<P, R, false, false>(a, grid, st);
        return a.bnd ? launch_stage_lane<P, R, true, true>(a, grid, st)
                     : launch_stage_lane<P, R, false, true>(a, grid, st);
    } else {
        return launch_stage_valu_np<4, P, R>(a, grid, st);
    }
}

template <typename R>
hipError_t launch_stage_valu(int N, int p, const StageArgs<R>& a, dim3 grid, hipStream_t st) {
    if (N == 1) {
        switch (p) {
            case 0: return launch_stage_valu_np<1, 0, R>(a, grid, st);
            case 1: return launch_stage_valu_np<1, 1, R>(a, grid, st);
            case 2: return launch_stage_valu_np<1, 2, R>(a, grid, st);
            case 3: return launch_stage_valu_np<1, 3, R>(a, grid, st);
            case 4: return launch_stage_valu_np<1, 4, R>(a, grid, st);
            case 5: return launch_stage_valu_np<1, 5, R>(a, grid, st);
        }
    } else if (N == 4) {
        switch (p) {
            case 0: return launch_euler<0, R>(a, grid, st);
            case 1: return launch_euler<1, R>(a, grid, st);
            case 2: return launch_euler<2, R>(a, grid, st);
            case 3: return launch_euler<3, R>(a, grid, st);
            case 4: return launch_euler<4, R>(a, grid, st);
            case 5: return launch_euler<5, R>(a, grid, st);
        }
    }
    return hipErrorInvalidValue;
}
template hipError_t launch_stage_valu<float>(int, int, const StageArgs<float>&, dim3, hipStream_t);
template hipError_t launch_stage_valu<double>(int, int, const StageArgs<double>&, dim3, hipStream_t);

template <typename R>
hipError_t launch_lambda(const R* u, const StateIx& ix, int K, double b0, const PhysP& ph, Ctrl* ctrl,
                         hipStream_t st) {
    hipLaunchKernelGGL(k_reset_lam, dim3(1), dim3(LAM_SLOTS), 0, st, ctrl);
    const dim3 grid(std::min((K + 255) / 256, 2048));
    if (ix.N == 1)
        hipLaunchKernelGGL((k_lambda<1, R>), grid, dim3(256), 0, st, u, ix, K, b0, ph, ctrl);
    else
        hipLaunchKernelGGL((k_lambda<4, R>), grid, dim3(256), 0, st, u, ix, K, b0, ph, ctrl);
    return hipGetLastError();
}
template hipError_t launch_lambda<float>(const float*, const StateIx&, int, double, const PhysP&, Ctrl*,
                                         hipStream_t);
template hipError_t launch_lambda<double>(const double*, const StateIx&, int, double, const PhysP&, Ctrl*,
                                          hipStream_t);

hipError_t launch_set_dt(Ctrl* ctrl, double dt, int advance, hipStream_t st) {
    hipLaunchKernelGGL(k_set_dt, dim3(1), dim3(LAM_SLOTS), 0, st, ctrl, dt, advance);
    return hipGetLastError();
}

template <int N, typename R>
static hipError_t launch_ic_np(int p, R* c, const StateIx& ix, const double* V, int K, const IcP& ic,
                               hipStream_t st) {
    dim3 grid((K + 127) / 128);
    switch (p) {
        case 0: hipLaunchKernelGGL((k_project_ic<N, 0, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        case 1: hipLaunchKernelGGL((k_project_ic<N, 1, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        case 2: hipLaunchKernelGGL((k_project_ic<N, 2, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        case 3: hipLaunchKernelGGL((k_project_ic<N, 3, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        case 4: hipLaunchKernelGGL((k_project_ic<N, 4, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        case 5: hipLaunchKernelGGL((k_project_ic<N, 5, R>), grid, dim3(128), 0, st, c, ix, V, K, ic); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename R>
hipError_t launch_project_ic(int p, R* c, const StateIx& ix, const double* V, int K, const IcP& ic, hipStream_t st) {
    if (ix.N == 1) return launch_ic_np<1, R>(p, c, ix, V, K, ic, st);
    return launch_ic_np<4, R>(p, c, ix, V, K, ic, st);
}
template hipError_t launch_project_ic<float>(int, float*, const StateIx&, const double*, int, const IcP&,
                                             hipStream_t);
template hipError_t launch_project_ic<double>(int, double*, const StateIx&, const double*, int, const IcP&,
                                              hipStream_t);

template <typename R>
hipError_t launch_audit(const R* c, const StateIx& ix, const double* Jd, int K, double b0, double gamma,
                        double* part, int nblocks, hipStream_t st) {
    if (ix.N == 1)
        hipLaunchKernelGGL((k_audit<1, R>), dim3(nblocks), dim3(256), 0, st, c, ix, Jd, K, b0, gamma, part);
    else
        hipLaunchKernelGGL((k_audit<4, R>), dim3(nblocks), dim3(256), 0, st, c, ix, Jd, K, b0, gamma, part);
    return hipGetLastError();
}
template hipError_t launch_audit<float>(const float*, const StateIx&, const double*, int, double, double, double*,
                                        int, hipStream_t);
template hipError_t launch_audit<double>(const double*, const StateIx&, const double*, int, double, double,
                                         double*, int, hipStream_t);

// ---------------------------------------------------------------------------
// State conversion on the device between the boundary's reference layout
// (FP64, c[var][mode][elem] in the caller's element order) and a state
// array of the bulk precision in layout `ix`.  perm[i] (Kp entries) is the
// caller's element of internal element i; padding elements carry element
// K-1's id.  One thread per (variable, internal element).
// ---------------------------------------------------------------------------
// The rows' pointers are arguments of their own, so that the loads of several
// modes are in flight (behind a struct they may be the output's, and each
// waits for the store before it: dg_rhs_device_noalloc through the scratch,
// Euler p = 5 FP32 at 800 triangles 105.7 -> 102.0 us).
template <typename R>
__global__ void __launch_bounds__(256) k_ref_to_state(const double* __restrict__ lo, const double* __restrict__ hi,
                                                     int split, R* __restrict__ dst, const int* __restrict__ perm,
                                                     StateIx ix, int K) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ix.N * ix.Kp) return;
    const int v = t / ix.Kp, i = t - v * ix.Kp;
    const size_t src = (size_t)perm[i];
    // eight at a time: the rows may lie in host memory, about 2 us away
    for (int m0 = 0; m0 < ix.NP; m0 += 8) {
        double x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int r = v * ix.NP + min(m0 + j, ix.NP - 1);
            x[j] = (r < split ? lo + (size_t)r * K : hi + (size_t)(r - split) * K)[src];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (m0 + j < ix.NP) dst[ix.at(v, m0 + j, i)] = (R)x[j];
    }
    // every slot of the layout is written: padding modes hold zeros
    for (int m = ix.NP; m < ix.slots(); m++) dst[ix.at(v, m, i)] = R(0);
}

template <typename R>
__global__ void __launch_bounds__(256) k_state_to_ref(const R* __restrict__ src, double* __restrict__ lo,
                                                     double* __restrict__ hi, int split, const int* __restrict__ perm,
                                                     StateIx ix, int K) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ix.N * K) return;
    const int v = t / K, i = t - v * K;
    const size_t dst = (size_t)perm[i];
#pragma unroll 4
    for (int m = 0; m < ix.NP; m++) {
        const int r = v * ix.NP + m;
        double* row = r < split ? lo + (size_t)r * K : hi + (size_t)(r - split) * K;
        row[dst] = (double)src[ix.at(v, m, i)];
    }
}

template <typename R>
hipError_t launch_ref_to_state(const RefRows& ref, R* dst, const int* perm, const StateIx& ix, int K, hipStream_t st) {
    const int n = ix.N * ix.Kp;
    hipLaunchKernelGGL((k_ref_to_state<R>), dim3((n + 255) / 256), dim3(256), 0, st, ref.lo, ref.hi, ref.split, dst,
                       perm, ix, K);
    return hipGetLastError();
}
template <typename R>
hipError_t launch_state_to_ref(const R* src, const RefRows& ref, const int* perm, const StateIx& ix, int K,
                               hipStream_t st) {
    const int n = ix.N * K;
    hipLaunchKernelGGL((k_state_to_ref<R>), dim3((n + 255) / 256), dim3(256), 0, st, src, ref.lo, ref.hi, ref.split,
                       perm, ix, K);
    return hipGetLastError();
}
template hipError_t launch_ref_to_state<float>(const RefRows&, float*, const int*, const StateIx&, int, hipStream_t);
template hipError_t launch_ref_to_state<double>(const RefRows&, double*, const int*, const StateIx&, int, hipStream_t);
template hipError_t launch_state_to_ref<float>(const float*, const RefRows&, const int*, const StateIx&, int,
                                               hipStream_t);
template hipError_t launch_state_to_ref<double>(const double*, const RefRows&, const int*, const StateIx&, int,
                                                hipStream_t);

// Fill the constant-memory tables of every order from the FP64 host tables.
template <typename R, int P>
static void fill_tab(TabP<R, P>& d) {
    Tables t = build_tables(P);
    constexpr int NP = TabP<R, P>::NP, NQ = TabP<R, P>::NQ, NQ1 = TabP<R, P>::NQ1;
    for (int m = 0; m < NP; m++) {
        for (int q = 0; q < NQ; q++) {
            d.B[m][q] = (R)t.basis[m * NQ + q];
            d.Gx[m][q] = (R)t.gx[m * NQ + q];
            d.Gy[m][q] = (R)t.gy[m * NQ + q];
        }
        for (int f = 0; f < 3; f++)
            for (int j = 0; j < NQ1; j++) d.S[f][m][j] = (R)t.side[(f * NP + m) * NQ1 + j];
        for (int v = 0; v < 3; v++) d.V[m][v] = (R)t.vertex[m * 3 + v];
    }
    for (int j = 0; j < NQ1; j++) d.W1[j] = (R)t.w1[j];
    for (int q = 0; q < NQ; q++) {
        d.R1[q] = (R)t.r1[q];
        d.R2[q] = (R)t.r2[q];
        d.W[q] = (R)t.w[q];
    }
}

template <typename R>
static void fill_all(TabAll<R>& a) {
    fill_tab<R, 0>(a.p0);
    fill_tab<R, 1>(a.p1);
    fill_tab<R, 2>(a.p2);
    fill_tab<R, 3>(a.p3);
    fill_tab<R, 4>(a.p4);
    fill_tab<R, 5>(a.p5);
}

hipError_t upload_tables() {
    static TabAll<double> h64;
    static TabAll<float> h32;
    fill_all<double>(h64);
    fill_all<float>(h32);
    hipError_t e = upload_tables_kernels(h64, h32);
    if (e == hipSuccess) e = upload_tables_mfma(h64, h32);
    if (e == hipSuccess) e = upload_tables_batch(h64, h32);
    return e;
}

}  // namespace dgmi

namespace dgmi {

// Streaming copy (16-byte vector loads and stores), the bandwidth reference
// for the roofline and the scale of the FETCH_SIZE / WRITE_SIZE counters.
// Streaming copy used as the bandwidth reference.  One 16-byte load and
// store per thread and iteration over a grid of 1024 workgroups: on MI355X
// this simple form measured faster than deeper unrolling or larger grids
// (about 5.6 TB/s for 1 GiB, read + write).
__global__ void __launch_bounds__(256) k_stream_copy(const float4* __restrict__ src, float4* __restrict__ dst,
                                                    int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// The same copy with four independent 16-byte loads in flight per thread
// before their stores (64 bytes per thread and iteration).
__global__ void __launch_bounds__(256) k_stream_copy4(const float4* __restrict__ src, float4* __restrict__ dst,
                                                     int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const float4 a = src[i], b = src[i + stride], c = src[i + 2 * stride], d = src[i + 3 * stride];
        dst[i] = a;
        dst[i + stride] = b;
        dst[i + 2 * stride] = c;
        dst[i + 3 * stride] = d;
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

// variant 0: k_stream_copy on 1024 workgroups; 1..3: k_stream_copy4 on
// 1024, 2048, 4096 workgroups
hipError_t launch_stream_copy(const void* src, void* dst, int64_t bytes, hipStream_t st, int variant) {
    const int64_t n = bytes / 16;
    if (variant == 0)
        hipLaunchKernelGGL(k_stream_copy, dim3(1024), dim3(256), 0, st, (const float4*)src, (float4*)dst, n);
    else
        hipLaunchKernelGGL(k_stream_copy4, dim3(512 << variant), dim3(256), 0, st, (const float4*)src, (float4*)dst, n);
    return hipGetLastError();
}

}  // namespace dgmi
