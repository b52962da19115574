// Host-visible launchers of the HIP kernels.
#pragma once
#include "dg_device.h"

namespace dgmi {

// initial-condition parameters passed by value to the projection kernel;
// also the state of inflow and outflow boundary sides
struct IcP {
    int kind;   // 0 constant, 1 Gaussian pulse, 2 vortex superposition, 3 supersonic vortex, 4 (x - y)^alpha
    int nv;
    double gamma;
    double gx, gy, gk;
    double Lx, Ly;
    double rho_inf, u_inf, v_inf, p_inf;
    double beta[4], vx[4], vy[4];
    double constant[4];
    double mach;  // supersonic vortex: Mach number at r = 1
    int fpow;     // supersonic vortex: powers rounded through float
    int alpha;    // (x - y)^alpha
};

// Initial condition U0(x, y) in FP64 (conserv_kernels.cu:167-187,
// euler.cu:31-59, supersonic.cu:28-38), on the host and the device.
__host__ __device__ inline double wrap_d(double d, double L) { return (L > 0) ? d - L * rint(d / L) : d; }

// a^b, or with fpow the reference's powf on double arguments: arguments and
// result rounded to float (the power itself here in FP64)
__host__ __device__ inline double ic_pow(double a, double b, int fpow) {
    return fpow ? (double)(float)pow((double)(float)a, (double)(float)b) : pow(a, b);
}

__host__ __device__ inline void ic_point(const IcP& ic, double x, double y, double* U) {
    if (ic.kind == 0) {
        for (int n = 0; n < 4; n++) U[n] = ic.constant[n];
        return;
    }
    if (ic.kind == 1) {
        double dx = wrap_d(x - ic.gx, ic.Lx), dy = wrap_d(y - ic.gy, ic.Ly);
        U[0] = exp(-ic.gk * (dx * dx + dy * dy));
        return;
    }
    if (ic.kind == 4) {
        // the advection prototype's test function (test_all.cu:21-51)
        const double u = pow(x - y, (double)ic.alpha);
        for (int n = 0; n < 4; n++) U[n] = u;
        return;
    }
    if (ic.kind == 3) {
        // supersonic vortex between two arcs (supersonic.cu:28-38): density
        // (1 + (gamma-1)/2 M^2 (1 - 1/r^2))^(1/(gamma-1)) with the reference's
        // literals 1.0125 and 2.5, speed M / r along the arcs, p = rho^gamma / gamma
        const double r = sqrt(x * x + y * y);
        U[0] = ic_pow(1 + 1.0125 * (1. - 1. / (r * r)), 2.5, ic.fpow);
        U[1] = U[0] * sin(atan(y / x)) * ic.mach / r;
        U[2] = U[0] * -cos(atan(y / x)) * ic.mach / r;
        const double pr = (1.0 / ic.gamma) * ic_pow(U[0], ic.gamma, ic.fpow);
        U[3] = 0.5 * U[0] * (ic.mach * ic.mach / (r * r)) + pr * (1. / (ic.gamma - 1.));
        return;
    }
    const double PI = 3.14159265358979323846;
    const double g = ic.gamma;
    double du = 0, dv = 0, dT = 0;
    for (int k = 0; k < ic.nv; k++) {
        double dx = wrap_d(x - ic.vx[k], ic.Lx), dy = wrap_d(y - ic.vy[k], ic.Ly);
        double r2 = dx * dx + dy * dy;
        double ex = exp(0.5 * (1. - r2));
        double beta = ic.beta[k];
        du += -beta / (2. * PI) * dy * ex;
        dv += beta / (2. * PI) * dx * ex;
        dT += -(g - 1.) * beta * beta / (8. * g * PI * PI) * ex * ex;
    }
    double T_inf = ic.p_inf / ic.rho_inf;
    double T = T_inf + dT;
    double rho = ic.rho_inf * pow(T / T_inf, 1. / (g - 1.));
    double pp = ic.p_inf * pow(rho / ic.rho_inf, g);
    double uu = ic.u_inf + du, vv = ic.v_inf + dv;
    U[0] = rho;
    U[1] = rho * uu;
    U[2] = rho * vv;
    U[3] = pp / (g - 1.) + 0.5 * rho * (uu * uu + vv * vv);
}

hipError_t upload_tables();
hipError_t upload_tables_kernels(const TabAll<double>& h64, const TabAll<float>& h32);
hipError_t upload_tables_mfma(const TabAll<double>& h64, const TabAll<float>& h32);
hipError_t upload_tables_batch(const TabAll<double>& h64, const TabAll<float>& h32);
// streaming copy variants of the bandwidth probe (0..STREAM_COPY_VARIANTS-1)
constexpr int STREAM_COPY_VARIANTS = 4;
hipError_t launch_stream_copy(const void* src, void* dst, int64_t bytes, hipStream_t st, int variant = 0);

template <typename R>
hipError_t launch_stage_valu(int N, int p, const StageArgs<R>& a, dim3 grid, hipStream_t st);
// packed geometry of the vector layout (StageArgs::lface, lmetric)
template <typename R>
hipError_t launch_lane_pack(const R* geo_e, const R* geo_f, const int* nbr, int Kp, void* lface, void* lmetric,
                            hipStream_t st);
// orders and physics whose lane kernel keeps its state in the vector layout
__host__ __device__ constexpr bool lane_vec(int N, int p) { return N == 4 && p <= 3; }
// Whether kernel kind `kind` has an instance on the caller's arrays
// (ST_RHS_REF): all but the Euler lane kernel at p = 4, 5, whose arithmetic
// and spills (0.4 ms at 131,072 triangles) leave the conversions no weight.
__host__ __device__ constexpr bool ref_rhs_supported(int N, int p, int kind) {
    return kind >= 2 || N == 1 || lane_vec(N, p);
}

// Extra per-solve data of the matrix-core kernel: per tile the halo element
// list [ntiles][hcap] and the sides the tile computes, [ntiles][tcap] records
// of 4 values in the bulk precision with `ntask` of them in use; per element
// 4 values (xr, yr, xs, ys) [Kp], padding elements replicating element K-1.
// A tile computes each of its sides once: the boundary sides, the sides to
// its halo, and of the sides between two of its elements the one whose
// record has the left element.  A record holds (nx, ny, f, word): f = len/4,
// negative for the side's left element, and the word (FP32 its bits, FP64
// its value) the offsets of the element's trace at point 0 of its face and
// of the neighbour's at its last point, in trace entries of 17 a slot, and
// the flags below.  Against three records per element and a side list built
// in LDS for every tile (per step of 4 stages): advection p = 4 FP32 524,288
// triangles 123.0 -> 116.9 us, Euler p = 3, 4 FP64 131,072 228.2 -> 225.3 and
// 246.3 -> 243.9, p = 4 FP32 524,288 374.8 -> 373.2.
constexpr int SIDE_OWN_BITS = 11, SIDE_NBR_BITS = 12;
constexpr uint32_t SIDE_INNER = 1u << 23;  // the neighbour is an element of the tile
constexpr uint32_t SIDE_BOUNDARY = 1u << 24;
constexpr int MFMA_SLOT_POINTS = 17;       // trace entries a slot: 16 points and 1 of padding (LDS banks)
struct SideTask {
    int ef;         // 3 * element + face
    uint32_t word;
};
struct MfmaArgs {
    const int* ntask;
    const int* halo;
    const void* sides;
    const void* metric4;
    int hcap;
    int tcap;
};
template <typename R>
hipError_t launch_mfma_pack(const R* geo_e, const R* geo_f, const int* nbr, const SideTask* tasks, int ntasks, int K,
                            int Kp, void* sides, void* metric4, hipStream_t st);

// matrix-core element kernel (FP32 or FP64, p = 1..4, state in the tile
// layout): 64-element tiles, 4 wavefronts per workgroup, persistent over the
// tiles of its XCD's range when the grid is smaller than the tile count;
// returns hipErrorInvalidValue for unsupported (N, p)
constexpr int MFMA_TILE_ELEMS = 64;
constexpr int MFMA_MAX_HALO = 64;
template <typename R>
hipError_t launch_stage_mfma(int N, int p, const StageArgs<R>& a, const MfmaArgs& mx, dim3 grid, hipStream_t st);
bool mfma_supported(int N, int p);
// dynamic LDS of a launch, `rs` = bytes per value of the bulk precision
size_t mfma_lds_bytes(int N, int hcap, int rs);
int mfma_resident_groups(int N, int p, int hcap, int rs, bool bnd);
hipError_t mfma_layout_probe(float* host_out);
hipError_t mfma_layout_probe_f64(double* host_out);
constexpr int VALU_TILE_ELEMS = 128;

// resets the solve's wave-speed slots and accumulates the state's maximum cell wave speed into them
template <typename R>
hipError_t launch_lambda(const R* u, const StateIx& ix, int K, double b0, const PhysP& ph, Ctrl* ctrl,
                         hipStream_t st);
// An FP64 array in the reference layout on the device, held in one or two
// pieces: rows (v*n_p + m) below `split` at lo, the others at hi.
struct RefRows {
    double *lo, *hi;
    int split;
};
// reference layout (FP64, caller's order) <-> state array in layout ix
template <typename R>
hipError_t launch_ref_to_state(const RefRows& ref, R* dst, const int* perm, const StateIx& ix, int K, hipStream_t st);
template <typename R>
hipError_t launch_state_to_ref(const R* src, const RefRows& ref, const int* perm, const StateIx& ix, int K,
                               hipStream_t st);
hipError_t launch_set_dt(Ctrl* ctrl, double dt, int advance, hipStream_t st);
template <typename R>
hipError_t launch_project_ic(int p, R* c, const StateIx& ix, const double* V, int K, const IcP& ic, hipStream_t st);
template <typename R>
hipError_t launch_audit(const R* c, const StateIx& ix, const double* Jd, int K, double b0, double gamma,
                        double* part, int nblocks, hipStream_t st);

// Ghost state UR of point j of a boundary side from the left trace UL
// (eval_left_right, conserv_kernels.cu:647-671): reflecting keeps rho and E
// and the velocity's component along the wall (supersonic.cu:64-108, wall
// normal precomputed per point); inflow and outflow take the problem's
// state at the point (euler.cu:177-241, precomputed in FP64).
template <int N, int NQ1, typename R>
__device__ __forceinline__ void boundary_ghost(const double* bnd, int w, int j, const R* UL, R* UR) {
    // the point's four values go to scalars first: indexing the pointer in a
    // loop made the compiler keep the ghost in a private (scratch) array
    const double* g = bnd + ((size_t)(w & NB_ELEM_MASK) * NQ1 + j) * 4;
    const double g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
    if (((w >> 28) & 3) == BC_REFLECTING) {
        UR[0] = UL[0];
        if constexpr (N == 4) {
            const R Nx = (R)g0, Ny = (R)g1;
            const R t = UL[1] * Ny - UL[2] * Nx;
            UR[1] = t * Ny;
            UR[2] = -t * Nx;
            UR[3] = UL[3];
        }
    } else {
        UR[0] = (R)g0;
        if constexpr (N == 4) {
            UR[1] = (R)g1;
            UR[2] = (R)g2;
            UR[3] = (R)g3;
        }
    }
}

}  // namespace dgmi
