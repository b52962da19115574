// Matrix-core (MFMA) processing of one 64-element tile, shared by the
// single-solve persistent kernel and the batched kernel.
//
// A workgroup of 4 wavefronts processes a tile of 64 consecutive (Morton)
// elements, one 16-element sub-tile per wavefront.  Per sub-tile and
// variable the element-local contractions are 16x16xK matrix products on
// v_mfma_f32_16x16x4f32 (FP32) or v_mfma_f64_16x16x4f64 (FP64) with elements
// as the N dimension:
//   volume interpolation  U[q][e]  = sum_m B[q][m]      u[m][e]      (K = 16)
//   face traces           T[pt][e] = sum_m S[pt][m]     u[m][e]      (K = 16)
//   volume projection     R[m][e]  = sum_q Gx[m][q] Fr[q][e] + Gy[m][q] Fs[q][e]  (K = 32)
//   surface projection    R[m][e] += sum_pt S[m][pt] w    G[pt][e]   (K = 16)
// where pt runs over the 3*(p+1) face points (padded to 16).  Each lane
// computes the volume fluxes of the points its accumulator registers hold;
// the reduction dimension of the projections is ordered the same way, so no
// data moves between lanes between the products.
//
// Neighbour traces come through LDS: every element's own face traces are
// written to LDS, and the tile's halo (neighbours outside the tile, listed
// per tile on the host) is traced into extra LDS slots.  The tile then
// evaluates the LLF flux of each of its sides once, spread evenly over its
// 256 lanes: a side between two of its elements is computed by one of them
// and written to both (the negation is exactly what the other would
// compute); a side to the halo is computed by the tile's element, and again
// by the neighbour's own tile, with identical operands, so the two
// contributions are bit-identical with opposite signs: race-free, no
// atomics, no face buffers in HBM.
#pragma once

#include <type_traits>

#include "dg_kernels.h"

namespace dgmi {

typedef float floatx4 __attribute__((ext_vector_type(4)));

typedef double doublex4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Per precision: the 16x16x4 product and where its operands and results
// sit.  Both take A[i][k] from lane i + 16k and B[k][j] from lane j + 16k.
// The FP32 product leaves D[4g + r][j] in register r of lane j + 16g, the
// FP64 product D[g + 4r][j]; pos(g, r) names that row.  Every reduction is
// ordered the same way (product s of lane group g takes index pos(g, s)),
// so a lane's B operands are the rows it holds in the output.  A mode
// step s whose modes pos(0..3, s) are all padding (FP64 up to p = 3: modes
// 4s..4s+3) is left out: p = 3 at 131,072 triangles 173.5 -> 166.2 us per step.
// Volume and face points are placed by the A tables of the interpolations:
// row i holds point qrow(i), so register r of lane group g holds point
// qpos(g, r) = g + 4r in both precisions.  Product step r of the
// projections then takes points 4r..4r+3, and a step whose points are all
// padding (4r >= the point count, p <= 3) is left out at compile time.
template <typename R>
struct MfmaT;
template <>
struct MfmaT<float> {
    using V = floatx4;
    __device__ __forceinline__ static V mma(float a, float b, V c) { return mfma4(a, b, c); }
    __host__ __device__ static constexpr int pos(int g, int r) { return 4 * g + r; }
    __host__ __device__ static constexpr int qpos(int g, int r) { return g + 4 * r; }
    __host__ __device__ static constexpr int qrow(int i) { return (i >> 2) + 4 * (i & 3); }
};
template <>
struct MfmaT<double> {
    using V = doublex4;
    __device__ __forceinline__ static V mma(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __host__ __device__ static constexpr int pos(int g, int r) { return g + 4 * r; }
    __host__ __device__ static constexpr int qpos(int g, int r) { return g + 4 * r; }
    __host__ __device__ static constexpr int qrow(int i) { return i; }
};

constexpr int MFMA_TILE = 64;

// whether mode step s of the mode reductions is issued (see above)
template <typename R, int NP>
__host__ __device__ constexpr bool mode_step_used(int s) {
    return MfmaT<R>::pos(0, s) < NP;
}

// LDS of a tile: the records of its sides [192] of 4 values (MfmaArgs), then
// traces [(64 + hcap)][17*N] values (16 points + 1 padding row so consecutive
// slots start in different banks), N variables innermost; `rs` = bytes per
// value (4 FP32, 8 FP64).
constexpr int MFMA_MAX_SIDES = MFMA_TILE * 3;
__host__ __device__ constexpr size_t mfma_tile_lds_bytes(int N, int hcap, int rs = 4) {
    return (size_t)MFMA_MAX_SIDES * 4 * rs + (size_t)(MFMA_TILE + hcap) * MFMA_SLOT_POINTS * N * rs;
}

// the traces of a tile's LDS, after the side records `fd`
template <typename V, typename R>
__device__ __forceinline__ R* tile_traces(V* fd) {
    return reinterpret_cast<R*>(fd + MFMA_MAX_SIDES);
}

// State access in the tile layout (StateIx): lane j + 16g of a wavefront
// moves the modes pos(g, 0..3) of its element and one variable.  Lanes whose
// group or register holds no mode read another lane's entry instead (in
// bounds; their operands meet zero matrix entries) and store nothing.
template <typename V>
__device__ __forceinline__ V tile_get(const DG_GLOBAL V* p, bool nt) {
    return nt ? __builtin_nontemporal_load(p) : *p;
}
template <int N, int P, typename R>
struct TileIo;
// FP32: one access of 16 bytes; groups of 4 modes
template <int N, int P>
struct TileIo<N, P, float> {
    using V = floatx4;
    static constexpr int G = tile_groups(n_modes(P)), VS = 16 * G;
    unsigned at;  // in units of 4 values: a scalar base and a 32-bit index
    __device__ __forceinline__ TileIo(int e, int g)
        : at((unsigned)((e >> 4) * (N * 16 * G) + (G == 4 ? g : min(g, G - 1)) * 16 + (e & 15))) {}
    __device__ __forceinline__ V load(const float* p, int v, bool nt = false) const {
        return tile_get((const DG_GLOBAL V*)p + (v * VS + at), nt);
    }
    __device__ __forceinline__ void store(float* p, int v, int g, V x) const {
        if (G == 4 || g < G) __builtin_nontemporal_store(x, (DG_GLOBAL V*)p + (v * VS + at));
    }
};
// FP64: pieces of 16 and 8 bytes (tile64_at).  Storing the used modes only
// instead of 16 slots cuts the state's bytes by 37% at p = 3 and 62% at p = 2,
// and 16-byte pieces a wavefront covers without gaps replace two halves of 32:
// per step p = 3 at 131,072 triangles 225.3 -> 173.5 us (at 524,288 786 -> 624),
// p = 2 at 32,768 74 -> 45.6, p = 4 at 131,072 243.7 -> 227.0, advection p = 3
// at 131,072 64.3 -> 54.9 and p = 1 at 2,048 18.0 -> 16.5.
template <int N, int P>
struct TileIo<N, P, double> {
    using V = doublex4;
    typedef double V2 __attribute__((ext_vector_type(2)));
    static constexpr int NP = n_modes(P), VS = 16 * tile64_slots(NP);
    static constexpr bool PAIRS = NP > 8;
    // lanes per register r whose group holds a mode
    __host__ __device__ static constexpr int groups(int r) { return NP - 4 * r < 4 ? NP - 4 * r : 4; }
    size_t block;
    int a, b;  // places of registers 0 (and 1) and of the next piece
    __device__ __forceinline__ TileIo(int e, int g) : block((size_t)(e >> 4) * (N * VS)) {
        const int j = e & 15;
        if constexpr (PAIRS) {
            a = (g * 16 + j) * 2;
            b = NP > 12 ? 128 + a : 128 + min(g, groups(2) - 1) * 16 + j;
        } else {
            a = min(g, groups(0) - 1) * 16 + j;
            b = 64 + min(g, NP > 4 ? groups(1) - 1 : 0) * 16 + j;
        }
    }
    __device__ __forceinline__ V load(const double* p, int v, bool nt = false) const {
        const DG_GLOBAL double* q = (const DG_GLOBAL double*)p + block + v * VS;
        if constexpr (PAIRS) {
            const V2 x = tile_get((const DG_GLOBAL V2*)(q + a), nt);
            if constexpr (NP > 12) {
                const V2 y = tile_get((const DG_GLOBAL V2*)(q + b), nt);
                return V{x[0], x[1], y[0], y[1]};
            }
            return V{x[0], x[1], tile_get(q + b, nt), 0.0};
        }
        const double x = tile_get(q + a, nt);
        if constexpr (NP > 4) return V{x, tile_get(q + b, nt), 0.0, 0.0};
        return V{x, 0.0, 0.0, 0.0};
    }
    __device__ __forceinline__ void store(double* p, int v, int g, V x) const {
        DG_GLOBAL double* q = (DG_GLOBAL double*)p + block + v * VS;
        if constexpr (PAIRS) {
            __builtin_nontemporal_store(V2{x[0], x[1]}, (DG_GLOBAL V2*)(q + a));
            if constexpr (NP > 12)
                __builtin_nontemporal_store(V2{x[2], x[3]}, (DG_GLOBAL V2*)(q + b));
            else if (g < groups(2))
                __builtin_nontemporal_store(x[2], q + b);
        } else {
            if (g < groups(0)) __builtin_nontemporal_store(x[0], q + a);
            if constexpr (NP > 4)
                if (g < groups(1)) __builtin_nontemporal_store(x[1], q + b);
        }
    }
};

// The five products' per-lane A operands (lane layout: A[i][k] from lane
// i + 16k, B[k][j] from lane j + 16k) as an LDS table [5][64] of 4 values:
// read where used, they would hold 20 registers.  The mode reductions (vol,
// tr) run mode pos(g, s) through product s in lane group g, so the B operand
// of a lane is its own modes as it loads them and the state in operand
// registers is already in the output layout of the projections.  A call fills
// the operands of product step s; the 4 wavefronts of a batch's workgroup take
// one each at the start of every run (by one wavefront: 64 ragged solves in
// FP32 657 -> 636 us per step).
enum { MFMA_A_VOL = 0, MFMA_A_TR = 1, MFMA_A_SP = 2, MFMA_A_GX = 3, MFMA_A_GY = 4, MFMA_A_SLOTS = 5 };

template <int P, typename R>
__device__ __forceinline__ void mfma_a_to_lds(typename MfmaT<R>::V* tabA, int s, int lane) {
    constexpr int NP = n_modes(P), NQ = n_quad_vol(P), NQ1 = P + 1, NPT = 3 * NQ1;
    const TabP<R, P>& T = tab<R, P>();
    const int g = lane >> 4, j = lane & 15;
    const int qj = MfmaT<R>::qrow(j);  // the point of A row j
    const int m = MfmaT<R>::pos(g, s), q = MfmaT<R>::qpos(g, s);
    R* t = reinterpret_cast<R*>(tabA + lane) + s;
    constexpr int SLOT = 64 * 4;
    // (loads unconditional with clamped indices, so that none waits for another)
    const int mc = min(m, NP - 1), jc = min(j, NP - 1), qc = min(q, NQ - 1), fc = min(q, NPT - 1);
    const int qjc = min(qj, NQ - 1), fjc = min(qj, NPT - 1);
    const R vol = T.B[mc][qjc], tr = T.S[fjc / NQ1][mc][fjc % NQ1];
    const R sp = T.S[fc / NQ1][jc][fc % NQ1] * T.W1[fc % NQ1], gx = T.Gx[jc][qc], gy = T.Gy[jc][qc];
    t[MFMA_A_VOL * SLOT] = (m < NP && qj < NQ) ? vol : R(0);
    t[MFMA_A_TR * SLOT] = (m < NP && qj < NPT) ? tr : R(0);
    t[MFMA_A_SP * SLOT] = (j < NP && q < NPT) ? sp : R(0);
    t[MFMA_A_GX * SLOT] = (j < NP && q < NQ) ? gx : R(0);
    t[MFMA_A_GY * SLOT] = (j < NP && q < NQ) ? gy : R(0);
}

// State operands of one tile held by one wavefront: its own sub-tile, and
// its share of the halo, dealt as (halo sub-tile, variable) pairs
// round-robin to the 4 wavefronts.
// REF: the state comes from the caller's FP64 array in the reference layout
// (ST_RHS_REF) and is held as read; `own` and `halo` give the operands in
// the bulk precision.
template <int N, int P, typename R = float, bool REF = false>
struct MfmaTileState {
    using V = typename MfmaT<R>::V;
    using VM = typename MfmaT<typename std::conditional<REF, double, R>::type>::V;
    static constexpr int HPW = (4 * N + 3) / 4;  // most halo pairs per wave (hcap <= 64)
    VM ub[N];
    VM hb[HPW];
    __device__ __forceinline__ static V bulk(const VM& x) {
        if constexpr (REF)
            return V{(R)x[0], (R)x[1], (R)x[2], (R)x[3]};
        else
            return x;
    }
    __device__ __forceinline__ V own(int v) const { return bulk(ub[v]); }
    __device__ __forceinline__ V halo(int q) const { return bulk(hb[q]); }
    // variable v, modes pos(g, 0..3) (padding modes read the last mode: they
    // meet zero matrix entries) of caller's element o
    __device__ __forceinline__ static VM load_ref(const double* __restrict__ x, int v, int K, int g, int o) {
        constexpr int NP = n_modes(P);
        VM r;
#pragma unroll
        for (int s = 0; s < 4; s++)
            r[s] = *(const DG_GLOBAL double*)((const char DG_GLOBAL*)(const DG_GLOBAL double*)x +
                                              ((size_t)(v * NP + min(MfmaT<R>::pos(g, s), NP - 1)) * K + o) * 8);
        return r;
    }
    __device__ __forceinline__ void load_ref_data(const StageArgs<R>& a, int tile, int w, int g, int j,
                                                  const int (&hid)[HPW]) {
        const int o = ref_elem(a, min(tile * MFMA_TILE + w * 16 + j, a.K - 1));
        int oh[HPW];
#pragma unroll
        for (int q = 0; q < HPW; q++) oh[q] = ref_elem(a, hid[q]);
#pragma unroll
        for (int v = 0; v < N; v++) ub[v] = load_ref(a.ref_u, v, a.K, g, o);
#pragma unroll
        for (int q = 0; q < HPW; q++) hb[q] = load_ref(a.ref_u, (w + 4 * q) % N, a.K, g, oh[q]);
    }
    // Halo element ids of this wave's pairs.  A halo state load depends on
    // its id, and waiting for an id waits for every load issued before it,
    // so the ids are requested ahead of the state loads that use them.
    // Ids and halo states are loaded for every slot q, pairs past the list
    // from its last entries (in bounds, unused): loads under a branch, with
    // registers zeroed on the other path, make the compiler wait for them
    // (and for everything issued before them) at the next write.
    __device__ __forceinline__ static void load_ids(const int* __restrict__ halo, int hcap, int tile, int w, int j,
                                                   int (&hid)[HPW]) {
        const int hlast = (hcap >> 4) - 1;
#pragma unroll
        for (int q = 0; q < HPW; q++) {
            const int hs = min((w + 4 * q) / N, hlast);
            hid[q] = gp(halo)[(unsigned)(tile * hcap + hs * 16 + j)];
        }
    }
    __device__ __forceinline__ void load_data(const R* __restrict__ u, int K, int tile, int w, int g, int j,
                                              const int (&hid)[HPW]) {
        const TileIo<N, P, R> io(min(tile * MFMA_TILE + w * 16 + j, K - 1), g);
#pragma unroll
        for (int v = 0; v < N; v++) ub[v] = io.load(u, v);
#pragma unroll
        for (int q = 0; q < HPW; q++) hb[q] = TileIo<N, P, R>(hid[q], g).load(u, (w + 4 * q) % N);
    }
    __device__ __forceinline__ void load_next(const StageArgs<R>& a, int tile, int w, int g, int j,
                                              const int (&hid)[HPW]) {
        if constexpr (REF)
            load_ref_data(a, tile, w, g, j, hid);
        else
            load_data(a.u, a.K, tile, w, g, j, hid);
    }
};

// Cell wave speed |u| + c of the new state's cell mean for the CFL step
// (euler.cu:252-278, in the bulk precision as the reference computes it):
// FP32 with the hardware reciprocal and square root, as the fluxes.
template <int N>
__device__ __forceinline__ float cell_speed_bulk(const PhysP& ph, const float* U) {
    if constexpr (N == 1) {
        const float ax = (float)ph.ax, ay = (float)ph.ay;
        return __builtin_amdgcn_sqrtf(ax * ax + ay * ay);
    } else {
        const float g = (float)ph.gamma;
        const float ir = __builtin_amdgcn_rcpf(U[0]);
        const float m2 = U[1] * U[1] + U[2] * U[2];
        const float pr = (g - 1.f) * (U[3] - 0.5f * m2 * ir);
        return __builtin_amdgcn_sqrtf(m2) * ir + __builtin_amdgcn_sqrtf(g * pr * ir);
    }
}
template <int N>
__device__ __forceinline__ double cell_speed_bulk(const PhysP& ph, const double* U) {
    return cell_speed<N>(ph, U);
}

template <int KIND>
constexpr bool rk_writes_acc() {
    return KIND == ST_RK4_2;
}

// Geometry of one tile from the packed arrays: the side record this thread
// stores to LDS (threads past tcap hold the tile's last again and store
// nothing, so the load is not under a branch), the number of sides, the
// affine map and the inverse mass of the lane's own element.  Padding
// elements replicate element K-1 in every geometry array.
template <typename R = float>
struct TileGeo {
    using V = typename MfmaT<R>::V;
    V f;
    int ntask;
    R xr, yr, xs, ys, ij;  // ij: the inverse mass 1/J (M = J*I), precomputed in FP64
    __device__ __forceinline__ void load(const StageArgs<R>& a, const MfmaArgs& mx, int tile, int el) {
        f = ((const DG_GLOBAL V*)mx.sides)[(unsigned)(tile * mx.tcap + min((int)threadIdx.x, mx.tcap - 1))];
        ntask = gp(mx.ntask)[(unsigned)tile];
        const unsigned ue = (unsigned)(tile * MFMA_TILE + el);
        const V m = ((const DG_GLOBAL V*)mx.metric4)[ue];
        xr = m[0];
        yr = m[1];
        xs = m[2];
        ys = m[3];
        ij = (gp(a.geo_e) + 4 * (size_t)a.Kp)[ue];
    }
};

// word of a side record (FP32: the bits of the 4th value, FP64:
// its value)
__device__ __forceinline__ int face_word(float x) { return __float_as_int(x); }
__device__ __forceinline__ int face_word(double x) { return (int)x; }

// LLF flux of one point of one side: record `r` (word `wd`), the element's
// trace at the point `own` and the neighbour's `nbt`, in the orientation of
// the element; written over `own`, and its negation over `nbt` when the
// neighbour is an element of the tile.  For a boundary side, `nw` is the
// side's neighbour word (the ghost data's index) and jo the point.
template <int N, int NQ1, typename R, bool BND>
__device__ __forceinline__ void side_flux(const StageArgs<R>& a, const typename MfmaT<R>::V r, int wd, R* own, R* nbt,
                                          int nw, int jo) {
    using V = typename MfmaT<R>::V;
    const bool left = r[2] < R(0);
    const bool inner = wd & SIDE_INNER;
    // boundary side (the element is its left element, the slot its own): the
    // ghost state of the point replaces the neighbour trace, which is not
    // read.  Only the BND instantiation carries this code, so the kernels
    // of meshes without boundary sides keep their register allocation.
    const bool bside = BND && (wd & SIDE_BOUNDARY);
    if constexpr (BND)
        if (bside) nbt = own;
    R G[N];
    if constexpr (N == 4) {
        // F(UL).n + F(UR).n, max of the two speeds and UL - UR with the sign
        // of this side folded into the speed
        R uo[N], un[N], Fo[N], Fb[N], so, sb;
        const V qo = *reinterpret_cast<const V*>(own), qn = *reinterpret_cast<const V*>(nbt);
#pragma unroll
        for (int v = 0; v < N; v++) {
            uo[v] = qo[v];
            un[v] = qn[v];
        }
        if constexpr (BND)
            if (bside) boundary_ghost<N, NQ1, R>(a.bnd, nw, jo, uo, un);
        normal_flux_speed<R>(a.phys, uo, r[0], r[1], Fo, so);
        normal_flux_speed<R>(a.phys, un, r[0], r[1], Fb, sb);
        const R lm = fmax(so, sb);
        const R lms = left ? lm : -lm;
#pragma unroll
        for (int v = 0; v < N; v++) G[v] = r[2] * fma(lms, uo[v] - un[v], Fo[v] + Fb[v]);
        *reinterpret_cast<V*>(own) = V{G[0], G[1], G[2], G[3]};
        if (inner && !bside) *reinterpret_cast<V*>(nbt) = V{-G[0], -G[1], -G[2], -G[3]};
    } else {
        R UL[N], UR[N];
        {
            const R uo = own[0], un = nbt[0];
            UL[0] = left ? uo : un;
            UR[0] = left ? un : uo;
        }
        if constexpr (BND)
            if (bside) boundary_ghost<N, NQ1, R>(a.bnd, nw, jo, UL, UR);
        R fxl[N], fyl[N], fxr[N], fyr[N];
        flux<N, R>(a.phys, UL, fxl, fyl);
        flux<N, R>(a.phys, UR, fxr, fyr);
        const R lm = llf_speed<N, R>(a.phys, UL, UR, r[0], r[1]);
        const R coef = R(2) * r[2];
        G[0] = coef * (R(0.5) * ((fxl[0] + fxr[0]) * r[0] + (fyl[0] + fyr[0]) * r[1] + lm * (UL[0] - UR[0])));
        own[0] = G[0];
        if (inner && !bside) nbt[0] = -G[0];
    }
}

// Software-pipelined body of the persistent single-solve kernel.  On entry
// `st` and `gc` hold the state and geometry of `tile`, and `hid` the halo
// ids of `next`.  Once the volume interpolation has consumed the state, the
// tile's RK registers (c, acc) are requested and then the state of `next`
// into the same registers; after the face fluxes the geometry of `next` and
// the halo ids of `next2` are requested, ahead of this tile's stores.  The
// vector-memory counter retires in issue order and counts stores, so every
// load a later wait is for is issued before the stores that wait need not
// cover (the scheduling barriers keep that order).  `next` and `next2` are
// tiles of this launch (the caller repeats the last tile where the walk
// ends), so no load sits under a branch.  The A operands are read from the
// LDS table `tabA`.
template <int N, int P, int KIND, typename R, bool BND = false>
__device__ __forceinline__ double mfma_process_tile_pipe(const StageArgs<R>& a, const MfmaArgs& mx,
                                                         const typename MfmaT<R>::V* tabA,
                                                         MfmaTileState<N, P, R, KIND == ST_RHS_REF>& st,
                                                         int (&hid)[MfmaTileState<N, P, R>::HPW], TileGeo<R>& gc,
                                                         R dt, int tile, int next, int next2,
                                                         typename MfmaT<R>::V* fd, R* ts) {
    using M = MfmaT<R>;
    using V = typename M::V;
    constexpr int NP = n_modes(P), NQ = n_quad_vol(P), NQ1 = P + 1, NPT = 3 * NQ1;
    constexpr int TILE = MFMA_TILE;
    constexpr int TS = MFMA_SLOT_POINTS * N;
    constexpr bool LAST = (KIND == ST_RK4_4 || KIND == ST_RK2_2);
    using RK = RkNeeds<KIND>;
    constexpr int HPW = MfmaTileState<N, P, R>::HPW;
    static_assert(NP <= 16 && NQ <= 16 && NPT <= 16, "order too high for 16x16 tiles");
    const int K = a.K;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int g = lane >> 4, j = lane & 15;
    const int npairs = (mx.hcap >> 4) * N;
    const int base = tile * TILE;
    const int el = w * 16 + j;
    const int e = base + el;
    const bool valid = e < K;
    const int ee = valid ? e : K - 1;

    const R xr = gc.xr, yr = gc.yr, xs = gc.xs, ys = gc.ys;

    // ---- phase 1: face traces of the own sub-tile and of this wave's halo pairs ----
    // (points qpos(g, 0..3) of every lane are written: a slot holds 16 points
    // plus a padding row; points >= 3(p+1) are read by the surface
    // projection only to be replaced by zero)
    const V Atr = tabA[MFMA_A_TR * 64 + lane];
    constexpr bool REF = KIND == ST_RHS_REF;
    V ub[N];
#pragma unroll
    for (int v = 0; v < N; v++) ub[v] = st.own(v);
    {
        V T[N];
#pragma unroll
        for (int v = 0; v < N; v++) {
            T[v] = V{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 4; s++)
                if (mode_step_used<R, NP>(s)) T[v] = M::mma(Atr[s], ub[v][s], T[v]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            R* dst = ts + el * TS + M::qpos(g, i) * N;
            if constexpr (N == 4)
                *reinterpret_cast<V*>(dst) = V{T[0][i], T[1][i], T[2][i], T[3][i]};
            else
                dst[0] = T[0][i];
        }
    }
#pragma unroll
    for (int q = 0; q < HPW; q++) {
        const int pr = w + 4 * q;
        if (pr < npairs) {
            const int slot = TILE + (pr / N) * 16 + j, v = pr % N;
            V acc = {0, 0, 0, 0};
            const V hb = st.halo(q);
#pragma unroll
            for (int s = 0; s < 4; s++)
                if (mode_step_used<R, NP>(s)) acc = M::mma(Atr[s], hb[s], acc);
#pragma unroll
            for (int i = 0; i < 4; i++) ts[slot * TS + M::qpos(g, i) * N + v] = acc[i];
        }
    }
    if ((int)threadIdx.x < mx.tcap) fd[threadIdx.x] = gc.f;

    // ---- phase 2: volume, side fluxes, surface, inverse mass, RK update ----
    V U[N];
    const V Avol = tabA[MFMA_A_VOL * 64 + lane];
#pragma unroll
    for (int v = 0; v < N; v++) {
        V acc = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (mode_step_used<R, NP>(s)) acc = M::mma(Avol[s], ub[v][s], acc);
        U[v] = acc;
    }
    // RK registers of this tile, then the next tile's state (st is dead
    // after this block).  For a stage whose input is the RK base state the
    // operand registers already hold it in the output layout.  c and acc are
    // read once per launch and the outputs are not read again in it: their
    // accesses carry the non-temporal hint, which keeps the 4 MB L2 of an
    // XCD for the stage input, whose lines neighbouring tiles read again as
    // halo (measured: 0.135 -> 0.122 ms per stage at 524,288 triangles, p = 4;
    // the hint on the geometry loads measured slower).
    // The wave runs at raised priority while it issues its loads, so a wave
    // with requests to make gets the issue slot before waves computing
    // (measured 1.5% faster per step at 524,288 triangles, p = 4).
    __builtin_amdgcn_s_setprio(2);
    const TileIo<N, P, R> io(ee, g);
    V cr[N], ar[N];
#pragma unroll
    for (int v = 0; v < N; v++) {
        cr[v] = V{0, 0, 0, 0};
        ar[v] = V{0, 0, 0, 0};
        if constexpr (RK::C_FROM_INPUT) cr[v] = ub[v];
        if constexpr (RK::ACC_FROM_INPUT) ar[v] = ub[v];
        if constexpr (sizeof(R) == 4) {
            if constexpr (RK::LOAD_C) cr[v] = io.load(a.c, v, true);
            if constexpr (RK::LOAD_ACC) ar[v] = io.load(a.acc, v, true);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    st.load_next(a, next, w, g, j, hid);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    V Rv[N];
#pragma unroll
    for (int v = 0; v < N; v++) Rv[v] = V{0, 0, 0, 0};
    const V Agx = tabA[MFMA_A_GX * 64 + lane], Agy = tabA[MFMA_A_GY * 64 + lane];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // volume point q = qpos(g, i): flux, metric, reduction step i (steps
        // of padding points only are left out)
        if (4 * i >= NQ) continue;
        R Uq[N], fx[N], fy[N];
#pragma unroll
        for (int v = 0; v < N; v++) Uq[v] = U[v][i];
        const bool qv = M::qpos(g, i) < NQ;
        if (N == 4 && !qv) Uq[0] = R(1);  // padding point: keep the flux finite
        if constexpr (N == 4) {
            metric_flux<R>(a.phys, Uq, xr, yr, xs, ys, fx, fy);  // fx, fy hold Fr, Fs
#pragma unroll
            for (int v = 0; v < N; v++) {
                Rv[v] = M::mma(Agx[i], qv ? fx[v] : R(0), Rv[v]);
                Rv[v] = M::mma(Agy[i], qv ? fy[v] : R(0), Rv[v]);
            }
        } else {
            flux<N, R>(a.phys, Uq, fx, fy);
#pragma unroll
            for (int v = 0; v < N; v++) {
                const R fr = qv ? fx[v] * ys - fy[v] * xs : R(0);
                const R fs = qv ? fy[v] * xr - fx[v] * yr : R(0);
                Rv[v] = M::mma(Agx[i], fr, Rv[v]);
                Rv[v] = M::mma(Agy[i], fs, Rv[v]);
            }
        }
    }
    __syncthreads();

    // ---- phase 2b: the LLF flux of each side of the tile, once ----
    // (after the volume terms, which use only this wave's registers, so the
    // waves meet at the barrier with the next tile's loads long in flight)
    // Work item (side k, point jo); the 64-item blocks of a
    // round go to the wavefronts in an order that rotates with the tile, so
    // the partial last round falls to each wavefront in turn.  The flux is
    // computed in the orientation of the record's element and written over
    // that element's trace at the point; a side between two elements of the
    // tile also writes its negation over the other element's trace, which is
    // bit for bit what that element would compute (the sums and maxima of the
    // two sides' terms commute and the sign flips are exact).  Each trace
    // entry of the tile's elements belongs to one side and one point, so the
    // item that reads it is the only one that writes it.
    {
        const int nitem = gc.ntask * NQ1;
        const int wblk = ((w + tile) & 3) * 64;
        for (int r0 = 0; r0 < nitem; r0 += 256) {
            if (r0 + wblk >= nitem) continue;  // uniform over the wavefront
            const int it = r0 + wblk + lane;
            if (it < nitem) {
                const int k = it / NQ1, jo = it - k * NQ1;
                const V rec = fd[k];
                const int wd = face_word(rec[3]);
                const int oo = wd & ((1 << SIDE_OWN_BITS) - 1);
                const int no = (wd >> SIDE_OWN_BITS) & ((1 << SIDE_NBR_BITS) - 1);
                int nw = 0;
                if constexpr (BND) {
                    const int eo = oo / MFMA_SLOT_POINTS, f = (oo - eo * MFMA_SLOT_POINTS) / NQ1;
                    nw = gp(a.nbr)[f * a.Kp + base + eo];
                }
                side_flux<N, NQ1, R, BND>(a, rec, wd, ts + (oo + jo) * N, ts + (no - jo) * N, nw, jo);
            }
        }
    }
    __syncthreads();

#pragma unroll
    for (int i = 0; i < 4; i++) {
        // own face point pt = qpos(g, i): its flux from phase 2b (point slots
        // past 3(p+1) hold stale traces and meet zero; steps of such slots
        // only are left out)
        if (4 * i >= NPT) continue;
        const int pt = M::qpos(g, i);
        const R* gq = ts + el * TS + pt * N;
        R G[N];
        if constexpr (N == 4) {
            const V q = *reinterpret_cast<const V*>(gq);
#pragma unroll
            for (int v = 0; v < N; v++) G[v] = pt < NPT ? q[v] : R(0);
        } else {
            G[0] = pt < NPT ? gq[0] : R(0);
        }
        const V Asp = tabA[MFMA_A_SP * 64 + lane];
#pragma unroll
        for (int v = 0; v < N; v++) Rv[v] = M::mma(Asp[i], G[v], Rv[v]);
    }

    // geometry of the next tile and halo ids of the one after, requested
    // before this tile's stores
    const R cj = gc.ij * dt;
    __builtin_amdgcn_s_setprio(2);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (sizeof(R) == 8) {
        // FP64 requests c and acc here instead, after the fluxes: their 64
        // registers are then not live across the face fluxes, which lets two
        // workgroups share a CU (0.409 -> 0.323 ms per stage at 524,288
        // triangles, p = 4); FP32 measured no gain from the same move
#pragma unroll
        for (int v = 0; v < N; v++) {
            if constexpr (RK::LOAD_C) cr[v] = io.load(a.c, v, true);
            if constexpr (RK::LOAD_ACC) ar[v] = io.load(a.acc, v, true);
        }
    }
    gc.load(a, mx, next, el);
    MfmaTileState<N, P>::load_ids(mx.halo, mx.hcap, next2, w, j, hid);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);

    if constexpr (REF) {
        // k into the caller's array; lane holds modes m = pos(g, i)
        if (valid) {
            const int o = ref_elem(a, e);
#pragma unroll
            for (int v = 0; v < N; v++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (M::pos(g, i) < NP)
                        *(DG_GLOBAL double*)((char DG_GLOBAL*)(DG_GLOBAL double*)a.ref_k +
                                             ((size_t)(v * NP + M::pos(g, i)) * K + o) * 8) = (double)(cj * Rv[v][i]);
        }
        __syncthreads();  // the next tile reuses the LDS
        return 0.0;
    }

    // inverse mass and the RK stage update; lane holds modes m = pos(g, i)
    const TileIo<N, P, R> so(e, g);
    R c0[N];
    double lam = 0.0;
#pragma unroll
    for (int v = 0; v < N; v++) {
        V o, an;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            R t = R(0);
            o[i] = rk_update<KIND, R>(cr[v][i], ar[v][i], cj * Rv[v][i], &t);
            an[i] = t;
        }
        // padding elements (e >= K) compute a copy of element K-1 into their own slots
        if constexpr (rk_writes_acc<KIND>()) so.store(a.acc, v, g, an);
        so.store(a.out, v, g, o);
        c0[v] = o[0];
    }
    if constexpr (LAST) {
        if (g == 0 && valid) {  // mode 0 = pos(0, 0) sits in register 0 of lane group 0
            R Uc[4];
            const R b0 = tab<R, P>().B[0][0];
#pragma unroll
            for (int v = 0; v < N; v++) Uc[v] = c0[v] * b0;
            lam = (double)cell_speed_bulk<N>(a.phys, Uc);
        }
    }
    __syncthreads();  // the next tile reuses the LDS
    return lam;
}

}  // namespace dgmi
