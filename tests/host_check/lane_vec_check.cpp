// Host build of the Euler lane body in the vector layout (lane_process,
// dg_lane_body.h) against the general lane body (valu_process, mode-major
// rows, the reference's operation order) on the same state and mesh: every
// element, padding included, every stage kind, buffers of exactly the device
// sizes (built with -fsanitize=address).
//
//   lane_vec_check <mesh.pmsh> <p: 1..3> <precision: 0 FP64 | 1 FP32>
#include <hip/hip_runtime.h>
inline int __float_as_int(float x) { int i; memcpy(&i, &x, 4); return i; }
inline float __int_as_float(int i) { float x; memcpy(&x, &i, 4); return x; }
#define LANE_FENCE()
#define LANE_KEEP(x)
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <vector>

#include "dg_geometry.h"
#include "dg_mesh.h"
#include "dg_lane_body.h"
#include "dg_valu_body.h"

using namespace dgmi;

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
    }
    for (int j = 0; j < NQ1; j++) d.W1[j] = (R)t.w1[j];
}

template <int P, typename R, int KIND>
static bool one(StageArgs<R> a, StageArgs<R> b, const StateIx& im, const StateIx& iv, const std::vector<R>& ltab,
                int threads) {
    a.kind = b.kind = KIND;
    double la = 0, lb = 0;
    const auto go = [] { return true; };
    const auto dt = [&] { return (R)b.ctrl->dt; };
    for (int e = 0; e < threads; e++) {
        if (a.bnd) {
            la = std::max(la, valu_process<4, P, R, true>(a, e, KIND));
            lb = std::max(lb, lane_process<P, KIND, R, true, false>(b, e, ltab.data(), go, dt));
        } else {
            la = std::max(la, valu_process<4, P, R, false>(a, e, KIND));
            lb = std::max(lb, lane_process<P, KIND, R, false, true>(b, e, ltab.data(), go, dt));
        }
    }
    // states of order 1, updates below 1, some hundred roundings each
    const double tol = 1000 * (double)std::numeric_limits<R>::epsilon();
    double worst = std::fabs(la - lb);
    for (int v = 0; v < 4; v++)
        for (int m = 0; m < n_modes(P); m++)
            for (int e = 0; e < a.K; e++) {
                worst = std::max(worst, std::fabs((double)a.out[im.at(v, m, e)] - (double)b.out[iv.at(v, m, e)]));
                worst = std::max(worst, std::fabs((double)a.acc[im.at(v, m, e)] - (double)b.acc[iv.at(v, m, e)]));
            }
    printf("  kind %d: largest difference %.3e (bound %.3e)\n", KIND, worst, tol);
    return worst <= tol;
}

template <typename R, int P>
static int run(const Mesh& m) {
    constexpr int N = 4, NP = n_modes(P), NQ1 = P + 1;
    const int K = m.K, Kp = (K + 63) / 64 * 64;
    std::vector<int> perm = morton_order(m);
    ElemGeometry g;
    std::string why = elem_geometry(m, perm, 0, g);
    if (!why.empty()) return 1;
    const StateIx im{N, NP, Kp, LAYOUT_MODES}, iv{N, NP, Kp, sizeof(R) == 4 ? LAYOUT_VEC32 : LAYOUT_VEC64};
    std::vector<R> um(im.elems()), uv(iv.elems()), cm(um), cv(uv), om(um), ov(uv), am(um), av(uv);
    std::vector<R> ge(5 * (size_t)Kp), gf(9 * (size_t)Kp), lf(12 * (size_t)Kp), lm(4 * (size_t)Kp);
    std::vector<int> nbr(3 * (size_t)Kp);
    unsigned seed = 12345;
    auto rnd = [&] { return (double)((seed = seed * 1664525u + 1013904223u) >> 8) / (1 << 24) - 0.5; };
    for (int i = 0; i < Kp; i++) {
        const int e = std::min(i, K - 1);
        const double map[5] = {g.xr[e], g.yr[e], g.xs[e], g.ys[e], 1.0 / g.J[e]};
        for (int k = 0; k < 5; k++) ge[k * (size_t)Kp + i] = (R)map[k];
        for (int k = 0; k < 4; k++) lm[4 * (size_t)i + k] = (R)map[k];
        for (int f = 0; f < 3; f++) {
            const double face[3] = {g.fnx[f][e], g.fny[f][e], g.flen[f][e]};
            for (int k = 0; k < 3; k++) {
                gf[(3 * f + k) * (size_t)Kp + i] = (R)face[k];
                lf[4 * ((size_t)f * Kp + i) + k] = (R)face[k];
            }
            const int w = g.nbr[f][e];
            nbr[f * (size_t)Kp + i] = w;
            if (sizeof(R) == 4) memcpy(&lf[4 * ((size_t)f * Kp + i) + 3], &w, 4);
            else lf[4 * ((size_t)f * Kp + i) + 3] = (R)w;
        }
        for (int v = 0; v < N; v++)
            for (int k = 0; k < NP; k++) {
                const R x = (R)((k == 0 ? (v == 0 ? 1.4 : v == 3 ? 3.5 : 0.2) : 0.0) + 0.02 * rnd());
                const R y = (R)rnd();
                um[im.at(v, k, i)] = uv[iv.at(v, k, i)] = x;
                cm[im.at(v, k, i)] = cv[iv.at(v, k, i)] = y;
                am[im.at(v, k, i)] = av[iv.at(v, k, i)] = (R)(y + 0.5);
            }
    }
    std::vector<double> bnd((size_t)g.bfaces.size() * NQ1 * 4, 0.0);
    for (size_t b = 0; b < g.bfaces.size(); b++)
        for (int j = 0; j < NQ1; j++) {
            double* o = &bnd[(b * NQ1 + j) * 4];
            if (g.bfaces[b].kind == BC_REFLECTING) { o[0] = 0.6; o[1] = 0.8; }
            else { o[0] = 1.2; o[1] = 0.3; o[2] = -0.1; o[3] = 2.9; }
        }
    Ctrl ctrl{};
    ctrl.dt = 1e-3;
    ctrl.active = 1;
    StageArgs<R> a{};
    a.u = um.data(); a.c = cm.data(); a.acc = am.data(); a.out = om.data();
    a.geo_e = ge.data(); a.geo_f = gf.data(); a.nbr = nbr.data();
    a.lface = lf.data(); a.lmetric = lm.data();
    a.ctrl = &ctrl; a.lam_bits = &ctrl.lam_bits;
    a.K = K; a.Kp = Kp; a.phys.gamma = 1.4;
    a.bnd = g.bfaces.empty() ? nullptr : bnd.data();
    StageArgs<R> b = a;
    b.u = uv.data(); b.c = cv.data(); b.acc = av.data(); b.out = ov.data();
    std::vector<R> ltab(LaneTab<P>::SIZE);
    for (int i = 0; i < 3; i++) LaneTab<P>::fill(ltab.data(), i, 3);
    const int threads = ((Kp + 127) / 128 + 7) / 8 * 8 * 128;
    bool ok = one<P, R, ST_RHS>(a, b, im, iv, ltab, threads) && one<P, R, ST_RK4_1>(a, b, im, iv, ltab, threads) &&
              one<P, R, ST_RK4_2>(a, b, im, iv, ltab, threads) && one<P, R, ST_RK4_3>(a, b, im, iv, ltab, threads) &&
              one<P, R, ST_RK4_4>(a, b, im, iv, ltab, threads) && one<P, R, ST_RK2_1>(a, b, im, iv, ltab, threads) &&
              one<P, R, ST_RK2_2>(a, b, im, iv, ltab, threads);
    printf("p=%d %s K=%d boundary faces %zu: %s\n", P, sizeof(R) == 8 ? "FP64" : "FP32", K, g.bfaces.size(),
           ok ? "bodies agree" : "BODIES DIFFER");
    return ok ? 0 : 2;
}

template <typename R>
static int by_p(const Mesh& m, int p) {
    return p == 1 ? run<R, 1>(m) : p == 2 ? run<R, 2>(m) : p == 3 ? run<R, 3>(m) : 3;
}

int main(int argc, char** argv) {
    if (argc != 4) return 4;
    fill_tab(c_tab64.p1);
    fill_tab(c_tab64.p2);
    fill_tab(c_tab64.p3);
    fill_tab(c_tab32.p1);
    fill_tab(c_tab32.p2);
    fill_tab(c_tab32.p3);
    Mesh m;
    std::string why = read_pmsh(argv[1], m);
    if (!why.empty()) return 1;
    return atoi(argv[3]) ? by_p<float>(m, atoi(argv[2])) : by_p<double>(m, atoi(argv[2]));
}
