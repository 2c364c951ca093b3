// Host check of the short Newton iteration (newton_device.h) against the
// general assembly and LU (vanka_device.h): cells of several grids, on the
// edges, corners and inside, with grounded, floating and thickness-limited
// states, both grounding-derivative modes and both signs of every velocity,
// must take the same iterates; exp_mid, log_normal, pow_pos and sigm_mid must
// return the bits of the general forms.  Prints "ok <cells>" or the first
// mismatch.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

#define __host__
#define __device__
#define __forceinline__ inline
#define __restrict__
#include "glide_hip.h"
#include "newton_device.h"

using namespace glide;

static bool same(double a, double b) { return a == b || (a != a && b != b); }

static int functions()
{
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    for (int k = 0; k < 200000; k++) {
        const double x = (2.0 * U(rng) - 1.0) * 700.0;
        if (!same(exp_mid(x), dm_exp(x))) return std::printf("exp_mid(%.17g)\n", x), 1;
        const double y = std::ldexp(1.0 + U(rng), (int)(U(rng) * 2040) - 1020);
        if (!same(log_normal(y), dm_log(y))) return std::printf("log_normal(%.17g)\n", y), 1;
        for (double q : {-1.0 / 3.0, -4.0 / 3.0, 2.5, -300.0})
            if (!same(pow_pos(y, q), dm_pow(y, q))) return std::printf("pow_pos(%.17g, %g)\n", y, q), 1;
        const double z = (2.0 * U(rng) - 1.0) * 400.0;
        if (!same(sigm_mid(z, 0.1), sigm(z, 0.1))) return std::printf("sigm_mid(%.17g)\n", z), 1;
    }
    const double xs[] = {0.0, 1.0, 5e-324, 2.2250738585072014e-308, 1.7976931348623157e308, INFINITY, NAN, 1.4142135623730951};
    for (double x : xs)
        for (double q : {-1.0 / 3.0, 0.0, 2.0, -2.0})
            if (!same(pow_pos(x, q), dm_pow(x, q))) return std::printf("pow_pos(%g, %g)\n", x, q), 1;
    for (double z : {0.0, 1e9, -1e9, (double)NAN, (double)INFINITY})
        if (!same(sigm_mid(z, 0.1), sigm(z, 0.1))) return std::printf("sigm_mid(%g)\n", z), 1;
    for (double z : {200.0, -200.0, 1e9, -1e9, (double)NAN, (double)INFINITY, -(double)INFINITY})
        if (!sigm_clamped(z, 0.1) || !same(sigm_end(z, 0.1), sigm(z, 0.1))) return std::printf("sigm_end(%g)\n", z), 1;
    if (sigm_clamped(199.99, 0.1) || sigm_clamped(-199.99, 0.1)) return std::printf("sigm_clamped\n"), 1;
    return 0;
}

int main()
{
    if (functions()) return 1;
    std::mt19937_64 rng(99);
    std::uniform_real_distribution<double> U(0.5, 2.0), S(-1.0, 1.0), P(0.0, 1.0);
    const int sizes[][2] = {{2, 2}, {2, 9}, {3, 3}, {4, 7}, {16, 16}, {33, 20}};
    long cells = 0, limited = 0, floating = 0, clamped = 0;
    for (int gl = 0; gl < 2; gl++)
        for (double dt : {1.0, 10.0, 0.3})
            for (auto &sz : sizes) {
                const Params p{3.0, 1e-5, 1e-3, 1.0, 0.1, gl};
                const int ny = sz[0], nx = sz[1];
                const double dx = 1500.0, dxi = 1.0 / dx;
                for (int i = 0; i < ny; i++)
                    for (int j = 0; j < nx; j++)
                        for (int rep = 0; rep < 4; rep++) {
                            CellNbhd N;
                            double *d = reinterpret_cast<double *>(&N);
                            for (size_t k = 0; k < sizeof(CellNbhd) / sizeof(double); k++) d[k] = 0.0;
                            // viscosities: 0 outside the domain
                            auto eta = [&](int a, int b) {
                                return i + a < 0 || i + a >= ny || j + b < 0 || j + b >= nx ? 0.0 : 200.0 * U(rng);
                            };
                            N.e_c = eta(0, 0); N.e_l = eta(0, -1); N.e_r = eta(0, 1); N.e_t = eta(-1, 0); N.e_b = eta(1, 0);
                            N.e_tl = eta(-1, -1); N.e_tr = eta(-1, 1); N.e_bl = eta(1, -1); N.e_br = eta(1, 1);
                            auto thick = [&]() { return P(rng) < 0.3 ? 0.1 + P(rng) : 400.0 * U(rng); };
                            N.H_l = thick(); N.H_r = thick(); N.H_t = thick(); N.H_b = thick();
                            N.H_tl = thick(); N.H_tr = thick(); N.H_bl = thick(); N.H_br = thick();
                            auto bed = [&]() { return 600.0 * S(rng) - 200.0; };
                            N.bed_c = bed(); N.bed_l = bed(); N.bed_r = bed(); N.bed_t = bed(); N.bed_b = bed();
                            N.beta_c = U(rng); N.beta_l = U(rng); N.beta_r = U(rng); N.beta_t = U(rng); N.beta_b = U(rng);
                            double *vel[] = {&N.u_ll, &N.u_rr, &N.u_tl, &N.u_tr, &N.u_bl, &N.u_br,
                                             &N.v_lt, &N.v_lb, &N.v_rt, &N.v_rb, &N.v_tt, &N.v_bb};
                            for (double *q : vel) *q = 80.0 * S(rng);
                            N.f0 = S(rng); N.f1 = S(rng); N.f2 = rep == 0 ? 0.0 : S(rng); N.f3 = S(rng); N.f4 = 100.0 * S(rng);
                            nbhd_grounding(N, p);
                            const NewtonK K = newton_constants(dx, dt);
                            NewtonCell C;
                            C.e2 = 2.0 * N.e_c;
                            C.n_l = 2.0 * N.e_l * N.H_l; C.n_r = 2.0 * N.e_r * N.H_r;
                            C.n_t = 2.0 * N.e_t * N.H_t; C.n_b = 2.0 * N.e_b * N.H_b;
                            C.p_tl = (2.0 * N.e_tl * N.H_tl + C.n_t) + C.n_l;
                            C.p_tr = C.n_t + 2.0 * N.e_tr * N.H_tr;
                            C.n_bl = 2.0 * N.e_bl * N.H_bl; C.n_br = 2.0 * N.e_br * N.H_br;
                            auto surf = [](double b, double H) { return fmax(b, -0.917 * H) + H; };
                            auto drag = [&](const Ground &g, double beta) { return fma(g.g, beta, (1.0 - g.g) * p.water_drag); };
                            C.H_l = N.H_l; C.H_r = N.H_r; C.H_t = N.H_t; C.H_b = N.H_b;
                            C.S_l = surf(N.bed_l, N.H_l); C.S_r = surf(N.bed_r, N.H_r);
                            C.S_t = surf(N.bed_t, N.H_t); C.S_b = surf(N.bed_b, N.H_b);
                            C.be_l = drag(N.g_l, N.beta_l); C.be_r = drag(N.g_r, N.beta_r);
                            C.be_t = drag(N.g_t, N.beta_t); C.be_b = drag(N.g_b, N.beta_b);
                            C.bed = N.bed_c; C.beta = N.beta_c;
                            C.u_ll = N.u_ll; C.u_rr = N.u_rr; C.u_tl = N.u_tl; C.u_tr = N.u_tr; C.u_bl = N.u_bl; C.u_br = N.u_br;
                            C.v_lt = N.v_lt; C.v_lb = N.v_lb; C.v_rt = N.v_rt; C.v_rb = N.v_rb; C.v_tt = N.v_tt; C.v_bb = N.v_bb;
                            C.c_l = (N.v_lt - N.v_lb) * dxi; C.c_r = (N.v_rt - N.v_rb) * dxi;
                            C.d_t = N.u_tr - N.u_tl; C.d_b = N.u_br - N.u_bl;
                            C.f0 = N.f0; C.f1 = N.f1; C.f2 = N.f2; C.f3 = N.f3; C.f4 = N.f4;
                            const double th = rep == 1 ? 300.0 : 0.1;
                            C.th = th;
                            if (i >= 1 && i < ny - 1 && j >= 1 && j < nx - 1 && rep >= 2)
                                newton_edges<true>(C, K, i, j, ny, nx);
                            else
                                newton_edges<false>(C, K, i, j, ny, nx);
                            NewtonX x{60 * S(rng), 60 * S(rng), 60 * S(rng), 60 * S(rng), fmax(thick(), th)};
                            NewtonX y = x;
                            for (int it = 0; it < 6; it++) {
                                double J[25], r[5], e[5];
                                vanka_assemble<0>(N, p, i, j, ny, nx, dxi, dt, y.u_l, y.u_r, y.v_t, y.v_b, y.H, th, false, J, r);
                                limited += J[20] == 0.0 && J[21] == 0.0 && J[24] == 2.0;
                                floating += N.bed_c < -0.917 * y.H;
                                clamped += sigm_clamped(fma(0.917, y.H, N.bed_c), p.gl_c);
                                lu5_solve(J, r, e);
                                y.u_l -= 0.25 * e[0];
                                y.u_r -= 0.25 * e[1];
                                y.v_t -= 0.25 * e[2];
                                y.v_b -= 0.25 * e[3];
                                y.H -= 0.25 * e[4];
                                y.H = fmax(y.H, th);
                                newton_iterate(C, K, p, 1, x);
                                if (!same(x.u_l, y.u_l) || !same(x.u_r, y.u_r) || !same(x.v_t, y.v_t) ||
                                    !same(x.v_b, y.v_b) || !same(x.H, y.H)) {
                                    std::printf("cell (%d, %d) of %d x %d, gl %d, iteration %d: %.17g %.17g %.17g %.17g %.17g, "
                                                "not %.17g %.17g %.17g %.17g %.17g\n", i, j, ny, nx, gl, it, x.u_l, x.u_r, x.v_t,
                                                x.v_b, x.H, y.u_l, y.u_r, y.v_t, y.v_b, y.H);
                                    return 1;
                                }
                            }
                            cells++;
                        }
            }
    if (limited < 100 || floating < 100 || clamped < 100 || clamped > 6 * cells - 100) {
        std::printf("%ld limited, %ld floating, %ld clamped of %ld iterations\n", limited, floating, clamped, 6 * cells);
        return 1;
    }
    std::printf("ok %ld\n", cells);
    return 0;
}
