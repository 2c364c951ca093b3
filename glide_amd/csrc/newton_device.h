// newton_device.h - the damped Newton iteration of one cell's five unknowns
// (u_l, u_r, v_t, v_b, H), written for instruction count, and the reciprocal,
// division, exp, log and sigmoid forms it needs.
//
// The iteration is vanka_assemble<0> followed by lu5_solve (vanka_device.h)
// with the same rounding of every value.  A sweep is bound by FP64
// instruction issue (a wave64 FP64 instruction holds its SIMD for 4 cycles, and
// a dependent one can follow after 8, so two waves hide the latency), so what
// pays is to issue fewer of them.  What is left out, and why no bit changes:
//  - factors of 2, 4, 1/2, 1/4 and 1/8: scaling by a power of two is exact, so
//    2 eta H is held instead of eta H, and the factors of the stresses, fluxes
//    and averages ride on the constants 2/dx, 1/(2 dx) and 1/(8 dx);
//  - equal entries: sigma_xx and sigma_yy of the centre cell fill the velocity
//    block with +-t and +-2t, t = 2 eta H / dx^2 (rounded as in the assembly),
//    and the elimination keeps that pattern exactly: rows 2 and 3 hold
//    (B, -B) under row 1 and share C, so 5 entries are updated instead of 9;
//  - values that one cell shares between its faces: H_c + H_nb serves the
//    driving stress and the flux, the cell's drag and surface all four faces;
//  - u - 0.25 d as one fma (0.25 d is exact);
//  - the range handling of divisions, exp and log, whose arguments are in
//    range here (recip, exp_mid, log_normal below).
// 348 FP64 instructions an iteration instead of about 590 (781 VALU in all,
// interior form), 308 where the sigmoid is clamped (newton_iterate).  Measured
// per sweep, 10 iterations, with its apply pass: 32^2 20.2 -> 12.1 us, 512^2
// 65.1 -> 41.6 us; a 512^2 step to 1e-8 82.8 -> 56.8 ms.
// Terms that vanish at the domain edge are multiplied by a factor held per
// cell (1/(2 dx) or 0 per face, 1/dx or 0 per vertex), constants where the
// whole tile is interior.  The only differences from the assembly are signs of
// zeros, and non-finite states (which make the residual norm non-finite
// either way).
//
// Compiled for the host too (plain divisions there), where the tests compare
// it with the assembly bit by bit.
#pragma once

#include "vanka_device.h"

namespace glide {

// y refined to the accuracy that the division sequences below start from.
// These are the compiler's own FP64 division (v_rcp_f64, two Newton steps, a
// quotient and its correction) without v_div_scale and v_div_fixup, so the
// results are the correctly rounded ones for normal operands and quotients
// away from the exponent limits.  Measured in a chain on one wave: 58-71
// cycles for a division, 41-46 for recip.
__host__ __device__ __forceinline__ double recip_refined(double d)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(d);
    y = fma(y, fma(-d, y, 1.0), y);
    return fma(y, fma(-d, y, 1.0), y);
#else
    return 1.0 / d;
#endif
}
// n / d with y = recip_refined(d)
__host__ __device__ __forceinline__ double div_refined(double n, double d, double y)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double q = n * y;
    return fma(fma(-d, q, n), y, q);
#else
    (void)y;
    return n / d;
#endif
}
__host__ __device__ __forceinline__ double recip(double d)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = recip_refined(d);
    return fma(fma(-d, y, 1.0), y, y);
#else
    return 1.0 / d;
#endif
}

// dm_exp for |x| <= 700 (no special values, a normal result): the same
// reduction and polynomial, the scaling by 2^k in one instruction.
__host__ __device__ __forceinline__ double exp_mid(double x)
{
    const double kd = DM_FLOOR(fma(x, 1.4426950408889634, 0.5));
    const int k = (int)kd;
    const double r = fma(-kd, 4.7493250390316726e-07, fma(-kd, 0.6931467056274414, x));
    const double r2 = r * r;
    const double q0 = r + 1.0;
    const double q1 = fma(r, 0.16666666666666666, 0.5);
    const double q2 = fma(r, 0.008333333333333333, 0.041666666666666664);
    const double q3 = fma(r, 0.0001984126984126984, 0.001388888888888889);
    const double q4 = fma(r, 2.7557319223985893e-06, 2.48015873015873e-05);
    const double q5 = fma(r, 2.505210838544172e-08, 2.755731922398589e-07);
    const double q6 = fma(r, 1.6059043836821613e-10, 2.08767569878681e-09);
    const double r4 = r2 * r2;
    const double s0 = fma(r2, q1, q0);
    const double s1 = fma(r2, q3, q2);
    const double s2 = fma(r2, q5, q4);
    const double r8 = r4 * r4;
    const double t0 = fma(r4, s1, s0);
    const double t1 = fma(r4, q6, s2);
    const double p = fma(r8, t1, t0);
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ldexp(p, k);
#else
    return p * dm_pow2i(k);
#endif
}

// dm_log for normal, finite x > 0
__host__ __device__ __forceinline__ double log_normal(double x)
{
    const uint64_t b = dm_to_bits(x);
    int e = (int)(b >> 52) - 1023;
    double m = dm_from_bits((b & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL);
    const bool up = m > 1.4142135623730951;
    m = up ? m * 0.5 : m;
    e = up ? e + 1 : e;
    const double f = m - 1.0;
    const double d = 2.0 + f;
    const double s = div_refined(f, d, recip_refined(d));
    const double z = s * s;
    const double z2 = z * z;
    const double a0 = fma(z, 0.4, 0.6666666666666666);
    const double a1 = fma(z, 0.2222222222222222, 0.2857142857142857);
    const double a2 = fma(z, 0.15384615384615385, 0.18181818181818182);
    const double a3 = fma(z, 0.11764705882352941, 0.13333333333333333);
    const double a4 = fma(z, 0.09523809523809523, 0.10526315789473684);
    const double a5 = 0.08695652173913043;
    const double z4 = z2 * z2;
    const double b0 = fma(z2, a1, a0);
    const double b1 = fma(z2, a3, a2);
    const double b2 = fma(z2, a5, a4);
    const double z8 = z4 * z4;
    const double c0 = fma(z4, b1, b0);
    const double Q = z * fma(z8, b2, c0);
    const double hfsq = 0.5 * f * f;
    const double lm = f - fma(-s, hfsq + Q, hfsq);
    const double ed = (double)e;
    return fma(ed, 0.6931467056274414, fma(ed, 4.7493250390316726e-07, lm));
}

// dm_pow(x, p) for x >= 0: the short forms where x is normal and |p log x| <= 700
__host__ __device__ __forceinline__ double pow_pos(double x, double p)
{
    const double y = p * log_normal(x);
    double r = exp_mid(y);
    if (!(x >= 2.2250738585072014e-308 && x <= 1.7976931348623157e308 && fabs(y) <= 700.0)) r = dm_pow(x, p);
    return r;
}

// sigm (ssa_device.h): the clamped argument keeps exp in range and 1 + exp in [1, 4.9e8]
__host__ __device__ __forceinline__ double sigm_mid(double z, double c)
{
    const double s = fmin(fmax(c * z, -20.0), 20.0);
    return recip(1.0 + exp_mid(-s));
}
// sigm where the argument reaches the clamp (a NaN counts as -20, as in sigm):
// 1 / (1 + e^-20) and 1 / (1 + e^20)
__host__ __device__ __forceinline__ bool sigm_clamped(double z, double c) { return !(fabs(c * z) < 20.0); }
__host__ __device__ __forceinline__ double sigm_end(double z, double c)
{
    return c * z > 0.0 ? 0x1.ffffffee4b79ap-1 : 0x1.1b4865556b5d5p-29;
}

// a value that is the same in every lane, held in scalar registers
__host__ __device__ __forceinline__ double uniform(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t b = dm_to_bits(x);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return dm_from_bits((uint64_t)hi << 32 | lo);
#else
    return x;
#endif
}

// constants of a level
struct NewtonK {
    double dxi, dxi2, hdx, edx;   // 1/dx, 2/dx, 1/(2 dx), 1/(8 dx)
    double dt, rdt, idt;          // dt, recip_refined(dt), 1/dt
};
__host__ __device__ __forceinline__ NewtonK newton_constants(double dx, double dt)
{
    NewtonK K;
    K.dxi = uniform(1.0 / dx);
    K.dxi2 = uniform(2.0 * K.dxi);
    K.hdx = uniform(0.5 * K.dxi);
    K.edx = uniform(0.125 * K.dxi);
    K.dt = dt;
    K.rdt = uniform(recip_refined(dt));
    K.idt = uniform(1.0 / dt);
    return K;
}

// What the cell's iteration reads besides its unknowns.  n_* = 2 eta H of the
// neighbours, S_* their surface max(bed, -0.917 H) + H, be_* their drag
// g beta + (1 - g) water_drag.
struct NewtonCell {
    double e2;                      // 2 eta of the cell
    double n_l, n_r, n_t, n_b;
    double p_tl, p_tr, n_bl, n_br;  // (n_tl + n_t) + n_l, n_t + n_tr
    double H_l, H_r, H_t, H_b;
    double S_l, S_r, S_t, S_b;
    double be_l, be_r, be_t, be_b;
    double bed, beta, th;
    double u_ll, u_rr, u_tl, u_tr, u_bl, u_br, c_l, c_r, d_t, d_b;   // c_l = (v_lt - v_lb)/dx, d_t = u_tr - u_tl
    double v_lt, v_lb, v_rt, v_rb, v_tt, v_bb;
    double f0, f1, f2, f3, f4;
    double F_l, F_r, F_t, F_b;      // 1/(2 dx), or 0 on a face of the domain edge
    double V_tl, V_tr, V_bl, V_br;  // 1/dx, or 0 on a vertex of the domain edge
};

// edge factors of cell (i, j); interior tiles take the constants
template <bool INTERIOR>
__host__ __device__ __forceinline__ void newton_edges(NewtonCell &C, const NewtonK &K, int i, int j, int ny, int nx)
{
    const bool l = INTERIOR || j > 0, r = INTERIOR || j + 1 < nx, t = INTERIOR || i > 0, b = INTERIOR || i + 1 < ny;
    C.F_l = l ? K.hdx : 0.0;
    C.F_r = r ? K.hdx : 0.0;
    C.F_t = t ? K.hdx : 0.0;
    C.F_b = b ? K.hdx : 0.0;
    C.V_tl = t && l ? K.dxi : 0.0;
    C.V_tr = t && r ? K.dxi : 0.0;
    C.V_bl = b && l ? K.dxi : 0.0;
    C.V_br = b && r ? K.dxi : 0.0;
}

struct NewtonX {
    double u_l, u_r, v_t, v_b, H;
};

// What the cell's own thickness gives: drag, surface and its slope, calving rate
// times (1 - g), d mass row / d H without the fluxes, d drag / d H.
struct NewtonCentre {
    double be, S, sl, cal, qH, db;
};
// CLAMPED: the cell's sigmoid argument reaches its clamp; GL: p.gl_derivatives
template <bool CLAMPED, bool GL>
__host__ __device__ __forceinline__ NewtonCentre newton_centre(const NewtonCell &C, const NewtonK &K, const Params &p, double H)
{
    NewtonCentre M;
    const double z = fma(0.917, H, C.bed);
    const double g = CLAMPED ? sigm_end(z, p.gl_c) : sigm_mid(z, p.gl_c);
    const double g1 = 1.0 - g;
    M.be = fma(g, C.beta, g1 * p.water_drag);
    const double Hf = -0.917 * H;
    M.S = fmax(C.bed, Hf) + H;
    M.sl = C.bed > Hf ? 1.0 : 1.0 + -0.917;   // 1 + d base / d H
    M.cal = p.calving_rate * g1;
    M.qH = K.idt + M.cal;
    M.db = 0.0;
    if (GL) {
        const double dg = 0.917 * (p.gl_c * g * g1);
        M.qH = K.idt - fma(p.calving_rate * H, dg, -M.cal);
        M.db = dg * (C.beta - p.water_drag);
    }
    return M;
}

// The block [[a0, t2, t, -t, c0], [t2, a1, -t, t, c1], [t, -t, a2, t2, c2],
// [-t, t, t2, a3, c3], [q0, q1, q2, q3, qH]] and its right-hand side
struct NewtonSystem {
    double a0, a1, a2, a3, t, c0, c1, c2, c3, q0, q1, q2, q3, qH;
    double r0, r1, r2, r3, r4;
};
// ADJ: the block alone, its mass row the identity where `masked`
template <bool GL, bool ADJ>
__host__ __device__ __forceinline__ NewtonSystem newton_system(const NewtonCell &C, const NewtonK &K, const NewtonCentre &M,
                                                              const NewtonX &x, bool masked)
{
    const double u_l = x.u_l, u_r = x.u_r, v_t = x.v_t, v_b = x.v_b, H = x.H;
    const double be = M.be, S = M.S, sl = M.sl;
    // mass row (J20..J23 = q0..q3, J24 = qH): H/dt, calving, the four upwind fluxes
    double r4 = div_refined(H, K.dt, K.rdt) - C.f4;
    double qH = M.qH;
    r4 = r4 + M.cal * H;
    const double s_l = C.H_l + H, s_r = H + C.H_r, s_t = C.H_t + H, s_b = H + C.H_b;
    double q0, q1, q2, q3;
    {   // twice the flux and its derivatives; the factors F carry 1/(2 dx)
        const double d = H - C.H_l, f = fma(s_l, u_l, -(fabs(u_l) * d));
        q0 = fma(copysign(1.0, u_l), d, -s_l) * C.F_l;
        qH = fma(-(u_l - fabs(u_l)), C.F_l, qH);
        r4 = fma(-f, C.F_l, r4);
    }
    {
        const double d = C.H_r - H, f = fma(s_r, u_r, -(fabs(u_r) * d));
        q1 = -fma(copysign(1.0, u_r), d, -s_r) * C.F_r;
        qH = fma(u_r + fabs(u_r), C.F_r, qH);
        r4 = fma(f, C.F_r, r4);
    }
    {
        const double d = C.H_t - H, f = fma(s_t, v_t, -(fabs(v_t) * d));
        q2 = -fma(copysign(1.0, v_t), d, -s_t) * C.F_t;
        qH = fma(v_t + fabs(v_t), C.F_t, qH);
        r4 = fma(f, C.F_t, r4);
    }
    {
        const double d = H - C.H_b, f = fma(s_b, v_b, -(fabs(v_b) * d));
        q3 = fma(copysign(1.0, v_b), d, -s_b) * C.F_b;
        qH = fma(-(v_b - fabs(v_b)), C.F_b, qH);
        r4 = fma(-f, C.F_b, r4);
    }
    if (ADJ ? masked : (H - K.dt * r4) <= C.th) {
        q0 = q1 = q2 = q3 = 0.0;
        qH = 1.0;
        r4 = H - C.th;
    }

    // momentum rows: right-hand sides r0..r3, diagonals a0..a3, H column c0..c3
    double r0 = -C.f0, r1 = -C.f1, r2 = -C.f2, r3 = -C.f3;
    const double n = H * C.e2;   // 2 eta H
    const double t = (n * K.dxi) * K.dxi, t2 = t + t;
    double a0 = -t2, a1 = -t2, a2 = -t2, a3 = -t2;
    double c0, c1, c2, c3;
    {   // sigma_xx, sigma_yy of the cell
        const double du = u_r - u_l, dv = v_t - v_b;
        const double ex = fma(du, K.dxi2, dv * K.dxi), ey = fma(du, K.dxi, dv * K.dxi2);
        const double sx = n * ex, sy = n * ey;
        r0 = fma(sx, K.dxi, r0);
        r1 = fma(-sx, K.dxi, r1);
        r2 = fma(-sy, K.dxi, r2);
        r3 = fma(sy, K.dxi, r3);
        const double jx = (ex * C.e2) * K.dxi, jy = (ey * C.e2) * K.dxi;
        c0 = jx;
        c1 = -jx;
        c2 = -jy;
        c3 = jy;
    }
    {   // ... of the four neighbours
        const double s = C.n_l * fma(u_l - C.u_ll, K.dxi2, C.c_l);
        r0 = fma(-s, K.dxi, r0);
        a0 = fma(-(C.n_l * K.dxi), K.dxi2, a0);
    }
    {
        const double s = C.n_r * fma(C.u_rr - u_r, K.dxi2, C.c_r);
        r1 = fma(s, K.dxi, r1);
        a1 = fma(-(C.n_r * K.dxi), K.dxi2, a1);
    }
    {
        const double s = C.n_t * fma(C.d_t, K.dxi, (C.v_tt - v_t) * K.dxi2);
        r2 = fma(s, K.dxi, r2);
        a2 = fma(-(C.n_t * K.dxi), K.dxi2, a2);
    }
    {
        const double s = C.n_b * fma(C.d_b, K.dxi, (v_b - C.v_bb) * K.dxi2);
        r3 = fma(-s, K.dxi, r3);
        a3 = fma(-(C.n_b * K.dxi), K.dxi2, a3);
    }
    // sigma_xy of the four vertices: e = 2 eps_xy, m = 8 eta H
    {   // top left
        const double e = fma(C.u_tl - u_l, C.V_tl, (v_t - C.v_lt) * C.V_tl), m = C.p_tl + n;
        const double s = m * e, d = m * C.V_tl, h = e * C.e2;
        r0 = fma(s, K.edx, r0);
        a0 = fma(-d, K.edx, a0);
        c0 = fma(h, K.edx, c0);
        r2 = fma(-s, K.edx, r2);
        a2 = fma(-d, K.edx, a2);
        c2 = fma(-h, K.edx, c2);
    }
    {   // top right
        const double e = fma(C.u_tr - u_r, C.V_tr, (C.v_rt - v_t) * C.V_tr), m = (C.p_tr + n) + C.n_r;
        const double s = m * e, d = m * C.V_tr, h = e * C.e2;
        r1 = fma(s, K.edx, r1);
        a1 = fma(-d, K.edx, a1);
        c1 = fma(h, K.edx, c1);
        r2 = fma(s, K.edx, r2);
        a2 = fma(-d, K.edx, a2);
        c2 = fma(h, K.edx, c2);
    }
    {   // bottom left
        const double e = fma(u_l - C.u_bl, C.V_bl, (v_b - C.v_lb) * C.V_bl), m = ((C.n_l + n) + C.n_bl) + C.n_b;
        const double s = m * e, d = m * C.V_bl, h = e * C.e2;
        r0 = fma(-s, K.edx, r0);
        a0 = fma(-d, K.edx, a0);
        c0 = fma(-h, K.edx, c0);
        r3 = fma(-s, K.edx, r3);
        a3 = fma(-d, K.edx, a3);
        c3 = fma(-h, K.edx, c3);
    }
    {   // bottom right
        const double e = fma(u_r - C.u_br, C.V_br, (C.v_rb - v_b) * C.V_br), m = ((n + C.n_r) + C.n_b) + C.n_br;
        const double s = m * e, d = m * C.V_br, h = e * C.e2;
        r1 = fma(-s, K.edx, r1);
        a1 = fma(-d, K.edx, a1);
        c1 = fma(-h, K.edx, c1);
        r3 = fma(s, K.edx, r3);
        a3 = fma(-d, K.edx, a3);
        c3 = fma(h, K.edx, c3);
    }
    {   // basal drag
        const double b_l = C.be_l + be, b_r = be + C.be_r, b_t = C.be_t + be, b_b = be + C.be_b;
        r0 = fma(-0.5, b_l * u_l, r0);
        a0 = fma(-0.5, b_l, a0);
        r1 = fma(-0.5, b_r * u_r, r1);
        a1 = fma(-0.5, b_r, a1);
        r2 = fma(-0.5, b_t * v_t, r2);
        a2 = fma(-0.5, b_t, a2);
        r3 = fma(-0.5, b_b * v_b, r3);
        a3 = fma(-0.5, b_b, a3);
        if (GL) {
            c0 = c0 + -0.5 * M.db * u_l;
            c1 = c1 + -0.5 * M.db * u_r;
            c2 = c2 + -0.5 * M.db * v_t;
            c3 = c3 + -0.5 * M.db * v_b;
        }
    }
    {   // driving stress
        const double d_l = S - C.S_l, d_r = C.S_r - S, d_t = C.S_t - S, d_b = S - C.S_b;
        r0 = r0 - (s_l * d_l) * C.F_l;
        c0 = c0 - fma(s_l * sl, C.F_l, d_l * C.F_l);
        r1 = r1 - (s_r * d_r) * C.F_r;
        c1 = c1 - fma(-(s_r * sl), C.F_r, d_r * C.F_r);
        r2 = r2 - (s_t * d_t) * C.F_t;
        c2 = c2 - fma(-(s_t * sl), C.F_t, d_t * C.F_t);
        r3 = r3 - (s_b * d_b) * C.F_b;
        c3 = c3 - fma(s_b * sl, C.F_b, d_b * C.F_b);
    }
    return {a0, a1, a2, a3, t, c0, c1, c2, c3, q0, q1, q2, q3, qH, r0, r1, r2, r3, r4};
}

// x = A^-1 r as lu5_solve takes it
__host__ __device__ __forceinline__ void newton_solve(const NewtonSystem &A, double &x0, double &x1, double &x2, double &x3,
                                                      double &x4)
{
    const double t = A.t, t2 = t + t, a0 = A.a0, c0 = A.c0, r0 = A.r0;
    double a1 = A.a1, a2 = A.a2, a3 = A.a3, c1 = A.c1, c2 = A.c2, c3 = A.c3, q1 = A.q1, q2 = A.q2, q3 = A.q3, qH = A.qH;
    const double i0 = recip(a0);
    const double m = t * i0, m2 = m + m, l0 = A.q0 * i0;   // column 0 below a0: m2, m, -m, l0
    a1 = fma(-m2, t2, a1);
    const double B = fma(-m2, t, -t);
    c1 = fma(-m2, c0, c1);
    a2 = fma(-m, t, a2);
    const double Cc = fma(m, t, t2);
    c2 = fma(-m, c0, c2);
    a3 = fma(-m, t, a3);
    c3 = fma(m, c0, c3);
    q1 = fma(-l0, t2, q1);
    q2 = fma(-l0, t, q2);
    q3 = fma(l0, t, q3);
    qH = fma(-l0, c0, qH);
    const double i1 = recip(a1);
    const double k = B * i1, l1 = q1 * i1;               // column 1: k, -k, l1
    a2 = fma(-k, B, a2);
    const double D = fma(k, B, Cc);
    c2 = fma(-k, c1, c2);
    a3 = fma(-k, B, a3);
    c3 = fma(k, c1, c3);
    q2 = fma(-l1, B, q2);
    q3 = fma(l1, B, q3);
    qH = fma(-l1, c1, qH);
    const double i2 = recip(a2);
    const double w = D * i2, l2 = q2 * i2;
    a3 = fma(-w, D, a3);
    c3 = fma(-w, c2, c3);
    q3 = fma(-l2, D, q3);
    qH = fma(-l2, c2, qH);
    const double i3 = recip(a3);
    const double l3 = q3 * i3;
    qH = fma(-l3, c3, qH);
    const double i4 = recip(qH);
    const double y1 = fma(-m2, r0, A.r1);
    const double y2 = fma(-k, y1, fma(-m, r0, A.r2));
    const double y3 = fma(-w, y2, fma(k, y1, fma(m, r0, A.r3)));
    const double y4 = fma(-l3, y3, fma(-l2, y2, fma(-l1, y1, fma(-l0, r0, A.r4))));
    x4 = y4 * i4;
    x3 = fma(-c3, x4, y3) * i3;
    x2 = fma(-D, x3, fma(-c2, x4, y2)) * i2;
    x1 = fma(-B, x2, fma(B, x3, fma(-c1, x4, y1))) * i1;
    x0 = fma(-t2, x1, fma(-t, x2, fma(t, x3, fma(-c0, x4, r0)))) * i0;
}

// One damped iteration x -= 0.25 A^-1 r, H = max(H, th)
template <bool CLAMPED, bool GL>
__host__ __device__ __forceinline__ void newton_step(const NewtonCell &C, const NewtonK &K, const Params &p, NewtonX &x)
{
    NewtonSystem A = newton_system<GL, false>(C, K, newton_centre<CLAMPED, GL>(C, K, p, x.H), x, false);
    A.a0 = A.a0 - 1.0;
    A.a1 = A.a1 - 1.0;
    A.a2 = A.a2 - 1.0;
    A.a3 = A.a3 - 1.0;
    A.qH = A.qH + 1.0;
    double x0, x1, x2, x3, x4;
    newton_solve(A, x0, x1, x2, x3, x4);
    x.u_l = fma(-0.25, x0, x.u_l);
    x.u_r = fma(-0.25, x1, x.u_r);
    x.v_t = fma(-0.25, x2, x.v_t);
    x.v_b = fma(-0.25, x3, x.v_b);
    x.H = fmax(fma(-0.25, x4, x.H), C.th);
}

// d = A^-T r of the adjoint block (vanka_assemble<1>): the velocity block is
// symmetric, so the transpose swaps the H column and the mass row.
template <bool GL>
__host__ __device__ __forceinline__ void newton_adjoint(const NewtonCell &C, const NewtonK &K, const NewtonCentre &M,
                                                        const NewtonX &x, bool masked, const double r[5], double d[5])
{
    const NewtonSystem A = newton_system<GL, true>(C, K, M, x, masked);
    newton_solve({A.a0, A.a1, A.a2, A.a3, A.t, A.q0, A.q1, A.q2, A.q3, A.c0, A.c1, A.c2, A.c3, A.qH, r[0], r[1], r[2], r[3], r[4]},
                 d[0], d[1], d[2], d[3], d[4]);
}

// n_newton iterations.  Ice 200 m above or below flotation (at the default
// sharpness) has its sigmoid clamped; where every lane of the wave has, which
// is most of a sheet, an iteration takes the clamped form's 5 instructions for
// the 40 of exp and division.  The branch selects whole iterations, so that each form is
// scheduled as one block: the sigmoid's chain hides among the rest of the
// assembly (as a branch of its own it cost waves at a grounding line 1.4%).
// Ten sweeps of 1024^2: 1632 -> 1480 us.
// AHEAD: the wave's issue priority rises half way (vanka_fold_tile).
template <bool AHEAD = false>
__host__ __device__ __forceinline__ void newton_iterate(const NewtonCell &C, const NewtonK &K, const Params &p, int n_newton,
                                               NewtonX &x)
{
    if (p.gl_derivatives) {
        for (int k = 0; k < n_newton; k++) newton_step<false, true>(C, K, p, x);
        return;
    }
    for (int k = 0; k < n_newton; k++) {
#if defined(__HIP_DEVICE_COMPILE__)
        if (AHEAD && 2 * k >= n_newton) __builtin_amdgcn_s_setprio(2);
#endif
        bool clamped = sigm_clamped(fma(0.917, x.H, C.bed), p.gl_c);
#if defined(__HIP_DEVICE_COMPILE__)
        clamped = __builtin_amdgcn_ballot_w64(!clamped) == 0;
#endif
        if (clamped)
            newton_step<true, false>(C, K, p, x);
        else
            newton_step<false, false>(C, K, p, x);
    }
}

}  // namespace glide
