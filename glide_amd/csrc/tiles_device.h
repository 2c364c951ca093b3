// tiles_device.h - tile bodies shared by the single-level and the batched
// (ensemble) kernels: the cell-viscosity LDS tile, the residual stencil, the
// forward Vanka smoother, its gather-apply pass and the local-smoother block
// activation.  Each body works on one (bx, by) tile of TX x TY points or
// cells with a (TX, TY) thread block, so a kernel may run it once per
// workgroup (one tile per block) or in a loop over many tiles (persistent
// batched launches).  The per-point arithmetic does not depend on the tile
// shape, so every shape gives bitwise-identical results.
#pragma once

#include "newton_device.h"

namespace glide {

// records msg as glide_last_error() and returns code (host side)
int set_error(int code, const char *msg);

constexpr int RB = 14;  // reference launch-block interior (glide/grid.py:184-186)
constexpr int NXCD = 8; // XCDs per MI355X

__host__ __device__ inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// Persistent tile loop.  With at least as many workgroups as tiles each
// workgroup runs tile blockIdx.x (the hardware dispatcher balances them).
// Otherwise workgroups loop over tiles: workgroups are dispatched round-robin
// over the XCDs (workgroup b runs on XCD b % 8), the tiles are cut into chunks
// of up to TCH consecutive tiles (neighbours sharing halo rows; smaller when
// there are few tiles, so every XCD gets at least two chunks) dealt
// round-robin to the XCDs, and each XCD's workgroups walk its chunks' tiles.
// Halos then meet in one L2 while work clustered in space (the local
// smoother's active blocks) still spreads over all XCDs.  The launch must
// have at least 8 workgroups.
constexpr int TCH = 8;
__host__ __device__ inline int tile_chunk(int total)
{
    const int tch = total / (2 * NXCD);
    return tch < 1 ? 1 : tch > TCH ? TCH : tch;
}

__host__ __device__ inline size_t n_u(int ny, int nx) { return (size_t)ny * (nx + 1); }
__host__ __device__ inline size_t n_v(int ny, int nx) { return (size_t)(ny + 1) * nx; }
__host__ __device__ inline size_t n_c(int ny, int nx) { return (size_t)ny * nx; }
__host__ __device__ inline size_t n_t(int ny, int nx) { return n_u(ny, nx) + n_v(ny, nx) + n_c(ny, nx); }

// Byte offsets of a tile's neighbourhood in a row-major field of `cols` columns:
// a base that is the same for the whole tile (row rb, column cb) and 32-bit
// offsets from it, so an access is one instruction (scalar base plus vector
// offset) where 64-bit element arithmetic took four to six.  (r, c) must not
// lie before (rb, cb) and at most 2^16 columns times some 20 rows after it.
struct TileField {
    uint32_t pitch;
    size_t org;
    __device__ __forceinline__ TileField(int cols, int rb, int cb) : pitch(8u * (uint32_t)cols), org((size_t)rb * cols + cb) {}
    __device__ __forceinline__ const char *base(const double *a) const { return (const char *)(a + org); }
};
__device__ __forceinline__ double ld_off(const char *base, uint32_t off) { return *(const double *)(base + off); }

template <class Body>
__device__ __forceinline__ void tile_loop(int total, const Body &body)
{
    const int G = gridDim.x, b = blockIdx.x;
    const bool one = G >= total;   // tile b only; one loop for both cases, so that the body is compiled once
    const int tch = tile_chunk(total);
    const int x = b % NXCD, lane = b / NXCD;
    const int nwg = (G - x + NXCD - 1) / NXCD;
    const int nchunks = (total + tch - 1) / tch;
    const int my_chunks = nchunks > x ? (nchunks - x + NXCD - 1) / NXCD : 0;
    const int first = one ? 0 : lane, end = one ? 1 : my_chunks * tch, step = one ? 1 : nwg;
    for (int k = first; k < end; k += step) {
        const int t = one ? b : (x + NXCD * (k / tch)) * tch + k % tch;
        if (t < total) body(t);
    }
}

// The same values, unknown to the compiler: a loop's body that takes them computes
// what follows from them anew instead of holding it in registers over the loop.
__device__ __forceinline__ GlideGeom opaque(GlideGeom g)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(g.ny), "+s"(g.nx), "+s"(g.dx), "+s"(g.dt));
#endif
    return g;
}
__device__ __forceinline__ Params opaque(Params p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p.n), "+s"(p.eps_reg), "+s"(p.water_drag), "+s"(p.calving_rate), "+s"(p.gl_c), "+s"(p.gl_derivatives));
#endif
    return p;
}

// One tile per workgroup with the tiles dealt to the XCDs in chunks of up to
// TCH consecutive tiles, as tile_loop deals them: workgroup b (on XCD b % 8)
// takes tile (x + 8 c) tch + o for x = b % 8, c = (b / 8) / tch, o = (b / 8)
// % tch.  Over a grid of a multiple of 8 tch workgroups this is a bijection;
// workgroups whose tile is past the last one (t >= total) have no tile.  With
// tiles numbered down the columns a chunk's neighbours share the tall halos in
// one L2: against tile b row by row, local sweeps (vanka_fold_tile) of 387 x 501
// 38.8 -> 36.7 us, of 1024^2 146 -> 140, full ones of 256^2 14.4 -> 13.8, of 512^2
// 37.4 -> 36.6.
__host__ __device__ __forceinline__ int chunked_tile(int b, int total)
{
    const int tch = tile_chunk(total), k = b / NXCD;
    return (b % NXCD + NXCD * (k / tch)) * tch + k % tch;
}
__host__ __device__ inline int chunked_grid(int total)
{
    const int span = NXCD * tile_chunk(total);
    return (total + span - 1) / span * span;
}

// ---------------------------------------------------------------------------
// viscosity tile: cells [i0-1, i0+TY] x [j0-1, j0+TX] into LDS (0 outside)
// ---------------------------------------------------------------------------
template <int TX, int TY>
__device__ __forceinline__ void fill_eta_tile(double (*eta_s)[TX + 2], int i0, int j0, const double *__restrict__ u,
                                              const double *__restrict__ v, const double *__restrict__ B,
                                              const Params &p, double dx, int ny, int nx)
{
    int tid = threadIdx.y * TX + threadIdx.x;
    for (int k = tid; k < (TY + 2) * (TX + 2); k += TX * TY) {
        int a = k / (TX + 2), b = k - a * (TX + 2);
        int ci = i0 - 1 + a, cj = j0 - 1 + b;
        eta_s[a][b] = (ci >= 0 && ci < ny && cj >= 0 && cj < nx) ? eta_cell(ci, cj, u, v, B, p, dx, ny, nx) : 0.0;
    }
}

// 2 eta of cell (i, j) (eta_cell, ssa_device.h) from its face velocities and
// the next ones along each face's line (u_tl = u[i-1, j], v_lt = v[i, j-1], ...):
// the factors of 1/2 of the corner shear rates, their mean square and eta
// itself are exact and ride on one constant; corners on the domain edge get
// the factor 0.
__device__ __forceinline__ double eta2_from(int i, int j, int ny, int nx, double u_l, double u_r, double v_t, double v_b,
                                            double u_tl, double u_tr, double u_bl, double u_br, double v_lt,
                                            double v_rt, double v_lb, double v_rb, double Bc, const Params &p,
                                            double glen_exp, double dxi)
{
    const double dudx = (u_r - u_l) * dxi, dvdy = (v_t - v_b) * dxi;
    const bool t = i > 0, b = i < ny - 1, l = j > 0, r = j < nx - 1;
    const double V_tl = t && l ? dxi : 0.0, V_tr = t && r ? dxi : 0.0, V_bl = b && l ? dxi : 0.0, V_br = b && r ? dxi : 0.0;
    const double e_tl = fma(u_tl - u_l, V_tl, (v_t - v_lt) * V_tl);
    const double e_tr = fma(u_tr - u_r, V_tr, (v_rt - v_t) * V_tr);
    const double e_bl = fma(u_l - u_bl, V_bl, (v_b - v_lb) * V_bl);
    const double e_br = fma(u_r - u_br, V_br, (v_rb - v_b) * V_br);
    const double e2 = fma(e_br, e_br, fma(e_bl, e_bl, fma(e_tr, e_tr, e_tl * e_tl)));
    const double eII = fma(0.0625, e2, fma(dudx, dvdy, fma(dvdy, dvdy, dudx * dudx))) + p.eps_reg;
    return Bc * pow_pos(eII, glen_exp);
}
// ---------------------------------------------------------------------------
// Residual r = F(U) - f (- sub)  (glide/cuda/residuals.cu:6-292), LDS-staged:
// the tile's u and v (two-ring halo) are staged once; every cell of the tile
// and the ring around it then yields 2 eta H, its normal stresses, surface and
// drag, and every vertex its shear stress, each evaluated once into LDS; each
// point sums its rows from LDS.
//
// Every row sums its terms in the order of the reference and the oracle, and
// every term has their rounding: what differs is powers of two, which are
// exact (2 eta H in eta H's place, the factors of the stresses, drags, fluxes
// and averages on the constants 1/(2 dx) and 1/(8 dx)), the range handling of
// the divisions, exp and log (newton_device.h), and terms that vanish at the
// domain edge, which get a factor of 0.  So the bits are the same up to the
// sign of zeros.
//
// Bound by FP64 issue: about half of it is the power law and the sigmoid per
// haloed cell.  512^2: 11.5 -> 8.7 us; 1024^2 on new data each pass: 47.9 ->
// 33.0 us (3.6 TB/s of compulsory traffic; 23 us at the rate of a large copy).
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct ResidLDS {
    double u[TY + 4][TX + 4];   // u[i0-2+a][j0-2+b] (clamped)
    double v[TY + 4][TX + 4];   // v[i0-2+a][j0-2+b] (clamped)
    double H[TY + 2][TX + 2];   // cells [i0-1+a][j0-1+b] (clamped); likewise:
    double S[TY + 2][TX + 2];   // surface max(bed, -0.917 H) + H
    double be[TY + 2][TX + 2];  // drag g beta + (1 - g) water_drag
    double n[TY + 2][TX + 2];   // 2 eta H (0 outside the domain)
    double sx[TY + 2][TX + 2];  // sigma_xx, sigma_yy (0 outside the domain)
    double sy[TY + 2][TX + 2];
    double cal[TY][TX];         // calving sink of cell [i0+a][j0+b]
    double sxy[TY + 1][TX + 1]; // 8 sigma_xy at vertex [i0+a][j0+b]
};

// The tiles cover the cells only (cdiv(nx, TX) x cdiv(ny, TY)); where a tile
// ends exactly at the last column (row), its last lane (row of threads) also
// computes the u faces at j = nx (v faces at i = ny), so the extra face column
// and row need no tiles of their own.
template <int TX, int TY>
__device__ __forceinline__ void residual_tile_lds(const GlideGeom &g, const Params &p, double *__restrict__ r,
                                                  const double *__restrict__ U, const double *__restrict__ f,
                                                  const double *__restrict__ sub, const double *__restrict__ bed,
                                                  const double *__restrict__ B, const double *__restrict__ beta,
                                                  const double *__restrict__ mask, const double *__restrict__ gamma,
                                                  int bx, int by, ResidLDS<TX, TY> &S)
{
    constexpr int NT = TX * TY, NC = ((TY + 2) * (TX + 2) + NT - 1) / NT;
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    const double *u = U, *v = U + nu, *H = U + nu + nv;
    const int i0 = by * TY, j0 = bx * TX;
    const int tid = threadIdx.y * TX + threadIdx.x;
    const NewtonK K = newton_constants(g.dx, g.dt);
    const double glen_exp = (1.0 - p.n) / (2.0 * p.n);
    // 1. stage u and v; the cells' other inputs go to registers meanwhile
    double h[NC], bd[NC], bt[NC], Bc[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
        if (k < (TY + 2) * (TX + 2)) {
            const size_t kc = (size_t)clampi(i0 - 1 + a, 0, ny - 1) * nx + clampi(j0 - 1 + b, 0, nx - 1);
            h[q] = H[kc];
            bd[q] = bed[kc];
            bt[q] = beta[kc];
            Bc[q] = B[kc];
        }
    }
    for (int k = tid; k < (TY + 4) * (TX + 4); k += NT) {
        const int a = k / (TX + 4), b = k - a * (TX + 4);
        S.u[a][b] = ld_u(u, i0 - 2 + a, j0 - 2 + b, ny, nx);
        S.v[a][b] = ld_v(v, i0 - 2 + a, j0 - 2 + b, ny, nx);
    }
    __syncthreads();
    // 2. per cell (a, b): global (i0-1+a, j0-1+b), its u and v at [a+1][b+1]
#pragma unroll
    for (int q = 0; q < NC; q++) {
        const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
        if (k >= (TY + 2) * (TX + 2)) break;
        const int ci = i0 - 1 + a, cj = j0 - 1 + b;
        const double u_l = S.u[a + 1][b + 1], u_r = S.u[a + 1][b + 2], v_t = S.v[a + 1][b + 1], v_b = S.v[a + 2][b + 1];
        double n = 0.0;
        if (ci >= 0 && ci < ny && cj >= 0 && cj < nx)
            n = eta2_from(ci, cj, ny, nx, u_l, u_r, v_t, v_b, S.u[a][b + 1], S.u[a][b + 2], S.u[a + 2][b + 1],
                          S.u[a + 2][b + 2], S.v[a + 1][b], S.v[a + 1][b + 2], S.v[a + 2][b], S.v[a + 2][b + 2], Bc[q], p,
                          glen_exp, K.dxi) *
                h[q];
        const double du = u_r - u_l, dv = v_t - v_b;
        S.n[a][b] = n;
        S.sx[a][b] = n * fma(du, K.dxi2, dv * K.dxi);
        S.sy[a][b] = n * fma(du, K.dxi, dv * K.dxi2);
        const double gr = sigm_mid(fma(0.917, h[q], bd[q]), p.gl_c), g1 = 1.0 - gr;
        S.H[a][b] = h[q];
        S.S[a][b] = fmax(bd[q], -0.917 * h[q]) + h[q];
        S.be[a][b] = fma(gr, bt[q], g1 * p.water_drag);
        if (a >= 1 && a <= TY && b >= 1 && b <= TX) S.cal[a - 1][b - 1] = p.calving_rate * g1 * h[q];
    }
    __syncthreads();
    // 3. per vertex shear stress, 0 on the domain edge
    for (int k = tid; k < (TY + 1) * (TX + 1); k += NT) {
        const int a = k / (TX + 1), b = k - a * (TX + 1);   // vertex (i0 + a, j0 + b): cells [a..a+1][b..b+1]
        const int vi = i0 + a, vj = j0 + b;
        const double V = vi > 0 && vi < ny && vj > 0 && vj < nx ? K.dxi : 0.0;
        const double m = ((S.n[a][b] + S.n[a][b + 1]) + S.n[a + 1][b]) + S.n[a + 1][b + 1];
        S.sxy[a][b] = m * fma(S.u[a + 1][b + 2] - S.u[a + 2][b + 2], V, (S.v[a + 2][b + 2] - S.v[a + 2][b + 1]) * V);
    }
    __syncthreads();
    // 4. rows of point (i, j): cell (i < ny, j < nx), u face (i < ny), v face (j < nx)
    auto rows = [&](int i, int j) {
        const int a = i - i0 + 1, b = j - j0 + 1;   // cell (i, j) in the one-ring arrays
        const bool il = j > 0, ir = j + 1 < nx, it = i > 0, ib = i + 1 < ny;
        const double H_c = S.H[a][b], H_l = S.H[a][b - 1], H_t = S.H[a - 1][b];
        const double u_l = S.u[a + 1][b + 1], v_t = S.v[a + 1][b + 1];
        const double s_l = H_l + H_c, s_t = H_t + H_c;
        const double F_l = il && j < nx ? K.hdx : 0.0, F_t = it && i < ny ? K.hdx : 0.0;
        if (i < ny && j < nx) {
            const size_t kc = (size_t)i * nx + j;
            const double H_r = S.H[a][b + 1], H_b = S.H[a + 1][b], u_r = S.u[a + 1][b + 2], v_b = S.v[a + 2][b + 1];
            const double F_r = ir ? K.hdx : 0.0, F_b = ib ? K.hdx : 0.0;
            double rH = div_refined(H_c, K.dt, K.rdt) - (f ? f[nu + nv + kc] : 0.0);
            rH += S.cal[a - 1][b - 1];
            rH -= fma(s_l, u_l, -(fabs(u_l) * (H_c - H_l))) * F_l;
            rH += fma(H_c + H_r, u_r, -(fabs(u_r) * (H_r - H_c))) * F_r;
            rH += fma(s_t, v_t, -(fabs(v_t) * (H_t - H_c))) * F_t;
            rH -= fma(H_c + H_b, v_b, -(fabs(v_b) * (H_c - H_b))) * F_b;
            const double m = mask[kc], th = gamma[kc];
            const double val = (1.0 - m) * rH + m * (H_c - th);
            const size_t k = nu + nv + kc;
            r[k] = sub ? val - sub[k] : val;
        }
        if (i < ny) {
            const size_t k = (size_t)i * (nx + 1) + j;
            double ru = f ? -f[k] : -0.0;
            ru += S.sx[a][b] * K.dxi;
            ru -= S.sx[a][b - 1] * K.dxi;
            ru += S.sxy[a - 1][b - 1] * K.edx;
            ru -= S.sxy[a][b - 1] * K.edx;
            ru = fma(-0.5, (S.be[a][b - 1] + S.be[a][b]) * u_l, ru);
            ru -= (s_l * (S.S[a][b] - S.S[a][b - 1])) * F_l;
            r[k] = sub ? ru - sub[k] : ru;
        }
        if (j < nx) {
            const size_t k = nu + (size_t)i * nx + j;
            double rv = f ? -f[k] : -0.0;
            rv += S.sy[a - 1][b] * K.dxi;
            rv -= S.sy[a][b] * K.dxi;
            rv -= S.sxy[a - 1][b - 1] * K.edx;
            rv += S.sxy[a - 1][b] * K.edx;
            rv = fma(-0.5, (S.be[a - 1][b] + S.be[a][b]) * v_t, rv);
            rv -= (s_t * (S.S[a - 1][b] - S.S[a][b])) * F_t;
            r[k] = sub ? rv - sub[k] : rv;
        }
    };
    const int i = i0 + threadIdx.y, j = j0 + threadIdx.x;
    if (i > ny || j > nx) return;
    rows(i, j);
    if (j == nx - 1 && j0 + TX == nx && i < ny) rows(i, nx);   // u face at j = nx
    if (i == ny - 1 && i0 + TY == ny && j < nx) rows(ny, j);   // v face at i = ny
}

template <class EtaFn>
__device__ __forceinline__ CellNbhd load_nbhd(int i, int j, int ny, int nx, size_t nu, size_t nv,
                                              const double *__restrict__ u, const double *__restrict__ v,
                                              const double *__restrict__ H, const double *__restrict__ f,
                                              const double *__restrict__ bed, const double *__restrict__ beta,
                                              const EtaFn &E)
{
    CellNbhd N;
    N.e_c = E(i, j); N.e_l = E(i, j - 1); N.e_r = E(i, j + 1); N.e_t = E(i - 1, j); N.e_b = E(i + 1, j);
    N.e_tl = E(i - 1, j - 1); N.e_tr = E(i - 1, j + 1); N.e_bl = E(i + 1, j - 1); N.e_br = E(i + 1, j + 1);
    N.H_l = ld_c(H, i, j - 1, ny, nx); N.H_r = ld_c(H, i, j + 1, ny, nx);
    N.H_t = ld_c(H, i - 1, j, ny, nx); N.H_b = ld_c(H, i + 1, j, ny, nx);
    N.H_tl = ld_c(H, i - 1, j - 1, ny, nx); N.H_tr = ld_c(H, i - 1, j + 1, ny, nx);
    N.H_bl = ld_c(H, i + 1, j - 1, ny, nx); N.H_br = ld_c(H, i + 1, j + 1, ny, nx);
    N.bed_c = ld_c(bed, i, j, ny, nx); N.bed_l = ld_c(bed, i, j - 1, ny, nx); N.bed_r = ld_c(bed, i, j + 1, ny, nx);
    N.bed_t = ld_c(bed, i - 1, j, ny, nx); N.bed_b = ld_c(bed, i + 1, j, ny, nx);
    N.beta_c = ld_c(beta, i, j, ny, nx); N.beta_l = ld_c(beta, i, j - 1, ny, nx);
    N.beta_r = ld_c(beta, i, j + 1, ny, nx); N.beta_t = ld_c(beta, i - 1, j, ny, nx);
    N.beta_b = ld_c(beta, i + 1, j, ny, nx);
    N.u_ll = ld_u(u, i, j - 1, ny, nx); N.u_rr = ld_u(u, i, j + 2, ny, nx);
    N.u_tl = ld_u(u, i - 1, j, ny, nx); N.u_tr = ld_u(u, i - 1, j + 1, ny, nx);
    N.u_bl = ld_u(u, i + 1, j, ny, nx); N.u_br = ld_u(u, i + 1, j + 1, ny, nx);
    N.v_lt = ld_v(v, i, j - 1, ny, nx); N.v_lb = ld_v(v, i + 1, j - 1, ny, nx);
    N.v_rt = ld_v(v, i, j + 1, ny, nx); N.v_rb = ld_v(v, i + 1, j + 1, ny, nx);
    N.v_tt = ld_v(v, i - 1, j, ny, nx); N.v_bb = ld_v(v, i + 2, j, ny, nx);
    if (f) {
        N.f0 = ld_u(f, i, j, ny, nx); N.f1 = ld_u(f, i, j + 1, ny, nx);
    N.f2 = ld_v(f + nu, i, j, ny, nx); N.f3 = ld_v(f + nu, i + 1, j, ny, nx);
    N.f4 = ld_v(f + nu + nv, i, j, ny, nx);
    } else {
        N.f0 = N.f1 = N.f2 = N.f3 = N.f4 = 0.0;
    }

    return N;
}

// ---------------------------------------------------------------------------
// What a Vanka sweep derives per cell from its input state, staged once for
// the tile's cells and the ring around them: 2 eta and 2 eta H (0 outside the
// domain), and H, surface and drag (those of the clamped cell outside it).
// Each thread then reads its neighbours' values instead of evaluating four
// neighbour sigmoids of its own.
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct VankaLDS {
    double e2[TY + 2][TX + 2];
    double n[TY + 2][TX + 2];
    double H[TY + 2][TX + 2];
    double S[TY + 2][TX + 2];
    double be[TY + 2][TX + 2];
};

// cell [a][b]'s neighbours from the staged values; what follows from those and the faces
template <int TX, int TY>
__device__ __forceinline__ void cell_from_lds(NewtonCell &C, const VankaLDS<TX, TY> &L, const NewtonK &K, int a, int b)
{
    C.e2 = L.e2[a][b];
    C.n_l = L.n[a][b - 1];
    C.n_r = L.n[a][b + 1];
    C.n_t = L.n[a - 1][b];
    C.n_b = L.n[a + 1][b];
    C.p_tl = (L.n[a - 1][b - 1] + C.n_t) + C.n_l;
    C.p_tr = C.n_t + L.n[a - 1][b + 1];
    C.n_bl = L.n[a + 1][b - 1];
    C.n_br = L.n[a + 1][b + 1];
    C.H_l = L.H[a][b - 1];
    C.H_r = L.H[a][b + 1];
    C.H_t = L.H[a - 1][b];
    C.H_b = L.H[a + 1][b];
    C.S_l = L.S[a][b - 1];
    C.S_r = L.S[a][b + 1];
    C.S_t = L.S[a - 1][b];
    C.S_b = L.S[a + 1][b];
    C.be_l = L.be[a][b - 1];
    C.be_r = L.be[a][b + 1];
    C.be_t = L.be[a - 1][b];
    C.be_b = L.be[a + 1][b];
    C.c_l = (C.v_lt - C.v_lb) * K.dxi;
    C.c_r = (C.v_rt - C.v_rb) * K.dxi;
    C.d_t = C.u_tr - C.u_tl;
    C.d_b = C.u_br - C.u_bl;
}

// A thread's share of the staged cells [i0-1, i0+TY] x [j0-1, j0+TX], cell q =
// tid + q TX TY: load() issues all its reads, compute() evaluates and stores
// to LDS.  Between the two the thread issues its own cell's reads as well, so a
// tile waits out one memory latency instead of three (two workgroups per CU
// leave little else to run meanwhile); together with 32-bit offsets a sweep's
// staging at 1024^2 went from 53.3 to 50.8 us.  INTERIOR: the cells lie in [1, ny-2] x
// [1, nx-2], so nothing is clamped.
template <bool INTERIOR, int TX, int TY>
struct VankaStage {
    static constexpr int NT = TX * TY, NALL = (TY + 2) * (TX + 2), NC = (NALL + NT - 1) / NT;
    double u[NC][6], v[NC][6];   // rows i-1, i, i+1 of u x columns j, j+1; rows i, i+1 of v x columns j-1, j, j+1
    double h[NC], bd[NC], bt[NC], Bc[NC];

    __device__ __forceinline__ void load(int i0, int j0, int rb, int cb, const double *__restrict__ U,
                                         const double *__restrict__ bed, const double *__restrict__ B,
                                         const double *__restrict__ beta, int ny, int nx)
    {
        const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
        const TileField tu(nx + 1, rb, cb), tc(nx, rb, cb);
        const char *bu = tu.base(U), *bv = tc.base(U + nu), *bH = tc.base(U + nu + nv), *bbed = tc.base(bed),
                   *bB = tc.base(B), *bbeta = tc.base(beta);
        const int tid = threadIdx.y * TX + threadIdx.x;
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
            if (k >= NALL) break;
            const int ci = i0 - 1 + a, cj = j0 - 1 + b;
            const int ic = INTERIOR ? ci : clampi(ci, 0, ny - 1), jc = INTERIOR ? cj : clampi(cj, 0, nx - 1);
            const uint32_t r0 = ic - rb, c0 = 8u * (jc - cb), u0 = r0 * tu.pitch, v0 = r0 * tc.pitch, kc = v0 + c0;
            // row i+1 of v and column j+1 of u exist for every cell
            const uint32_t v1 = v0 + tc.pitch;
            const uint32_t ut = INTERIOR || ic > 0 ? u0 - tu.pitch : u0, ub = INTERIOR || ic < ny - 1 ? u0 + tu.pitch : u0;
            const uint32_t cl = INTERIOR || jc > 0 ? c0 - 8 : c0, cr = INTERIOR || jc < nx - 1 ? c0 + 8 : c0;
            h[q] = ld_off(bH, kc);
            bd[q] = ld_off(bbed, kc);
            bt[q] = ld_off(bbeta, kc);
            Bc[q] = ld_off(bB, kc);
            u[q][0] = ld_off(bu, ut + c0);
            u[q][1] = ld_off(bu, ut + c0 + 8);
            u[q][2] = ld_off(bu, u0 + c0);
            u[q][3] = ld_off(bu, u0 + c0 + 8);
            u[q][4] = ld_off(bu, ub + c0);
            u[q][5] = ld_off(bu, ub + c0 + 8);
            v[q][0] = ld_off(bv, v0 + cl);
            v[q][1] = ld_off(bv, v0 + c0);
            v[q][2] = ld_off(bv, v0 + cr);
            v[q][3] = ld_off(bv, v1 + cl);
            v[q][4] = ld_off(bv, v1 + c0);
            v[q][5] = ld_off(bv, v1 + cr);
        }
    }
    __device__ __forceinline__ void compute(VankaLDS<TX, TY> &L, int i0, int j0, const Params &p, double dxi, int ny,
                                            int nx) const
    {
        const double glen_exp = (1.0 - p.n) / (2.0 * p.n);
        const int tid = threadIdx.y * TX + threadIdx.x;
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
            if (k >= NALL) break;
            const int ci = i0 - 1 + a, cj = j0 - 1 + b;
            double e2 = 0.0;
            if (INTERIOR || (ci >= 0 && ci < ny && cj >= 0 && cj < nx))
                e2 = eta2_from(INTERIOR ? 1 : ci, INTERIOR ? 1 : cj, INTERIOR ? 3 : ny, INTERIOR ? 3 : nx, u[q][2], u[q][3],
                               v[q][1], v[q][4], u[q][0], u[q][1], u[q][4], u[q][5], v[q][0], v[q][2], v[q][3], v[q][5],
                               Bc[q], p, glen_exp, dxi);
            const double g = sigm_mid(fma(0.917, h[q], bd[q]), p.gl_c);
            L.e2[a][b] = e2;
            L.n[a][b] = e2 * h[q];
            L.H[a][b] = h[q];
            L.S[a][b] = fmax(bd[q], -0.917 * h[q]) + h[q];
            L.be[a][b] = fma(g, bt[q], (1.0 - g) * p.water_drag);
        }
    }
};

// ---------------------------------------------------------------------------
// One cell's Vanka update (glide/cuda/vanka.cu:56-439): the tile's cells are
// staged (VankaStage), then each thread takes its cell's neighbourhood, runs
// n_newton damped Newton iterations (newton_iterate) and returns the per-cell
// deltas.  (i, j) is the cell, (i0, j0) the tile's first cell, so that the cell
// is [i - i0 + 1][j - j0 + 1] of the staged arrays.  INTERIOR: the tile's ring
// lies in [1, ny-2] x [1, nx-2], so no read is clamped and no term vanishes.
// ---------------------------------------------------------------------------
template <bool INTERIOR, int TX, int TY>
__device__ __forceinline__ void vanka_cell_deltas(const GlideGeom &g, const Params &p, const NewtonK &K,
                                                  VankaLDS<TX, TY> &L, const double *__restrict__ U,
                                                  const double *__restrict__ f, const double *__restrict__ bed,
                                                  const double *__restrict__ B, const double *__restrict__ beta,
                                                  const double *__restrict__ gamma, int n_newton, int i0, int j0, int i,
                                                  int j, double d5[5])
{
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    // a row and column not after the first that the tile's cells read
    const int rb = INTERIOR ? i0 - 2 : max(i0 - 2, 0), cb = INTERIOR ? j0 - 2 : max(j0 - 2, 0);
    VankaStage<INTERIOR, TX, TY> stage;
    stage.load(i0, j0, rb, cb, U, bed, B, beta, ny, nx);
    const TileField tu(nx + 1, rb, cb), tc(nx, rb, cb);
    const char *bu = tu.base(U), *bv = tc.base(U + nu), *fu = tu.base(f), *fv = tc.base(f + nu),
               *fH = tc.base(f + nu + nv);
    // rows i-1, i, i+1 of u and i-1, i, i+1, i+2 of v; columns j-1, j, j+1 and, of u, j+2 (clamped at the edge)
    const uint32_t r0 = i - rb, c0 = 8u * (j - cb);
    const uint32_t u0 = r0 * tu.pitch, v0 = r0 * tc.pitch, v1 = v0 + tc.pitch;
    const uint32_t ut = INTERIOR || i > 0 ? u0 - tu.pitch : u0, ub = INTERIOR || i < ny - 1 ? u0 + tu.pitch : u0;
    const uint32_t vt = INTERIOR || i > 0 ? v0 - tc.pitch : v0, vb = INTERIOR || i < ny - 1 ? v1 + tc.pitch : v1;
    const uint32_t cl = INTERIOR || j > 0 ? c0 - 8 : c0, cr = INTERIOR || j < nx - 1 ? c0 + 8 : c0;
    const uint32_t crr = INTERIOR || j < nx - 1 ? c0 + 16 : c0 + 8;
    NewtonX x;
    NewtonCell C;
    x.u_l = ld_off(bu, u0 + c0);
    x.u_r = ld_off(bu, u0 + c0 + 8);
    x.v_t = ld_off(bv, v0 + c0);
    x.v_b = ld_off(bv, v1 + c0);
    C.u_ll = ld_off(bu, u0 + cl);
    C.u_rr = ld_off(bu, u0 + crr);
    C.u_tl = ld_off(bu, ut + c0);
    C.u_tr = ld_off(bu, ut + c0 + 8);
    C.u_bl = ld_off(bu, ub + c0);
    C.u_br = ld_off(bu, ub + c0 + 8);
    C.v_lt = ld_off(bv, v0 + cl);
    C.v_lb = ld_off(bv, v1 + cl);
    C.v_rt = ld_off(bv, v0 + cr);
    C.v_rb = ld_off(bv, v1 + cr);
    C.v_tt = ld_off(bv, vt + c0);
    C.v_bb = ld_off(bv, vb + c0);
    C.f0 = ld_off(fu, u0 + c0);
    C.f1 = ld_off(fu, u0 + c0 + 8);
    C.f2 = ld_off(fv, v0 + c0);
    C.f3 = ld_off(fv, v1 + c0);
    C.f4 = ld_off(fH, v0 + c0);
    C.bed = ld_off(tc.base(bed), v0 + c0);
    C.beta = ld_off(tc.base(beta), v0 + c0);
    C.th = ld_off(tc.base(gamma), v0 + c0);
    stage.compute(L, i0, j0, p, K.dxi, ny, nx);
    __syncthreads();
    const int a = i - i0 + 1, b = j - j0 + 1;
    x.H = L.H[a][b];
    const NewtonX x0 = x;
    cell_from_lds(C, L, K, a, b);
    newton_edges<INTERIOR>(C, K, i, j, ny, nx);
    newton_iterate(C, K, p, n_newton, x);
    d5[0] = 0.5 * (x.u_l - x0.u_l);
    d5[1] = 0.5 * (x.u_r - x0.u_r);
    d5[2] = 0.5 * (x.v_t - x0.v_t);
    d5[3] = 0.5 * (x.v_b - x0.v_b);
    d5[4] = x.H - x0.H;
}

// ---------------------------------------------------------------------------
// Forward Vanka: per-cell damped Newton (glide/cuda/vanka.cu:3-439, 844-1295)
// cd (5 x nc, structure of arrays) receives 0.5*(x - x0) for the four faces
// and (H - H0) for the cell.
// ---------------------------------------------------------------------------
template <int TX, int TY, bool LOCAL>
__device__ __forceinline__ void vanka_tile(const GlideGeom &g, const Params &p, const double *__restrict__ U,
                                           const double *__restrict__ f, const double *__restrict__ bed,
                                           const double *__restrict__ B, const double *__restrict__ beta,
                                           const double *__restrict__ gamma, const unsigned char *__restrict__ blk,
                                           int nbx, int n_newton, double *__restrict__ cd, int bx, int by,
                                           VankaLDS<TX, TY> &L)
{
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx), nc = n_c(ny, nx);
    const int i0 = by * TY, j0 = bx * TX;
    const int i = i0 + threadIdx.y, j = j0 + threadIdx.x;
    const bool mine = (i < ny && j < nx);
    // A local sweep smooths every cell of a tile that holds an active cell:
    // the apply pass reads only the active cells' updates, so the idle
    // cells' chains change nothing, and a wave with part of its lanes idle
    // ran its Newton chain up to 2.3x slower than a full wave (measured on
    // the 64^2 to 512^2 levels).
    if (LOCAL) {
        if (!__syncthreads_or(mine && blk[(i / RB) * nbx + j / RB])) return;   // uniform: the whole tile is idle
    }
    const NewtonK K = newton_constants(g.dx, g.dt);
    double d5[5];
    // the whole per-cell body is instantiated twice so that no value is live
    // across the branch; threads past the level's edge take its nearest cell
    if (i0 >= 2 && i0 + TY <= ny - 2 && j0 >= 2 && j0 + TX <= nx - 2)
        vanka_cell_deltas<true>(g, p, K, L, U, f, bed, B, beta, gamma, n_newton, i0, j0, i, j, d5);
    else
        vanka_cell_deltas<false>(g, p, K, L, U, f, bed, B, beta, gamma, n_newton, i0, j0, min(i, ny - 1), min(j, nx - 1),
                                 d5);
    if (!mine) return;
    const size_t ci = (size_t)i * nx + j;
#pragma unroll
    for (int q = 0; q < 5; q++) cd[q * nc + ci] = d5[q];
}

// Gather the per-cell updates: U += 0.5 * delta (glide/grid.py:305-317)
template <int TX, int TY, bool LOCAL>
__device__ __forceinline__ void apply_tile(int ny, int nx, double *__restrict__ U, const double *__restrict__ cd,
                                           const unsigned char *__restrict__ blk, int nbx, int bx, int by)
{
    const int i = by * TY + threadIdx.y, j = bx * TX + threadIdx.x;
    if (i > ny || j > nx) return;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx), nc = n_c(ny, nx);
    auto act = [&](int ci, int cj) { return !LOCAL || blk[(ci / RB) * nbx + cj / RB] != 0; };
    if (i < ny) {
        double d = 0.0;
        if (j > 0 && act(i, j - 1)) d = d + cd[nc + (size_t)i * nx + j - 1];
        if (j < nx && act(i, j)) d = d + cd[(size_t)i * nx + j];
        U[(size_t)i * (nx + 1) + j] += 0.5 * d;
    }
    if (j < nx) {
        double d = 0.0;
        if (i > 0 && act(i - 1, j)) d = d + cd[3 * nc + (size_t)(i - 1) * nx + j];
        if (i < ny && act(i, j)) d = d + cd[2 * nc + (size_t)i * nx + j];
        U[nu + (size_t)i * nx + j] += 0.5 * d;
    }
    if (i < ny && j < nx) {
        size_t ci = (size_t)i * nx + j;
        double d = act(i, j) ? cd[4 * nc + ci] : 0.0;
        U[nu + nv + ci] += 0.5 * d;
    }
}

// ---------------------------------------------------------------------------
// A sweep of a large level without an apply pass: from the state U into Uo
// (another buffer).  Inside a tile the faces' updates meet in LDS; a face
// between two tiles keeps its value in Uo, and the two cells' updates of it
// go to the pending arrays, which whoever reads the face in the next sweep
// adds (k_fold_finish after the last one): v faces on the tiles' top rows,
// u faces on their left columns.  So a sweep reads and writes the state once
// where the two kernels wrote five values a cell, read them again and read and
// wrote the state; and the tile's state is staged in LDS, 5.5 loads a thread
// where each took its cells' 56 through the vector cache.  Same bits as
// vanka_tile and apply_tile.  A sweep of ten, before and
// after: 256^2 17.2 -> 14.0 us, 387 x 501 local 44.2 -> 40.2, 512^2 42.7 -> 38.0,
// 1024^2 149 -> 138.
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct FoldLDS {
    VankaLDS<TX, TY> L;
    double u[TY + 4][TX + 3];   // rows i0-2 .. i0+TY+1, face columns j0-1 .. j0+TX+1 (clamped)
    double v[TY + 3][TX + 4];   // face rows i0-1 .. i0+TY+1, columns j0-2 .. j0+TX+1 (clamped)
    double cdr[TY][TX], cdb[TY][TX];   // the cells' updates of their right and bottom faces
};
// pending updates: v faces of row by * TY from the cells above and below, u
// faces of column bx * TX from the cells at the left and right
struct FoldPending {
    double *top, *bot, *lft, *rgt;
    __host__ __device__ FoldPending(double *a, int ny, int nx, int ntx, int nty)
        : top(a), bot(a + (size_t)nty * nx), lft(a + 2 * (size_t)nty * nx), rgt(a + 2 * (size_t)nty * nx + (size_t)ny * ntx)
    {
    }
    __host__ __device__ static size_t doubles(int ny, int nx, int ntx, int nty)
    {
        return 2 * (size_t)nty * nx + 2 * (size_t)ny * ntx;
    }
};
// the scratch of 5 nc doubles holds the other state and two sets of pending updates
__host__ __device__ inline bool fold_fits(int ny, int nx, int tx, int ty)
{
    return n_t(ny, nx) + 2 * FoldPending::doubles(ny, nx, cdiv(nx, tx), cdiv(ny, ty)) <= 5 * n_c(ny, nx);
}
template <int TX, int TY>
__host__ __device__ inline FoldPending fold_pending(double *scratch, int ny, int nx, int set)
{
    const int ntx = cdiv(nx, TX), nty = cdiv(ny, TY);
    return FoldPending(scratch + n_t(ny, nx) + set * FoldPending::doubles(ny, nx, ntx, nty), ny, nx, ntx, nty);
}

// stages the tile's faces, its own cell and what follows from them; then as vanka_cell_deltas
template <bool INTERIOR, int TX, int TY>
__device__ __forceinline__ void fold_cell(const GlideGeom &g, const Params &p, const NewtonK &K, FoldLDS<TX, TY> &F,
                                          const double *__restrict__ U, const FoldPending &P, bool first,
                                          const double *__restrict__ f, const double *__restrict__ bed,
                                          const double *__restrict__ B, const double *__restrict__ beta,
                                          const double *__restrict__ gamma, int n_newton, bool second, int bx, int by,
                                          int i, int j, NewtonX &x, NewtonX &x0)
{
    constexpr int NT = TX * TY, UC = TX + 3, VC = TX + 4, NU = (TY + 4) * UC, NV = (TY + 3) * VC;
    constexpr int QU = (NU + NT - 1) / NT, QV = (NV + NT - 1) / NT, NALL = (TY + 2) * (TX + 2), QC = (NALL + NT - 1) / NT;
    static_assert(2 * VC <= NT && 2 * (TY + 4) <= NT, "one pending face a thread");
    const int ny = g.ny, nx = g.nx, i0 = by * TY, j0 = bx * TX;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    const int rb = INTERIOR ? i0 - 2 : max(i0 - 2, 0), cb = INTERIOR ? j0 - 2 : max(j0 - 2, 0);
    const TileField tu(nx + 1, rb, cb), tc(nx, rb, cb);
    const char *bu = tu.base(U), *bv = tc.base(U + nu), *bH = tc.base(U + nu + nv), *bbed = tc.base(bed),
               *bB = tc.base(B), *bbeta = tc.base(beta);
    const int tid = threadIdx.y * TX + threadIdx.x;
    auto clip = [](int k, int n) { return INTERIOR ? k : clampi(k, 0, n); };
    double ur[QU], vr[QV], h[QC], bd[QC], bt[QC], Bc[QC];
#pragma unroll
    for (int q = 0; q < QU; q++) {
        const int k = tid + q * NT, r = k / UC, c = k - r * UC;
        if (k >= NU) break;
        ur[q] = ld_off(bu, (clip(i0 - 2 + r, ny - 1) - rb) * tu.pitch + 8u * (clip(j0 - 1 + c, nx) - cb));
    }
#pragma unroll
    for (int q = 0; q < QV; q++) {
        const int k = tid + q * NT, r = k / VC, c = k - r * VC;
        if (k >= NV) break;
        vr[q] = ld_off(bv, (clip(i0 - 1 + r, ny) - rb) * tc.pitch + 8u * (clip(j0 - 2 + c, nx - 1) - cb));
    }
#pragma unroll
    for (int q = 0; q < QC; q++) {
        const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
        if (k >= NALL) break;
        const uint32_t kc = (clip(i0 - 1 + a, ny - 1) - rb) * tc.pitch + 8u * (clip(j0 - 1 + b, nx - 1) - cb);
        h[q] = ld_off(bH, kc);
        bd[q] = ld_off(bbed, kc);
        bt[q] = ld_off(bbeta, kc);
        Bc[q] = ld_off(bB, kc);
    }
    // the faces with pending updates: v on rows i0 and i0 + TY, u on columns j0 and j0 + TX
    const bool top = !first && by > 0, bot = !first && i0 + TY < ny, lft = !first && bx > 0, rgt = !first && j0 + TX < nx;
    double pv = 0.0, pu = 0.0;
    const int vs = tid >= VC, vc = tid - vs * VC, us = tid & 1, ru = tid >> 1;   // thread's row and column of v, of u
    const bool pend_v = tid < 2 * VC && (vs ? bot : top), pend_u = tid < 2 * (TY + 4) && (us ? rgt : lft);
    if (pend_v) {
        const size_t k = (size_t)(by + vs) * nx + clip(j0 - 2 + vc, nx - 1);
        const double a = P.bot[k], b = P.top[k];
        pv = ld_off(bv, (i0 + vs * TY - rb) * tc.pitch + 8u * (clip(j0 - 2 + vc, nx - 1) - cb)) + 0.5 * ((0.0 + a) + b);
    }
    if (pend_u) {
        const int r = clip(i0 - 2 + ru, ny - 1);
        const size_t k = (size_t)(bx + us) * ny + r;
        const double a = P.rgt[k], b = P.lft[k];
        pu = ld_off(bu, (r - rb) * tu.pitch + 8u * (j0 + us * TX - cb)) + 0.5 * ((0.0 + a) + b);
    }
    NewtonCell C;
    {
        const uint32_t r0 = i - rb, c0 = 8u * (j - cb), u0 = r0 * tu.pitch + c0, v0 = r0 * tc.pitch + c0;
        const char *fu = tu.base(f), *fv = tc.base(f + nu);
        C.f0 = ld_off(fu, u0);
        C.f1 = ld_off(fu, u0 + 8);
        C.f2 = ld_off(fv, v0);
        C.f3 = ld_off(fv, v0 + tc.pitch);
        C.f4 = ld_off(tc.base(f + nu + nv), v0);
        C.bed = ld_off(bbed, v0);
        C.beta = ld_off(bbeta, v0);
        C.th = ld_off(tc.base(gamma), v0);
    }
#pragma unroll
    for (int q = 0; q < QU; q++) {
        const int k = tid + q * NT, r = k / UC, c = k - r * UC;
        if (k < NU && !(c == 1 && lft) && !(c == TX + 1 && rgt)) F.u[r][c] = ur[q];
    }
#pragma unroll
    for (int q = 0; q < QV; q++) {
        const int k = tid + q * NT, r = k / VC, c = k - r * VC;
        if (k < NV && !(r == 1 && top) && !(r == TY + 1 && bot)) F.v[r][c] = vr[q];
    }
    if (pend_v) F.v[1 + vs * TY][vc] = pv;
    if (pend_u) F.u[ru][1 + us * TX] = pu;
    __syncthreads();
    const double glen_exp = (1.0 - p.n) / (2.0 * p.n);
#pragma unroll
    for (int q = 0; q < QC; q++) {
        const int k = tid + q * NT, a = k / (TX + 2), b = k - a * (TX + 2);
        if (k >= NALL) break;
        const int ci = i0 - 1 + a, cj = j0 - 1 + b;
        double e2 = 0.0;
        if (INTERIOR || (ci >= 0 && ci < ny && cj >= 0 && cj < nx))
            e2 = eta2_from(INTERIOR ? 1 : ci, INTERIOR ? 1 : cj, INTERIOR ? 3 : ny, INTERIOR ? 3 : nx, F.u[a + 1][b],
                           F.u[a + 1][b + 1], F.v[a][b + 1], F.v[a + 1][b + 1], F.u[a][b], F.u[a][b + 1], F.u[a + 2][b],
                           F.u[a + 2][b + 1], F.v[a][b], F.v[a][b + 2], F.v[a + 1][b], F.v[a + 1][b + 2], Bc[q], p,
                           glen_exp, K.dxi);
        const double sg = sigm_mid(fma(0.917, h[q], bd[q]), p.gl_c);
        F.L.e2[a][b] = e2;
        F.L.n[a][b] = e2 * h[q];
        F.L.H[a][b] = h[q];
        F.L.S[a][b] = fmax(bd[q], -0.917 * h[q]) + h[q];
        F.L.be[a][b] = fma(sg, bt[q], (1.0 - sg) * p.water_drag);
    }
    __syncthreads();
    const int a = i - i0, b = j - j0;
    x.u_l = F.u[a + 2][b + 1];
    x.u_r = F.u[a + 2][b + 2];
    x.v_t = F.v[a + 1][b + 2];
    x.v_b = F.v[a + 2][b + 2];
    C.u_ll = F.u[a + 2][b];
    C.u_rr = F.u[a + 2][b + 3];
    C.u_tl = F.u[a + 1][b + 1];
    C.u_tr = F.u[a + 1][b + 2];
    C.u_bl = F.u[a + 3][b + 1];
    C.u_br = F.u[a + 3][b + 2];
    C.v_lt = F.v[a + 1][b + 1];
    C.v_lb = F.v[a + 2][b + 1];
    C.v_rt = F.v[a + 1][b + 3];
    C.v_rb = F.v[a + 2][b + 3];
    C.v_tt = F.v[a][b + 2];
    C.v_bb = F.v[a + 3][b + 2];
    cell_from_lds(C, F.L, K, a + 1, b + 1);
    newton_edges<INTERIOR>(C, K, i, j, ny, nx);
    x.H = F.L.H[a + 1][b + 1];
    x0 = x;
    if (second)
        __builtin_amdgcn_s_setprio(1);
    else
        __builtin_amdgcn_s_setprio(0);
    newton_iterate<true>(C, K, p, n_newton, x);
    __builtin_amdgcn_s_setprio(3);
}

// Pi, Po: pending updates of the last sweep and of this one; first: there are none yet
//
// Issue priorities: a Newton chain issues in nearly every cycle by itself, so two
// workgroups on a CU that start together share the issue, end together and then
// leave it idle while the next two wait for memory.  The second 256 workgroups
// (the second one on each of 256 CUs) run their chains ahead of the first, a
// chain's second half goes before other's first half, and what loads and stores
// goes before both, so that one stages while the other computes.  A sweep of
// ten: 512^2 37.9 -> 34.7 us, 1024^2 136 -> 130, 1024^2 local 151 -> 141.
template <int TX, int TY, bool LOCAL>
__device__ __forceinline__ void vanka_fold_tile(const GlideGeom &g, const Params &p, const double *__restrict__ U,
                                                double *__restrict__ Uo, const FoldPending &Pi, const FoldPending &Po,
                                                bool first, const double *__restrict__ f, const double *__restrict__ bed,
                                                const double *__restrict__ B, const double *__restrict__ beta,
                                                const double *__restrict__ gamma, const unsigned char *__restrict__ blk,
                                                int nbx, int n_newton, int bx, int by, FoldLDS<TX, TY> &F)
{
    __builtin_amdgcn_s_setprio(3);
    const bool second = blockIdx.x >> 8 & 1;
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    const int i0 = by * TY, j0 = bx * TX, a = threadIdx.y, b = threadIdx.x;
    const int i = i0 + a, j = j0 + b;
    const bool in = i < ny && j < nx;
    const bool act = !LOCAL || (in && blk[(i / RB) * nbx + j / RB] != 0);
    const size_t ku = (size_t)i * (nx + 1) + j, kv = nu + (size_t)i * nx + j, kH = nu + nv + (size_t)i * nx + j;
    // faces between tiles at this cell
    const bool pt = a == 0 && by > 0, pb = a == TY - 1 && i + 1 < ny, pl = b == 0 && bx > 0, pr = b == TX - 1 && j + 1 < nx;
    const size_t kt = (size_t)by * nx + j, kl = (size_t)bx * ny + i;
    if (LOCAL) {
        if (!__syncthreads_or(act)) {   // uniform: the whole tile is idle.  Both buffers hold its inner points from the first sweep on
            if (!in) return;
            if (pt || first) Uo[kv] = pt && !first ? U[kv] + 0.5 * ((0.0 + Pi.bot[kt]) + Pi.top[kt]) : U[kv];
            if (pl || first) Uo[ku] = pl && !first ? U[ku] + 0.5 * ((0.0 + Pi.rgt[kl]) + Pi.lft[kl]) : U[ku];
            if (first) {
                Uo[kH] = U[kH];
                if (j == nx - 1) Uo[ku + 1] = U[ku + 1];
                if (i == ny - 1) Uo[kv + nx] = U[kv + nx];
            }
            if (pt) Po.top[kt] = 0.0;
            if (pb) Po.bot[kt + nx] = 0.0;
            if (pl) Po.lft[kl] = 0.0;
            if (pr) Po.rgt[kl + ny] = 0.0;
            return;
        }
    }
    const NewtonK K = newton_constants(g.dx, g.dt);
    NewtonX x, x0;
    // as in vanka_tile
    if (i0 >= 2 && i0 + TY <= ny - 2 && j0 >= 2 && j0 + TX <= nx - 2)
        fold_cell<true>(g, p, K, F, U, Pi, first, f, bed, B, beta, gamma, n_newton, second, bx, by, i, j, x, x0);
    else
        fold_cell<false>(g, p, K, F, U, Pi, first, f, bed, B, beta, gamma, n_newton, second, bx, by, min(i, ny - 1),
                         min(j, nx - 1), x, x0);
    // an idle cell's updates count as 0
    const double d0 = act ? 0.5 * (x.u_l - x0.u_l) : 0.0, d1 = act ? 0.5 * (x.u_r - x0.u_r) : 0.0;
    const double d2 = act ? 0.5 * (x.v_t - x0.v_t) : 0.0, d3 = act ? 0.5 * (x.v_b - x0.v_b) : 0.0;
    const double dH = act ? x.H - x0.H : 0.0;
    F.cdr[a][b] = d1;
    F.cdb[a][b] = d3;
    __syncthreads();
    if (!in) return;
    double d = 0.0;
    if (b > 0) d = d + F.cdr[a][b - 1];
    Uo[ku] = pl ? x0.u_l : x0.u_l + 0.5 * (d + d0);
    d = 0.0;
    if (a > 0) d = d + F.cdb[a - 1][b];
    Uo[kv] = pt ? x0.v_t : x0.v_t + 0.5 * (d + d2);
    Uo[kH] = x0.H + 0.5 * dH;
    if (j == nx - 1) Uo[ku + 1] = x0.u_r + 0.5 * (0.0 + d1);
    if (i == ny - 1) Uo[kv + nx] = x0.v_b + 0.5 * (0.0 + d3);
    if (pt) Po.top[kt] = d2;
    if (pb) Po.bot[kt + nx] = d3;
    if (pl) Po.lft[kl] = d0;
    if (pr) Po.rgt[kl + ny] = d1;
}

// adds the last sweep's pending updates of tile (bx, by)'s top row and left column; a wave a tile
template <int TX, int TY>
__device__ __forceinline__ void fold_finish_tile(int ny, int nx, double *__restrict__ U, const FoldPending &P, int bx, int by,
                                                 int lane)
{
    static_assert(TX == 64 && TY <= 64, "a wave covers the tile's top row and left column");
    const int i0 = by * TY, j0 = bx * TX, j = j0 + lane, i = i0 + lane;
    if (by > 0 && j < nx) {
        const size_t k = (size_t)by * nx + j;
        U[n_u(ny, nx) + (size_t)i0 * nx + j] += 0.5 * ((0.0 + P.bot[k]) + P.top[k]);
    }
    if (bx > 0 && lane < TY && i < ny) {
        const size_t k = (size_t)bx * ny + i;
        U[(size_t)i * (nx + 1) + j0] += 0.5 * ((0.0 + P.rgt[k]) + P.lft[k]);
    }
}

// Several Vanka sweeps in one launch, for levels whose sweeps leave most of the
// chip idle: there a sweep by itself is one wave's Newton chain (0.61 us an
// iteration) and as much again for the launch, the first loads and the stores
// (5.9 us at 16^2 to 128^2).  A workgroup of MS x MS threads keeps MS x MS
// cells' state in LDS, one cell a thread, and runs ns sweeps on it.  A cell's
// update reads faces that cells up to 2 away update, so 2 rows and columns a
// sweep go stale at each side of the tile that is not the level's edge; what
// is left of the tile after ns sweeps is the (MS + 1 - 4 ns)^2 cells that the
// workgroup owns (their left and top faces, the level's last face column and
// row where its cells reach them).  Level dimensions up to MS have no such
// sides and any number of sweeps.  Cells are computed by several workgroups,
// from the same inputs with the same bits as by vanka_tile and apply_tile.
// A sweep of ten, before (one to a launch, its apply pass in the kernel) and
// after: 16^2 12.0 -> 7.7 us, 32^2 12.0 -> 9.1, 64^2 12.3 -> 9.1, 128^2 12.5 -> 10.0.
// At 13 x 13 cells a workgroup and one sweep a launch it still beats the sweep
// and apply kernels: 208^2 15.2 -> 12.7 us.  The 128^2 reference step took 24.4 ms,
// 17.7 now.
constexpr int MS = 16;
struct MultiLDS {
    double u[MS + 2][MS + 1];   // rows i0-1 .. i0+MS (clamped), face columns j0 .. j0+MS
    double v[MS + 1][MS + 2];   // face rows i0 .. i0+MS, columns j0-1 .. j0+MS (clamped)
    double H[MS + 2][MS + 2], n[MS + 2][MS + 2], S[MS + 2][MS + 2], be[MS + 2][MS + 2];   // the cells and a ring
    double cdr[MS][MS], cdb[MS][MS];   // the cells' updates of their right and bottom faces
};
// cells of a dimension of n that a workgroup owns after ns sweeps
__host__ __device__ inline int multi_own(int n, int ns) { return n <= MS ? n : MS + 1 - 4 * ns; }
// first cell of the tile that owns cells io ..: 2 ns more at the top and left, and inside the level where that has room
__host__ __device__ inline int multi_origin(int io, int n, int ns)
{
    const int o = io - 2 * ns < n - MS ? io - 2 * ns : n - MS;
    return o > 0 ? o : 0;
}

template <bool LOCAL>
__device__ __forceinline__ void vanka_multi_tile(const GlideGeom &g, const Params &p, const double *U, double *Uo,
                                                 const double *__restrict__ f, const double *__restrict__ bed,
                                                 const double *__restrict__ B, const double *__restrict__ beta,
                                                 const double *__restrict__ gamma, const unsigned char *__restrict__ blk,
                                                 int nbx, int n_newton, int ns, int bx, int by, MultiLDS &L)
{
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    const int oy = multi_own(ny, ns), ox = multi_own(nx, ns);
    const int io = by * oy, jo = bx * ox;   // owned cells [io, io + oy) x [jo, jo + ox)
    const int i0 = multi_origin(io, ny, ns), j0 = multi_origin(jo, nx, ns);
    const int tid = threadIdx.y * MS + threadIdx.x;
    const bool in = i0 + (int)threadIdx.y < ny && j0 + (int)threadIdx.x < nx;
    // threads past the level's edge run its nearest cell and drop the result (a
    // wave with idle lanes ran its chain slower)
    const int i = min(i0 + (int)threadIdx.y, ny - 1), j = min(j0 + (int)threadIdx.x, nx - 1), a = i - i0, b = j - j0;
    for (int k = tid; k < (MS + 2) * (MS + 1); k += MS * MS) {
        const int ru = k / (MS + 1), cu = k - ru * (MS + 1);
        L.u[ru][cu] = U[(size_t)clampi(i0 - 1 + ru, 0, ny - 1) * (nx + 1) + min(j0 + cu, nx)];
        const int rv = k / (MS + 2), cv = k - rv * (MS + 2);
        L.v[rv][cv] = U[nu + (size_t)min(i0 + rv, ny) * nx + clampi(j0 - 1 + cv, 0, nx - 1)];
    }
    const size_t ku = (size_t)i * (nx + 1) + j, kv = nu + (size_t)i * nx + j, kc = (size_t)i * nx + j;
    double H = U[nu + nv + kc];
    const bool act = !LOCAL || blk[(i / RB) * nbx + j / RB] != 0;
    if (!LOCAL || __syncthreads_or(in && act)) {   // uniform
        NewtonCell C;
        C.f0 = f[ku];
        C.f1 = f[ku + 1];
        C.f2 = f[kv];
        C.f3 = f[kv + nx];
        C.f4 = f[nu + nv + kc];
        C.bed = bed[kc];
        C.beta = beta[kc];
        C.th = gamma[kc];
        const double Bc = B[kc], glen_exp = (1.0 - p.n) / (2.0 * p.n);
        const NewtonK K = newton_constants(g.dx, g.dt);
        newton_edges<false>(C, K, i, j, ny, nx);
        for (int k = tid; k < (MS + 2) * (MS + 2); k += MS * MS) {   // the ring: 0 beyond the level's edge and the tile
            (&L.H[0][0])[k] = 0.0;
            (&L.n[0][0])[k] = 0.0;
            (&L.S[0][0])[k] = 0.0;
            (&L.be[0][0])[k] = 0.0;
        }
        const int bl = max(b - 1, 0), br = min(b + 2, MS), at = max(a - 1, 0), ab = min(a + 2, MS);
        for (int s = 0; s < ns; s++) {
            __syncthreads();   // the state (and, first, the cleared ring) is there
            NewtonX x;
            x.u_l = L.u[a + 1][b];
            x.u_r = L.u[a + 1][b + 1];
            x.v_t = L.v[a][b + 1];
            x.v_b = L.v[a + 1][b + 1];
            x.H = H;
            C.u_tl = L.u[a][b];
            C.u_tr = L.u[a][b + 1];
            C.u_bl = L.u[a + 2][b];
            C.u_br = L.u[a + 2][b + 1];
            C.v_lt = L.v[a][b];
            C.v_rt = L.v[a][b + 2];
            C.v_lb = L.v[a + 1][b];
            C.v_rb = L.v[a + 1][b + 2];
            C.u_ll = L.u[a + 1][bl];
            C.u_rr = L.u[a + 1][br];
            C.v_tt = L.v[at][b + 1];
            C.v_bb = L.v[ab][b + 1];
            C.e2 = eta2_from(i, j, ny, nx, x.u_l, x.u_r, x.v_t, x.v_b, C.u_tl, C.u_tr, C.u_bl, C.u_br, C.v_lt, C.v_rt,
                             C.v_lb, C.v_rb, Bc, p, glen_exp, K.dxi);
            const double sg = sigm_mid(fma(0.917, H, C.bed), p.gl_c), be = fma(sg, C.beta, (1.0 - sg) * p.water_drag);
            if (in) {
                L.H[a + 1][b + 1] = H;
                L.n[a + 1][b + 1] = C.e2 * H;
                L.S[a + 1][b + 1] = fmax(C.bed, -0.917 * H) + H;
                L.be[a + 1][b + 1] = be;
                // beyond the level's edge stands the edge cell's drag
                if (i == 0) L.be[a][b + 1] = be;
                if (i == ny - 1) L.be[a + 2][b + 1] = be;
                if (j == 0) L.be[a + 1][b] = be;
                if (j == nx - 1) L.be[a + 1][b + 2] = be;
            }
            __syncthreads();
            C.n_l = L.n[a + 1][b];
            C.n_r = L.n[a + 1][b + 2];
            C.n_t = L.n[a][b + 1];
            C.n_b = L.n[a + 2][b + 1];
            C.p_tl = (L.n[a][b] + C.n_t) + C.n_l;
            C.p_tr = C.n_t + L.n[a][b + 2];
            C.n_bl = L.n[a + 2][b];
            C.n_br = L.n[a + 2][b + 2];
            C.H_l = L.H[a + 1][b];
            C.H_r = L.H[a + 1][b + 2];
            C.H_t = L.H[a][b + 1];
            C.H_b = L.H[a + 2][b + 1];
            C.S_l = L.S[a + 1][b];
            C.S_r = L.S[a + 1][b + 2];
            C.S_t = L.S[a][b + 1];
            C.S_b = L.S[a + 2][b + 1];
            C.be_l = L.be[a + 1][b];
            C.be_r = L.be[a + 1][b + 2];
            C.be_t = L.be[a][b + 1];
            C.be_b = L.be[a + 2][b + 1];
            C.c_l = (C.v_lt - C.v_lb) * K.dxi;
            C.c_r = (C.v_rt - C.v_rb) * K.dxi;
            C.d_t = C.u_tr - C.u_tl;
            C.d_b = C.u_br - C.u_bl;
            const NewtonX x0 = x;
            newton_iterate(C, K, p, n_newton, x);
            // an idle cell's updates count as 0
            const double d0 = act ? 0.5 * (x.u_l - x0.u_l) : 0.0, d1 = act ? 0.5 * (x.u_r - x0.u_r) : 0.0;
            const double d2 = act ? 0.5 * (x.v_t - x0.v_t) : 0.0, d3 = act ? 0.5 * (x.v_b - x0.v_b) : 0.0;
            const double dH = act ? x.H - x0.H : 0.0;
            if (in) {
                L.cdr[a][b] = d1;
                L.cdb[a][b] = d3;
            }
            __syncthreads();   // all have read the state, too
            H = x0.H + 0.5 * dH;
            if (in) {
                double d = 0.0;
                if (b > 0) d = d + L.cdr[a][b - 1];
                L.u[a + 1][b] = x0.u_l + 0.5 * (d + d0);
                d = 0.0;
                if (a > 0) d = d + L.cdb[a - 1][b];
                L.v[a][b + 1] = x0.v_t + 0.5 * (d + d2);
                if (j == nx - 1) L.u[a + 1][b + 1] = x0.u_r + 0.5 * (0.0 + d1);
                if (i == ny - 1) L.v[a + 1][b + 1] = x0.v_b + 0.5 * (0.0 + d3);
            }
        }
    }
    // each thread stores the points that it updated itself
    if (LOCAL) __syncthreads();   // or, in an idle tile, that others loaded
    if (in && i >= io && i < io + oy && j >= jo && j < jo + ox) {
        Uo[ku] = L.u[a + 1][b];
        Uo[kv] = L.v[a][b + 1];
        Uo[nu + nv + kc] = H;
        if (j == nx - 1) Uo[ku + 1] = L.u[a + 1][b + 1];
        if (i == ny - 1) Uo[kv + nx] = L.v[a + 1][b + 1];
    }
}

// Local-smoother activation: one 16x16 workgroup per 14x14 reference block
// reads its 16x16 footprint (glide/solver.py:148-154, glide/cuda/vanka.cu:870-888).
__device__ __forceinline__ void activation_block(int ny, int nx, const double *__restrict__ r,
                                                 const double *__restrict__ U, const double *__restrict__ gamma,
                                                 unsigned char *__restrict__ blk, int bx, int by, int nbx,
                                                 int *__restrict__ any_active = nullptr)
{
    const int i = by * RB - 1 + (int)threadIdx.y, j = bx * RB - 1 + (int)threadIdx.x;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    int bad = 0;
    if (i >= 0 && i < ny && j >= 0 && j < nx) {
        size_t ci = (size_t)i * nx + j;
        double a = r[nu + nv + ci], b = U[nu + nv + ci] - gamma[ci];
        double fb = a + b - sqrt(a * a + b * b);
        double te = fabs(r[(size_t)i * (nx + 1) + j + 1]) + fabs(r[(size_t)i * (nx + 1) + j]) +
                    fabs(r[nu + (size_t)(i + 1) * nx + j]) + fabs(r[nu + (size_t)i * nx + j]) + fabs(fb);
        bad = te > 0.01;
    }
    int any = __syncthreads_or(bad);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        blk[by * nbx + bx] = (unsigned char)(any != 0);
        if (any && any_active) *any_active = 1;   // every writer stores the same value
    }
}

// ---------------------------------------------------------------------------
// Bilinear prolongation samples (glide/cuda/utility.cu:180-337)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double bilin(double ty, double tx, double v00, double v01, double v10, double v11)
{
    return (1.0 - ty) * ((1.0 - tx) * v00 + tx * v01) + ty * ((1.0 - tx) * v10 + tx * v11);
}
// coarse sample helper: value of (a[k] - b[k]) when b != NULL, else a[k]
__device__ __forceinline__ double cdiff(const double *__restrict__ a, const double *__restrict__ b, size_t k)
{
    return b ? a[k] - b[k] : a[k];
}
// bilinear u prolongation of (uc - wc) at fine face (j, i) (utility.cu:180-232)
__device__ __forceinline__ double prol_u_at(const double *uc, const double *wc, int j, int i, int nyc, int nxc)
{
    double Jf = (j - 0.5) * 0.5, If = i * 0.5;
    Jf = fmax(0.0, fmin(Jf, (double)(nyc - 1)));
    If = fmax(0.0, fmin(If, (double)nxc));
    int Jl = (int)Jf, Il = (int)If;
    int Jh = min(Jl + 1, nyc - 1), Ih = min(Il + 1, nxc);
    double ty = Jf - Jl, tx = If - Il;
    size_t s = nxc + 1;
    return bilin(ty, tx, cdiff(uc, wc, Jl * s + Il), cdiff(uc, wc, Jl * s + Ih), cdiff(uc, wc, Jh * s + Il),
                 cdiff(uc, wc, Jh * s + Ih));
}
// utility.cu:235-287
__device__ __forceinline__ double prol_v_at(const double *vc, const double *wc, int j, int i, int nyc, int nxc)
{
    double Jf = j * 0.5, If = (i - 0.5) * 0.5;
    Jf = fmax(0.0, fmin(Jf, (double)nyc));
    If = fmax(0.0, fmin(If, (double)(nxc - 1)));
    int Jl = (int)Jf, Il = (int)If;
    int Jh = min(Jl + 1, nyc), Ih = min(Il + 1, nxc - 1);
    double ty = Jf - Jl, tx = If - Il;
    size_t s = nxc;
    return bilin(ty, tx, cdiff(vc, wc, Jl * s + Il), cdiff(vc, wc, Jl * s + Ih), cdiff(vc, wc, Jh * s + Il),
                 cdiff(vc, wc, Jh * s + Ih));
}
// utility.cu:289-337
__device__ __forceinline__ double prol_H_at(const double *hc, const double *wc, int j, int i, int nyc, int nxc)
{
    double Jf = (j - 0.5) * 0.5, If = (i - 0.5) * 0.5;
    Jf = fmax(0.0, fmin(Jf, (double)(nyc - 1)));
    If = fmax(0.0, fmin(If, (double)(nxc - 1)));
    int Jl = (int)Jf, Il = (int)If;
    int Jh = min(Jl + 1, nyc - 1), Ih = min(Il + 1, nxc - 1);
    double ty = Jf - Jl, tx = If - Il;
    size_t s = nxc;
    return bilin(ty, tx, cdiff(hc, wc, Jl * s + Il), cdiff(hc, wc, Jl * s + Ih), cdiff(hc, wc, Jh * s + Il),
                 cdiff(hc, wc, Jh * s + Ih));
}

// ---------------------------------------------------------------------------
// Linearisation, LDS-staged like the residual: JVP j = J(U) d
// (glide/cuda/residuals.cu:299-579) and the gather-form VJP l = J(U)^T lambda
// (residuals.cu:586-1023; the (u, v) block through its symmetry, as a JVP
// along lambda with a zero thickness direction).  Every cell of the tile and
// the ring around it yields 2 eta H and its derivative, the directional
// derivatives of its normal stresses, its surface, drag and the direction (or
// lambda_H (1 - mask)) once into LDS, every vertex the derivative of its shear
// stress; each point then sums its terms from LDS.  The velocities are read
// from the caches, where a tile's rows stay, which leaves the LDS to four
// workgroups per CU instead of three.
//
// Rounding as in the residual: every output sums its terms in the per-point
// form's order, with powers of two on the constants, the short exp and log,
// and a factor of 0 where a term vanishes at the domain edge, so the bits are
// those of the per-point form up to the sign of zeros.  On new data each pass,
// JVP of 512^2 21.2 -> 14.6 us, VJP of 333 x 517 16.5 -> 14.5; in the caches, JVP of
// 1024^2 71 -> 49 (the staged form before, which kept the velocities in LDS and
// evaluated each face's terms).
//
// The tiles cover the cells (cdiv(nx, TX) x cdiv(ny, TY)); the faces at j = nx
// and i = ny go with the last tiles as in the residual.
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct LinLDS {
    // cells [i0-1+a][j0-1+b], clamped
    double n[TY + 2][TX + 2];    // 2 eta H (0 outside the domain)
    double hd[TY + 2][TX + 2];   // H (2 eta)' (0 outside)
    double eh[TY + 2][TX + 2];   // JVP: 2 eta H' (0 outside); VJP: 2 eta
    double tx[TY + 2][TX + 2], ty[TY + 2][TX + 2];   // derivatives of sigma_xx, sigma_yy (0 outside)
    double H[TY + 2][TX + 2];
    double dH[TY + 2][TX + 2];   // direction, or lambda_H (1 - mask)
    double S[TY + 2][TX + 2];    // surface
    double sl[TY + 2][TX + 2];   // d surface / d H
    double be[TY + 2][TX + 2];   // drag
    double db[TY + 2][TX + 2];   // d drag / d H (gl_derivatives)
    double cd[TY][TX];           // -d calving / d H of cell [i0+a][j0+b]
    double txy[TY + 1][TX + 1];  // 8 x derivative of sigma_xy, vertices [i0+a][j0+b]
};

// the general form's eII^q and its derivative factor, for arguments out of the short forms' range
__device__ __forceinline__ void glen_pow_dual(double x, double q, double &v, double &c)
{
    const double lg = log_normal(x), y0 = q * lg, y1 = (q - 1.0) * lg;
    v = exp_mid(y0);
    c = q * exp_mid(y1);
    if (!(x >= 2.2250738585072014e-308 && x <= 1.7976931348623157e308 && fabs(y0) <= 700.0 && fabs(y1) <= 700.0)) {
        if (x == 0.0) {   // dm_pow's own value at 0 (only reachable with eps_reg = 0)
            v = dm_pow(x, q);
            c = q * dm_pow(x, q - 1.0);
        } else {
            const double l = dm_log(x);
            v = dm_exp(q * l);
            c = q * dm_exp((q - 1.0) * l);
        }
    }
}

template <int TX, int TY>
struct LinLDS0 : LinLDS<TX, TY> {
    __device__ __forceinline__ void keep(int, int, double, double) {}
};
// ... with the smoother's 2 eta and 2 eta H, whose viscosity rounds differently (fma, eta2_from)
template <int TX, int TY>
struct AdjLDS : LinLDS<TX, TY> {
    double s_e2[TY + 2][TX + 2], s_n[TY + 2][TX + 2];
    __device__ __forceinline__ void keep(int a, int b, double e2, double n)
    {
        s_e2[a][b] = e2;
        s_n[a][b] = n;
    }
};

// One tile: stage() fills the LDS (all threads), then the rows may be asked
// for: u faces (i0.., j0..j0+TX), v faces (i0..i0+TY, j0..), cells.  ADJ: LDS is an AdjLDS.
template <int TX, int TY, bool VJP, bool ADJ, int NT = TX * TY>
struct LinTile {
    using LDS = typename std::conditional<ADJ, AdjLDS<TX, TY>, LinLDS0<TX, TY>>::type;
    static constexpr int NALL = (TY + 2) * (TX + 2);
    LDS &S;
    const Params &p;
    const int ny, nx, i0, j0, rb, cb;
    const TileField tu, tc;
    const char *bu, *bv, *bH, *du, *dv, *dH, *bbed, *bB, *bbeta, *bmask;
    const NewtonK K;

    __device__ __forceinline__ LinTile(LDS &S_, const GlideGeom &g, const Params &p_, const double *__restrict__ U,
                                       const double *__restrict__ D, const double *__restrict__ bed,
                                       const double *__restrict__ B, const double *__restrict__ beta,
                                       const double *__restrict__ mask, int bx, int by)
        : S(S_), p(p_), ny(g.ny), nx(g.nx), i0(by * TY), j0(bx * TX), rb(max(i0 - 2, 0)), cb(max(j0 - 2, 0)),
          tu(nx + 1, rb, cb), tc(nx, rb, cb), K(newton_constants(g.dx, g.dt))
    {
        const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
        bu = tu.base(U), bv = tc.base(U + nu), bH = tc.base(U + nu + nv);
        du = tu.base(D), dv = tc.base(D + nu), dH = tc.base(D + nu + nv);
        bbed = tc.base(bed), bB = tc.base(B), bbeta = tc.base(beta), bmask = tc.base(mask);
    }
    // byte offsets of (row, column), clamped to the field
    __device__ __forceinline__ uint32_t ou(int i, int j) const
    {
        return (uint32_t)(clampi(i, 0, ny - 1) - rb) * tu.pitch + 8u * (clampi(j, 0, nx) - cb);
    }
    __device__ __forceinline__ uint32_t ov(int i, int j) const
    {
        return (uint32_t)(clampi(i, 0, ny) - rb) * tc.pitch + 8u * (clampi(j, 0, nx - 1) - cb);
    }

    __device__ __forceinline__ void stage() const
    {
        const int tid = threadIdx.y * TX + threadIdx.x;
        const double glen_exp = (1.0 - p.n) / (2.0 * p.n);
        // 1. per cell
    #pragma unroll 1
        for (int k = tid; k < NALL; k += NT) {
            const int a = k / (TX + 2), b = k - a * (TX + 2);
            const int ci = i0 - 1 + a, cj = j0 - 1 + b;
            const int ic = clampi(ci, 0, ny - 1), jc = clampi(cj, 0, nx - 1);
            const uint32_t r0 = ic - rb, c0 = 8u * (jc - cb), u0 = r0 * tu.pitch + c0, v0 = r0 * tc.pitch + c0;
            const double h = ld_off(bH, v0), bd = ld_off(bbed, v0), bt = ld_off(bbeta, v0);
            double hd = ld_off(dH, v0);
            if (VJP) hd = hd * (1.0 - ld_off(bmask, v0));
            double n = 0.0, nh = 0.0, ne = 0.0, tx = 0.0, ty = 0.0, se = 0.0;
            if (ic == ci && jc == cj) {
                const uint32_t v1 = v0 + tc.pitch;   // row i+1 of v and column j+1 of u exist for every cell
                const bool t = ci > 0, bo = ci < ny - 1, l = cj > 0, r = cj < nx - 1;
                const uint32_t ut = t ? u0 - tu.pitch : u0, ub = bo ? u0 + tu.pitch : u0, cl = l ? 8u : 0u, cr = r ? 8u : 0u;
                const double u_l = ld_off(bu, u0), u_r = ld_off(bu, u0 + 8), v_t = ld_off(bv, v0), v_b = ld_off(bv, v1);
                const double x_l = ld_off(du, u0), x_r = ld_off(du, u0 + 8), y_t = ld_off(dv, v0), y_b = ld_off(dv, v1);
                const double V_tl = t && l ? K.dxi : 0.0, V_tr = t && r ? K.dxi : 0.0, V_bl = bo && l ? K.dxi : 0.0,
                             V_br = bo && r ? K.dxi : 0.0;
                // corner shear rates (doubled) and their derivatives
                const double e_tl = (ld_off(bu, ut) - u_l) * V_tl + (v_t - ld_off(bv, v0 - cl)) * V_tl;
                const double e_tr = (ld_off(bu, ut + 8) - u_r) * V_tr + (ld_off(bv, v0 + cr) - v_t) * V_tr;
                const double e_bl = (u_l - ld_off(bu, ub)) * V_bl + (v_b - ld_off(bv, v1 - cl)) * V_bl;
                const double e_br = (u_r - ld_off(bu, ub + 8)) * V_br + (ld_off(bv, v1 + cr) - v_b) * V_br;
                const double d_tl = (ld_off(du, ut) - x_l) * V_tl + (y_t - ld_off(dv, v0 - cl)) * V_tl;
                const double d_tr = (ld_off(du, ut + 8) - x_r) * V_tr + (ld_off(dv, v0 + cr) - y_t) * V_tr;
                const double d_bl = (x_l - ld_off(du, ub)) * V_bl + (y_b - ld_off(dv, v1 - cl)) * V_bl;
                const double d_br = (x_r - ld_off(du, ub + 8)) * V_br + (ld_off(dv, v1 + cr) - y_b) * V_br;
                const double a_ = u_r - u_l, b_ = v_t - v_b;
                const double ux = a_ * K.dxi, vy = b_ * K.dxi, uxd = (x_r - x_l) * K.dxi, vyd = (y_t - y_b) * K.dxi;
                const double e2 = ((e_tl * e_tl + e_tr * e_tr) + e_bl * e_bl) + e_br * e_br;
                const double e2d = ((fma(e_tl, d_tl, d_tl * e_tl) + fma(e_tr, d_tr, d_tr * e_tr)) + fma(e_bl, d_bl, d_bl * e_bl)) +
                                   fma(e_br, d_br, d_br * e_br);
                if (ADJ) {
                    se = eta2_from(ci, cj, ny, nx, u_l, u_r, v_t, v_b, ld_off(bu, ut), ld_off(bu, ut + 8), ld_off(bu, ub),
                                             ld_off(bu, ub + 8), ld_off(bv, v0 - cl), ld_off(bv, v0 + cr), ld_off(bv, v1 - cl),
                                             ld_off(bv, v1 + cr), ld_off(bB, v0), p, glen_exp, K.dxi);
                }
                const double eII = fma(0.0625, e2, (ux * ux + vy * vy) + ux * vy) + p.eps_reg;
                const double eIId = fma(0.0625, e2d, (fma(ux, uxd, uxd * ux) + fma(vy, vyd, vyd * vy)) + fma(ux, vyd, uxd * vy));
                double pv, pc;
                glen_pow_dual(eII, glen_exp, pv, pc);
                const double Bc = ld_off(bB, v0);
                const double ev = pv * Bc, ed = (pc * eIId) * Bc;   // 2 eta and its derivative
                n = ev * h;
                nh = h * ed;
                ne = VJP ? ev : ev * hd;
                const double nd = VJP ? nh : nh + ne;
                const double ex = fma(a_, K.dxi2, b_ * K.dxi), ey = fma(a_, K.dxi, b_ * K.dxi2);
                const double p1 = n * K.dxi, p2 = p1 + p1;
                tx = (((p2 * x_r - p2 * x_l) + p1 * y_t) - p1 * y_b) + ex * nd;
                ty = (((p1 * x_r - p1 * x_l) + p2 * y_t) - p2 * y_b) + ey * nd;
            }
            const double z = fma(0.917, h, bd), gr = sigm_mid(z, p.gl_c), g1 = 1.0 - gr, Hf = -0.917 * h;
            double njd = p.calving_rate * g1, db = 0.0;
            if (p.gl_derivatives) {
                const double dg = 0.917 * (p.gl_c * gr * g1);
                njd = -fma(p.calving_rate * h, dg, -njd);
                db = dg * (bt - p.water_drag);
            }
            S.n[a][b] = n;
            S.keep(a, b, se, se * h);
            S.hd[a][b] = nh;
            S.eh[a][b] = ne;
            S.tx[a][b] = tx;
            S.ty[a][b] = ty;
            S.H[a][b] = h;
            S.dH[a][b] = hd;
            S.S[a][b] = fmax(bd, Hf) + h;
            S.sl[a][b] = bd > Hf ? 1.0 : 1.0 + -0.917;
            S.be[a][b] = fma(gr, bt, g1 * p.water_drag);
            S.db[a][b] = db;
            if (a >= 1 && a <= TY && b >= 1 && b <= TX) S.cd[a - 1][b - 1] = njd;
        }
        __syncthreads();
        // 2. per vertex, 0 on the domain edge
    #pragma unroll 1
        for (int k = tid; k < (TY + 1) * (TX + 1); k += NT) {
            const int a = k / (TX + 1), b = k - a * (TX + 1);   // vertex (i0 + a, j0 + b): cells [a..a+1][b..b+1]
            const int vi = i0 + a, vj = j0 + b;
            double t8 = 0.0;
            if (vi > 0 && vi < ny && vj > 0 && vj < nx) {
                const uint32_t ub = (uint32_t)(vi - rb) * tu.pitch + 8u * (vj - cb), ut = ub - tu.pitch;
                const uint32_t vr = (uint32_t)(vi - rb) * tc.pitch + 8u * (vj - cb), vl = vr - 8;
                const double m = ((S.n[a][b] + S.n[a][b + 1]) + S.n[a + 1][b]) + S.n[a + 1][b + 1];
                const double md =
                    VJP ? ((S.hd[a][b] + S.hd[a][b + 1]) + S.hd[a + 1][b]) + S.hd[a + 1][b + 1]
                        : ((((((S.hd[a][b] + S.eh[a][b]) + S.hd[a][b + 1]) + S.eh[a][b + 1]) + S.hd[a + 1][b]) + S.eh[a + 1][b]) +
                           S.hd[a + 1][b + 1]) +
                              S.eh[a + 1][b + 1];
                const double q = m * K.dxi;
                const double x = fma(ld_off(bu, ut) - ld_off(bu, ub), K.dxi, (ld_off(bv, vr) - ld_off(bv, vl)) * K.dxi);
                t8 = (((q * ld_off(du, ut) - q * ld_off(du, ub)) - q * ld_off(dv, vl)) + q * ld_off(dv, vr)) + x * md;
            }
            S.txy[a][b] = t8;
        }
        __syncthreads();
    }
    // u face (i, j): J_u d (glide/cuda/residuals.cu:378-499)
    __device__ __forceinline__ double u_row(int i, int j) const
    {
        const int a = i - i0 + 1, b = j - j0 + 1;
        const uint32_t o = ou(i, j);
        const double u_l = ld_off(bu, o), x_l = ld_off(du, o);
        const double H_l = S.H[a][b - 1], H_c = S.H[a][b], s = H_l + H_c, F = j > 0 && j < nx ? K.hdx : 0.0;
        double d = S.tx[a][b] * K.dxi;
        d -= S.tx[a][b - 1] * K.dxi;
        d += S.txy[a - 1][b - 1] * K.edx;
        d -= S.txy[a][b - 1] * K.edx;
        double q = (S.be[a][b - 1] + S.be[a][b]) * x_l;
        if (!VJP) {
            if (p.gl_derivatives)
                q = (q + (S.db[a][b - 1] * u_l) * S.dH[a][b - 1]) + (S.db[a][b] * u_l) * S.dH[a][b];
            d = fma(-0.5, q, d);
            const double dS = (S.S[a][b] - S.S[a][b - 1]) * F;
            d -= fma(-(s * S.sl[a][b - 1]), F, dS) * S.dH[a][b - 1] + fma(s * S.sl[a][b], F, dS) * S.dH[a][b];
        } else {   // plus the mass rows through the fluxes of this face
            d = fma(-0.5, q, d);
            const double D2 = fma(-copysign(1.0, u_l), H_c - H_l, s);
            d = ((S.dH[a][b - 1] * D2) * F - (S.dH[a][b] * D2) * F) + d;
        }
        return d;
    }
    // v face (i, j) (residuals.cu:501-576)
    __device__ __forceinline__ double v_row(int i, int j) const
    {
        const int a = i - i0 + 1, b = j - j0 + 1;
        const uint32_t o = ov(i, j);
        const double v_t = ld_off(bv, o), y_t = ld_off(dv, o);
        const double H_t = S.H[a - 1][b], H_c = S.H[a][b], s = H_t + H_c, F = i > 0 && i < ny ? K.hdx : 0.0;
        double d = S.ty[a - 1][b] * K.dxi;
        d -= S.ty[a][b] * K.dxi;
        d -= S.txy[a - 1][b - 1] * K.edx;
        d += S.txy[a - 1][b] * K.edx;
        double q = (S.be[a - 1][b] + S.be[a][b]) * y_t;
        if (!VJP) {
            if (p.gl_derivatives)
                q = (q + (S.db[a - 1][b] * v_t) * S.dH[a - 1][b]) + (S.db[a][b] * v_t) * S.dH[a][b];
            d = fma(-0.5, q, d);
            const double dS = (S.S[a - 1][b] - S.S[a][b]) * F;
            d -= fma(s * S.sl[a - 1][b], F, dS) * S.dH[a - 1][b] + fma(-(s * S.sl[a][b]), F, dS) * S.dH[a][b];
        } else {
            d = fma(-0.5, q, d);
            const double D2 = fma(-copysign(1.0, v_t), H_t - H_c, s);
            d = ((S.dH[a][b] * D2) * F - (S.dH[a - 1][b] * D2) * F) + d;
        }
        return d;
    }
    // cell (i, j)
    __device__ __forceinline__ double h_row(int i, int j) const
    {
        const int a = i - i0 + 1, b = j - j0 + 1;
        const uint32_t u0 = ou(i, j), v0 = ov(i, j), v1 = v0 + tc.pitch;
        const double u_l = ld_off(bu, u0), u_r = ld_off(bu, u0 + 8), v_t = ld_off(bv, v0), v_b = ld_off(bv, v1);
        const double x_l = ld_off(du, u0), x_r = ld_off(du, u0 + 8), y_t = ld_off(dv, v0), y_b = ld_off(dv, v1);
        const double F_l = j > 0 ? K.hdx : 0.0, F_r = j + 1 < nx ? K.hdx : 0.0, F_t = i > 0 ? K.hdx : 0.0,
                     F_b = i + 1 < ny ? K.hdx : 0.0;
        const double H = S.H[a][b], H_l = S.H[a][b - 1], H_r = S.H[a][b + 1], H_t = S.H[a - 1][b], H_b = S.H[a + 1][b];
        const double s_l = H_l + H, s_r = H + H_r, s_t = H_t + H, s_b = H + H_b;
        const double m_l = u_l - fabs(u_l), q_r = u_r + fabs(u_r), q_t = v_t + fabs(v_t), m_b = v_b - fabs(v_b);
        const double h = S.dH[a][b], h_l = S.dH[a][b - 1], h_r = S.dH[a][b + 1], h_t = S.dH[a - 1][b], h_b = S.dH[a + 1][b];
        if (!VJP) {   // mass row (residuals.cu:343-375)
            double d = div_refined(h, K.dt, K.rdt);
            d += S.cd[a - 1][b - 1] * h;
            d -= ((fma(-copysign(1.0, u_l), H - H_l, s_l) * x_l + (u_l + fabs(u_l)) * h_l) + m_l * h) * F_l;
            d += ((fma(-copysign(1.0, u_r), H_r - H, s_r) * x_r + q_r * h) + (u_r - fabs(u_r)) * h_r) * F_r;
            d += ((fma(-copysign(1.0, v_t), H_t - H, s_t) * y_t + (v_t - fabs(v_t)) * h_t) + q_t * h) * F_t;
            d -= ((fma(-copysign(1.0, v_b), H - H_b, s_b) * y_b + m_b * h) + (v_b + fabs(v_b)) * h_b) * F_b;
            const double m = ld_off(bmask, v0);
            return (1.0 - m) * d + m * h;
        }
        // VJP: every row's derivative with respect to H(i, j).  Own mass row (residuals.cu:648-690)
        double acc = div_refined(h, K.dt, K.rdt);
        acc += h * S.cd[a - 1][b - 1];
        acc -= (h * m_l) * F_l;
        acc += (h * q_r) * F_r;
        acc += (h * q_t) * F_t;
        acc -= (h * m_b) * F_b;
        acc += ld_off(dH, v0) * ld_off(bmask, v0);
        // neighbours' mass rows through the shared faces
        acc += (h_l * m_l) * F_l;
        acc -= (h_r * q_r) * F_r;
        acc -= (h_t * q_t) * F_t;
        acc += (h_b * m_b) * F_b;
        // momentum rows through eta*H of this cell: normal stresses
        const double e2 = S.eh[a][b];
        {
            const double du_ = u_r - u_l, dv_ = v_t - v_b;
            const double ex = fma(du_, K.dxi2, dv_ * K.dxi), ey = fma(du_, K.dxi, dv_ * K.dxi2);
            acc += ((x_l * ex) * e2) * K.dxi;
            acc -= ((x_r * ex) * e2) * K.dxi;
            acc -= ((y_t * ey) * e2) * K.dxi;
            acc += ((y_b * ey) * e2) * K.dxi;
        }
        // shear stresses of the four corner vertices
        {
            const uint32_t ut = i > 0 ? u0 - tu.pitch : u0, ub = i < ny - 1 ? u0 + tu.pitch : u0, cl = j > 0 ? 8u : 0u,
                           cr = j < nx - 1 ? 8u : 0u;
            const double V_tl = i > 0 && j > 0 ? K.dxi : 0.0, V_tr = i > 0 && j < nx - 1 ? K.dxi : 0.0,
                         V_bl = i < ny - 1 && j > 0 ? K.dxi : 0.0, V_br = i < ny - 1 && j < nx - 1 ? K.dxi : 0.0;
            double e = fma(ld_off(bu, ut) - u_l, V_tl, (v_t - ld_off(bv, v0 - cl)) * V_tl);
            double w = ((x_l - ld_off(du, ut)) - y_t) + ld_off(dv, v0 - cl);
            acc += ((w * e) * e2) * K.edx;
            e = fma(ld_off(bu, ut + 8) - u_r, V_tr, (ld_off(bv, v0 + cr) - v_t) * V_tr);
            w = ((x_r - ld_off(du, ut + 8)) - ld_off(dv, v0 + cr)) + y_t;
            acc += ((w * e) * e2) * K.edx;
            e = fma(u_l - ld_off(bu, ub), V_bl, (v_b - ld_off(bv, v1 - cl)) * V_bl);
            w = ((ld_off(du, ub) - x_l) - y_b) + ld_off(dv, v1 - cl);
            acc += ((w * e) * e2) * K.edx;
            e = fma(u_r - ld_off(bu, ub + 8), V_br, (ld_off(bv, v1 + cr) - v_b) * V_br);
            w = ((ld_off(du, ub + 8) - x_r) - ld_off(dv, v1 + cr)) + y_b;
            acc += ((w * e) * e2) * K.edx;
        }
        // basal drag (grounding-line derivatives) and driving stress on the four faces
        const double Sc = S.S[a][b], sl = S.sl[a][b], db = -0.5 * S.db[a][b];
        if (p.gl_derivatives) acc += x_l * (db * u_l);
        acc -= x_l * fma(s_l * sl, F_l, (Sc - S.S[a][b - 1]) * F_l);
        if (p.gl_derivatives) acc += x_r * (db * u_r);
        acc -= x_r * fma(-(s_r * sl), F_r, (S.S[a][b + 1] - Sc) * F_r);
        if (p.gl_derivatives) acc += y_t * (db * v_t);
        acc -= y_t * fma(-(s_t * sl), F_t, (S.S[a - 1][b] - Sc) * F_t);
        if (p.gl_derivatives) acc += y_b * (db * v_b);
        acc -= y_b * fma(s_b * sl, F_b, (Sc - S.S[a + 1][b]) * F_b);
        return acc;
    }
};

// VJP: out = base - l when base != NULL (the adjoint residual f_adj - J^T lambda).
// STREAM: the output bypasses the caches (a level that they don't hold).
template <int TX, int TY, bool VJP, int NT, bool STREAM = false>
__device__ __forceinline__ void lin_tile_lds(const GlideGeom &g, const Params &p, double *__restrict__ out,
                                             const double *__restrict__ base, const double *__restrict__ U,
                                             const double *__restrict__ D, const double *__restrict__ bed,
                                             const double *__restrict__ B, const double *__restrict__ beta,
                                             const double *__restrict__ mask, int bx, int by, LinLDS0<TX, TY> &S)
{
    const LinTile<TX, TY, VJP, false, NT> T(S, g, p, U, D, bed, B, beta, mask, bx, by);
    T.stage();
    if (threadIdx.y >= TY) return;   // threads that only staged
    const int ny = g.ny, nx = g.nx, i = T.i0 + threadIdx.y, j = T.j0 + threadIdx.x;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    if (i > ny || j > nx) return;
    auto emit = [&](size_t k, double val) {
        if (VJP && base) val = base[k] - val;
        if (STREAM)
            __builtin_nontemporal_store(val, out + k);
        else
            out[k] = val;
    };
    auto urow = [&](int i, int j) { emit((size_t)i * (nx + 1) + j, T.u_row(i, j)); };
    auto vrow = [&](int i, int j) { emit(nu + (size_t)i * nx + j, T.v_row(i, j)); };
    if (i < ny) urow(i, j);
    if (j < nx) vrow(i, j);
    if (j == nx - 1 && T.j0 + TX == nx && i < ny) urow(i, nx);   // u face at j = nx
    if (i == ny - 1 && T.i0 + TY == ny && j < nx) vrow(ny, j);   // v face at i = ny
    if (i < ny && j < nx) emit(nu + nv + (size_t)i * nx + j, T.h_row(i, j));
}

// ---------------------------------------------------------------------------
// One colour of the adjoint smoother in one pass (glide/grid.py:319-330,
// glide/cuda/vanka.cu:441-840): r = f_adj - J^T lam, then every cell of the
// colour solves its transposed block against r and updates its five dofs.  A
// pass of its own for r and another for the solve cost two launches, two
// stagings and the trip of r through memory, each of them more than the
// arithmetic on the levels that fit the chip at once.
//
// The tiles read their neighbours' lam, so the updated lam goes to another
// array, every dof written once: by its cell of the colour (the cells of one
// colour own disjoint dofs), the thickness of the other cells and the domain
// edge faces of cells of the other colour by those.  The cells of the colour
// take the first half of the threads, so that whole waves solve.
// ---------------------------------------------------------------------------
template <int TX, int TY, int NT>
__device__ __forceinline__ void adjoint_tile(const GlideGeom &g, const Params &p, double *__restrict__ lam_out,
                                             double *__restrict__ r, const double *__restrict__ f_adj,
                                             const double *__restrict__ U, const double *__restrict__ lam,
                                             const double *__restrict__ bed, const double *__restrict__ B,
                                             const double *__restrict__ beta, const double *__restrict__ mask, int color,
                                             double omega, int bx, int by, AdjLDS<TX, TY> &S)
{
    const LinTile<TX, TY, true, true, NT> T(S, g, p, U, lam, bed, B, beta, mask, bx, by);
    T.stage();
    if (threadIdx.y >= TY) return;   // threads that only staged
    const int ny = g.ny, nx = g.nx;
    const size_t nu = n_u(ny, nx), nv = n_v(ny, nx);
    const int tid = threadIdx.y * TX + threadIdx.x, half = tid >= TX * TY / 2, q = tid - half * (TX * TY / 2);
    const int a = q / (TX / 2) + 1, i = T.i0 + a - 1, b = 2 * (q % (TX / 2)) + 1 + ((color + i + half) & 1), j = T.j0 + b - 1;
    if (i >= ny || j >= nx) return;
    const size_t ku = (size_t)i * (nx + 1) + j, kv0 = nu + (size_t)i * nx + j, kv1 = kv0 + nx, kh = kv0 + nv;
    if (half) {
        r[kh] = f_adj[kh] - T.h_row(i, j);
        lam_out[kh] = lam[kh];
        auto edge = [&](size_t k, double row) {
            r[k] = f_adj[k] - row;
            lam_out[k] = lam[k];
        };
        if (j == 0) edge(ku, T.u_row(i, 0));
        if (j == nx - 1) edge(ku + 1, T.u_row(i, nx));
        if (i == 0) edge(kv0, T.v_row(0, j));
        if (i == ny - 1) edge(kv1, T.v_row(ny, j));
        return;
    }
    double rhs[5], d[5];
    rhs[0] = f_adj[ku] - T.u_row(i, j);
    rhs[1] = f_adj[ku + 1] - T.u_row(i, j + 1);
    rhs[2] = f_adj[kv0] - T.v_row(i, j);
    rhs[3] = f_adj[kv1] - T.v_row(i + 1, j);
    rhs[4] = f_adj[kh] - T.h_row(i, j);
    r[ku] = rhs[0];
    r[ku + 1] = rhs[1];
    r[kv0] = rhs[2];
    r[kv1] = rhs[3];
    r[kh] = rhs[4];
    const char *bu = T.bu, *bv = T.bv;
    const uint32_t u0 = T.ou(i, j), v0 = T.ov(i, j), v1 = v0 + T.tc.pitch;
    const uint32_t ut = T.ou(i - 1, j), ub = T.ou(i + 1, j);
    NewtonX x;
    NewtonCell C{};
    x.u_l = ld_off(bu, u0);
    x.u_r = ld_off(bu, u0 + 8);
    x.v_t = ld_off(bv, v0);
    x.v_b = ld_off(bv, v1);
    x.H = S.H[a][b];
    C.u_tl = ld_off(bu, ut);
    C.u_tr = ld_off(bu, ut + 8);
    C.u_bl = ld_off(bu, ub);
    C.u_br = ld_off(bu, ub + 8);
    C.v_lt = ld_off(bv, T.ov(i, j - 1));
    C.v_lb = ld_off(bv, T.ov(i + 1, j - 1));
    C.v_rt = ld_off(bv, T.ov(i, j + 1));
    C.v_rb = ld_off(bv, T.ov(i + 1, j + 1));
    C.e2 = S.s_e2[a][b];
    C.n_l = S.s_n[a][b - 1];
    C.n_r = S.s_n[a][b + 1];
    C.n_t = S.s_n[a - 1][b];
    C.n_b = S.s_n[a + 1][b];
    C.p_tl = (S.s_n[a - 1][b - 1] + C.n_t) + C.n_l;
    C.p_tr = C.n_t + S.s_n[a - 1][b + 1];
    C.n_bl = S.s_n[a + 1][b - 1];
    C.n_br = S.s_n[a + 1][b + 1];
    C.H_l = S.H[a][b - 1];
    C.H_r = S.H[a][b + 1];
    C.H_t = S.H[a - 1][b];
    C.H_b = S.H[a + 1][b];
    C.S_l = S.S[a][b - 1];
    C.S_r = S.S[a][b + 1];
    C.S_t = S.S[a - 1][b];
    C.S_b = S.S[a + 1][b];
    C.be_l = S.be[a][b - 1];
    C.be_r = S.be[a][b + 1];
    C.be_t = S.be[a - 1][b];
    C.be_b = S.be[a + 1][b];
    newton_edges<false>(C, T.K, i, j, ny, nx);
    const double cd = S.cd[a - 1][b - 1];
    const NewtonCentre M{S.be[a][b], S.S[a][b], S.sl[a][b], 0.0, T.K.idt + cd, S.db[a][b]};
    const bool masked = mask[(size_t)i * nx + j] > 0.5;
    if (p.gl_derivatives)
        newton_adjoint<true>(C, T.K, M, x, masked, rhs, d);
    else
        newton_adjoint<false>(C, T.K, M, x, masked, rhs, d);
    lam_out[ku] = lam[ku] + 0.5 * omega * d[0];
    lam_out[ku + 1] = lam[ku + 1] + 0.5 * omega * d[1];
    lam_out[kv0] = lam[kv0] + 0.5 * omega * d[2];
    lam_out[kv1] = lam[kv1] + 0.5 * omega * d[3];
    lam_out[kh] = lam[kh] + omega * d[4];
}

}  // namespace glide
