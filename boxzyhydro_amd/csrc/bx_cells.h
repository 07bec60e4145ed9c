// bx_cells.h -- per-cell bodies of the exact call sequence (one reference
// subroutine's work on one cell), shared by the one-kernel-per-subroutine
// path (bx_exact.hip) and the batched boxes (bx_boxes.hip), so that both run
// the same arithmetic.  Arithmetic order follows the cited reference lines.
#pragma once

#include <type_traits>

#include "bx_internal.h"
#include "bx_math.h"

namespace bx {

// max-reduce non-negative doubles of a block (at most 1024 threads) into *dst
// (as IEEE bits)
__device__ __forceinline__ void block_max_to(double v, unsigned long long *dst)
{
    __shared__ double wmax[16];
    for (int off = 32; off > 0; off >>= 1) v = vmax(v, __shfl_xor(v, off, 64));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) wmax[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = wmax[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); k++) m = vmax(m, wmax[k]);
        // skip the atomic when the stored maximum is already larger
        const unsigned long long b = (unsigned long long)__double_as_longlong(m);
        if (b > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dst, b);
    }
}

// A maximum over a whole grid goes into kMaxSlots words, each in a cache line
// of its own, a block's share into the slot of its index; the host takes the
// largest.  One word for all cost about 9 ns per block: 46 us at 96^3 for a
// Courant pass that streams in 10.
__device__ __forceinline__ unsigned long long *max_slot(unsigned long long *slots)
{
    return slots + (blockIdx.x % kMaxSlots) * kMaxStride;
}

// 1-based (ix,iy,iz) of cell c (utils.f90:191-194 inverse)
__device__ __forceinline__ void coords(int64_t c, int nx, int ny, int &ix, int &iy, int &iz)
{
    int64_t plane = (int64_t)nx * ny;
    iz = (int)(c / plane) + 1;
    int64_t r = c - (int64_t)(iz - 1) * plane;
    iy = (int)(r / nx) + 1;
    ix = (int)(r - (int64_t)(iy - 1) * nx) + 1;
}

// init_grid.f90:81-107 ghost flag: 1 outer layer, 2 second layer, 0 interior
__device__ __forceinline__ int boundary_of(int ix, int iy, int iz, int nx, int ny, int nz)
{
    int f1 = (ix == 1 || ix == nx) || (iy == 1 || iy == ny) || (nz >= 6 && (iz == 1 || iz == nz));
    if (f1) return 1;
    int f2 = (ix == 2 || ix == nx - 1) || (iy == 2 || iy == ny - 1) || (nz >= 6 && (iz == 2 || iz == nz - 1));
    return f2 ? 2 : 0;
}

// One cell of the exact path in registers.
struct CellState {
    double U[5], v[3], p;
};

// state.f90:30-57, H2STAT=-1 branch: p, and E of a low-density cell
__device__ __forceinline__ void state_of(CellState &x, double gam, double seps, double muc, double rgas)
{
    const double rho = x.U[0];
    const double ekin = rho * 0.5 * (x.v[0] * x.v[0] + x.v[1] * x.v[1] + x.v[2] * x.v[2]);
    double eps = vmax(x.U[4] - ekin, seps);
    if (rho < 1e-4) {
        const double tk = vmin(5e3, x.p / (rho * rgas) * muc);
        const double pc = rho * tk * rgas / muc;
        x.p = pc;
        eps = pc / (gam - 1.0);
        x.U[4] = eps + ekin;
    } else {
        x.p = eps * (gam - 1.0);
    }
}

// velocity.f90:18-53: u = m/rho, vlimit clamp; returns max |u_d| before the
// clamp and whether it acted
__device__ __forceinline__ double velocity_of(CellState &x, double vlimit, double seps, bool &clamped)
{
    double vm = 0.0;
    const double rho = x.U[0];
    div_shared<3>(x.U + 1, rho, x.v);
    clamped = false;
    for (int d = 0; d < 3; d++) {
        vm = vmax(vm, fabs(x.v[d]));
        if (fabs(x.v[d]) > vlimit) clamped = true;
    }
    if (clamped) {
        double *m = x.U + 1, *v = x.v;
        double E = x.U[4];
        double ekin = 0.5 * (m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / rho;
        double speed = 0.0;
        for (int d = 0; d < 3; d++) speed = speed + v[d] * v[d];
        speed = sqrt(speed);
        for (int d = 0; d < 3; d++) {
            v[d] = v[d] * vlimit / speed;
            m[d] = v[d] * rho;
        }
        E = E - ekin;
        ekin = 0.5 * (m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / rho;
        x.U[4] = vmax(E, seps) + ekin;
    }
    return vm;
}

// source.f90:148-182 with the force g; with fluxangmom the terms of
// source.f90:73-90 come first (the pforce of source.f90:64-66 feeds nothing on
// the hydro path), x and y being the cell's centre
__device__ __forceinline__ void source_of(CellState &s, double dt, double g0, double g1, double g2, double seps,
                                          int ang, double x, double y)
{
    const double rho = s.U[0];
    double m0 = s.U[1], m1 = s.U[2], m2 = s.U[3];
    const double ux = s.v[0], uy = s.v[1], uz = s.v[2];
    if (ang) {
        const double r = sqrt(x * x + y * y);
        // r**4 as the reference's build evaluates it: a left-to-right product
        const double w = x * uy - y * ux, r4 = ((r * r) * r) * r;
        m1 = m1 + rho * (w * w) * y / r4 * dt;
        m0 = m0 + rho * (w * w) * x / r4 * dt;
    }
    m1 = m1 + (rho * g1) * dt;
    m0 = m0 + (rho * g0) * dt;
    m2 = m2 + (g2 * rho) * dt;
    const double ekin = 0.5 * (m0 * m0 + m1 * m1 + m2 * m2) / rho;
    s.U[1] = m0;
    s.U[2] = m1;
    s.U[3] = m2;
    s.U[4] = vmax(s.U[4] - ekin + dt * rho * (ux * g0 + uy * g1 + uz * g2), seps) + ekin;
}

// courant.f90:17-21: sum_d (c+|u_d|)/Delta_d
__device__ __forceinline__ double courant_of(const CellState &x, double ad, double dx, double dy, double dz)
{
    const double sound = sqrt(ad * x.p / x.U[0]);
    return (sound + fabs(x.v[0])) / dx + (sound + fabs(x.v[1])) / dy + (sound + fabs(x.v[2])) / dz;
}

__device__ __forceinline__ void state_cell(int64_t n, int64_t c, double *__restrict__ cons,
                                           const double *__restrict__ u, double *__restrict__ p,
                                           double *__restrict__ ad, double gam, double seps, double muc, double rgas)
{
    CellState x;
    x.U[0] = cons[c];
    x.U[4] = cons[4 * n + c];
    for (int d = 0; d < 3; d++) x.v[d] = u[d * n + c];
    const bool low = x.U[0] < 1e-4;
    if (low) x.p = p[c];
    state_of(x, gam, seps, muc, rgas);
    ad[c] = gam;
    if (low) cons[4 * n + c] = x.U[4];
    p[c] = x.p;
}

__device__ __forceinline__ double velocity_cell(int64_t n, int64_t c, double *__restrict__ cons,
                                                double *__restrict__ u, double vlimit, double seps)
{
    CellState x;
    for (int d = 0; d < 4; d++) x.U[d] = cons[d * n + c];
    x.U[4] = 0.0;
    bool clamped;
    double vm = 0.0;
    div_shared<3>(x.U + 1, x.U[0], x.v);
    for (int d = 0; d < 3; d++) vm = vmax(vm, fabs(x.v[d]));
    if (vm > vlimit || !(vm == vm) || fabs(x.v[0]) > vlimit || fabs(x.v[1]) > vlimit || fabs(x.v[2]) > vlimit) {
        x.U[4] = cons[4 * n + c];
        vm = velocity_of(x, vlimit, seps, clamped);
        if (clamped)
            for (int d = 1; d < 5; d++) cons[d * n + c] = x.U[d];
    }
    for (int d = 0; d < 3; d++) u[d * n + c] = x.v[d];
    return vm;
}

// courant.f90:17-21: the cell's sum_d (c+|u_d|)/Delta_d
__device__ __forceinline__ double courant_cell(int64_t n, int64_t c, const double *__restrict__ cons,
                                               const double *__restrict__ u, const double *__restrict__ p,
                                               const double *__restrict__ ad, double dx, double dy, double dz)
{
    CellState x;
    x.U[0] = cons[c];
    x.p = p[c];
    for (int d = 0; d < 3; d++) x.v[d] = u[d * n + c];
    return courant_of(x, ad[c], dx, dy, dz);
}

// source() on an interior cell with the gforce planes gf, or without them a
// uniform gravity vector g (the reference's g = -(phi(+)-phi(-))/(2d) = -0.0
// for phi=0)
__device__ __forceinline__ void source_cell(int64_t n, int64_t c, int nx, int ny, int nz, double *__restrict__ cons,
                                            const double *__restrict__ u, double dt, double g0, double g1, double g2,
                                            double seps, int ang, double dx, double dy,
                                            const double *__restrict__ gf)
{
    int ix, iy, iz;
    coords(c, nx, ny, ix, iy, iz);
    if (boundary_of(ix, iy, iz, nx, ny, nz) > 0) return;
    CellState x;
    for (int f = 0; f < 5; f++) x.U[f] = cons[f * n + c];
    for (int d = 0; d < 3; d++) x.v[d] = u[d * n + c];
    if (gf) {  // gforce(1:3, igrid) of calc_gforce / external_grav
        g0 = gf[c];
        g1 = gf[n + c];
        g2 = gf[2 * n + c];
    }
    source_of(x, dt, g0, g1, g2, seps, ang, centre(dx, ix, nx), centre(dy, iy, ny));
    for (int f = 1; f < 5; f++) cons[f * n + c] = x.U[f];
}

// utils.f90:314-403 as resolved on the host into (ghost, donor, momentum sign
// flips).  Donors that are ghosts are read from a snapshot taken first.
__device__ __forceinline__ void ghost_snapshot_one(int64_t n, int64_t ns, int64_t k, const int32_t *__restrict__ ssrc,
                                                   const double *__restrict__ planes, double *__restrict__ scratch)
{
    const int64_t s = ssrc[k];
    for (int f = 0; f < 5; f++) scratch[f * ns + k] = planes[f * n + s];
}

__device__ __forceinline__ void ghost_fill_one(int64_t n, int64_t k, const int32_t *__restrict__ dst,
                                               const int32_t *__restrict__ src, const int32_t *__restrict__ sign,
                                               double *__restrict__ planes, const double *__restrict__ scratch,
                                               int64_t ns)
{
    const int64_t d = dst[k];
    const int32_t s0 = src[k];
    const double *base;
    int64_t stride, s;
    if (s0 >= 0) {
        base = planes;
        stride = n;
        s = s0;
    } else {
        base = scratch;
        stride = ns;
        s = -(int64_t)s0 - 1;
    }
    const int sg = sign[k];
    planes[d] = base[s];
    for (int f = 1; f <= 3; f++) {
        double v = base[f * stride + s];
        planes[f * n + d] = ((sg >> (f - 1)) & 1) ? -v : v;
    }
    planes[4 * n + d] = base[4 * stride + s];
}

// ------------------------------------------ flux: one HLL flux per face
// The side of cell q in direction d (minus: pm=0, plus: pm=1) exactly as
// the reference forms it (flux.f90:253-295 slopes, 312-482 states).
// ANG: flux_ang.f90:301-482, with the r- and angular momenta, which get no
// transverse term.
struct AngGrid {
    double dx, dy, yoffset;
};
// the centre that flux_ang's momentum transform takes (with yoffset)
__device__ __forceinline__ AngCentre ang_centre(const AngGrid &g, int64_t c, int nx, int ny)
{
    const double x = centre(g.dx, (int)(c % nx) + 1, nx), y = centre(g.dy, (int)((c / nx) % ny) + 1, ny) + g.yoffset;
    return {x, y, sqrt(x * x + y * y)};
}
template <int d, bool ANG = false>
__device__ __forceinline__ Side<double> cell_side(int64_t q, int pm, int64_t n, int nx, int ny, int nz,
                                                 int64_t stride, const double *__restrict__ cons,
                                                 const double *__restrict__ u, const double *__restrict__ p,
                                                 const double *__restrict__ ad, double dt, double ds, double seps,
                                                 const AngGrid &ang = AngGrid{})
{
    int ix, iy, iz;
    coords(q, nx, ny, ix, iy, iz);
    const bool ghost = boundary_of(ix, iy, iz, nx, ny, nz) > 0;
    const double rho = cons[q], E = cons[4 * n + q];
    const double v[3] = {u[q], u[n + q], u[2 * n + q]};
    const double pc = p[q], gc = ad[q];
    const double eps = vmax(E - 0.5 * rho * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]), seps);
    const double sound = sqrt(pc * gc / rho);
    double su[3] = {0.0, 0.0, 0.0}, sp = 0.0, sd = 0.0, se = 0.0, sgm = 0.0;
    if (!ghost) {
        const int64_t cm = q - stride, cp = q + stride;
        for (int j = 0; j < 3; j++) su[j] = slope(u[j * n + cm], v[j], u[j * n + cp]);
        double em, ep;
        {
            const double r = cons[cm];
            const double a0 = u[cm], a1 = u[n + cm], a2 = u[2 * n + cm];
            em = vmax(cons[4 * n + cm] - 0.5 * r * (a0 * a0 + a1 * a1 + a2 * a2), seps);
        }
        {
            const double r = cons[cp];
            const double a0 = u[cp], a1 = u[n + cp], a2 = u[2 * n + cp];
            ep = vmax(cons[4 * n + cp] - 0.5 * r * (a0 * a0 + a1 * a1 + a2 * a2), seps);
        }
        sp = slope(p[cm], pc, p[cp]);
        sd = slope(cons[cm], rho, cons[cp]);
        se = slope(em, eps, ep);
        sgm = slope(ad[cm], gc, ad[cp]);
    }
    const double lp = vmax(v[d] + sound, 0.0) * dt / ds;
    const double lm = vmin(v[d] - sound, 0.0) * dt / ds;
    const double zc = 0.0 * (dt * 0.5 / ds);  // transverse terms: flux.f90:391-479
    double mi[7], pl[7];
    muscl(rho, lm, lp, sd, mi[0], pl[0]);
    for (int j = 0; j < 3; j++) muscl(v[j], lm, lp, su[j], mi[1 + j], pl[1 + j]);
    muscl(pc, lm, lp, sp, mi[4], pl[4]);
    muscl(eps, lm, lp, se, mi[5], pl[5]);
    muscl(gc, lm, lp, sgm, mi[6], pl[6]);
    const double *o = pm ? pl : mi;
    Side<double> sd7;
    sd7.d = o[0] + zc;
    sd7.v[0] = o[1] + zc;
    sd7.v[1] = o[2] + zc;
    sd7.v[2] = o[3] + zc;
    sd7.p = o[4] + zc;
    sd7.e = o[5] + zc;
    sd7.g = o[6] + zc;
    if constexpr (ANG) {
        double w[3][2];
        for (int k = -1; k <= 1; k++) {
            const int64_t e = ghost ? q : q + k * stride;
            ang_centre(ang, e, nx, ny).to(cons[n + e], cons[2 * n + e], w[k + 1][0], w[k + 1][1]);
        }
        double m[2], pp[2];
        for (int j = 0; j < 2; j++)
            muscl(w[1][j], lm, lp, ghost ? 0.0 : slope(w[0][j], w[1][j], w[2][j]), m[j], pp[j]);
        sd7.s1 = pm ? pp[0] : m[0];
        sd7.s2 = pm ? pp[1] : m[1];
    }
    return sd7;
}

// flux.f90:121-190 with each face computed once: F(d, c) is the HLL flux of
// the face between cell c and c + s_d (get_fluxes/flux_hll, flux.f90:486-590),
// for the faces some interior cell uses.  The reference forms every face
// twice, once from each side, from the same inputs and with the same result.
__device__ __forceinline__ void face_hll_cell(int64_t n, int64_t c, int nx, int ny, int nz, bool flatz,
                                              const double *__restrict__ cons, const double *__restrict__ u,
                                              const double *__restrict__ p, const double *__restrict__ ad,
                                              double *__restrict__ F, double dt, double dx, double dy, double dz,
                                              double seps)
{
    int ix, iy, iz;
    coords(c, nx, ny, ix, iy, iz);
    const bool in_c = boundary_of(ix, iy, iz, nx, ny, nz) == 0;
    const int64_t sz = flatz ? 0 : (int64_t)nx * ny;
    double f[5];
    // x face c+1/2: needed by c or c+1 when interior
    if (in_c || (ix < nx && boundary_of(ix + 1, iy, iz, nx, ny, nz) == 0)) {
        face_flux<double, 0>(cell_side<0>(c, 1, n, nx, ny, nz, 1, cons, u, p, ad, dt, dx, seps),
                             cell_side<0>(c + 1, 0, n, nx, ny, nz, 1, cons, u, p, ad, dt, dx, seps), f);
        for (int k = 0; k < 5; k++) F[(int64_t)k * n + c] = f[k];
    }
    if (in_c || (iy < ny && boundary_of(ix, iy + 1, iz, nx, ny, nz) == 0)) {
        face_flux<double, 1>(cell_side<1>(c, 1, n, nx, ny, nz, nx, cons, u, p, ad, dt, dy, seps),
                             cell_side<1>(c + nx, 0, n, nx, ny, nz, nx, cons, u, p, ad, dt, dy, seps), f);
        for (int k = 0; k < 5; k++) F[(int64_t)(5 + k) * n + c] = f[k];
    }
    if (in_c || (!flatz && iz < nz && boundary_of(ix, iy, iz + 1, nx, ny, nz) == 0)) {
        face_flux<double, 2>(cell_side<2>(c, 1, n, nx, ny, nz, sz, cons, u, p, ad, dt, dz, seps),
                             cell_side<2>(c + sz, 0, n, nx, ny, nz, sz, cons, u, p, ad, dt, dz, seps), f);
        for (int k = 0; k < 5; k++) F[(int64_t)(10 + k) * n + c] = f[k];
    }
}

// flux.f90:121-230 on the face fluxes: fluxtmp of an interior cell (zero on
// ghosts, flux.f90:51), the stage update and the floors
__device__ __forceinline__ void face_update_cell(int64_t n, int64_t c, int nx, int ny, int nz, bool flatz,
                                                 const double *__restrict__ F, double *__restrict__ cons,
                                                 const double *__restrict__ cons_old, int avg, double dt, double ayz,
                                                 double axz, double axy, double vol, double srho, double seps)
{
    int ix, iy, iz;
    coords(c, nx, ny, ix, iy, iz);
    double ftmp[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (boundary_of(ix, iy, iz, nx, ny, nz) == 0) {
        const int64_t sz = flatz ? 0 : (int64_t)nx * ny;
        for (int i = 0; i < 5; i++) {
            const double fx0 = F[(int64_t)i * n + c - 1], fx1 = F[(int64_t)i * n + c];
            const double fy0 = F[(int64_t)(5 + i) * n + c - nx], fy1 = F[(int64_t)(5 + i) * n + c];
            const double fz0 = F[(int64_t)(10 + i) * n + c - sz], fz1 = F[(int64_t)(10 + i) * n + c];
            ftmp[i] = -((ayz * (fx1 - fx0) + axz * (fy1 - fy0) + axy * (fz1 - fz0)) * dt / vol);
        }
    }
    double U[5];
    for (int i = 0; i < 5; i++) {
        const double ft = ftmp[i];
        const double cu = cons[(int64_t)i * n + c];
        U[i] = avg == 0 ? cu + ft : 0.5 * (cons_old[(int64_t)i * n + c] + cu + ft);
    }
    U[0] = vmax(U[0], srho);
    if (U[4] < 0.0) U[4] = 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) / U[0] + seps;
    for (int i = 0; i < 5; i++) cons[(int64_t)i * n + c] = U[i];
}

// The end of the flux subroutine on one cell with fluxtmp ft (flux.f90:205-228);
// ANG: in the transformed momenta, back to linear ones, then the floors
// (flux_ang.f90:223-281).
template <bool ANG>
__device__ __forceinline__ void flux_end(int64_t n, int64_t c, int nx, int ny, const double *__restrict__ cons,
                                         const double *__restrict__ cons_old, double *__restrict__ out, int avg,
                                         const double *ft, double srho, double seps, const AngGrid &ang)
{
    double cu[5], co[5] = {}, U[5];
    for (int i = 0; i < 5; i++) cu[i] = cons[i * n + c];
    if (avg)
        for (int i = 0; i < 5; i++) co[i] = cons_old[i * n + c];
    AngCentre tr;
    if constexpr (ANG) {
        tr = ang_centre(ang, c, nx, ny);
        double rm, am;
        tr.to(cu[1], cu[2], rm, am);
        cu[1] = rm;
        cu[2] = am;
        if (avg) {
            tr.to(co[1], co[2], rm, am);
            co[1] = rm;
            co[2] = am;
        }
    }
    for (int i = 0; i < 5; i++) U[i] = avg == 0 ? cu[i] + ft[i] : 0.5 * (co[i] + cu[i] + ft[i]);
    if constexpr (ANG) {
        double m1, m2;
        tr.back(U[1], U[2], m1, m2);
        U[1] = m1;
        U[2] = m2;
    }
    U[0] = vmax(U[0], srho);
    if (U[4] < 0.0) U[4] = 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) / U[0] + seps;
    for (int i = 0; i < 5; i++) out[i * n + c] = U[i];
}

// face_update_cell without the face planes: the six faces of an interior cell
// formed here, from cons, u, p and ad into the out planes.  ANG: flux_ang.f90.
template <bool ANG>
__device__ __forceinline__ void flux_cell(int64_t n, int64_t c, int nx, int ny, int nz, bool flatz,
                                          const double *__restrict__ cons, const double *__restrict__ u,
                                          const double *__restrict__ p, const double *__restrict__ ad,
                                          const double *__restrict__ cons_old, double *__restrict__ out, int avg,
                                          double dt, double dx, double dy, double dz, double srho, double seps,
                                          const AngGrid &ang)
{
    int ix, iy, iz;
    coords(c, nx, ny, ix, iy, iz);
    double ftmp[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (boundary_of(ix, iy, iz, nx, ny, nz) == 0) {
        const double axy = dy * dx, ayz = dy * dz, axz = dx * dz, vol = dx * dy * dz;
        const int64_t sz = flatz ? 0 : (int64_t)nx * ny;
        double f0[5], f1[5], s[5];
        auto faces = [&](auto dirc, int64_t st, double ds) {
            constexpr int d = decltype(dirc)::value;
            auto side = [&](int64_t q, int pm) {
                return cell_side<d, ANG>(q, pm, n, nx, ny, nz, st, cons, u, p, ad, dt, ds, seps, ang);
            };
            if constexpr (ANG) {
                const AngCentre at = ang_centre({dx, dy, 0.0}, c, nx, ny);
                double g[2];
                face_flux_ang<d>(side(c - st, 1), side(c, 0), at, at, f0, g);
                face_flux_ang<d>(side(c, 1), side(c + st, 0), at, at, f1, g);
            } else {
                face_flux<double, d>(side(c - st, 1), side(c, 0), f0);
                face_flux<double, d>(side(c, 1), side(c + st, 0), f1);
            }
        };
        faces(std::integral_constant<int, 0>{}, 1, dx);
        for (int i = 0; i < 5; i++) s[i] = ayz * (f1[i] - f0[i]);
        faces(std::integral_constant<int, 1>{}, nx, dy);
        for (int i = 0; i < 5; i++) s[i] = s[i] + axz * (f1[i] - f0[i]);
        faces(std::integral_constant<int, 2>{}, sz, dz);
        for (int i = 0; i < 5; i++) ftmp[i] = -((s[i] + axy * (f1[i] - f0[i])) * dt / vol);
    }
    flux_end<ANG>(n, c, nx, ny, cons, cons_old, out, avg, ftmp, srho, seps, ang);
}

}  // namespace bx
