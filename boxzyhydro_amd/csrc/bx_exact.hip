// bx_exact.hip -- the hydro step as the reference structures it: one kernel per
// reference subroutine, acting on device-resident SoA planes.  These kernels
// are the plain FP64 drop-in behind bx_state/bx_velocity/bx_courant/
// bx_source/bx_set_ghost_cells/bx_flux/bx_avisc, and the exact fallback of
// the fused step.  Arithmetic order follows the cited reference lines so the
// results are bit-identical to the reference's FP64 step.
#include <algorithm>
#include <cstring>
#include <utility>

#include "bx_cells.h"

namespace bx {

constexpr int kThreads = 256;

// --------------------------------------------------------------- velocity
__global__ __launch_bounds__(kThreads) void k_velocity(int64_t n, double *__restrict__ cons,
                                                      double *__restrict__ u, double vlimit,
                                                      double seps, unsigned long long *maxv)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const double vm = c < n ? velocity_cell(n, c, cons, u, vlimit, seps) : 0.0;
    if (maxv) block_max_to(vm, max_slot(maxv));
}

// ---------------------------------------------------------------- courant
// courant.f90:17-29: max over all cells
__global__ __launch_bounds__(kThreads) void k_courant(int64_t n, const double *__restrict__ cons,
                                                     const double *__restrict__ u,
                                                     const double *__restrict__ p,
                                                     const double *__restrict__ ad, double dx,
                                                     double dy, double dz, unsigned long long *rate)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    block_max_to(c < n ? courant_cell(n, c, cons, u, p, ad, dx, dy, dz) : 0.0, max_slot(rate));
}

// ----------------------------------------------------------------- source
__global__ __launch_bounds__(kThreads) void k_source(int64_t n, int nx, int ny, int nz,
                                                    double *__restrict__ cons,
                                                    const double *__restrict__ u, double dt,
                                                    double g0, double g1, double g2, double seps,
                                                    int ang, double dx, double dy,
                                                    const double *__restrict__ gf)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) source_cell(n, c, nx, ny, nz, cons, u, dt, g0, g1, g2, seps, ang, dx, dy, gf);
}

// ------------------------------------------------------------ ghost cells
__global__ __launch_bounds__(kThreads) void k_ghost_snapshot(int64_t n, int64_t ns,
                                                            const int32_t *__restrict__ ssrc,
                                                            const double *__restrict__ planes,
                                                            double *__restrict__ scratch)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ns) ghost_snapshot_one(n, ns, k, ssrc, planes, scratch);
}

__global__ __launch_bounds__(kThreads) void k_ghosts(int64_t n, int64_t ng, const int32_t *__restrict__ dst,
                                                    const int32_t *__restrict__ src,
                                                    const int32_t *__restrict__ sign,
                                                    double *__restrict__ planes,
                                                    const double *__restrict__ scratch, int64_t ns)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ng) ghost_fill_one(n, k, dst, src, sign, planes, scratch, ns);
}

// ------------------------------------------------------------------- flux
// flux_ang leaves cons_old, when avg = 1, transformed to r- and angular
// momentum and back (flux_ang.f90:40-61, 245-268)
__global__ __launch_bounds__(kThreads) void k_ang_old(int64_t n, int nx, int ny, double *__restrict__ cons_old,
                                                     AngGrid ang)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const AngCentre tr = ang_centre(ang, c, nx, ny);
    double rm, am, m1, m2;
    tr.to(cons_old[n + c], cons_old[2 * n + c], rm, am);
    tr.back(rm, am, m1, m2);
    cons_old[n + c] = m1;
    cons_old[2 * n + c] = m2;
}

// flux.f90:6-230 cell by cell: for grids that the tiles do not serve (slow
// null), and for a call whose tiled kernel met a value outside its range (*slow
// set), every cell again from the same inputs.
template <bool ANG>
__global__ __launch_bounds__(kThreads) void k_flux_cells(const unsigned int *__restrict__ slow, int64_t n, int nx,
                                                        int ny, int nz, bool flatz, const double *__restrict__ cons,
                                                        const double *__restrict__ u, const double *__restrict__ p,
                                                        const double *__restrict__ ad,
                                                        const double *__restrict__ cons_old, double *__restrict__ out,
                                                        int avg, double dt, double dx, double dy, double dz,
                                                        double srho, double seps, AngGrid ang)
{
    if (slow && *slow == 0u) return;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
        flux_cell<ANG>(n, c, nx, ny, nz, flatz, cons, u, p, ad, cons_old, out, avg, dt, dx, dy, dz, srho, seps, ang);
}

// the ghost cells of the flux's result: fluxtmp = 0 there (flux.f90:51), then
// the update and the floors; read only where a ghost's donor is a ghost
template <bool ANG>
__global__ __launch_bounds__(kThreads) void k_flux_ghosts(int64_t n, int nx, int ny, int64_t ng,
                                                         const int32_t *__restrict__ dst,
                                                         const double *__restrict__ cons,
                                                         const double *__restrict__ cons_old,
                                                         double *__restrict__ out, int avg, double srho, double seps,
                                                         AngGrid ang)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ng) return;
    const double ft[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    flux_end<ANG>(n, dst[k], nx, ny, cons, cons_old, out, avg, ft, srho, seps, ang);
}

// ------------------------------------------------------------------ avisc
// avisc.f90:13-24 with get_boundary (utils.f90:62-74).  Outer-layer cells
// (boundary=1) have only their donor in ineigh(1) in the reference and read
// ineigh(2:6)=0 (outside the array); here those neighbours are the cell itself.
__global__ __launch_bounds__(kThreads) void k_avisc(int64_t n, int nx, int ny, int nz, bool flatz,
                                                   const double *__restrict__ u, double *__restrict__ qq,
                                                   double ax, double ay, double az)
{
    int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    int ix, iy, iz;
    coords(c, nx, ny, ix, iy, iz);
    const int bnd = boundary_of(ix, iy, iz, nx, ny, nz);
    if (bnd == 0) {
        qq[c] = 0.0;
        qq[n + c] = 0.0;
        qq[2 * n + c] = 0.0;
        return;
    }
    const int64_t pl = (int64_t)nx * ny;
    int64_t nb[6];
    if (bnd == 2) {
        nb[0] = c + nx;
        nb[1] = c - nx;
        nb[2] = c + 1;
        nb[3] = c - 1;
        nb[4] = flatz ? c : c + pl;
        nb[5] = flatz ? c : c - pl;
    } else {
        for (int k = 0; k < 6; k++) nb[k] = c;
        if (ix == 1) nb[0] = c + 2;
        else if (ix == nx) nb[0] = c - 2;
        else if (iy == 1) nb[0] = c + 2 * (int64_t)nx;
        else if (iy == ny) nb[0] = c - 2 * (int64_t)nx;
        else if (iz == 1) nb[0] = flatz ? c : c + 2 * pl;
        else nb[0] = flatz ? c : c - 2 * pl;
    }
    for (int k = 0; k < 6; k++) {
        int jx, jy, jz;
        coords(nb[k], nx, ny, jx, jy, jz);
        if (boundary_of(jx, jy, jz, nx, ny, nz) > 0) nb[k] = c;
    }
    double t;
    t = vmin(0.0, u[nb[2]] - u[nb[3]]);
    qq[c] = ax * (t * t);
    t = vmin(0.0, u[n + nb[0]] - u[n + nb[1]]);
    qq[n + c] = ay * (t * t);
    t = vmin(0.0, u[2 * n + nb[4]] - u[2 * n + nb[5]]);
    qq[2 * n + c] = az * (t * t);
}

// ------------------------------------------------------------- launchers
int launch_state(bx_ctx *c) { return launch_pass(c, kState, 0.0, true); }

// The maximum of the slots to the (pinned) host word, and the slots cleared
// for the next kernel that forms one.  One small kernel in place of a clearing
// one before that kernel and a copy of the slots after it: 8 us less of each
// maximum.
static_assert(kMaxSlots <= 64, "a lane per slot");
__global__ __launch_bounds__(64) void k_take_max(unsigned long long *slots, unsigned long long *host)
{
    const int l = threadIdx.x;
    unsigned long long v = 0ull;  // non-negative doubles order as their bits
    if (l < kMaxSlots) {
        v = slots[l * kMaxStride];
        slots[l * kMaxStride] = 0ull;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    if (l == 0) *host = v;
}

static int take_max(bx_ctx *c)
{
    hipLaunchKernelGGL(k_take_max, dim3(1), dim3(64), 0, c->stream, c->dmax, c->hmax);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

// Before a kernel that forms a maximum: the slots are clear unless an earlier
// one's maximum was never read (an error in between).
int begin_max(bx_ctx *c)
{
    if (c->max_open)
        if (int rc = take_max(c)) return rc;
    c->max_open = true;
    return BX_OK;
}

// The grid-wide maximum of the last kernel that formed one (waits for it).
int read_max(bx_ctx *c, double *out)
{
    if (int rc = take_max(c)) return rc;
    c->max_open = false;
    BX_HIP(hipStreamSynchronize(c->stream));
    std::memcpy(out, c->hmax, sizeof(double));
    return BX_OK;
}

int launch_velocity(bx_ctx *c, bool want_maxv)
{
    if (want_maxv)
        if (int rc = begin_max(c)) return rc;
    hipLaunchKernelGGL(k_velocity, dim3(blocks_for(c->n, kThreads)), dim3(kThreads), 0, c->stream, c->n, c->cons, c->u,
                       c->prm.vlimit, c->prm.small_eps, want_maxv ? c->dmax : (unsigned long long *)nullptr);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

int launch_courant(bx_ctx *c)
{
    if (int rc = begin_max(c)) return rc;
    hipLaunchKernelGGL(k_courant, dim3(blocks_for(c->n, kThreads)), dim3(kThreads), 0, c->stream, c->n, c->cons, c->u,
                       c->p, c->adindx, c->prm.dx, c->prm.dy, c->prm.dz, c->dmax);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

int launch_ghosts(bx_ctx *c, double *planes5)
{
    if (c->nghost == 0) return BX_OK;
    if (c->nscratch > 0) {
        hipLaunchKernelGGL(k_ghost_snapshot, dim3(blocks_for(c->nscratch, kThreads)), dim3(kThreads), 0, c->stream,
                           c->n, c->nscratch, c->ghost_scratch_src, planes5, c->ghost_scratch);
        BX_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_ghosts, dim3(blocks_for(c->nghost, kThreads)), dim3(kThreads), 0, c->stream, c->n,
                       c->nghost, c->ghost_dst, c->ghost_src, c->ghost_sign, planes5, c->ghost_scratch,
                       c->nscratch);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

int launch_source(bx_ctx *c, double dt)
{
    hipLaunchKernelGGL(k_source, dim3(blocks_for(c->n, kThreads)), dim3(kThreads), 0, c->stream, c->n, c->nx,
                       c->ny, c->nz, c->cons, c->u, dt, c->grav[0], c->grav[1], c->grav[2], c->prm.small_eps,
                       c->prm.fluxangmom, c->prm.dx, c->prm.dy, c->grav_flags ? c->gforce : (const double *)nullptr);
    BX_HIP(hipGetLastError());
    return launch_ghosts(c, c->cons);
}

// The flux subroutine: the tiled kernel over the interior, the cell-by-cell one
// in its place where the data asks for it (the choice is made on the device),
// into the states planes, which then trade places with cons.  One kernel in
// place of face fluxes to memory and an update: 5.5 -> 2.2 ms for the two
// calls of a step at 256^3; with flux_ang in place of the interface states of
// every cell to 54 planes and the faces per cell: eight steps of a 120x120x24
// disk 2.52 -> 1.59 ms.
template <bool ANG>
static int flux_kernels(bx_ctx *c, int avg, double dt)
{
    double *out = c->states;
    const AngGrid ang{c->prm.dx, c->prm.dy, c->prm.yoffset};
    // Thin in x, a tile's 32 columns are mostly idle and the cells are faster: an
    // exact step of 1 x 512^2 interior cells 688 us against 921 in tiles, 2 x 512^2
    // 841 against 962, 1 x 180^2 144 against 184; 3 x 512^2 996 against 997, and
    // on 1 x 128^2, where the launches count, 118 against 117.  With flux_ang, whose
    // cells take half as long again, 1 x 512^2 1194 against 1492, 2 x 256^2 472
    // against 429.
    const int64_t rows = (int64_t)(c->ny - 4) * (c->flatz ? c->nz : c->nz - 4);
    const bool thin = c->nx - 4 <= (ANG ? 1 : 2) && rows >= (int64_t)16384 * (c->nx - 4);
    unsigned int *slow = nullptr;
    if (!thin && tile_fits(c, sizeof(double))) {
        slow = &c->dsc->slow[c->nflux & 1];
        unsigned int *next = &c->dsc->slow[(c->nflux + 1) & 1];
        c->nflux++;
        if (int rc = launch_tiled_flux(c, avg, dt, out, slow, next)) return rc;
    }
    // Few blocks where it mostly has nothing to do: a call of 192^3 cells that is
    // handed over (NaN, negative pressures) takes 3.9 ms with 256 of them, 2.5 with
    // 1024, 2.2 with 4096, but idle ones cost every call up to 1 us (four exact
    // steps of 31 x 54 x 79 cells 912 us with 256, 936 with 658).
    hipLaunchKernelGGL(k_flux_cells<ANG>, dim3(std::min(blocks_for(c->n, kThreads), slow ? 256u : 4096u)),
                       dim3(kThreads), 0, c->stream, slow, c->n, c->nx, c->ny, c->nz, c->flatz, c->cons, c->u, c->p,
                       c->adindx, c->cons_old, out, avg, dt, c->prm.dx, c->prm.dy, c->prm.dz, c->prm.small_rho,
                       c->prm.small_eps, ang);
    BX_HIP(hipGetLastError());
    if (c->nscratch > 0) {
        hipLaunchKernelGGL(k_flux_ghosts<ANG>, dim3(blocks_for(c->nghost, kThreads)), dim3(kThreads), 0, c->stream,
                           c->n, c->nx, c->ny, c->nghost, c->ghost_dst, c->cons, c->cons_old, out, avg,
                           c->prm.small_rho, c->prm.small_eps, ang);
        BX_HIP(hipGetLastError());
    }
    if (ANG && avg) {
        hipLaunchKernelGGL(k_ang_old, dim3(blocks_for(c->n, kThreads)), dim3(kThreads), 0, c->stream, c->n, c->nx,
                           c->ny, c->cons_old, ang);
        BX_HIP(hipGetLastError());
    }
    return BX_OK;
}

int launch_flux(bx_ctx *c, int avg, double dt, bool ghosts)
{
    if (int rc = c->prm.fluxangmom ? flux_kernels<true>(c, avg, dt) : flux_kernels<false>(c, avg, dt)) return rc;
    std::swap(c->cons, c->states);
    return ghosts ? launch_ghosts(c, c->cons) : BX_OK;
}

int launch_avisc(bx_ctx *c)
{
    hipLaunchKernelGGL(k_avisc, dim3(blocks_for(c->n, kThreads)), dim3(kThreads), 0, c->stream, c->n, c->nx,
                       c->ny, c->nz, c->flatz, c->u, c->qq, c->prm.avmag[0], c->prm.avmag[1], c->prm.avmag[2]);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

}  // namespace bx
