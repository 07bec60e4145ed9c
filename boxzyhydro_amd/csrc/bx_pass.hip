// bx_pass.hip -- the pointwise calls of the exact step in fused passes.
//
// Between two ghost fills or fluxes the reference's step (main.f90:211-555)
// runs several pointwise subroutines over the grid (state, velocity, source,
// courant).  A pass takes one cell through all of them in registers, in the
// same order and with the same operations: streaming passes are bound by HBM
// (a velocity after a state reads four of the five planes again), on small
// grids by dispatches.  Interior cells and ghosts are separate launches: the
// ghost launch goes first and forms, from the still untouched donor, what the
// donor's calls will leave in it, so that a set_ghost_cells between two
// subroutines needs no pass of its own.  This covers tables whose donors are
// all interior cells; grids with chained ghosts (walls in two directions) run
// the ghost fills as they stand and use the state + velocity pass over every
// cell.
//
// Tabulated EOS: a state() whose pressure, gamma and muc the next state()
// overwrites unread needs no table lookup (a random 128-byte line per cell),
// only the energy reset of a low-density cell: two of the five per step.
//
// Eight steps of a 128^3 cloud with tables 7.20 -> 5.36 ms, of a 120x120x24
// disk with flux_ang and a point mass 2.77 -> 2.52 ms; the calls one by one
// keep their own kernels.
#include "bx_cells.h"
#include "bx_eos_dev.h"

namespace bx {

constexpr int kPassThreads = 256;

struct PassArgs {
    int64_t n;
    int nx, ny, nz;
    double *cons, *u, *p, *ad, *mucp;  // ad: null where every cell already holds gamma; mucp: tabulated EOS
    double gam, seps, muc, rgas, vlimit, dt;
    double g0, g1, g2;
    const double *gf;
    int ang, disk, all;                // disk: nz == 1 with tables; all: take ghost cells too
    int inner;                         // a later pass of the step sets muc before any reader
    double dx, dy, dz;
    EosDev e;
    unsigned long long *rate;          // kMaxSlots slots
};

// state() on a cell.  TAB: state.f90:58-79; with `lookup` false the cell's p,
// gamma and muc are left as they are (only a low-density cell's p and E are set).
template <bool TAB>
__device__ __forceinline__ void pass_state(const PassArgs &a, CellState &x, double &ad, double &mu, int64_t c,
                                           bool lookup)
{
    if constexpr (!TAB) {
        state_of(x, a.gam, a.seps, a.muc, a.rgas);
        ad = a.gam;
    } else {
        const double rho = x.U[0];
        const double ekin = rho * 0.5 * (x.v[0] * x.v[0] + x.v[1] * x.v[1] + x.v[2] * x.v[2]);
        if (lookup) {
            const double eps = vmax(x.U[4] - ekin, a.seps);
            double tk, m, g;
            if (a.disk) {
                // nz == 1: the column is a disk of scale height hscale (state.f90:61-69)
                const int ix = (int)(c % a.nx) + 1, iy = (int)((c / a.nx) % a.ny) + 1;
                const double px = centre(a.dx, ix, a.nx), py = centre(a.dy, iy, a.ny);
                const double hscale = sqrt((ad - 1.0) * eps / (2.0 * ekin) * (px * px + py * py));
                get_gamma2(a.e, eps / (2.0 * hscale), rho / (2.0 * hscale), tk, m, g);
            } else {
                get_gamma2(a.e, eps, rho, tk, m, g);
            }
            ad = g;
            mu = m;
            x.p = rho * tk * a.rgas / m;
        }
        if (rho < 1e-4) {
            const double pc = a.rgas * a.e.tk_bgrnd / a.muc * rho;
            x.U[4] = pc / (a.gam - 1.0) + ekin;
            x.p = pc;
        }
    }
}

__device__ __forceinline__ void pass_source(const PassArgs &a, CellState &x, int64_t c)
{
    double g0 = a.g0, g1 = a.g1, g2 = a.g2;
    if (a.gf) {
        g0 = a.gf[c];
        g1 = a.gf[a.n + c];
        g2 = a.gf[2 * a.n + c];
    }
    double px = 0.0, py = 0.0;
    if (a.ang) {
        px = centre(a.dx, (int)(c % a.nx) + 1, a.nx);
        py = centre(a.dy, (int)((c / a.nx) % a.ny) + 1, a.ny);
    }
    source_of(x, a.dt, g0, g1, g2, a.seps, a.ang, px, py);
}

__device__ __forceinline__ void pass_velocity(const PassArgs &a, CellState &x)
{
    bool clamped;
    velocity_of(x, a.vlimit, a.seps, clamped);
}

__device__ __forceinline__ void load_cell(const PassArgs &a, int64_t c, CellState &x)
{
    for (int f = 0; f < 5; f++) x.U[f] = a.cons[f * a.n + c];
    for (int d = 0; d < 3; d++) x.v[d] = a.u[d * a.n + c];
}

// What a pass leaves of a cell; planes that a call cannot have changed are not
// written again.  x0: the cell as loaded.
template <int PASS, bool TAB, bool GHOST>
__device__ __forceinline__ void store_cell(const PassArgs &a, int64_t c, const CellState &x, const double *U0, double ad,
                                           double mu)
{
    for (int f = GHOST ? 0 : 1; f < 5; f++)
        if (GHOST || __double_as_longlong(x.U[f]) != __double_as_longlong(U0[f])) a.cons[f * a.n + c] = x.U[f];
    if (PASS != kState && PASS != kStateRate)
        for (int d = 0; d < 3; d++) a.u[d * a.n + c] = x.v[d];
    if (TAB && PASS == kEndNext && !a.disk) return;  // the next step's kBeforeFlux sets them before any reader
    a.p[c] = x.p;
    if (TAB || a.ad) a.ad[c] = ad;
    if constexpr (TAB)
        if (!a.inner) a.mucp[c] = mu;
}

// Each thread takes CPT cells a block apart (coalesced), so that the table
// lookups of its cells are in flight together.
template <int PASS, bool TAB, int CPT>
__global__ __launch_bounds__(kPassThreads) void k_pass(PassArgs a)
{
    const int64_t base = (int64_t)blockIdx.x * blockDim.x * CPT + threadIdx.x;
    CellState x[CPT];
    double U0[CPT][5], ad[CPT], mu[CPT];
    bool on[CPT];
    double rate = 0.0;
    const bool disk = TAB && a.disk;
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int64_t c0 = base + (int64_t)k * blockDim.x, c = c0 < a.n ? c0 : a.n - 1;
        on[k] = c0 < a.n;
        if (PASS != kState && PASS != kStateRate && !a.all) {
            int ix, iy, iz;
            coords(c, a.nx, a.ny, ix, iy, iz);
            on[k] = on[k] && boundary_of(ix, iy, iz, a.nx, a.ny, a.nz) == 0;
        }
        load_cell(a, c, x[k]);
        for (int f = 0; f < 5; f++) U0[k][f] = x[k].U[f];
        x[k].p = !TAB && x[k].U[0] < 1e-4 ? a.p[c] : 0.0;
        ad[k] = disk ? a.ad[c] : 0.0;
        mu[k] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int64_t c0 = base + (int64_t)k * blockDim.x, c = c0 < a.n ? c0 : a.n - 1;
        CellState &y = x[k];
        if (PASS == kBeforeFlux) pass_source(a, y, c);  // main.f90:289
        pass_state<TAB>(a, y, ad[k], mu[k], c, PASS < kEnd || disk);
        if (PASS != kState && PASS != kStateRate) pass_velocity(a, y);
        if (PASS >= kEnd) {
            pass_source(a, y, c);  // main.f90:490
            pass_state<TAB>(a, y, ad[k], mu[k], c, PASS == kEnd || disk);
            pass_velocity(a, y);
        }
        if (PASS == kEndNext) pass_state<TAB>(a, y, ad[k], mu[k], c, true);  // the next step's main.f90:232
        if (PASS == kEndNext || PASS == kStateRate)
            if (on[k]) rate = vmax(rate, courant_of(y, ad[k], a.dx, a.dy, a.dz));
    }
#pragma unroll
    for (int k = 0; k < CPT; k++)
        if (on[k]) store_cell<PASS, TAB, false>(a, base + (int64_t)k * blockDim.x, x[k], U0[k], ad[k], mu[k]);
    if (PASS == kEndNext || PASS == kStateRate) block_max_to(rate, max_slot(a.rate));
}

__device__ __forceinline__ void take_signed(CellState &x, const CellState &d, int sg)
{
    x.U[0] = d.U[0];
    for (int f = 1; f <= 3; f++) x.U[f] = ((sg >> (f - 1)) & 1) ? -d.U[f] : d.U[f];
    x.U[4] = d.U[4];
}

// The ghosts of a pass, before the interior's: entry k of a table whose donors
// are interior cells.  The ghost takes its donor's conserved values where the
// sequence fills the ghosts, and goes through the calls with its own velocity
// and pressure.
template <int PASS, bool TAB>
__global__ __launch_bounds__(kPassThreads) void k_pass_ghosts(PassArgs a, int64_t ng, const int32_t *__restrict__ dst,
                                                             const int32_t *__restrict__ src,
                                                             const int32_t *__restrict__ sign)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double rate = 0.0;
    if (k < ng) {
        const int64_t c = dst[k], s = src[k];
        const int sg = sign[k];
        const bool disk = TAB && a.disk;
        CellState x, d;
        load_cell(a, s, d);
        d.p = !TAB && d.U[0] < 1e-4 ? a.p[s] : 0.0;
        for (int q = 0; q < 3; q++) x.v[q] = a.u[q * a.n + c];
        x.p = TAB ? 0.0 : a.p[c];
        double ad = disk ? a.ad[c] : 0.0, mu = 0.0, adx = 0.0, mux = 0.0;
        if (PASS == kBeforeFlux) pass_source(a, d, s);  // main.f90:289, source.f90:199, main.f90:312
        take_signed(x, d, sg);
        pass_state<TAB>(a, x, ad, mu, c, PASS < kEnd || disk);
        pass_velocity(a, x);
        if (PASS >= kEnd) {
            pass_state<TAB>(a, d, adx, mux, s, false);
            pass_velocity(a, d);
            pass_source(a, d, s);  // main.f90:490, and the fills of source.f90:199 and main.f90:511
            take_signed(x, d, sg);
            pass_state<TAB>(a, x, ad, mu, c, PASS == kEnd || disk);
            pass_velocity(a, x);
        }
        if (PASS == kEndNext) {
            pass_state<TAB>(a, x, ad, mu, c, true);
            rate = courant_of(x, ad, a.dx, a.dy, a.dz);
        }
        store_cell<PASS, TAB, true>(a, c, x, nullptr, ad, mu);
    }
    if (PASS == kEndNext) block_max_to(rate, max_slot(a.rate));
}

static PassArgs pass_args(bx_ctx *c, double dt, bool all)
{
    PassArgs a{};
    a.n = c->n;
    a.nx = c->nx;
    a.ny = c->ny;
    a.nz = c->nz;
    a.cons = c->cons;
    a.u = c->u;
    a.p = c->p;
    a.ad = !c->eos && c->ad_uniform ? nullptr : c->adindx;
    a.gam = c->prm.gammafix;
    a.seps = c->prm.small_eps;
    a.muc = c->muc;
    a.rgas = c->rgas;
    a.vlimit = c->prm.vlimit;
    a.dt = dt;
    a.g0 = c->grav[0];
    a.g1 = c->grav[1];
    a.g2 = c->grav[2];
    a.gf = c->grav_flags ? c->gforce : nullptr;
    a.ang = c->prm.fluxangmom;
    a.all = all ? 1 : 0;
    a.dx = c->prm.dx;
    a.dy = c->prm.dy;
    a.dz = c->prm.dz;
    a.rate = c->dmax;
    if (c->eos) {
        a.e = c->eos->dev;
        a.mucp = c->eos->muc_plane;
        a.disk = c->nz == 1 ? 1 : 0;
    }
    return a;
}

template <bool TAB, int CPT>
static void go_pass(bx_ctx *c, int pass, const PassArgs &a)
{
    const dim3 grid(blocks_for(c->n, kPassThreads * CPT)), block(kPassThreads);
    switch (pass) {
    case kState: hipLaunchKernelGGL((k_pass<kState, TAB, CPT>), grid, block, 0, c->stream, a); break;
    case kStateRate: hipLaunchKernelGGL((k_pass<kStateRate, TAB, CPT>), grid, block, 0, c->stream, a); break;
    case kAfterFlux: hipLaunchKernelGGL((k_pass<kAfterFlux, TAB, CPT>), grid, block, 0, c->stream, a); break;
    case kBeforeFlux: hipLaunchKernelGGL((k_pass<kBeforeFlux, TAB, CPT>), grid, block, 0, c->stream, a); break;
    case kEnd: hipLaunchKernelGGL((k_pass<kEnd, TAB, CPT>), grid, block, 0, c->stream, a); break;
    default: hipLaunchKernelGGL((k_pass<kEndNext, TAB, CPT>), grid, block, 0, c->stream, a); break;
    }
}

template <bool TAB>
static void go_ghosts(bx_ctx *c, int pass, const PassArgs &a)
{
    const dim3 grid(blocks_for(c->nghost, kPassThreads)), block(kPassThreads);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, c->stream, a, c->nghost, c->ghost_dst, c->ghost_src, c->ghost_sign);
    };
    switch (pass) {
    case kAfterFlux: go(k_pass_ghosts<kAfterFlux, TAB>); break;
    case kBeforeFlux: go(k_pass_ghosts<kBeforeFlux, TAB>); break;
    case kEnd: go(k_pass_ghosts<kEnd, TAB>); break;
    default: go(k_pass_ghosts<kEndNext, TAB>); break;
    }
}

// A pass over every cell.  `filled`: the ghosts hold what the sequence's fill
// gives them (kState, kStateRate, or kAfterFlux after the fills); otherwise the
// pass fills them (no chained ghosts).
int launch_pass(bx_ctx *c, int pass, double dt, bool filled)
{
    if (pass == kEndNext || pass == kStateRate)
        if (int rc = begin_max(c)) return rc;
    PassArgs a = pass_args(c, dt, filled);
    a.inner = !filled && (pass == kBeforeFlux || pass == kAfterFlux) ? 1 : 0;
    if (!filled && c->nghost > 0) {
        if (c->eos) go_ghosts<true>(c, pass, a);
        else go_ghosts<false>(c, pass, a);
        BX_HIP(hipGetLastError());
    }
    if (c->eos) go_pass<true, 2>(c, pass, a);
    else go_pass<false, 1>(c, pass, a);
    BX_HIP(hipGetLastError());
    c->ad_uniform = !c->eos;
    return BX_OK;
}

}  // namespace bx
