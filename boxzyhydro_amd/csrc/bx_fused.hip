// bx_fused.hip -- the hydro step as one fused stencil kernel per RK stage.
//
// The reference step (main.f90:211-555) runs ~25 passes over the grid per
// step.  On a "regular" state -- every ghost cell a (sign-flipped) copy of an
// interior donor, u == m/rho bitwise, no cell below the rho<1e-4 EOS branch,
// no speed above vlimit -- every pass except the two flux stages is pointwise,
// so they are folded into the stencil kernels:
//
//   stage 1:  U^n -> source(0) energy re-round (source.f90:176-182), state,
//             velocity -> MUSCL/HLL predictor flux(0) (flux.f90) -> floors ->
//             U*, and the stale-velocity pressure p* of main.f90:351-355
//   stage 2:  U*, p*, U^n -> velocity -> corrector flux(1) with
//             cons_old = source(0)(U^n) -> floors -> state, velocity,
//             source(1) re-round (main.f90:374-515) -> U^{n+1}, plus the
//             next step's Courant rate (courant.f90:17-23) as a max-reduction
//
// Every arithmetic operation is the one the exact sequence (bx_exact.hip)
// performs on the same values, so the fused step is bit-identical to it; a
// cell that would take an irregular branch raises a flag and the host redoes
// the step with the exact sequence.
//
// Work decomposition (gfx950, wave64): by default each stage is one kernel,
// k_stage, a workgroup holding a tile of outputs (64 x 8, 64 x 4, 32 x 16 or
// 32 x 8 columns) with its +-2 halo in LDS and marching in z (bx_tile.h).  The tuning variants 0, 1 and 4
// (bx_tune) run the earlier form, two kernels per stage with every wave
// independent (no LDS, no block barriers):
//   * k_ydir: a wave holds 64 interior x-cells of one z-plane and marches in y
//     with a register queue; it writes the y-term of fluxtmp (FP64 planes).
//   * k_xz: a wave holds 64 cells of one interior row (lanes 2..61 output,
//     0,1,62,63 the x-halo; x-neighbours through wave shuffles) and marches in
//     z with a register queue; it adds the x- and z-terms in the reference's
//     order and applies the stage update.
// Both give the same bits.
#include <cmath>

#include "bx_cells.h"
#include "bx_tile.h"

namespace bx {

// One stage as one kernel: x-y tile of WX x TY outputs with its +-2 halo in
// LDS, marching in z (bx_tile.h: tile_stage).  P2: every spacing and the
// cell volume are powers of two (their divisions are multiplications), known
// at compile time, which keeps the spacings themselves out of the registers.
// V: StageKind; W: walls whose ghosts are read from their donors (bx_tile.h).
template <int STAGE, typename S, int TY, bool P2, int V, bool W, int WX>
__global__ __launch_bounds__(64 * tile_waves(TY, WX)) void k_stage(StageArgs a0)
{
    __shared__ TileLds<S, TY, V, WX> lds;
    StageArgs a = with_dt(a0);
    if constexpr (P2) {
        a.ds_pow2[0] = a.ds_pow2[1] = a.ds_pow2[2] = 1;
        a.vol_pow2 = 1;
    }
    // Workgroups go to the 8 XCDs in turn (workgroup id mod 8).  Give each
    // XCD a contiguous range of tiles, x fastest, so that the tiles in flight
    // on one XCD are neighbours and share their halo rows and boundary cache
    // lines in that XCD's L2.
    const unsigned gx = gridDim.x, gy = gridDim.y;
    unsigned T = gx * gy * gridDim.z;
    unsigned L = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    if constexpr (STAGE == 2 && W && sizeof(S) == 8) {
        if (a.ncorner > 0) {
            if ((int)L < a.ncorner) {
                static_assert(sizeof(lds) >= sizeof(double[3][2][5]), "the corner faces' buffer");
                if ((int)L < a.nd2) corner_block(a, (int)L, reinterpret_cast<double (*)[2][5]>(&lds));
                return;
            }
            L -= (unsigned)a.ncorner;
            T = gx * gy * (unsigned)((a.zhi - a.zlo + a.lz - 1) / a.lz);
            if (L >= T) return;
        }
    }
    const unsigned xcd = L & 7u, slot = L >> 3, q = T >> 3, rem = T & 7u;
    const unsigned t = xcd * q + (xcd < rem ? xcd : rem) + slot;
    tile_stage<STAGE, S, TY, V, W, WX>(a, lds, t % gx, (t / gx) % gy, t / (gx * gy));
}


// y-direction kernel: one launch over the interior (bx_waves.h: ydir_wave)
template <int STAGE, typename S>
__global__ __launch_bounds__(256) void k_ydir(StageArgs a0, S *__restrict__ Ey, int ly)
{
    const StageArgs a = with_dt(a0);
    ydir_wave<STAGE, S>(a, Ey, ly, blockIdx.x, blockIdx.y, blockIdx.z, wave_id());
}

// x/z kernel: one launch over the interior (bx_waves.h: xz_wave)
template <int STAGE, typename S, int OCC, bool PFE>
__global__ __launch_bounds__(256, OCC) void k_xz(StageArgs a0, const S *__restrict__ Ey)
{
    const StageArgs a = with_dt(a0);
    xz_wave<STAGE, S, PFE>(a, Ey, blockIdx.x, blockIdx.z, wave_id());
}

// -------------------------------------------------------------- helpers
// p: null keeps the pressure plane (written by the fused corrector with gravity)
__global__ __launch_bounds__(256) void k_materialize(int64_t n, const double *__restrict__ cons,
                                                    double *__restrict__ u, double *__restrict__ p,
                                                    double *__restrict__ ad, double gam, double seps)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) materialize_cell(n, c, cons, u, p, ad, gam, seps);
}

__global__ __launch_bounds__(256) void k_regular(int64_t n, const double *__restrict__ cons,
                                                const double *__restrict__ u, double gam, double seps,
                                                double dx, double dy, double dz, unsigned int *flags,
                                                unsigned long long *rate)
{
    unsigned int flg = 0;
    double rt = 0.0;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
        rt = vmax(rt, regular_cell(n, c, cons, u, gam, seps, dx, dy, dz, flg));
    if (flg) atomicOr(flags, flg);
    block_max_to(rt, rate + (blockIdx.x % kRateSlots) * kMaxStride);
}

template <typename S>
__global__ __launch_bounds__(256) void k_ghosts6(int64_t n, int64_t ng, const int32_t *__restrict__ dst,
                                                const int32_t *__restrict__ src,
                                                const int32_t *__restrict__ sign, S *__restrict__ planes,
                                                S *__restrict__ pstar)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ng) ghost6_one<S>(n, k, dst, src, sign, planes, pstar);
}

// FP64 <-> FP32 copies of the 5 conserved planes (mixed form hand-over)
__global__ __launch_bounds__(256) void k_narrow(int64_t m, const double *__restrict__ a, float *__restrict__ b)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) b[i] = (float)a[i];
}

__global__ __launch_bounds__(256) void k_widen(int64_t m, const float *__restrict__ a, double *__restrict__ b)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) b[i] = (double)a[i];
}

// ----------------------------------------------------------------- host
static bool is_pow2(double d)
{
    int e;
    double m = std::frexp(d, &e);
    return m == 0.5;
}

StageArgs base_args(bx_ctx *c, double dt)
{
    StageArgs a{};
    a.n = c->n;
    a.nx = c->nx;
    a.ny = c->ny;
    a.nz = c->nz;
    a.flatz = c->flatz ? 1 : 0;
    a.zlo = c->flatz ? 0 : 2;
    a.zhi = c->flatz ? c->nz : c->nz - 2;
    a.lz = c->fused_lz;
    a.dt = dt;
    const double ds[3] = {c->prm.dx, c->prm.dy, c->prm.dz};
    for (int d = 0; d < 3; d++) {
        a.ds[d] = ds[d];
        a.inv_ds[d] = 1.0 / ds[d];
        a.ds_pow2[d] = is_pow2(ds[d]) ? 1 : 0;
    }
    const double dx = ds[0], dy = ds[1], dz = ds[2];
    a.axy = dy * dx;
    a.ayz = dy * dz;
    a.axz = dx * dz;
    a.vol = dx * dy * dz;
    a.inv_vol = 1.0 / a.vol;
    a.vol_pow2 = is_pow2(a.vol) ? 1 : 0;
    a.gam = c->prm.gammafix;
    a.gm1 = c->prm.gammafix - 1.0;
    a.seps = c->prm.small_eps;
    a.srho = c->prm.small_rho;
    a.vlimit = c->prm.vlimit;
    a.flags = &c->dsc->flags;
    a.nd2 = c->nd2;
    a.d2cell = c->d2_src;
    a.d2ubar = c->d2_ubar;
    a.d2dst = c->d2_dst;
    a.d2sign = c->d2_sign;
    a.gf = c->grav_flags ? c->gfused : nullptr;
    return a;
}

// the grid of the tiled kernels: tiles of wx x ty columns by chunks of lz
// planes, and a.ncorner workgroups more
static dim3 tile_grid(const bx_ctx *c, const StageArgs &a, int ty, int wx)
{
    const unsigned gx = (unsigned)((c->nx - 4 + wx - 1) / wx), gy = (unsigned)((c->ny - 4 + ty - 1) / ty);
    return dim3(gx, gy, (unsigned)((a.zhi - a.zlo + a.lz - 1) / a.lz) + ((unsigned)a.ncorner + gx * gy - 1) / (gx * gy));
}

template <int STAGE, typename S, int TY, int WX, bool W>
static int launch_tile_w(bx_ctx *c, const StageArgs &a)
{
    const bool p2 = a.ds_pow2[0] && a.ds_pow2[1] && a.ds_pow2[2] && a.vol_pow2;
    const dim3 grid = tile_grid(c, a, TY, WX), block(64 * tile_waves(TY, WX));
    if constexpr (sizeof(S) == 8 && TY * WX == 512 && !W) {
        if (a.gf) {
            // the power-of-two forms spill 2 and 7 VGPRs at 168; the general
            // ones (163, no spill) give the same bits and are ~1 % faster
            hipLaunchKernelGGL((k_stage<STAGE, S, TY, false, kGravity, false, WX>), grid, block, 0, c->stream, a);
            BX_HIP(hipGetLastError());
            return BX_OK;
        }
    }
    if (a.gf) return set_error(BX_ERR_UNSUPPORTED, "fused step with gravity: FP64 64 x 8 or 32 x 16 tiles only");
    if (p2)
        hipLaunchKernelGGL((k_stage<STAGE, S, TY, true, kPlain, W, WX>), grid, block, 0, c->stream, a);
    else
        hipLaunchKernelGGL((k_stage<STAGE, S, TY, false, kPlain, W, WX>), grid, block, 0, c->stream, a);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

template <int STAGE, typename S, int TY, int WX>
static int launch_tile(bx_ctx *c, const StageArgs &a)
{
    bool w = false;
    for (int i = 0; i < 6; i++) w = w || (a.gmap && a.wall[i]);
    return w ? launch_tile_w<STAGE, S, TY, WX, true>(c, a) : launch_tile_w<STAGE, S, TY, WX, false>(c, a);
}

template <int STAGE, typename S>
static int launch_stage(bx_ctx *c, const StageArgs &a, hipEvent_t mid, S *eflux)
{
    if (c->grav_flags && !a.gf) return set_error(BX_ERR_STATE, "fused step with gravity before its force planes");
    if (c->fused_occ >= 10) {
        if (mid) BX_HIP(hipEventRecord(mid, c->stream));
        switch (c->fused_occ) {
        case kTile64x4: return launch_tile<STAGE, S, 4, 64>(c, a);
        case kTile64x8: return launch_tile<STAGE, S, 8, 64>(c, a);
        case kTile32x8: return launch_tile<STAGE, S, 8, 32>(c, a);
        default: break;
        }
        if constexpr (sizeof(S) == 8) return launch_tile<STAGE, S, 16, 32>(c, a);
        return set_error(BX_ERR_UNSUPPORTED, "mixed form: no 32 x 16 tiles");
    }
    if (a.gf) return set_error(BX_ERR_UNSUPPORTED, "fused step with gravity: the tiled kernel only (variant 11)");
    const int nzi = a.zhi - a.zlo;
    const int ly = c->fused_ly;
    {
        const unsigned gx = (unsigned)((c->nx - 4 + 63) / 64);
        const unsigned gy = (unsigned)((nzi + 3) / 4);
        const unsigned gz = (unsigned)((c->ny - 4 + ly - 1) / ly);
        hipLaunchKernelGGL((k_ydir<STAGE, S>), dim3(gx, gy, gz), dim3(256), 0, c->stream, a, eflux, ly);
        BX_HIP(hipGetLastError());
    }
    if (mid) BX_HIP(hipEventRecord(mid, c->stream));
    {
        const int64_t nwaves = ((int64_t)(c->ny - 4) * c->nx + kSegOut - 1) / kSegOut;
        const unsigned gx = (unsigned)((nwaves + 3) / 4);
        const unsigned gy = 1;
        const unsigned gz = (unsigned)((nzi + a.lz - 1) / a.lz);
        const S *ey = eflux;
        if (c->fused_occ == 4)
            hipLaunchKernelGGL((k_xz<STAGE, S, 4, false>), dim3(gx, gy, gz), dim3(256), 0, c->stream, a, ey);
        else if (c->fused_occ == 1)
            hipLaunchKernelGGL((k_xz<STAGE, S, 1, true>), dim3(gx, gy, gz), dim3(256), 0, c->stream, a, ey);
        else
            hipLaunchKernelGGL((k_xz<STAGE, S, 3, false>), dim3(gx, gy, gz), dim3(256), 0, c->stream, a, ey);
        BX_HIP(hipGetLastError());
    }
    return BX_OK;
}

// The flux subroutine on interior cells (bx_tile.h, stages 3 and 4): cons ->
// out, with cons_old for avg = 1.  slow: the word that records a value outside
// the tile's range; slow_next: cleared for the next call.
int launch_tiled_flux(bx_ctx *c, int avg, double dt, double *out, unsigned int *slow, unsigned int *slow_next)
{
    StageArgs a = base_args(c, dt);
    a.uin = c->cons;
    a.uold = c->cons_old;
    a.pin = c->p;
    a.vel = c->u;
    a.ad = c->adindx;
    a.uout = out;
    a.gf = nullptr;
    a.flags = slow;
    a.clear = slow_next;
    a.yoffset = c->prm.yoffset;
    a.p_class = kPositive | (c->flatz ? 0 : kPositiveZero);
    // gamma from its plane unless every cell holds gammafix; with it as a
    // seventh field the 64 x 8 tile, and with the eighth and ninth of flux_ang
    // either tile of eight owner waves, is too large for LDS
    const bool vg = !c->ad_uniform, ang = c->prm.fluxangmom != 0;
    unsigned tiles = tile_bit(kTile64x4) | tile_bit(kTile32x8);
    if (!ang) tiles |= tile_bit(kTile32x16) | (vg ? 0u : tile_bit(kTile64x8));
    const int tile = tile_split(c, false, tiles, &a.lz);
    const bool p2 = a.ds_pow2[0] && a.ds_pow2[1] && a.ds_pow2[2] && a.vol_pow2;
    auto go = [&](auto stage, auto rows, auto cols, auto pow2, auto kind) {
        constexpr int TY = decltype(rows)::value, WX = decltype(cols)::value;
        hipLaunchKernelGGL((k_stage<decltype(stage)::value, double, TY, decltype(pow2)::value, decltype(kind)::value,
                                    false, WX>),
                           tile_grid(c, a, TY, WX), dim3(64 * tile_waves(TY, WX)), 0, c->stream, a);
    };
    auto with_stage = [&](auto rows, auto cols, auto pow2, auto kind) {
        if (avg == 0) go(std::integral_constant<int, 3>{}, rows, cols, pow2, kind);
        else go(std::integral_constant<int, 4>{}, rows, cols, pow2, kind);
    };
    auto with_spacing = [&](auto rows, auto cols, auto kind) {
        if (p2) with_stage(rows, cols, std::true_type{}, kind);
        else with_stage(rows, cols, std::false_type{}, kind);
    };
    using R4 = std::integral_constant<int, 4>;
    using R8 = std::integral_constant<int, 8>;
    using R16 = std::integral_constant<int, 16>;
    using C32 = std::integral_constant<int, 32>;
    using C64 = std::integral_constant<int, 64>;
    auto with_tile = [&](auto kind) {
        constexpr int V = decltype(kind)::value;
        if constexpr (V == kPlain)
            if (tile == kTile64x8) return with_spacing(R8{}, C64{}, kind);
        if constexpr (!has_ang(V))
            if (tile == kTile32x16) return with_spacing(R16{}, C32{}, kind);
        if (tile == kTile32x8) return with_spacing(R8{}, C32{}, kind);
        with_spacing(R4{}, C64{}, kind);
    };
    if (ang && vg) with_tile(std::integral_constant<int, kAngGamma>{});
    else if (ang) with_tile(std::integral_constant<int, kAng>{});
    else if (vg) with_tile(std::integral_constant<int, kGamma>{});
    else with_tile(std::integral_constant<int, kPlain>{});
    BX_HIP(hipGetLastError());
    return BX_OK;
}

// the pressure plane of the materialised state at the corner ghosts (the
// value the last fused step's fix-up recorded)
__global__ __launch_bounds__(64) void k_corner_pressure(int nd2, const int32_t *__restrict__ dst,
                                                        const double *__restrict__ ubar, double *__restrict__ p)
{
    const int j = threadIdx.x;
    if (j < nd2) p[dst[j]] = ubar[6 * j + 5];
}

int launch_materialize(bx_ctx *c)
{
    hipLaunchKernelGGL(k_materialize, dim3(blocks_for(c->n, 256)), dim3(256), 0, c->stream, c->n, c->cons, c->u,
                       c->p_fused ? (double *)nullptr : c->p, c->adindx, c->prm.gammafix, c->prm.small_eps);
    BX_HIP(hipGetLastError());
    c->ad_uniform = true;
    if (c->nd2 > 0 && c->prm.precision == BX_PREC_FP64) {  // the mixed form copies the donors
        hipLaunchKernelGGL(k_corner_pressure, dim3(1), dim3(64), 0, c->stream, c->nd2, c->d2_dst, c->d2_ubar, c->p);
        BX_HIP(hipGetLastError());
    }
    return BX_OK;
}

// Whether the fused kernels compute this context's step (no allocation).
int fused_supported(const bx_ctx *c)
{
    if (c->nscratch > 0 && !c->fghost_ok)
        return set_error(BX_ERR_UNSUPPORTED, "fused step needs the ghost donors of a pair of set_ghost_cells calls "
                                             "to resolve to interior cells within two levels");
    if (!tile_fits(c, c->prm.precision == BX_PREC_MIXED ? sizeof(float) : sizeof(double)))
        return set_error(BX_ERR_UNSUPPORTED, "fused step: an x-y plane is beyond the stage kernels' 32-bit offsets or "
                                             "launch grid");
    if (c->grav[0] != 0.0 || c->grav[1] != 0.0 || c->grav[2] != 0.0)
        return set_error(BX_ERR_UNSUPPORTED, "fused step assumes zero gravity");
    if (c->prm.fluxangmom) return set_error(BX_ERR_UNSUPPORTED, "fused step fluxes linear momentum (fluxangmom off)");
    if (c->grav_flags & BX_GRAV_EXTERNAL)
        return set_error(BX_ERR_UNSUPPORTED, "fused step with gravity: a given potential only (no point mass, whose "
                                             "force needs the corrector's mass moments before source(1))");
    if (c->eos) return set_error(BX_ERR_UNSUPPORTED, "fused step assumes a fixed gamma (H2STAT=-1)");
    return BX_OK;
}

// The tile and z chunk of the tiled kernels: they march in z chunks of the
// interior planes (any length: nzi/m rounded up for m chunks).  A workgroup's
// time is (planes it marches) x (time per plane) + a start that does not
// depend on the chunk (launch, the first planes of the z queue), so the choice
// minimises that over the rounds of workgroups each CU takes; ties go to the
// longer chunk and the tile listed first.  Constants in us for both stages
// together, from sweeps of the chunk at 16^3..256^3 (MI355X):
//   FP64, eight owner waves: one workgroup per CU (LDS), 13 per plane + 33.
//     Tiles of 32 columns fill the lanes where the interior width is just
//     above a multiple of 64: 96^3 interior cells 187 us in 64 x 8 tiles, 154
//     in 32 x 16; where both fill them they take 1 % more (128^3 302, 294).
//   FP64, four owner waves: one workgroup per CU, 8.5 per plane + 30: half the
//     rows per CU, so faster where the wide tiles leave CUs idle (32^3 with
//     one plane each 41 us in 64 x 4 and 38 in 32 x 8 tiles, 46 in wide ones),
//     and slower where they fill the chip (256^3: 2.5 against 1.95 ms).
//   Mixed, four owner waves: several workgroups share a CU and its issue
//     slots, so the time is (workgroups per CU) x (chunk + 2 planes), with one
//     alone on its CU, which waits for its own latencies, counted as 1.6.
//     192^3: chunk 28 489 us, 32 545 us; 96^3 interior: 105 us in 64 x 4
//     tiles, 85 in 32 x 8; 100 x 130 x 90: 131, 132.
// tiles: the set to choose from (tile_bit).
int tile_split(const bx_ctx *c, bool mixed, unsigned tiles, int *lz)
{
    const int nzi = c->flatz ? c->nz : c->nz - 4;
    struct Shape {
        int tile, wx, ty;
        double plane, start, mixed;
    };
    static const Shape shapes[] = {
        {kTile64x8, 64, 8, 13.0, 33.0, 0.0},
        {kTile32x16, 32, 16, 13.2, 33.3, 0.0},
        {kTile64x4, 64, 4, 8.5, 30.0, 1.0},
        {kTile32x8, 32, 8, 9.0, 28.0, 1.02},
    };
    double best = HUGE_VAL;
    int at = kTile64x4;
    *lz = nzi;
    for (const Shape &t : shapes) {
        if (!(tiles & tile_bit(t.tile))) continue;
        const int64_t n = (int64_t)((c->nx - 4 + t.wx - 1) / t.wx) * ((c->ny - 4 + t.ty - 1) / t.ty);
        for (int m = 1; m <= nzi && m <= 4 * c->ncu; m++) {
            const int l = (nzi + m - 1) / m;
            const double rounds = (double)((n * ((nzi + l - 1) / l) + c->ncu - 1) / c->ncu);
            const double cost = mixed ? t.mixed * std::fmax(rounds, 1.6) * (l + 2) : rounds * (t.plane * l + t.start);
            if (cost < best) {
                best = cost;
                *lz = l;
                at = t.tile;
            }
        }
    }
    return at;
}

// The rule's work split of the stage kernels for a grid.  The y chunk only
// serves the two-kernel variants; gravity has the tiles of eight owner waves
// only.
void default_split(const bx_ctx *c, int *ly, int *lz, int *tile)
{
    const int64_t want = 2 * 1024;
    const int nzi = c->flatz ? c->nz : c->nz - 4;
    *ly = 64;
    while (*ly > 8 && (int64_t)((c->nx - 4 + 63) / 64) * nzi * ((c->ny - 4 + *ly - 1) / *ly) < want) *ly /= 2;
    const bool mixed = c->prm.precision == BX_PREC_MIXED;
    const unsigned wide = tile_bit(kTile64x8) | tile_bit(kTile32x16);
    const unsigned narrow = tile_bit(kTile64x4) | tile_bit(kTile32x8);
    *tile = tile_split(c, mixed, mixed ? narrow : (c->grav_flags ? wide : wide | narrow), lz);
}

// The context's split: the rule's unless bx_tune chose one.  Allocates nothing.
void fused_defaults(bx_ctx *c)
{
    int ly, lz, tile;
    default_split(c, &ly, &lz, &tile);
    if (c->fused_ly == 0) c->fused_ly = ly;
    if (c->fused_lz == 0) {
        c->fused_lz = lz;
        c->fused_occ = tile;
    }
}

// Ghost table shallow, allocation of the fused buffers.
int fused_prepare(bx_ctx *c)
{
    if (int rc = fused_supported(c)) return rc;
    if (c->prm.precision == BX_PREC_MIXED) {
        const size_t pf = sizeof(float) * (size_t)c->n;
        if (!c->cons32) BX_HIP(hipMalloc((void **)&c->cons32, 5 * pf));
        if (!c->ustar32) BX_HIP(hipMalloc((void **)&c->ustar32, 5 * pf));
        if (!c->unext32) BX_HIP(hipMalloc((void **)&c->unext32, 5 * pf));
        if (!c->pstar32) BX_HIP(hipMalloc((void **)&c->pstar32, pf));
    }
    const size_t pb = sizeof(double) * (size_t)c->n;
    if (!c->eflux) BX_HIP(hipMalloc((void **)&c->eflux, 5 * pb));
    if (!c->ustar) BX_HIP(hipMalloc((void **)&c->ustar, 5 * pb));
    if (!c->unext) BX_HIP(hipMalloc((void **)&c->unext, 5 * pb));
    if (!c->pstar) BX_HIP(hipMalloc((void **)&c->pstar, pb));
    fused_defaults(c);
    return BX_OK;
}

// Flags and Courant rate of the current (exact-path) state; ghosts must hold
// copies of their donors, which the exact sequence guarantees after a step.
int launch_regular_check(bx_ctx *c)
{
    BX_HIP(hipMemsetAsync(&c->dsc->flags, 0, sizeof(unsigned int), c->stream));
    BX_HIP(hipMemsetAsync(c->dsc->rate[0], 0, sizeof(c->dsc->rate[0]), c->stream));
    hipLaunchKernelGGL(k_regular, dim3(reduce_blocks(c->n)), dim3(256), 0, c->stream, c->n, c->cons, c->u,
                       c->prm.gammafix, c->prm.small_eps, c->prm.dx, c->prm.dy, c->prm.dz, &c->dsc->flags,
                       c->dsc->rate[0]);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

// corners: whether to fill the two-level corner ghosts too (the last nd2
// entries of the table) or leave what the fix-up wrote
template <typename S>
static int ghosts6(bx_ctx *c, S *planes, S *pstar, bool corners = true)
{
    const int64_t ng = c->nghost - (corners ? 0 : c->nd2);
    if (ng <= 0) return BX_OK;
    hipLaunchKernelGGL(k_ghosts6<S>, dim3(blocks_for(ng, 256)), dim3(256), 0, c->stream, c->n, ng,
                       c->ghost_dst, c->nscratch ? c->fghost_src : c->ghost_src,
                       c->nscratch ? c->fghost_sign : c->ghost_sign, planes, pstar);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

__global__ __launch_bounds__(192) void k_corner_ghosts(StageArgs a0)
{
    __shared__ double F[3][2][5];
    const StageArgs a = with_dt(a0);
    corner_block(a, blockIdx.x, F);
}

// after the corrector, and after any ghost fill of un that writes these ghosts (b: the corrector's arguments)
static int corner_ghosts(bx_ctx *c, const StageArgs &b)
{
    if (c->nd2 == 0) return BX_OK;
    hipLaunchKernelGGL(k_corner_ghosts, dim3((unsigned)c->nd2), dim3(192), 0, c->stream, b);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

int narrow_cons(bx_ctx *c)
{
    hipLaunchKernelGGL(k_narrow, dim3(blocks_for(5 * c->n, 256)), dim3(256), 0, c->stream, 5 * c->n, c->cons,
                       c->cons32);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

int widen_cons(bx_ctx *c)
{
    hipLaunchKernelGGL(k_widen, dim3(blocks_for(5 * c->n, 256)), dim3(256), 0, c->stream, 5 * c->n, c->cons32,
                       c->cons);
    BX_HIP(hipGetLastError());
    return BX_OK;
}

// With gravity the corrector also writes the pressure plane (the state after
// source(1), which takes the velocity from before the kick); returns that
// plane for the ghost fill, null without gravity.
template <typename S>
static S *grav_pressure(bx_ctx *c, StageArgs &b)
{
    if constexpr (sizeof(S) == 8) {
        if (b.gf) {
            b.pout = c->p;
            return c->p;
        }
    }
    return nullptr;
}

// Whether the stage kernels read donors in place of ghost cells.  Gravity with
// walls reads its ghosts from memory: the signs take the gravity form over its
// registers (12 to 19 VGPRs spilled).
static bool reads_donors(const bx_ctx *c)
{
    bool wall = false;
    for (int i = 0; i < 6; i++) wall = wall || c->prm.no_outflow[i];
    return c->axis_ghosts && c->fused_occ >= 10 && !(c->grav_flags && wall);
}

static void read_donors(const bx_ctx *c, StageArgs &a)
{
    a.gmap = 1;
    for (int i = 0; i < 6; i++) a.wall[i] = c->prm.no_outflow[i] ? 1 : 0;
}

// One fused step u0 -> us, ps -> un from a regular state, with full dt `dt`
// or, for par = 0 or 1, with dt formed on the device from slot[par] and
// rate[par] (left in slot[par^1], logged in log[cap]).  The Courant rate of
// U^{n+1} is left in rate[0] or rate[par^1]; irregular branches
// are added to the flags.  fill: the ghost cells of us, ps and un hold their
// donors' values afterwards (otherwise those of the stage inputs need not,
// and those of un do not, but for the corner ghosts).
template <typename S>
static int enqueue_step(bx_ctx *c, double dt, int par, double *log, int cap, S *u0, S *us, S *ps, S *un,
                        bool fill_us, bool fill_un)
{
    int rc;
    const bool donors = reads_donors(c);
    unsigned long long *rate = c->dsc->rate[par < 0 ? 0 : par ^ 1];
    StageArgs a = base_args(c, dt);
    if (donors) read_donors(c, a);
    StageArgs b = a;
    if (par >= 0) {
        a.slot = &c->dsc->slot[par];
        a.slot_next = &c->dsc->slot[par ^ 1];
        a.rate_in = c->dsc->rate[par];
        a.cfl = c->prm.cfl;
        a.log = log;
        a.log_cap = cap;
        b.dtp = &c->dsc->slot[par ^ 1].dt;
    }
    a.rate_next = rate;
    a.uin = u0;
    a.uout = us;
    a.pout = ps;
    b.uin = us;
    b.pin = ps;
    b.uold = u0;
    b.uout = un;
    b.rate = rate;
    b.rate_mask = kRateSlots - 1;
    // The corner ghosts take their inputs from stage 1's output alone (through
    // the donors), so they run in workgroups of stage 2's launch, ahead of its
    // tiles: 13.7 us less on each step's path than in a launch of their own.
    const bool corners = sizeof(S) == 8 && donors && c->nd2 > 0;
    if (corners) b.ncorner = (c->nd2 + 7) & ~7;
    S *pfin = grav_pressure<S>(c, b);
    if (c->prof_on) BX_HIP(hipEventRecord(c->ev[0], c->stream));
    if ((rc = launch_stage<1, S>(c, a, c->prof_on ? c->ev[1] : nullptr, (S *)c->eflux))) return rc;
    if (c->prof_on) BX_HIP(hipEventRecord(c->ev[2], c->stream));
    if ((fill_us || !donors) && (rc = ghosts6<S>(c, us, ps))) return rc;
    if (c->prof_on) BX_HIP(hipEventRecord(c->ev[3], c->stream));
    if ((rc = launch_stage<2, S>(c, b, c->prof_on ? c->ev[4] : nullptr, (S *)c->eflux))) return rc;
    if (c->prof_on) BX_HIP(hipEventRecord(c->ev[5], c->stream));
    if ((fill_un || !donors) && (rc = ghosts6<S>(c, un, pfin, !corners))) return rc;
    if constexpr (sizeof(S) == 8)
        if (!corners) return corner_ghosts(c, b);
    return BX_OK;
}

// ------------------------------------------------------ runs of steps
// Two fused steps, u0 -> un -> u0, with dt from the device scalars.
template <typename S>
static int enqueue_pair(bx_ctx *c, S *u0, S *us, S *ps, S *un)
{
    int rc;
    if ((rc = enqueue_step<S>(c, 0.0, 0, c->chunk_dts, kChunkSteps, u0, us, ps, un, false, false))) return rc;
    return enqueue_step<S>(c, 0.0, 1, c->chunk_dts, kChunkSteps, un, us, ps, u0, false, false);
}

static int enqueue_current_pair(bx_ctx *c)
{
    return c->state_in_32 ? enqueue_pair<float>(c, c->cons32, c->ustar32, c->pstar32, c->unext32)
                          : enqueue_pair<double>(c, c->cons, c->ustar, c->pstar, c->unext);
}

// The ghost cells of the current state after a run of pairs.
static int fill_after_run(bx_ctx *c)
{
    if (!reads_donors(c)) return BX_OK;
    if (c->state_in_32) return ghosts6<float>(c, c->cons32, (float *)nullptr);
    return ghosts6<double>(c, c->cons, c->grav_flags ? c->p : (double *)nullptr, false);
}

void drop_step_graphs(bx_ctx *c)
{
    for (int i = 0; i < 2; i++) {
        if (c->sexec[i]) (void)hipGraphExecDestroy(c->sexec[i]);
        if (c->sgraph[i]) (void)hipGraphDestroy(c->sgraph[i]);
        c->sexec[i] = nullptr;
        c->sgraph[i] = nullptr;
        c->skey[i] = c->skey2[i] = nullptr;
    }
}

// The captured pair that starts from the current state buffer (captured on
// first use; one per buffer parity and precision, two kept).
static int pair_exec(bx_ctx *c, hipGraphExec_t *out)
{
    const bool f32 = c->state_in_32;
    const void *key = f32 ? (const void *)c->cons32 : (const void *)c->cons;
    const void *key2 = f32 ? (const void *)c->unext32 : (const void *)c->unext;
    for (int i = 0; i < 2; i++)
        if (c->sexec[i] && c->skey[i] == key && c->skey2[i] == key2) {
            *out = c->sexec[i];
            return BX_OK;
        }
    const int slot = c->sexec[0] ? (c->sexec[1] ? c->snext : 1) : 0;
    c->snext = 1 - slot;
    if (c->sexec[slot]) (void)hipGraphExecDestroy(c->sexec[slot]);
    if (c->sgraph[slot]) (void)hipGraphDestroy(c->sgraph[slot]);
    c->sexec[slot] = nullptr;
    c->sgraph[slot] = nullptr;
    c->skey[slot] = c->skey2[slot] = nullptr;
    BX_HIP(hipStreamSynchronize(c->stream));
    BX_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue_current_pair(c);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(c->stream, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    BX_HIP(e);
    hipGraphExec_t x = nullptr;
    const hipError_t ei = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (ei != hipSuccess) {
        (void)hipGraphDestroy(g);
        return hip_check(ei, "hipGraphInstantiate");
    }
    c->sgraph[slot] = g;
    c->sexec[slot] = x;
    c->skey[slot] = key;
    c->skey2[slot] = key2;
    *out = x;
    return BX_OK;
}

int run_step_pairs(bx_ctx *c, int pairs, bool graph)
{
    int rc;
    if (!c->chunk_dts) BX_HIP(hipMalloc((void **)&c->chunk_dts, sizeof(double) * kChunkSteps));
    if (graph) {
        hipGraphExec_t x = nullptr;
        if ((rc = pair_exec(c, &x))) return rc;
        for (int i = 0; i < pairs; i++) BX_HIP(hipGraphLaunch(x, c->stream));
    } else {
        for (int i = 0; i < pairs; i++)
            if ((rc = enqueue_current_pair(c))) return rc;
    }
    return fill_after_run(c);
}

int fused_step_into(bx_ctx *c, double dt, double *u0, double *us, double *ps, double *un, bool reset_flags)
{
    if (reset_flags) BX_HIP(hipMemsetAsync(&c->dsc->flags, 0, sizeof(unsigned int), c->stream));
    return enqueue_step<double>(c, dt, -1, nullptr, 0, u0, us, ps, un, true, true);
}

__global__ void k_clear_scalars(unsigned int *flags, unsigned long long *rate)
{
    if (threadIdx.x == 0) *flags = 0u;
    rate[threadIdx.x * kMaxStride] = 0ull;
}

// One FP64 fused step u0 -> us, ps -> un (ey: the y-term planes) on the
// context's stream with the flags and the Courant rate (kRateSlots slots)
// accumulated into the given device words, which a kernel clears first (no memset nodes, so the sequence can be captured).
// Allocates nothing; the tile defaults must be set (fused_defaults).
int fused_step_words(bx_ctx *c, double dt, const double *u0, double *us, double *ps, double *un, double *ey,
                     unsigned int *flags, unsigned long long *rate)
{
    if (c->grav_flags) return set_error(BX_ERR_UNSUPPORTED, "this fused step entry takes no gravity configuration");
    int rc;
    hipLaunchKernelGGL(k_clear_scalars, dim3(1), dim3(kRateSlots), 0, c->stream, flags, rate);
    BX_HIP(hipGetLastError());
    StageArgs a = base_args(c, dt);
    a.flags = flags;
    a.uin = u0;
    a.uout = us;
    a.pout = ps;
    if ((rc = launch_stage<1, double>(c, a, nullptr, ey))) return rc;
    if ((rc = ghosts6<double>(c, us, ps))) return rc;
    StageArgs b = base_args(c, dt);
    b.flags = flags;
    b.uin = us;
    b.pin = ps;
    b.uold = u0;
    b.uout = un;
    b.rate = rate;
    b.rate_mask = kRateSlots - 1;
    if ((rc = launch_stage<2, double>(c, b, nullptr, ey))) return rc;
    if ((rc = ghosts6<double>(c, un, (double *)nullptr))) return rc;
    return corner_ghosts(c, b);
}

// Step k of a run whose dts are formed on the device (scalars of step 0 in
// slot[0], its rate in rate[0]), logged into log[cap]
int fused_step_device_dt(bx_ctx *c, int k, double *u0, double *us, double *ps, double *un, double *log, int cap)
{
    return enqueue_step<double>(c, 0.0, k & 1, log, cap, u0, us, ps, un, true, true);
}

int fused_step(bx_ctx *c, double dt)
{
    BX_HIP(hipMemsetAsync(&c->dsc->flags, 0, sizeof(unsigned int), c->stream));
    if (c->prm.precision == BX_PREC_MIXED)
        return enqueue_step<float>(c, dt, -1, nullptr, 0, c->cons32, c->ustar32, c->pstar32, c->unext32, false, true);
    return enqueue_step<double>(c, dt, -1, nullptr, 0, c->cons, c->ustar, c->pstar, c->unext, false, true);
}

}  // namespace bx
