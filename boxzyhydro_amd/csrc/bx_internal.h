// bx_internal.h -- context layout and launch helpers shared by the HIP sources.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "boxzy.h"
#include "bx_runs.h"

namespace bx {

struct HostPipe;

constexpr int kMaxSlots = 32, kMaxStride = 16;  // slots of a grid-wide maximum, and 8-byte words from one to the next

constexpr int kMaxD2 = 64;  // two-level ghost compositions a context may have (one wave)

// Slots of the fused step's Courant rate (a power of two, one row of 16 lanes
// reads them).  Every wave of stage 2 looks at the rate and adds its share:
// 784 waves on one word took half of a 32^3 stage 2 (22.6 us, with slots 13.3).
constexpr int kRateSlots = 16;

// The step scalars of main.f90 as a device-dt step leaves them.
struct StepSlot {
    double dt;       // full dt of the step (main.f90:342)
    double dtold;    // main.f90:271
    double time;     // at the step's start (main.f90:545 advances it)
    double endtime;
    int step;        // main.f90:213
    int logk;        // steps of the current run so far (index into its dt log)
};

// Scalars that live on the device so whole steps can run without host syncs.
// Device-dt steps alternate between the two slots and rates (a step reads one
// and writes the other), so that no workgroup reads what another one writes.
struct DevScalars {
    // Courant max-rate (non-negative doubles as bits), ping-pong, each in
    // kRateSlots words of a cache line each: a rate is their maximum
    unsigned long long rate[2][kRateSlots * kMaxStride];
    unsigned int flags;               // irregular-branch flags raised by the fused kernels
    unsigned int pad;
    StepSlot slot[2];
    unsigned int slow[2];             // FLAG_SLOW of a tiled flux call; calls alternate between the two words
};
inline unsigned long long rate_bits(const DevScalars *s, int par)
{
    unsigned long long m = 0ull;
    for (int i = 0; i < kRateSlots; i++) m = s->rate[par][i * kMaxStride] > m ? s->rate[par][i * kMaxStride] : m;
    return m;
}
inline void set_rate_bits(DevScalars *s, int par, unsigned long long bits)
{
    for (int i = 0; i < kRateSlots; i++) s->rate[par][i * kMaxStride] = i == 0 ? bits : 0ull;
}

// flags bits
enum : unsigned int {
    FLAG_LOWRHO = 1u,  // a state() call met rho<1e-4 (state.f90:52-56)
    FLAG_CLAMP = 2u,   // a velocity() call met |u_i|>vlimit (velocity.f90:33)
    FLAG_FLOOR = 8u,   // a floor of the stage update acted (flux.f90:225-228, the source re-round
                       // or the p* eps floor); informational: the step is exact either way
    FLAG_SLOW = 16u,   // the tiled flux met a value outside its range (bx_stage.h prims)
    FLAG_IRREGULAR = FLAG_LOWRHO | FLAG_CLAMP,
};

}  // namespace bx

struct bx_ctx {
    bx_params prm;
    int device;
    hipStream_t stream;
    int nx, ny, nz;
    int64_t n;        // ngrid
    int64_t nghost;
    double muc, rgas;
    double grav[3];   // uniform gravity acceleration; -0.0 from phi=0 (utils.f90:566-568)
    bool flatz;       // nz<6: z neighbours are the cell itself (init_grid.f90:241-247)

    // exact-path device state, SoA planes of n doubles
    double *cons;      // 5 planes: rho, mx, my, mz, E
    double *cons_old;  // 5 planes
    double *u;         // 3 planes
    double *p;
    double *adindx;
    double *qq;        // 3 planes
    double *states;    // 5 planes: the exact flux's result, which trades places with cons
    bool ad_uniform;   // every cell of adindx holds gammafix
    unsigned nflux;    // tiled flux calls so far (parity: which slow word a call uses)
    int ncu;           // compute units of the device

    // ghost table: ghost cell id, donor (>=0: cell id; <0: -(scratch slot+1)),
    // sign bits (bit k flips momentum k); scratch holds pre-fill values of
    // ghost donors (5 planes of nscratch)
    int32_t *ghost_dst;
    int32_t *ghost_src;
    int32_t *ghost_sign;
    int32_t *ghost_scratch_src;
    double *ghost_scratch;
    int64_t nscratch;
    // the same table composed over a pair of set_ghost_cells calls (every call
    // site of the step makes two in a row): ghost dst[k] <- +-(interior cell
    // fsrc[k]), exact when each scratch donor's own donor is an interior cell
    // (fghost_ok); equal to the table above when nscratch == 0
    int32_t *fghost_src;
    int32_t *fghost_sign;
    bool fghost_ok;
    // every ghost's composed donor is the per-axis one (axis_donor), an
    // interior cell: the tiled kernels then read donors in place of ghosts
    bool axis_ghosts;
    // ghosts whose pair leaves the pre-pair value of another ghost h2 (whose
    // own pair gives an interior cell v): the corner ghosts of a box walled
    // in y and z.  After a step such a ghost holds +-(v's corrector result
    // before source(1)); a fix-up kernel after the corrector's ghost fill
    // writes it (d2_ubar: 6 doubles per entry, its scratch, the last one the
    // ghost's pressure for the materialised planes).  fghost_src/sign map
    // them to v for the other fills.
    int nd2;
    int32_t *d2_dst;   // ghost cell
    int32_t *d2_src;   // interior cell v
    int32_t *d2_sign;  // sign bits of the composition
    double *d2_ubar;

    // fused-path state
    double *ustar;     // 5 planes: stage-1 result U*
    double *pstar;     // stage-2 pressure p* (stale-velocity EOS, main.f90:351-355)
    double *unext;     // 5 planes: stage-2 result U^{n+1}
    bool fused_valid;  // device cons holds a regular state (see bx_step)
    bool fused_ready;  // fused buffers allocated, ghost table shallow
    bool fused_unsupported;
    bool ghosts_filled;  // ghost cells hold their donors' values (after any exact step)
    int fused_ly, fused_lz;  // y rows and z planes per wave of the stage kernels
    int fused_occ;           // stage kernel variant: 0, 1, 4 two kernels; from 10 one tiled kernel (Tile)
    double *eflux;           // 5 planes: y-term of fluxtmp (FP64)
    bool prof_on;
    hipEvent_t ev[6];   // per stage: before the y kernel, between the two kernels, after the x/z kernel
    double prof_ms[4];  // summed durations: y kernel stage 1, x/z kernel stage 1, y kernel stage 2, x/z kernel stage 2
    int64_t prof_steps;
    bool aux_stale;    // u, p planes not materialised since the last fused step
    bool old_stale;    // cons_old not materialised since the last fused step
    int64_t fallbacks;
    int64_t nfused, nexact;  // steps bx_step took with the fused kernels / the exact sequence

    // captured pairs of fused steps (BX_STEP_GRAPH), keyed by the state buffer
    // they start from (the pair returns the state to it) and the other one
    // (the exact path's flux trades the state buffer for another)
    hipGraph_t sgraph[2];
    hipGraphExec_t sexec[2];
    const void *skey[2], *skey2[2];
    int snext;             // the slot the next capture replaces
    void *chunk0;          // 5 planes: the state at the start of a replayed chunk (rollback)
    bx::RunPacing runs;    // when the next run may be taken
    int64_t graph_steps;   // steps taken from replays (kept, not undone)
    double *chunk_dts;     // dt of each step of a chunk
    double *stage;         // device staging of host transfers (Fortran layout), stage_len doubles
    int64_t stage_len;
    struct bx::HostPipe *pipe;  // pinned slots of large host transfers (bx_transfer.hip), or null

    unsigned long long *dmax, *hmax;  // slots of a grid-wide maximum (bx_cells.h), and a pinned word for it
    bool max_open;                    // a kernel has added to the slots since they were last taken and cleared

    bx::DevScalars *dsc;   // device scalars
    bx::DevScalars *hsc;   // pinned host mirror

    // mixed-precision planes (FP32 storage)
    float *cons32, *ustar32, *unext32, *pstar32;
    bool state_in_32;  // the current state lives in cons32 (mixed form)

    struct bx_adj *adj;  // adjoint store (bx_adjoint.hip), or null
    struct bx_eos *eos;  // tabulated EOS (bx_eos.hip), or null for a fixed gamma

    // gravity (bx_gravity.hip): a given potential and per-cell gforce(3,n) planes
    int grav_flags;                // BX_GRAV_* bits, 0 = uniform -0.0 force of phi = 0
    double obj_mass, obj_radius;   // external_grav point mass (parameters.f90:83-86)
    double *phi;                   // n
    double *gforce;                // 3 planes
    double *grav_sums;             // centre-of-mass sums (3) and tree partials
    // The fused step with a potential (BX_GRAV_POTENTIAL alone): gforce is
    // settled when it was computed from the current phi (gforce_gen ==
    // phi_gen), so that source(0) and source(1) of a step see the same force;
    // gfused is gforce with the ghosts filled as their donors' (sign flips of
    // the momenta), built from generation gfused_gen.  p_fused: the pressure
    // plane holds what the last step's exact sequence would leave (written by
    // the fused corrector), so materialising keeps it.
    int64_t phi_gen, gforce_gen, gfused_gen;
    double *gfused;  // 3 planes
    bool p_fused;
};

namespace bx {

int set_error(int code, const std::string &msg);
int hip_check(hipError_t e, const char *what);

#define BX_HIP(call)                                             \
    do {                                                         \
        hipError_t _e = (call);                                  \
        if (_e != hipSuccess) return bx::hip_check(_e, #call);   \
    } while (0)

// blocks of a reduction over n cells into one word (256 threads, each taking
// every gridDim-th 256 cells), or of a kernel that mostly has nothing to do
inline unsigned int reduce_blocks(int64_t n) { return (unsigned int)((n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024); }

inline unsigned int blocks_for(int64_t n, int threads)
{
    return (unsigned int)((n + threads - 1) / threads);
}

// kernels launched by the C-ABI (defined in bx_exact.hip / bx_fused.hip)
int launch_state(bx_ctx *c);
int launch_velocity(bx_ctx *c, bool want_maxv);
int launch_courant(bx_ctx *c);
int launch_source(bx_ctx *c, double dt);
int launch_ghosts(bx_ctx *c, double *planes5);
// ghosts: whether to fill the ghost cells after it (flux.f90:231)
int launch_flux(bx_ctx *c, int avg, double dt, bool ghosts);
int launch_tiled_flux(bx_ctx *c, int avg, double dt, double *out, unsigned int *slow, unsigned int *slow_next);
// tiles of the tiled kernels (fused_occ of the fused step): columns x rows;
// 64 x 4 and 32 x 8 have four waves of owners, the others eight
enum Tile : int { kTile64x4 = 10, kTile64x8 = 11, kTile32x8 = 12, kTile32x16 = 13 };
constexpr unsigned tile_bit(int tile) { return 1u << (tile - kTile64x4); }
// Whether the stage kernels reach every cell of a grid with elements of `size`
// bytes: they address a cell by its plane and a 32-bit byte offset within it,
// and the rows of tiles (at least 4 rows of cells each) are the launch's y
// dimension.
inline bool tile_fits(int64_t nx, int64_t ny, size_t size)
{
    return nx * ny <= (int64_t)(((uint64_t)1 << 32) / size) && (ny - 4 + 3) / 4 <= 65535;
}
inline bool tile_fits(const bx_ctx *c, size_t size) { return tile_fits(c->nx, c->ny, size); }
int tile_split(const bx_ctx *c, bool mixed, unsigned tiles, int *lz);
void default_split(const bx_ctx *c, int *ly, int *lz, int *tile);
int launch_avisc(bx_ctx *c);
int launch_materialize(bx_ctx *c);
int launch_regular_check(bx_ctx *c);
int fused_step(bx_ctx *c, double dt);
// one FP64 fused step U^n=u0 -> U*=us, p*=ps -> U^{n+1}=un (ghosts filled); the rate is zeroed
// first, the flags too when reset_flags (else they accumulate over steps)
int fused_step_into(bx_ctx *c, double dt, double *u0, double *us, double *ps, double *un, bool reset_flags);
// the same, step k of a run, with dt formed on the device from the current
// Courant rate (the device scalars carry time, dtold, step and endtime, at the
// run's start in slot[0] and rate[0]; after k steps in [k & 1]); flags
// accumulate and each dt is logged into log[cap]
int fused_step_device_dt(bx_ctx *c, int k, double *u0, double *us, double *ps, double *un, double *log, int cap);
void adjoint_free(bx_ctx *c);
void eos_free(bx_ctx *c);
void gravity_free(bx_ctx *c);
int launch_calc_gforce(bx_ctx *c);
int launch_external_grav(bx_ctx *c);
bool grav_settled(const bx_ctx *c);
int grav_fused_planes(bx_ctx *c);
// the pointwise calls of the exact step in fused passes (bx_pass.hip)
enum Pass : int {
    kState = 0,       // state
    kStateRate = 1,   // state, Courant rate                           main.f90:232-241
    kAfterFlux = 2,   // (ghosts,) state, velocity                     :351-355
    kBeforeFlux = 3,  // source, (ghosts,) state, velocity             :289-318
    kEnd = 4,         // (ghosts,) state, velocity, source, (ghosts,) state, velocity  :374-515
    kEndNext = 5,     // kEnd, then the next step's kStateRate
};
int launch_pass(bx_ctx *c, int pass, double dt, bool filled);
int begin_max(bx_ctx *c);
int read_max(bx_ctx *c, double *out);
int fused_prepare(bx_ctx *c);
// `pairs` pairs of fused steps from the current state (device dt, flags
// accumulating), replayed from a captured graph (BX_STEP_GRAPH) or enqueued;
// the scalars must be on the device
int run_step_pairs(bx_ctx *c, int pairs, bool graph);
void drop_step_graphs(bx_ctx *c);
int narrow_cons(bx_ctx *c);
int widen_cons(bx_ctx *c);

// The ghost table of a grid (bx_ghost_table's gd, gs, gg, gx) composed over a
// pair of set_ghost_cells calls: ghost gd[k] <- +-(interior cell src[k]); ok
// when every entry resolves, the two-level corner ghosts (entries d2at, see
// bx_ctx) among them.
struct GhostPair {
    std::vector<int32_t> src, sign;
    std::vector<size_t> d2at;
    std::vector<int32_t> d2dst, d2src, d2sign;
    bool ok;
};
void compose_ghosts(int64_t n, const std::vector<int32_t> &gd, const std::vector<int32_t> &gs,
                    const std::vector<int32_t> &gg, const std::vector<int32_t> &gx, GhostPair &out);

// Large host transfers (bx_transfer.hip).  A transfer is cut into chunks of
// whole units (bytes); worker w of kWorkers calls, with `self`, for the bytes
// [off, off+len) of the host array: get (download) enqueues whatever forms
// them on the device and returns where they are; room (upload) says where they
// go and put enqueues what follows the copy.  Device memory a callback hands
// out must be w's own.  Without a pipe (small transfers, no pinned memory)
// chunks of at most stage_bytes (0: any size) go one after another with w = 0.
// Calls return after the transfer.
struct PipeChunk {
    hipError_t (*get)(void *self, size_t off, size_t len, int w, const void **src);
    hipError_t (*room)(void *self, size_t off, size_t len, int w, void **to);
    hipError_t (*put)(void *self, size_t off, size_t len, int w);
    size_t stage_bytes;
};
constexpr size_t kPipeMin = size_t(8) << 20;  // smaller transfers are copied directly
size_t pipe_stage_bytes();                    // device staging that gives every worker a slot of its own
size_t pipe_slot_bytes();
int pipe_download(HostPipe **slot, int device, hipStream_t stream, char *dst, size_t bytes, size_t unit,
                  const PipeChunk &chunk, void *self);
int pipe_upload(HostPipe **slot, int device, hipStream_t stream, const char *src, size_t bytes, size_t unit,
                const PipeChunk &chunk, void *self);
void pipe_free(HostPipe *p);

}  // namespace bx
