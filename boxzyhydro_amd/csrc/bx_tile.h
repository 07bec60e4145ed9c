// bx_tile.h -- one RK stage of the fused step as a single kernel: a workgroup
// holds an x-y tile of the grid with its +-2 halo in LDS and marches in z.
//
// Tile: WX x-cells by TY rows of outputs.  With WX = 64 the workgroup has TY+4
// waves, wave w with row r = w-2 of the tile (rows -2..TY+1, the two outer
// rows on each side being the y-halo), a cell per lane.  With WX = 32 a wave
// holds two rows, and the x-edges have waves of their own: for 16 rows again
// 12 waves, 8 of them owners.  Grids whose interior width lies just above a
// multiple of 64 fill the lanes of narrow tiles (tile_split chooses): at 96^3
// interior cells the step takes 154 us in place of 187, at 160x144x128 with
// gravity 498 in place of 572.  The primitives of a plane are
// kept in a tile in LDS with one column of x-halo on each side; there are two
// such tiles, for planes k and k+1.  Every row writes its primitives one
// plane ahead, so that the tile of plane k is complete when plane k starts.
// Per z-plane k:
//
//   A  owner rows 0..TY-1 take the z face k+1/2 from their register queue in
//      z (the primitives of plane k from the tile, k+1 and k+2 in registers)
//      and park the z flux difference of plane k in LDS; every row writes its
//      primitives of plane k+1 into the other tile.  The edge wave
//      (with WX = 64 wave r=TY+1, else one per 8 rows) takes the x-edges of
//      the owner rows on plane k+1: columns -2,-1,0 and WX-2..WX+1, seven
//      lanes per row, their primitives (columns -1 and WX go into the
//      plane-(k+1) tile) and x-states.
//   B  owner rows form their x-states from the neighbours' primitives
//      (flux.f90:253-351, 391-479), the x-faces l-1/2 (the left plus state
//      from the next lower lane, or column -1's for column 0) and with face
//      l+1/2 (next higher lane, or face WX-1/2) the x flux difference, parked
//      in LDS; then their y-states, publishing the y-plus state (row r-1's
//      is needed by row r's face r-1/2).  Row -1 publishes its y-plus state,
//      row TY keeps its y-minus state.                            -- barrier
//   C  owner rows and row TY evaluate their face y r-1/2 and publish it over
//      the y-plus state they read (no other row reads that slot).  The
//      edge wave publishes the x-plus state of column -1 and evaluates face
//      x WX-1/2 of plane k+1 (the owners read plane k's in B).    -- barrier
//   D  owner rows read face y r+1/2 and apply the stage update and
//      everything pointwise up to the next stage (as the two-kernel form
//      does).
//
// A and B need no barrier between them: the tile they write in A is read
// from the next plane on, and the y-plus slot row r writes in B is read in
// D only by row r itself.  Every wave runs a loop of its own role with the
// same two barriers per plane (and one before the first), so that no
// register holds a value of another role.  Each face and each cell's
// primitives are evaluated once per workgroup, except at the tile's edges:
// the y-halo costs 4 rows of primitives, 2 rows of states and 1 row of faces
// per TY rows; the x-edges 7 cells of primitives, states and faces per row
// (one wave pass).
// Ghost cells (StageArgs::gmap): a ghost holds its donor's values, so the loads
// of a ghost take the donor's address instead (per lane in x and y, per plane
// in z: the tile's cells keep their own coordinates for the slopes and the
// outputs), and at a wall (W) the normal velocity changes sign.  The ghost
// cells of the stage's input then need no fill before it: two dispatches less
// per step (4.6 us each on small grids, 33 us each at 256^3).
// Stages 3 and 4 are the flux subroutine of the exact path (flux(0), flux(1)):
// the same march over the planes cons, u, p (and adindx) as they stand, ghosts
// from memory, ending with flux.f90:205-228.  With flux_ang (has_ang) two more
// fields are reconstructed, and each x and y face is projected twice, for the
// cell above and the cell below it.
// Every arithmetic operation is the one the exact sequence performs on the
// same values, so the results are bit-identical to it.
#pragma once

#include <type_traits>

#include "bx_stage.h"
#include "bx_waves.h"

namespace bx {

// A wave of a tile of WX columns holds 64 columns of one row or 32 of two.
// Its waves: halo rows, owner rows, and the x-edges of the owner rows, 7 lanes
// to a row, kEdgeRows rows to a wave (with 64 columns the one edge wave has a
// halo row besides).
constexpr int kEdgeRows = 8;
constexpr int tile_waves(int TY, int WX)
{
    return WX == 64 ? TY + 4 : TY / 2 + 2 + (TY + kEdgeRows - 1) / kEdgeRows;
}

template <typename S, int TY, int V = kPlain, int WX = 64>
struct TileLds {
    static constexpr int RS = WX + 2;  // row stride of the primitive tile: columns -1..WX
    static constexpr int NF = 6 + (has_gamma(V) ? 1 : 0) + (has_ang(V) ? 2 : 0);
    S P[2][NF][(TY + 4) * RS];     // rho, u0, u1, u2, p, eps (, gamma) (, r- and angular momentum) of planes k, k+1 (tile k&1), rows -2..TY+1
    S Sy[NF][(TY + 1) * WX];       // y-plus states of rows -1..TY-1 (index r+1), then y-face r-1/2 (index r)
    S SxL[NF][TY];                 // x-plus state of column -1, per owner row
    S FxR[5][TY];                  // x-face flux WX-1/2, per owner row
    double Dx[5][TY * WX];         // x flux difference of each owner cell (phase B to D)
    double Dz[5][TY * WX];         // z flux difference of each owner cell (phase A to D)
};

template <typename S, int F, int N>
__device__ __forceinline__ void store_w(S (&P)[F][N], int idx, const W6<S> &w)
{
    if constexpr (F == 7 || F == 9) P[6][idx] = w.g;
    if constexpr (F >= 8) {
        P[F - 2][idx] = w.rm;
        P[F - 1][idx] = w.am;
    }
    P[0][idx] = w.d;
    P[1][idx] = w.u0;
    P[2][idx] = w.u1;
    P[3][idx] = w.u2;
    P[4][idx] = w.p;
    P[5][idx] = w.e;
}

template <typename S, int F, int N>
__device__ __forceinline__ W6<S> fetch_w(const S (&P)[F][N], int idx)
{
    W6<S> w;
    w.g = w.rm = w.am = S(0);
    if constexpr (F == 7 || F == 9) w.g = P[6][idx];
    if constexpr (F >= 8) {
        w.rm = P[F - 2][idx];
        w.am = P[F - 1][idx];
    }
    w.d = P[0][idx];
    w.u0 = P[1][idx];
    w.u1 = P[2][idx];
    w.u2 = P[3][idx];
    w.p = P[4][idx];
    w.e = P[5][idx];
    return w;
}

template <typename S, int F, int N>
__device__ __forceinline__ void store_side(S (&B)[F][N], int idx, const Side<S> &s)
{
    if constexpr (F == 7 || F == 9) B[6][idx] = s.g;
    if constexpr (F >= 8) {
        B[F - 2][idx] = s.s1;
        B[F - 1][idx] = s.s2;
    }
    B[0][idx] = s.d;
    B[1][idx] = s.v[0];
    B[2][idx] = s.v[1];
    B[3][idx] = s.v[2];
    B[4][idx] = s.p;
    B[5][idx] = s.e;
}

template <typename S, int F, int N>
__device__ __forceinline__ Side<S> fetch_side(const S (&B)[F][N], int idx, S gam)
{
    Side<S> s;
    s.d = B[0][idx];
    s.v[0] = B[1][idx];
    s.v[1] = B[2][idx];
    s.v[2] = B[3][idx];
    s.p = B[4][idx];
    s.e = B[5][idx];
    s.g = gam;
    if constexpr (F == 7 || F == 9) s.g = B[6][idx];
    if constexpr (F >= 8) {
        s.s1 = B[F - 2][idx];
        s.s2 = B[F - 1][idx];
    }
    return s;
}

// value of the next lower column; column 0 takes `edge`
template <int WX, typename T>
__device__ __forceinline__ T from_lower(T v, T edge, int col)
{
    const T w = wave_shift_t<0x138>(v, edge);  // wave_shr:1
    return WX < 64 && col == 0 ? edge : w;
}

// value of the next higher column; the last column takes `edge`
template <int WX, typename T>
__device__ __forceinline__ T from_upper(T v, T edge, int col)
{
    const T w = wave_shift_t<0x130>(v, edge);  // wave_shl:1
    return WX < 64 && col == WX - 1 ? edge : w;
}

// Where a tile's row (or edge lane) at column x and row y reads its cells, and
// at walls the sign bits of the velocity components there (0 or the sign bit
// of the high word; the z component per plane).  prims() of a cell with a
// negated momentum is prims() of the cell with the velocity negated, bit for
// bit: quotients and products by a sign are exact.
template <typename S, bool W>
struct Donor {
    unsigned off;     // byte offset within a plane
    unsigned sx, sy;  // W only
    __device__ __forceinline__ Donor(const StageArgs &a, int x, int y)
    {
        int xd = min(max(x, 0), a.nx - 1), yd = min(max(y, 0), a.ny - 1);
        sx = sy = 0u;
        if (a.gmap) {
            if (W) {
                sx = axis_flip(xd, a.nx, a.wall[0], a.wall[1]) ? 0x80000000u : 0u;
                sy = axis_flip(yd, a.ny, a.wall[2], a.wall[3]) ? 0x80000000u : 0u;
            }
            xd = axis_donor(xd, a.nx, W && a.wall[0], W && a.wall[1]);
            yd = axis_donor(yd, a.ny, W && a.wall[2], W && a.wall[3]);
        }
        off = (unsigned)(yd * a.nx + xd) * (unsigned)sizeof(S);
    }
    // plane k's element offset (uniform)
    static __device__ __forceinline__ int64_t plane(const StageArgs &a, int64_t plane, int k)
    {
        if (a.gmap && !a.flatz) k = axis_donor(k, a.nz, W && a.wall[4], W && a.wall[5]);
        return (int64_t)k * plane;
    }
    static __device__ __forceinline__ S flip(S v, unsigned m)
    {
        if constexpr (sizeof(S) == 8)
            return __longlong_as_double(__double_as_longlong(v) ^ (long long)((unsigned long long)m << 32));
        else
            return __int_as_float(__float_as_int(v) ^ (int)m);
    }
    __device__ __forceinline__ void signs(const StageArgs &a, int k, W6<S> &w) const
    {
        if constexpr (W) {
            w.u0 = flip(w.u0, sx);
            w.u1 = flip(w.u1, sy);
            const bool fz = a.gmap && !a.flatz && axis_flip(k, a.nz, a.wall[4], a.wall[5]);
            w.u2 = flip(w.u2, fz ? 0x80000000u : 0u);
            no_minus_zero(w);
        }
    }
};

// flux_ang: a column's centre as the transform of the momenta takes it (with
// yoffset) and as the pressure projection does (without), for the column and
// its lower neighbours in x and y.
template <int V>
struct AngColumn {
    AngCentre at, lowx, lowy;  // projection (get_fluxes_ang: no yoffset)
    AngCentre tr;              // transform
    __device__ __forceinline__ AngColumn(const StageArgs &a, int x, int y)
    {
        if constexpr (has_ang(V)) {
            const double cx = centre(a.ds[0], x + 1, a.nx), cy = centre(a.ds[1], y + 1, a.ny);
            const double lx = centre(a.ds[0], x, a.nx), ly = centre(a.ds[1], y, a.ny), ty = cy + a.yoffset;
            at = {cx, cy, sqrt(cx * cx + cy * cy)};
            lowx = {lx, cy, sqrt(lx * lx + cy * cy)};
            lowy = {cx, ly, sqrt(cx * cx + ly * ly)};
            tr = {cx, ty, sqrt(cx * cx + ty * ty)};
        }
    }
    // the cell's r- and angular momentum; outside the finite slopes' range the
    // call goes to the cell-by-cell kernel
    template <typename S>
    __device__ __forceinline__ void momenta(const Raw<S> &v, W6<S> &w, unsigned int &flg) const
    {
        if constexpr (has_ang(V)) {
            tr.to(v.g1, v.g2, w.rm, w.am);
            if (!(fabs(w.rm) + fabs(w.am) <= 1e60)) flg |= FLAG_SLOW;
        }
    }
};

// the flux of a face for the cell above it (F) and, with flux_ang, the two
// momentum fluxes of the cell below it (G)
template <typename S, int dir, int V>
__device__ __forceinline__ void stage_face(const Side<S> &L, const Side<S> &R, const AngColumn<V> &col, S F[5], S G[2])
{
    if constexpr (has_ang(V)) face_flux_ang<dir>(L, R, col.at, dir == 0 ? col.lowx : col.lowy, F, G);
    else face_flux<S, dir>(L, R, F);
}

// Per-tile constants of one stage; col, row: the lane's place in the tile.
struct TileGeom {
    int nx, ny, nz;
    int64_t n, plane;
    int x0, j0, row, col;
    int edge;  // first owner row of an edge wave, else -1
    int kb, ke;
};

// The end of the flux subroutine at an interior cell (flux.f90:205-228): the
// stage update with fluxtmp ft and the floors.
template <int STAGE, int V>
__device__ __forceinline__ void flux_update(const StageArgs &a, double ui[5], double uo[5], const double ft[5],
                                            const W6<double> &q0, const AngColumn<V> &col, int64_t c, unsigned coff)
{
    double U[5];
    if constexpr (has_ang(V)) {
        ui[1] = q0.rm;
        ui[2] = q0.am;
        if (STAGE == 4) {
            double rm, am;
            col.tr.to(uo[1], uo[2], rm, am);
            uo[1] = rm;
            uo[2] = am;
        }
    }
    for (int i = 0; i < 5; i++) U[i] = STAGE == 3 ? ui[i] + ft[i] : 0.5 * (uo[i] + ui[i] + ft[i]);
    if constexpr (has_ang(V)) {
        double m1, m2;
        col.tr.back(U[1], U[2], m1, m2);
        U[1] = m1;
        U[2] = m2;
    }
    U[0] = floor_at(U[0], a.srho);
    if (U[4] < 0.0) U[4] = 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) / U[0] + a.seps;
    for (int i = 0; i < 5; i++) elem<double>(a.uout, (int64_t)i * a.n + c, coff) = U[i];
}

// Owner rows 0..TY-1: the register queue in z and the stage update.  The
// primitives of plane k are read back from the tile where needed, and the x
// and z flux differences are parked in LDS until the update, to keep the
// registers live across the barriers few.
template <int STAGE, typename S, int TY, int V, bool W, int WX>
__device__ __forceinline__ void tile_owner(const StageArgs &a, TileLds<S, TY, V, WX> &L, const TileGeom &g,
                                           unsigned int &flg, double &rmax)
{
    constexpr int RS = TileLds<S, TY, V, WX>::RS;
    const int col = g.col, row = g.row, nx = g.nx, ny = g.ny, nz = g.nz;
    const int64_t n = g.n;
    const int x = g.x0 + col, y = g.j0 + row;
    const Donor<S, W> me(a, x, y);
    const unsigned coff = me.off;
    const AngColumn<V> ang(a, min(x, nx - 1), min(y, ny - 1));
    const bool xy_ghost = x < 2 || x > nx - 3 || y < 2 || y > ny - 3;
    const bool is_out = !xy_ghost;
    const S gamS = S(a.gam);
    auto zplane = [&](int k) -> int64_t { return Donor<S, W>::plane(a, g.plane, k); };
    auto zghost = [&](int k) -> bool { return !a.flatz && (k < 2 || k > nz - 3); };
    const int c = (row + 2) * RS + col + 1;  // this cell in the primitive tiles
    const int o = row * WX + col;           // this cell's slot in the per-owner buffers

    W6<S> q2{};  // primitives of plane k+1 (k+2 after the z face of plane k)
    S cs0 = S(0), cs1 = S(0);
    Side<S> zp_prev{};
    S Fz_prev[5] = {S(0), S(0), S(0), S(0), S(0)};
    Raw<S> nxt;
    const int kb = g.kb, ke = g.ke;
    if (!a.flatz) {
        auto at = [&](int k) -> W6<S> {
            const Raw<S> v = load_raw<STAGE, S, V>(a, zplane(k), coff);
            W6<S> w = prims<STAGE, S, V>(a, v, flg);
            me.signs(a, k, w);
            ang.momenta(v, w, flg);
            return w;
        };
        const W6<S> t0 = at(kb - 2), t1 = at(kb - 1), t2 = at(kb), t3 = at(kb + 1);
        Side<S> zmi, zpl;
        dir_states<2, S, V>(t0, t1, t2, sound_at<V>(t1, a), xy_ghost || zghost(kb - 1), a, zmi, zpl);
        zp_prev = zpl;
        cs1 = sound_at<V>(t2, a);
        dir_states<2, S, V>(t1, t2, t3, cs1, xy_ghost || zghost(kb), a, zmi, zpl);
        S gz[2];
        stage_face<S, 2, V>(zp_prev, zmi, ang, Fz_prev, gz);
        zp_prev = zpl;
        store_w(L.P[kb & 1], c, t2);  // plane kb
        q2 = t3;
        nxt = load_raw<STAGE, S, V>(a, zplane(kb + 2), coff);
    } else {
        const Raw<S> v = load_raw<STAGE, S, V>(a, zplane(kb), coff);
        W6<S> w = prims<STAGE, S, V>(a, v, flg);
        me.signs(a, kb, w);
        ang.momenta(v, w, flg);
        cs1 = sound_at<V>(w, a);
        store_w(L.P[kb & 1], c, w);
        if (kb + 1 < ke) nxt = load_raw<STAGE, S, V>(a, zplane(kb + 1), coff);
    }
    __syncthreads();  // every row's primitives of plane kb are in the tile

    for (int k = kb; k < ke; k++) {
        const bool ghost_k = xy_ghost || zghost(k);
        const int t = k & 1;
        // A: the z face k+1/2 and the z flux difference of plane k; plane
        // k+1 into the other tile
        if (!a.flatz) {
            const W6<S> q1 = q2;
            cs0 = cs1;
            const Raw<S> cur = nxt;
            // plane k+3 (the last iteration reloads a plane, so that the queue
            // needs no branch)
            nxt = load_raw<STAGE, S, V>(a, zplane(min(k + 3, nz - 1)), coff);
            q2 = prims<STAGE, S, V>(a, cur, flg);
            me.signs(a, k + 2, q2);
            ang.momenta(cur, q2, flg);
            cs1 = sound_at<V>(q1, a);
            Side<S> zmi1, zpl1;
            dir_states<2, S, V>(fetch_w(L.P[t], c), q1, q2, cs1, xy_ghost || zghost(k + 1), a, zmi1, zpl1);
            S Fz1[5], gz[2];
            stage_face<S, 2, V>(zp_prev, zmi1, ang, Fz1, gz);
            for (int i = 0; i < 5; i++) {
                L.Dz[i][o] = (double)Fz1[i] - (double)Fz_prev[i];
                Fz_prev[i] = Fz1[i];
            }
            zp_prev = zpl1;
            if (k + 1 < ke) store_w(L.P[t ^ 1], c, q1);
        } else {
            cs0 = cs1;
            if (k + 1 < ke) {
                const Raw<S> cur = nxt;
                nxt = load_raw<STAGE, S, V>(a, zplane(min(k + 2, ke - 1)), coff);
                W6<S> w = prims<STAGE, S, V>(a, cur, flg);
                me.signs(a, k + 1, w);
                ang.momenta(cur, w, flg);
                cs1 = sound_at<V>(w, a);
                store_w(L.P[t ^ 1], c, w);
            }
        }
        // B (no barrier: plane k's tile was complete before the last one): x-states, x-faces and the x flux difference; y-states
        {
            const W6<S> q0 = fetch_w(L.P[t], c);
            Side<S> xmi, xpl;
            dir_states<0, S, V>(fetch_w(L.P[t], c - 1), q0, fetch_w(L.P[t], c + 1), cs0, ghost_k, a, xmi, xpl);
            Side<S> xl;
            xl.d = from_lower<WX>(xpl.d, L.SxL[0][row], col);
            xl.v[0] = from_lower<WX>(xpl.v[0], L.SxL[1][row], col);
            xl.v[1] = from_lower<WX>(xpl.v[1], L.SxL[2][row], col);
            xl.v[2] = from_lower<WX>(xpl.v[2], L.SxL[3][row], col);
            xl.p = from_lower<WX>(xpl.p, L.SxL[4][row], col);
            xl.e = from_lower<WX>(xpl.e, L.SxL[5][row], col);
            xl.g = gamS;
            constexpr int NF = TileLds<S, TY, V, WX>::NF;
            if constexpr (has_gamma(V)) xl.g = from_lower<WX>(xpl.g, L.SxL[6][row], col);
            if constexpr (has_ang(V)) {
                xl.s1 = from_lower<WX>(xpl.s1, L.SxL[NF - 2][row], col);
                xl.s2 = from_lower<WX>(xpl.s2, L.SxL[NF - 1][row], col);
            }
            S Fx0[5], gx[2];
            stage_face<S, 0, V>(xl, xmi, ang, Fx0, gx);  // face l-1/2
            for (int i = 0; i < 5; i++) {
                // face l+1/2, as this cell has it
                const S fx1 = from_upper<WX>(has_ang(V) && (i == 1 || i == 2) ? gx[i - 1] : Fx0[i], L.FxR[i][row], col);
                L.Dx[i][o] = (double)fx1 - (double)Fx0[i];
            }
        }
        Side<S> ymi;
        {
            Side<S> ypl;
            dir_states<1, S, V>(fetch_w(L.P[t], c - RS), fetch_w(L.P[t], c), fetch_w(L.P[t], c + RS), cs0, ghost_k, a,
                          ymi, ypl);
            store_side(L.Sy, (row + 1) * WX + col, ypl);
        }
        __syncthreads();
        // C: face y r-1/2, published over the y-plus state of row r-1
        S Fy0[5], gy[2];
        stage_face<S, 1, V>(fetch_side(L.Sy, row * WX + col, gamS), ymi, ang, Fy0, gy);
        for (int i = 0; i < 5; i++)  // as row r-1 has it
            L.Sy[i][row * WX + col] = has_ang(V) && (i == 1 || i == 2) ? gy[i - 1] : Fy0[i];
        // the update's loads go out before the barrier and run under it (coff is
        // a cell of the plane for every lane)
        const int64_t cz = (int64_t)k * g.plane;  // an interior plane
        S ri[5], ro[5];
        for (int i = 0; i < 5; i++) {
            ri[i] = elem<S>(a.uin, (int64_t)i * n + cz, coff);
            ro[i] = STAGE == 2 || STAGE == 4 ? elem<S>(a.uold, (int64_t)i * n + cz, coff) : S(0);
        }
        __syncthreads();
        // D: face y r+1/2 and the update
        if (is_out) {
            double ui[5], uo[5], sd[5], ft[5];
            for (int i = 0; i < 5; i++) {
                ui[i] = ri[i];
                uo[i] = ro[i];
            }
            for (int i = 0; i < 5; i++) {
                // flux.f90:188-190 in the reference's order, accumulated in FP64
                const S fy1 = L.Sy[i][(row + 1) * WX + col];
                const double ey = (double)(S)(a.axz * ((double)fy1 - (double)Fy0[i]));
                const double dz = a.flatz ? 0.0 : L.Dz[i][o];
                const double s = (a.ayz * L.Dx[i][o] + ey) + a.axy * dz;
                sd[i] = s * a.dt;
            }
            div_all<5>(sd, a.vol, a.inv_vol, a.vol_pow2, ft);
            for (int i = 0; i < 5; i++) ft[i] = -ft[i];
            if constexpr (STAGE >= 3) flux_update<STAGE, V>(a, ui, uo, ft, fetch_w(L.P[t], c), ang, cz, coff);
            else stage_update<STAGE, S, V == kGravity>(a, ui, uo, ft, fetch_w(L.P[t], c), cz, coff, flg, rmax);
        }
    }
}

// Halo rows -2, -1 and TY: their primitives, the y-states of rows -1 and TY,
// and face y TY-1/2.
template <int STAGE, typename S, int TY, int V, bool W, int WX>
__device__ __forceinline__ void tile_halo(const StageArgs &a, TileLds<S, TY, V, WX> &L, const TileGeom &g,
                                          unsigned int &flg)
{
    constexpr int RS = TileLds<S, TY, V, WX>::RS;
    const int col = g.col, row = g.row, nx = g.nx, ny = g.ny, nz = g.nz;
    const int x = g.x0 + col, y = g.j0 + row;
    const Donor<S, W> me(a, x, y);
    const unsigned coff = me.off;
    const AngColumn<V> ang(a, min(x, nx - 1), min(y, ny - 1));
    const bool xy_ghost = x < 2 || x > nx - 3 || y < 2 || y > ny - 3;
    const S gamS = S(a.gam);
    auto zplane = [&](int k) -> int64_t { return Donor<S, W>::plane(a, g.plane, k); };
    auto zghost = [&](int k) -> bool { return !a.flatz && (k < 2 || k > nz - 3); };
    const int c = (row + 2) * RS + col + 1;
    const int kb = g.kb, ke = g.ke;
    Raw<S> nxt;
    auto put = [&](int k, const Raw<S> &raw) {
        W6<S> w = prims<STAGE, S, V>(a, raw, flg);
        me.signs(a, k, w);
        ang.momenta(raw, w, flg);
        store_w(L.P[k & 1], c, w);
    };
    put(kb, load_raw<STAGE, S, V>(a, zplane(kb), coff));
    if (kb + 1 < ke) nxt = load_raw<STAGE, S, V>(a, zplane(kb + 1), coff);
    __syncthreads();  // as the owners' first barrier
    for (int k = kb; k < ke; k++) {
        const int t = k & 1;
        if (k + 1 < ke) {
            // A: primitives of plane k+1 into the other tile
            const Raw<S> cur = nxt;
            nxt = load_raw<STAGE, S, V>(a, zplane(min(k + 2, ke - 1)), coff);
            put(k + 1, cur);
        }
        Side<S> ymi;
        if (row == -1 || row == TY) {
            // B: y-states of plane k
            const W6<S> w = fetch_w(L.P[t], c);
            Side<S> ypl;
            dir_states<1, S, V>(fetch_w(L.P[t], c - RS), w, fetch_w(L.P[t], c + RS), sound_at<V>(w, a),
                          xy_ghost || zghost(k), a, ymi, ypl);
            if (row == -1) store_side(L.Sy, col, ypl);
        }
        __syncthreads();
        if (row == TY) {
            S F[5], gy[2];
            stage_face<S, 1, V>(fetch_side(L.Sy, TY * WX + col, gamS), ymi, ang, F, gy);
            for (int i = 0; i < 5; i++)
                L.Sy[i][TY * WX + col] = has_ang(V) && (i == 1 || i == 2) ? gy[i - 1] : F[i];
        }
        __syncthreads();
    }
}

// An edge wave: the x-edges of kEdgeRows owner rows one plane ahead (and with
// 64 columns its own halo row TY+1).  Lane 7*i+j holds column
// {-2,-1,0,WX-2,WX-1,WX,WX+1}[j] of owner row g.edge + i.
template <int STAGE, typename S, int TY, int V, bool W, int WX>
__device__ __forceinline__ void tile_edge(const StageArgs &a, TileLds<S, TY, V, WX> &L, const TileGeom &g,
                                          unsigned int &flg)
{
    constexpr int RS = TileLds<S, TY, V, WX>::RS;
    static_assert(7 * kEdgeRows <= 64 && (WX < 64 || TY <= kEdgeRows), "x-edge lanes of the owner rows");
    constexpr bool kHalo = WX == 64;
    const int lane = threadIdx.x & 63;
    const int col = g.col, row = g.row, nx = g.nx, ny = g.ny, nz = g.nz;
    const int x = g.x0 + col, y = g.j0 + row;
    const Donor<S, W> me(a, x, y);
    const unsigned coff = me.off;
    const AngColumn<V> ang(a, min(x, nx - 1), min(y, ny - 1));
    const S gamS = S(a.gam);
    auto zplane = [&](int k) -> int64_t { return Donor<S, W>::plane(a, g.plane, k); };
    auto zghost = [&](int k) -> bool { return !a.flatz && (k < 2 || k > nz - 3); };
    const int c = (row + 2) * RS + col + 1;

    const int er = lane / 7, ej = lane - 7 * er, erow = g.edge + er;
    const bool e_on = er < kEdgeRows && erow < TY;
    const int ecol = ej < 3 ? ej - 2 : ej + WX - 5;
    const int ex = g.x0 + ecol, ey = g.j0 + erow;
    const Donor<S, W> em(a, ex, ey);
    const AngColumn<V> eang(a, min(max(ex, 0), nx - 1), min(ey, ny - 1));
    const unsigned eoff = em.off;
    const bool e_xy_ghost = ex < 2 || ex > nx - 3 || ey < 2 || ey > ny - 3;

    // the three parts of the x-edge items of plane k
    W6<S> ew{};
    Side<S> emi{}, epl{};
    auto edge_prims = [&](int k, const Raw<S> &raw) {
        ew = prims<STAGE, S, V>(a, raw, flg);
        em.signs(a, k, ew);
        eang.momenta(raw, ew, flg);
        if (ej == 1 || ej == 5) store_w(L.P[k & 1], (erow + 2) * RS + ecol + 1, ew);
    };
    // neighbours within a row's seven lanes through whole-wave shifts (the
    // lanes whose neighbour lies in another row or outside the wave are not
    // used: columns -1, WX-1 and WX take columns -2..0 and WX-2..WX+1)
    auto edge_states = [&](int k) {
        dir_states<0, S, V>(lane_below_w(ew), ew, lane_above_w(ew), sound_at<V>(ew, a), e_xy_ghost || zghost(k), a, emi, epl);
    };
    auto edge_publish = [&]() {
        if (ej == 1) store_side(L.SxL, erow, epl);
        Side<S> xl;
        xl.d = lane_below(epl.d);
        xl.v[0] = lane_below(epl.v[0]);
        xl.v[1] = lane_below(epl.v[1]);
        xl.v[2] = lane_below(epl.v[2]);
        xl.p = lane_below(epl.p);
        xl.e = lane_below(epl.e);
        xl.g = gamS;
        if constexpr (has_gamma(V)) xl.g = lane_below(epl.g);
        if constexpr (has_ang(V)) {
            xl.s1 = lane_below(epl.s1);
            xl.s2 = lane_below(epl.s2);
        }
        if (ej == 5) {
            S F[5], gx[2];
            stage_face<S, 0, V>(xl, emi, eang, F, gx);  // face WX-1/2, as column WX-1 has it
            for (int i = 0; i < 5; i++) L.FxR[i][erow] = has_ang(V) && (i == 1 || i == 2) ? gx[i - 1] : F[i];
        }
    };

    const int kb = g.kb, ke = g.ke;
    Raw<S> nxt{};
    auto put = [&](int k, const Raw<S> &raw) {
        W6<S> w = prims<STAGE, S, V>(a, raw, flg);
        me.signs(a, k, w);
        ang.momenta(raw, w, flg);
        store_w(L.P[k & 1], c, w);
    };
    if (kHalo) {
        put(kb, load_raw<STAGE, S, V>(a, zplane(kb), coff));
        if (kb + 1 < ke) nxt = load_raw<STAGE, S, V>(a, zplane(kb + 1), coff);
    }
    Raw<S> enxt{};
    if (e_on) {
        edge_prims(kb, load_raw<STAGE, S, V>(a, zplane(kb), eoff));
        edge_states(kb);
        edge_publish();
        if (kb + 1 < ke) enxt = load_raw<STAGE, S, V>(a, zplane(kb + 1), eoff);
    }
    __syncthreads();  // as the owners' first barrier
    for (int k = kb; k < ke; k++) {
        const bool more = k + 1 < ke;
        if (more) {
            // A: primitives of plane k+1, its own row and the x-edges
            if (kHalo) {
                const Raw<S> cur = nxt;
                nxt = load_raw<STAGE, S, V>(a, zplane(min(k + 2, ke - 1)), coff);
                put(k + 1, cur);
            }
            if (e_on) {
                const Raw<S> ecur = enxt;
                enxt = load_raw<STAGE, S, V>(a, zplane(min(k + 2, ke - 1)), eoff);
                edge_prims(k + 1, ecur);
                edge_states(k + 1);  // B
            }
        }
        __syncthreads();
        if (e_on && more) edge_publish();  // C: the owners read plane k's in B
        __syncthreads();
    }
}

// One stage over the tile (bx, by) of WX x TY outputs and the z planes of chunk bz.
// V: StageKind.  W: some side is a wall (read only with gmap).
template <int STAGE, typename S, int TY, int V, bool W, int WX>
__device__ __forceinline__ void tile_stage(const StageArgs &a, TileLds<S, TY, V, WX> &L, unsigned bx, unsigned by,
                                           unsigned bz)
{
    constexpr int RPW = 64 / WX, kHalos = 2 / RPW, kOwners = TY / RPW;  // rows of a wave; waves of a halo; owner waves
    TileGeom g;
    g.nx = a.nx;
    g.ny = a.ny;
    g.nz = a.nz;
    g.n = a.n;
    g.plane = (int64_t)a.nx * a.ny;
    g.x0 = 2 + (int)bx * WX;
    g.j0 = 2 + (int)by * TY;
    // waves in order of their rows -2..TY+1, with 32 columns then the edge waves
    const int w = wave_id(), lane = threadIdx.x & 63;
    g.row = RPW * w - 2 + (RPW > 1 ? lane / WX : 0);
    g.col = lane & (WX - 1);
    g.edge = WX == 64 ? (w == TY + 3 ? 0 : -1) : (w >= kOwners + 2 * kHalos ? kEdgeRows * (w - kOwners - 2 * kHalos) : -1);
    g.kb = a.zlo + (int)bz * a.lz;
    g.ke = min(g.kb + a.lz, a.zhi);
    if (g.kb >= g.ke) return;  // uniform over the workgroup
    unsigned int flg = 0;
    double rmax = 0.0;
    if (w >= kHalos && w < kHalos + kOwners) {
        // The owner rows are the critical path between the barriers; each SIMD
        // holds two of them and one halo or edge wave, which is older and would
        // win the issue arbitration by age: the owners issue first
        // (2.06 -> 2.00 ms per step at 256^3).
        __builtin_amdgcn_s_setprio(1);
        tile_owner<STAGE, S, TY, V, W, WX>(a, L, g, flg, rmax);
    }
    else if (g.edge >= 0) tile_edge<STAGE, S, TY, V, W, WX>(a, L, g, flg);
    else tile_halo<STAGE, S, TY, V, W, WX>(a, L, g, flg);
    if (flg) atomicOr(a.flags, flg);
    if (STAGE == 2) wave_max_to(rmax, rate_slot(a, bx + by + bz + (unsigned)w));
}

// The two-level corner ghosts after the corrector's ghost fill.  The exact
// sequence leaves such a ghost holding +-(its interior cell v's corrector
// result before source(1)); that value reaches the results only through the
// next step's Courant rate (courant.f90:11-15 runs over every cell) and the
// stored state.  Three waves per ghost evaluate v's corrector update
// again from the corrector's inputs with the tiled kernel's operations (its
// six faces, flux.f90:121-190, and the update of flux.f90:213-228), park the
// result before source(1), write the ghost and give its Courant rate (the
// state and velocity of main.f90:232 and of the step's last velocity call,
// state.f90:30-57, velocity.f90:18-21).  The kernel is a serial chain of
// divisions and roots on a step's critical path: one wave takes each
// direction and one lane each of its two faces, so that a sixth of the faces
// lies on the chain (with one lane per ghost taking all six: 18.0 us).
//
// corner_prims: the primitives of the cell o cells from v along axis dir,
// ghosts as the tiles read them.
__device__ __forceinline__ W6<double> corner_prims(const StageArgs &a, int64_t v, int dir, int o, unsigned int &flg)
{
    const int64_t plane = (int64_t)a.nx * a.ny;
    const int x = (int)(v % a.nx) + (dir == 0 ? o : 0), y = (int)((v / a.nx) % a.ny) + (dir == 1 ? o : 0);
    const int z = (int)(v / plane) + (dir == 2 ? o : 0);
    const Donor<double, true> me(a, x, y);
    W6<double> w = load_prims<2, double>(a, Donor<double, true>::plane(a, plane, z), me.off, flg);
    me.signs(a, z, w);
    return w;
}

// corner_faces: wave d of the three, lane h: face h of direction d, between the
// cells h-1 and h from v, into F (then a barrier before corner_update)
__device__ __forceinline__ void corner_faces(const StageArgs &a, int j, int d, int h, double (*F)[2][5],
                                             unsigned int &flg)
{
    if (h >= 2) return;
    const int64_t v = a.d2cell[j];
    const int64_t plane = (int64_t)a.nx * a.ny;
    const int ix = (int)(v % a.nx), iy = (int)((v / a.nx) % a.ny), iz = (int)(v / plane);
    double f[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    auto face = [&](auto dirc) {
        constexpr int dir = decltype(dirc)::value;
        W6<double> w[4];
        for (int i = 0; i < 4; i++) w[i] = corner_prims(a, v, dir, h - 2 + i, flg);
        Side<double> mi[2], pl[2];
        for (int i = 0; i < 2; i++) {
            const int o = h - 1 + i;
            const int x = ix + (dir == 0 ? o : 0), y = iy + (dir == 1 ? o : 0), z = iz + (dir == 2 ? o : 0);
            const bool gh = x < 2 || x > a.nx - 3 || y < 2 || y > a.ny - 3 || (!a.flatz && (z < 2 || z > a.nz - 3));
            dir_states<dir>(w[i], w[i + 1], w[i + 2], sound_of(w[i + 1], a.gam), gh, a, mi[i], pl[i]);
        }
        face_flux<double, dir>(pl[0], mi[1], f);
    };
    if (d == 0) face(std::integral_constant<int, 0>{});
    else if (d == 1) face(std::integral_constant<int, 1>{});
    else if (!a.flatz) face(std::integral_constant<int, 2>{});
    for (int i = 0; i < 5; i++) F[d][h][i] = f[i];
}

// corner_update: one lane, once F is complete; returns the ghost's Courant rate
__device__ __forceinline__ double corner_update(const StageArgs &a, int j, const double (*F)[2][5], int64_t gcell,
                                                int sg, unsigned int &flg)
{
    const int64_t v = a.d2cell[j];
    const W6<double> q0 = corner_prims(a, v, 0, 0, flg);
    double ui[5], uo[5], ft[5];
    for (int i = 0; i < 5; i++) {
        ui[i] = elem<double>(a.uin, (int64_t)i * a.n + v, 0u);
        uo[i] = elem<double>(a.uold, (int64_t)i * a.n + v, 0u);
        const double dx = F[0][1][i] - F[0][0][i];
        const double ey = a.axz * (F[1][1][i] - F[1][0][i]);
        const double dz = a.flatz ? 0.0 : F[2][1][i] - F[2][0][i];
        const double sm = (a.ayz * dx + ey) + a.axy * dz;
        ft[i] = -div_by(sm * a.dt, a.vol, a.inv_vol, a.vol_pow2);
    }
    double rv = 0.0;
    // rewrites U^{n+1} of v with the bits the tiled kernel wrote and parks
    // the result before source(1) in d2ubar (with gravity also p of v)
    if (a.gf) stage_update<2, double, true>(a, ui, uo, ft, q0, v, 0u, flg, rv, true);
    else stage_update<2, double>(a, ui, uo, ft, q0, v, 0u, flg, rv, true);
    double U[5];
    for (int i = 0; i < 5; i++) U[i] = a.d2ubar[6 * j + i];
    // the pressure the exact sequence leaves in the ghost: the state call
    // after the last ghost pair (main.f90:511-513) takes the velocity of
    // the previous velocity call, when the ghost held h2's value from
    // before the third pair, 0.5*(cons_old + U* + 0) of v up to signs
    // (flux.f90:213, cons_old = U^n after source(0), which leaves rho as
    // it is and, without gravity, m too; with gravity m is kicked by v's
    // force); the signs drop out of |u|^2
    {
        double rc = 0.5 * ((uo[0] + ui[0]) + 0.0);
        rc = vmax(rc, a.srho);
        double mo[3] = {uo[1], uo[2], uo[3]};
        if (a.gf) {
            const double g[3] = {a.gf[v], a.gf[a.n + v], a.gf[2 * a.n + v]};
            const double m[3] = {uo[1], uo[2], uo[3]};
            grav_momenta(uo[0], m, g, a.dt * 0.5, mo);
        }
        double uc[3];
        for (int d = 0; d < 3; d++) uc[d] = (0.5 * ((mo[d] + ui[1 + d]) + 0.0)) / rc;
        const double ek = U[0] * 0.5 * (uc[0] * uc[0] + uc[1] * uc[1] + uc[2] * uc[2]);
        a.d2ubar[6 * j + 5] = vmax(U[4] - ek, a.seps) * a.gm1;
    }
    for (int f = 1; f <= 3; f++)
        if ((sg >> (f - 1)) & 1) U[f] = -U[f];
    double *un = (double *)a.uout;
    for (int i = 0; i < 5; i++) un[(int64_t)i * a.n + gcell] = U[i];
    const double v0 = U[1] / U[0], v1 = U[2] / U[0], v2 = U[3] / U[0];
    const double ekin = U[0] * 0.5 * (v0 * v0 + v1 * v1 + v2 * v2);
    const double p = vmax(U[4] - ekin, a.seps) * a.gm1;
    const double snd = sqrt(a.gam * p / U[0]);
    return div_by(snd + fabs(v0), a.ds[0], a.inv_ds[0], a.ds_pow2[0]) +
         div_by(snd + fabs(v1), a.ds[1], a.inv_ds[1], a.ds_pow2[1]) +
         div_by(snd + fabs(v2), a.ds[2], a.inv_ds[2], a.ds_pow2[2]);
}

// one corner ghost by a workgroup of at least three waves
__device__ __forceinline__ void corner_block(const StageArgs &a, int j, double (*F)[2][5])
{
    const int d = wave_id();
    double rt = 0.0;
    unsigned int flg = 0;
    if (d < 3) corner_faces(a, j, d, threadIdx.x & 63, F, flg);
    __syncthreads();
    if (threadIdx.x == 0) rt = corner_update(a, j, F, a.d2dst[j], a.d2sign[j], flg);
    if (flg) atomicOr(a.flags, flg);
    if (d == 0) wave_max_to(rt, rate_slot(a, (unsigned)j));
}

}  // namespace bx
