// ads_el_tile.h -- several time levels of the elastic forward scheme per launch.
//
// A workgroup takes one tile of one shot: a core and a halo of 4 cells per level around it.  The
// fields of the whole extent live in registers: a lane holds one column, a wavefront R consecutive
// rows.  The y neighbours come from the adjacent lanes (DPP moves), the x neighbours from the lane's
// own rows and, within two rows of a wavefront's edge, through LDS.  A level is two phases (stress and
// velocity), each of which reads two cells to either side, so what is wrong beyond the extent moves
// inward 4 cells a level and never reaches the core.  Only core cells are stored.  Sources are added
// inside the tile.
//
// Included by ads_elastic.hip after its state and coefficient types.
#pragma once

#include "ads_tile.h"

namespace ads {

constexpr int ET_NW = 8;  // wavefronts per workgroup

// What a tile's extent holds: cells inside the identity rectangle only; any rows but only its columns
// (x profile); any columns but only its rows (y profile); anything.
enum { ET_PLAIN = 0, ET_X = 1, ET_Y = 2, ET_XY = 3 };

// Point lists of (shot, tile, wavefront): groups of one register row and field type, their cells in
// column order.  key.x = column in the extent | core << 8, key.y = the plan's number of the unique
// (cell, type), whose entries are ent[eptr[key.y]] .. of the shot.
struct ElPoints {
    const int32_t *ptr;
    const int4 *grp;  // row | type << 8, first key, end key
    const int2 *key;
    const int64_t *eptr, *ent;
};

template <typename T> struct ElFwdTile {
    const int4 *tiles;  // two per tile: core (i0, i1, j0, j1); extent (ie, je, rows | columns << 16, kind)
    int ntiles, nb, act;
    int n, nt;  // levels n .. n + nt - 1
    ElCoef<T> c;
    // states: field q of level l, shot s at u + (l mod NS) ls + q fs + s ss; memory variables
    // likewise from m, outside the box mb (full grid: mb.H == 0)
    T *u, *m;
    int64_t ls, fs, ss, mls, mfs, mss;
    int NS;
    FrameBox mb;
    const int64_t *nstep;
    ElPoints src;
    T *pre;  // stresses before injection, one per key and slot (stride pls); may be null
    int64_t pls;
    const T *rho, *lam, *mu;
    // full-grid memory variables: read from m, written after the launch's last level to mo
    T *mo;
    const T *srcv;
    const int64_t *srcv_off, *nsrc;
};
__device__ inline void recompute(uint32_t &v) { asm volatile("" : "+v"(v)); }
// a wave-uniform value that the compiler takes for a new one at each use (see recompute)
__device__ inline int opaque(int v)
{
    uint32_t x = (uint32_t)v;
    recompute(x);
    return __builtin_amdgcn_readfirstlane((int)x);
}

// A tile as one wavefront sees it.
template <int R> struct ElView {
    int i0, i1, j0, j1, lane, w, r0, last, j, jc;
    uint32_t core, rA, rB;  // rows of the core; rows of the update ranges' parts A and B
    FwPart fc;              // this column's
    bool own;               // a core column
    __device__ inline ElView(const int4 c, const int4 e, int NX, int NY, int sub)
    {
        i0 = c.x, i1 = c.y, j0 = c.z, j1 = c.w;
        lane = threadIdx.x % WAVE, w = wave_id();
        const int ne = e.z & 0xffff, ce = e.z >> 16;
        r0 = e.x + w * R;
        last = e.x + ne - 1;
        j = e.y + lane;
        jc = e.y + min(lane, ce - 1);
        own = j >= j0 && j < j1;
        core = row_mask<R>(r0, i0, i1);
        if (sub) {
            rA = rB = row_mask<R>(r0, 2, NX);
            fc.A = fc.B = j >= 2 && j <= NY - 1;
        } else {
            rA = row_mask<R>(r0, 1, NX);
            rB = row_mask<R>(r0, 2, NX + 1);
            fc.A = j >= 2 && j <= NY;
            fc.B = j >= 1 && j <= NY - 1;
        }
    }
};

template <typename T> struct ElLds {
    T row[4][3][ET_NW][WAVE];  // vx, vy, sxx, sxy: three rows per wavefront
    T plane[ET_NW][WAVE];
};
// Rows around a wavefront's own: `lo` rows above and 3 - lo below of one field, from the neighbouring
// wavefronts (beyond the tile: any value).
template <int LO, typename T, int R>
__device__ inline void put_rows(T (&l)[3][ET_NW][WAVE], const T (&f)[R], int w, int lane)
{
    // the wavefront below reads the last LO rows, the one above the first 3 - LO
#pragma unroll
    for (int k = 0; k < LO; k++) l[k][w][lane] = f[R - LO + k];
#pragma unroll
    for (int k = 0; k < 3 - LO; k++) l[LO + k][w][lane] = f[k];
}
template <int LO, typename T>
__device__ inline void get_rows(const T (&l)[3][ET_NW][WAVE], T (&h)[3], int w, int lane)
{
    const int wu = max(w - 1, 0), wd = min(w + 1, ET_NW - 1);
#pragma unroll
    for (int k = 0; k < LO; k++) h[k] = l[k][wu][lane];
#pragma unroll
    for (int k = LO; k < 3; k++) h[k] = l[k][wd][lane];
}
// row r of a field with its neighbour rows: r in [-LO, R + 3 - LO)
template <int LO, typename T, int R> __device__ inline T at_row(const T (&f)[R], const T (&h)[3], int r)
{
    return r < 0 ? h[r + LO < 0 ? 0 : r + LO] : (r >= R ? h[LO + r - R > 2 ? 2 : LO + r - R] : f[r]);
}

// Applies the wavefront's point groups: f(row, type, hit value of this column) with uniform row and type.
// val(key) gives a key's value; the columns without a key get 0 and hit = false.
struct ElGroups {
    int lo, hi;
    __device__ inline ElGroups(const ElPoints &p, int64_t at)
        : lo(__builtin_amdgcn_readfirstlane(p.ptr[at])), hi(__builtin_amdgcn_readfirstlane(p.ptr[at + 1]))
    {
    }
};
template <typename T, typename V, typename F>
__device__ inline void el_points(const ElPoints &p, const ElGroups &gs, int lane, T *plane, V &&val, F &&f)
{
    for (int g = gs.lo; g < gs.hi; g++) {
        const int4 q = p.grp[g];
        const int k = q.y + lane;
        const bool has = k < q.z;
        const int2 key = has ? p.key[k] : make_int2(0, -1);
        const T v = has ? val(key) : T(0);
        plane[lane] = T(0);
        __builtin_amdgcn_wave_barrier();
        if (has) plane[key.x & 63] = v;
        __builtin_amdgcn_wave_barrier();
        const T add = plane[lane];
        __builtin_amdgcn_wave_barrier();
        f(__builtin_amdgcn_readfirstlane(q.x & 0xff), __builtin_amdgcn_readfirstlane(q.x >> 8), add, key, has);
    }
}

// ---------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------
template <typename T, int SUB, int R, int KIND>
__device__ inline void el_fwd_tile_body(const ElFwdTile<T> &a, const int4 c4, const int4 e4, int s, int tile, int nt,
                                        ElLds<T> &lds)
{
    constexpr bool XM = KIND == ET_X || KIND == ET_XY, YM = KIND == ET_Y || KIND == ET_XY, GEN = KIND != ET_PLAIN;
    const ElCoef<T> &c = a.c;
    const ElView<R> t(c4, e4, c.NX, c.NY, SUB);
    const int lane = t.lane, w = t.w;
    const T dt = c.dt, ihx = c.ihx, ihy = c.ihy;
    const uint32_t pb = (uint32_t)c.P * (uint32_t)sizeof(T);
    const uint32_t jcb = (uint32_t)t.jc * (uint32_t)sizeof(T);
    uint32_t ro[R];  // byte offset of the lane's cell in each row, clamped to the extent
#pragma unroll
    for (int r = 0; r < R; r++) ro[r] = (uint32_t)min(t.r0 + r, t.last) * pb + jcb;
    int slot = a.n % a.NS;
    const int sl = slot >= 1 ? slot - 1 : a.NS - 1;
    const T *__restrict__ ui = a.u + (int64_t)sl * a.ls + (int64_t)s * a.ss;
    T X[R], Y[R], XX[R], YY[R], XY[R], LA[R + 1], MU[R + 1], RH[R + 1];
#pragma unroll
    for (int r = 0; r < R; r++) {
        X[r] = *at_off(ui + VX * a.fs, ro[r]);
        Y[r] = *at_off(ui + VY * a.fs, ro[r]);
        XX[r] = *at_off(ui + SXX * a.fs, ro[r]);
        YY[r] = *at_off(ui + SYY * a.fs, ro[r]);
        XY[r] = *at_off(ui + SXY * a.fs, ro[r]);
    }
#pragma unroll
    for (int r = 0; r <= R; r++) {
        const uint32_t o = (uint32_t)min(t.r0 + r, c.NX + 1) * pb;
        LA[r] = *at_off(at_off(a.lam, o), jcb);
        MU[r] = *at_off(at_off(a.mu, o), jcb);
        RH[r] = *at_off(at_off(a.rho, o), jcb);
    }
    // memory variables: m1, m3, m5, m7 of the x profile, m2, m4, m6, m8 of the y profile
    T mx[XM ? 4 : 1][XM ? R : 1] = {}, my[YM ? 4 : 1][YM ? R : 1] = {};
    const MvCol mc = mv_col(a.mb, t.jc);
    auto mvi = [&](int i) -> int { return a.mb.H ? mv_at(a.mb, mc, i) : i * c.P + t.jc; };
    if constexpr (GEN) {
        const T *__restrict__ mi = a.m + (int64_t)(a.mo ? 0 : sl) * a.mls + (int64_t)s * a.mss;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int o = mvi(min(t.r0 + r, t.last));
            if (o >= 0) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if constexpr (XM) mx[k][r] = mi[(2 * k) * a.mfs + o];
                    if constexpr (YM) my[k][r] = mi[(2 * k + 1) * a.mfs + o];
                }
            }
        }
    }
    const ProfRow<T> py = YM ? prof_col(c, t.jc) : ProfRow<T>{};
    const int64_t ns = a.nsrc[s];
    const ElGroups sg(a.src, ((int64_t)s * a.ntiles + tile) * ET_NW + w);
    const T *__restrict__ srow = a.srcv + a.srcv_off[s] + (int64_t)(a.n - 1) * ns;
    for (int q = 0; q < nt; q++) {
#pragma unroll
        for (int r = 0; r <= R; r++) {
            recompute(LA[r]);
            recompute(MU[r]);
            recompute(RH[r]);
        }
        // (profiles and row masks are formed at each level, or they fill the scalar registers)
        const int r0 = opaque(t.r0);
        const uint32_t rA = (uint32_t)opaque((int)t.rA), rB = (uint32_t)opaque((int)t.rB);
        put_rows<1>(lds.row[0], X, w, lane);
        put_rows<2>(lds.row[1], Y, w, lane);
        __syncthreads();
        T hx[3], hy[3];
        get_rows<1>(lds.row[0], hx, w, lane);
        get_rows<2>(lds.row[1], hy, w, lane);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const ProfRow<T> px = XM ? prof_row(c, min(r0 + r, t.last)) : ProfRow<T>{};
            const T x = X[r], y = Y[r];
            const T vym = lane_west(y), vyp = lane_east(y), vymm = lane_west(vym);
            const T vxm = lane_west(x), vxp = lane_east(x), vxpp = lane_east(vxp);
            const T mue = lane_east(MU[r]);
            if (!GEN || ((rA >> r & 1) && t.fc.A)) {
                const T lb = SUB ? LA[r] : T(0.5) * (LA[r + 1] + LA[r]);
                const T mb = SUB ? MU[r] : T(0.5) * (MU[r + 1] + MU[r]);
                const T lm = lb + T(2) * mb;
                T dx = (T(27) * at_row<1>(X, hx, r + 1) - T(27) * x - at_row<1>(X, hx, r + 2) + at_row<1>(X, hx, r - 1)) * ihx;
                T dy = (T(27) * y - T(27) * vym - vyp + vymm) * ihy;
                if constexpr (XM) {
                    mx[0][r] = px.bh * mx[0][r] + px.ah * dx;
                    dx += mx[0][r];
                }
                if constexpr (YM) {
                    my[0][r] = py.bf * my[0][r] + py.af * dy;
                    dy += my[0][r];
                }
                XX[r] += (lm * dx + lb * dy) * dt;
                YY[r] += (lm * dy + lb * dx) * dt;
            }
            if (!GEN || ((rB >> r & 1) && t.fc.B)) {
                const T mb = SUB ? MU[r] : T(0.5) * (MU[r] + mue);
                T dx = (T(27) * y - T(27) * at_row<2>(Y, hy, r - 1) - at_row<2>(Y, hy, r + 1) + at_row<2>(Y, hy, r - 2)) * ihx;
                T dy = (T(27) * vxp - T(27) * x - vxpp + vxm) * ihy;
                if constexpr (XM) {
                    mx[1][r] = px.bf * mx[1][r] + px.af * dx;
                    dx += mx[1][r];
                }
                if constexpr (YM) {
                    my[1][r] = py.bh * my[1][r] + py.ah * dy;
                    dy += my[1][r];
                }
                XY[r] += mb * (dx + dy) * dt;
            }
        }
        put_rows<2>(lds.row[2], XX, w, lane);
        put_rows<1>(lds.row[3], XY, w, lane);
        __syncthreads();
        get_rows<2>(lds.row[2], hx, w, lane);
        get_rows<1>(lds.row[3], hy, w, lane);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const ProfRow<T> px = XM ? prof_row(c, min(r0 + r, t.last)) : ProfRow<T>{};
            const T b = XY[r], g = YY[r];
            const T xym = lane_west(b), xyp = lane_east(b), xymm = lane_west(xym);
            const T yym = lane_west(g), yyp = lane_east(g), yypp = lane_east(yyp);
            const T re0 = lane_east(RH[r]), re1 = lane_east(RH[r + 1]);
            if (!GEN || ((rB >> r & 1) && t.fc.A)) {
                T dx = (T(27) * XX[r] - T(27) * at_row<2>(XX, hx, r - 1) - at_row<2>(XX, hx, r + 1) + at_row<2>(XX, hx, r - 2)) * ihx;
                T dy = (T(27) * b - T(27) * xym - xyp + xymm) * ihy;
                if constexpr (XM) {
                    mx[2][r] = px.bf * mx[2][r] + px.af * dx;
                    dx += mx[2][r];
                }
                if constexpr (YM) {
                    my[2][r] = py.bf * my[2][r] + py.af * dy;
                    dy += my[2][r];
                }
                X[r] += (dx + dy) * dt / RH[r];
            }
            if (!GEN || ((rA >> r & 1) && t.fc.B)) {
                const T rb = SUB ? RH[r] : T(0.25) * (RH[r] + RH[r + 1] + re1 + re0);
                T dx = (T(27) * at_row<1>(XY, hy, r + 1) - T(27) * b - at_row<1>(XY, hy, r + 2) + at_row<1>(XY, hy, r - 1)) * ihx;
                T dy = (T(27) * yyp - T(27) * g - yypp + yym) * ihy;
                if constexpr (XM) {
                    mx[3][r] = px.bh * mx[3][r] + px.ah * dx;
                    dx += mx[3][r];
                }
                if constexpr (YM) {
                    my[3][r] = py.bh * my[3][r] + py.ah * dy;
                    dy += my[3][r];
                }
                Y[r] += (dx + dy) * dt / rb;
            }
        }
        // sources, added to the finished level (the velocity update reads the stresses before them)
        T *__restrict__ pre = a.pre ? a.pre + (int64_t)slot * a.pls : nullptr;
        if (a.n + q <= a.nstep[s])
            el_points<T>(
                a.src, sg, lane, lds.plane[w],
                [&](int2 key) {
                    T v = T(0);
                    for (int64_t e = a.src.eptr[key.y]; e < a.src.eptr[key.y + 1]; e++) v += srow[a.src.ent[e]];
                    return v;
                },
                [&](int row, int type, T add, int2 key, bool has) {
                    T old = T(0);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const bool at_r = r == row;  // uniform
                        old = at_r ? (type == SXX ? XX[r] : type == SYY ? YY[r] : XY[r]) : old;
                        X[r] += at_r && type == VX ? add : T(0);
                        Y[r] += at_r && type == VY ? add : T(0);
                        XX[r] += at_r && type == SXX ? add : T(0);
                        YY[r] += at_r && type == SYY ? add : T(0);
                        XY[r] += at_r && type == SXY ? add : T(0);
                    }
                    if (pre && type >= SXX) {
                        lds.plane[w][lane] = old;
                        __builtin_amdgcn_wave_barrier();
                        if (has && (key.x >> 8)) pre[key.y] = lds.plane[w][key.x & 63];
                        __builtin_amdgcn_wave_barrier();
                    }
                });
        srow += ns;
        T *__restrict__ uo = a.u + (int64_t)slot * a.ls + (int64_t)s * a.ss;
        if (t.own) {
#pragma unroll
            for (int r = 0; r < R; r++)
                if (t.core >> r & 1) {
                    *at_off(uo + VX * a.fs, ro[r]) = X[r];
                    *at_off(uo + VY * a.fs, ro[r]) = Y[r];
                    *at_off(uo + SXX * a.fs, ro[r]) = XX[r];
                    *at_off(uo + SYY * a.fs, ro[r]) = YY[r];
                    *at_off(uo + SXY * a.fs, ro[r]) = XY[r];
                }
            if constexpr (GEN) {
                if (!a.mo || q == nt - 1) {
                    T *__restrict__ mo = (a.mo ? a.mo : a.m + (int64_t)slot * a.mls) + (int64_t)s * a.mss;
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const int o = t.core >> r & 1 ? mvi(t.r0 + r) : -1;
                        if (o >= 0) {
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                mo[(2 * k) * a.mfs + o] = XM ? mx[XM ? k : 0][XM ? r : 0] : T(0);
                                mo[(2 * k + 1) * a.mfs + o] = YM ? my[YM ? k : 0][YM ? r : 0] : T(0);
                            }
                        }
                    }
                }
            }
        }
        slot = slot + 1 == a.NS ? 0 : slot + 1;
    }
}
// Bound by latency on small grids (two barriers, one round of loads and of stores per launch, two
// wavefronts per SIMD), by the vector units on large ones: 56 % of a launch's cells are halo at two
// levels.  4 rows per wavefront hold an FP64 cell's 5 fields, 3 parameters and 8 memory variables in
// 220 registers; 6 rows spill (134 x 97, 4 shots: 19.2 against 11.3 us per level), 2 rows leave no
// core at two levels.  The same tiles in the adjoint (both phases in one launch, 15 inputs a cell)
// were slower than its streaming kernels nearly everywhere (600 x 600, 16 shots, FP32: 314 against 190
// us per level) and are not kept.
template <typename T, int SUB, int R>
__global__ __launch_bounds__(WAVE *ET_NW) void el_fwd_tile(const ElFwdTile<T> a)
{
    __shared__ __align__(16) ElLds<T> lds;
    TileMap m{a.ntiles, a.act, 1, a.nb};
    int z, s, tile;
    if (!decode_tile(m, z, s, tile, (int)blockIdx.x)) return;  // workgroup-uniform
    const int4 c = a.tiles[2 * tile], e = a.tiles[2 * tile + 1];
    const int nt = a.mo ? a.nt : min(a.nt, (int)a.nstep[s] - a.n + 1);
    if (e.w == ET_PLAIN) el_fwd_tile_body<T, SUB, R, ET_PLAIN>(a, c, e, s, tile, nt, lds);
    else if (e.w == ET_X) el_fwd_tile_body<T, SUB, R, ET_X>(a, c, e, s, tile, nt, lds);
    else if (e.w == ET_Y) el_fwd_tile_body<T, SUB, R, ET_Y>(a, c, e, s, tile, nt, lds);
    else el_fwd_tile_body<T, SUB, R, ET_XY>(a, c, e, s, tile, nt, lds);
}

// Traces of levels lo + 1 .. hi from their slots: 8 receivers by 32 levels per workgroup.
template <typename T>
__global__ __launch_bounds__(256) void el_record(const T *__restrict__ u, int64_t ls, int64_t fs, int64_t ss, int NS, int lo,
                                                 int hi, const int64_t *__restrict__ rcv_ptr,
                                                 const int64_t *__restrict__ rcv_key, const int64_t *__restrict__ nstep,
                                                 T *__restrict__ traces, const int64_t *__restrict__ trace_off)
{
    const int s = blockIdx.z, n = lo + 1 + (int)blockIdx.y * 32 + (int)(threadIdx.x & 31);
    const int64_t r = (int64_t)blockIdx.x * 8 + threadIdx.x / 32;
    if (n > hi || n > nstep[s] || r >= rcv_ptr[s + 1] - rcv_ptr[s]) return;
    const int64_t key = rcv_key[rcv_ptr[s] + r];
    traces[trace_off[s] + r * (nstep[s] + 1) + n] = u[(int64_t)(n % NS) * ls + (key & 7) * fs + (int64_t)s * ss + (key >> 3)];
}

// ---------------------------------------------------------------------------------------------
// tiles and point lists (host)
// ---------------------------------------------------------------------------------------------
struct ElTileHost {
    int i0, i1, j0, j1, ie, je, ne, ce, kind;
};
// The tiles of the padded grid for launches of `levels` levels, `rows` rows each; R: the rectangle in which the CPML is the
// identity and every update range holds.
static inline std::vector<ElTileHost> el_tiles(int NX, int NY, int levels, int rows, const Rect &R)
{
    std::vector<ElTileHost> out;
    const int H = 4 * levels;
    const std::vector<int> ci = tile_cuts(0, NX + 2, H, NX + 2, rows), cj = tile_cuts(0, NY + 2, H, NY + 2, WAVE);
    for (size_t p = 0; p + 1 < ci.size(); p++)
        for (size_t q = 0; q + 1 < cj.size(); q++) {
            ElTileHost t{ci[p], ci[p + 1], cj[q], cj[q + 1], 0, 0, 0, 0, 0};
            t.ie = std::max(t.i0 - H, 0);
            t.je = std::max(t.j0 - H, 0);
            t.ne = std::min(t.i1 + H, NX + 2) - t.ie;
            t.ce = std::min(t.j1 + H, NY + 2) - t.je;
            const bool px = t.ie >= R.iL && t.ie + t.ne <= R.iR, py = t.je >= R.jL && t.je + t.ce <= R.jR;
            t.kind = px ? (py ? ET_PLAIN : ET_Y) : (py ? ET_X : ET_XY);
            out.push_back(t);
        }
    return out;
}
// Point lists (ElPoints) of unique keys key[c] = (i * P + j) * 8 + type, c in [ptr[s], ptr[s + 1]) of shot s.
struct ElPointLists {
    std::vector<int32_t> ptr;
    std::vector<int4> grp;
    std::vector<int2> key;
};
static inline ElPointLists el_point_lists(const std::vector<ElTileHost> &tiles, int rowsw, int64_t P,
                                          const std::vector<int64_t> &ptr, const std::vector<int64_t> &key)
{
    // row and column ranges of the tiles are a product: the tiles of a cell are found through the
    // distinct row and column bands
    std::vector<int> rows, cols;  // first tile of each band of rows; of each band of columns
    for (size_t q = 0; q < tiles.size(); q++) {
        if (tiles[q].j0 == tiles[0].j0) rows.push_back((int)q);
        if (tiles[q].i0 == tiles[0].i0) cols.push_back((int)q);
    }
    struct Ent {
        uint64_t at;  // tile, wavefront, row, type, column
        int32_t c, own;
    };
    ElPointLists o;
    const size_t nt = tiles.size(), ns = ptr.size() - 1;
    o.ptr.assign(ns * nt * ET_NW + 1, 0);
    std::vector<Ent> es;
    for (size_t s = 0; s < ns; s++) {
        es.clear();
        for (int64_t c = ptr[s]; c < ptr[s + 1]; c++) {
            const int type = (int)(key[c] & 7), i = (int)((key[c] >> 3) / P), j = (int)((key[c] >> 3) % P);
            for (int rq : rows) {
                const ElTileHost &a = tiles[rq];
                if (i < a.ie || i >= a.ie + a.ne) continue;
                for (int cq : cols) {
                    const size_t q = (size_t)rq + cq;
                    const ElTileHost &t = tiles[q];
                    if (j < t.je || j >= t.je + t.ce) continue;
                    const int r = i - t.ie, own = i >= t.i0 && i < t.i1 && j >= t.j0 && j < t.j1;
                    es.push_back(Ent{((((uint64_t)q * ET_NW + r / rowsw) << 8 | (uint64_t)(r % rowsw)) << 8 | (uint64_t)type) << 8 |
                                         (uint64_t)(j - t.je),
                                     (int32_t)c, own});
                }
            }
        }
        std::sort(es.begin(), es.end(), [](const Ent &x, const Ent &y) { return x.at < y.at; });
        size_t e = 0;
        for (size_t q = 0; q < nt * ET_NW; q++) {
            o.ptr[s * nt * ET_NW + q] = (int32_t)o.grp.size();
            for (; e < es.size() && es[e].at >> 24 == q; e++) {
                if (e == 0 || es[e].at >> 8 != es[e - 1].at >> 8)
                    o.grp.push_back(make_int4((int)(es[e].at >> 16 & 0xff) | (int)(es[e].at >> 8 & 0xff) << 8,
                                              (int)o.key.size(), (int)o.key.size(), 0));
                o.key.push_back(make_int2((int)(es[e].at & 0xff) | es[e].own << 8, es[e].c));
                o.grp.back().z = (int)o.key.size();
            }
        }
    }
    o.ptr[ns * nt * ET_NW] = (int32_t)o.grp.size();
    if (o.grp.empty()) o.grp.push_back(make_int4(0, 0, 0, 0));
    if (o.key.empty()) o.key.push_back(make_int2(0, 0));
    return o;
}

}  // namespace ads
