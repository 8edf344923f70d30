// ads_ac_tile.h -- several time levels of the acoustic scheme per launch, forward and adjoint.
//
// A workgroup takes one tile of one shot: the tile's core and a halo around it wide enough for the
// launch's levels.  The state of the whole extent lives in registers for all of them: a lane holds
// one column, a wavefront R consecutive rows.  The j neighbours come from the adjacent lanes (DPP
// moves), the i neighbours from the lane's own rows and, at a wavefront's first and last row,
// through LDS (two rows per wavefront and field, double-buffered: one barrier per level).  Cells of
// the halo are stepped too; what they read beyond the extent is wrong, and that error moves inward
// one cell per level (two where kernel 0's phi/psi follow the new u), so it never reaches the core.
// Only core cells are stored.  Every value is the single-level expression in the same order, so the
// wavefields equal single-level stepping bit for bit.
#pragma once

#include "ads_common.h"
#include "ads_stencil.h"
#include "ads_tile.h"

namespace ads {

// Point lists of (shot, tile): the distinct source (or interior receiver) cells inside the tile's
// extent, sorted by row and column.  ptr[shot * ntiles + tile] indexes cell; cell[q] is (row << 8 |
// column within the extent, first entry), its entries end where the next cell's begin; ent holds
// the source (receiver) numbers within the shot, in their order.
struct PointList {
    const int32_t *ptr;
    const int2 *cell;
    const int32_t *ent;
};

// What the forward and the adjoint tile kernels share.
template <typename T> struct TileCommon {
    const int4 *tiles;  // two per tile: core (i0, i1, j0, j1); extent (ie, je, rows | columns << 16, kind)
    int ntiles, nb, act, NX, NY, P;
    AcCoef<T> k;
    const T *C, *sx, *ty;
    const uint8_t *nearx, *neary;
    // wavefield levels: level l of shot s at u + (l mod NS) * lstride + s * sstride
    T *u;
    int64_t lstride, sstride;
    int NS;
    const int32_t *nstep;  // record length per shot (plan order)
    PointList src;
    const T *srcv;
    const int64_t *srcv_off, *nsrc;
};

// What a tile's extent holds: interior cells that no PML term reaches; those, the x PML with the rows next
// to it and ring rows (tau = 0 on every column and its neighbours); the y PML likewise; anything.  Each kind is a straight-line body of its own: the
// x PML's coefficients are scalars of the row, the y PML's are registers of the lane.
enum { TILE_PLAIN = 0, TILE_X = 1, TILE_Y = 2, TILE_XY = 3 };

template <typename T> struct FwdTile : TileCommon<T> {
    int n, nt;              // levels n .. n + nt - 1
    const T *phi, *psi;     // level n - 1, stride fstride per shot
    T *phio, *psio;         // level n + nt - 1 (plstride 0), or level n + t at phio + t * plstride
    int64_t fstride, plstride;
};

template <typename T> struct AdjTile : TileCommon<T> {
    int n, nt, Sg;          // levels n down to n - nt + 1; shots per workgroup
    const T *P1, *P2, *F, *G;  // P^{n+1}, P^{n+2}, F^{n+1}, G^{n+1}
    T *P1o, *P2o, *Fo, *Go;    // P^m, P^{m+1}, F^m, G^m of the lowest level m
    int64_t fstride;
    T *gC;                  // one array (gstride) per group of Sg shots
    int64_t gstride;
    PointList rcv;
    const T *resid;
    const int64_t *trace_off, *rcv_ptr;
    const T *dense;         // dense cotangent of u: level l of shot s at dense + l * lstride + s * sstride
};

// The scheme's expressions, shared by every kernel of the acoustic plan so that single- and multi-level
// stepping round alike.  The unit is compiled without contraction; a product is fused only where it is
// exact (a multiplication by 2), which changes no result.
template <typename T> __device__ inline T ac_fma(T a, T b, T c);
template <> __device__ inline float ac_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <> __device__ inline double ac_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
// num / d.  FP64: from inv = 1 / d rounded to nearest, the quotient estimate and one residual correction give
// the correctly rounded quotient (Markstein 1990), then the hardware's fix-up for infinities and zeros;
// the PML divides by 1 + (sigma + tau) dt / 2, which does not change from level to level, and 4 instructions
// take the place of about 20.  FP32 divides: the residual underflows where the quotient nears the
// denormal range, as it does ahead of every wavefront, and one bit there changes every later rounding.
__device__ inline float ac_div(float num, float d, float) { return num / d; }
__device__ inline double ac_div(double num, double d, double inv)
{
    const double q = num * inv;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-q, d, num), inv, q), d, num);
}
template <typename T> __device__ inline T ac_lap(const AcCoef<T> &k, T wc, T ws, T wn, T we, T ww)
{
    return k.cx * ac_fma(T(-2), wc, ws + wn) + k.cy * ac_fma(T(-2), wc, we + ww);
}
template <typename T> __device__ inline T ac_plain(T wc, T wold, T C, T lap)
{
    return ac_fma(T(2), wc, -wold) + C * lap;
}
// The PML update before the division by 1 + h: a2 = 2 - sigma tau dt^2, e = 1 - h, h = (sigma + tau) dt / 2,
// dphi and dpsi the differences of the neighbours' phi and psi
template <typename T>
__device__ inline T ac_pml_num(const AcCoef<T> &k, T a2, T e, T wc, T wold, T C, T lap, T dphi, T dpsi)
{
    return a2 * wc + C * lap + k.ex * dphi + k.ey * dpsi - e * wold;
}
// phi^n = (1 - dt sigma) phi + C (tau - sigma) fx dv, psi^n = (1 - dt tau) psi - C (tau - sigma) fy dv;
// d1 the damping factor, ct = C (tau - sigma).  Taken on the interior's PML cells only: elsewhere phi and psi stay
// the 0 that they start from, also beside a dv that is not finite.  (The tiles tell those cells by
// C (tau + sigma) != 0, with C = 0 outside the interior, which costs no register over the levels and no time;
// flags of the cell cost up to 2.6 %.)
template <typename T> __device__ inline T ac_phi(const AcCoef<T> &k, T d1, T phi, T ct, T dv)
{
    return d1 * phi + ct * k.fx * dv;
}
template <typename T> __device__ inline T ac_psi(const AcCoef<T> &k, T d1, T psi, T ct, T dv)
{
    return d1 * psi - ct * k.fy * dv;
}

// Columns per lane.  The kernels' register arrays have this last dimension, of 1, only because their code comes
// out better with it: without it the same expressions take other registers and scalar spills, and the adjoint is
// slower (517 x 389, 6 shots, FP32 gradient 7.18 -> 7.43 ms; 200 x 66, 8 shots, FP64 15.5 -> 15.7 ms).
constexpr int VEC = 1;

// A tile as one wavefront sees it.
struct TileView {
    int i0, i1, j0, j1;  // core
    int r0, nr;          // global row of register row 0, rows inside the extent
    int lane, w, j;      // j: the lane's first column
    int jc, last;        // the column and the last row that the lane's loads are clamped to: what lies
                         // beyond the extent repeats its edge and is never stored
    int jend;            // one past the extent's last column
};
template <int R> __device__ inline TileView tile_view(const int4 c, const int4 e)
{
    TileView v;
    v.i0 = c.x, v.i1 = c.y, v.j0 = c.z, v.j1 = c.w;
    v.lane = threadIdx.x & (WAVE - 1);
    v.w = wave_id();
    const int ne = e.z & 0xffff, ce = e.z >> 16;
    v.r0 = e.x + v.w * R;
    v.nr = min(max(ne - v.w * R, 0), R);
    v.j = e.y + v.lane;
    v.jc = e.y + min(v.lane, ce - 1);
    v.last = e.x + ne - 1;
    v.jend = e.y + ce;
    return v;
}
// Stores rows r of x whose bit is set in `rows` (wave-uniform) from the lanes whose column j lies in
// [j0, j1); ro: byte offset of each row (wave-uniform), jb of the lane's column.
template <typename T, int R>
__device__ inline void store_rows(T *base, const uint32_t *ro, uint32_t jb, const T (&x)[R][VEC], uint32_t rows, int j,
                                  int j0, int j1)
{
    if (j < j0 || j >= j1) return;
    if (rows == (1u << R) - 1) {
#pragma unroll
        for (int r = 0; r < R; r++) vst(at_off(at_off(base, ro[r]), jb), x[r]);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (rows >> r & 1) vst(at_off(at_off(base, ro[r]), jb), x[r]);
    }
}

// PML coefficients of a lane's cells.  sg: sigma per row (scalars).  TILE_X: e, 1 + h, its reciprocal and d1
// per row (scalars); TILE_Y: the same per column; TILE_XY: the reciprocal per cell, the rest formed where it
// is used.
template <typename T, int R, int KIND> struct PmlCoef {
    static constexpr bool X = KIND == TILE_X, Y = KIND == TILE_Y, XY = KIND == TILE_XY;
    T sg[R], re[X ? R : 1], rh[X ? R : 1], ri[X ? R : 1], rd[X || XY ? R : 1];
    T tu[VEC], te[Y ? VEC : 1], th[Y ? VEC : 1], ti[Y ? VEC : 1], tk[VEC], inv[XY ? R : 1][VEC];
    uint32_t rin, nx;        // interior rows, rows next to the x PML or in it
    bool jin[VEC], ny[VEC];  // interior columns, columns next to the y PML or in it
    __device__ inline void load(const TileView &t, const TileCommon<T> &a, const AcCoef<T> &k)
    {
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            const bool cok = t.j < t.jend;
            jin[e] = t.j >= 1 && t.j <= a.NY && cok;
            tu[e] = !X && cok ? a.ty[t.j] : T(0);
            tk[e] = T(1) - k.dt * tu[e];
            ny[e] = !X && cok && a.neary[t.j] != 0;
            if constexpr (Y) {
                te[e] = T(1) - tu[e] * k.hdt;
                th[e] = T(1) + tu[e] * k.hdt;
                ti[e] = T(1) / th[e];
            }
        }
        rin = nx = 0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = t.r0 + r;
            const bool ok = r < t.nr;
            rin |= ok && i >= 1 && i <= a.NX ? 1u << r : 0u;
            nx |= !Y && ok && a.nearx[i] != 0 ? 1u << r : 0u;
            sg[r] = Y ? T(0) : uniform(a.sx[min(i, t.last)]);
            if constexpr (X) {
                re[r] = uniform(T(1) - sg[r] * k.hdt);
                rh[r] = uniform(T(1) + sg[r] * k.hdt);
                ri[r] = uniform(T(1) / (T(1) + sg[r] * k.hdt));
            }
            if constexpr (X || XY) rd[r] = uniform(T(1) - k.dt * sg[r]);
            if constexpr (XY)
#pragma unroll
                for (int e = 0; e < VEC; e++) inv[r][e] = T(1) / (T(1) + (sg[r] + tu[e]) * k.hdt);
        }
        rin = __builtin_amdgcn_readfirstlane(rin);
        nx = __builtin_amdgcn_readfirstlane(nx);
    }
    // inside the PML
    __device__ inline bool pml(int r, int e) const { return (!X && tu[e] != T(0)) || (!Y && sg[r] != T(0)); }
    // tau + sigma
    __device__ inline T sum(int r, int e) const { return X ? sg[r] : Y ? tu[e] : sg[r] + tu[e]; }
    // tau - sigma
    __device__ inline T c(int r, int e) const { return X ? -sg[r] : Y ? tu[e] : tu[e] - sg[r]; }
    __device__ inline T a2(int r, int e, const AcCoef<T> &k) const { return XY ? T(2) - sg[r] * tu[e] * k.dt2 : T(2); }
    __device__ inline T e(int r, int q, const AcCoef<T> &k) const
    {
        if constexpr (X) return re[r];
        else if constexpr (Y) return te[q];
        else return T(1) - (sg[r] + tu[q]) * k.hdt;
    }
    // x / (1 + h)
    __device__ inline T div(T x, int r, int q, const AcCoef<T> &k) const
    {
        if constexpr (X) return ac_div(x, rh[r], ri[r]);
        else if constexpr (Y) return ac_div(x, th[q], ti[q]);
        else return ac_div(x, T(1) + (sg[r] + tu[q]) * k.hdt, inv[r][q]);
    }
    // the PML formula holds; the plain one elsewhere
    __device__ inline bool near(int r, int e) const { return (!Y && (nx >> r & 1)) || (!X && ny[e]); }
    __device__ inline T d1(int r) const
    {
        if constexpr (Y) return T(1);
        else return rd[r];
    }
    __device__ inline bool in(int r, int e) const { return (Y || (rin >> r & 1)) && (X || jin[e]); }
};

// One wavefront's part of a point list: cells [lo, hi) in rows row0 .. row0 + nrow - 1 of the
// extent, and the mask of those rows that hold a cell.  Values go through a small LDS plane (one
// value per row and lane, zero when idle): a lane per cell writes, every lane reads its column.
struct WavePoints {
    int lo, hi;
    uint32_t rows;
};
template <int NROW>
__device__ inline WavePoints wave_points(const PointList &p, int64_t at, int row0, int lane)
{
    WavePoints o{0, 0, 0u};
    const int q0 = p.ptr[at], q1 = p.ptr[at + 1];
    if (q1 <= q0) return o;
    int before = 0, upto = 0;
    for (int q = q0; q < q1; q += WAVE) {
        const int row = q + lane < q1 ? p.cell[q + lane].x >> 8 : 0x7fff;
        before += __popcll(__ballot(row < row0));
        upto += __popcll(__ballot(row < row0 + NROW));
        const int k = row - row0;
#pragma unroll
        for (int r = 0; r < NROW; r++) o.rows |= __ballot(k == r) ? 1u << r : 0u;
    }
    o.lo = q0 + before;
    o.hi = q0 + upto;
    return o;
}

// Adds dt^2 srcv[lev - 1, .] at the wavefront's source cells to rows of B, entry by entry in
// source order (Core.jl:593-601).  `first`: the value of the lane's own first cell and entry.
template <typename T, int R>
__device__ inline void add_points(const TileCommon<T> &a, const WavePoints &wp, int row0, int lane,
                                  T (*__restrict__ plane)[WAVE], const T *__restrict__ srow, T first,
                                  T (&B)[R][VEC])
{
    for (int k = 0;; k++) {
        bool any = false;
        for (int q = wp.lo + lane; q < wp.hi; q += WAVE) {
            const int2 c = a.src.cell[q];
            if (c.y + k >= a.src.cell[q + 1].y) continue;
            const T v = k == 0 && q < wp.lo + WAVE ? first : srow[a.src.ent[c.y + k]];
            plane[(c.x >> 8) - row0][c.x & 255] = v * a.k.dt2;
            any = true;
        }
        if (!__ballot(any)) break;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < R; r++)
            if (wp.rows >> r & 1) {  // uniform
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    B[r][e] += plane[r][lane];
                    plane[r][lane] = T(0);
                }
            }
        __builtin_amdgcn_wave_barrier();
    }
}
// first-entry value of the lane's own cell at a level's srcv row
template <typename T>
__device__ inline T first_point(const PointList &p, const WavePoints &wp, int lane, const T *__restrict__ row)
{
    const int q = wp.lo + lane;
    return q < wp.hi ? row[p.ent[p.cell[q].y]] : T(0);
}
// Sum over a cell's entries of row[entry] (in order), for every cell of the wavefront, into plane.
template <typename T, int W>
__device__ inline void sum_points(const PointList &p, const WavePoints &wp, int row0, int lane,
                                  T (*__restrict__ plane)[W], const T *__restrict__ row, T first, T scale)
{
    for (int q = wp.lo + lane; q < wp.hi; q += WAVE) {
        const int2 c = p.cell[q];
        const int e1 = p.cell[q + 1].y;
        T v = q < wp.lo + WAVE ? first * scale : row[p.ent[c.y]] * scale;
        for (int e = c.y + 1; e < e1; e++) v += row[p.ent[e]] * scale;
        plane[(c.x >> 8) - row0][c.x & 255] = v;
    }
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------
template <typename T, int V, int R, int NW, bool PML> struct FwdTileLds {
    T u[2][NW][2][WAVE];
    T p[PML ? 2 : 0][NW][2][WAVE];            // phi rows
    T v[PML && V == 0 ? 2 : 0][NW][2][WAVE];  // u^n before the sources
    T plane[NW][R][WAVE];
};

template <typename T, int V, int R, int NW, int KIND>
__device__ inline void fwd_tile_body(const FwdTile<T> &a, const TileView &t, int s, int tile, int nt,
                                     FwdTileLds<T, V, R, NW, KIND != TILE_PLAIN> &lds)
{
    constexpr bool PML = KIND != TILE_PLAIN;
    const AcCoef<T> k = a.k;
    const int lane = t.lane, w = t.w, j = t.j;
    const uint32_t jb = (uint32_t)j * (uint32_t)sizeof(T), jcb = (uint32_t)t.jc * (uint32_t)sizeof(T);
    const int lrow = w * R;  // first register row within the extent
    const T zero[VEC] = {};
#pragma unroll
    for (int r = 0; r < R; r++) vst(&lds.plane[w][r][lane], zero);
    uint32_t ro[R];  // byte offset of each row, clamped to the extent (wave-uniform)
#pragma unroll
    for (int r = 0; r < R; r++) ro[r] = (uint32_t)min(t.r0 + r, t.last) * ((uint32_t)a.P * (uint32_t)sizeof(T));
    T C[R][VEC];
#pragma unroll
    for (int r = 0; r < R; r++) vld(C[r], at_off(at_off(a.C, ro[r]), jcb));
    const uint32_t core = row_mask<R>(t.r0, t.i0, t.i1);  // core rows (wave-uniform)
    const int wu = max(w - 1, 0), wd = min(w + 1, NW - 1);

    int par = 0;
    int slot = a.n % a.NS;
    const int sl1 = slot >= 1 ? slot - 1 : a.NS - 1, sl2 = sl1 >= 1 ? sl1 - 1 : a.NS - 1;
    T *__restrict__ ub = a.u + (int64_t)s * a.sstride;
    const T *__restrict__ w1 = ub + (int64_t)sl1 * a.lstride;
    const T *__restrict__ w0 = ub + (int64_t)sl2 * a.lstride;
    const T *__restrict__ phi = a.phi + (int64_t)s * a.fstride;
    const T *__restrict__ psi = a.psi + (int64_t)s * a.fstride;
    T A[R][VEC], B[R][VEC], F[R][VEC], G[R][VEC];
#pragma unroll
    for (int r = 0; r < R; r++) {
        vld(A[r], at_off(at_off(w1, ro[r]), jcb));
        vld(B[r], at_off(at_off(w0, ro[r]), jcb));
        if constexpr (PML) {
            vld(F[r], at_off(at_off(phi, ro[r]), jcb));
            vld(G[r], at_off(at_off(psi, ro[r]), jcb));
        }
    }
    const WavePoints wp = wave_points<R>(a.src, (int64_t)s * a.ntiles + tile, lrow, lane);
    const int64_t ns = a.nsrc[s];
    const T *__restrict__ srow = a.srcv + a.srcv_off[s] + (int64_t)(a.n - 1) * ns;
    T pv = first_point(a.src, wp, lane, srow);
    PmlCoef<T, R, KIND> pc;
    if constexpr (PML) {
        pc.load(t, a, k);
#pragma unroll
        for (int r = 0; r < R; r++)  // so that phi = psi = 0 outside the interior
#pragma unroll
            for (int e = 0; e < VEC; e++) C[r][e] = pc.in(r, e) ? C[r][e] : T(0);
    }
    auto level = [&](T (&X)[R][VEC], T (&Y)[R][VEC], int q) {  // X = u^{n-1}; Y: u^{n-2} in, u^n out
        if constexpr (PML) {
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                recompute(pc.tu[e]);
#pragma unroll
                for (int r = 0; r < R; r++) recompute(C[r][e]);
            }
        }
        vst(&lds.u[par][w][0][lane], X[0]);
        vst(&lds.u[par][w][1][lane], X[R - 1]);
        if constexpr (PML) {
            vst(&lds.p[par][w][0][lane], F[0]);
            vst(&lds.p[par][w][1][lane], F[R - 1]);
        }
        __syncthreads();
        // rows r0 - 1 and r0 + R (beyond the tile's first and last row: any value)
        T un_[VEC], us_[VEC], fn[VEC], fs_[VEC];
        vld(un_, &lds.u[par][wu][1][lane]);
        vld(us_, &lds.u[par][wd][0][lane]);
        if constexpr (PML) {
            vld(fn, &lds.p[par][wu][1][lane]);
            vld(fs_, &lds.p[par][wd][0][lane]);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            T F_[VEC], G_[VEC];
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                const T wc = X[r][e], wn = r > 0 ? X[r > 0 ? r - 1 : r][e] : un_[e];
                const T ws = r < R - 1 ? X[r < R - 1 ? r + 1 : r][e] : us_[e];
                const T we = lane_east(X[r][e]), ww = lane_west(X[r][e]);
                const T lap = ac_lap(k, wc, ws, wn, we, ww);
                if constexpr (!PML) {
                    Y[r][e] = ac_plain(wc, Y[r][e], C[r][e], lap);
                } else {
                    const T fs = r < R - 1 ? F[r < R - 1 ? r + 1 : r][e] : fs_[e];
                    T out = ac_plain(wc, Y[r][e], C[r][e], lap);
                    if (!pc.X || pc.near(r, e)) {  // uniform for TILE_X
                        const T num = ac_pml_num(k, pc.a2(r, e, k), pc.e(r, e, k), wc, Y[r][e], C[r][e], lap, fs - fn[e],
                                                 lane_east(G[r][e]) - lane_west(G[r][e]));
                        out = pc.near(r, e) ? pc.div(num, r, e, k) : out;
                    }
                    Y[r][e] = pc.in(r, e) ? out : T(0);
                    if constexpr (V == 1) {
                        const T ct = C[r][e] * pc.c(r, e);
                        F_[e] = F[r][e];
                        G_[e] = G[r][e];
                        if (C[r][e] * pc.sum(r, e) != T(0)) {
                            F_[e] = ac_phi(k, pc.d1(r), F[r][e], ct, ws - wn);
                            G_[e] = ac_psi(k, pc.tk[e], G[r][e], ct, we - ww);
                        }
                    }
                    fn[e] = F[r][e];
                }
            }
            if constexpr (PML && V == 1) {
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    F[r][e] = F_[e];
                    G[r][e] = G_[e];
                }
            }
        }
        if constexpr (V == 0 && PML) {  // phi/psi from u^n before the sources
            vst(&lds.v[par][w][0][lane], Y[0]);
            vst(&lds.v[par][w][1][lane], Y[R - 1]);
            __syncthreads();
            T vn_[VEC], vs_[VEC];
            vld(vn_, &lds.v[par][wu][1][lane]);
            vld(vs_, &lds.v[par][wd][0][lane]);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    const T vn = r > 0 ? Y[r > 0 ? r - 1 : r][e] : vn_[e];
                    const T vs = r < R - 1 ? Y[r < R - 1 ? r + 1 : r][e] : vs_[e];
                    const T ve = lane_east(Y[r][e]), vw = lane_west(Y[r][e]);  // (by every lane)
                    const T ct = C[r][e] * pc.c(r, e);
                    if (C[r][e] * pc.sum(r, e) != T(0)) {
                        F[r][e] = ac_phi(k, pc.d1(r), F[r][e], ct, vs - vn);
                        G[r][e] = ac_psi(k, pc.tk[e], G[r][e], ct, ve - vw);
                    }
                }
        }
        // the next level's value is loaded inside the same branch: a load carried to the loop's end
        // on the other path would make every level wait for its own stores
        if (wp.hi > wp.lo) {
            add_points<T, R>(a, wp, lrow, lane, lds.plane[w], srow, pv, Y);
            srow += ns;
            if (q + 1 < nt) pv = first_point(a.src, wp, lane, srow);
        }
        store_rows(ub + (int64_t)slot * a.lstride, ro, jb, Y, core, j, t.j0, t.j1);
        if constexpr (PML) {
            if (a.plstride != 0 || q == nt - 1) {
                const int64_t o = (int64_t)s * a.fstride + (int64_t)q * a.plstride;
                store_rows(a.phio + o, ro, jb, F, core, j, t.j0, t.j1);
                store_rows(a.psio + o, ro, jb, G, core, j, t.j0, t.j1);
            }
        }
        slot = slot + 1 == a.NS ? 0 : slot + 1;
        par ^= 1;
    };
    for (int q = 0; q < nt; q += 2) {
        level(A, B, q);
        if (q + 1 < nt) level(B, A, q + 1);
    }
}

// RN (RP): rows per wavefront of a plain (PML) tile.  What bounds it: at 1000^2 x 32
// shots FP32 with 7 levels per launch (63 us per level; one level per launch takes 104) the vector units
// issue two thirds of the time, half of that for the PML tiles and 40 % for the halo, and 3.3 TB/s move,
// mostly stores; a workgroup's loads do not overlap its own levels, so several per CU have to.
// FP32 asks for three (69 VGPRs): 63 us, two 63, four (64 VGPRs, some spilled) 74.
template <typename T, int V, int RN, int RP, int NW>
__global__ __launch_bounds__(NW *WAVE) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 4)))
void ac_fwd_tile(const FwdTile<T> a)
{
    using LP = FwdTileLds<T, V, RP, NW, true>;
    using LN = FwdTileLds<T, V, RN, NW, false>;
    __shared__ __align__(16) char raw[sizeof(LP) > sizeof(LN) ? sizeof(LP) : sizeof(LN)];
    TileMap m{a.ntiles, a.act, 1, a.nb};
    int z, s, tile;
    if (!decode_tile(m, z, s, tile, (int)blockIdx.x)) return;  // workgroup-uniform
    const int4 c = a.tiles[2 * tile], e = a.tiles[2 * tile + 1];
    const int nt = min(a.nt, a.nstep[s] - a.n + 1);
    LP &lp = *reinterpret_cast<LP *>(raw);
    if (e.w == TILE_PLAIN)
        fwd_tile_body<T, V, RN, NW, TILE_PLAIN>(a, tile_view<RN>(c, e), s, tile, nt,
                                                     *reinterpret_cast<LN *>(raw));
    else if (e.w == TILE_X)
        fwd_tile_body<T, V, RP, NW, TILE_X>(a, tile_view<RP>(c, e), s, tile, nt, lp);
    else if (e.w == TILE_Y)
        fwd_tile_body<T, V, RP, NW, TILE_Y>(a, tile_view<RP>(c, e), s, tile, nt, lp);
    else
        fwd_tile_body<T, V, RP, NW, TILE_XY>(a, tile_view<RP>(c, e), s, tile, nt, lp);
}

// ---------------------------------------------------------------------------------------------
// adjoint
// ---------------------------------------------------------------------------------------------
template <typename T, int V, int R, int NW, bool PML> struct AdjTileLds {
    T p[2][NW][2][WAVE];
    T f[PML ? 2 : 0][NW][2][WAVE];  // C (tau - sigma) F rows
    T plane[NW][R + (PML ? 2 : 0)][WAVE];
};

template <typename T, int V, int R, int NW, int KIND, bool DENSE>
__device__ inline void adj_tile_body(const AdjTile<T> &a, const TileView &t, int g, int tile,
                                     AdjTileLds<T, V, R, NW, KIND != TILE_PLAIN> &lds)
{
    constexpr bool PML = KIND != TILE_PLAIN;
    constexpr bool UN = V == 0 && PML;  // kernel 0 also reads u^n before its sources
    constexpr int RD = DENSE ? R : 1, RV = UN ? R + 2 : 1;
    const AcCoef<T> k = a.k;
    const int lane = t.lane, w = t.w, j = t.j;
    const uint32_t jb = (uint32_t)j * (uint32_t)sizeof(T), jcb = (uint32_t)t.jc * (uint32_t)sizeof(T);
    const int lrow = w * R;
    const int m = a.n - a.nt + 1;
    const uint32_t core = row_mask<R>(t.r0, t.i0, t.i1);  // core rows (wave-uniform)
    const int wu = max(w - 1, 0), wd = min(w + 1, NW - 1);
    const T zero[VEC] = {};
#pragma unroll
    for (int r = 0; r < R + (PML ? 2 : 0); r++) vst(&lds.plane[w][r][lane], zero);

    PmlCoef<T, R, KIND> pc;
    if constexpr (PML) pc.load(t, a, k);
    uint32_t ro[R + 2];  // byte offset of rows r0 - 1 .. r0 + R, clamped to the extent and the grid
#pragma unroll
    for (int q = 0; q < R + 2; q++)
        ro[q] = (uint32_t)min(max(t.r0 - 1 + q, 0), t.last) * ((uint32_t)a.P * (uint32_t)sizeof(T));
    T C[R + 2][VEC], acc[R][VEC];
#pragma unroll
    for (int q = 0; q < R + 2; q++) vld(C[q], at_off(at_off(a.C, ro[q]), jcb));
#pragma unroll
    for (int r = 0; r < R; r++) vzero(acc[r]);

    int par = 0;
    const int s1 = min(a.act, (g + 1) * a.Sg);
    for (int s = g * a.Sg; s < s1; s++) {
        const int top = min(a.n, a.nstep[s]);  // a shot enters at its own last level, from zero
        const int64_t fo_ = (int64_t)s * a.fstride;
        T A[R][VEC], B[R][VEC], F[R][VEC], G[R][VEC];
#pragma unroll
        for (int r = 0; r < R; r++) {
            vld(A[r], at_off(at_off(a.P1 + fo_, ro[r + 1]), jcb));
            vld(B[r], at_off(at_off(a.P2 + fo_, ro[r + 1]), jcb));
            if constexpr (PML) {
                vld(F[r], at_off(at_off(a.F + fo_, ro[r + 1]), jcb));
                vld(G[r], at_off(at_off(a.G + fo_, ro[r + 1]), jcb));
            }
        }
        const T *__restrict__ ub = a.u + (int64_t)s * a.sstride;
        // rows r0 - 1 .. r0 + R of level l; wavefronts without core rows need none
        auto load_u = [&](int l, T (&U)[R + 2][VEC]) {
            if (core == 0) return;  // uniform
            const T *__restrict__ ul = ub + (int64_t)(l % a.NS) * a.lstride;
#pragma unroll
            for (int q = 0; q < R + 2; q++) vld(U[q], at_off(at_off(ul, ro[q]), jcb));
        };
        auto load_d = [&](int l, T (&D)[RD][VEC]) {
            const T *__restrict__ dl = a.dense + (int64_t)s * a.sstride + (int64_t)l * a.lstride;
#pragma unroll
            for (int r = 0; r < RD; r++) vld(D[r], at_off(at_off(dl, ro[r + 1]), jcb));
        };
        T U[R + 2][VEC] = {}, UX[R + 2][VEC] = {}, VN[RV][VEC], D[RD][VEC], DX[RD][VEC] = {};
        load_u(top - 1, U);
        if constexpr (UN) {
#pragma unroll
            for (int q = 0; q < RV; q++) vzero(VN[q]);
            if constexpr (RV == R + 2) load_u(top, VN);
        }
        if constexpr (DENSE) load_d(top, D);
        WavePoints wr{0, 0, 0u}, wsrc{0, 0, 0u};
        const T *__restrict__ rrow = nullptr;
        const T *__restrict__ srow = nullptr;
        int64_t nrc = 0, ns = 0;
        T rv = T(0);
        if constexpr (!DENSE) {
            wr = wave_points<R>(a.rcv, (int64_t)s * a.ntiles + tile, lrow, lane);
            nrc = a.rcv_ptr[s + 1] - a.rcv_ptr[s];
            rrow = a.resid + a.trace_off[s] + (int64_t)top * nrc;
            rv = first_point(a.rcv, wr, lane, rrow);
        }
        if constexpr (UN) {
            wsrc = wave_points<R + 2>(a.src, (int64_t)s * a.ntiles + tile, lrow - 1, lane);
            ns = a.nsrc[s];
            srow = a.srcv + a.srcv_off[s] + (int64_t)(top - 1) * ns;
        }

        // X = P^{n+1}; Y: P^{n+2} in, P^n out; U = u^{n-1}, UX receives u^{n-2} (D, DX likewise)
        auto level = [&](T (&X)[R][VEC], T (&Y)[R][VEC], T (&U)[R + 2][VEC], T (&UX)[R + 2][VEC], T (&D)[RD][VEC],
                         T (&DX)[RD][VEC], int n) {
            if constexpr (PML) {
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    recompute(pc.tu[e]);
#pragma unroll
                    for (int q = 0; q < R + 2; q++) recompute(C[q][e]);
                }
            }
            vst(&lds.p[par][w][0][lane], X[0]);
            vst(&lds.p[par][w][1][lane], X[R - 1]);
            // (C (tau - sigma)) F of a row
            auto fq = [&](int r, T (&o)[VEC]) {
#pragma unroll
                for (int e = 0; e < VEC; e++) o[e] = C[r + 1][e] * pc.c(r, e) * F[r][e];
            };
            // F^n, G^n and their dL/dC terms: dpi, dpj the differences of P^{n+1}, dvi, dvj those of the
            // field that phi/psi^n read
            auto adj_phipsi = [&](int r, int e, T dpi, T dpj, T dvi, T dvj, T &F, T &G, T &acc) {
                const T c = pc.c(r, e);
                const bool pml = pc.in(r, e) && pc.pml(r, e);
                if constexpr (V == 1) {  // (a dv that is not finite makes the cell's other term so, too)
                    F = pml ? pc.d1(r) * F + k.ex * dpi : T(0);
                    G = pml ? pc.tk[e] * G + k.ey * dpj : T(0);
                    acc = ac_fma(F * c * k.fx, dvi, acc);
                    acc = ac_fma(G * -c * k.fy, dvj, acc);
                } else if (pml) {  // elsewhere F and G stay 0, and nothing joins acc beside any dv
                    F = pc.d1(r) * F + k.ex * dpi;
                    G = pc.tk[e] * G + k.ey * dpj;
                    acc = ac_fma(F * c * k.fx, dvi, acc);
                    acc = ac_fma(G * -c * k.fy, dvj, acc);
                }
            };
            if constexpr (PML && V == 1) {
                T q0[VEC], q1[VEC];
                fq(0, q0);
                fq(R - 1, q1);
                vst(&lds.f[par][w][0][lane], q0);
                vst(&lds.f[par][w][1][lane], q1);
            }
            // the next level's inputs, in flight during this one
            if (n > m) {
                load_u(n - 2, UX);
                if constexpr (DENSE) load_d(n - 1, DX);
            }
            __syncthreads();
            T pn_[VEC], ps_[VEC];
            vld(pn_, &lds.p[par][wu][1][lane]);
            vld(ps_, &lds.p[par][wd][0][lane]);
            if constexpr (UN) {  // F^n, G^n and their dL/dC terms, with u^n before its sources
                if (wsrc.hi > wsrc.lo) {
                    sum_points(a.src, wsrc, lrow - 1, lane, lds.plane[w], srow,
                               first_point(a.src, wsrc, lane, srow), k.dt2);
#pragma unroll
                    for (int q = 0; q < RV; q++)
                        if (wsrc.rows >> q & 1) {
#pragma unroll
                            for (int e = 0; e < VEC; e++) VN[q][e] -= lds.plane[w][q][lane];
                            vst(&lds.plane[w][q][lane], zero);
                        }
                    __builtin_amdgcn_wave_barrier();
                    srow -= ns;
                }
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const T pn = r > 0 ? X[r > 0 ? r - 1 : r][e] : pn_[e];
                        const T ps = r < R - 1 ? X[r < R - 1 ? r + 1 : r][e] : ps_[e];
                        const T dp = lane_west(X[r][e]) - lane_east(X[r][e]);
                        const T dvj = lane_east(VN[UN ? r + 1 : 0][e]) - lane_west(VN[UN ? r + 1 : 0][e]);
                        adj_phipsi(r, e, pn - ps, dp, VN[UN ? r + 2 : 0][e] - VN[UN ? r : 0][e], dvj, F[r][e], G[r][e], acc[r][e]);
                    }
                T q0[VEC], q1[VEC];
                fq(0, q0);
                fq(R - 1, q1);
                vst(&lds.f[par][w][0][lane], q0);
                vst(&lds.f[par][w][1][lane], q1);
                __syncthreads();
            }
            T fn[VEC], fs_[VEC], fc[VEC], fs[VEC];
            if constexpr (PML) {
                vld(fn, &lds.f[par][wu][1][lane]);
                vld(fs_, &lds.f[par][wd][0][lane]);
                fq(0, fc);
            }
            if (wr.hi > wr.lo) sum_points(a.rcv, wr, lrow, lane, lds.plane[w], rrow, rv, T(1));
            T qn[VEC], qc[VEC], qs[VEC];
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                qn[e] = C[0][e] * pn_[e];
                qc[e] = C[1][e] * X[0][e];
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                T gq[VEC];
#pragma unroll
                for (int e = 0; e < VEC; e++)
                    qs[e] = C[r + 2][e] * (r < R - 1 ? X[r < R - 1 ? r + 1 : r][e] : ps_[e]);
                if constexpr (PML) {
                    if (r < R - 1) fq(r < R - 1 ? r + 1 : r, fs);
                    else {
#pragma unroll
                        for (int e = 0; e < VEC; e++) fs[e] = fs_[e];
                    }
#pragma unroll
                    for (int e = 0; e < VEC; e++) gq[e] = C[r + 1][e] * -pc.c(r, e) * G[r][e];
                }
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    const T p1c = X[r][e];
                    const T lapq = ac_lap(k, qc[e], qs[e], qn[e], lane_east(qc[e]), lane_west(qc[e]));
                    T Pv = ac_fma(T(2), p1c, lapq) - Y[r][e];
                    if constexpr (DENSE) Pv += D[r][e];
                    if constexpr (PML) {
                        if (!pc.X || pc.near(r, e)) {  // uniform for TILE_X
                            T U_ = pc.a2(r, e, k) * p1c + lapq - pc.e(r, e, k) * Y[r][e] + k.fx * (fn[e] - fs[e]) +
                                   k.fy * (lane_west(gq[e]) - lane_east(gq[e]));
                            if constexpr (DENSE) U_ += D[r][e];
                            Pv = pc.near(r, e) ? pc.div(U_, r, e, k) : Pv;
                        }
                        Pv = pc.in(r, e) ? Pv : T(0);
                    }
                    Y[r][e] = Pv;
                }
                if (wr.rows >> r & 1) {  // uniform: receiver residuals on this row
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const T add = lds.plane[w][r][lane];
                        if constexpr (PML) Y[r][e] += pc.div(add, r, e, k);
                        else Y[r][e] += add;
                    }
                    vst(&lds.plane[w][r][lane], zero);
                }
#pragma unroll
                for (int e = 0; e < VEC; e++)
                    acc[r][e] = ac_fma(Y[r][e],
                                       ac_lap(k, U[r + 1][e], U[r + 2][e], U[r][e], lane_east(U[r + 1][e]), lane_west(U[r + 1][e])),
                                       acc[r][e]);
                if constexpr (PML && V == 1) {
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const T pn = r > 0 ? X[r > 0 ? r - 1 : r][e] : pn_[e];
                        const T ps = r < R - 1 ? X[r < R - 1 ? r + 1 : r][e] : ps_[e];
                        adj_phipsi(r, e, pn - ps, lane_west(X[r][e]) - lane_east(X[r][e]), U[r + 2][e] - U[r][e],
                                   lane_east(U[r + 1][e]) - lane_west(U[r + 1][e]), F[r][e], G[r][e], acc[r][e]);
                    }
                }
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    qn[e] = qc[e];
                    qc[e] = qs[e];
                    if constexpr (PML) {
                        fn[e] = fc[e];
                        fc[e] = fs[e];
                    }
                }
            }
            if (wr.hi > wr.lo) {
                __builtin_amdgcn_wave_barrier();
                rrow -= nrc;
                if (n > m) rv = first_point(a.rcv, wr, lane, rrow);
            }
            if constexpr (UN) {
#pragma unroll
                for (int q = 0; q < RV; q++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) VN[q][e] = U[q][e];
            }
            par ^= 1;
        };
        auto store = [&](const T (&X)[R][VEC], const T (&Y)[R][VEC]) {  // X = P^{m+1}, Y = P^m
            store_rows(a.P1o + fo_, ro + 1, jb, Y, core, j, t.j0, t.j1);
            store_rows(a.P2o + fo_, ro + 1, jb, X, core, j, t.j0, t.j1);
            if constexpr (PML) {
                store_rows(a.Fo + fo_, ro + 1, jb, F, core, j, t.j0, t.j1);
                store_rows(a.Go + fo_, ro + 1, jb, G, core, j, t.j0, t.j1);
            }
        };
        int n = top;
        for (;;) {
            level(A, B, U, UX, D, DX, n);
            if (n-- == m) {
                store(A, B);
                break;
            }
            level(B, A, UX, U, DX, D, n);
            if (n-- == m) {
                store(B, A);
                break;
            }
        }
    }
    T *__restrict__ gC = a.gC + (int64_t)g * a.gstride;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (!(core >> r & 1)) continue;  // uniform
        T *p = at_off(at_off(gC, ro[r + 1]), jb);
#pragma unroll
        for (int e = 0; e < VEC; e++)
            if (j >= t.j0 && j < t.j1 && (!PML || pc.in(r, e))) p[e] += acc[r][e];
    }
}

// Bounds as in the forward; 1000^2 x 32 shots FP32, 7 levels per launch: 94 us per level (one level per
// launch and a receiver launch: 178).  Two workgroups per CU in FP32 (128 VGPRs with a few spilled): 100
// against 147 us with one (no spills) and 203 with three, eight shots per workgroup.
template <typename T, int V, int RN, int RP, int NW, bool DENSE>
__global__ __launch_bounds__(NW *WAVE) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2)))
void ac_adj_tile(const AdjTile<T> a)
{
    using LP = AdjTileLds<T, V, RP, NW, true>;
    using LN = AdjTileLds<T, V, RN, NW, false>;
    __shared__ __align__(16) char raw[sizeof(LP) > sizeof(LN) ? sizeof(LP) : sizeof(LN)];
    TileMap m{a.ntiles, (a.act + a.Sg - 1) / a.Sg, 1, a.nb};
    int z, g, tile;
    if (!decode_tile(m, z, g, tile, (int)blockIdx.x)) return;  // workgroup-uniform
    const int4 c = a.tiles[2 * tile], e = a.tiles[2 * tile + 1];
    LP &lp = *reinterpret_cast<LP *>(raw);
    if (e.w == TILE_PLAIN)
        adj_tile_body<T, V, RN, NW, TILE_PLAIN, DENSE>(a, tile_view<RN>(c, e), g, tile,
                                                            *reinterpret_cast<LN *>(raw));
    else if (e.w == TILE_X)
        adj_tile_body<T, V, RP, NW, TILE_X, DENSE>(a, tile_view<RP>(c, e), g, tile, lp);
    else if (e.w == TILE_Y)
        adj_tile_body<T, V, RP, NW, TILE_Y, DENSE>(a, tile_view<RP>(c, e), g, tile, lp);
    else
        adj_tile_body<T, V, RP, NW, TILE_XY, DENSE>(a, tile_view<RP>(c, e), g, tile, lp);
}

// ---------------------------------------------------------------------------------------------
// tiles and point lists (host)
// ---------------------------------------------------------------------------------------------
struct TileHost {
    int i0, i1, j0, j1, ie, je, ne, ce, kind;
};

// Tiles covering rows [ilo, ihi) x columns [jlo, jhi) with halo H; sx, ty: the damping profiles of the
// padded axes (as the kernels read them).
struct TileGrid {
    int NX, NY, rowsN, rowsP;  // interior cells; rows of a plain / PML tile
    std::vector<int> px, py;        // prefix counts of the rows (columns) in the PML or next to it
    std::vector<int> rx, ry;        // of those on the ring
};
template <typename T>
static inline TileGrid tile_grid(const std::vector<T> &sx, const std::vector<T> &ty, int rowsN, int rowsP)
{
    TileGrid g{(int)sx.size() - 2, (int)ty.size() - 2, rowsN, rowsP, {0}, {0}, {0}, {0}};
    auto count = [](const std::vector<T> &f, std::vector<int> &near, std::vector<int> &ring) {
        for (size_t q = 0; q < f.size(); q++) {
            const bool n = f[q] != T(0) || (q > 0 && f[q - 1] != T(0)) || (q + 1 < f.size() && f[q + 1] != T(0));
            near.push_back(near.back() + n);
            ring.push_back(ring.back() + (q == 0 || q + 1 == f.size()));
        }
    };
    count(sx, g.px, g.rx);
    count(ty, g.py, g.ry);
    return g;
}
static inline int tile_kind(const TileGrid &g, const TileHost &t)
{
    auto any = [](const std::vector<int> &c, int a, int n) { return c[a + n] != c[a]; };
    const bool dx = any(g.px, t.ie, t.ne), dy = any(g.py, t.je, t.ce);
    const bool rx = any(g.rx, t.ie, t.ne), ry = any(g.ry, t.je, t.ce);
    if (!dx && !dy && !rx && !ry) return TILE_PLAIN;
    if (!dy && !ry) return TILE_X;
    if (!dx && !rx) return TILE_Y;
    return TILE_XY;
}
static inline void add_tiles(std::vector<TileHost> &out, const TileGrid &g, int ilo, int ihi, int jlo, int jhi, int H,
                             bool plain)
{
    if (ihi <= ilo || jhi <= jlo) return;
    const std::vector<int> ci = tile_cuts(ilo, ihi, H, g.NX + 2, plain ? g.rowsN : g.rowsP);
    const std::vector<int> cj = tile_cuts(jlo, jhi, H, g.NY + 2, WAVE);
    for (size_t p = 0; p + 1 < ci.size(); p++)
        for (size_t q = 0; q + 1 < cj.size(); q++) {
            TileHost t{ci[p], ci[p + 1], cj[q], cj[q + 1], 0, 0, 0, 0, 0};
            t.ie = std::max(t.i0 - H, 0);
            t.je = std::max(t.j0 - H, 0);
            t.ne = std::min(t.i1 + H, g.NX + 2) - t.ie;
            t.ce = std::min(t.j1 + H, g.NY + 2) - t.je;
            t.kind = tile_kind(g, t);
            if (!plain && t.kind == TILE_PLAIN) t.kind = TILE_X;  // holds a PML tile's rows
            out.push_back(t);
        }
}

// The tiles of a grid for launches of up to `levels` levels; R: the cells that no PML term reaches.  The
// plain scheme and kernel 1 lose one halo cell per level, kernel 0's PML cells two (phi/psi follow the
// new u).  Either every tile is a PML tile, or bands of them surround plain tiles, which hold more rows;
// whichever gives the smaller sum of tiles (a PML tile counted as a plain one: fewer cells, more work).
static inline std::vector<TileHost> make_tiles(int variant, int levels, const Rect &R, const TileGrid &g)
{
    std::vector<TileHost> a, b;
    const int H = variant == 0 ? 2 * levels : levels, X = g.NX + 2, Y = g.NY + 2;
    add_tiles(a, g, 0, X, 0, Y, H, false);
    const Rect Q{R.iL + levels, R.iR - levels, R.jL + levels, R.jR - levels};
    if (Q.iR <= Q.iL || Q.jR <= Q.jL) return a;
    add_tiles(b, g, Q.iL, Q.iR, Q.jL, Q.jR, levels, true);
    for (const TileHost &t : b)
        if (t.kind != TILE_PLAIN) return a;
    add_tiles(b, g, 0, Q.iL, 0, Y, H, false);
    add_tiles(b, g, Q.iL, Q.iR, 0, Q.jL, H, false);
    add_tiles(b, g, Q.iL, Q.iR, Q.jR, Y, H, false);
    add_tiles(b, g, Q.iR, X, 0, Y, H, false);
    return b.size() <= a.size() ? b : a;
}

// Point lists of every (shot, tile) for points (i, j) of shots ptr[s] .. ptr[s+1] (see PointList).
struct PointLists {
    std::vector<int32_t> ptr, ent;
    std::vector<int2> cell;
};
static inline PointLists make_points(const std::vector<TileHost> &tiles, int NX, int NY,
                                     const std::vector<int64_t> &ptr, const std::vector<int64_t> &pi,
                                     const std::vector<int64_t> &pj, bool interior)
{
    constexpr int BIN = 32;
    const int nbj = (NY + 2 + BIN - 1) / BIN, nbi = (NX + 2 + BIN - 1) / BIN;
    std::vector<std::vector<int32_t>> bins((size_t)nbi * nbj);
    for (size_t q = 0; q < tiles.size(); q++) {
        const TileHost &t = tiles[q];
        for (int x = t.ie / BIN; x <= (t.ie + t.ne - 1) / BIN; x++)
            for (int y = t.je / BIN; y <= (t.je + t.ce - 1) / BIN; y++) bins[(size_t)x * nbj + y].push_back((int32_t)q);
    }
    struct Key {
        uint64_t at;   // tile, row, column
        int32_t ent;
    };
    PointLists o;
    const size_t nt = tiles.size(), ns = ptr.size() - 1;
    o.ptr.assign(ns * nt + 1, 0);
    std::vector<Key> ks;
    for (size_t s = 0; s < ns; s++) {
        ks.clear();
        for (int64_t e = ptr[s]; e < ptr[s + 1]; e++) {
            const int i = (int)pi[e], j = (int)pj[e];
            if (interior && (i < 1 || i > NX || j < 1 || j > NY)) continue;
            for (int32_t q : bins[(size_t)(i / BIN) * nbj + j / BIN]) {
                const TileHost &t = tiles[q];
                if (i < t.ie || i >= t.ie + t.ne || j < t.je || j >= t.je + t.ce) continue;
                ks.push_back(Key{(uint64_t)q << 16 | (uint64_t)(i - t.ie) << 8 | (uint64_t)(j - t.je), (int32_t)(e - ptr[s])});
            }
        }
        std::sort(ks.begin(), ks.end(), [](const Key &x, const Key &y) { return x.at < y.at || (x.at == y.at && x.ent < y.ent); });
        size_t z = 0;
        for (size_t q = 0; q < nt; q++) {
            o.ptr[s * nt + q] = (int32_t)o.cell.size();
            for (; z < ks.size() && ks[z].at >> 16 == q; z++) {
                if (z == 0 || ks[z].at != ks[z - 1].at)
                    o.cell.push_back(make_int2((int)(ks[z].at & 0xffff), (int)o.ent.size()));
                o.ent.push_back(ks[z].ent);
            }
        }
    }
    o.ptr[ns * nt] = (int32_t)o.cell.size();
    o.cell.push_back(make_int2(0, (int)o.ent.size()));
    if (o.ent.empty()) o.ent.push_back(0);
    return o;
}

}  // namespace ads
