// ads_acoustic.hip -- acoustic PML time stepper for gfx950: forward, hand-written adjoint,
// checkpointed multi-shot batches, full-history drop-in, kernel-shape autotuner.
//
// Scheme (src/Core.jl:528-549 / AcousticOneStepCpu.h:1-48), interior cell (i, j):
//   u^n = [(2 - s t dt^2) w + C lap(w) + ex (phi_{i+1} - phi_{i-1}) + ey (psi_{j+1} - psi_{j-1})
//          - (1 - (s+t) dt/2) wold] / (1 + (s+t) dt/2),
//   lap(w) = cx (w_{i+1} + w_{i-1} - 2w) + cy (w_{j+1} + w_{j-1} - 2w),  cx = dt^2/hx^2
//   phi^n = (1 - dt s) phi + C (t - s) fx (v_{i+1} - v_{i-1}),  fx = dt/(2hx)
//   psi^n = (1 - dt t) psi + C (s - t) fy (v_{j+1} - v_{j-1})
// with w = u^{n-1}, wold = u^{n-2}, v = u^n before source injection (PropagatorKernel 0) or
// v = w (PropagatorKernel 1/2).  s = sigma_x(i), t = tau_y(j) (separable, Core.jl:738-761).
// phi/psi are non-zero only where s or t is (the PML strips); interior cells skip them.
//
// Adjoint (exact transpose of the discrete loop; P^n = dL/du^n / d, d = 1 + (s+t) dt/2):
//   dL/du^n = R^n + (2 - s t dt^2) P^{n+1} + lap(C P^{n+1}) - (1 - (s+t) dt/2) P^{n+2}
//             + fx [Cp_{i-1} F_{i-1} - Cp_{i+1} F_{i+1}] + fy [Cq_{j-1} G_{j-1} - Cq_{j+1} G_{j+1}]
//   F^n = (1 - dt s) F^{n+1} + ex (P^{n+1}_{i-1} - P^{n+1}_{i+1})    (dL/dphi^n), G likewise
//   dL/dC += P^n lap(u^{n-1}) + F^n (t - s) fx (v_{i+1} - v_{i-1}) + G^n (s - t) fy (...)
// where Cp = C (t - s), Cq = C (s - t) and F in the dL/du^n line is F^{n+1} (kernel 1) or F^n
// (kernel 0).  Receiver residuals R^n are added after the stencil pass by a per-cell gather.
//
// Both sweeps run several time levels per launch over tiles held in registers (ads_ac_tile.h).  Stepping the
// forward one level per launch (ads_acoustic_plan_set_blocking(1)) uses the kernels below: the interior
// rectangle, where no PML term reaches, with one 16-byte vector of depth cells per lane and row, and the
// frame around it with one cell per lane.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <limits>
#include <map>
#include <memory>
#include <tuple>
#include <type_traits>
#include <vector>

#include "ads_common.h"
#include "ads_schedule.h"
#include "ads_stencil.h"

namespace ads {

template <typename T> struct AcCoef {
    T cx, cy, ex, ey, fx, fy, dt, hdt, dt2;
};

template <typename T> AcCoef<T> make_coef(double dt, double hx, double hy)
{
    AcCoef<T> k;
    k.cx = (T)(dt * dt / (hx * hx));
    k.cy = (T)(dt * dt / (hy * hy));
    k.ex = (T)(dt * dt / (2.0 * hx));
    k.ey = (T)(dt * dt / (2.0 * hy));
    k.fx = (T)(dt / (2.0 * hx));
    k.fy = (T)(dt / (2.0 * hy));
    k.dt = (T)dt;
    k.hdt = (T)(dt / 2.0);
    k.dt2 = (T)(dt * dt);
    return k;
}

}  // namespace ads
#include "ads_ac_tile.h"
namespace ads {

// Field addressing: level pointer + shot * stride.
template <typename T> struct Lv {
    T *p;
    int64_t stride;
    __device__ __host__ T *at(int s) const { return p + (int64_t)s * stride; }
};
template <typename T> inline Lv<const T> cst(Lv<T> a) { return Lv<const T>{a.p, a.stride}; }

template <typename T> __device__ inline T ldg(const T *p, int64_t i, bool ok) { return ok ? p[i] : T(0); }

// ---------------------------------------------------------------------------------------------
// forward step: u^n (pre-source) and, for kernel 1, phi^n/psi^n
// ---------------------------------------------------------------------------------------------
template <typename T> struct FwdArgs {
    Lv<T> u;
    Lv<const T> w, wold, phi, psi;
    Lv<T> phio, psio;
    const T *C, *sx, *ty;
    const uint8_t *nearx, *neary;
    int NX, NY, P, act, Sg;
    TileMap map;
    AcCoef<T> k;
};

// Rectangle forward: u^n = 2 w - wold + C lap(w).  A wavefront owns RPT rows x (64 lanes x VEC
// depth cells); a workgroup loops over a group of Sg shots, SB at a time, issuing every load of
// those SB shots before the first store, so each wavefront keeps SB shots' rows in flight.
template <typename T, int RPT, int VEC, int SB>
__device__ inline void fwd_rect_body(const FwdArgs<T> &a, const Rect &R, int bid)
{
    int g, strip, tj;
    if (!decode_tile(a.map, g, strip, tj, bid)) return;
    const int lane = threadIdx.x & (WAVE - 1), wv = wave_id();
    const int j0 = R.jL + (tj * WAVE + lane) * VEC;
    const int ib = R.iL + (strip * NWAVES + wv) * RPT;
    if (ib >= R.iR) return;  // wave-uniform
    const int P = a.P, nr = min(RPT, R.iR - ib);
    const bool act = j0 < R.jR;
    const bool le = lane == 0 && act;                                // reads j0-1 >= jL-1 >= 0
    const bool re = act && (lane == WAVE - 1 || j0 + VEC == R.jR);  // reads j0+VEC <= jR <= NY+1
    const AcCoef<T> k = a.k;
    T Cr[RPT][VEC];
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        if (act && r < nr) vld(Cr[r], a.C + (int64_t)(ib + r) * P + j0);
        else vzero(Cr[r]);
    }
    const int s1 = min(a.act, (g + 1) * a.Sg);
    for (int s = g * a.Sg; s < s1; s += SB) {
        T W[SB][RPT + 2][VEC], WO[SB][RPT][VEC], EL[SB][RPT], ER[SB][RPT];
#pragma unroll
        for (int b = 0; b < SB; b++) {
            if (s + b >= s1) break;  // uniform
            const T *__restrict__ w = a.w.at(s + b);
            const T *__restrict__ wo = a.wold.at(s + b);
#pragma unroll
            for (int q = 0; q < RPT + 2; q++) {  // rows iL-1 .. iR lie inside [0, NX+1]
                if (act && q <= nr + 1) vld(W[b][q], w + (int64_t)(ib - 1 + q) * P + j0);
                else vzero(W[b][q]);
            }
#pragma unroll
            for (int r = 0; r < RPT; r++) {
                const int64_t row = (int64_t)(ib + r) * P;
                if (act && r < nr) vld(WO[b][r], wo + row + j0);
                else vzero(WO[b][r]);
                EL[b][r] = le && r < nr ? w[row + j0 - 1] : T(0);
                ER[b][r] = re && r < nr ? w[row + j0 + VEC] : T(0);
            }
        }
#pragma unroll
        for (int b = 0; b < SB; b++) {
            if (s + b >= s1) break;
            T *__restrict__ u = a.u.at(s + b);
#pragma unroll
            for (int r = 0; r < RPT; r++) {
                if (r >= nr) break;  // uniform
                T wl, wr;
                lr_of(W[b][r + 1], EL[b][r], ER[b][r], lane, re, wl, wr);
                T out[VEC];
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    const T wc = W[b][r + 1][e];
                    const T ww = e == 0 ? wl : W[b][r + 1][e - 1];
                    const T we = e == VEC - 1 ? wr : W[b][r + 1][e + 1];
                    const T lap = ac_lap(k, wc, W[b][r + 2][e], W[b][r][e], we, ww);
                    out[e] = ac_plain(wc, WO[b][r][e], Cr[r][e], lap);
                }
                if (act) vst(u + (int64_t)(ib + r) * P + j0, out);
            }
        }
    }
}

// Frame forward, one depth cell per lane.  A workgroup takes one frame item and its four
// wavefronts take every fourth shot of the group, so the thin PML strips still fill the GPU.
// Only lanes with a cell near the PML read phi/psi; cells of the padding ring get u = 0
// (sources are added afterwards).
template <typename T, int V>
__device__ inline void fwd_frame_body(const FwdArgs<T> &a, const TileMap &map,
                                      const int4 *__restrict__ items, int nitems, int bid)
{
    int g, blk, tj;
    if (!decode_tile(map, g, blk, tj, bid)) return;
    const int lane = threadIdx.x & (WAVE - 1), wv = wave_id();
    const int it = blk;  // one item per workgroup; its 4 wavefronts take every 4th shot
    if (it >= nitems) return;  // workgroup-uniform
    const int4 m = items[it];
    const int ib = m.x, nr = m.y, j = m.z + lane;
    const int NX = a.NX, NY = a.NY, P = a.P;
    const bool act = j < m.w;
    const bool le = lane == 0 && act && j >= 1;
    const bool re = act && (lane == WAVE - 1 || j + 1 == m.w);
    const bool reok = re && j + 1 <= NY + 1;
    const AcCoef<T> k = a.k;
    const bool jin = j >= 1 && j <= NY;
    const T tu = act ? a.ty[j] : T(0);
    const bool ny = act && a.neary[j] != 0;
    bool rin[FRPT], nx[FRPT];
    T sg[FRPT], Cr[FRPT];
    bool lp = false;
#pragma unroll
    for (int r = 0; r < FRPT; r++) {
        const int i = ib + r;
        const bool ok = r < nr;
        rin[r] = ok && i >= 1 && i <= NX;
        nx[r] = ok && a.nearx[i] != 0;
        sg[r] = ok ? a.sx[i] : T(0);
        Cr[r] = act && rin[r] ? a.C[(int64_t)i * P + j] : T(0);
        lp |= rin[r] && jin && (nx[r] || ny);
    }
    lp = lp && act;
    const int s1 = min(a.act, (g + 1) * a.Sg);
    for (int s = g * a.Sg + wv; s < s1; s += NWAVES) {
        const T *__restrict__ w = a.w.at(s);
        const T *__restrict__ wo = a.wold.at(s);
        const T *__restrict__ phi = a.phi.at(s);
        const T *__restrict__ psi = a.psi.at(s);
        T W[FRPT + 2], WO[FRPT], PH[FRPT + 2], PS[FRPT], EL[FRPT], ER[FRPT], SL[FRPT], SR[FRPT];
#pragma unroll
        for (int q = 0; q < FRPT + 2; q++) {
            const int i = ib - 1 + q;
            const bool ok = act && q <= nr + 1 && i >= 0 && i <= NX + 1;
            W[q] = ok ? w[(int64_t)i * P + j] : T(0);
            PH[q] = ok && lp ? phi[(int64_t)i * P + j] : T(0);
        }
#pragma unroll
        for (int r = 0; r < FRPT; r++) {
            const int64_t row = (int64_t)(ib + r) * P;
            WO[r] = act && rin[r] ? wo[row + j] : T(0);
            PS[r] = lp && rin[r] ? psi[row + j] : T(0);
            EL[r] = le && rin[r] ? w[row + j - 1] : T(0);
            ER[r] = reok && rin[r] ? w[row + j + 1] : T(0);
            SL[r] = le && lp && rin[r] ? psi[row + j - 1] : T(0);
            SR[r] = reok && lp && rin[r] ? psi[row + j + 1] : T(0);
        }
        T *__restrict__ u = a.u.at(s);
#pragma unroll
        for (int r = 0; r < FRPT; r++) {
            if (r >= nr) break;  // uniform
            const int64_t row = (int64_t)(ib + r) * P;
            T wv1[1] = {W[r + 1]}, pv1[1] = {PS[r]};
            T ww, we, pw, pe;
            lr_of(wv1, EL[r], ER[r], lane, re, ww, we);
            lr_of(pv1, SL[r], SR[r], lane, re, pw, pe);
            const T wc = W[r + 1], wn = W[r], ws = W[r + 2];
            const T lap = ac_lap(k, wc, ws, wn, we, ww);
            const T s_ = sg[r], Cij = Cr[r];
            const bool in = rin[r] && jin;
            const bool near = nx[r] || ny;
            const T plain = ac_plain(wc, WO[r], Cij, lap);
            const T den = T(1) + (s_ + tu) * k.hdt;
            const T num = ac_pml_num(k, T(2) - s_ * tu * k.dt2, T(1) - (s_ + tu) * k.hdt, wc, WO[r], Cij, lap, PH[r + 2] - PH[r], pe - pw);
            const T out = in ? (near ? ac_div(num, den, T(1) / den) : plain) : T(0);
            if (act) u[row + j] = out;
            if (V == 1 && lp) {
                const bool pml = in && (s_ != T(0) || tu != T(0));
                a.phio.at(s)[row + j] = pml ? ac_phi(k, T(1) - k.dt * s_, PH[r + 1], Cij * (tu - s_), ws - wn) : T(0);
                a.psio.at(s)[row + j] = pml ? ac_psi(k, T(1) - k.dt * tu, PS[r], Cij * (tu - s_), we - ww) : T(0);
            }
        }
    }
}

// kernel 0: phi^n/psi^n from the new u (before sources), PML cells only.  The PML lies in the
// frame: one workgroup per (frame item, 4 shots), a wavefront per shot, a lane per column.
template <typename T>
__global__ __launch_bounds__(256) void ac_fwd_phipsi(
    Lv<const T> u_, Lv<const T> phi_, Lv<const T> psi_, Lv<T> phio, Lv<T> psio,
    const T *__restrict__ C, const T *__restrict__ sx, const T *__restrict__ ty,
    const uint8_t *__restrict__ pmlx, const uint8_t *__restrict__ pmly, int NX, int NY, int P,
    AcCoef<T> k, const int4 *__restrict__ items, int act)
{
    const int4 m = items[blockIdx.x];
    const int j = m.z + (threadIdx.x & 63);
    const int s = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (s >= act || j >= m.w || j < 1 || j > NY) return;
    const T *__restrict__ u = u_.at(s);
    const T tu = ty[j];
    for (int r = 0; r < m.y; r++) {
        const int i = m.x + r;
        if (i < 1 || i > NX || !(pmlx[i] | pmly[j])) continue;
        const int64_t ij = (int64_t)i * P + j;
        const T sg = sx[i], Cij = C[ij];
        phio.at(s)[ij] = ac_phi(k, T(1) - k.dt * sg, phi_.at(s)[ij], Cij * (tu - sg), u[ij + P] - u[ij - P]);
        psio.at(s)[ij] = ac_psi(k, T(1) - k.dt * tu, psi_.at(s)[ij], Cij * (tu - sg), u[ij + 1] - u[ij - 1]);
    }
}

// Per-shot source injection at level n (u[cell] += dt^2 * srcv[n-1, q] in source order,
// Core.jl:593-601).  One workgroup per shot; shots are in plan order.
template <typename T>
__global__ __launch_bounds__(256) void ac_add_sources(
    Lv<T> u_, int n, const int64_t *__restrict__ us_ptr, const int64_t *__restrict__ us_cell,
    const int64_t *__restrict__ us_eptr, const int64_t *__restrict__ us_ent, const T *__restrict__ srcv,
    const int64_t *__restrict__ srcv_off, const int64_t *__restrict__ nsrc, T dt2)
{
    const int s = blockIdx.x;
    T *__restrict__ u = u_.at(s);
    const T *__restrict__ row = srcv + srcv_off[s] + (int64_t)(n - 1) * nsrc[s];
    for (int64_t c = us_ptr[s] + threadIdx.x; c < us_ptr[s + 1]; c += blockDim.x) {
        const int64_t cell = us_cell[c];
        T acc = u[cell];
        for (int64_t e = us_eptr[c]; e < us_eptr[c + 1]; e++) acc += row[us_ent[e]] * dt2;
        u[cell] = acc;
    }
}

// Receiver sampling of a whole forward segment at once, trace[n, r] = u^n[rcv_r] for levels
// lo < n <= hi, from the checkpoint slot ring (level n in slot n mod NS; sources already added).
// Grid: (levels, shots).
template <typename T>
__global__ __launch_bounds__(256) void ac_record(const T *__restrict__ seg, int64_t NS, int64_t slot_stride,
                                                 int64_t npad, int64_t lo, const int64_t *__restrict__ nstep,
                                                 const int64_t *__restrict__ rcv_ptr,
                                                 const int64_t *__restrict__ rcv_cell, T *__restrict__ traces,
                                                 const int64_t *__restrict__ trace_off)
{
    const int64_t n = lo + 1 + blockIdx.x;
    const int s = blockIdx.y;
    if (nstep[s] < n) return;
    const T *__restrict__ u = seg + (n % NS) * slot_stride + (int64_t)s * npad;
    const int64_t r0 = rcv_ptr[s], nr = rcv_ptr[s + 1] - r0;
    T *__restrict__ tr = traces + trace_off[s] + n * nr;
    for (int64_t r = threadIdx.x; r < nr; r += blockDim.x) tr[r] = u[rcv_cell[r0 + r]];
}

// One level of the whole grid: workgroups [0, nfb) take the frame items (tile map fmap), the rest the
// rectangle tiles (a.map).
template <typename T, int RPT, int VEC, int SB, int V>
__global__ __launch_bounds__(WAVE *NWAVES) void ac_fwd_level(const FwdArgs<T> a, const Rect R,
                                                              const TileMap fmap,
                                                              const int4 *__restrict__ items,
                                                              int nitems, int nfb)
{
    const int b = (int)blockIdx.x;
    if (b < nfb) fwd_frame_body<T, V>(a, fmap, items, nitems, b);
    else fwd_rect_body<T, RPT, VEC, SB>(a, R, b - nfb);
}

// model (caller layout, (NX+2) x (NY+2)) -> C (pitched), squared if asked
template <typename T>
__global__ void k_model_in(const T *__restrict__ m, T *__restrict__ C, int NX, int NY, int P, int sq)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    if (j >= NY + 2) return;
    const T v = m[(int64_t)i * (NY + 2) + j];
    C[(int64_t)i * P + j] = sq ? v * v : v;
}

// one dense level of every shot into a history (shot stride hs)
template <typename T>
__global__ void k_level_copy(const T *__restrict__ src, T *__restrict__ dst, int64_t hs, int64_t n)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) dst[(int64_t)blockIdx.y * hs + q] = src[(int64_t)blockIdx.y * n + q];
}

// sum of the shot-group accumulators (pitched) -> gradient in caller layout (x 2m if squared)
template <typename T>
__global__ void k_grad_out(const T *__restrict__ gC, int64_t stride, int ngroups,
                           const T *__restrict__ m, T *__restrict__ g, int NX, int NY, int P, int sq)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    if (j >= NY + 2) return;
    const int64_t q = (int64_t)i * P + j, o = (int64_t)i * (NY + 2) + j;
    T acc = T(0);
    for (int s = 0; s < ngroups; s++) acc += gC[(int64_t)s * stride + q];
    g[o] = sq ? T(2) * m[o] * acc : acc;
}


// ---------------------------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------------------------
struct Shape {
    int rpt = 2, sg = 8, sb = 1;  // rows per wavefront, shots per workgroup, shots per batch
};

// Shape of the tile kernels: 8 wavefronts of 8 rows (plain tiles) or 4 rows (PML tiles, whose state is
// larger) by 64 columns.  Compared at 1000^2 x 32 shots FP32, each against the 8 / 4 of its time: forward us per
// level with 16 wavefronts of 4 / 4 rows 69 against 66, 8 / 8 rows 77, 4 / 4 rows 82, two columns per lane 67 (the
// adjoint 267 against 88).  5 and 6 rows of a PML tile: the whole gradient 84.6 and 99.0 ms against 82.5,
// and 200 x 66 x 8 shots FP64 18.0 and 26.7 against 15.6.
constexpr int TILE_WAVES = 8, TILE_RN = 8, TILE_RP = 4;

struct AcPlanBase {
    ads_acoustic_params p{};
    int dtype = ADS_F32;
    int variant = 0;  // 0 or 1
    int64_t NX = 0, NY = 0, Pitch = 0, Npad = 0, Ndense = 0, NMAX = 0, nshots = 0;
    std::vector<int64_t> order;         // plan position -> caller shot
    std::vector<int64_t> nstep_sorted;  // per plan position
    std::vector<int64_t> srcv_off_caller, trace_off_caller;  // per caller shot
    int64_t srcv_elems = 0, trace_elems = 0;
    std::vector<int> active;  // active[n] = #shots with nstep >= n
    std::vector<double> sx, ty;
    // phi/psi vanish on the quiet box (no damping profile acts there): checkpoint records keep
    // the nfr cells outside it
    FrameBox fbox{};
    int64_t nfr = 0;
    // snapshot slots of the reversal schedule (< 0: one per segment start, the one-level scheme)
    int64_t snapshots = -1;
    std::vector<uint8_t> pmlx, pmly, nearx, neary;
    double f_pml = 0.0;  // fraction of interior cells inside the PML strips
    // Single-level forward: rows per wavefront, shots per workgroup, shots per batch; adjoint: shots per
    // workgroup (its other entries have no effect)
    Shape fwd_shape{2, 16, 1}, adj_shape{2, 1, 1};
    int tuned = 0;
    // device tables (cells of the pitched layout)
    DevBuf d_sx, d_ty, d_pmlx, d_pmly, d_nearx, d_neary;
    DevBuf d_us_ptr, d_us_eptr, d_us_ent, d_us_cell, d_nsrc, d_srcv_off;
    DevBuf d_rcv_ptr, d_rcv_cell, d_trace_off, d_nstep_sorted;
    // single-level forward: the interior rectangle (columns rounded inwards to vectors) and the frame
    Rect rect{};
    DevBuf d_items;
    int nitems = 0;
    // blocking: levels per forward launch asked for (1: one, 2: the multi-level tiles); blk_ok: no source
    // lies in the rectangle, which is not empty.  blk_ok decides nothing here: ads_acoustic_plan_blocking
    // reports it
    bool blk_ok = false;
    int blocking = 2;
    // tiles of the multi-level kernels (plan and history layout) and their source / receiver lists
    int ntiles = 0;
    DevBuf d_tiles, d_ts_ptr, d_ts_cell, d_ts_ent, d_tr_ptr, d_tr_cell, d_tr_ent;
    DevBuf d_nstep32;
    int tile_levels = 4;  // levels per launch of the tile kernels (choose_levels)
    // hipGraph replay of whole checkpoint segments (forward sweep, recomputation, adjoint
    // sweep), keyed by everything the captured launches depend on
    struct GraphKey {
        int kind, record, set;  // set: the phi/psi buffer or adjoint state set that the segment starts from
        int64_t lo, hi, ns;  // ns: slots of the workspace layout (fixes every slot address)
        // model: the workspace's C, which lies behind the checkpoints and so moves with the snapshot count
        const void *ws, *model, *srcv, *traces, *resid;
        bool operator<(const GraphKey &o) const
        {
            return std::tie(kind, record, set, lo, hi, ns, ws, model, srcv, traces, resid) <
                   std::tie(o.kind, o.record, o.set, o.lo, o.hi, o.ns, o.ws, o.model, o.srcv, o.traces, o.resid);
        }
    };
    // A cached graph also records its last use: the key holds the caller's trace / residual
    // addresses, so fresh buffers on every FWI iteration would otherwise add graphs without
    // bound.  The cache keeps at most graph_cap() graphs and evicts the least recently used.
    struct CachedGraph {
        hipGraphExec_t exec;
        uint64_t used;
    };
    std::map<GraphKey, CachedGraph> graphs;
    uint64_t graph_clock = 0;
    hipStream_t cap_stream = nullptr;  // capture needs a stream other than the null stream
    int use_graph = 0;
    void drop_graphs()
    {
        if (!graphs.empty()) (void)hipDeviceSynchronize();  // none may still be executing
        for (auto &kv : graphs) (void)hipGraphExecDestroy(kv.second.exec);
        graphs.clear();
    }
    // one gradient's worth of segment graphs (forward, recomputation and adjoint sweeps of M
    // segments) for two buffer sets, so alternating calls keep their graphs
    static size_t graph_cap(int64_t M) { return (size_t)std::max<int64_t>(16, 6 * M + 8); }
    void evict_lru()
    {
        auto victim = graphs.begin();
        for (auto it = graphs.begin(); it != graphs.end(); ++it)
            if (it->second.used < victim->second.used) victim = it;
        (void)hipDeviceSynchronize();  // the evicted graph may still be executing
        (void)hipGraphExecDestroy(victim->second.exec);
        graphs.erase(victim);
    }
    // The histories step every shot over all NSTEP levels, so each record has to be that long; the shortest
    // is the last in plan order.
    int check_history() const
    {
        if (nstep_sorted.back() != p.NSTEP)
            ADS_FAIL(ADS_ERR_SHAPE, "history mode needs nstep == NSTEP for every shot (shot %lld has %lld of %lld)",
                     (long long)order.back(), (long long)nstep_sorted.back(), (long long)p.NSTEP);
        return ADS_OK;
    }
    virtual ~AcPlanBase()
    {
        drop_graphs();
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
    }
};

static int validate_params(const ads_acoustic_params *p)
{
    if (!p) ADS_FAIL(ADS_ERR_ARG, "null params");
    if (p->NX < 1 || p->NY < 1 || p->NSTEP < 1)
        ADS_FAIL(ADS_ERR_SHAPE, "NX, NY, NSTEP must be >= 1 (got %lld, %lld, %lld)",
                 (long long)p->NX, (long long)p->NY, (long long)p->NSTEP);
    if ((p->NX + 2) * (((p->NY + 2 + 63) / 64) * 64) >= (int64_t)1 << 31 || p->NX + 2 > (1 << 24))
        ADS_FAIL(ADS_ERR_SHAPE, "grid too large for 32-bit cell indexing within a shot");
    if (!(p->DELTAT > 0) || !(p->DELTAX > 0) || !(p->DELTAY > 0))
        ADS_FAIL(ADS_ERR_ARG, "DELTAT, DELTAX, DELTAY must be > 0");
    if (p->PropagatorKernel < 0 || p->PropagatorKernel > 2)
        ADS_FAIL(ADS_ERR_ARG, "PropagatorKernel must be 0, 1 or 2");
    return ADS_OK;
}

template <typename T> struct AcPlan : AcPlanBase {
    AcCoef<T> k;

    static unsigned grid_of(const TileMap &m) { return cdiv(m.nb, NXCD) * NXCD; }

    static constexpr int VECP = sizeof(T) == 4 ? 4 : 2;  // pitched layout: 16-byte vectors
    static TileMap tiles_of(int ntj, int nstrips, int ngroups) { return TileMap{ntj, nstrips, ngroups, ntj * nstrips * ngroups}; }
    static bool empty(const Rect &R) { return R.iR <= R.iL || R.jR <= R.jL; }
    // single-level launch: rows per wavefront 1/2/4, shots per batch 1/2 (2 with 1-2 rows)
    template <int RPT, int SB> void launch_level(FwdArgs<T> a, hipStream_t st)
    {
        const int ng = (int)cdiv(a.act, a.Sg);
        a.map = empty(rect) ? TileMap{}
                            : tiles_of((int)cdiv(rect.jR - rect.jL, WAVE * VECP), (int)cdiv(rect.iR - rect.iL, NWAVES * RPT), ng);
        const TileMap fm = tiles_of(1, nitems, ng);
        const int nfb = (int)grid_of(fm);
        const unsigned nb = (unsigned)nfb + grid_of(a.map);
        const int4 *it = d_items.as<int4>();
        if (nb == 0) return;
        if (variant == 1) ac_fwd_level<T, RPT, VECP, SB, 1><<<nb, WAVE * NWAVES, 0, st>>>(a, rect, fm, it, nitems, nfb);
        else ac_fwd_level<T, RPT, VECP, SB, 0><<<nb, WAVE * NWAVES, 0, st>>>(a, rect, fm, it, nitems, nfb);
    }
    void launch_shape(const FwdArgs<T> &a, const Shape &sh, hipStream_t st)
    {
        if (sh.sb == 2 && sh.rpt == 1) launch_level<1, 2>(a, st);
        else if (sh.sb == 2 && sh.rpt == 2) launch_level<2, 2>(a, st);
        else if (sh.rpt == 1) launch_level<1, 1>(a, st);
        else if (sh.rpt == 4) launch_level<4, 1>(a, st);
        else launch_level<2, 1>(a, st);
    }

    // What a launch has to move, for the profile: one value per interior cell and shot
    double cell_bytes() const { return (double)NX * (double)NY * sizeof(T); }
    double fwd_level_bytes(int act) const  // single-level forward
    {
        return (double)act * cell_bytes() * (4.0 + (variant == 1 ? 4.0 : 2.0) * f_pml);
    }
    int64_t group_arrays() const { return (int64_t)cdiv(nshots, adj_shape.sg); }

    // ---- workspace layout for checkpoint interval K ----
    struct WS {
        int64_t K, NS, M, S;  // interval, slots, segments, snapshot slots
        // P^{n+1}, P^{n+2}, F^{n+1}, G^{n+1} in two sets: an adjoint launch reads one and writes the other
        T *seg, *phi[2], *psi[2], *P[4], *F[2], *G[2], *gC, *ckpt, *C, *resid;
        double *loss, *part;
        std::vector<size_t> ck_off;  // element offset of each snapshot slot in ckpt
        // The buffer that holds phi/psi of the level that the next forward launch starts from.  State of one
        // call, like the rest of this struct: several threads may run a plan, each on its own workspace.
        int cur = 0;
    };
    int64_t seg_level(const WS &w, int64_t m) const { return std::min<int64_t>(1 + m * w.K, NMAX); }
    int64_t snap_slots(int64_t M, int64_t snaps) const
    {
        const int64_t one = std::max<int64_t>(M - 1, 0);
        return snaps < 0 ? one : std::min(snaps, one);
    }
    // a record of the state at level a for `act` shots: u^a, u^{a-1} (full grid), phi^a and
    // psi^a (cells outside the quiet box)
    size_t rec_elems(int act) const { return (size_t)act * (2 * (size_t)Npad + 2 * (size_t)nfr); }
    int rec_act(int64_t a) const { return active[std::min<int64_t>(a + 1, NMAX)]; }
    int64_t seg_count(int64_t K) const { return NMAX >= 2 ? (NMAX - 1 + K - 1) / K : 0; }
    void layout(WS &w, Carve &cv, int64_t K) const { layout(w, cv, K, snapshots); }
    void layout(WS &w, Carve &cv, int64_t K, int64_t snaps) const
    {
        if (K < 1) K = 1;
        if (K > std::max<int64_t>(NMAX - 1, 1)) K = std::max<int64_t>(NMAX - 1, 1);
        w.K = K;
        w.M = seg_count(K);
        w.NS = std::min<int64_t>(K + 2, NMAX + 1);
        const size_t F = (size_t)nshots * Npad * sizeof(T);
        w.seg = (T *)cv.take(F * w.NS);
        for (int q = 0; q < 2; q++) {
            w.phi[q] = (T *)cv.take(F);
            w.psi[q] = (T *)cv.take(F);
        }
        for (int q = 0; q < 4; q++) w.P[q] = (T *)cv.take(F);
        for (int q = 0; q < 2; q++) {
            w.F[q] = (T *)cv.take(F);
            w.G[q] = (T *)cv.take(F);
        }
        w.gC = (T *)cv.take((size_t)nshots * Npad * sizeof(T));  // up to one array per shot
        // snapshot slots: one-level, slot q holds state q+1 and is sized for the shots active
        // there; binomial, any slot may hold any state and is sized for the most active shots
        w.S = snap_slots(w.M, snaps);
        w.ck_off.assign((size_t)w.S, 0);
        size_t ck = 0;
        for (int64_t q = 0; q < w.S; q++) {
            w.ck_off[q] = ck;
            const int64_t a = w.S >= w.M - 1 ? 1 + (q + 1) * w.K : 1 + w.K;
            ck += (rec_elems(rec_act(a)) + 63) & ~size_t(63);
        }
        w.ckpt = (T *)cv.take(ck * sizeof(T));
        w.C = (T *)cv.take((size_t)Npad * sizeof(T));
        w.resid = (T *)cv.take((size_t)std::max<int64_t>(trace_elems, 1) * sizeof(T));
        w.loss = (double *)cv.take(64);
        w.part = (double *)cv.take(MISFIT_BLOCKS * sizeof(double));
    }
    Lv<T> phl(const WS &w, int q) const { return Lv<T>{w.phi[q], Npad}; }
    Lv<T> psl(const WS &w, int q) const { return Lv<T>{w.psi[q], Npad}; }
    size_t ws_size(int64_t K) const { return ws_size(K, snapshots); }
    size_t ws_size(int64_t K, int64_t snaps) const
    {
        WS w;
        Carve cv(nullptr, 0);
        layout(w, cv, K, snaps);
        return cv.off + 256;
    }

    // Fastest (K, S) whose workspace fits `budget`.  Cost model in shot-levels: the forward
    // and the adjoint sweep each pass every active shot's levels once (an adjoint level costs
    // ADJ_COST forward levels: 451 / 337 us at 2000^2 x 64 shots FP32, 94 / 63 at 1000^2 x 32), and the
    // reversal schedule adds its segment rebuilds, which alone rank the schedules.
    static constexpr double ADJ_COST = 1.4;
    int choose_schedule(size_t budget, int64_t *Kout, int64_t *Sout) const
    {
        double total = 0.0;
        for (int64_t n = 2; n <= NMAX; n++) total += active[n];
        auto ws = [&](int64_t K, int64_t S) { return ws_size(K, S); };
        auto work = [&](int64_t K, int64_t M) {
            std::vector<double> w((size_t)M, 0.0);
            for (int64_t m = 0; m < M; m++) {
                const int64_t a = std::min<int64_t>(1 + m * K, NMAX), b = std::min<int64_t>(a + K, NMAX);
                for (int64_t n = a + 1; n <= b; n++) w[m] += active[n];
            }
            return w;
        };
        return ads::choose_schedule(budget, NMAX - 1, total, ADJ_COST, ws, work, *Kout, *Sout)
                   ? ADS_OK
                   : ADS_ERR_WORKSPACE;
    }

    Lv<T> slot(const WS &w, int64_t n) const
    {
        return Lv<T>{w.seg + (size_t)(n % w.NS) * nshots * Npad, Npad};
    }

    int prepare_C(T *C, const void *model, int P, hipStream_t st)
    {
        k_model_in<T><<<dim3(cdiv(NY + 2, 256), NX + 2), 256, 0, st>>>((const T *)model, C, (int)NX,
                                                                      (int)NY, P, p.square_velocity);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    // Runs body(stream) directly, or -- with graphs on and no event profiling -- captures it
    // once on a private stream into a graph and replays that graph on st.
    template <class F> int replay(const GraphKey &key, int64_t M, hipStream_t st, F &&body)
    {
        if (!use_graph || prof_enabled()) return body(st);
        auto it = graphs.find(key);
        if (it == graphs.end()) {
            while (!graphs.empty() && graphs.size() >= graph_cap(M)) evict_lru();
            if (!cap_stream) ADS_HIP(hipStreamCreateWithFlags(&cap_stream, hipStreamNonBlocking));
            ADS_HIP(hipStreamBeginCapture(cap_stream, hipStreamCaptureModeThreadLocal));
            const int rc = body(cap_stream);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(cap_stream, &g);
            if (rc != ADS_OK) {
                if (g) (void)hipGraphDestroy(g);
                return rc;
            }
            ADS_HIP(e);
            hipGraphExec_t ex = nullptr;
            const hipError_t ei = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            ADS_HIP(ei);
            it = graphs.emplace(key, CachedGraph{ex, 0}).first;
        }
        it->second.used = ++graph_clock;
        ADS_HIP(hipGraphLaunch(it->second.exec, st));
        return ADS_OK;
    }

    // one level: the stencil, phi/psi from the new u (kernel 0), sources
    int fwd_step(WS &w, int n, const T *srcv, hipStream_t st, const Shape &shape)
    {
        const int act = active[n], cur = w.cur;
        if (act <= 0) return ADS_OK;
        w.cur ^= 1;
        FwdArgs<T> a{slot(w, n), cst(slot(w, n - 1)), cst(slot(w, n - 2)), cst(phl(w, cur)), cst(psl(w, cur)),
                     phl(w, cur ^ 1), psl(w, cur ^ 1), w.C, d_sx.as<T>(), d_ty.as<T>(), d_nearx.as<uint8_t>(),
                     d_neary.as<uint8_t>(), (int)NX, (int)NY, (int)Pitch, act, std::min(shape.sg, act), TileMap{}, k};
        int pr = prof_start(ADS_PROF_AC_FWD, st);
        launch_shape(a, shape, st);
        prof_stop(pr, st, fwd_level_bytes(act));
        if (variant == 0 && nitems > 0)
            ac_fwd_phipsi<T><<<dim3((unsigned)nitems, cdiv(act, NWAVES)), 256, 0, st>>>(
                cst(a.u), a.phi, a.psi, a.phio, a.psio, a.C, d_sx.as<T>(), d_ty.as<T>(), d_pmlx.as<uint8_t>(),
                d_pmly.as<uint8_t>(), (int)NX, (int)NY, (int)Pitch, k, d_items.as<int4>(), act);
        ac_add_sources<T><<<act, 256, 0, st>>>(a.u, n, d_us_ptr.as<int64_t>(), d_us_cell.as<int64_t>(),
                                               d_us_eptr.as<int64_t>(), d_us_ent.as<int64_t>(), srcv,
                                               d_srcv_off.as<int64_t>(), d_nsrc.as<int64_t>(), k.dt2);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    // forward over levels lo+1..hi from the state held in slots/phi (record traces if asked)
    int run_forward(WS &w, int64_t lo, int64_t hi, const T *srcv, T *traces, int record, hipStream_t st,
                    const Shape *sh = nullptr)
    {
        if (sh) return run_forward_levels(w, lo, hi, srcv, traces, record, st, sh);
        GraphKey key{0, record, w.cur, lo, hi, w.NS, w.seg, w.C, srcv, traces, nullptr};
        const int end = w.cur ^ (fwd_launches(lo, hi) & 1);
        ADS_TRY(replay(key, w.M, st, [&](hipStream_t s) { return run_forward_levels(w, lo, hi, srcv, traces, record, s); }));
        w.cur = end;
        return ADS_OK;
    }
    void tile_common(TileCommon<T> &a, const T *C, int P, int act, const T *srcv) const
    {
        a.tiles = d_tiles.as<int4>();
        a.ntiles = ntiles;
        a.act = act;
        a.NX = (int)NX;
        a.NY = (int)NY;
        a.P = P;
        a.k = k;
        a.C = C;
        a.sx = d_sx.as<T>();
        a.ty = d_ty.as<T>();
        a.nearx = d_nearx.as<uint8_t>();
        a.neary = d_neary.as<uint8_t>();
        a.nstep = d_nstep32.as<int32_t>();
        a.src = PointList{d_ts_ptr.as<int32_t>(), d_ts_cell.as<int2>(), d_ts_ent.as<int32_t>()};
        a.srcv = srcv;
        a.srcv_off = d_srcv_off.as<int64_t>();
        a.nsrc = d_nsrc.as<int64_t>();
    }
    // Each of a launch's first `act` shots has to have the launch's level `lo`, the first that the forward
    // steps and the last of the adjoint: the kernels count their levels from there on.  Looked at here: one
    // branch for it in the adjoint tile kernel cost 2 % of a 1000^2 gradient (other scalar spills).
    int check_levels(int act, int lo) const
    {
        if (act < 1 || act > nshots || nstep_sorted[act - 1] < lo)
            ADS_FAIL(ADS_ERR_SHAPE, "a shot of the launch has no level %d", lo);
        return ADS_OK;
    }
    int launch_fwd_tile(FwdTile<T> &a, hipStream_t st)
    {
        ADS_TRY(check_levels(a.act, a.n));
        a.nb = a.ntiles * a.act;
        const unsigned nb = cdiv(a.nb, NXCD) * NXCD;
        double levels = 0.0;
        for (int q = 0; q < a.nt; q++) levels += active[a.n + q];
        int pr = prof_start(ADS_PROF_AC_FWD, st);
        if (variant == 1) ac_fwd_tile<T, 1, TILE_RN, TILE_RP, TILE_WAVES><<<nb, TILE_WAVES * WAVE, 0, st>>>(a);
        else ac_fwd_tile<T, 0, TILE_RN, TILE_RP, TILE_WAVES><<<nb, TILE_WAVES * WAVE, 0, st>>>(a);
        // per launch: u^{n-1}, u^{n-2}, C and phi/psi once, phi/psi back once, every level's u
        prof_stop(pr, st, cell_bytes() * (levels + a.act * (3.0 + 4.0 * f_pml)), a.nt);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }
    // one adjoint launch: levels a.n down to a.n - a.nt + 1
    template <bool DENSE> int launch_adj_tile(AdjTile<T> &a, hipStream_t st)
    {
        ADS_TRY(check_levels(a.act, a.n - a.nt + 1));
        a.Sg = std::min(adj_shape.sg, a.act);  // (any count is accepted; the kernel adds it to act)
        a.nb = a.ntiles * (int)cdiv(a.act, a.Sg);
        const unsigned nb = cdiv(a.nb, NXCD) * NXCD;
        double levels = 0.0;
        for (int q = 0; q < a.nt; q++) levels += active[a.n - q];
        int pr = prof_start(ADS_PROF_AC_ADJ, st);
        if (variant == 1) ac_adj_tile<T, 1, TILE_RN, TILE_RP, TILE_WAVES, DENSE><<<nb, TILE_WAVES * WAVE, 0, st>>>(a);
        else ac_adj_tile<T, 0, TILE_RN, TILE_RP, TILE_WAVES, DENSE><<<nb, TILE_WAVES * WAVE, 0, st>>>(a);
        // per launch: P^{n+1}, P^{n+2} and F/G in and out, C and dL/dC in and out once per group of shots, and
        // every level's u (kernel 0's PML: one more) and dense cotangent
        const double per_shot = 4.0 + (variant == 1 ? 4.0 : 5.0) * f_pml;
        prof_stop(pr, st, cell_bytes() * ((DENSE ? 2.0 : 1.0) * levels + a.act * per_shot + 3.0 * cdiv(a.act, a.Sg)), a.nt);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }
    // Adjoint of levels hi .. lo + 1 of the plan layout from state set `set`; launches toggle the set.
    int adj_launches(int64_t lo, int64_t hi) const { return (int)cdiv(hi - lo, tile_levels); }
    int adj_levels(const WS &w, int64_t lo, int64_t hi, int set, const T *srcv, const T *resid, hipStream_t st)
    {
        for (int64_t n = hi; n > lo; set ^= 1) {
            AdjTile<T> a{};
            a.n = (int)n;
            a.nt = (int)std::min<int64_t>(tile_levels, n - lo);
            n -= a.nt;
            const int act = active[n + 1];
            if (act <= 0) continue;
            tile_common(a, w.C, (int)Pitch, act, srcv);
            a.u = w.seg;
            a.lstride = nshots * Npad;
            a.sstride = Npad;
            a.NS = (int)w.NS;
            a.P1 = w.P[2 * set];
            a.P2 = w.P[2 * set + 1];
            a.F = w.F[set];
            a.G = w.G[set];
            a.P1o = w.P[2 * (set ^ 1)];
            a.P2o = w.P[2 * (set ^ 1) + 1];
            a.Fo = w.F[set ^ 1];
            a.Go = w.G[set ^ 1];
            a.fstride = Npad;
            a.gC = w.gC;
            a.gstride = Npad;
            a.rcv = PointList{d_tr_ptr.as<int32_t>(), d_tr_cell.as<int2>(), d_tr_ent.as<int32_t>()};
            a.resid = resid;
            a.trace_off = d_trace_off.as<int64_t>();
            a.rcv_ptr = d_rcv_ptr.as<int64_t>();
            ADS_TRY(launch_adj_tile<false>(a, st));
        }
        return ADS_OK;
    }
    // launches that move phi/psi on over levels lo+1..hi (levels without active shots launch nothing)
    int fwd_launches(int64_t lo, int64_t hi) const
    {
        const int step = blocking == 2 ? tile_levels : 1;
        int n = 0;
        for (int64_t l = lo + 1; l <= hi; l += step) n += active[l] > 0;
        return n;
    }
    int run_forward_levels(WS &w, int64_t lo, int64_t hi, const T *srcv, T *traces, int record, hipStream_t st,
                           const Shape *sh = nullptr)
    {
        if (blocking == 1 || sh) {
            for (int64_t n = lo + 1; n <= hi; n++) ADS_TRY(fwd_step(w, (int)n, srcv, st, sh ? *sh : fwd_shape));
        } else {
            for (int64_t n = lo + 1; n <= hi; n += tile_levels) {
                if (active[n] <= 0) continue;
                FwdTile<T> a{};
                tile_common(a, w.C, (int)Pitch, active[n], srcv);
                a.u = w.seg;
                a.lstride = nshots * Npad;
                a.sstride = Npad;
                a.NS = (int)w.NS;
                a.n = (int)n;
                a.nt = (int)std::min<int64_t>(tile_levels, hi - n + 1);
                a.phi = w.phi[w.cur];
                a.psi = w.psi[w.cur];
                a.phio = w.phi[w.cur ^ 1];
                a.psio = w.psi[w.cur ^ 1];
                a.fstride = Npad;
                w.cur ^= 1;
                ADS_TRY(launch_fwd_tile(a, st));
            }
        }
        if (record && traces && hi > lo && trace_elems > 0) {
            ac_record<T><<<dim3((unsigned)(hi - lo), (unsigned)nshots), 256, 0, st>>>(
                w.seg, w.NS, nshots * Npad, Npad, lo, d_nstep_sorted.as<int64_t>(), d_rcv_ptr.as<int64_t>(),
                d_rcv_cell.as<int64_t>(), traces, d_trace_off.as<int64_t>());
            ADS_LAUNCH_CHECK();
        }
        return ADS_OK;
    }

    int frame_copy(bool unpack, Lv<T> f, T *rec, int act, hipStream_t st)
    {
        if (nfr <= 0 || act <= 0) return ADS_OK;
        const dim3 g(cdiv(nfr, 256), (unsigned)act);
        if (unpack) k_frame_copy<T, true><<<g, 256, 0, st>>>(f.p, Npad, rec, fbox, (int)Pitch);
        else k_frame_copy<T, false><<<g, 256, 0, st>>>(f.p, Npad, rec, fbox, (int)Pitch);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    // state at level a (u^a, u^{a-1}, phi^a, psi^a; active shots are a prefix) into slot q
    int save_ckpt(const WS &w, int64_t q, int64_t a, hipStream_t st)
    {
        const int act = rec_act(a);
        const size_t U = (size_t)act * Npad, R = (size_t)act * nfr;
        T *dst = w.ckpt + w.ck_off[q];
        ADS_HIP(hipMemcpyAsync(dst, slot(w, a).p, U * sizeof(T), hipMemcpyDeviceToDevice, st));
        ADS_HIP(hipMemcpyAsync(dst + U, slot(w, a - 1).p, U * sizeof(T), hipMemcpyDeviceToDevice, st));
        ADS_TRY(frame_copy(false, phl(w, w.cur), dst + 2 * U, act, st));
        ADS_TRY(frame_copy(false, psl(w, w.cur), dst + 2 * U + R, act, st));
        return ADS_OK;
    }

    // slot q (q < 0: the zero state at level 1) back into the slot ring and phi/psi buffers.
    // The buffers' quiet-box cells are zero: every forward clears them and no pass writes a
    // non-zero value there.
    int restore_ckpt(const WS &w, int64_t q, int64_t a, hipStream_t st)
    {
        const int act = rec_act(a);
        const size_t U = (size_t)act * Npad, R = (size_t)act * nfr;
        if (q < 0) {
            ADS_HIP(hipMemsetAsync(slot(w, 0).p, 0, U * sizeof(T), st));
            ADS_HIP(hipMemsetAsync(slot(w, 1).p, 0, U * sizeof(T), st));
            ADS_HIP(hipMemsetAsync(phl(w, w.cur).p, 0, U * sizeof(T), st));
            ADS_HIP(hipMemsetAsync(psl(w, w.cur).p, 0, U * sizeof(T), st));
            return ADS_OK;
        }
        const T *src = w.ckpt + w.ck_off[q];
        ADS_HIP(hipMemcpyAsync(slot(w, a).p, src, U * sizeof(T), hipMemcpyDeviceToDevice, st));
        ADS_HIP(hipMemcpyAsync(slot(w, a - 1).p, src + U, U * sizeof(T), hipMemcpyDeviceToDevice, st));
        ADS_TRY(frame_copy(true, phl(w, w.cur), const_cast<T *>(src) + 2 * U, act, st));
        ADS_TRY(frame_copy(true, psl(w, w.cur), const_cast<T *>(src) + 2 * U + R, act, st));
        return ADS_OK;
    }

    int check_ws(WS &w, void *ws, size_t wsb, int64_t K)
    {
        Carve cv(ws, wsb);
        layout(w, cv, K);
        if (!ws || !cv.ok())
            ADS_FAIL(ADS_ERR_WORKSPACE, "workspace too small: need %zu bytes, got %zu", cv.off, wsb);
        return ADS_OK;
    }

    int forward(const void *model, const void *srcv, void *traces, void *ws, size_t wsb,
                int64_t K, hipStream_t st)
    {
        WS w;
        ADS_TRY(check_ws(w, ws, wsb, K));
        const size_t F = (size_t)nshots * Npad * sizeof(T);
        ADS_TRY(prepare_C(w.C, model, (int)Pitch, st));
        ADS_HIP(hipMemsetAsync(slot(w, 0).p, 0, F, st));
        ADS_HIP(hipMemsetAsync(slot(w, 1).p, 0, F, st));
        for (int q = 0; q < 2; q++) {
            ADS_HIP(hipMemsetAsync(w.phi[q], 0, F, st));
            ADS_HIP(hipMemsetAsync(w.psi[q], 0, F, st));
        }
        if (traces && trace_elems) ADS_HIP(hipMemsetAsync(traces, 0, trace_elems * sizeof(T), st));
        // the reversal schedule's first descent: the states it keeps, in level order
        Reversal rv(w.M, w.S);
        const auto path = rv.first_path();
        size_t pi = 0;
        for (int64_t m = 0; m < w.M; m++) {
            const int64_t a = seg_level(w, m), b = seg_level(w, m + 1);
            if (pi < path.size() && path[pi].first == m) ADS_TRY(save_ckpt(w, path[pi++].second, a, st));
            ADS_TRY(run_forward(w, a, b, (const T *)srcv, (T *)traces, traces != nullptr, st));
        }
        return ADS_OK;
    }

    int zero_adjoint_state(const WS &w, hipStream_t st)
    {
        const size_t F = (size_t)nshots * Npad * sizeof(T);
        for (int q = 0; q < 4; q++) ADS_HIP(hipMemsetAsync(w.P[q], 0, F, st));
        for (int q = 0; q < 2; q++) {
            ADS_HIP(hipMemsetAsync(w.F[q], 0, F, st));
            ADS_HIP(hipMemsetAsync(w.G[q], 0, F, st));
        }
        ADS_HIP(hipMemsetAsync(w.gC, 0, (size_t)group_arrays() * Npad * sizeof(T), st));
        return ADS_OK;
    }

    int backward(const void *model, const void *srcv, const T *resid, void *grad, void *ws,
                 size_t wsb, int64_t K, hipStream_t st)
    {
        WS w;
        ADS_TRY(check_ws(w, ws, wsb, K));
        ADS_TRY(zero_adjoint_state(w, st));
        const T *sv = (const T *)srcv;
        struct Ops {
            AcPlan *pl;
            WS &w;
            const T *sv, *resid;
            hipStream_t st;
            int set;  // state set of the next adjoint launch
            int restore(int64_t m, int64_t q) { return pl->restore_ckpt(w, q, pl->seg_level(w, m), st); }
            int save(int64_t m, int64_t q) { return pl->save_ckpt(w, q, pl->seg_level(w, m), st); }
            int forward(int64_t m0, int64_t m1)  // segment by segment: one cached graph each
            {
                for (int64_t m = m0; m < m1; m++)
                    ADS_TRY(pl->run_forward(w, pl->seg_level(w, m), pl->seg_level(w, m + 1), sv, nullptr, 0, st));
                return ADS_OK;
            }
            int adjoint(int64_t m)
            {
                const int64_t a = pl->seg_level(w, m), b = pl->seg_level(w, m + 1);
                GraphKey key{1, 0, set, a, b, w.NS, w.seg, w.C, sv, nullptr, resid};
                ADS_TRY(pl->replay(key, w.M, st, [&](hipStream_t s) { return pl->adj_levels(w, a, b, set, sv, resid, s); }));
                set ^= pl->adj_launches(a, b) & 1;
                return ADS_OK;
            }
        } ops{this, w, sv, resid, st, 0};
        Reversal rv(w.M, w.S);
        ADS_TRY(rv.run(ops));
        k_grad_out<T><<<dim3(cdiv(NY + 2, 256), NX + 2), 256, 0, st>>>(
            w.gC, Npad, (int)group_arrays(), (const T *)model, (T *)grad, (int)NX, (int)NY,
            (int)Pitch, p.square_velocity);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    int misfit(const WS &w, const T *traces, const T *obs, hipStream_t st)
    {
        launch_misfit<T>(traces, obs, w.resid, trace_elems, w.part, w.loss, st);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    // ---- autotuner: times the single-level forward's shapes and the adjoint tiles' shot groups ----
    int autotune(const void *model, const void *srcv, void *ws, size_t wsb, int64_t K, int reps,
                 hipStream_t st)
    {
        drop_graphs();  // captured segments embed the kernel shapes
        WS w;
        ADS_TRY(check_ws(w, ws, wsb, K));
        if (NMAX < 3) {  // nothing worth timing
            tuned = 1;
            return ADS_OK;
        }
        const T *sv = (const T *)srcv;
        ADS_TRY(prepare_C(w.C, model, (int)Pitch, st));
        const size_t F = (size_t)nshots * Npad * sizeof(T);
        for (int64_t q = 0; q < std::min<int64_t>(w.NS, 4); q++) ADS_HIP(hipMemsetAsync(slot(w, q).p, 0, F, st));
        for (int q = 0; q < 2; q++) {
            ADS_HIP(hipMemsetAsync(w.phi[q], 0, F, st));
            ADS_HIP(hipMemsetAsync(w.psi[q], 0, F, st));
        }
        const int rpts[3] = {1, 2, 4};
        std::vector<int> sgs;
        for (int sg = 1; sg <= std::max<int64_t>(nshots, 1) && sg <= 32; sg *= 2) sgs.push_back(sg);
        if (reps < 1) reps = 3;
        hipEvent_t e0, e1;
        ADS_HIP(hipEventCreate(&e0));
        ADS_HIP(hipEventCreate(&e1));
        auto timeit = [&](auto &&body) -> float {
            body();  // warm
            (void)hipEventRecord(e0, st);
            for (int r = 0; r < reps; r++) body();
            (void)hipEventRecord(e1, st);
            (void)hipEventSynchronize(e1);
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            return ms;
        };
        int64_t n0 = std::min<int64_t>(2, NMAX);
        float best = 1e30f;
        Shape bf = fwd_shape;
        for (int rp : rpts)
            for (int sg : sgs)
                for (int sb = 1; sb <= std::min(2, sg); sb++) {
                    if (sb == 2 && rp >= 4) continue;
                    Shape sh{rp, sg, sb};
                    float ms = timeit([&] { (void)run_forward(w, n0 - 1, n0 + 1 <= NMAX ? n0 + 1 : n0, sv, nullptr, 0, st, &sh); });
                    if (ms < best) best = ms, bf = sh;
                }
        fwd_shape = bf;
        ADS_TRY(zero_adjoint_state(w, st));
        if (trace_elems) ADS_HIP(hipMemsetAsync(w.resid, 0, (size_t)trace_elems * sizeof(T), st));
        best = 1e30f;
        int bs = adj_shape.sg;
        const int64_t top = std::min<int64_t>(NMAX, 1 + std::min<int64_t>(w.K, tile_levels));
        for (int sg : sgs) {
            adj_shape.sg = sg;
            float ms = timeit([&] { (void)adj_levels(w, 1, top, 0, sv, w.resid, st); });
            if (ms < best) best = ms, bs = sg;
        }
        adj_shape.sg = bs;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        tuned = 1;
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }

    // ---- full-history drop-in (every shot has NSTEP levels, dense caller layout) ----
    int forward_history(const void *model, const void *srcv, void *u_hist, void *phi_hist,
                        void *psi_hist, void *scratch, hipStream_t st)
    {
        const int pitch = (int)(NY + 2);
        const int64_t Lv_ = NMAX + 1;
        const size_t H = (size_t)nshots * Lv_ * Ndense * sizeof(T);
        T *C = (T *)scratch;
        const size_t F = (size_t)nshots * Ndense;
        T *pp[2] = {(T *)scratch + Ndense, (T *)scratch + Ndense + F};
        T *qq[2] = {(T *)scratch + Ndense + 2 * F, (T *)scratch + Ndense + 3 * F};
        ADS_TRY(prepare_C(C, model, pitch, st));
        const int64_t hs = Lv_ * Ndense;
        // levels 0 and 1; every later level is written whole
        ADS_HIP(hipMemset2DAsync(u_hist, hs * sizeof(T), 0, (size_t)std::min<int64_t>(2, Lv_) * Ndense * sizeof(T),
                                 (size_t)nshots, st));
        if (phi_hist) ADS_HIP(hipMemsetAsync(phi_hist, 0, H, st));
        if (psi_hist) ADS_HIP(hipMemsetAsync(psi_hist, 0, H, st));
        // Both auxiliary histories: the tiles write every level into them.  Neither: two scratch buffers of
        // each, toggled by every launch.  One alone: the buffers with a level per launch, and a copy of the
        // level (a shot stride of its own for each of the two costs the tile kernel 3 to 5 %: scalar spills).
        const bool aux = phi_hist && psi_hist;
        T *one = aux ? nullptr : (T *)(phi_hist ? phi_hist : psi_hist);
        if (!aux)
            for (int q = 0; q < 2; q++) {
                ADS_HIP(hipMemsetAsync(pp[q], 0, F * sizeof(T), st));
                ADS_HIP(hipMemsetAsync(qq[q], 0, F * sizeof(T), st));
            }
        int set = 0;
        for (int64_t n = 2; n <= NMAX; set ^= 1) {
            FwdTile<T> a{};
            tile_common(a, C, pitch, (int)nshots, (const T *)srcv);
            a.u = (T *)u_hist;
            a.lstride = Ndense;
            a.sstride = hs;
            a.NS = std::numeric_limits<int>::max();
            a.n = (int)n;
            a.nt = one ? 1 : (int)std::min<int64_t>(tile_levels, NMAX - n + 1);
            a.phi = aux ? (const T *)phi_hist + (n - 1) * Ndense : pp[set];
            a.psi = aux ? (const T *)psi_hist + (n - 1) * Ndense : qq[set];
            a.phio = aux ? (T *)phi_hist + n * Ndense : pp[set ^ 1];
            a.psio = aux ? (T *)psi_hist + n * Ndense : qq[set ^ 1];
            a.fstride = aux ? hs : Ndense;
            a.plstride = aux ? Ndense : 0;
            ADS_TRY(launch_fwd_tile(a, st));
            if (one) {
                k_level_copy<T><<<dim3(cdiv(Ndense, 256), (unsigned)nshots), 256, 0, st>>>(
                    phi_hist ? a.phio : a.psio, one + n * Ndense, hs, Ndense);
                ADS_LAUNCH_CHECK();
            }
            n += a.nt;
        }
        return ADS_OK;
    }

    int backward_history(const void *model, const void *srcv, const void *u_hist,
                         const void *g_hist, void *grad, void *scratch, hipStream_t st)
    {
        const int pitch = (int)(NY + 2);
        const int64_t Lv_ = NMAX + 1;
        const size_t F = (size_t)nshots * Ndense;
        T *C = (T *)scratch;
        T *b = (T *)scratch + Ndense;
        T *P[4] = {b, b + F, b + 2 * F, b + 3 * F}, *Fa[2] = {b + 4 * F, b + 5 * F}, *Ga[2] = {b + 6 * F, b + 7 * F};
        T *gC = b + 8 * F;
        ADS_TRY(prepare_C(C, model, pitch, st));
        ADS_HIP(hipMemsetAsync(b, 0, 9 * F * sizeof(T), st));
        const int64_t hs = Lv_ * Ndense;
        int set = 0;
        for (int64_t n = NMAX; n >= 2; set ^= 1) {
            AdjTile<T> a{};
            tile_common(a, C, pitch, (int)nshots, (const T *)srcv);
            a.u = (T *)u_hist;
            a.lstride = Ndense;
            a.sstride = hs;
            a.NS = std::numeric_limits<int>::max();
            a.n = (int)n;
            a.nt = (int)std::min<int64_t>(tile_levels, n - 1);
            n -= a.nt;
            a.P1 = P[2 * set];
            a.P2 = P[2 * set + 1];
            a.F = Fa[set];
            a.G = Ga[set];
            a.P1o = P[2 * (set ^ 1)];
            a.P2o = P[2 * (set ^ 1) + 1];
            a.Fo = Fa[set ^ 1];
            a.Go = Ga[set ^ 1];
            a.fstride = Ndense;
            a.gC = gC;
            a.gstride = Ndense;
            a.dense = (const T *)g_hist;
            ADS_TRY(launch_adj_tile<true>(a, st));
        }
        k_grad_out<T><<<dim3(cdiv(NY + 2, 256), NX + 2), 256, 0, st>>>(
            gC, Ndense, (int)group_arrays(), (const T *)model, (T *)grad, (int)NX, (int)NY, pitch,
            p.square_velocity);
        ADS_LAUNCH_CHECK();
        return ADS_OK;
    }
    size_t history_scratch() const { return ((size_t)Ndense + 9 * (size_t)nshots * Ndense) * sizeof(T); }
};

// The tiles of the multi-level kernels and their point lists.
// Levels per launch.  More levels read and write the state and launch less often, but widen the halo (by
// one cell a level, kernel 0's PML by two) and so need more tiles.
// Where all workgroups of an adjoint launch are on the card at once (one per CU in FP64, two in FP32) a
// launch takes as long as one of them, and the more levels the better: the most that still fit.  ms of a
// call with kernel 0 for 4 / 5 / 6 / 7 levels (largest that fits in brackets): 200^2 solver FP64 9.8 / 9.0 /
// 8.3 / [7.9]; 300 x 280 solver FP64 4.8 / 4.7 / [4.4] / 5.6; 1501 x 401 forward FP32 3.25 / [2.9] / 3.4 /
// 4.6; 200 x 66, 8 shots, FP64 [15.6] / 21.0 / 19.4 / 30.9; 300 x 200, 1 shot, FP32 2.4 / 2.2 / 2.0 / [1.9].
// Beyond that the work counts: the tiles, a PML tile at 2.2 of a plain one (half the rows, four times the
// instructions), per level.  ms for 3 / 4 levels, the model's choice in brackets: 400 x 800, 24 shots, FP32
// [31.7] / 33.9; 1000^2, 32 shots, FP32 24.2 / [22.4]; 700 x 600, 16 shots, FP64 10.4 / [10.0].  Kernel 1
// takes 7: us per level, forward + adjoint, for 5 / 6 / 7 / 8 / 10 levels at 1000^2 x 32 shots FP32 66 + 99, 65 +
// 101, 63 + 101, 63 + 103, 71 + 123; at 2000^2 x 64 396 + 538, 388 + 498, 380 + 499, 401 + 505, 421 + 576.
static int choose_levels(int variant, int64_t nshots, size_t elem, const Rect &R, const TileGrid &g)
{
    const int64_t fit = elem == 4 ? 512 : 256;
    for (int L = variant == 0 ? 7 : 12; L >= (variant == 0 ? 3 : 8); L--)
        if ((int64_t)make_tiles(variant, L, R, g).size() * nshots <= fit) return L;
    if (variant == 1) return 7;
    int best = 4;
    double least = 0.0;
    for (int L = 3; L <= 5; L++) {
        double c = 0.0;
        for (const TileHost &t : make_tiles(variant, L, R, g)) c += t.kind == TILE_PLAIN ? 1.0 : 2.2;
        if (least == 0.0 || c / L < least) least = c / L, best = L;
    }
    return best;
}

template <typename T>
static int build_tiles(AcPlan<T> *P, const Rect &R, const std::vector<int64_t> &sp,
                       const std::vector<int64_t> &si, const std::vector<int64_t> &sj, const std::vector<int64_t> &rp,
                       const std::vector<int64_t> &ri, const std::vector<int64_t> &rj)
{
    const int NX = (int)P->NX, NY = (int)P->NY;
    const std::vector<T> sx(P->sx.begin(), P->sx.end()), ty(P->ty.begin(), P->ty.end());
    const TileGrid grid = tile_grid(sx, ty, TILE_WAVES * TILE_RN, TILE_WAVES * TILE_RP);
    P->tile_levels = choose_levels(P->variant, P->nshots, sizeof(T), R, grid);
    const std::vector<TileHost> tiles = make_tiles(P->variant, P->tile_levels, R, grid);
    std::vector<int4> t;
    for (const TileHost &q : tiles) {
        t.push_back(make_int4(q.i0, q.i1, q.j0, q.j1));
        t.push_back(make_int4(q.ie, q.je, q.ne | q.ce << 16, q.kind));
    }
    P->ntiles = (int)tiles.size();
    ADS_TRY(P->d_tiles.upload(t));
    const PointLists s = make_points(tiles, NX, NY, sp, si, sj, false);
    ADS_TRY(P->d_ts_ptr.upload(s.ptr));
    ADS_TRY(P->d_ts_cell.upload(s.cell));
    ADS_TRY(P->d_ts_ent.upload(s.ent));
    const PointLists r = make_points(tiles, NX, NY, rp, ri, rj, true);
    ADS_TRY(P->d_tr_ptr.upload(r.ptr));
    ADS_TRY(P->d_tr_cell.upload(r.cell));
    ADS_TRY(P->d_tr_ent.upload(r.ent));
    return ADS_OK;
}

template <typename T>
static int build_plan(const ads_acoustic_params *p, const ads_shot_geometry *g, AcPlan<T> *P)
{
    ADS_TRY(validate_params(p));
    if (!g || g->nshots < 1 || !g->src_ptr || !g->rcv_ptr)
        ADS_FAIL(ADS_ERR_ARG, "geometry: need nshots >= 1, src_ptr and rcv_ptr");
    P->p = *p;
    P->variant = p->PropagatorKernel == 0 ? 0 : 1;
    P->NX = p->NX;
    P->NY = p->NY;
    P->Pitch = ((p->NY + 2 + WAVE - 1) / WAVE) * WAVE;
    P->Npad = (p->NX + 2) * P->Pitch;
    // the stencil kernels address one field of one shot with 32-bit byte offsets
    if ((uint64_t)P->Npad * sizeof(T) >= (uint64_t(1) << 32))
        ADS_FAIL(ADS_ERR_ARG, "grid too large: one padded field of one shot must be below 4 GiB");
    P->Ndense = (p->NX + 2) * (p->NY + 2);
    P->nshots = g->nshots;
    P->k = make_coef<T>(p->DELTAT, p->DELTAX, p->DELTAY);
    P->fwd_shape = Shape{2, (int)std::min<int64_t>(16, g->nshots), 1};
    const int64_t ns = g->nshots;
    if (g->src_ptr[0] != 0 || g->rcv_ptr[0] != 0) ADS_FAIL(ADS_ERR_ARG, "src_ptr/rcv_ptr must start at 0");
    std::vector<int64_t> nstep(ns);
    for (int64_t s = 0; s < ns; s++) {
        nstep[s] = g->nstep ? g->nstep[s] : p->NSTEP;
        if (nstep[s] < 1 || nstep[s] > p->NSTEP)
            ADS_FAIL(ADS_ERR_SHAPE, "shot %lld: nstep %lld outside [1, NSTEP=%lld]", (long long)s,
                     (long long)nstep[s], (long long)p->NSTEP);
        if (g->src_ptr[s + 1] < g->src_ptr[s] || g->rcv_ptr[s + 1] < g->rcv_ptr[s])
            ADS_FAIL(ADS_ERR_ARG, "src_ptr/rcv_ptr must be non-decreasing");
    }
    // plan order: longest record first, so the shots active at level n are a prefix
    P->order.resize(ns);
    for (int64_t s = 0; s < ns; s++) P->order[s] = s;
    std::stable_sort(P->order.begin(), P->order.end(),
                     [&](int64_t a, int64_t b) { return nstep[a] > nstep[b]; });
    P->NMAX = nstep[P->order[0]];
    P->nstep_sorted.resize(ns);
    for (int64_t q = 0; q < ns; q++) P->nstep_sorted[q] = nstep[P->order[q]];
    P->active.assign(P->NMAX + 2, 0);
    for (int64_t n = 0; n <= P->NMAX + 1; n++) {
        int c = 0;
        for (int64_t q = 0; q < ns; q++) c += P->nstep_sorted[q] >= n;
        P->active[n] = c;
    }
    // caller-order offsets of srcv and traces
    P->srcv_off_caller.resize(ns);
    P->trace_off_caller.resize(ns);
    int64_t so = 0, to = 0;
    for (int64_t s = 0; s < ns; s++) {
        P->srcv_off_caller[s] = so;
        P->trace_off_caller[s] = to;
        so += nstep[s] * (g->src_ptr[s + 1] - g->src_ptr[s]);
        to += (nstep[s] + 1) * (g->rcv_ptr[s + 1] - g->rcv_ptr[s]);
    }
    P->srcv_elems = so;
    P->trace_elems = to;
    // validated 1-based (i, j) in plan order
    auto check = [&](const int64_t *I, const int64_t *J, int64_t e, const char *what) -> int {
        int64_t i = I[e], j = J[e];
        if (i < 1 || i > p->NX + 2 || j < 1 || j > p->NY + 2)
            ADS_FAIL(ADS_ERR_INDEX, "%s %lld at (%lld, %lld) is outside the padded grid [1, %lld] x [1, %lld]",
                     what, (long long)e, (long long)i, (long long)j, (long long)(p->NX + 2),
                     (long long)(p->NY + 2));
        return ADS_OK;
    };
    std::vector<int64_t> sp(ns + 1, 0), rp(ns + 1, 0), si, sj, ri, rj, nsrc(ns), soff(ns), toff(ns);
    for (int64_t q = 0; q < ns; q++) {
        int64_t s = P->order[q];
        if (g->src_ptr[s + 1] > g->src_ptr[s] && (!g->srci || !g->srcj))
            ADS_FAIL(ADS_ERR_ARG, "srci/srcj are null");
        if (g->rcv_ptr[s + 1] > g->rcv_ptr[s] && (!g->rcvi || !g->rcvj))
            ADS_FAIL(ADS_ERR_ARG, "rcvi/rcvj are null");
        for (int64_t e = g->src_ptr[s]; e < g->src_ptr[s + 1]; e++) {
            ADS_TRY(check(g->srci, g->srcj, e, "source"));
            si.push_back(g->srci[e] - 1);
            sj.push_back(g->srcj[e] - 1);
        }
        for (int64_t e = g->rcv_ptr[s]; e < g->rcv_ptr[s + 1]; e++) {
            ADS_TRY(check(g->rcvi, g->rcvj, e, "receiver"));
            ri.push_back(g->rcvi[e] - 1);
            rj.push_back(g->rcvj[e] - 1);
        }
        sp[q + 1] = (int64_t)si.size();
        rp[q + 1] = (int64_t)ri.size();
        nsrc[q] = g->src_ptr[s + 1] - g->src_ptr[s];
        soff[q] = P->srcv_off_caller[s];
        toff[q] = P->trace_off_caller[s];
    }
    auto flat = [&](const std::vector<int64_t> &I, const std::vector<int64_t> &J) {
        std::vector<int64_t> f(I.size());
        for (size_t e = 0; e < I.size(); e++) f[e] = I[e] * P->Pitch + J[e];
        return f;
    };
    const CellLists us = build_cell_lists(ns, sp.data(), flat(si, sj));
    ADS_TRY(P->d_us_ptr.upload(us.shot_ptr));
    ADS_TRY(P->d_us_eptr.upload(us.ent_ptr));
    ADS_TRY(P->d_us_ent.upload(us.ent));
    ADS_TRY(P->d_us_cell.upload(us.cell));
    ADS_TRY(P->d_rcv_cell.upload(flat(ri, rj)));
    // PML profiles and flags
    P->sx.resize(p->NX + 2);
    P->ty.resize(p->NY + 2);
    ADS_TRY(ads_acoustic_pml_profiles(p, P->sx.data(), P->ty.data()));
    P->fbox = quiet_box(P->sx, P->ty);
    P->nfr = P->fbox.cells();
    std::vector<T> sxT(P->sx.begin(), P->sx.end()), tyT(P->ty.begin(), P->ty.end());
    auto flags = [](const std::vector<T> &v, std::vector<uint8_t> &pm, std::vector<uint8_t> &nr) {
        size_t L = v.size();
        pm.assign(L, 0);
        nr.assign(L, 0);
        for (size_t q = 0; q < L; q++) pm[q] = v[q] != T(0);
        for (size_t q = 0; q < L; q++)
            nr[q] = pm[q] | (q > 0 ? pm[q - 1] : 0) | (q + 1 < L ? pm[q + 1] : 0);
    };
    flags(sxT, P->pmlx, P->nearx);
    flags(tyT, P->pmly, P->neary);
    {
        int64_t cnt = 0;
        for (int64_t i = 1; i <= p->NX; i++)
            for (int64_t j = 1; j <= p->NY; j++) cnt += (P->pmlx[i] | P->pmly[j]) != 0;
        P->f_pml = (double)cnt / ((double)p->NX * (double)p->NY);
    }
    ADS_TRY(P->d_sx.upload(sxT));
    ADS_TRY(P->d_ty.upload(tyT));
    // plain rows/columns: interior and no PML formula needed
    std::vector<uint8_t> px(p->NX + 2, 0), py(p->NY + 2, 0);
    for (int64_t i = 1; i <= p->NX; i++) px[i] = !P->nearx[i];
    for (int64_t j = 1; j <= p->NY; j++) py[j] = !P->neary[j];
    Rect plain;
    {
        std::vector<int4> items;
        split_grid(px, py, p->NX, p->NY, 1, plain, items);  // no vector rounding
        split_grid(px, py, p->NX, p->NY, AcPlan<T>::VECP, P->rect, items);
        P->nitems = (int)items.size();
        ADS_TRY(P->d_items.upload(items));
        const Rect &R = P->rect;
        bool src_in = false;
        for (size_t e = 0; e < si.size(); e++)
            src_in |= si[e] >= R.iL && si[e] < R.iR && sj[e] >= R.jL && sj[e] < R.jR;
        P->blk_ok = !src_in && R.iR - R.iL > 2 && R.jR - R.jL > 2;
    }
    ADS_TRY(P->d_pmlx.upload(P->pmlx));
    ADS_TRY(P->d_pmly.upload(P->pmly));
    ADS_TRY(P->d_nearx.upload(P->nearx));
    ADS_TRY(P->d_neary.upload(P->neary));
    ADS_TRY(P->d_nsrc.upload(nsrc));
    ADS_TRY(P->d_srcv_off.upload(soff));
    ADS_TRY(P->d_rcv_ptr.upload(rp));
    ADS_TRY(P->d_trace_off.upload(toff));
    ADS_TRY(P->d_nstep_sorted.upload(P->nstep_sorted));
    ADS_TRY(P->d_nstep32.upload(std::vector<int32_t>(P->nstep_sorted.begin(), P->nstep_sorted.end())));
    ADS_TRY(build_tiles(P, plain, sp, si, sj, rp, ri, rj));
    // Shots per adjoint workgroup: a workgroup keeps its model rows and dL/dC in registers over its shots,
    // so more shots save their traffic as long as every CU still has four workgroups; past four shots the
    // last workgroups' tail costs more.  us per level, FP32, for 1 / 2 / 4 / 8 shots: 1000^2 x 32 shots 119 /
    // 98 / 94 / 100, kernel 0 - / 152 / 137 / 147; for 2 / 4 / 8: 2000^2 x 64 546 / 490 / 499.
    P->adj_shape.sg = (int)std::min<int64_t>(4, std::max<int64_t>(1, (int64_t)P->ntiles * ns / 1024));
    return ADS_OK;
}

}  // namespace ads

using namespace ads;

struct ads_acoustic_plan {
    std::unique_ptr<AcPlanBase> impl;
};

template <typename F> static int dispatch(ads_acoustic_plan *pl, F &&f)
{
    if (!pl || !pl->impl) ADS_FAIL(ADS_ERR_ARG, "null plan");
    if (pl->impl->dtype == ADS_F64) return f(*static_cast<AcPlan<double> *>(pl->impl.get()));
    return f(*static_cast<AcPlan<float> *>(pl->impl.get()));
}

extern "C" {

int ads_acoustic_plan_create(const ads_acoustic_params *p, const ads_shot_geometry *g, int dtype,
                             ads_acoustic_plan **out)
{
    clear_error();
    if (!out) ADS_FAIL(ADS_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (dtype != ADS_F32 && dtype != ADS_F64) ADS_FAIL(ADS_ERR_ARG, "dtype must be ADS_F32 or ADS_F64");
    auto pl = std::make_unique<ads_acoustic_plan>();
    int rc;
    if (dtype == ADS_F64) {
        auto P = std::make_unique<AcPlan<double>>();
        P->dtype = dtype;
        rc = build_plan<double>(p, g, P.get());
        pl->impl = std::move(P);
    } else {
        auto P = std::make_unique<AcPlan<float>>();
        P->dtype = dtype;
        rc = build_plan<float>(p, g, P.get());
        pl->impl = std::move(P);
    }
    if (rc != ADS_OK) return rc;
    *out = pl.release();
    return ADS_OK;
}

int ads_acoustic_plan_destroy(ads_acoustic_plan *plan)
{
    delete plan;
    return ADS_OK;
}

int ads_acoustic_plan_sizes(const ads_acoustic_plan *plan, int64_t *srcv_elems,
                            int64_t *trace_elems, int64_t *srcv_off, int64_t *trace_off)
{
    clear_error();
    if (!plan || !plan->impl) ADS_FAIL(ADS_ERR_ARG, "null plan");
    const AcPlanBase &b = *plan->impl;
    if (srcv_elems) *srcv_elems = b.srcv_elems;
    if (trace_elems) *trace_elems = b.trace_elems;
    for (int64_t s = 0; s < b.nshots; s++) {
        if (srcv_off) srcv_off[s] = b.srcv_off_caller[s];
        if (trace_off) trace_off[s] = b.trace_off_caller[s];
    }
    return ADS_OK;
}

size_t ads_acoustic_plan_workspace_size(const ads_acoustic_plan *plan, int64_t K)
{
    if (!plan || !plan->impl) return 0;
    if (plan->impl->dtype == ADS_F64) return static_cast<AcPlan<double> *>(plan->impl.get())->ws_size(K);
    return static_cast<AcPlan<float> *>(plan->impl.get())->ws_size(K);
}

int64_t ads_acoustic_plan_choose_interval(const ads_acoustic_plan *plan, size_t budget)
{
    if (!plan || !plan->impl) return 0;
    // One-level schedule: the fewest segments M whose interval fits, then the shortest
    // interval with that M: every segment but the last is recomputed, so K = ceil(levels / M)
    // minimises the recomputation ((M - 1) K levels) among the intervals that need M segments.
    const int64_t L = std::max<int64_t>(plan->impl->NMAX - 1, 1);
    for (int64_t M = 1; M <= L; M++) {
        const int64_t K = (L + M - 1) / M;
        const size_t need = plan->impl->dtype == ADS_F64
                                ? static_cast<AcPlan<double> *>(plan->impl.get())->ws_size(K, -1)
                                : static_cast<AcPlan<float> *>(plan->impl.get())->ws_size(K, -1);
        if (need <= budget) return K;
        if (K == 1) break;
    }
    return 0;
}

int ads_acoustic_plan_set_snapshots(ads_acoustic_plan *plan, int64_t snapshots)
{
    clear_error();
    if (!plan || !plan->impl) ADS_FAIL(ADS_ERR_ARG, "null plan");
    plan->impl->snapshots = snapshots < 0 ? -1 : snapshots;
    return ADS_OK;
}

int64_t ads_acoustic_plan_snapshots(const ads_acoustic_plan *plan)
{
    return plan && plan->impl ? plan->impl->snapshots : -1;
}

int ads_acoustic_plan_choose_schedule(ads_acoustic_plan *plan, size_t budget, int64_t *K, int64_t *S)
{
    clear_error();
    if (!plan || !plan->impl || !K || !S) ADS_FAIL(ADS_ERR_ARG, "null argument");
    const int rc = plan->impl->dtype == ADS_F64
                       ? static_cast<AcPlan<double> *>(plan->impl.get())->choose_schedule(budget, K, S)
                       : static_cast<AcPlan<float> *>(plan->impl.get())->choose_schedule(budget, K, S);
    if (rc != ADS_OK) ADS_FAIL(rc, "no checkpoint schedule fits %zu bytes", budget);
    plan->impl->snapshots = *S;
    return ADS_OK;
}

int ads_acoustic_plan_forward(ads_acoustic_plan *plan, const void *model, const void *srcv,
                              void *traces, void *ws, size_t wsb, int64_t K, ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv) ADS_FAIL(ADS_ERR_ARG, "null model/srcv");
    return dispatch(plan, [&](auto &P) { return P.forward(model, srcv, traces, ws, wsb, K, S(stream)); });
}

int ads_acoustic_plan_backward(ads_acoustic_plan *plan, const void *model, const void *srcv,
                               const void *grad_traces, void *grad_model, void *ws, size_t wsb,
                               int64_t K, ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv || !grad_traces || !grad_model) ADS_FAIL(ADS_ERR_ARG, "null argument");
    return dispatch(plan, [&](auto &P) {
        using R = typename std::remove_const<decltype(P.k.dt)>::type;
        return P.backward(model, srcv, (const R *)grad_traces, grad_model, ws, wsb, K, S(stream));
    });
}

int ads_acoustic_plan_gradient(ads_acoustic_plan *plan, const void *model, const void *srcv,
                               const void *observed, double *loss, void *grad_model, void *traces,
                               void *ws, size_t wsb, int64_t K, ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv || !observed || !grad_model) ADS_FAIL(ADS_ERR_ARG, "null argument");
    return dispatch(plan, [&](auto &P) -> int {
        using R = typename std::remove_const<decltype(P.k.dt)>::type;
        typename std::remove_reference<decltype(P)>::type::WS w;
        ADS_TRY(P.check_ws(w, ws, wsb, K));
        // traces go to the caller's buffer if given, else into the residual area (reused)
        R *tr = traces ? (R *)traces : w.resid;
        ADS_TRY(P.forward(model, srcv, tr, ws, wsb, K, S(stream)));
        ADS_TRY(P.misfit(w, tr, (const R *)observed, S(stream)));
        if (loss) ADS_HIP(hipMemcpyAsync(loss, w.loss, sizeof(double), hipMemcpyDeviceToDevice, S(stream)));
        return P.backward(model, srcv, w.resid, grad_model, ws, wsb, K, S(stream));
    });
}

int ads_acoustic_plan_autotune(ads_acoustic_plan *plan, const void *model, const void *srcv,
                               void *ws, size_t wsb, int64_t K, int reps, int *shape_out,
                               ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv) ADS_FAIL(ADS_ERR_ARG, "null argument");
    return dispatch(plan, [&](auto &P) -> int {
        ADS_TRY(P.autotune(model, srcv, ws, wsb, K, reps, S(stream)));
        if (shape_out) {
            const Shape *sh[2] = {&P.fwd_shape, &P.adj_shape};
            for (int q = 0; q < 2; q++) {
                shape_out[3 * q] = sh[q]->rpt;
                shape_out[3 * q + 1] = sh[q]->sg;
                shape_out[3 * q + 2] = sh[q]->sb;
            }
        }
        return ADS_OK;
    });
}

int ads_acoustic_plan_set_shape(ads_acoustic_plan *plan, const int *shape)
{
    clear_error();
    if (!shape) ADS_FAIL(ADS_ERR_ARG, "null shape");
    for (int q = 0; q < 2; q++) {
        const int rpt = shape[3 * q], sg = shape[3 * q + 1], sb = shape[3 * q + 2];
        if (rpt != 1 && rpt != 2 && rpt != 4 && !(q == 0 && (rpt == 8 || rpt == 16)))
            ADS_FAIL(ADS_ERR_ARG, "rows per wavefront must be 1, 2 or 4 (8 or 16 for the forward)");
        if (sg < 1) ADS_FAIL(ADS_ERR_ARG, "shots per workgroup must be >= 1");
        if (sb != 1 && sb != 2) ADS_FAIL(ADS_ERR_ARG, "shots per batch must be 1 or 2");
        if (sb == 2 && rpt >= 4) ADS_FAIL(ADS_ERR_ARG, "shots per batch 2 needs 1 or 2 rows per wavefront");
    }
    return dispatch(plan, [&](auto &P) -> int {
        P.fwd_shape = Shape{shape[0], shape[1], shape[2]};  // 8 or 16 rows: 2 rows
        P.adj_shape = Shape{shape[3], shape[4], shape[5]};
        P.drop_graphs();
        return ADS_OK;
    });
}

int ads_acoustic_plan_set_graph(ads_acoustic_plan *plan, int enable)
{
    clear_error();
    return dispatch(plan, [&](auto &P) -> int {
        P.use_graph = enable ? 1 : 0;
        if (!enable) P.drop_graphs();
        return ADS_OK;
    });
}

int ads_acoustic_plan_set_frame_rows(ads_acoustic_plan *plan, int rows)
{
    clear_error();
    if (rows != 0 && rows != 4 && rows != 8 && rows != 16 && rows != 32 && rows != 64)
        ADS_FAIL(ADS_ERR_ARG, "frame rows must be 0, 4, 8, 16, 32 or 64, got %d", rows);
    return dispatch(plan, [&](auto &) -> int { return ADS_OK; });
}

int ads_acoustic_plan_set_blocking(ads_acoustic_plan *plan, int levels)
{
    clear_error();
    if (levels != 1 && levels != 2) ADS_FAIL(ADS_ERR_ARG, "levels must be 1 or 2, got %d", levels);
    return dispatch(plan, [&](auto &P) -> int {
        if (P.blocking != levels) P.drop_graphs();
        P.blocking = levels;
        return ADS_OK;
    });
}

int ads_acoustic_plan_blocking(const ads_acoustic_plan *plan)
{
    if (!plan || !plan->impl) return 0;
    return plan->impl->blocking == 2 && plan->impl->blk_ok ? 2 : 1;
}

int ads_acoustic_plan_forward_history(ads_acoustic_plan *plan, const void *model,
                                      const void *srcv, void *u_hist, void *phi_hist,
                                      void *psi_hist, void *scratch, ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv || !u_hist || !scratch) ADS_FAIL(ADS_ERR_ARG, "null argument");
    return dispatch(plan, [&](auto &P) -> int {
        ADS_TRY(P.check_history());
        return P.forward_history(model, srcv, u_hist, phi_hist, psi_hist, scratch, S(stream));
    });
}

int ads_acoustic_plan_backward_history(ads_acoustic_plan *plan, const void *model,
                                       const void *srcv, const void *u_hist,
                                       const void *grad_u_hist, void *grad_model, void *scratch,
                                       ads_stream_t stream)
{
    clear_error();
    if (!model || !srcv || !u_hist || !grad_u_hist || !grad_model || !scratch)
        ADS_FAIL(ADS_ERR_ARG, "null argument");
    return dispatch(plan, [&](auto &P) -> int {
        ADS_TRY(P.check_history());
        return P.backward_history(model, srcv, u_hist, grad_u_hist, grad_model, scratch, S(stream));
    });
}

size_t ads_acoustic_plan_history_scratch_size(const ads_acoustic_plan *plan)
{
    if (!plan || !plan->impl) return 0;
    if (plan->impl->dtype == ADS_F64)
        return static_cast<AcPlan<double> *>(plan->impl.get())->history_scratch();
    return static_cast<AcPlan<float> *>(plan->impl.get())->history_scratch();
}

}  // extern "C"
