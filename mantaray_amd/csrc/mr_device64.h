// mr_device64.h -- the fp64-interpolation mode (MR_PREC_FP64_INTERP): field
// queries, the right-hand side, and its vector-Jacobian product, for the
// differentiable path.
//
// The reference interpolates in f32 (interpolator.rs:39-84 over f32 corner
// values), so its trajectories are piecewise constant in the field values at
// the scale of an f32 ulp and have no useful derivative with respect to
// them.  This mode keeps the reference's algorithm (the same fractional
// index, cell rule, bilinear formula with its corner and det == 0 exits, and
// cell-difference gradients) but evaluates all of it in f64 on the f64 values,
// with the bathymetry queried at the f64 point instead of its f32 rounding:
//
//   index   (p - a0) / |a1 - a0|         (cartesian_current.rs:244, in f64)
//   cell    floor, or n-2 on the last node (cartesian_current.rs:283-339)
//   value   ((a00 + a10 u) + a01 w) + (a11 u) w, u = (y - y_j) RN(1/(y_j+1 - y_j)),
//           w = (x - x_i) RN(1/(x_i+1 - x_i))   (interpolator.rs:59-83, in f64)
//   slopes  (D - A) RN(1/(x1 - x0)), (B - A) RN(1/(y1 - y0))
//
//   (the change of basis m01 = -dtx/det, m10 = -bty/det with det = -dtx bty
//   is the reciprocal of the cell's size along each axis, here rounded once;
//   the slopes are the cell difference times the rounded reciprocal of the
//   signed first spacing, within an ulp of the reference's quotient)
//
// Field values come from kernel arguments (pointers to the raw f64 arrays),
// so a caller can differentiate with respect to them and change them between
// calls without rebuilding anything; what depends only on the axes (an
// AxisCell64 per axis cell) is tabulated once per field.  As in the reference
// mode, each lane holds cells in registers (a Slot64 per field, or one for
// both where they lie on the same grid) and loads the cell a coming
// evaluation will most likely need ahead of it.
//
// Linearisation.  With u, w the bilinear fractions of the query, the value is
//   v = wA A + wB B + wC C + wD D,  wA = (1-u)(1-w), wB = u(1-w), wC = u w,
//   wD = (1-u) w,
// its derivative along x is (a01 + a11 u) m10 and along y (a10 + a11 w) m01;
// the cell-difference slopes are constant inside a cell.  The right-hand
// side (wave_ray_path.rs:118-150) with k = |k|, e = k/k, q = k h,
// T = tanh q, S = sech^2 q, sigma = sqrt(g k T):
//   dx/dt = cg e + U,   cg = (g/2)(T + q S)/sigma
//   dk/dt = c grad h - (grad U)^T k,   c = -k sigma / sinh(2q)
// has the partial derivatives
//   d sigma/dk = cg,  d sigma/dh = (g/2) k^2 S / sigma
//   N = T + q S,  dN/dq = 2 S (1 - q T)
//   d cg/dk = (g/2)(h N_q - N cg/sigma)/sigma
//   d cg/dh = (g/2)(k N_q - N sigma_h/sigma)/sigma
//   d c/dk  = c (1/k + cg/sigma - 2 h coth 2q)
//   d c/dh  = c (sigma_h/sigma - 2 k coth 2q),  coth 2q = (T + 1/T)/2
// and d(cg e)/dk = cg_k e e^T + (cg/k)(I - e e^T).
#pragma once

#include "mr_device.h"

namespace mr {

// Numeric parameters of a field in fp64 mode (per lane, in VGPRs).
struct Grid64View {
    int kind;                             // BK_* for a bathymetry, CK_* for a current
    int nx, ny, ncx;                      // grid; ncx = nx - 1
    int an;                               // ArrayDepth (an x an)
    uint32_t oob_from;                    // first cell (row-major) with a corner past the data
    double a0x, a0y;                      // first coordinate of each axis
    double sx, sy, inv_sx, inv_sy;        // |a1 - a0| and RN(1/|a1 - a0|)
    double nxm1, nym1;                    // n - 1
    double rxs, rys;                      // RN(1/(a1 - a0)), signed: the slope factors
    double h, h0, x0, y0, dhdx, dhdy;     // ConstantDepth / ConstantSlope, widened
    double u, v;                          // ConstantCurrent
    float gx0, gy0, ginv_x, ginv_y;       // cell guess for prefetch, in f32
    float gmax_x, gmax_y;                 // (f32)(n - 2)
};

// What a query needs of cell i along one axis.  [lo, hi] is the cell's fast
// interval: the f64 index's cell [T[i], T[i+1]) narrowed to the open interval
// between the cell's nodes (a[i], a[i+1]), both ends included (empty as lo >
// hi or NaN).  A target inside on both axes is in the cell and on none of
// its node lines, so the bilinear value needs neither the corner exit nor
// the det == 0 exit; other targets of the cell (rare: the node coordinates
// themselves, and cells that err) take the full query.
struct AxisCell64 {                       // 32 B
    double lo, hi;
    double a, r;                          // a[i]; RN(1/(a[i+1] - a[i]))
};

// Device arrays of a field in fp64 mode (kernel arguments).
struct Grid64Ptrs {
    const AxisCell64 *xc, *yc;            // per axis cell
    const double *xn, *yn;                // node coordinates
    const float *arr;                     // ArrayDepth values
    const void *view;                     // the field's Grid64View, for the full queries
};

// A gridded value at a point with what its derivatives need.
struct Val64 {
    double val;                           // interpolated value
    double gx, gy;                        // cell-difference slopes
    double dx, dy;                        // derivative of the interpolant along x, y
};

// The cell of a query: flat index of corner A (B = A + nx, C = A + nx + 1,
// D = A + 1) and the bilinear fractions.
struct Cell64 {
    uint32_t iA;
    double u, w;
};

// One cell held per lane: its axis cells and the four corners of NV value
// arrays (depth; u and v; or all three), as the pairs (A, D) and (B, C) that
// lie next to each other in memory.  A slot holds only cells whose corners
// all lie in the data; one never loaded has NaN intervals, which contain no
// point.
template <int NV>
struct Slot64 {
    mr_d2 xt = {MR_NAN_INIT, MR_NAN_INIT}, yt = {MR_NAN_INIT, MR_NAN_INIT};   // (lo, hi)
    mr_d2 xa = {0.0, 0.0}, ya = {0.0, 0.0};                                   // (a, r)
    mr_d2 ad[NV] = {}, bc[NV] = {};
    uint32_t iA = 0;
};

// Cell of (x, y), or ok = false where the reference's index or corner
// lookup errs (a NaN target included); i1 = j1 = 0 then.
__device__ __forceinline__ bool locate64(const Grid64View &G, double x, double y, int &i1,
                                         int &j1)
{
    bool ok = true;
    const double fx = index64(x, G.a0x, G.sx, G.inv_sx, G.nxm1, ok);
    const double fy = index64(y, G.a0y, G.sy, G.inv_sy, G.nym1, ok);
    i1 = ok ? __builtin_elementwise_min((int)fx, G.nx - 2) : 0;
    j1 = ok ? __builtin_elementwise_min((int)fy, G.ny - 2) : 0;
    ok = ok & ((uint32_t)j1 * (uint32_t)G.ncx + (uint32_t)i1 < G.oob_from);
    i1 = ok ? i1 : 0;
    j1 = ok ? j1 : 0;
    return ok;
}

// How far (x, y) is outside the slot's fast interval, as a word that is
// below OUT64 exactly inside: the distances to the four bounds are all
// non-negative and finite there, and the high words of negative, infinite
// and NaN doubles are all at or above 0x7ff00000.  (Four f64 compares and
// the scalar ANDs of their masks took longer; f64 min and max would have
// their loaded operands quieted first.)
constexpr uint32_t OUT64 = 0x7ff00000u;

__device__ __forceinline__ uint32_t hi_word(double v)
{
    return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32);
}

template <int NV>
__device__ __forceinline__ uint32_t off_slot64(const Slot64<NV> &s, double x, double y)
{
    const uint32_t a = hi_word(x - s.xt.x), b = hi_word(s.xt.y - x);
    const uint32_t c = hi_word(y - s.yt.x), d = hi_word(s.yt.y - y);
    return __builtin_elementwise_max(__builtin_elementwise_max(a, b),
                                     __builtin_elementwise_max(c, d));
}

// two neighbouring values of an array
__device__ __forceinline__ mr_d2 gld_pair(const double *p, uint32_t i)
{
    typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
    return *(const MR_GLOBAL pair *)((const MR_GLOBAL char *)p + i * 8u);
}

// Start loading cell (i1, j1) into s, for a cell whose corners lie in the
// data; vals: the NV value arrays.
template <int NV>
__device__ __forceinline__ void slot64_load(const Grid64View &G, const Grid64Ptrs &P,
                                            const double *const (&vals)[NV], Slot64<NV> &s,
                                            int i1, int j1)
{
    const MR_GLOBAL mr_d2 *xc =
        (const MR_GLOBAL mr_d2 *)((const MR_GLOBAL char *)P.xc + (uint32_t)i1 * 32u);
    const MR_GLOBAL mr_d2 *yc =
        (const MR_GLOBAL mr_d2 *)((const MR_GLOBAL char *)P.yc + (uint32_t)j1 * 32u);
    s.xt = xc[0];
    s.xa = xc[1];
    s.yt = yc[0];
    s.ya = yc[1];
    const uint32_t iA = __umul24((uint32_t)G.nx, (uint32_t)j1) + (uint32_t)i1;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        s.ad[q] = gld_pair(vals[q], iA);
        s.bc[q] = gld_pair(vals[q], iA + (uint32_t)G.nx);
    }
    s.iA = iA;
}

// Start loading the cell that (x, y) most likely lies in (guessed in f32,
// clamped into the grid; used only to choose what to load), unless a corner
// of it is past the data (oob: the first such cell).
template <int NV>
__device__ __forceinline__ void slot64_prefetch(const Grid64View &G, const Grid64Ptrs &P,
                                                const double *const (&vals)[NV], uint32_t oob,
                                                Slot64<NV> &s, double x, double y)
{
    const int i1 = guess_cell((float)x, G.gx0, G.ginv_x, G.gmax_x);
    const int j1 = guess_cell((float)y, G.gy0, G.ginv_y, G.gmax_y);
    if (__umul24((uint32_t)j1, (uint32_t)G.ncx) + (uint32_t)i1 < oob)
        slot64_load<NV>(G, P, vals, s, i1, j1);
}

// interpolator::bilinear in f64 on a cell (ad, bc: its corners; (x0, rx),
// (y0, ry): its origin and reciprocal sizes), without its exits, and the
// cell-difference slopes.
__device__ __forceinline__ Val64 cell64_value(const Grid64View &G, mr_d2 ad, mr_d2 bc, mr_d2 xa,
                                              mr_d2 ya, double u, double w)
{
    const double a10 = bc.x - ad.x, a01 = ad.y - ad.x;
    const double a11 = ((bc.y - ad.x) - a10) - a01;
    Val64 r;
    r.val = ((ad.x + a10 * u) + a01 * w) + (a11 * u) * w;
    r.gx = a01 * G.rxs;
    r.gy = a10 * G.rys;
    r.dx = (a01 + a11 * u) * xa.y;
    r.dy = (a10 + a11 * w) * ya.y;
    return r;
}

// the bilinear fractions of a target in the slot's cell
template <int NV>
__device__ __forceinline__ Cell64 slot64_cell(const Slot64<NV> &s, double x, double y)
{
    return Cell64{s.iA, s.ya.y * (y - s.ya.x), s.xa.y * (x - s.xa.x)};
}

// The full query of the N value arrays of a gridded field at (x, y): its
// cell by the reference's index, with the exits of interpolator::bilinear (a
// target on a node returns that corner, first of A, B, C, D; det == 0 errs
// anywhere else).  Returns false where the reference errs.
template <int N>
__device__ __forceinline__ bool full64(const Grid64View &G, const Grid64Ptrs &P,
                                       const double *const (&vals)[N], double x, double y,
                                       Val64 (&v)[N], Cell64 &c)
{
    int i1, j1;
    bool ok = locate64(G, x, y, i1, j1);
    Slot64<N> s;
    if (ok) slot64_load<N>(G, P, vals, s, i1, j1);
    const double xb = ok ? P.xn[i1 + 1] : 0.0, yb = ok ? P.yn[j1 + 1] : 0.0;
    wait_vmem();
    c = slot64_cell<N>(s, x, y);
    const bool xl = x == s.xa.x, xr = x == xb, yl = y == s.ya.x, yr = y == yb;
    const bool node = (xl | xr) & (yl | yr);
#pragma unroll
    for (int q = 0; q < N; ++q) {
        v[q] = cell64_value(G, s.ad[q], s.bc[q], s.xa, s.ya, c.u, c.w);
        if (node) v[q].val = xl ? (yl ? s.ad[q].x : s.bc[q].x) : (yr ? s.bc[q].y : s.ad[q].y);
    }
    return ok & (node | ((xb - s.xa.x) * (yb - s.ya.x) != 0.0));
}

// Bathymetry in fp64 mode, analytic kinds in place and gridded depth by the
// full query.  Returns ok = false where the reference errs; h is NaN (not an
// error) for a NaN point (cartesian_netcdf3.rs:102-105) and outside an
// ArrayDepth.  cell is meaningful for BK_GRID only.
template <int BK>
__device__ __forceinline__ bool bathy64(const Grid64View &B, const Grid64Ptrs &P,
                                        const double *depth, double x, double y, Val64 &h,
                                        Cell64 &cell)
{
    cell.iA = 0; cell.u = 0.0; cell.w = 0.0;
    h.dx = 0.0; h.dy = 0.0;
    const bool nn = __builtin_isnan(x) || __builtin_isnan(y);
    if (BK == BK_CONSTANT) {                               // constant_depth.rs:34-40
        h.val = nn ? MR_NAN : B.h;
        h.gx = 0.0; h.gy = 0.0;
        return true;
    } else if (BK == BK_SLOPE) {                           // constant_slope.rs:63-74
        h.val = nn ? MR_NAN : (B.h0 + B.dhdx * (x - B.x0)) + B.dhdy * (y - B.y0);
        h.gx = B.dhdx; h.gy = B.dhdy;
        h.dx = B.dhdx; h.dy = B.dhdy;
        return true;
    } else if (BK == BK_ARRAY) {                           // array_depth.rs:26-33
        const uint64_t xi = x > 0.0 ? (x >= 1.8446744073709552e19 ? UINT64_MAX : (uint64_t)x) : 0;
        const uint64_t yi = y > 0.0 ? (y >= 1.8446744073709552e19 ? UINT64_MAX : (uint64_t)y) : 0;
        h.gx = 0.0; h.gy = 0.0;
        if (xi >= (uint64_t)B.an || yi >= (uint64_t)B.an) {
            h.val = MR_NAN;
            return true;
        }
        h.val = (double)P.arr[xi * (uint64_t)B.an + yi];
        return true;
    } else {                                               // cartesian_netcdf3.rs:98-135
        const double *const vals[1] = {depth};
        Val64 v[1];
        bool ok = full64<1>(B, P, vals, x, y, v, cell);
        h = v[0];
        if (nn) {
            h.val = MR_NAN; h.gx = MR_NAN; h.gy = MR_NAN;
            ok = true;
        }
        return ok;
    }
}

// Current in fp64 mode, a gridded one by the full query; ok = false where
// the reference errs (no NaN guard: a NaN point errs,
// cartesian_current.rs:492-495).
template <int CK>
__device__ __forceinline__ bool current64(const Grid64View &C, const Grid64Ptrs &P,
                                          const double *cu, const double *cv, double x, double y,
                                          Val64 &u, Val64 &v, Cell64 &cell)
{
    cell.iA = 0; cell.u = 0.0; cell.w = 0.0;
    if (CK == CK_CONSTANT) {                               // constant_current.rs:66-76
        u.val = C.u; v.val = C.v;
        u.gx = u.gy = u.dx = u.dy = 0.0;
        v.gx = v.gy = v.dx = v.dy = 0.0;
        return true;
    } else {                                               // cartesian_current.rs:487-542
        const double *const vals[2] = {cu, cv};
        Val64 w[2];
        const bool ok = full64<2>(C, P, vals, x, y, w, cell);
        u = w[0];
        v = w[1];
        return ok;
    }
}

// Field values of one fp64 evaluation.
struct Fields64 {
    const double *depth, *u, *v;
};

// The cells a lane holds for one evaluation.  SH: depth and current lie on
// the same f64 axes, so one slot (b) holds depth, u and v; the tests,
// fractions and axis cells of a second one are saved.
template <int BK, int CK, bool SH>
struct Slots64 {
    Slot64<SH ? 3 : 1> b;
    Slot64<2> c;
};

// Load the cells that (x, y) most likely lies in: every one (a ray's first
// cells, or a segment's), or those of held that do not contain it.
template <int BK, int CK, bool SH, bool ALL>
__device__ __forceinline__ void load64(const Grid64View &B, const Grid64Ptrs &BP,
                                       const Grid64View &C, const Grid64Ptrs &CP,
                                       const Fields64 &F, const Slots64<BK, CK, SH> &held,
                                       Slots64<BK, CK, SH> &s, double x, double y)
{
    if constexpr (SH) {
        const double *const vals[3] = {F.depth, F.u, F.v};
        if (ALL || off_slot64(held.b, x, y) >= OUT64)
            slot64_prefetch<3>(C, CP, vals, __builtin_elementwise_min(B.oob_from, C.oob_from),
                               s.b, x, y);
    } else {
        if constexpr (BK == BK_GRID) {
            const double *const vals[1] = {F.depth};
            if (ALL || off_slot64(held.b, x, y) >= OUT64)
                slot64_prefetch<1>(B, BP, vals, B.oob_from, s.b, x, y);
        }
        if constexpr (CK == CK_GRID) {
            const double *const vals[2] = {F.u, F.v};
            if (ALL || off_slot64(held.c, x, y) >= OUT64)
                slot64_prefetch<2>(C, CP, vals, C.oob_from, s.c, x, y);
        }
    }
}

template <int BK, int CK, bool SH>
__device__ __forceinline__ void load_guess64(const Grid64View &B, const Grid64Ptrs &BP,
                                             const Grid64View &C, const Grid64Ptrs &CP,
                                             const Fields64 &F, Slots64<BK, CK, SH> &s, double x,
                                             double y)
{
    load64<BK, CK, SH, true>(B, BP, C, CP, F, s, s, x, y);
}

// s_waitcnt on the vector memory count alone, for counts up to 63 (gfx9
// splits vmcnt over bits 3:0 and 15:14; expcnt and lgkmcnt at their no-wait
// maxima).
template <int N>
__device__ __forceinline__ void vm_wait_upto()
{
    static_assert(N >= 0 && N < 64, "vmcnt below 64");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Start loading, into n, the cells of (x, y) that q does not hold.
template <int BK, int CK, bool SH>
__device__ __forceinline__ void prefetch64(const Grid64View &B, const Grid64Ptrs &BP,
                                           const Grid64View &C, const Grid64Ptrs &CP,
                                           const Fields64 &F, const Slots64<BK, CK, SH> &q,
                                           Slots64<BK, CK, SH> &n, double x, double y)
{
    load64<BK, CK, SH, false>(B, BP, C, CP, F, q, n, x, y);
}

// The fields of one fp64 evaluation, with their cells.
struct Point64 {
    Val64 h, u, v;
    Cell64 bc, cc;
    bool okb, okc;
};

// The fields at (x, y) from the cells in hand: the gridded queries' own
// operations for a target inside the slots' fast intervals, with no branch
// and no load.  Returns OUT64 or more where that does not hold (a target
// outside them, a NaN target), and those lanes must take point64_full.
template <int BK, int CK, bool SH>
__device__ __forceinline__ uint32_t point64_fast(const Grid64View &B, const Grid64Ptrs &BP,
                                                 const Grid64View &C, const Grid64Ptrs &CP,
                                                 const Fields64 &F,
                                                 const Slots64<BK, CK, SH> &sl, double x,
                                                 double y, Point64 &p)
{
    uint32_t off = 0;
    p.okb = true;
    p.okc = true;
    if constexpr (BK == BK_GRID) {
        off = off_slot64(sl.b, x, y);
        p.bc = slot64_cell(sl.b, x, y);
        p.h = cell64_value(B, sl.b.ad[0], sl.b.bc[0], sl.b.xa, sl.b.ya, p.bc.u, p.bc.w);
    } else {
        p.okb = bathy64<BK>(B, BP, F.depth, x, y, p.h, p.bc);
    }
    if constexpr (SH) {
        p.cc = p.bc;
        p.u = cell64_value(C, sl.b.ad[1], sl.b.bc[1], sl.b.xa, sl.b.ya, p.cc.u, p.cc.w);
        p.v = cell64_value(C, sl.b.ad[2], sl.b.bc[2], sl.b.xa, sl.b.ya, p.cc.u, p.cc.w);
    } else if constexpr (CK == CK_GRID) {
        const uint32_t offc = off_slot64(sl.c, x, y);
        off = __builtin_elementwise_max(off, offc);
        p.cc = slot64_cell(sl.c, x, y);
        p.u = cell64_value(C, sl.c.ad[0], sl.c.bc[0], sl.c.xa, sl.c.ya, p.cc.u, p.cc.w);
        p.v = cell64_value(C, sl.c.ad[1], sl.c.bc[1], sl.c.xa, sl.c.ya, p.cc.u, p.cc.w);
    } else {
        p.okc = current64<CK>(C, CP, F.u, F.v, x, y, p.u, p.v, p.cc);
    }
    return off;
}

// ... and by the full queries, on views loaded for the occasion: most of a
// view serves only them, and held in registers all the time it would push
// what every evaluation uses into accumulation registers (or scratch).
template <int BK, int CK>
__device__ __forceinline__ void point64_full(const Grid64Ptrs &BP, const Grid64Ptrs &CP,
                                             const Fields64 &F, double x, double y, Point64 &p)
{
    const Grid64View B = load_view<Grid64View>(BP.view);
    const Grid64View C = load_view<Grid64View>(CP.view);
    p.okb = bathy64<BK>(B, BP, F.depth, x, y, p.h, p.bc);
    p.okc = current64<CK>(C, CP, F.u, F.v, x, y, p.u, p.v, p.cc);
}

// Whether any lane must take point64_full, as one compare and one scalar
// branch: the mask intrinsic is not folded into the test inside the block.
// The callers mark it unlikely (an expectation inside this function would be
// lost when it is inlined), so that the block is laid out after the loop; in
// its place it costs a taken branch at every evaluation (16,384 rays x 2000
// steps of a forward and its sweep 5.32 -> 5.20 ms).
template <int BK, int CK>
__device__ __forceinline__ bool any_off64(uint32_t off)
{
    if (BK != BK_GRID && CK != CK_GRID) return false;
    return __builtin_amdgcn_uicmp(off, OUT64, 35 /* >= */) != 0;
}

// WaveRayPath::system in fp64 mode, with the cells held in sl.  As rhs_rec()
// does for the reference precision, every lane first evaluates with the
// cells in hand, and the lanes whose target is not inside them evaluate
// again with the full queries.
template <int BK, int CK, bool SH, int MATH>
__device__ __forceinline__ void rhs64(const Grid64View &B, const Grid64Ptrs &BP,
                                      const Grid64View &C, const Grid64Ptrs &CP,
                                      const Fields64 &F, const Slots64<BK, CK, SH> &sl,
                                      const FastConsts &K, double x, double y, double kx,
                                      double ky, double &dx, double &dy, double &dkx,
                                      double &dky)
{
    Point64 p;
    auto system = [&] {
        odes<MATH, depth_is_flat<BK>(), CK == CK_CONSTANT>(K, p.okb ? p.h.val : MR_NAN, p.h.gx, p.h.gy, p.okc, p.u.val, p.v.val, p.u.gx,
                   p.u.gy, p.v.gx, p.v.gy, kx, ky, dx, dy, dkx, dky);
    };
    const uint32_t off = point64_fast<BK, CK, SH>(B, BP, C, CP, F, sl, x, y, p);
    system();
    if (__builtin_expect(any_off64<BK, CK>(off), 0)) {
        __asm__ volatile("");
        if (off >= OUT64) {
            point64_full<BK, CK>(BP, CP, F, x, y, p);
            system();
        }
    }
}

// ---------------------------------------------------------------------------
// Adjoint accumulation into the value grids.  A ray stays in one cell for
// many evaluations, so each lane sums its contributions to the four corners of
// the cell in hand, and the gradient grid takes them (hardware f64 atomics)
// only when it moves to another cell, and once at the end.  With 64 lanes
// some lane leaves its cell in most steps, a few lanes an instruction; and
// vmcnt counts atomics with loads and retires both in order, so in a wave
// that also loads cells an atomic holds up the next cell's loads, for a
// microsecond and more on a grid larger than L2.  So the sums of a left cell
// go to a queue in LDS, and once it holds a wave's worth, all lanes add one
// entry each.  A wave that loads no cells (the chain of the four-wave sweep)
// adds them at once (NoQueue).  N arrays on one grid share the cell test (u and v; on shared
// axes the depth too).
constexpr int QUEUE64 = 128;               // entries; at most 63 before a push of up to 64

template <int N>
struct CellSums {
    uint32_t iA = 0xFFFFFFFFu;             // no cell yet
    double s[N][4] = {};                   // corners A, B, C, D
};

// A wave's queue in LDS: [1 + 4 N][QUEUE64] doubles, each entry's cell and
// sums, and the number of entries after them.  The number lives in LDS as
// well: lanes join and leave the sweep at their own steps, and a register
// copy of a lane that sat out a push would be stale.
template <int N>
struct CellQueue {
    double *e;
    static constexpr int words = (1 + 4 * N) * QUEUE64 + 1;
    __device__ __forceinline__ int *count() const
    {
        return reinterpret_cast<int *>(e + (words - 1));
    }
};

// lanes of mask below this one
__device__ __forceinline__ int lanes_below(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Adds the queue's last entries to the gradient grids (null: not wanted)
// until fewer than `keep` are left.  Two neighbouring lanes take one entry,
// corners A and D and then B and C, which lie next to each other: the two
// atomics of a pair go out as one request (every request goes to memory, and
// their number is what the drains cost).
template <int N>
__device__ __forceinline__ void queue_drain(CellQueue<N> &q, double *const (&grad)[N],
                                            uint32_t nx, int keep)
{
    const uint64_t active = __builtin_amdgcn_ballot_w64(true);
    const int n = __popcll(active), rank = lanes_below(active);
    int count = *q.count();
    // (an odd lane out, as when a wave's last lane drains alone, takes both
    // corners by turns)
    const int pairs = n > 1 ? n / 2 : 1, side = n > 1 ? rank & 1 : 0;
    while (count >= keep) {
        const int take = __builtin_elementwise_min(pairs, count);
        if ((n > 1 ? rank / 2 : 0) < take) {
            const double *e = q.e + (count - take + rank / 2);
            const uint32_t iA = (uint32_t)__builtin_bit_cast(uint64_t, e[0]);
            for (int d = side; d < 2; d += n > 1 ? 2 : 1) {
                // sums A, B, C, D at 1 .. 4
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    if (!grad[k]) continue;
                    unsafeAtomicAdd(grad[k] + iA + d, e[(4 * k + (d ? 4 : 1)) * QUEUE64]);
                    unsafeAtomicAdd(grad[k] + iA + nx + d, e[(4 * k + (d ? 3 : 2)) * QUEUE64]);
                }
            }
        }
        count -= take;
    }
    *q.count() = count;
}

// Puts the sums of the lanes that have any into the queue (leave: the lanes
// to take), and empties it down to less than a wave's worth.
template <int N>
__device__ __forceinline__ void queue_push(CellQueue<N> &q, CellSums<N> &s, bool leave,
                                           double *const (&grad)[N], uint32_t nx)
{
    const bool put = leave & (s.iA != 0xFFFFFFFFu);
    const uint64_t mask = __builtin_amdgcn_ballot_w64(put);
    const int count = *q.count();
    if (put) {
        double *e = q.e + (count + lanes_below(mask));
        e[0] = __builtin_bit_cast(double, (uint64_t)s.iA);
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c) e[(1 + 4 * k + c) * QUEUE64] = s.s[k][c];
    }
    *q.count() = count + __popcll(mask);
    // (other lanes of the wave read them back)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    queue_drain<N>(q, grad, nx, 64);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// In a queue's place where a lane's sums go straight to the grids: in the
// chain wave of the four-wave sweep (16,384 rays x 2000 steps) the queue took
// 3.04 ms over a flat depth and 3.74 on shared axes, this 2.81 and 3.50, and
// sums with a cell test for each array 2.91 and 4.09.
template <int N>
struct NoQueue {
    static constexpr int words = 0;
};
template <int N>
__device__ __forceinline__ void queue_push(NoQueue<N> &, CellSums<N> &s, bool leave,
                                           double *const (&grad)[N], uint32_t nx)
{
    if (leave & (s.iA != 0xFFFFFFFFu)) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if (!grad[k]) continue;
            unsafeAtomicAdd(grad[k] + s.iA, s.s[k][0]);
            unsafeAtomicAdd(grad[k] + s.iA + nx, s.s[k][1]);
            unsafeAtomicAdd(grad[k] + s.iA + nx + 1u, s.s[k][2]);
            unsafeAtomicAdd(grad[k] + s.iA + 1u, s.s[k][3]);
        }
    }
}
template <int N>
__device__ __forceinline__ void queue_drain(NoQueue<N> &, double *const (&)[N], uint32_t, int)
{
}

// Adds the cotangents of one query to the sums of its cell: vb on the
// interpolated values, gxb and gyb on the cell-difference slopes.
template <int N, class Queue>
__device__ __forceinline__ void sums_add(CellSums<N> &s, Queue &q,
                                         double *const (&grad)[N], uint32_t nx,
                                         const Cell64 &cell, double rxs, double rys,
                                         const double (&vb)[N], const double (&gxb)[N],
                                         const double (&gyb)[N])
{
    if (__builtin_expect(__builtin_amdgcn_uicmp(cell.iA, s.iA, 33 /* != */) != 0, 0)) {
        __asm__ volatile("");
        const bool moved = cell.iA != s.iA;
        queue_push(q, s, moved, grad, nx);
        if (moved) {
            s = CellSums<N>{};
            s.iA = cell.iA;
        }
    }
    const double u = cell.u, w = cell.w;
    const double u1 = 1.0 - u, w1 = 1.0 - w;
    const double wa = u1 * w1, wb = u * w1, wc = u * w, wd = u1 * w;   // corner weights
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double gx = gxb[k] * rxs, gy = gyb[k] * rys;
        s.s[k][0] += vb[k] * wa - (gx + gy);
        s.s[k][1] += vb[k] * wb + gy;
        s.s[k][2] += vb[k] * wc;
        s.s[k][3] += vb[k] * wd + gx;
    }
}

// Gradient grids of an adjoint sweep (null: not wanted).
struct Grads64 {
    double *depth, *u, *v;
};

// The sums and queues of a sweep: of the depth alone and of the current's two
// arrays, or of all three on shared axes.
template <int BK, int CK, bool SH, template <int> class Queue = CellQueue>
struct Sums64 {
    static constexpr int NB = SH ? 3 : 1;
    static constexpr bool queued = Queue<1>::words > 0;
    static constexpr int words = (BK == BK_GRID ? Queue<NB>::words : 0) +
                                 (!SH && CK == CK_GRID ? Queue<2>::words : 0);
    CellSums<NB> b;
    CellSums<2> c;
    Queue<NB> qb;
    Queue<2> qc;

    // lds: `words` doubles of the wave's own
    __device__ __forceinline__ explicit Sums64(double *lds)
    {
        if constexpr (queued) {
            qb.e = lds;
            qc.e = lds + (BK == BK_GRID ? Queue<NB>::words : 0);
            if (BK == BK_GRID) *qb.count() = 0;
            if (!SH && CK == CK_GRID) *qc.count() = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    // the last sums of every lane, called by the whole wave
    __device__ __forceinline__ void finish(const Grads64 &Gr, uint32_t bnx, uint32_t cnx)
    {
        if constexpr (SH) {
            double *const g[3] = {Gr.depth, Gr.u, Gr.v};
            queue_push(qb, b, true, g, bnx);
            queue_drain(qb, g, bnx, 1);
        } else {
            if constexpr (BK == BK_GRID) {
                double *const g[1] = {Gr.depth};
                queue_push(qb, b, true, g, bnx);
                queue_drain(qb, g, bnx, 1);
            }
            if constexpr (CK == CK_GRID) {
                double *const g[2] = {Gr.u, Gr.v};
                queue_push(qc, c, true, g, cnx);
                queue_drain(qc, g, cnx, 1);
            }
        }
    }
};

// Adds one evaluation's field cotangents to the sums: hvb, hgx, hgy those of
// the depth query, g that of the derivatives (whose first two are also those
// of u and v), at the wavenumber (kx, ky).
template <int BK, int CK, bool SH, template <int> class Queue>
__device__ __forceinline__ void fields_add(const Grid64View &B, const Grid64View &C,
                                           const Grads64 &Gr, Sums64<BK, CK, SH, Queue> &sums,
                                           const Cell64 &bc, bool okb, const Cell64 &cc, bool okc,
                                           double hvb, double hgx, double hgy, const double g[4],
                                           double kx, double ky)
{
    // (a state of a finite row never errs; the guards keep a misuse in bounds)
    if constexpr (SH) {
        double *const grad[3] = {Gr.depth, Gr.u, Gr.v};
        if ((Gr.depth || Gr.u || Gr.v) && okb && okc)
            sums_add(sums.b, sums.qb, grad, (uint32_t)C.nx, cc, C.rxs, C.rys, {hvb, g[0], g[1]},
                        {hgx, -g[2] * kx, -g[2] * ky}, {hgy, -g[3] * kx, -g[3] * ky});
    } else {
        if constexpr (BK == BK_GRID) {
            double *const grad[1] = {Gr.depth};
            if (Gr.depth && okb)
                sums_add(sums.b, sums.qb, grad, (uint32_t)B.nx, bc, B.rxs, B.rys, {hvb}, {hgx},
                            {hgy});
        }
        if constexpr (CK == CK_GRID) {
            double *const grad[2] = {Gr.u, Gr.v};
            if ((Gr.u || Gr.v) && okc)
                sums_add(sums.c, sums.qc, grad, (uint32_t)C.nx, cc, C.rxs, C.rys, {g[0], g[1]},
                            {-g[2] * kx, -g[2] * ky}, {-g[3] * kx, -g[3] * ky});
        }
    }
}

// The linearisation of rhs64 at one stage point, as a record of LIN_N
// doubles, so that the cotangent chain can run apart from the (costlier)
// field queries and dispersion terms:
//   [0, 16)   M, row-major: the state cotangent is z = M g for a cotangent g
//             of (dx/dt, dy/dt, dkx/dt, dky/dt)
//   [16, 20)  hb: the depth-value cotangent is hb . g
//   20, 21, 22  c, kx, ky: the slope cotangents (g2 c, g3 c), (-g2 kx, -g3 kx),
//             (-g2 ky, -g3 ky) of depth, u and v
//   23, 24    bathymetry cell fractions (u, w); 25, 26 the current's
//   27        the two cells' corner-A indices, bit-packed (all ones: none)
constexpr int LIN_N = 28;

__device__ __forceinline__ double pack_cells(uint32_t b, uint32_t c)
{
    return __builtin_bit_cast(double, ((uint64_t)c << 32) | (uint64_t)b);
}
__device__ __forceinline__ void unpack_cells(double v, uint32_t &b, uint32_t &c)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    b = (uint32_t)u;
    c = (uint32_t)(u >> 32);
}

// Whether lin_apply reads field f of a linearisation record for the field
// kinds BK, CK (the only fields a ring is given): the depth terms (16-20, 23,
// 24) for gridded depth, the current's (21, 22, 25, 26) for a gridded
// current, and with a flat depth (depth_is_flat: zero slopes and derivatives)
// not the four zeros of M's x and y rows.  On shared cells (SH) the current's
// fractions serve the depth too.
template <int BK, int CK, bool SH>
__device__ constexpr bool lin_field_used(int f)
{
    if (f < 16)
        return !depth_is_flat<BK>() || f == 0 || f == 1 || f == 4 || f == 5 || f >= 8;
    if (f == 27) return true;
    if (SH && (f == 23 || f == 24)) return false;
    if (f <= 20 || f == 23 || f == 24) return BK == BK_GRID;
    return CK == CK_GRID;
}

// The linearisation record of one evaluation from its field values (the
// arithmetic of rhs64_lin below).
template <int BK, int CK>
__device__ __forceinline__ void lin_record(const FastConsts &K, const Val64 &h, const Val64 &u,
                                           const Val64 &v, const Cell64 &bc, const Cell64 &cc,
                                           bool okb, bool okc, double kx, double ky,
                                           double R[LIN_N])
{
    const double hh = h.val;
    const double k2 = __builtin_fma(kx, kx, ky * ky);
    const double rk = rsq_nr(k2);
    const double k = k2 * rk;
    const double ex = kx * rk, ey = ky * rk;
    const double q = k * hh;
    double e, em;
    exp_pair(q, e, em, K);
    const double ope = 1.0 + e;
    // one reciprocal square root, W = 1/sqrt(g k (1-e)(1+e)), gives the
    // reciprocal D = 1/((1-e)(1+e)) = g k W^2 and 1/sigma = W (1+e), as
    // sigma^2 = g k tanh(kh) = g k (1-e)/(1+e)
    const double gk = K.g * k;
    const double W = rsq_nr((gk * em) * ope);
    const double D = gk * (W * W);
    const double iope = em * D;
    const double T = em * iope;
    const double S = (4.0 * e) * (iope * iope);
    if (depth_is_flat<BK>()) {
        // no depth gradient: the rows of M are the current's and the
        // c_g k/|k| terms only
        const double rs = W * ope;
        const double N = __builtin_fma(q, S, T);
        const double cg = K.half_g * N * rs;
        const double Nq = 2.0 * S * (1.0 - q * T);
        const double cg_k = K.half_g * rs * (hh * Nq - N * cg * rs);
        const double tk = cg * rk;
        const double a = cg_k - tk;
        R[0] = u.dx; R[1] = v.dx; R[2] = 0.0; R[3] = 0.0;
        R[4] = u.dy; R[5] = v.dy; R[6] = 0.0; R[7] = 0.0;
        R[8] = a * ex * ex + tk; R[9] = a * ex * ey; R[10] = -u.gx; R[11] = -u.gy;
        R[12] = a * ey * ex; R[13] = a * ey * ey + tk; R[14] = -v.gx; R[15] = -v.gy;
        R[16] = 0.0; R[17] = 0.0; R[18] = 0.0; R[19] = 0.0; R[20] = 0.0;
        R[21] = kx; R[22] = ky;
        R[23] = 0.0; R[24] = 0.0; R[25] = cc.u; R[26] = cc.w;
        R[27] = pack_cells(0xFFFFFFFFu, (CK == CK_GRID && okc) ? cc.iA : 0xFFFFFFFFu);
        return;
    }
    const double invT = (ope * ope) * D;
    const double gkT = gk * T;
    const double rs = W * ope;
    const double sigma = gkT * rs;
    const double N = __builtin_fma(q, S, T);
    const double cg = K.half_g * N * rs;
    const double c = (-2.0 * k) * e * sigma * D;
    const double sig_h = K.half_g * (k * k) * S * rs;
    const double Nq = 2.0 * S * (1.0 - q * T);
    const double cg_k = K.half_g * rs * (hh * Nq - N * cg * rs);
    const double cg_h = K.half_g * rs * (k * Nq - N * sig_h * rs);
    const double coth2 = 0.5 * (T + invT);
    const double c_k = c * (rk + cg * rs - 2.0 * hh * coth2);
    const double c_h = c * (sig_h * rs - 2.0 * k * coth2);
    const double tk = cg * rk;
    const double hb[4] = {cg_h * ex, cg_h * ey, c_h * h.gx, c_h * h.gy};
    const double a = cg_k - tk;
    // rows of M (the partial derivatives of f, transposed)
    R[0] = hb[0] * h.dx + u.dx; R[1] = hb[1] * h.dx + v.dx;
    R[2] = hb[2] * h.dx;        R[3] = hb[3] * h.dx;
    R[4] = hb[0] * h.dy + u.dy; R[5] = hb[1] * h.dy + v.dy;
    R[6] = hb[2] * h.dy;        R[7] = hb[3] * h.dy;
    R[8] = a * ex * ex + tk;    R[9] = a * ex * ey;
    R[10] = c_k * ex * h.gx - u.gx; R[11] = c_k * ex * h.gy - u.gy;
    R[12] = a * ey * ex;        R[13] = a * ey * ey + tk;
    R[14] = c_k * ey * h.gx - v.gx; R[15] = c_k * ey * h.gy - v.gy;
    R[16] = hb[0]; R[17] = hb[1]; R[18] = hb[2]; R[19] = hb[3];
    R[20] = c; R[21] = kx; R[22] = ky;
    R[23] = bc.u; R[24] = bc.w; R[25] = cc.u; R[26] = cc.w;
    // a state of a finite row never errs; the marks keep a misuse in bounds
    R[27] = pack_cells((BK == BK_GRID && okb) ? bc.iA : 0xFFFFFFFFu,
                       (CK == CK_GRID && okc) ? cc.iA : 0xFFFFFFFFu);
}

template <int BK, int CK, bool SH>
__device__ __forceinline__ void rhs64_lin(const Grid64View &B, const Grid64Ptrs &BP,
                                          const Grid64View &C, const Grid64Ptrs &CP,
                                          const Fields64 &F, const Slots64<BK, CK, SH> &sl,
                                          const FastConsts &K, double x, double y, double kx,
                                          double ky, double R[LIN_N])
{
    // as rhs64: first with the cells in hand, then the full queries for the
    // lanes whose target is not inside them
    Point64 p;
    const uint32_t off = point64_fast<BK, CK, SH>(B, BP, C, CP, F, sl, x, y, p);
    lin_record<BK, CK>(K, p.h, p.u, p.v, p.bc, p.cc, p.okb, p.okc, kx, ky, R);
    if (__builtin_expect(any_off64<BK, CK>(off), 0)) {
        __asm__ volatile("");
        if (off >= OUT64) {
            point64_full<BK, CK>(BP, CP, F, x, y, p);
            lin_record<BK, CK>(K, p.h, p.u, p.v, p.bc, p.cc, p.okb, p.okc, kx, ky, R);
        }
    }
}

// Applies a linearisation record R to the cotangent g: z = M g, and the
// field-value cotangents to the sums.
template <int BK, int CK, bool SH, template <int> class Queue>
__device__ __forceinline__ void lin_apply(const double R[LIN_N], const Grid64View &B,
                                          const Grid64View &C, const Grads64 &Gr,
                                          Sums64<BK, CK, SH, Queue> &sums, const double g[4],
                                          double z[4])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z[i] = R[4 * i] * g[0] + R[4 * i + 1] * g[1];
        if (!depth_is_flat<BK>() || i >= 2)    // (R[2], R[3], R[6], R[7] are zero)
            z[i] += R[4 * i + 2] * g[2] + R[4 * i + 3] * g[3];
    }
    uint32_t ib, ic;
    unpack_cells(R[27], ib, ic);
    double hbar = 0.0;
    if (BK == BK_GRID)
        hbar = (R[16] * g[0] + R[17] * g[1]) + (R[18] * g[2] + R[19] * g[3]);
    fields_add(B, C, Gr, sums, Cell64{ib, R[23], R[24]}, ib != 0xFFFFFFFFu,
                           Cell64{ic, R[25], R[26]}, ic != 0xFFFFFFFFu, hbar, g[2] * R[20],
                           g[3] * R[20], g, R[21], R[22]);
}

// The fields of a record that lin_apply reads, and where each stands among
// them.
template <int BK, int CK, bool SH>
__device__ constexpr int lin_place(int f)
{
    int n = 0;
    for (int g = 0; g < f; ++g) n += lin_field_used<BK, CK, SH>(g) ? 1 : 0;
    return n;
}

// rhs64 and its linearisation at once, for a flat depth (depth_is_flat): the
// record R and the derivatives, which share the field values and most of the
// dispersion terms.  The derivatives are rhs64's own, bitwise (the same odes
// on the same values, in the forward's math mode): the stage points formed
// from them are then those the forward evaluated, so none of a finite row's
// errs.  Derivatives from the record's group velocity, an ulp off, take about
// eight operations a stage less (262,144 rays x 3000 steps of a forward and
// its sweep 65.4 against 66.2 ms), but put a stage point that the forward met
// on the grid's edge outside it, and one at a cell line into the next cell,
// whose values may be missing.
template <int BK, int CK, int MATH>
__device__ __forceinline__ void rhs64_with_lin(const Grid64View &B, const Grid64Ptrs &BP,
                                               const Grid64View &C, const Grid64Ptrs &CP,
                                               const Fields64 &F,
                                               const Slots64<BK, CK, false> &sl,
                                               const FastConsts &K, const double s[4],
                                               double R[LIN_N], double d[4])
{
    static_assert(depth_is_flat<BK>(), "no depth gradient");
    Point64 p;
    auto eval = [&] {
        lin_record<BK, CK>(K, p.h, p.u, p.v, p.bc, p.cc, p.okb, p.okc, s[2], s[3], R);
        odes<MATH, true, CK == CK_CONSTANT>(K, p.okb ? p.h.val : MR_NAN, p.h.gx, p.h.gy, p.okc,
                                            p.u.val, p.v.val, p.u.gx, p.u.gy, p.v.gx, p.v.gy,
                                            s[2], s[3], d[0], d[1], d[2], d[3]);
    };
    const uint32_t off = point64_fast<BK, CK, false>(B, BP, C, CP, F, sl, s[0], s[1], p);
    eval();
    if (__builtin_expect(any_off64<BK, CK>(off), 0)) {
        __asm__ volatile("");
        if (off >= OUT64) {
            point64_full<BK, CK>(BP, CP, F, s[0], s[1], p);
            eval();
        }
    }
}

// Vector-Jacobian product of rhs64 at (x, y, kx, ky): given the cotangent
// (g0, g1, g2, g3) of (dx/dt, dy/dt, dkx/dt, dky/dt), adds the state
// cotangent to (bx, by, bkx, bky) and the field-value cotangents to the
// accumulators.  The dispersion terms are evaluated with the closed forms of
// the fast mode whatever the forward's math mode: only the derivative
// depends on them.  The state must be one at which rhs64 is finite.
template <int BK, int CK, bool SH>
__device__ __forceinline__ void rhs64_vjp(const Grid64View &B, const Grid64Ptrs &BP,
                                          const Grid64View &C, const Grid64Ptrs &CP,
                                          const Fields64 &F, const Slots64<BK, CK, SH> &sl,
                                          const Grads64 &Gr, Sums64<BK, CK, SH> &sums,
                                          const FastConsts &K, double x, double y, double kx,
                                          double ky, double g0, double g1, double g2, double g3, double &bx,
                                          double &by, double &bkx, double &bky)
{
    // the field values as in rhs64: from the cells in hand, then the full
    // queries for the lanes whose target is not inside them (the product and
    // the accumulation below run once, after both)
    Point64 p;
    const uint32_t off = point64_fast<BK, CK, SH>(B, BP, C, CP, F, sl, x, y, p);
    if (__builtin_expect(any_off64<BK, CK>(off), 0)) {
        __asm__ volatile("");
        if (off >= OUT64) point64_full<BK, CK>(BP, CP, F, x, y, p);
    }
    const Val64 &h = p.h, &u = p.u, &v = p.v;
    const Cell64 &bc = p.bc, &cc = p.cc;
    const bool okb = p.okb, okc = p.okc;
    const double hh = h.val;
    const double k2 = __builtin_fma(kx, kx, ky * ky);
    const double rk = rsq_nr(k2);                       // 1/k
    const double k = k2 * rk;
    const double ex = kx * rk, ey = ky * rk;
    const double q = k * hh;
    double e, em;
    exp_pair(q, e, em, K);                               // e = exp(-2q), em = 1 - e
    const double ope = 1.0 + e;
    // 1/((1-e)(1+e)) and 1/sigma from one reciprocal square root, as in
    // lin_record
    const double gk = K.g * k;
    const double W = rsq_nr((gk * em) * ope);
    const double D = gk * (W * W);
    const double iope = em * D;
    const double T = em * iope;                         // tanh q
    const double S = (4.0 * e) * (iope * iope);         // sech^2 q
    const double rs = W * ope;                          // 1/sigma
    const double N = __builtin_fma(q, S, T);
    const double cg = K.half_g * N * rs;
    const double Nq = 2.0 * S * (1.0 - q * T);
    const double cg_k = K.half_g * rs * (hh * Nq - N * cg * rs);
    const double P = g0 * ex + g1 * ey;                 // cotangent of cg
    const double tk = cg * rk;
    double hvb = 0.0, hgx = 0.0, hgy = 0.0;             // cotangents of the depth query
    if (depth_is_flat<BK>()) {
        // no depth gradient: the terms of c and of the depth cotangent vanish
        bkx += (cg_k * P) * ex + tk * (g0 - P * ex) - g2 * u.gx - g3 * u.gy;
        bky += (cg_k * P) * ey + tk * (g1 - P * ey) - g2 * v.gx - g3 * v.gy;
        bx += g0 * u.dx + g1 * v.dx;
        by += g0 * u.dy + g1 * v.dy;
    } else {
        const double invT = (ope * ope) * D;            // 1/tanh q
        const double sigma = (gk * T) * rs;
        const double c = (-2.0 * k) * e * sigma * D;
        const double sig_h = K.half_g * (k * k) * S * rs;   // d sigma / dh
        const double cg_h = K.half_g * rs * (k * Nq - N * sig_h * rs);
        const double coth2 = 0.5 * (T + invT);
        const double c_k = c * (rk + cg * rs - 2.0 * hh * coth2);
        const double c_h = c * (sig_h * rs - 2.0 * k * coth2);
        const double cbar = g2 * h.gx + g3 * h.gy;      // cotangent of c
        const double hbar = cg_h * P + c_h * cbar;
        bkx += (cg_k * P) * ex + tk * (g0 - P * ex) + (c_k * cbar) * ex - g2 * u.gx - g3 * u.gy;
        bky += (cg_k * P) * ey + tk * (g1 - P * ey) + (c_k * cbar) * ey - g2 * v.gx - g3 * v.gy;
        bx += hbar * h.dx + g0 * u.dx + g1 * v.dx;
        by += hbar * h.dy + g0 * u.dy + g1 * v.dy;
        hvb = hbar;
        hgx = g2 * c;
        hgy = g3 * c;
    }
    const double g[4] = {g0, g1, g2, g3};
    fields_add(B, C, Gr, sums, bc, okb, cc, okc, hvb, hgx, hgy, g, kx, ky);
}

}  // namespace mr
